"""GPU tests of paths inside the kernels that depend on the data or on how a shape meets the tiles, against
the fp32 oracle with the tolerances of the parity tests (out max-abs 2e-2, gradients relative L2 5e-2)."""
import pytest
import torch

from oracle.attention_oracle import attention_backward, attention_forward, reference_grads
from triton_flashattn_amd import AlibiBias, flash_attention_fn, flash_attention_qkvpacked_fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_forward_reference_point_of_growing_scores(gpu_device, D, dtype):
    """The reference point of the exponentials is raised only when their sum grows past a limit: scores that grow
    (or fall) along the keys slowly, by a few powers of two per key and by jumps beyond the range of fp16, with
    and without a bias, from one to several key steps and with a ragged last one."""
    g = torch.Generator().manual_seed(D)
    for slope, N, causal, bias_kind in [(0.05, 333, False, None), (1.5, 333, False, "f"), (-1.5, 256, False, None),
                                        (0.4, 300, True, None), (25.0, 150, False, None), (1.5, 160, True, "b")]:
        M = N if causal else 70
        q = torch.randn(1, M, 2, D, generator=g)
        k = torch.randn(1, N, 2, D, generator=g) * 0.5
        q[..., 0], k[..., 0] = 4.0, torch.arange(N).float()[None, :, None] * (slope / 4.0)
        q, k, v = (t.to(dtype).to(gpu_device) for t in (q, k, torch.randn(1, N, 2, D, generator=g)))
        bias = None
        if bias_kind == "f":
            bias = torch.randn(1, 2, M, N, generator=g).to(dtype).to(gpu_device)
        elif bias_kind == "b":
            bias = torch.rand(1, 2, M, N, generator=g) > 0.5
            bias[..., 0] = True
            bias = bias.to(gpu_device)
        with torch.no_grad():
            out = flash_attention_fn(q, k, v, bias, causal, 1.0)
        ref, _ = attention_forward(q, k, v, bias, causal, 1.0)
        # scores reach 3750 (25 x 150): the two fp32 sums of a score may differ by 2^-22 of that in natural units,
        # so a weight by 1e-3 and the output (values up to 4) by less than the tolerance
        err = (out.float() - ref).abs().max().item()
        assert err <= 2e-2, (slope, N, causal, bias_kind, err)


@pytest.mark.parametrize("kind", [None, "dense", "row"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,causal", [(32, False), (64, False), (128, True), (256, False)])
def test_forward_error_where_few_keys_carry_a_row(gpu_device, D, causal, dtype, kind):
    """Scores of standard deviation 8, where one weight is most of a row: it is 1, which rounds to itself, whenever it
    raised the reference point, so that the output's own rounding is most of its error (1.13 to 1.15 times it, 1.19 with
    a running maximum that is raised at 2^8; 1.26 to 1.37 where the point is left behind further)."""
    g = torch.Generator().manual_seed(D)
    S, H = 700, 8
    q, k, v = (torch.randn(2, S, H, D, generator=g).to(gpu_device) for _ in range(3))
    q, k, v = q.to(dtype), (k * (8 if kind is None else 1)).to(dtype), v.to(dtype)
    bias = None
    if kind is not None:
        bias = (torch.randn((2, H, S, S) if kind == "dense" else (2, H, 1, S), generator=g) * 8).to(dtype).to(gpu_device)
    with torch.no_grad():
        out = flash_attention_fn(q, k, v, bias, causal).double()
    qd, kd, vd = (t.double().transpose(1, 2).contiguous() for t in (q, k, v))
    s = qd @ kd.transpose(2, 3).contiguous() * D ** -0.5
    s = s if bias is None else s + bias.double()
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=gpu_device).triu(1), float("-inf"))
    ref = (s.softmax(-1) @ vd).transpose(1, 2)
    assert (out - ref).norm() <= 1.22 * (ref.to(dtype).double() - ref).norm()


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_forward_of_biases_that_grow_along_the_keys(gpu_device, D, dtype):
    """The rules for raising the reference point under a distance penalty: rows that grow in every block, in every few,
    up to the diagonal and down behind it, all the way or not at all, with a ragged last step and rows that start masked."""
    g = torch.Generator().manual_seed(D)
    H = 6
    slopes = torch.tensor([3.0, 0.7, 0.2, 0.05, 0.0, -0.5])
    for M, N, causal in [(333, 333, True), (256, 256, True), (150, 1000, False), (130, 321, False)]:
        q, k, v = (torch.randn(1, n, H, D, generator=g).to(dtype).to(gpu_device) for n in (M, N, N))
        penalty = AlibiBias(slopes.abs().to(gpu_device))
        dist = penalty.materialize(M, N)
        row = slopes[None, :, None, None].to(gpu_device) * torch.arange(N, device=gpu_device)
        masked = dist.clone()
        masked[..., :70] = float("-inf")
        if causal:
            masked[..., torch.arange(M) < 70, 0] = 0.0
        for name, bias, dense in [("alibi", penalty, dist), ("tensor", dist.to(dtype), dist.to(dtype)), ("fp32", dist, dist),
                                  ("row", row, row), ("row16", row.to(dtype), row.to(dtype)), ("masked", masked, masked)]:
            with torch.no_grad():
                out = flash_attention_fn(q, k, v, bias, causal)
            ref, _ = attention_forward(q, k, v, dense.expand(1, H, M, N), causal)
            # biases reach 3000: a bias times log2 e and its fp32 sum with the score are off by 2^-12 at most, a weight by
            # 2e-4, the output (values up to 4.5) by 1e-3 and by its own rounding
            err = (out.float() - ref).abs().max().item()
            assert err <= 2e-2, (name, M, N, causal, err)


def rel_l2(a, b):
    """||a - b|| / ||b||, measured against an RMS floor of 1e-3 where the reference is zero up to rounding."""
    return ((a.float() - b).norm() / b.norm().clamp_min(1e-3 * b.numel() ** 0.5)).item()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias_kind", [None, "dense", "row", "alibi", "bool"])
def test_backward_ragged_tiles_with_low_scores(gpu_device, D, bias_kind):
    """Keys past N and rows past M run through the unmasked steps of the backward kernels: their probabilities,
    2^(0 - LSE) with an LSE far below zero, overflow, and nothing of them may reach a result."""
    g = torch.Generator().manual_seed(D)
    for M, N, causal in [(517, 130, False), (450, 321, False), (333, 1, False), (389, 389, True), (97, 640, False)]:
        if bias_kind == "alibi" and N == 1:
            continue
        mk = lambda n: torch.randn(1, n, 2, D, generator=g)
        q, k, v, do = mk(M), mk(N), mk(N), mk(M)
        # scores of about -144, with an ordinary spread: were a weight near one, its dS = P (dP - delta) would be the
        # difference of two nearly equal numbers, and delta carries the rounding of the bf16 output, 2^-8 of |o| |do|
        q[..., 0], k[..., 0], scale = 34.0, -34.0 - torch.rand(1, N, 2, generator=g) / 4, 0.125
        q, k, v = (t.bfloat16().to(gpu_device).requires_grad_(True) for t in (q, k, v))
        do = do.bfloat16().to(gpu_device)
        bias, dense, grad_of = None, None, None
        if bias_kind in ("dense", "row"):
            shape = (1, 2, M if bias_kind == "dense" else 1, N)
            bias = (torch.randn(shape, generator=g) - 100.0).bfloat16().to(gpu_device).requires_grad_(True)
            dense, grad_of = bias.detach(), bias
        elif bias_kind == "alibi":
            slopes = torch.tensor([0.02, 0.1], device=gpu_device).requires_grad_(True)
            bias, grad_of = AlibiBias(slopes), slopes
            dense = bias.materialize(M, N).detach()
        elif bias_kind == "bool":
            bias = dense = (torch.rand(1, 2, M, N, generator=g) > 0.3).index_fill(3, torch.tensor([0]), True).to(gpu_device)
        out = flash_attention_fn(q, k, v, bias, causal, scale)
        wanted = [q, k, v] + ([] if grad_of is None else [grad_of])
        grads = torch.autograd.grad(out, wanted, do)
        full = None if dense is None else dense.expand(1, 2, M, N)
        o, lse = attention_forward(q.detach(), k.detach(), v.detach(), full, causal, scale)
        dq, dk, dv, db, _ = attention_backward(do, q.detach(), k.detach(), v.detach(), o, lse, full, causal, scale)
        assert (out.float() - o).abs().max().item() <= 2 ** -7 * v.abs().max().item(), (M, N)  # P and out in bf16
        for name, a, b in zip("qkv", grads, (dq, dk, dv)):
            assert rel_l2(a, b) <= 5e-2, (name, M, N, causal)
        if bias_kind == "dense":
            assert rel_l2(grads[3], db) <= 5e-2, (M, N)
        elif bias_kind == "row":
            # a sum over M rows of terms that the kernel rounds nowhere: bounded by the size of its terms, and where
            # they vanish (one key: dP - delta is the rounding of two equal sums of D products) by M such roundings
            limit = 1e-2 * db.abs().sum(2).max() + M * D * 2 ** -22
            assert (grads[3].float() - db.sum(2, keepdim=True)).abs().max() <= limit, (M, N)
        elif bias_kind == "alibi":
            i, j = torch.arange(M, device=gpu_device)[:, None], torch.arange(N, device=gpu_device)[None, :]
            terms = db[0] * -(i * (N / M) - j).abs()
            assert (grads[3] - terms.sum((1, 2))).abs().max() <= 1e-2 * terms.abs().sum((1, 2)).max(), (M, N)


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
def test_gradient_of_a_shared_bias(gpu_device, D):
    """A bias shared by batches and / or heads: its gradient is summed over the pairs in one kernel, in tiles of 128
    rows and 64 keys, the pairs split between work-groups where the tiles are few (all cases but the last two)."""
    g = torch.Generator().manual_seed(D)
    cases = [((1, 3, 128, 64), 5, 3, torch.bfloat16, False), ((1, 2, 129, 65), 7, 2, torch.float32, False),
             ((2, 1, 197, 197), 2, 3, torch.float16, True), ((1, 1, 2, 3), 3, 3, torch.float32, False),
             ((1, 1, 127, 333), 2, 5, torch.bfloat16, False), ((1, 1, 64, 64), 1, 2, torch.float32, True)]
    if D <= 64:
        cases += [((1, 8, 520, 520), 2, 8, torch.float32, True), ((1, 8, 300, 770), 3, 8, torch.bfloat16, False)]
    for shape, B, H, bias_dtype, causal in cases:
        M, N = shape[2:]
        dtype = torch.float16 if bias_dtype == torch.float16 else torch.bfloat16
        mk = lambda n: torch.randn(B, n, H, D, generator=g).to(dtype).to(gpu_device).requires_grad_(True)
        q, k, v, do = mk(M), mk(N), mk(N), mk(M).detach()
        bias = torch.randn(shape, generator=g).to(bias_dtype).to(gpu_device).requires_grad_(True)
        out = flash_attention_fn(q, k, v, bias, causal)
        grads = torch.autograd.grad(out, (q, k, v, bias), do)
        again = torch.autograd.grad(flash_attention_fn(q, k, v, bias, causal), bias, do)[0]
        assert torch.equal(grads[3], again)
        full = bias.detach().expand(B, H, M, N)
        o, lse = attention_forward(q.detach(), k.detach(), v.detach(), full, causal)
        dq, dk, dv, db, _ = attention_backward(do, q.detach(), k.detach(), v.detach(), o, lse, full, causal)
        for name, a, b in zip(("dq", "dk", "dv", "dbias"), grads, (dq, dk, dv, db.sum_to_size(shape))):
            assert rel_l2(a, b) <= 5e-2, (name, shape, B, H, causal, rel_l2(a, b))


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
def test_pairs_that_share_a_bias(gpu_device, D):
    """The walk over the (batch, head) pairs of a tile: several pairs to a work-group, over heads and batches, shares that
    start in the middle of a batch, an empty last share, one, two and three pairs without shares; rows that are accessed
    four elements at a time and rows that are not (odd lengths, a padded pitch, transposed)."""
    g = torch.Generator().manual_seed(D)
    cases = [((1, 1, 300, 300), 6, 8, torch.bfloat16, True), ((300, 300), 3, 16, torch.float32, False),
             ((2, 1, 260, 200), 2, 24, torch.bfloat16, False), ((1, 8, 300, 300), 7, 8, torch.float32, False),
             ((1, 16, 300, 200), 3, 16, torch.float16, False), ((1, 24, 260, 129), 2, 24, torch.bfloat16, False),
             ((3, 1, 1000, 310), 3, 2, torch.bfloat16, False), ((1, 33, 130, 257), 4, 33, torch.float32, False)]
    for i, (shape, B, H, bias_dtype, causal) in enumerate(cases):
        M, N = shape[-2:]
        dtype = torch.float16 if bias_dtype == torch.float16 else torch.bfloat16
        mk = lambda n: torch.randn(B, n, H, D, generator=g).to(dtype).to(gpu_device).requires_grad_(True)
        q, k, v, do = mk(M), mk(N), mk(N), mk(M).detach()
        bias = torch.randn(shape, generator=g).to(bias_dtype).to(gpu_device)
        if i % 3 == 1:
            bias = torch.nn.functional.pad(bias, (0, 4))[..., :N]
        elif i % 3 == 2:
            bias = bias.transpose(-1, -2).contiguous().transpose(-1, -2)
        bias.requires_grad_(True)
        got = torch.autograd.grad(flash_attention_fn(q, k, v, bias, causal), bias, do)[0]
        full = bias.detach().expand(B, H, M, N)
        o, lse = attention_forward(q.detach(), k.detach(), v.detach(), full, causal)
        want = attention_backward(do, q.detach(), k.detach(), v.detach(), o, lse, full, causal)[3].sum_to_size(shape)
        # (the terms are rounded once each, in the products: the sum over the pairs adds no error of its own)
        assert got.shape == want.shape and rel_l2(got, want) <= 2e-2, (shape, B, H, causal, rel_l2(got, want))


@pytest.mark.parametrize("d_qk,d_v", [(8, 8), (24, 24), (40, 56), (80, 80), (96, 40), (72, 120), (64, 128)])
def test_head_dims_below_the_kernels(gpu_device, d_qk, d_v):
    """Head dims that are whole 16-byte chunks run at the next head dim of the kernels without padded copies: both
    directions, plain, split over the keys, with masks and causal, and nothing is written past a row."""
    g = torch.Generator().manual_seed(d_qk)
    for B, M, N, H, causal, kind in [(2, 130, 130, 2, True, None), (1, 77, 200, 3, False, "dense"), (2, 64, 333, 2, False, "bool"),
                                     (1, 40, 2200, 1, False, None), (2, 257, 257, 2, False, None)]:
        mk = lambda n, d: torch.randn(B, n, H, d, generator=g).bfloat16().to(gpu_device).requires_grad_(True)
        # (the tensors are slices of wider ones, whose other columns hold NaN)
        wide = lambda n, d: torch.cat([mk(n, d).detach(), torch.full((B, n, H, 8), float("nan"), device=gpu_device, dtype=torch.bfloat16)], -1)
        q, k, v, do = (wide(M, d_qk)[..., :d_qk].requires_grad_(True), wide(N, d_qk)[..., :d_qk].requires_grad_(True),
                       wide(N, d_v)[..., :d_v].requires_grad_(True), mk(M, d_v).detach())
        bias = None
        if kind == "dense":
            bias = torch.randn(B, H, M, N, generator=g).bfloat16().to(gpu_device).requires_grad_(True)
        elif kind == "bool":
            bias = (torch.rand(B, H, M, N, generator=g) > 0.3).index_fill(3, torch.tensor([0]), True).to(gpu_device)
        out = flash_attention_fn(q, k, v, bias, causal)
        wanted = [q, k, v] + ([bias] if kind == "dense" else [])
        grads = torch.autograd.grad(out, wanted, do)
        b = None if bias is None else bias.detach()
        o, lse = attention_forward(q.detach(), k.detach(), v.detach(), b, causal)
        dq, dk, dv, db, _ = attention_backward(do, q.detach(), k.detach(), v.detach(), o, lse, b, causal)
        assert out.shape == o.shape and (out.float() - o).abs().max().item() <= 2e-2
        for name, a, ref in zip(("dq", "dk", "dv", "dbias"), grads, (dq, dk, dv, db)):
            assert a.shape == ref.shape and rel_l2(a, ref) <= 5e-2, (name, M, N, causal, kind)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,d_v", [(8, 8), (24, 24), (40, 40), (64, 64), (72, 72), (80, 80), (120, 120), (128, 128), (8, 128), (56, 72)])
def test_infinite_keys_at_head_dims_below_the_kernels(gpu_device, d, d_v, dtype):
    """A key of -inf in one column, met by positive queries, has scores of -inf and a weight of zero, as at the head dims
    of the kernels: everything but the column of dQ that multiplies it stays finite."""
    g = torch.Generator().manual_seed(d)
    for M, N, causal, kind in [(130, 200, False, None), (97, 333, False, "bool"), (64, 2500, False, None), (150, 150, True, "dense")]:
        mk = lambda n, w=d: torch.randn(2, n, 2, w, generator=g).to(dtype)
        q, k, v, do = mk(M), mk(N), mk(N, d_v), mk(M, d_v)
        q[..., 0] = q[..., 0].abs() + 0.1
        k[:, 1::3, :, 0] = float("-inf")
        ins = [t.to(gpu_device).requires_grad_(True) for t in (q, k, v)]
        do = do.to(gpu_device)
        bias = None
        if kind == "bool":
            bias = (torch.rand(2, 2, M, N, generator=g) > 0.3).index_fill(3, torch.tensor([0]), True).to(gpu_device)
        elif kind == "dense":
            bias = torch.randn(2, 2, M, N, generator=g).to(dtype).to(gpu_device)
        out = flash_attention_fn(*ins, bias, causal)
        dq, dk, dv = torch.autograd.grad(out, ins, do)
        q, k, v = (t.detach() for t in ins)
        o, lse = attention_forward(q, k, v, bias, causal)
        want = attention_backward(do, q, k, v, o, lse, bias, causal)
        assert o.isfinite().all() and (out.float() - o).abs().max().item() <= 2e-2, (M, N, kind)
        for name, a, b in (("dq", dq[..., 1:], want[0][..., 1:]), ("dk", dk, want[1]), ("dv", dv, want[2])):
            assert b.isfinite().all() and rel_l2(a, b) <= 5e-2, (name, M, N, kind)


def test_host_path_equals_the_autograd_classes(gpu_device):
    """flash_attention_fn goes through the C++ host path; FlashAttentionFn, called directly, through Python and ctypes:
    the same kernels on the same arguments, bit for bit, for every kind of bias, layout and set of wanted gradients."""
    from triton_flashattn_amd.flash_attention import FlashAttentionFn, FlashAttentionQKVPackedFn, flash_attention_qkvpacked_fn
    dev, g = gpu_device, torch.Generator().manual_seed(0)
    B, M, N, H, D = 2, 75, 131, 4, 64
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    slopes = torch.tensor([0.5, 0.1, 0.02, 0.01], device=dev)
    biases = [None, rnd(B, H, M, N), rnd(1, H, M, N).float(), rnd(H, 1, N).half(), rnd(N), rnd(M, N), rnd(B, 1, 1, N) > -1.0, slopes]
    for i, bias in enumerate(biases):
        for want in ((1, 1, 1, 1), (1, 0, 0, 0), (0, 1, 0, 1), (0, 0, 1, 0), (0, 0, 0, 1)):
            if want == (0, 0, 0, 1) and (bias is None or bias.dtype == torch.bool):
                continue
            # sequence-major, head-major, and rows that the kernels cannot read in place
            q = rnd(B, M, H, D) if i % 3 == 0 else rnd(B, H, M, D).transpose(1, 2) if i % 3 == 1 else rnd(B, M, H, D + 2)[..., :D]
            inputs = [q, rnd(B, N, H, D), rnd(B, N, H, D)]
            is_alibi = bias is slopes
            extra = None if bias is None else bias.clone()
            leaves = []
            for t, w in zip(inputs + ([] if extra is None or extra.dtype == torch.bool else [extra]), want):
                t.requires_grad_(bool(w))
                if w:
                    leaves.append(t)
            do = rnd(B, M, H, D) if i % 2 else rnd(B, M, H, 1).expand(B, M, H, D)
            ours = flash_attention_fn(*inputs, AlibiBias(extra) if is_alibi else extra, False)
            ref = FlashAttentionFn.apply(*inputs, None if is_alibi else extra, False, None, extra if is_alibi else None)
            assert "AttentionNode" in ours.grad_fn.name()
            assert torch.equal(ours, ref)
            for a, b in zip(torch.autograd.grad(ours, leaves, do), torch.autograd.grad(ref, leaves, do)):
                assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b), (i, want)
    qkv = rnd(B, M, 3, H, D).requires_grad_(True)
    for bias in (None, rnd(1, H, M, M).requires_grad_(True)):
        leaves, do = [qkv] + ([] if bias is None else [bias]), rnd(B, M, H, D)
        ours, ref = flash_attention_qkvpacked_fn(qkv, bias, True), FlashAttentionQKVPackedFn.apply(qkv, bias, True, None, None)
        for a, b in zip((ours,) + torch.autograd.grad(ours, leaves, do), (ref,) + torch.autograd.grad(ref, leaves, do)):
            assert torch.equal(a, b)
    # without gradients the host path goes below autograd
    with torch.no_grad():
        assert torch.equal(flash_attention_qkvpacked_fn(qkv, None, True), FlashAttentionQKVPackedFn.apply(qkv, None, True, None, None))
        for bias in biases:
            for q in (rnd(B, M, H, D), rnd(B, H, M, D).transpose(1, 2), rnd(B, M, H, D + 2)[..., :D]):
                k, v, is_alibi = rnd(B, N, H, D), rnd(B, N, H, D), bias is slopes
                ref = FlashAttentionFn.apply(q, k, v, None if is_alibi else bias, False, None, bias if is_alibi else None)
                assert torch.equal(flash_attention_fn(q, k, v, AlibiBias(bias) if is_alibi else bias, False), ref)
    with pytest.raises(ValueError):
        flash_attention_fn(qkv[:, :, 0], qkv[:, :5, 1], qkv[:, :5, 2], None, True)


def test_host_path_with_hooks_views_and_transforms(gpu_device):
    """What programs put around an autograd function: saved-tensor hooks whose tensors come back elsewhere or changed,
    a bias written to before the backward, tracing and transforms.  (What a hook may hand back wrongly is turned into
    an error on the host; nothing is launched for it.)"""
    dev, g = gpu_device, torch.Generator().manual_seed(0)
    B, S, H, D = 2, 75, 4, 64
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    q, k, v = (rnd(B, S, H, D).requires_grad_(True) for _ in range(3))
    do, bias = rnd(B, S, H, D), rnd(H, S, S)
    want = torch.autograd.grad(flash_attention_fn(q, k, v, bias), (q, k, v), do)
    # through host memory and back, and as tensors of another layout
    with torch.autograd.graph.save_on_cpu():
        out = flash_attention_fn(q, k, v, bias)
    for a, b in zip(torch.autograd.grad(out, (q, k, v), do), want):
        assert torch.equal(a, b)
    strided = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2) if t.dim() == 4 and t.shape[-1] == D else t
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, strided):
        out = flash_attention_fn(q, k, v, bias)
    for a, b in zip(torch.autograd.grad(out, (q, k, v), do), want):
        assert torch.equal(a, b)
    for spoil in (lambda t: t.cpu(), lambda t: t[:, :7], lambda t: t.float() if t.dtype == torch.bfloat16 else t.bfloat16(),
                  lambda t: t.cpu() if t.dim() == 3 else t, lambda t: t[0]):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, spoil):
            out = flash_attention_fn(q, k, v, bias)
        with pytest.raises(ValueError):
            out.backward(do)
    # a bias with a missing dimension is read again by the backward, where the kernels can read it in place
    bias = rnd(H, 1, S)
    out = flash_attention_fn(q, k, v, bias)
    bias.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(do)
    # a trace runs the kernels on the inputs it is given later
    call = lambda a, b, c: flash_attention_fn(a, b, c, None, True)
    one, other = [rnd(B, S, H, D) for _ in range(3)], [rnd(B, S, H, D) for _ in range(3)]
    traced = torch.jit.trace(call, one, check_trace=False)
    assert torch.equal(traced(*other), call(*other))
    # a transform is refused, also where it wraps none of the arguments
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: call(*one) * x)(rnd(3, 1))


@pytest.mark.parametrize("D", [64, 72, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_dq_of_few_rows(gpu_device, D, causal):
    """Up to 64 query rows the dQ kernel takes rows of Q, dO and O by other loads than above: around that line, with every kind of
    bias, by the kernel that forms delta itself and, with keys enough for several work-groups to share them, by shares."""
    for M, N in ([(5, 5), (33, 33), (64, 64), (65, 65)] if causal else [(1, 70), (31, 2100), (63, 33), (64, 129), (65, 129), (97, 64)]):
        g = torch.Generator().manual_seed(M + N)
        q, k, v, do = (torch.randn(2, s, 3, D, generator=g).bfloat16().to(gpu_device) for s in (M, N, N, M))
        ins = [t.requires_grad_(True) for t in (q, k, v)]
        dense = torch.randn(2, 3, M, N, generator=g).to(gpu_device)
        # (the first key is visible: scores of a row without a visible key are -1e6, rounded to 2^-4, and its weights off by 6 %)
        mask = (dense > -1.5) | (torch.arange(N, device=gpu_device) == 0)
        alibi = AlibiBias(torch.tensor([0.5, 0.25, 0.1], device=gpu_device))
        for bias in (None, mask, dense.bfloat16(), dense, mask[:, :1, :1], dense[:1, :, :1].bfloat16(), alibi):
            got = torch.autograd.grad(flash_attention_fn(*ins, bias, causal), ins, do)
            full = alibi.materialize(M, N) if bias is alibi else bias
            ref = reference_grads(*[t.detach() for t in ins], None if full is None else full.expand(2, 3, M, N), do, causal)
            for name, a in zip(("dq", "dk", "dv"), got):
                assert (a.float() - ref[name]).norm() <= 5e-2 * ref[name].norm(), (name, M, N, D, causal, type(bias))


@pytest.mark.parametrize("D", [72, 80, 96])
def test_dk_dv_of_few_keys_at_head_dim_96(gpu_device, D):
    """Up to 64 keys the kernel of head dim 96 takes K and V in and gradients out by other ways than above: around that line,
    waves without a key among them, and strided gradients (the packed function)."""
    for M, N, causal in [(70, 5, False), (70, 31, False), (33, 33, True), (200, 64, False), (64, 64, True), (64, 65, False), (97, 97, True)]:
        g = torch.Generator().manual_seed(M + N + D)
        q, k, v, do = (torch.randn(2, s, 3, D, generator=g).bfloat16().to(gpu_device) for s in (M, N, N, M))
        mask = torch.ones(2, 1, 1, N, dtype=torch.bool, device=gpu_device)
        mask[1, ..., N // 2 + 1:] = False
        for bias in (None, mask, AlibiBias(torch.tensor([0.5, 0.25, 0.1], device=gpu_device))):
            ins = [t.detach().requires_grad_(True) for t in (q, k, v)]
            got = torch.autograd.grad(flash_attention_fn(*ins, bias, causal), ins, do)
            full = bias.materialize(M, N) if isinstance(bias, AlibiBias) else bias
            ref = reference_grads(q, k, v, None if full is None else full.expand(2, 3, M, N), do, causal)
            if M == N:
                qkv = torch.stack((q, k, v), 2).requires_grad_(True)
                packed, = torch.autograd.grad(flash_attention_qkvpacked_fn(qkv, bias, causal), qkv, do)
                for i in range(3):
                    assert torch.equal(packed[:, :, i], got[i]), (i, M, N, D, type(bias))
            for name, a in zip(("dk", "dv"), got[1:]):
                assert (a.float() - ref[name]).norm() <= 5e-2 * ref[name].norm(), (name, M, N, D, causal, type(bias))


def test_ragged_fp32_bias_written_to_before_the_backward(gpu_device):
    """A bias whose rows the kernels do not fetch in 16-byte chunks is copied where a backward may follow: the gradients are
    those of the bias that the forward saw, also of a tensor that autograd would not save."""
    g = torch.Generator().manual_seed(3)
    q, k, v, do = (torch.randn(2, 75, 2, 64, generator=g).bfloat16().to(gpu_device) for _ in range(4))
    bias = torch.randn(2, 2, 75, 75, generator=g).to(gpu_device)
    with torch.inference_mode():
        inference = bias.clone()
    ins = [t.requires_grad_(True) for t in (q, k, v)]
    want = torch.autograd.grad(flash_attention_fn(*ins, bias), ins, do)
    for b in (inference, bias):
        out = flash_attention_fn(*ins, b)
        assert "AttentionNode" in out.grad_fn.name()
        if b is bias:
            bias.zero_()
        for x, y in zip(torch.autograd.grad(out, ins, do), want):
            assert torch.equal(x, y)


def test_host_path_raises_what_the_launchers_raise(gpu_device):
    """A problem that the library refuses (2^28 keys, as views of one: nothing is allocated or launched) is a
    NativeLibraryError, in the forward and in the backward, which meets it through a hook; no memory is an OutOfMemoryError."""
    from triton_flashattn_amd import _native
    q, k, v = (torch.randn(1, n, 1, 64, device=gpu_device).bfloat16().requires_grad_(True) for n in (3, 1, 1))
    many = lambda t: t.detach().expand(1, 1 << 28, 1, 64) if t.shape == k.shape else t
    with torch.no_grad(), pytest.raises(_native.NativeLibraryError, match="bad shape"):
        flash_attention_fn(q, many(k), many(v))
    with pytest.raises(_native.NativeLibraryError, match="bad shape"):
        flash_attention_fn(q, many(k), many(v))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, many):
        out = flash_attention_fn(q, k, v)
    with pytest.raises(_native.NativeLibraryError, match="bad shape"):
        torch.autograd.grad(out, q, torch.ones_like(out))
    with torch.no_grad(), pytest.raises(torch.OutOfMemoryError):
        flash_attention_fn(q.expand(1 << 12, 3, 1 << 18, 64), k.expand(1 << 12, 1, 1 << 18, 64), v.expand(1 << 12, 1, 1 << 18, 64))


@pytest.mark.parametrize("kind", [None, "row", "bool", "dense", "alibi"])
def test_few_rows_against_many_keys(gpu_device, kind):
    """Few query tiles split their keys into up to 32 shares, short tiles into shares of 256 keys: both directions at
    the edges of that rule (no share, two, ragged last ones, 32, and rounding that leaves fewer than asked for), with
    whole shares behind the end of a sequence, masked by False or by a bias of -inf.  A dense bias takes the dQ
    kernel that reads dS, split as well."""
    g = torch.Generator().manual_seed(5)
    for B, M, N, H, D in [(1, 1, 511, 2, 64), (1, 1, 513, 2, 128), (2, 7, 1111, 1, 32), (1, 1, 8191, 1, 128), (1, 16, 8448, 2, 64),
                          (3, 130, 1700, 2, 128), (1, 256, 2049, 3, 16), (2, 257, 4096, 1, 64), (1, 5, 2304, 1, 256), (1, 64, 2560, 8, 128)]:
        mk = lambda n: torch.randn(B, n, H, D, generator=g).bfloat16().to(gpu_device)
        q, k, v, do = mk(M), mk(N), mk(N), mk(M)
        bias, dense, grad_of = None, None, []
        # (the last sequence ends inside the first share, and its last keys are whole masked shares)
        ends = torch.tensor([N - 3] * (B - 1) + [max(1, min(200, N // 2))])
        live = (torch.arange(N)[None] < ends[:, None])[:, None, None].to(gpu_device)
        if kind == "row":
            bias = dense = torch.zeros(B, 1, 1, N, device=gpu_device).masked_fill(~live, float("-inf"))
        elif kind == "bool":
            bias = dense = live
        elif kind == "dense":
            bias = torch.randn(B, H, M, N, generator=g).bfloat16().to(gpu_device).masked_fill(~live, float("-inf"))
            # ... and one sequence starts with masked keys
            bias[0, :, :, :min(300, N // 3) if B > 1 else 33] = float("-inf")
            bias = dense = bias.requires_grad_(True)
            grad_of = [bias]
        elif kind == "alibi":
            bias = AlibiBias(torch.linspace(0.01, 0.3, H).to(gpu_device))
            dense = bias.materialize(M, N)
        ins = [t.requires_grad_(True) for t in (q, k, v)]
        out = flash_attention_fn(q, k, v, bias, False)
        grads = torch.autograd.grad(out, ins + grad_of, do)
        q, k, v = (t.detach() for t in ins)
        full = None if dense is None else dense.detach().expand(B, H, M, N)
        o, lse = attention_forward(q, k, v, full, False)
        want = attention_backward(do, q, k, v, o, lse, full, False)[:3 + len(grad_of)]
        assert (out.float() - o).abs().max().item() <= 2e-2, (kind, B, M, N, H, D)
        for name, a, b in zip(("dq", "dk", "dv", "dbias"), grads, want):
            assert rel_l2(a, b) <= 5e-2, (name, kind, B, M, N, H, D, rel_l2(a, b))
