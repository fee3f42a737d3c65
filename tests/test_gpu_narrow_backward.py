"""GPU tests of the dK / dV / dBias kernel of the smaller head dims where its tiles end, and of the kernels of head dim 96,
against the fp32 oracle with the tolerances of the parity tests."""
import pytest
import torch

from oracle.attention_oracle import attention_backward, attention_forward
from test_gpu_parity import check, make_inputs, rel_l2, run_oracle, run_ours
from test_gpu_parity_edges import _launch_directly
from triton_flashattn_amd import AlibiBias, _native, flash_attention_fn

pytestmark = pytest.mark.gpu

# Largest error of a gradient that is summed inside the kernels over the sum of its terms' magnitudes, against 64 bits and
# with the kernel's own output in delta, so that nothing but fp32 sums and exponentials is left: 2.0e-7 over head dims 32 to
# 128 and 33 to 1100 rows; four times that.
SUM_RTOL = 8e-7


def dscores(q, k, v, do, out, dense, causal):
    """dS (B, H, M, N) of the output that the kernels returned, in 64 bits."""
    q, k, v, out = (t.detach() for t in (q, k, v, out))
    _, lse = attention_forward(q, k, v, dense, causal, dtype=torch.float64)
    return attention_backward(do, q, k, v, out, lse, dense, causal, dtype=torch.float64)[3]


def add_trend(v, do, causal):
    """Adds to the first column of v a slope over the keys and to that of do its counterpart over the rows, so that the terms
    of a slope's gradient do not cancel between rows or tiles: a tile that is lost shows."""
    M, N = do.shape[1], v.shape[1]
    i, j = (torch.arange(n, device=v.device)[None, :, None] / n for n in (M, N))
    v[..., 0] += 6.0 * j
    do[..., 0] += 6.0 if causal else 6.0 - 12.0 * i


def check_slope_gradient(got, ds, causal, tag):
    """The gradient of ALiBi slopes, the sum of -|i N / M - j| dS per head; no 32 keys of a wave may be lost in it."""
    M, N = ds.shape[2:]
    i, j = torch.arange(M, device=ds.device)[:, None], torch.arange(N, device=ds.device)[None, :]
    terms = ds * -(i * (N / M) - j).abs()
    # (a row's delta, common to its terms, may be off by 2^-22 of |dO| |O|, ten times the terms' own dP - delta: 3e-6 of one row)
    limit = SUM_RTOL * (1 + 4 / M) * terms.abs().sum((0, 2, 3))
    for first in range(0, N, 32):
        # (causal: the last key alone is seen by the last row alone, at distance 0)
        if not (causal and first == N - 1):
            assert (terms[..., first:first + 32].sum((0, 2, 3)).abs() > limit).all(), ("a loss of 32 keys would not show", tag, first)
    assert ((got - terms.sum((0, 2, 3))).abs() <= limit).all(), (tag, got, terms.sum((0, 2, 3)))


def check_row_gradient(got, ds, rounding, tag):
    """The gradient of a (1, H, 1, N) bias, the sum of dS over batches and rows, key by key: rounded to the bias's type and off
    by the limit of the sum and the rounding of its terms (H, N)."""
    want, size = ds.sum((0, 2)), ds.abs().sum((0, 2))
    info = torch.finfo(got.dtype)  # (below its least normal number a type's steps do not shrink: 2^-24 in fp16)
    limit = info.eps / 2 * want.abs().clamp_min(info.tiny) + SUM_RTOL * size + rounding
    for first in range(0, ds.shape[3], 32):
        if ds.shape[3] > 1:
            part = slice(first, first + 32)
            assert (want[:, part].abs() > 2 * limit[:, part]).any(), ("a loss of 32 keys would not show", tag, first)
    error = (got[0, :, 0].double() - want).abs()
    assert (error <= limit).all(), (tag, (error / limit).max().item())


def check_summed_gradient(kind, q, k, v, do, leaf, causal, tag):
    """The gradient of ALiBi slopes (kind "alibi") or of a (1, H, 1, N) bias on inputs whose terms do not cancel."""
    M, N, H = q.shape[1], k.shape[1], q.shape[2]
    v, do = v.detach().float(), do.float()
    add_trend(v, do, causal)
    v, do = v.to(q.dtype), do.to(q.dtype)
    if kind == "alibi":  # slopes that leave the farthest keys some weight; causal, that leave some to the last keys, which few rows see
        leaf = (torch.linspace(0.05, 0.2, H) if causal else torch.linspace(2.0, 6.0, H) / N).to(q.device).requires_grad_(True)
    bias = AlibiBias(leaf) if kind == "alibi" else leaf
    dense = bias.materialize(M, N) if kind == "alibi" else bias.expand(-1, -1, M, -1)
    out = flash_attention_fn(q.detach(), k.detach(), v, bias, causal)
    got, = torch.autograd.grad(out, leaf, do)
    dense = dense.detach().expand(q.shape[0], H, M, N)
    ds = dscores(q, k, v, do, out, dense, causal)
    if kind == "alibi":
        check_slope_gradient(got, ds, causal, tag)
    else:
        # dP and delta: 2^-22 of the sum of |dO| |V| at most, times P, whose sums over the rows are dV of a dO of ones
        _, lse = attention_forward(q.detach(), k.detach(), v, dense, causal, dtype=torch.float64)
        weight = attention_backward(torch.ones_like(do), q.detach(), k.detach(), v, out, lse, dense, causal, dtype=torch.float64)[2][..., 0]
        size = (do.abs().amax(1, keepdim=True).double() * v.abs().double()).sum(3)
        check_row_gradient(got, ds, 2.0 ** -22 * (weight * size).sum(0).T, tag)


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("kind", [None, "bool", "bf16", "f16", "f32"])
def test_edges_of_steps_waves_and_tiles(gpu_device, D, kind):
    """Row counts around its 32-row blocks, its steps of two and the first of its steady-state steps; key counts around the
    32 keys of a wave (waves without keys among them) and the 128 of a work-group; a bias of q's type, of the other 16-bit
    type and in fp32, with and without a gradient."""
    for i, (M, N, causal) in enumerate([(1, 1, False), (31, 33, False), (33, 96, False), (64, 128, False), (65, 129, False),
                                        (127, 100, False), (193, 161, False), (321, 264, False), (1, 1, True), (33, 33, True),
                                        (64, 64, True), (97, 97, True), (128, 128, True), (200, 200, True), (391, 391, True)]):
        q, k, v, do, bias = make_inputs(gpu_device, 1, M, N, 3, D, torch.bfloat16, kind, seed=10 * i + D, trainable=i % 3 != 2)
        check(run_ours(q, k, v, do, bias, causal), run_oracle(q, k, v, do, bias, causal), str((D, kind, M, N, causal)))


@pytest.mark.parametrize("d_qk,d_v", [(96, 96), (72, 88), (96, 64), (8, 96)])
@pytest.mark.parametrize("kind", [None, "alibi", "row", "boolrow", "dense", "f16", "f32"])
def test_head_dims_up_to_96(gpu_device, d_qk, d_v, kind):
    """Head dims between 64 and 96 run at 96, in bf16 and fp16 in turn: rows of 192 bytes in LDS, the edges of steps and tiles, keys
    split between work-groups in both directions, rows of a bias that are too long for LDS (causal: their keys are not split),
    bias tiles of q's type ("dense"), in fp16 and in fp32, and neighbouring columns that hold NaN."""
    g = torch.Generator().manual_seed(d_qk + d_v)
    shapes = [(1, 1, 1, False), (1, 33, 65, False), (2, 64, 128, False), (1, 129, 193, False), (1, 40, 2200, False),
              (1, 257, 257, True), (2, 128, 128, True), (1, 391, 391, True)]
    if kind in ("row", "boolrow"):
        shapes += [(1, 4200, 4200, True), (1, 4133, 4133, True)]
    for i, (B, M, N, causal) in enumerate(shapes):
        if kind == "alibi" and N == 1:
            continue
        H = 2
        dtype = torch.float16 if i % 2 else torch.bfloat16
        wide = lambda n, d: torch.cat([torch.randn(B, n, H, d, generator=g), torch.full((B, n, H, 8), float("nan"))], -1).to(dtype).to(gpu_device)[..., :d]
        q, k, v, do = (t.requires_grad_(i < 3) for i, t in enumerate((wide(M, d_qk), wide(N, d_qk), wide(N, d_v), wide(M, d_v))))
        bias, dense, grad_of = None, None, None
        if kind == "alibi":
            grad_of = torch.tensor([0.02, 0.3], device=gpu_device).requires_grad_(True)
            bias = AlibiBias(grad_of)
            dense = bias.materialize(M, N).detach()
        elif kind in ("row", "dense", "f16", "f32"):
            bdt = {"f16": torch.float16, "f32": torch.float32}.get(kind, dtype)
            bias = grad_of = torch.randn(1, H, 1 if kind == "row" else M, N, generator=g).expand(1 if kind == "row" else B, -1, -1, -1)
            bias = grad_of = bias.to(bdt).contiguous().to(gpu_device).requires_grad_(True)
            dense = bias.detach()
        elif kind == "boolrow":
            bias = dense = (torch.rand(B, 1, 1, N, generator=g) > 0.3).index_fill(3, torch.tensor([0]), True).to(gpu_device)
        out = flash_attention_fn(q, k, v, bias, causal)
        grads = torch.autograd.grad(out, [q, k, v] + ([] if grad_of is None else [grad_of]), do)
        full = None if dense is None else dense.expand(B, H, M, N)
        o, lse = attention_forward(q.detach(), k.detach(), v.detach(), full, causal)
        dq, dk, dv, db, _ = attention_backward(do, q.detach(), k.detach(), v.detach(), o, lse, full, causal)
        assert (out.float() - o).abs().max().item() <= 2e-2, (M, N, causal)
        for name, a, b in zip("qkv", grads, (dq, dk, dv)):
            assert rel_l2(a, b) <= 5e-2, (name, M, N, causal)
        if kind in ("dense", "f16", "f32"):
            assert rel_l2(grads[3], db) <= 5e-2, (M, N)
        elif kind in ("row", "alibi"):
            check_summed_gradient(kind, q, k, v, do, grad_of, causal, (M, N, causal))


class AtHeadDim:
    """The library, whose launchers take the tensors' first d columns for all there are."""

    def __init__(self, lib, d):
        self.lib, self.d = lib, d

    def __getattr__(self, name):
        return getattr(self.lib, name)

    def fa_fwd(self, args, stream):
        return self.lib.fa_fwd_dims(args, self.d, self.d, stream)

    def fa_bwd_stages(self, args, stream, stages):
        return self.lib.fa_bwd_stages_dims(args, self.d, self.d, stream, stages)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["bool", "bf16", "f16", "f32"])
def test_bias_tiles_that_are_only_read_at_head_dim_96(gpu_device, monkeypatch, dtype, kind):
    """Straight to the kernels, rows of the bias that allow aligned 16-byte accesses and (elsewhere the public functions pad
    them) rows that do not; the columns behind the head dim hold NaN."""
    lib = _native.load()
    for i, (B, M, N, d, causal) in enumerate([(2, 129, 192, 96, False), (1, 33, 65, 72, False), (1, 200, 333, 88, False), (1, 391, 391, 96, True)]):
        q, k, v, do, bias = make_inputs(gpu_device, B, M, N, 2, 128, dtype, kind, seed=i, trainable=False)
        ref = run_oracle(*(t[..., :d] for t in (q, k, v, do)), bias, causal, 128 ** -0.5)
        for t in (q, k, v, do):
            t[..., d:] = float("nan")
        monkeypatch.setattr(_native, "load", lambda: AtHeadDim(lib, d))
        res = _launch_directly(q, k, v, do, bias, None, causal)
        check({n: None if t is None else t[..., :d] for n, t in res.items()}, dict(ref, dbias=None), str((M, N, d)))


@pytest.mark.parametrize("kind", [None, "bool", "bf16", "f32", "alibi", "row"])
def test_tiles_of_64_keys_at_head_dim_128(gpu_device, kind):
    """Few query rows at head dim 128 take 64-key tiles: around the line (512 rows, 1024 with a causal mask), key counts
    around a tile and a wave, and the slope and row gradients that are summed per tile."""
    g = torch.Generator().manual_seed(7)
    H = 2
    for M, N, causal in [(1, 63, False), (33, 64, False), (100, 65, False), (512, 97, False), (513, 130, False), (96, 333, False),
                         (64, 64, True), (161, 161, True), (1000, 1000, True), (1025, 1025, True)]:
        q, k, v, do, bias = make_inputs(gpu_device, 1, M, N, H, 128, torch.bfloat16, kind if kind in ("bool", "bf16", "f32") else None,
                                        seed=M, trainable=False)
        if kind in (None, "bool", "bf16", "f32"):
            check(run_ours(q, k, v, do, bias, causal), run_oracle(q, k, v, do, bias, causal), str((kind, M, N, causal)))
            continue
        if kind == "alibi":
            grad_of = torch.tensor([0.02, 0.3], device=gpu_device).requires_grad_(True)
            bias = AlibiBias(grad_of)
            dense = bias.materialize(M, N).detach()
        else:
            bias = grad_of = torch.randn(1, H, 1, N, generator=g).bfloat16().to(gpu_device).requires_grad_(True)
            dense = bias.detach()
        ins = [t.requires_grad_(True) for t in (q, k, v)]
        grads = torch.autograd.grad(flash_attention_fn(*ins, bias, causal), ins + [grad_of], do)
        ref = run_oracle(q.detach(), k.detach(), v.detach(), do, dense.expand(1, H, M, N), causal)
        for name, a in zip(("dq", "dk", "dv"), grads):
            assert rel_l2(a, ref[name]) <= 5e-2, (name, M, N, causal)
        check_summed_gradient(kind, q, k, v, do, grad_of, causal, (M, N, causal))


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("kind", ["bool", "bf16", "f32"])
def test_biases_that_a_pair_of_waves_takes(gpu_device, D, kind):
    """Up to head dim 64 biases of at least 512 (masks 1500, head dim 16 1025) rows go to the kernel of two waves per 32 keys, an fp32 one with a
    gradient also in whole rounds of as many tiles as there are CUs and, causal, with fewer rows: around the lines, with ragged rows and keys,
    rows of the bias that are whole chunks and rows that are not."""
    for M, N, H, causal in [(511, 130, 2, False), (512, 97, 2, False), (513, 264, 2, False), (640, 33, 1, False),
                            (545, 136, 140, False), (1281, 130, 256, False), (1280, 33, 300, False), (2049, 65, 400, False), (1499, 70, 2, False), (1500, 264, 2, False), (1525, 130, 1, False),
                            (1025, 264, 20, False), (1, 1, 2, True), (33, 33, 2, True), (200, 200, 2, True), (512, 512, 2, True), (577, 577, 2, True), (650, 650, 1, True), (1500, 1500, 16, True)]:
        for trainable in (True, False):
            q, k, v, do, bias = make_inputs(gpu_device, 1, M, N, H, D, torch.bfloat16, kind, seed=M + D, trainable=trainable)
            check(run_ours(q, k, v, do, bias, causal), run_oracle(q, k, v, do, bias, causal), str((D, kind, M, N, H, causal, trainable)))


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("kind", ["bf16", "f16", "f32"])
def test_bias_and_gradient_rows_that_allow_no_aligned_accesses(gpu_device, D, kind):
    """Straight to the kernels, rows of an odd number of keys, dense (fp32: read 4 bytes to a lane; else, and the gradient,
    element by element), with a padded pitch (16 bytes at a time) and, the bias, every second column of a wider tensor
    (element by element), the gradient dense, with a padded pitch, or none."""
    for i, (M, N, causal) in enumerate([(70, 197, False), (131, 131, True), (33, 5, False), (300, 129, False)]):
        q, k, v, do, bias = make_inputs(gpu_device, 2, M, N, 2, D, torch.bfloat16, kind, seed=D + i, trainable=False)
        ref = run_oracle(q, k, v, do, bias, causal)
        wide = torch.full((2, 2, M, -(-N // 8) * 8), float("nan"), dtype=bias.dtype, device=gpu_device)
        wide[..., :N] = bias
        apart = torch.full((2, 2, M, 2 * N), float("nan"), dtype=bias.dtype, device=gpu_device)
        apart[..., ::2] = bias
        for b in (bias, wide[..., :N], apart[..., ::2]):
            for out in (torch.empty_like(bias), torch.empty_like(wide)[..., :N], None):
                res = _launch_directly(q, k, v, do, b, out, causal)
                check(res, ref, str((D, kind, M, N, causal, b.stride(), None if out is None else out.stride())))


def test_tiles_of_64_or_128_keys_with_an_fp32_bias(gpu_device):
    """An fp32 bias that is only read at head dim 128, in few and in many tiles, around the lines between 64 and 128 keys."""
    for M, N, H, causal in [(320, 65, 520, False), (321, 65, 520, False), (513, 65, 2, False), (512, 130, 260, False),
                            (321, 321, 350, True), (320, 320, 350, True), (1000, 1000, 2, True)]:
        q, k, v, do, bias = make_inputs(gpu_device, 1, M, N, H, 128, torch.bfloat16, "f32", seed=M, trainable=False)
        check(run_ours(q, k, v, do, bias, causal), run_oracle(q, k, v, do, bias, causal), str((M, N, H, causal)))


def test_alibi_of_long_tiles_at_head_dim_96(gpu_device):
    """dK, dV and the slope gradient of ALiBi at head dims up to 96 around the line between the kernels of 96 and 128: 1024
    rows, and more tiles than there are CUs."""
    for M, N, H, causal, d in [(1024, 130, 1, False, 96), (1025, 130, 2, False, 72), (1100, 1100, 1, True, 96), (1030, 130, 130, False, 88)]:
        g = torch.Generator().manual_seed(M)
        q, k, v, do = (torch.randn(1, n, H, d, generator=g) for n in (M, N, N, M))
        add_trend(v, do, causal)
        q, k, v, do = (t.bfloat16().to(gpu_device) for t in (q, k, v, do))
        slopes = torch.linspace(0.01, 0.002, H, device=gpu_device).requires_grad_(True)
        dense = AlibiBias(slopes).materialize(M, N).detach()
        ins = [t.requires_grad_(True) for t in (q, k, v)]
        out = flash_attention_fn(*ins, AlibiBias(slopes), causal)
        grads = torch.autograd.grad(out, ins + [slopes], do)
        ref = run_oracle(q.detach(), k.detach(), v.detach(), do, dense, causal)
        for name, a in zip(("dq", "dk", "dv"), grads):
            assert rel_l2(a, ref[name]) <= 5e-2, (name, M, N, causal)
        check_slope_gradient(grads[3], dscores(q, k, v, do, out, dense, causal), causal, (M, N))
