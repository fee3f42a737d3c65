"""GPU tests of paths inside the kernels that depend on the data or on how a shape meets the tiles, against
the fp32 oracle with the tolerances of the parity tests (out max-abs 2e-2, gradients relative L2 5e-2)."""
import pytest
import torch

from oracle.attention_oracle import attention_forward
from triton_flashattn_amd import flash_attention_fn

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
