"""GPU tests of the dK / dV / dBias kernel of head dims up to 64 where its tiles end, against the fp32 oracle with the
tolerances of the parity tests."""
import pytest
import torch

from test_gpu_parity import check, make_inputs, run_oracle, run_ours

pytestmark = pytest.mark.gpu


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
