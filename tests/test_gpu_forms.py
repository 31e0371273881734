"""The forms of the kernels that a rule on sizes picks, at the edges of their ranges, against the oracle."""
import sys

import numpy as np
import pytest
import torch

from helpers import SEED_CONSTANTS, assert_close, make_inputs, rargs

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]
SIXTEEN = [torch.bfloat16, torch.float16]


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _both_ops(oracle, shape, dtype, **tuning):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_bias_tl
    M, K, N, H, BK, BN = shape
    _say(shape, dtype, tuning)
    (x, hw, dy), (x64, hw64, dy64) = make_inputs(M, K, N, H, dtype, seed=M + K)
    bias = torch.randn((N,), generator=torch.Generator().manual_seed(4)).to(dtype)
    with _lib.tuning(**tuning):
        y = rz_linear_forward_bias_tl(x, hw, bias.cuda(), 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
        dx = rz_linear_backward_input_grad_tl(dy, hw, 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, N, BK, BN, R1024, 0.75) + bias.double().numpy(), dtype, "y")
    assert_close(dx.float().cpu().numpy(), oracle.input_grad(dy64, hw64, K, BK, BN, R1024, 0.75), dtype, "dx")


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("split", [-1, 2, 4, 5])   # whole; finished in the kernel; by a second kernel
@pytest.mark.parametrize("shape", [
    (32, 640, 1280, 20000, 32, 64),      # complete tiles and steps
    (1, 640, 1280, 20000, 64, 64),       # one row
    (31, 700, 1100, 20000, 32, 64),      # last step and last column tile partial, rows of whole pieces (K) and not (N)
    (17, 641, 1023, 20000, 16, 128),     # nothing a multiple of anything
    (32, 128, 128, 20000, 64, 32),       # fewer steps than stages
    (5, 9, 900, 20000, 32, 64),          # a row of little more than one piece
], ids=lambda s: "x".join(map(str, s)))
def test_at_most_32_rows(oracle, shape, dtype, split):
    _both_ops(oracle, shape, dtype, tile=128, split=split)


@pytest.mark.parametrize("dtype", [torch.float32] + SIXTEEN, ids=str)
@pytest.mark.parametrize("shape", [
    (20, 64, 64, 70001, 64, 64),          # one tile, H one beyond a multiple of the span
    (20, 1024, 1024, 65536, 32, 32),      # 1024 tiles: half a round of looks
    (20, 1040, 2048, 99999, 32, 32),      # 2112 tiles: a second round; partial tiles
    (20, 2048, 2048, 262144, 32, 32),     # 4096 tiles, the most
    (20, 999, 1001, 65537, 16, 64),       # partial tiles in both directions, last span of one element
    (20, 1024, 1024, 45000, 64, 64),      # every list longer than one batch of loads
], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("accumulate", [False, True])
def test_fold_of_few_tiles(oracle, shape, dtype, accumulate):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H, BK, BN = shape
    _say(shape, dtype, accumulate)
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, dtype, seed=K)
    before = torch.randn((H,), generator=torch.Generator().manual_seed(2))
    out = before.cuda()
    R = _lib.hash_constants(*rargs(R1024))
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5) + (before.double().numpy() if accumulate else 0.0)
    # (fp32 tiles and sums whatever the layer's type: M products and at most a few hundred tiles per element)
    for plans in (False, True):
        out.copy_(before)
        with _lib.tuning(fold=1, lds_image=-1, window=-1):
            assert _lib.plan_query(2, M, K, N, H, BK, BN, _lib.dtype_code(x), _lib.WG_DHW_F32)["mode"] == "fold"
            _, dbias = weight_grad_hashed(x, dy, 0.5, M, K, N, H, R, BK, BN, out=out, accumulate=accumulate,
                                          with_bias_grad=True, use_layer_plan=plans)
        assert np.abs(out.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()
        assert_close(dbias.float().cpu().numpy(), dy64.sum(0), dtype, "bias gradient")
