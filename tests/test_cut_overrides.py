"""Cut forward / input-grad contractions of at most 32 rows under the overrides that keep the square 128 tile (register
staging, the single-stage form): the plan must be one that this tile's kernel takes."""
import pytest
import torch

from helpers import SEED_CONSTANTS, assert_close, make_inputs, rargs

R1024 = SEED_CONSTANTS[1024]
OVERRIDES = [dict(clamp=-1), dict(stages=1), dict(clamp=-1, stages=1)]
# (M, K, N: 16-bit forward under any of them)
SHAPES = [(1, 2048, 512), (17, 4100, 4097), (17, 2049, 9001)]


@pytest.mark.parametrize("override", OVERRIDES, ids=str)
@pytest.mark.parametrize("split", [0, 3])
def test_a_tile_that_is_mostly_padding_is_left_to_the_second_kernel(override, split):
    """A batch of fewer rows than the tile never finishes its own cut (a 32 x 128 tile does, but it is staged
    directly only), however many slices the plan has; without overrides it does."""
    from rzlinear_amd import _lib
    cut = 0
    for code in (_lib.RZ_BF16, _lib.RZ_F16):
        for M in (1, 7, 31, 32):
            for K in (1000, 2048, 4100, 8192, 10240):
                for N in (512, 1031, 2048, 10240):
                    for op in (0, 1):
                        with _lib.tuning(split=split, **override):
                            q = _lib.plan_query(op, M, K, N, 1 << 20, 32, 64, code)
                        if q["mode"] == "split" and q["tile"] == 128:
                            cut += 1
                            assert q["step"] == 64 and q["shares"] == 0, (op, M, K, N, q)
    assert cut > 50
    assert _lib.plan_query(0, 1, 2048, 512, 1 << 20, 32, 64, _lib.RZ_BF16)["shares"] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("override", OVERRIDES, ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("split", [0, 3])
def test_cuts_under_the_overrides(oracle, shape, dtype, override, split):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_tl
    M, K, N = shape
    H, BK, BN = 20000, 32, 64
    print(shape, dtype, override, split, flush=True)
    (x, hw, _), (x64, hw64, _) = make_inputs(M, K, N, H, dtype, seed=M + K)
    with _lib.tuning(split=split, **override):
        y = rz_linear_forward_tl(x, hw, 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
        dx = rz_linear_backward_input_grad_tl(x, hw, 0.75, M, N, K, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, N, BK, BN, R1024, 0.75), dtype, "y")
    assert_close(dx.float().cpu().numpy(), oracle.input_grad(x64, hw64, N, BK, BN, R1024, 0.75), dtype, "dx")
