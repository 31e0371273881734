"""The baseline configurations at their full sizes, on the GPU.

The CPU oracle would take minutes there, so the check is assembled from pieces that are pinned
elsewhere: the index map comes from the materialiser (bit-exact against the oracle in
test_gpu_parity.py, and checked against the oracle again here at full size), the dense products
are float64 torch.matmul on the GPU, and the reduction into hashed_weight is torch's index_add_
— the reference tests' own design (python/tests/test_rz_linear.py:21-33,:77-90)."""
import sys

import numpy as np
import pytest
import torch

from helpers import SEED_CONSTANTS, TOL, ULP, rargs, ROUNDING, stored_tile_bytes

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]

# name -> (M, K, N, H, dtype, input distributions[, (BK, BN)]); 64 x 64 tiles, as benchmarked, unless
# given: the reference's own benchmark grid (python/bench/bench.py:10-11 in the reference: K = N = 10240,
# compress_ratio 0.0625, M = 32, 128, 1024) runs on its launchers' default 32 x 64 tile.  "normal":
# X ~ N(0,1), dY ~ N(0,1); "relu": X = relu(N(0,1)), dY ~ N(0, variance 1e-2), the
# recommendation-MLP-like configuration.  hashed_weight ~ U(-1/sqrt(K), 1/sqrt(K)) throughout.
CONFIGS = {
    "square1024_bf16": (1024, 1024, 1024, 16384, torch.bfloat16, "normal"),
    "square1024_fp32": (1024, 1024, 1024, 16384, torch.float32, "normal"),
    "square2048_bf16": (2048, 2048, 2048, 16384, torch.bfloat16, "normal"),
    "square2048_fp32": (2048, 2048, 2048, 16384, torch.float32, "normal"),
    "square4096_bf16": (4096, 4096, 4096, 16778, torch.bfloat16, "normal"),
    "square4096_fp32": (4096, 4096, 4096, 16778, torch.float32, "normal"),
    "rec_mlp_bf16": (16384, 512, 1024, 5243, torch.bfloat16, "relu"),
    "ffn_bf16": (8192, 4096, 16384, 67109, torch.bfloat16, "normal"),
    "collision_fp32": (32768, 2048, 2048, 32768, torch.float32, "normal"),
    "grid_32_10240_fp32": (32, 10240, 10240, 6553600, torch.float32, "normal", (32, 64)),
    "grid_128_10240_bf16": (128, 10240, 10240, 6553600, torch.bfloat16, "normal", (32, 64)),
    "grid_1024_10240_bf16": (1024, 10240, 10240, 6553600, torch.bfloat16, "normal", (32, 64)),
    "grid_1024_10240_fp32": (1024, 10240, 10240, 6553600, torch.float32, "normal", (32, 64)),
}
_index_maps = {}   # (K, N, H, BK, BN) -> index map on the device (the grid's is 105 M entries: computed once)


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _rel(out, ref):
    ref = ref.double()
    return float((out.double() - ref).abs().max() / ref.abs().max())


def _check(out, ref, dtype, what, slack=None):
    """The stated normalised tolerance and the element-wise rounding bound of helpers.assert_close
    (with its allowance `slack` per element, if any), evaluated on the GPU (the tensors are large)."""
    ref = ref.double()
    err = (out.double() - ref).abs()
    scale = float(ref.abs().max())
    assert torch.isfinite(out).all(), what
    assert float(err.max()) / scale <= TOL[dtype], "%s: normalised max error %.3g" % (what, float(err.max()) / scale)
    excess = err / (ULP[dtype] * ref.abs() + 1e-5 * scale + (0.0 if slack is None else slack))
    worst = float(excess.max())
    assert worst <= 1.0, "%s: %.2f x the element-wise bound at flat index %d (%d elements beyond it)" % (
        what, worst, int(excess.argmax()), int((excess > 1.0).sum()))


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_baseline_configuration_at_full_size(oracle, name):
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_tl
    from rzlinear_amd.impl.RzLinearIdx import rz_linear_weight_tl
    M, K, N, H, dtype, dist = CONFIGS[name][:6]
    BK, BN = CONFIGS[name][6] if len(CONFIGS[name]) > 6 else (64, 64)
    _say("full size", name)
    g = torch.Generator().manual_seed(77)
    x = torch.randn((M, K), generator=g)
    hw = ((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype).cuda()
    dy = torch.randn((M, N), generator=g)
    if dist == "relu":
        x, dy = torch.relu(x), dy * 0.1
    x, dy = x.to(dtype).cuda(), dy.to(dtype).cuda()
    kw = dict(BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)

    # index map: materialise arange(H) in fp32 (exact), compare with the oracle's map
    if (K, N, H, BK, BN) not in _index_maps:
        _index_maps.clear()
        idx = rz_linear_weight_tl(torch.arange(H, dtype=torch.float32, device="cuda"), K, N, H, *rargs(R1024), **kw).long()
        assert np.array_equal(idx.cpu().numpy(), oracle.index_map(K, N, H, BK, BN, R1024))
        _index_maps[(K, N, H, BK, BN)] = idx
    idx = _index_maps[(K, N, H, BK, BN)]
    W = hw.double()[idx]

    y = rz_linear_forward_tl(x, hw, 1.0, M, K, N, H, *rargs(R1024), **kw)
    dx, dhw = rz_linear_backward_tl(x, hw, dy, 1.0, M, K, N, H, *rargs(R1024), **kw)
    torch.cuda.synchronize()
    _check(y, x.double() @ W, dtype, "Y")
    _check(dx, dy.double() @ W.t(), dtype, "dX")
    dW = x.double().t() @ dy.double()
    ref = torch.zeros((H,), dtype=torch.float64, device="cuda").index_add_(0, idx.reshape(-1), dW.reshape(-1))
    # (a 16-bit layer whose weight gradient goes through the fold keeps the tiles of X^T.dY in its own dtype:
    #  every stored value, one per element of X^T.dY and slice of M, is rounded once before the slots are
    #  added up in fp32 — see helpers.stored_tiles_slack)
    slack = None
    if dtype != torch.float32:
        from rzlinear_amd import _lib
        code = _lib.RZ_BF16 if dtype == torch.bfloat16 else _lib.RZ_F16
        folds = [_lib.plan_query(2, M, K, N, H, BK, BN, code, planned=p) for p in (False, True)
                 if stored_tile_bytes((M, K, N, H, BK, BN), code, p) == 2]
        for q in folds:
            step = q["slice_len"] if q["slices"] > 1 else M
            stored = sum((x[m:m + step].double().t() @ dy[m:m + step].double()).abs() for m in range(0, M, step))
            s = torch.zeros((H,), dtype=torch.float64, device="cuda").index_add_(0, idx.reshape(-1), stored.reshape(-1))
            slack = s if slack is None else torch.maximum(slack, s)
            del stored
        if slack is not None:
            slack = ROUNDING[dtype] * slack
    _check(dhw, ref, dtype, "dHW", slack)
    # mass conservation, a check that does not go through the index map: every element of
    # X^T.dY lands in exactly one slot
    assert abs(float(dhw.double().sum() - dW.sum())) <= TOL[dtype] * float(dW.abs().sum()) / 10


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=lambda d: str(d).split(".")[-1])
def test_row_pitches_that_break_16_byte_alignment(oracle, dtype):
    """Complete tiles (the kernels without bounds checks, direct-to-LDS staging for bf16) on
    operands whose rows start at odd element offsets."""
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_tl
    M, K, N, H, BK, BN = 512, 512, 768, 9000, 64, 64
    _say("odd row pitch", dtype)
    g = torch.Generator().manual_seed(78)
    xbig = torch.randn((M, K + 3), generator=g).to(dtype).cuda()
    dybig = torch.randn((M, N + 5), generator=g).to(dtype).cuda()
    x, dy = xbig[:, 1:K + 1], dybig[:, 3:N + 3]
    assert x.stride(0) == K + 3 and x.data_ptr() % 16 != 0
    hw = ((torch.rand((H + 1,), generator=g) * 2 - 1) / K ** 0.5).to(dtype).cuda()[1:]   # odd start as well
    kw = dict(BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    y = rz_linear_forward_tl(x, hw, 1.0, M, K, N, H, *rargs(R1024), **kw)
    dx, dhw = rz_linear_backward_tl(x, hw, dy, 1.0, M, K, N, H, *rargs(R1024), **kw)
    torch.cuda.synchronize()
    x64, hw64, dy64 = (t.double().cpu().numpy() for t in (x, hw, dy))
    f = lambda t: t.float().cpu().numpy()
    from helpers import rel_err
    assert rel_err(f(y), oracle.forward(x64, hw64, N, BK, BN, R1024)) <= TOL[dtype]
    assert rel_err(f(dx), oracle.input_grad(dy64, hw64, K, BK, BN, R1024)) <= TOL[dtype]
    assert rel_err(f(dhw), oracle.weight_grad(x64, dy64, H, BK, BN, R1024)) <= TOL[dtype]
