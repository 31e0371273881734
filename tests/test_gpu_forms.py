"""The forms of the kernels that a rule on sizes picks, at the edges of their ranges, against the oracle."""
import sys

import numpy as np
import pytest
import torch

from helpers import SEED_CONSTANTS, assert_close, make_inputs, rargs, rounded_tiles_slack, stored_tile_bytes

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]
SIXTEEN = [torch.bfloat16, torch.float16]


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _forward_and_mirrored_input_grad(oracle, shape, dtype, split, tile, slices, finished):
    """The forward of (M, K, N) and the input-grad of (M, N, K), which the planner prices alike, under the plan that
    is expected; finished in the kernel or, where the plan stays the same, by a second one: the same bits."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_bias_tl
    M, K, N, H, BK, BN = shape
    _say(shape, dtype, split)
    (x, hw, _), (x64, hw64, _) = make_inputs(M, K, N, H, dtype, seed=M + K)
    bias = torch.randn((N,), generator=torch.Generator().manual_seed(4)).to(dtype)
    out = []
    for finish in (0, -1):
        with _lib.tuning(split=split, finish=finish):
            for q in (_lib.plan_query(0, M, K, N, H, BK, BN, _lib.dtype_code(x)), _lib.plan_query(1, M, N, K, H, BK, BN, _lib.dtype_code(x))):
                if finish == 0:
                    assert (q["tile"], q["slices"], q["shares"]) == (tile, slices, finished)
                same_plan = (q["tile"], q["slices"]) == (tile, slices)
            if not same_plan:   # (priced without the finish, another tile may be the better one)
                continue
            y = rz_linear_forward_bias_tl(x, hw, bias.cuda(), 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
            dx = rz_linear_backward_input_grad_tl(x, hw, 0.75, M, N, K, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
            out.append((y, dx))
    y, dx = out[0]
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, N, BK, BN, R1024, 0.75) + bias.double().numpy(), dtype, "y")
    assert_close(dx.float().cpu().numpy(), oracle.input_grad(x64, hw64, N, BK, BN, R1024, 0.75), dtype, "dx")
    for a, b in zip(out[0], out[-1]):
        np.testing.assert_array_equal(a.float().cpu().numpy(), b.float().cpu().numpy())


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("shape,split,slices,finished", [
    ((32, 2048, 2048, 20000, 32, 64), 0, 8, 1),      # complete tiles and steps, as many slices as the kernel finishes
    ((32, 2048, 2048, 20000, 64, 64), 3, 3, 1),      # an incomplete last slice
    ((1, 2048, 2048, 20000, 64, 64), 4, 4, 1),       # one row
    ((31, 4111, 4099, 20000, 32, 64), 5, 5, 1),      # odd row pitch, last step and last column tile partial
    ((17, 4100, 4097, 20000, 16, 128), 6, 6, 1),     # ... in other hashed tiles
    ((7, 2049, 2040, 20000, 128, 32), 0, 6, 1),
], ids=str)
def test_16_bit_at_most_32_rows(oracle, shape, split, slices, finished, dtype):
    _forward_and_mirrored_input_grad(oracle, shape, dtype, split, 128, slices, finished)


@pytest.mark.parametrize("dtype,shape,slices", [
    (torch.bfloat16, (32, 2048, 2048, 20000, 32, 64), 8),
    (torch.float16, (1, 2048, 512, 20000, 32, 64), 8),
    (torch.bfloat16, (7, 2049, 2040, 20000, 128, 32), 6),
    (torch.float32, (32, 1024, 1024, 20000, 32, 64), 6),
], ids=str)
def test_a_captured_cut_takes_the_second_kernel_with_the_same_bits(dtype, shape, slices):
    """A stream under capture gets no counters: the same plan, its planes added by the second kernel.  (The `finish`
    override, which does that too, may change the plan.)"""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearForward import forward_hashed
    M, K, N, H, BK, BN = shape
    _say("captured", shape, dtype)
    (x, hw, _), _ = make_inputs(M, K, N, H, dtype, seed=M + K)
    bias = torch.randn((N,), generator=torch.Generator().manual_seed(4)).to(dtype).cuda()
    q = _lib.plan_query(0, M, K, N, H, BK, BN, _lib.dtype_code(x))
    assert (q["slices"], q["shares"]) == (slices, 1)

    def forward():
        return forward_hashed(x, hw, bias, 0.75, M, K, N, H, _lib.hash_constants(*rargs(R1024)), BK, BN, 2)

    forward()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = forward()
    for replay in range(3):
        x.copy_(torch.randn((M, K), generator=torch.Generator().manual_seed(replay)).to(dtype))
        finished = forward()
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, finished), replay


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
def test_16_bit_at_most_32_rows_uncut(oracle, dtype):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_tl
    M, K, N, H, BK, BN = 5, 9, 9000, 20000, 32, 64   # (rows of little more than one 16-byte piece)
    (x, hw, _), (x64, hw64, _) = make_inputs(M, K, N, H, dtype, seed=1)
    assert _lib.plan_query(0, M, K, N, H, BK, BN, _lib.dtype_code(x))["tile"] == 128
    y = rz_linear_forward_tl(x, hw, 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, N, BK, BN, R1024, 0.75), dtype, "y")


@pytest.mark.parametrize("shape,split,slices,finished", [
    ((32, 1024, 1024, 20000, 32, 64), 0, 6, 1),
    ((32, 1024, 1024, 20000, 32, 64), 8, 8, 1),
    ((32, 2048, 1024, 20000, 64, 64), 16, 16, 0),
], ids=str)
def test_fp32_32_rows(oracle, shape, split, slices, finished):
    _forward_and_mirrored_input_grad(oracle, shape, torch.float32, split, 32, slices, finished)


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


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("shape", [
    (64, 1024, 1024, 20000, 32, 64),      # 16 tiles, four stages, complete
    (70, 650, 1100, 20000, 64, 64),       # partial tiles and last step
    (65, 129, 131, 20000, 16, 128),       # one step and a bit, odd row pitches
    (50, 40, 72, 20000, 32, 64),          # less than one step
    (1030, 300, 1040, 20000, 32, 64),     # more tiles than compute units: two stages
    (1025, 257, 1099, 20000, 64, 32),     # ... partial, odd row pitches
], ids=lambda s: "x".join(map(str, s)))
def test_16_bit_64_tile(oracle, shape, dtype):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import input_grad_hashed, weight_grad_hashed
    from rzlinear_amd.impl.RzLinearForward import forward_hashed
    M, K, N, H, BK, BN = shape
    _say(shape, dtype)
    (x, hw, dy), (x64, hw64, dy64) = make_inputs(M, K, N, H, dtype, seed=M)
    R = _lib.hash_constants(*rargs(R1024))
    with _lib.tuning(tile=64, split=-1, window=-1):
        y = forward_hashed(x, hw, None, 0.75, M, K, N, H, R, BK, BN, 2)
        dx = input_grad_hashed(dy, hw, 0.75, M, K, N, H, R, BK, BN, 2)
        dhw, dbias = weight_grad_hashed(x, dy, 0.75, M, K, N, H, R, BK, BN, out=torch.empty(H, device="cuda"), with_bias_grad=True)
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, N, BK, BN, R1024, 0.75), dtype, "y")
    assert_close(dx.float().cpu().numpy(), oracle.input_grad(dy64, hw64, K, BK, BN, R1024, 0.75), dtype, "dx")
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.75)
    assert np.abs(dhw.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()   # (fp32 sums of exact products)
    assert_close(dbias.float().cpu().numpy(), dy64.sum(0), dtype, "bias gradient")


@pytest.mark.parametrize("dtype", [torch.float32] + SIXTEEN, ids=str)
@pytest.mark.parametrize("shape", [
    (4096, 512, 512, 5243, 64, 64),       # sixteen slices of 128 tiles, complete
    (4090, 500, 1000, 20000, 32, 64),     # eight, partial tiles and a partial last slice
    (8191, 511, 509, 9000, 64, 64),       # odd row pitches
], ids=lambda s: "x".join(map(str, s)))
def test_weight_grad_in_whole_slices_per_xcd(oracle, shape, dtype):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H, BK, BN = shape
    _say(shape, dtype)
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, dtype, seed=M)
    q = _lib.plan_query(2, M, K, N, H, BK, BN, _lib.dtype_code(x), _lib.WG_DHW_F32, True)
    assert q["mode"] == "lds_image" and q["slices"] % 8 == 0, q
    dhw, dbias = weight_grad_hashed(x, dy, 0.75, M, K, N, H, _lib.hash_constants(*rargs(R1024)), BK, BN,
                                    out=torch.empty(H, device="cuda"), with_bias_grad=True)
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.75)
    # (fp32 sums of M products and about a hundred tiles per element)
    assert np.abs(dhw.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()
    assert_close(dbias.float().cpu().numpy(), dy64.sum(0), dtype, "bias gradient")


@pytest.mark.parametrize("dtype", [torch.float32] + SIXTEEN, ids=str)
@pytest.mark.parametrize("shape", [
    (32, 512, 256, 60000, 32, 64),    # one workgroup of the bias gradient, complete
    (33, 512, 264, 60000, 32, 64),    # a second one of eight columns
    (3, 300, 1001, 60000, 32, 32),    # fewer rows than row groups, odd row pitch
], ids=lambda s: "x".join(map(str, s)))
def test_bias_gradient_behind_the_windows(oracle, shape, dtype):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H, BK, BN = shape
    _say(shape, dtype)
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, dtype, seed=M)
    with _lib.tuning(window=1, fold=-1, lds_image=-1):
        assert _lib.plan_query(2, M, K, N, H, BK, BN, _lib.dtype_code(x), _lib.WG_DHW_F32, True)["mode"] == "window"
        dhw, dbias = weight_grad_hashed(x, dy, 0.75, M, K, N, H, _lib.hash_constants(*rargs(R1024)), BK, BN,
                                        out=torch.empty(H, device="cuda"), with_bias_grad=True)
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.75)
    assert np.abs(dhw.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()   # (fp32 sums of exact products)
    assert_close(dbias.float().cpu().numpy(), dy64.sum(0), dtype, "bias gradient")


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("extents", [(256, 512), (256, 384), (250, 391)], ids=str)   # (both tiles complete; the 128 tile; neither)
@pytest.mark.parametrize("steps,rest", [(1, 0), (2, 0), (3, 0), (4, 0), (5, 0), (6, 0), (7, 0), (9, 0), (36, 0),
                                        (0, 17), (1, 1), (2, 31), (3, 32), (4, 63), (5, 33), (7, 33), (8, 33), (9, 63),
                                        (10, 1), (11, 40), (12, 17), (17, 8)], ids=str)
@pytest.mark.parametrize("tile", [128, 256])
def test_16_bit_pipelined_tiles_at_few_steps(oracle, tile, steps, rest, extents, dtype):
    """The loops that load several R steps of 64 elements ahead: fewer steps than are in flight, every remainder of the
    stages, a partial last step, past the first bank of the offset table; the 256 tile's two loops on either side of the rule that chooses; complete and ragged tiles; all
    three operations, dHW through LDS images and through stored tiles, bias gradient included."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl, weight_grad_hashed
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_bias_tl
    r, (a, b), H, BK, BN = 64 * steps + rest, extents, 20000, 32, 64
    _say(tile, r, extents, dtype)
    R = _lib.hash_constants(*rargs(R1024))
    bias = torch.randn((b,), generator=torch.Generator().manual_seed(4)).to(dtype)
    with _lib.tuning(tile=tile, split=-1):
        (x, hw, _), (x64, hw64, _) = make_inputs(a, r, b, H, dtype, seed=r)
        y = rz_linear_forward_bias_tl(x, hw, bias.cuda(), 0.75, a, r, b, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
        assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, b, BK, BN, R1024, 0.75) + bias.double().numpy(), dtype, "y")
        (_, hw, dy), (_, hw64, dy64) = make_inputs(a, b, r, H, dtype, seed=r)
        dx = rz_linear_backward_input_grad_tl(dy, hw, 0.75, a, b, r, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
        assert_close(dx.float().cpu().numpy(), oracle.input_grad(dy64, hw64, b, BK, BN, R1024, 0.75), dtype, "dx")
    (x, _, dy), (x64, _, dy64) = make_inputs(r, a, b, H, dtype, seed=r)
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5)
    for how in ({"window": -1}, {"lds_image": -1, "window": -1, "fold": 2}):
        out = torch.empty((H,), dtype=torch.float32, device="cuda")
        with _lib.tuning(tile=tile, **how):
            _, dbias = weight_grad_hashed(x, dy, 0.5, r, a, b, H, R, BK, BN, out=out, with_bias_grad=True)
        # (fp32 sums of exact products: at most r of them per stored value and a few dozen values per slot)
        assert np.abs(out.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()
        assert_close(dbias.float().cpu().numpy(), dy64.sum(0), dtype, "bias gradient")


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("extents", [(2048, 2304), (2030, 2299)], ids=str)
@pytest.mark.parametrize("r", [8, 64, 65, 128, 191, 192, 256, 300, 320, 384, 1000, 1088, 2300], ids=str)
def test_16_bit_pairs_of_tiles(oracle, extents, r, dtype):
    """288 tiles of 128 are more than compute units: pairs, 144 workgroups of 256 x 128 — fewer steps than its three stages
    hold, every remainder of them, a partial last step, past the first bank of the offset table; complete and ragged."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_bias_tl
    (a, b), H, BK, BN = extents, 20000, 32, 64
    _say(r, extents, dtype)
    bias = torch.randn((b,), generator=torch.Generator().manual_seed(4)).to(dtype)
    (x, hw, _), (x64, hw64, _) = make_inputs(a, r, b, H, dtype, seed=r)
    with _lib.tuning(split=-1):
        for op, K, N in ((0, r, b), (1, b, r)):
            q = _lib.plan_query(op, a, K, N, H, BK, BN, _lib.dtype_code(x))
            assert (q["tile"], q["slices"], q["workgroups"], q["step"]) == (128, 1, 144, 64)
        y = rz_linear_forward_bias_tl(x, hw, bias.cuda(), 0.75, a, r, b, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
        dx = rz_linear_backward_input_grad_tl(x, hw, 0.75, a, b, r, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, b, BK, BN, R1024, 0.75) + bias.double().numpy(), dtype, "y")
    assert_close(dx.float().cpu().numpy(), oracle.input_grad(x64, hw64, b, BK, BN, R1024, 0.75), dtype, "dx")


def _odd_pitch(t, before):
    """A view with the values of t inside rows of odd pitch, at an odd start, with infinities and NaN all around it."""
    cols = t.shape[1]
    big = torch.full((t.shape[0], before + cols + 2 + (before + cols + 1) % 2), float("inf"), dtype=t.dtype, device=t.device)
    big[:, ::2] = float("nan")
    view = big[:, before:before + cols]
    view.copy_(t)
    assert view.stride(0) % 2 == 1 and view.data_ptr() % 16 != 0
    return view


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("extents", [(256, 512), (250, 391)], ids=str)
@pytest.mark.parametrize("r", [17, 64, 191, 256, 300, 1088], ids=str)
@pytest.mark.parametrize("tile", [128, 256])
def test_16_bit_pipelined_tiles_in_odd_pitches(oracle, tile, r, extents, dtype):
    """Operands that are part of wider rows: what lies behind a row's last element (infinities and NaN) is fetched with it and
    must be cleared in LDS, in both halves of the 256 tile's rows; all three operations, dHW through images and stored tiles."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl, weight_grad_hashed
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_tl
    (a, b), H, BK, BN = extents, 20000, 32, 64
    _say(tile, r, extents, dtype)
    R = _lib.hash_constants(*rargs(R1024))
    kw = dict(BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    with _lib.tuning(tile=tile, split=-1):
        (x, hw, _), (x64, hw64, _) = make_inputs(a, r, b, H, dtype, seed=r)
        y = rz_linear_forward_tl(_odd_pitch(x, 1), hw, 0.75, a, r, b, H, *rargs(R1024), **kw)
        assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, b, BK, BN, R1024, 0.75), dtype, "y")
        (_, hw, dy), (_, hw64, dy64) = make_inputs(a, b, r, H, dtype, seed=r)
        dx = rz_linear_backward_input_grad_tl(_odd_pitch(dy, 3), hw, 0.75, a, b, r, H, *rargs(R1024), **kw)
        assert_close(dx.float().cpu().numpy(), oracle.input_grad(dy64, hw64, b, BK, BN, R1024, 0.75), dtype, "dx")
    (x, _, dy), (x64, _, dy64) = make_inputs(r, a, b, H, dtype, seed=r)
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5)
    for how in ({"window": -1}, {"lds_image": -1, "window": -1, "fold": 2}):
        out = torch.empty((H,), dtype=torch.float32, device="cuda")
        with _lib.tuning(tile=tile, **how):
            _, dbias = weight_grad_hashed(_odd_pitch(x, 3), _odd_pitch(dy, 1), 0.5, r, a, b, H, R, BK, BN, out=out, with_bias_grad=True)
        # (fp32 sums of exact products: at most r of them per stored value and a few dozen values per slot)
        assert np.abs(out.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()
        assert_close(dbias.float().cpu().numpy(), dy64.sum(0), dtype, "bias gradient")


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("extents", [(2048, 2304), (2030, 2299)], ids=str)
@pytest.mark.parametrize("r", [65, 192, 300], ids=str)
def test_16_bit_pairs_of_tiles_in_odd_pitches(oracle, extents, r, dtype):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_tl
    (a, b), H, BK, BN = extents, 20000, 32, 64
    _say(r, extents, dtype)
    (x, hw, _), (x64, hw64, _) = make_inputs(a, r, b, H, dtype, seed=r)
    wide, kw = _odd_pitch(x, 1), dict(BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)
    with _lib.tuning(split=-1):
        for op, K, N in ((0, r, b), (1, b, r)):
            q = _lib.plan_query(op, a, K, N, H, BK, BN, _lib.dtype_code(x))
            assert (q["tile"], q["slices"], q["workgroups"], q["step"]) == (128, 1, 144, 64)
        y = rz_linear_forward_tl(wide, hw, 0.75, a, r, b, H, *rargs(R1024), **kw)
        dx = rz_linear_backward_input_grad_tl(wide, hw, 0.75, a, b, r, H, *rargs(R1024), **kw)
    assert_close(y.float().cpu().numpy(), oracle.forward(x64, hw64, b, BK, BN, R1024, 0.75), dtype, "y")
    assert_close(dx.float().cpu().numpy(), oracle.input_grad(x64, hw64, b, BK, BN, R1024, 0.75), dtype, "dx")


@pytest.mark.parametrize("shape,mode,tile", [
    ((96, 449, 6200, 27389, 64, 64), "lds_image", 128),        # images of the 128 tile, K odd
    ((2000, 2043, 2051, 20000, 32, 64), "lds_image", 256),     # slices, a partial last one
    ((1948, 2184, 1810, 197652, 64, 64), "fold", 256),         # stored slices in fp32
    ((2322, 536, 3404, 91227, 64, 64), "fold", 128),
], ids=str)
def test_16_bit_weight_grad_plans_in_odd_pitches(oracle, shape, mode, tile):
    """The plans that sizes pick by themselves, on operands inside wider rows."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H, BK, BN = shape
    _say(shape)
    q = _lib.plan_query(2, M, K, N, H, BK, BN, _lib.RZ_BF16)
    assert (q["mode"], q["tile"]) == (mode, tile), q
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, torch.bfloat16, seed=M)
    dhw, dbias = weight_grad_hashed(_odd_pitch(x, 1), _odd_pitch(dy, 3), 0.5, M, K, N, H, _lib.hash_constants(*rargs(R1024)), BK, BN,
                                    with_bias_grad=True)
    assert_close(dhw.float().cpu().numpy(), oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5), torch.bfloat16, "dHW")
    assert_close(dbias.float().cpu().numpy(), dy64.sum(0), torch.bfloat16, "bias gradient")


@pytest.mark.parametrize("shape,slices", [((200, 6000, 6000, 20000, 32, 64), 5), ((896, 3968, 2368, 20000, 64, 64), 3), ((900, 4001, 2371, 20000, 32, 64), 3)], ids=str)
def test_16_bit_cut_pairs_of_tiles(oracle, shape, slices):
    """Pairs over slices of the contraction, their planes added by the second kernel or in the kernel: the same bits."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearForward import rz_linear_forward_bias_tl
    M, K, N, H, BK, BN = shape
    _say(shape)
    (x, hw, _), (x64, hw64, _) = make_inputs(M, K, N, H, torch.bfloat16, seed=3)
    bias = torch.randn((N,), generator=torch.Generator().manual_seed(4)).bfloat16()
    out = []
    for finish in (0, -1):
        with _lib.tuning(split=slices, finish=finish):
            q = _lib.plan_query(0, M, K, N, H, BK, BN, _lib.RZ_BF16)
            assert (q["tile"], q["slices"], q["workgroups"]) == (128, slices, -(-M // 256) * -(-N // 128) * slices)
            out.append(rz_linear_forward_bias_tl(x, hw, bias.cuda(), 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN))
    assert torch.equal(out[0], out[1])
    assert_close(out[0].float().cpu().numpy(), oracle.forward(x64, hw64, N, BK, BN, R1024, 0.75) + bias.double().numpy(), torch.bfloat16, "y")


@pytest.mark.parametrize("shape,tile,slices", [
    ((1963, 1344, 3328, 279552, 64, 64), 256, 2),     # added by atomics when cut no further than those allow
    ((1948, 2184, 1810, 197652, 64, 64), 256, 2),     # odd row pitches, partial tiles and a partial last step
    ((4846, 519, 1167, 41000, 64, 64), 128, 5),       # the fewest tiles
    ((2322, 536, 3404, 91227, 64, 64), 128, 3),
], ids=str)
def test_16_bit_weight_grad_in_stored_slices(oracle, shape, tile, slices):
    """Slices of M stored tile by tile are partial sums and kept in fp32: only dHW itself is rounded."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H, BK, BN = shape
    _say(shape)
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, torch.bfloat16, seed=M)
    R = _lib.hash_constants(*rargs(R1024))
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5)
    q = _lib.plan_query(2, M, K, N, H, BK, BN, _lib.RZ_BF16)
    assert (q["mode"], q["tile"], q["slices"]) == ("fold", tile, slices)
    assert all(stored_tile_bytes(shape, _lib.RZ_BF16, planned) == 4 for planned in (False, True))
    for plans in (False, True):
        dhw, dbias = weight_grad_hashed(x, dy, 0.5, M, K, N, H, R, BK, BN, with_bias_grad=True, use_layer_plan=plans)
        assert_close(dhw.float().cpu().numpy(), ref, torch.bfloat16, "dHW")
        assert_close(dbias.float().cpu().numpy(), dy64.sum(0), torch.bfloat16, "bias gradient")


def test_static_scratch_takes_the_cut_that_fits(oracle):
    """rz_weight_grad stores two or more slices for this problem, more than the static scratch holds; the static entry point
    keeps the plan that it would hold, folded in a fixed order."""
    import ctypes
    from rzlinear_amd import _lib
    lib = _lib.load()
    M, K, N, H, BK, BN = 1878, 781, 4746, 185331, 64, 64
    assert _lib.plan_query(2, M, K, N, H, BK, BN, _lib.RZ_BF16)["slices"] > 1
    assert lib.rz_weight_grad_workspace_bytes(M, K, N, H, BK, BN, _lib.RZ_BF16) > 32 << 20
    _say("static scratch, fewer slices", (M, K, N, H))
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, torch.bfloat16, seed=72)
    # (its tiles are whole sums over M, rounded once to bf16; the slices of the other entry points are kept in fp32)
    slack = rounded_tiles_slack(oracle, x64, dy64, (M, K, N, H, BK, BN), R1024, 0.5, torch.bfloat16, M)
    R = (ctypes.c_int32 * 8)(*R1024)
    out = [torch.full((H,), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    for o in out:
        _lib.check(lib.rz_weight_grad_static(x.data_ptr(), dy.data_ptr(), o.data_ptr(), M, K, N, H, BK, BN, R, 0.5, K, N,
                                             _lib.RZ_BF16, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    assert_close(out[0].float().cpu().numpy(), oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5), torch.bfloat16, "dHW", slack=slack)


@pytest.mark.parametrize("shape,slices", [
    ((96, 449, 6200, 27389, 64, 64), 1),       # 196 workgroups, odd rows, partial tiles
    ((933, 849, 463, 24001, 32, 64), 8),
    ((96, 8768, 2496, 8233, 32, 64), 1),       # 1380 workgroups, two on a compute unit
], ids=str)
def test_16_bit_image_in_128_tiles(oracle, shape, slices):
    """Images of the 128 tile where the fitted times prefer it to the 256 tile."""
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H, BK, BN = shape
    _say(shape)
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, torch.bfloat16, seed=M)
    q = _lib.plan_query(2, M, K, N, H, BK, BN, _lib.RZ_BF16)
    assert (q["mode"], q["tile"], q["slices"]) == ("lds_image", 128, slices)
    dhw, dbias = weight_grad_hashed(x, dy, 0.5, M, K, N, H, _lib.hash_constants(*rargs(R1024)), BK, BN, with_bias_grad=True)
    assert_close(dhw.float().cpu().numpy(), oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5), torch.bfloat16, "dHW")
    assert_close(dbias.float().cpu().numpy(), dy64.sum(0), torch.bfloat16, "bias gradient")


@pytest.mark.parametrize("dtype", SIXTEEN, ids=str)
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_mfma_probe_multiplies_what_it_says(mode, dtype):
    """Every mode does the same work: with operands of one, a thread adds up 128 accumulators of 64 products per step."""
    from rzlinear_amd import _lib
    wgs, steps = 3, 5
    operands = torch.ones((32768,), dtype=dtype, device="cuda")
    out = torch.zeros((wgs * 512,), dtype=torch.float32, device="cuda")
    ticks = torch.zeros((2 * wgs,), dtype=torch.int64, device="cuda")
    _lib.check(_lib.load().rz_mfma_probe(operands.data_ptr(), out.data_ptr(), ticks.data_ptr(), wgs, steps, mode,
                                         _lib.dtype_code(operands), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out.cpu(), torch.full((wgs * 512,), 128.0 * 64 * steps))   # (whole numbers: exact in fp32)
    assert bool((ticks[::2] > 0).all())
