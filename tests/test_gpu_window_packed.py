"""The window kernel's operands as MFMA fragments (made by a kernel of the same call where the workspace has room) and its
several images of a small window, at the edges of both, against the oracle and against the forms without that workspace."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import SEED_CONSTANTS, TOL, make_inputs, rargs, rel_err

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]
# (M, K, N, H, BK, BN)
CASES = [
    (1, 3001, 4095, 700001, 32, 64),      # one row: a group that is nearly empty; rows that are not whole pieces, odd H
    (16, 3001, 2051, 380000, 32, 64),     # a group exactly; windows of 1488, sixteen images
    (17, 2047, 3003, 400000, 64, 64),     # ... and one row more
    (33, 2080, 4104, 1000000, 64, 64),    # whole pieces, little to gain: staged whether there is room or not
    (64, 1025, 4099, 1300000, 32, 128),   # two units side by side; windows of 5080, four images
    (47, 2100, 2100, 200000, 128, 32),    # 32-column units
    (257, 1030, 1030, 66000, 64, 64),     # many groups of rows; tiles that reach beyond K and N: fragments of zeros
    (31, 4096, 4100, 3300000, 64, 64),    # one image, though two would fit beside the fragments
    (18, 4100, 6000, 7000000, 32, 64),    # two rounds of windows, one image
    (9, 4096, 8192, 40000, 64, 64),       # more units meet a window than its list holds: images over several rounds
]


def _call(lib, x, dy, out, ws, nbytes, plan, shape, code, tuning):
    from rzlinear_amd import _lib
    M, K, N, H, BK, BN = shape
    R = _lib.hash_constants(*rargs(R1024))
    stream = torch.cuda.current_stream().cuda_stream
    if plan is None:
        st = lib.rz_weight_grad_hashed(x.data_ptr(), dy.data_ptr(), out.data_ptr(), None, ws, nbytes, M, K, N, H, BK, BN, R, 2, 0.5,
                                       x.stride(0), dy.stride(0), code, 0, tuning, stream)
    else:
        st = lib.rz_weight_grad_planned(x.data_ptr(), dy.data_ptr(), out.data_ptr(), None, ws, nbytes, plan.data_ptr(), plan.numel() * 4,
                                        M, K, N, H, BK, BN, R, 2, 0.5, x.stride(0), dy.stride(0), code, 0, tuning, stream)
    _lib.check(st)
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", CASES, ids=lambda s: "x".join(map(str, s)))
def test_fragments_and_images(oracle, shape, dtype):
    from rzlinear_amd import _lib
    M, K, N, H, BK, BN = shape
    print("packed window", shape, dtype, flush=True)
    (x, _, dy), (x64, _, dy64) = make_inputs(M, K, N, H, dtype, seed=5)
    ref = oracle.weight_grad(x64, dy64, H, BK, BN, R1024, 0.5)
    # rows at an odd pitch, starting at an odd element, between NaN: nothing outside the operands is used
    wide = []
    for t in (x, dy):
        w = torch.full((M + 2, t.shape[1] + 5), float("nan"), dtype=dtype, device=t.device)
        w[1:M + 1, 3:3 + t.shape[1]] = t
        wide.append(w[1:M + 1, 3:3 + t.shape[1]])
    lib = _lib.load()
    code = _lib.dtype_code(x)
    t = _lib.Tuning(window=1)
    tuning = ctypes.byref(t)
    need = lib.rz_weight_grad_hashed_workspace_bytes(M, K, N, H, BK, BN, code, 0, 0, tuning)
    offsets = -(-K // BK) * -(-N // BN) * 4
    plan = _lib.layer_plan(K, N, H, BK, BN, _lib.hash_constants(*rargs(R1024)), 2, x.device)
    ws = torch.full((need + 512,), 255, dtype=torch.uint8, device=x.device)   # (fragments and offsets of NaN and -1)
    got = {}
    for name, (a, b), at, nbytes, p in (
            ("packed", (x, dy), ws.data_ptr(), need, None),
            ("planned", (x, dy), ws.data_ptr(), need, plan),
            ("wide rows", wide, ws.data_ptr(), need, plan),
            ("workspace at four bytes", (x, dy), ws.data_ptr() + 4, need, None),
            ("offsets alone", (x, dy), ws.data_ptr(), (offsets + 255) // 256 * 256, None),
            ("no workspace", (x, dy), None, 0, plan)):
        ws.fill_(255)
        out = torch.full((H,), float("nan"), dtype=dtype, device=x.device)
        _call(lib, a, b, out, at, nbytes, p, shape, code, tuning)
        got[name] = out
        assert rel_err(out.float().cpu().numpy(), ref) <= TOL[dtype], name
        assert (out.float().cpu().numpy()[ref == 0] == 0).all(), name
        assert bool((ws[need + 256:] == 255).all()), name   # (nothing behind the workspace)
    for name in got:   # (as many images either way)
        assert torch.equal(got[name], got["packed"]), name


def test_workspace_query_has_room_for_the_fragments_of_a_planned_call():
    """With a layer plan the window kernel is taken for batches that go elsewhere without one: the workspace is asked for
    without saying which, and holds the fragments either way."""
    from rzlinear_amd import _lib
    lib = _lib.load()
    differ = 0
    for M, K, N, H in ((m, k, n, k * n // 16) for m in (8, 64, 128, 256) for k in (1024, 2048, 4096) for n in (2048, 5120)):
        for code in (_lib.RZ_F32, _lib.RZ_BF16):
            planned = _lib.plan_query(2, M, K, N, H, 64, 64, code, planned=True)["mode"]
            differ += planned != _lib.plan_query(2, M, K, N, H, 64, 64, code)["mode"]
            if planned == "window" and code == _lib.RZ_BF16 and M >= 128 and K >= 2048:   # (where they are worth it)
                need = lib.rz_weight_grad_hashed_workspace_bytes(M, K, N, H, 64, 64, code, 0, 0, None)
                assert need >= (M + 15) // 16 * 16 * (K + N) * 2, (M, K, N)
    assert differ > 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (31, 4096, 4100, 3300000, 64, 64),   # windows of 12892: two images would fit beside the fragments, one beside the staging area
    (20, 2100, 4096, 1664000, 32, 64),   # ... of 6500: four and two
    (64, 1001, 3333, 1100000, 64, 128),  # ... of 4300: eight and four; element by element without the fragments
    (40, 2048, 2048, 262144, 32, 32),    # ... of 1024: sixteen either way
], ids=lambda s: "x".join(map(str, s)))
def test_the_bits_do_not_depend_on_the_workspace(shape, dtype):
    """The same order of the sums with the operands as fragments, and without room for them."""
    from rzlinear_amd import _lib
    M, K, N, H, BK, BN = shape
    print("window bits", shape, dtype, flush=True)
    (x, _, dy), _ = make_inputs(M, K, N, H, dtype, seed=6)
    lib = _lib.load()
    code = _lib.dtype_code(x)
    t = _lib.Tuning(window=1)
    tuning = ctypes.byref(t)
    need = lib.rz_weight_grad_hashed_workspace_bytes(M, K, N, H, BK, BN, code, 0, 0, tuning)
    ws = torch.empty((need,), dtype=torch.uint8, device=x.device)
    plan = _lib.layer_plan(K, N, H, BK, BN, _lib.hash_constants(*rargs(R1024)), 2, x.device)
    got = []
    for at, nbytes, p in ((ws.data_ptr(), need, None), (ws.data_ptr(), need, plan), (None, 0, plan)):
        out = torch.full((H,), float("nan"), dtype=dtype, device=x.device)
        _call(lib, x, dy, out, at, nbytes, p, shape, code, tuning)
        got.append(out)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (20, 2047, 3003, 700001, 64, 64),
    (33, 2080, 4104, 1000000, 64, 128),   # rows of whole pieces
    (7, 1030, 1030, 200000, 128, 32),
], ids=lambda s: "x".join(map(str, s)))
def test_infinities_stay_where_w_has_elements(oracle, shape, dtype):
    """One infinite gradient reaches the places of its column of W, one infinite input those of its row, and none of the places
    that a tile at the edge of W spans beyond it."""
    from rzlinear_amd import _lib
    M, K, N, H, BK, BN = shape
    print("window infinities", shape, dtype, flush=True)
    (x, _, dy), _ = make_inputs(M, K, N, H, dtype, seed=7)
    x[x == 0] = 1
    dy[dy == 0] = 1
    k_inf, n_inf = K - 3, N - 2
    x[M - 1, k_inf] = float("inf")
    dy[M // 2, n_inf] = float("-inf")
    idx = oracle.index_map(K, N, H, BK, BN, R1024)
    touched = np.zeros(H, dtype=bool)
    touched[idx[k_inf]] = True
    touched[idx[:, n_inf]] = True
    lib = _lib.load()
    code = _lib.dtype_code(x)
    t = _lib.Tuning(window=1)
    tuning = ctypes.byref(t)
    need = lib.rz_weight_grad_hashed_workspace_bytes(M, K, N, H, BK, BN, code, 0, 0, tuning)
    ws = torch.empty((need,), dtype=torch.uint8, device=x.device)
    plan = _lib.layer_plan(K, N, H, BK, BN, _lib.hash_constants(*rargs(R1024)), 2, x.device)
    for at, nbytes in ((ws.data_ptr(), need), (None, 0)):
        out = torch.zeros((H,), dtype=dtype, device=x.device)
        _call(lib, x, dy, out, at, nbytes, plan, shape, code, tuning)
        assert ((~torch.isfinite(out)).cpu().numpy() == touched).all()
