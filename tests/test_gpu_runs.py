"""16-bit forward / input-grad in runs of equal length (rz_gemm_runs_kernel) against float32 products of the materialised W."""
import sys

import pytest
import torch

from helpers import SEED_CONSTANTS, assert_close, rargs

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]


def _calls(op, shape, dtype):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import rz_linear_backward_input_grad_tl
    from rzlinear_amd.impl.RzLinearForward import forward_hashed
    from rzlinear_amd.impl.RzLinearIdx import rz_linear_idx_tl
    M, K, N, H, BK, BN = shape
    print(op, shape, dtype, flush=True)
    sys.stdout.flush()
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn((M, K if op == 0 else N), generator=g).to(dtype).cuda()
    hw = ((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype).cuda()
    bias = torch.randn((N,), generator=g).to(dtype).cuda()
    consts = _lib.hash_constants(*rargs(R1024))

    def run():
        if op == 0:
            return forward_hashed(x, hw, bias, 0.75, M, K, N, H, consts, BK, BN, 2)
        return rz_linear_backward_input_grad_tl(x, hw, 0.75, M, K, N, H, *rargs(R1024), BLOCK_SIZE_K=BK, BLOCK_SIZE_N=BN)

    def reference(oracle):
        W = torch.from_numpy(oracle.index_map(K, N, H, BK, BN, R1024)).cuda()
        W = hw.float()[W.reshape(-1).long()].reshape(K, N)
        y = x.float() @ (W if op == 0 else W.t().contiguous()) * 0.75
        return y + bias.float() if op == 0 else y

    q = _lib.plan_query(op, M, K, N, H, BK, BN, _lib.dtype_code(x))
    return x, run, reference, q


CASES = [
    (0, (1024, 10240, 10240, 655360, 32, 64), 256, 3, torch.bfloat16),   # complete tiles, ends of tiles in pieces
    (1, (1024, 10240, 10240, 655360, 32, 64), 256, 3, torch.float16),
    (0, (3328, 7680, 10624, 81592, 64, 64), 128, 4, torch.bfloat16),     # whole rounds of 256 x 128 ahead
    (1, (5031, 4002, 6371, 100000, 64, 64), 256, 0, torch.bfloat16),     # whole rounds ahead, nothing a multiple of anything
    (0, (8864, 9146, 934, 100000, 32, 64), 256, 0, torch.float16),
    (1, (7114, 2563, 6678, 16384, 64, 64), 128, 3, torch.float16),       # ragged 256 x 128
]


@pytest.mark.parametrize("op,shape,tile,slices,dtype", CASES, ids=str)
def test_runs(oracle, op, shape, tile, slices, dtype):
    """The plan that is meant, right results, and the same bits again: whoever comes last at a tile, over a used workspace, and
    with the parts added up by a second kernel."""
    from rzlinear_amd import _lib
    x, run, reference, q = _calls(op, shape, dtype)
    assert q["windows"] > 0 and q["tile"] == tile and (slices == 0 or q["slices"] == slices), q
    first = run()
    assert_close(first.float().cpu().numpy(), reference(oracle).cpu().numpy(), dtype, "y" if op == 0 else "dx")
    for _ in range(4):
        assert torch.equal(run(), first)
    with _lib.tuning(finish=-1):
        assert _lib.plan_query(op, *shape, _lib.dtype_code(x)) == {**q, "shares": 0}
        assert torch.equal(run(), first)


@pytest.mark.parametrize("op,shape,tile,slices,dtype", CASES[:4:3], ids=str)
def test_captured_runs_are_added_up_by_a_second_kernel(op, shape, tile, slices, dtype):
    """A stream under capture gets no counters; the bits are the same, replay after replay."""
    x, run, _, _ = _calls(op, shape, dtype)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run()
    for replay in range(3):
        x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(replay)).to(dtype))
        finished = run()
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, finished), replay


def test_runs_on_several_streams_at_once():
    """Every stream has counters of its own."""
    op, shape, _, _, dtype = CASES[2]
    x, run, _, _ = _calls(op, shape, dtype)
    want = run()
    streams = [torch.cuda.Stream() for _ in range(4)]
    torch.cuda.synchronize()
    got = []
    for _ in range(2):
        for s in streams:
            with torch.cuda.stream(s):
                got.append(run())
    torch.cuda.synchronize()
    assert all(torch.equal(g, want) for g in got)


def _ws_call(op, x, hw, bias, out, ld_in, ld_out, ws, nbytes, shape, tuning=None):
    """rz_forward_hashed / rz_input_grad_hashed over a workspace and pitches of the test's choice; returns the status."""
    from rzlinear_amd import _lib
    M, K, N, H, BK, BN = shape
    lib = _lib.load()
    R = _lib.hash_constants(*rargs(R1024))
    stream = torch.cuda.current_stream().cuda_stream
    code = _lib.dtype_code(x)
    if op == 0:
        st = lib.rz_forward_hashed(x.data_ptr(), hw.data_ptr(), bias.data_ptr(), out.data_ptr(), ws, nbytes, M, K, N, H, BK, BN, R, 2, 0.75,
                                   ld_in, ld_out, code, tuning, stream)
    else:
        st = lib.rz_input_grad_hashed(x.data_ptr(), hw.data_ptr(), out.data_ptr(), ws, nbytes, M, K, N, H, BK, BN, R, 2, 0.75, ld_in, ld_out,
                                      code, tuning, stream)
    torch.cuda.synchronize()
    return st


def _need(op, shape, code, tuning=None):
    from rzlinear_amd import _lib
    lib = _lib.load()
    return (lib.rz_forward_hashed_workspace_bytes if op == 0 else lib.rz_input_grad_hashed_workspace_bytes)(*shape, code, tuning)


def _operands(op, shape, dtype, seed=4):
    M, K, N, H, BK, BN = shape
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((M, K if op == 0 else N), generator=g).to(dtype).cuda()
    hw = ((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype).cuda()
    bias = torch.randn((N,), generator=g).to(dtype).cuda()
    return x, hw, bias, torch.empty((M, N if op == 0 else K), dtype=dtype, device="cuda")


@pytest.mark.parametrize("op,shape,tile,slices,dtype", [CASES[0], CASES[3], CASES[5]], ids=str)
def test_runs_over_any_workspace_address_and_pitch(op, shape, tile, slices, dtype):
    """The planes are read and written two floats at a time: a workspace at any address has room to align them.  Rows of the operand and the
    result at odd pitches, between NaN and values that must stay."""
    from rzlinear_amd import _lib
    print("runs at odd addresses", op, shape, dtype, flush=True)
    x, hw, bias, out = _operands(op, shape, dtype)
    M, cols, J = shape[0], x.shape[1], out.shape[1]
    need = _need(op, shape, _lib.dtype_code(x))
    ws = torch.full((need + 256,), 255, dtype=torch.uint8, device="cuda")
    assert _ws_call(op, x, hw, bias, out, cols, J, ws.data_ptr(), need, shape) == 0
    wide_x = torch.full((M + 1, cols + 3), float("nan"), dtype=dtype, device="cuda")
    wide_x[:M, :cols] = x
    wide_out = torch.full((M + 1, J + 5), 7.0, dtype=dtype, device="cuda")
    for shift in (4, 1, 12):
        ws.fill_(255)
        out2 = wide_out[:M, :J]
        out2.fill_(float("nan"))
        assert _ws_call(op, wide_x, hw, bias, wide_out, cols + 3, J + 5, ws.data_ptr() + shift, need, shape) == 0
        assert torch.equal(out2, out), shift
        assert bool((wide_out[:, J:] == 7).all()) and bool((wide_out[M] == 7).all())
        assert bool((ws[:shift] == 255).all()) and bool((ws[need + shift:] == 255).all())


@pytest.mark.parametrize("op,shape,tile,slices,dtype", [CASES[0], CASES[3]], ids=str)
def test_runs_keep_infinities_and_nan_where_they_belong(op, shape, tile, slices, dtype):
    """A row with one infinite or NaN element gives a row without finite ones; the other rows have the bits they have without it."""
    print("runs with infinities", op, shape, dtype, flush=True)
    from rzlinear_amd import _lib
    x, hw, bias, out = _operands(op, shape, dtype)
    hw[hw == 0] = 1
    M, cols, J = shape[0], x.shape[1], out.shape[1]
    need = _need(op, shape, _lib.dtype_code(x))
    ws = torch.empty((need,), dtype=torch.uint8, device="cuda")
    assert _ws_call(op, x, hw, bias, out, cols, J, ws.data_ptr(), need, shape) == 0
    rows = {0: float("inf"), 255: float("nan"), M // 2: float("-inf"), M - 1: float("inf")}
    for i, (row, v) in enumerate(rows.items()):
        x[row, (cols - 1) * i // 3] = v
    got = torch.empty_like(out)
    assert _ws_call(op, x, hw, bias, got, cols, J, ws.data_ptr(), need, shape) == 0
    finite = torch.isfinite(got)
    keep = torch.ones(M, dtype=torch.bool, device="cuda")
    keep[list(rows)] = False
    assert not bool(finite[~keep].any()) and torch.equal(got[keep], out[keep])


@pytest.mark.parametrize("op,shape,dtype,slices_bytes", [
    (0, (3328, 7680, 10624, 81592, 64, 64), torch.bfloat16, 0),
    (1, (1895, 5660, 15920, 100000, 32, 64), torch.float16, 0),
    (0, (1024, 10240, 10240, 655360, 32, 64), torch.bfloat16, 3 * 1024 * 10240 * 4),   # (slices need planes too)
], ids=str)
def test_a_call_without_room_for_runs_does_what_it_would_without_them(op, shape, dtype, slices_bytes):
    """No workspace, or too little for the planes of runs: whole tiles, or slices, as such calls have always been accepted; an error only
    where slices need more."""
    import ctypes
    from rzlinear_amd import _lib
    print("no room for runs", op, shape, dtype, flush=True)
    x, hw, bias, out = _operands(op, shape, dtype)
    M, cols, J = shape[0], x.shape[1], out.shape[1]
    code = _lib.dtype_code(x)
    assert _lib.plan_query(op, *shape, code)["windows"] > 0
    need = _need(op, shape, code)
    assert slices_bytes < need
    ws = torch.empty((need,), dtype=torch.uint8, device="cuda")
    runs, whole = torch.empty_like(out), torch.empty_like(out)
    assert _ws_call(op, x, hw, bias, runs, cols, J, ws.data_ptr(), need, shape) == 0
    assert _ws_call(op, x, hw, bias, whole, cols, J, None, 0, shape, ctypes.byref(_lib.Tuning(split=-1))) == 0

    def close(a):
        return float((a.float() - whole.float()).abs().max() / whole.float().abs().max()) <= 2e-2
    assert close(runs)
    assert _ws_call(op, x, hw, bias, out, cols, J, None, 0, shape) == (0 if slices_bytes == 0 else -7)
    if slices_bytes > 0:
        assert _ws_call(op, x, hw, bias, out, cols, J, ws.data_ptr(), slices_bytes - 1, shape) == -7
    out.fill_(float("nan"))
    ws.fill_(255)
    assert _ws_call(op, x, hw, bias, out, cols, J, ws.data_ptr(), slices_bytes, shape) == 0 and close(out)
    assert bool((ws[slices_bytes:] == 255).all())
    again = torch.empty_like(out)
    assert _ws_call(op, x, hw, bias, again, cols, J, ws.data_ptr(), need - 1, shape) == 0 and torch.equal(again, out)
