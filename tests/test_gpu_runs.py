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
        assert _lib.plan_query(op, *shape, _lib.dtype_code(x))["shares"] == 0
        same = _lib.plan_query(op, *shape, _lib.dtype_code(x))["windows"] == q["windows"]
        if same:   # (priced without the finish, another plan may be the better one)
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
