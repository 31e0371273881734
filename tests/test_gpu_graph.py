"""The entry points enqueue kernels only (no allocation, no synchronisation, no memset nodes), so
a training step can be captured in a HIP graph and replayed.  Every replay is compared with the
eager result of the same inputs, with eager work and synchronisations between replays."""
import ctypes
import sys

import pytest
import torch

from helpers import SEED_CONSTANTS, rargs

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("cfg", [
    (512, 512, 768, 9000, torch.bfloat16),      # LDS-image weight-grad, direct staging
    (96, 1024, 512, 70000, torch.float32),      # atomic scatter (zero-fill kernel inside the graph), split forward
    (32, 4096, 4096, 1 << 20, torch.bfloat16),  # window kernel (offset table built inside the graph)
    (520, 4096, 4096, 200000, torch.bfloat16),  # tile-by-tile output + fold kernel + reduction of its images
], ids=lambda c: "x".join(map(str, c[:4])) + "-" + str(c[4]).split(".")[-1])
def test_step_captured_in_a_graph_replays_correctly(cfg):
    from rzlinear_amd import _lib
    M, K, N, H, dtype = cfg
    BK = BN = 64
    _say("graph capture", cfg)
    lib = _lib.load()
    R = (ctypes.c_int32 * 8)(*R1024)
    code = {torch.float32: 0, torch.bfloat16: 1}[dtype]
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(9)
    x = torch.randn((M, K), generator=g).to(dtype).to(dev)
    hw = ((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype).to(dev)
    dy = torch.randn((M, N), generator=g).to(dtype).to(dev)
    bias = torch.randn((N,), generator=g).to(dtype).to(dev)
    y = torch.empty((M, N), dtype=dtype, device=dev)
    dx = torch.empty((M, K), dtype=dtype, device=dev)
    dhw = torch.empty((H,), dtype=dtype, device=dev)
    dbias = torch.empty((N,), dtype=dtype, device=dev)
    fws = lib.rz_forward_workspace_bytes(M, K, N, H, BK, BN, code)
    iws = lib.rz_input_grad_workspace_bytes(M, K, N, H, BK, BN, code)
    wws = lib.rz_weight_grad_ex_workspace_bytes(M, K, N, H, BK, BN, code, 0, 0)
    wbs = lib.rz_weight_grad_ex_workspace_bytes(M, K, N, H, BK, BN, code, 0, 1)
    bufs = [torch.empty((max(n, 16),), dtype=torch.uint8, device=dev) for n in (fws, iws, wws, wbs)]

    def step(stream):
        _lib.check(lib.rz_forward_ws(x.data_ptr(), hw.data_ptr(), bias.data_ptr(), y.data_ptr(), bufs[0].data_ptr(),
                                     fws, M, K, N, H, BK, BN, R, 0.5, K, N, code, stream))
        _lib.check(lib.rz_input_grad_ws(dy.data_ptr(), hw.data_ptr(), dx.data_ptr(), bufs[1].data_ptr(), iws,
                                        M, K, N, H, BK, BN, R, 0.5, N, K, code, stream))
        # with the bias gradient first; the call without it comes last and decides dhw (for the
        # third configuration that is the window kernel, whose result is reproducible)
        _lib.check(lib.rz_weight_grad_ex(x.data_ptr(), dy.data_ptr(), dhw.data_ptr(), dbias.data_ptr(),
                                         bufs[3].data_ptr(), wbs, M, K, N, H, BK, BN, R, 0.5, K, N, code, 0, stream))
        _lib.check(lib.rz_weight_grad_ex(x.data_ptr(), dy.data_ptr(), dhw.data_ptr(), None, bufs[2].data_ptr(), wws,
                                         M, K, N, H, BK, BN, R, 0.5, K, N, code, 0, stream))

    # warm up on a side stream (first launches set kernel attributes), then capture
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(side.cuda_stream)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(torch.cuda.current_stream().cuda_stream)

    outs = (y, dx, dhw, dbias)
    for replay in range(4):
        # new inputs, written by ordinary eager kernels
        x.copy_(torch.randn((M, K), generator=g).to(dtype))
        dy.copy_(torch.randn((M, N), generator=g).to(dtype))
        hw.copy_(((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype))
        step(torch.cuda.current_stream().cuda_stream)      # eager reference
        torch.cuda.synchronize()
        eager = [t.clone() for t in outs]
        for t in outs:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(("y", "dx", "dhw", "dbias"), outs, eager):
            if name == "dhw" and cfg[3] == 70000:
                # atomic scatter: summation order differs from run to run
                assert torch.allclose(a.float(), b.float(), rtol=1e-4, atol=1e-4 * float(b.float().abs().max())), (name, replay)
            else:
                assert torch.equal(a, b), (name, replay)


@pytest.mark.parametrize("shape", [
    (16, 1024, 2048, 524288),     # by windows with a layer plan, by atomics without
    (32, 4096, 4096, 1 << 20),    # by windows, or folded without
    (520, 4096, 4096, 200000),    # folded
], ids=str)
@pytest.mark.parametrize("native", [True, False], ids=["module", "launcher"])
def test_a_layer_without_a_plan_is_captured_without_one(oracle, shape, native):
    """A layer plan is built with a copy that a capture does not take: a backward that is captured before the layer has one goes without, as
    calls of paths that have none always have.  The kernels are warm: another layer of the same shape has run."""
    import numpy as np
    from helpers import TOL, rel_err
    from rzlinear_amd import RzLinear, _lib
    from rzlinear_amd.impl.RzLinearBackward import weight_grad_hashed
    M, K, N, H = shape
    dtype, BK, BN = torch.bfloat16, 64, 64
    _say("capture without a plan", shape, native)
    g = torch.Generator().manual_seed(2)
    x = torch.randn((M, K), generator=g).to(dtype).cuda().requires_grad_(True)
    dy = torch.randn((M, N), generator=g).to(dtype).cuda()
    layers = [RzLinear(K, N, hashed_weight=torch.nn.Parameter(((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype)), seed=seed, dtype=dtype,
                       block_size_k=BK, block_size_n=BN).cuda() for seed in (31, 32)]

    def backward(layer, with_plans=None):
        if native:
            return torch.autograd.grad(layer(x), (layer._hashed_weight,), dy)[0]
        R = _lib.hash_constants(*rargs([int(v) for v in layer._random_numbers]))
        return weight_grad_hashed(x.detach(), dy, layer._init_factor, M, K, N, H, R, BK, BN, use_layer_plan=with_plans)[0]

    _lib.clear_layer_plans()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        backward(layers[0])
        _lib.use_layer_plans = False
        try:
            backward(layers[0])   # (the kernels of the way without a plan)
        finally:
            _lib.use_layer_plans = True
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    plans = len(_lib._layer_plans)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dhw = backward(layers[1])
    assert len(_lib._layer_plans) == plans
    for replay in range(3):
        with torch.no_grad():
            x.copy_(torch.randn((M, K), generator=g).to(dtype))
        dhw.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        ref = oracle.weight_grad(x.detach().double().cpu().numpy(), dy.double().cpu().numpy(), H, BK, BN,
                                 [int(v) for v in layers[1]._random_numbers], layers[1]._init_factor)
        assert rel_err(dhw.float().cpu().numpy(), ref) <= TOL[dtype], replay
    eager = backward(layers[1])   # (which builds the plan: a capture from now on has it)
    assert len(_lib._layer_plans) == plans + 1
    assert rel_err(eager.float().cpu().numpy(), np.asarray(ref)) <= TOL[dtype]
