"""Input-grad and weight-grad of a backward pass in one launch, against the two by themselves."""
import pytest
import torch

from helpers import SEED_CONSTANTS, make_inputs

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]
BF16, FP16, FP32 = torch.bfloat16, torch.float16, torch.float32

# (M, K, N, H, BK, BN), dtype: every pair of kernels, complete and ragged, at its smallest and around a round of workgroups
PAIRS = [
    ((96, 320, 192, 8192, 32, 64), BF16),          # 64 with 64, four stages, a ragged M
    ((1, 8, 9, 4096, 32, 64), BF16),               # ... one tile each, rows that are not whole pieces
    ((263, 286, 163, 8192, 64, 64), FP16),         # ... three slices of M
    ((128, 1024, 1024, 65536, 32, 64), BF16),      # ... more workgroups than compute units: two stages; stored tiles
    ((128, 256, 256, 16384, 32, 64), FP16),        # 64 with 128, complete
    ((160, 320, 1536, 8192, 64, 64), BF16),        # ... the input-grad cut
    ((337, 885, 1501, 13268, 32, 64), FP16),       # ... ragged, three slices of M
    ((62, 1001, 1203, 65536, 32, 64), BF16),       # ... stored tiles
    ((1024, 1024, 1024, 65536, 64, 64), FP32),     # fp32 64 with 64
    ((300, 135, 961, 16384, 64, 64), FP32),        # ... both cut, ragged
    ((61, 8384, 448, 234752, 64, 64), FP32),       # ... many more workgroups than compute units, of a short loop: apart
    ((2048, 1024, 1024, 20000, 64, 64), BF16),     # 128 with 128
    ((3738, 679, 525, 8192, 64, 64), FP16),        # ... ragged, eight slices (whole ones to an XCD)
    ((3072, 2048, 2048, 31340, 64, 64), BF16),     # 256 x 128 with 256
    ((3001, 2047, 1531, 31340, 64, 64), FP16),     # ... nothing a multiple of anything
    ((6144, 2048, 1536, 31340, 64, 64), BF16),     # 256 with 256
    ((6011, 2050, 1530, 31340, 64, 64), BF16),
    ((14456, 556, 802, 27869, 64, 64), BF16),      # 256 with 128, seven slices
    ((5056, 2304, 256, 36864, 64, 64), FP16),
    ((4288, 2304, 4544, 654336, 64, 64), BF16),    # 256 with 256, apart: no compute unit would be done sooner
    ((513, 6143, 6145, 300000, 64, 64), BF16),     # 256 x 128 with 256, stored tiles, ragged
    ((128, 2048, 4096, 400000, 32, 64), BF16),     # windows of dHW: no launch in common
    ((16384, 512, 1024, 5243, 64, 64), BF16),      # 256 x 128 with 128
    ((5001, 1030, 1021, 20000, 64, 64), FP16),
    ((2048, 4096, 1024, 262144, 32, 64), BF16),    # ... stored tiles
]


def _both_and_apart(shape, dtype, dhw_dtype=None, accumulate=False):
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import backward_hashed, input_grad_hashed, weight_grad_hashed
    M, K, N, H, BK, BN = shape
    print(shape, dtype, flush=True)
    (x, hw, dy), _ = make_inputs(M, K, N, H, dtype, seed=M + N)
    R = _lib.hash_constants(*[R1024[7 - i] for i in range(8)])
    before = torch.randn((H,), generator=torch.Generator().manual_seed(9)).cuda().to(dhw_dtype or dtype)
    outs = [before.clone() if accumulate else torch.full_like(before, float("nan")) for _ in range(2)]
    both = backward_hashed(x, hw, dy, 0.75, M, K, N, H, R, BK, BN, out=outs[0], accumulate=accumulate, with_bias_grad=True)
    dx = input_grad_hashed(dy, hw, 0.75, M, K, N, H, R, BK, BN, _lib.HASH_TWO_LEVEL)
    dhw, db = weight_grad_hashed(x, dy, 0.75, M, K, N, H, R, BK, BN, out=outs[1], accumulate=accumulate, with_bias_grad=True)
    return both, (dx, dhw, db)


@pytest.mark.parametrize("shape,dtype", PAIRS, ids=str)
def test_same_bits_as_apart(shape, dtype):
    both, apart = _both_and_apart(shape, dtype)
    for name, a, b in zip(("dx", "dhw", "dbias"), both, apart):
        assert torch.isfinite(b.float()).all() and torch.equal(a, b), name


@pytest.mark.parametrize("shape,dtype", PAIRS, ids=str)
def test_same_fp32_bits_of_the_bias_gradient(shape, dtype):
    # (in fp32: rounded to 16 bits, sums in another order hardly ever differ)
    from rzlinear_amd import _lib
    M, K, N, H, BK, BN = shape
    print(shape, dtype, flush=True)
    (x, hw, dy), _ = make_inputs(M, K, N, H, dtype, seed=M + N)
    R = _lib.hash_constants(*[R1024[7 - i] for i in range(8)])
    lib, code, flags, stream = _lib.load(), _lib.dtype_code(x), _lib.WG_DHW_F32 | _lib.WG_DBIAS_F32, _lib.require_gpu(x, hw, dy)
    sizes = (M, K, N, H, BK, BN)
    ws = [_lib.workspace(n + 256, x.device) for n in (lib.rz_input_grad_hashed_workspace_bytes(*sizes, code, None),
                                                      lib.rz_weight_grad_hashed_workspace_bytes(*sizes, code, flags, 1, None))]
    dx, dhw = torch.empty_like(x), torch.empty((H,), device=x.device)
    together, apart = (torch.full((N,), float("nan"), device=x.device) for _ in range(2))
    _lib.check(lib.rz_linear_backward_hashed(
        x.data_ptr(), dy.data_ptr(), hw.data_ptr(), dx.data_ptr(), dhw.data_ptr(), together.data_ptr(), ws[0].data_ptr(), ws[0].numel(),
        ws[1].data_ptr(), ws[1].numel(), None, 0, *sizes, R, _lib.HASH_TWO_LEVEL, 0.75, K, N, K, code, flags, None, stream))
    _lib.check(lib.rz_weight_grad_hashed(
        x.data_ptr(), dy.data_ptr(), dhw.data_ptr(), apart.data_ptr(), ws[1].data_ptr(), ws[1].numel(), *sizes, R, _lib.HASH_TWO_LEVEL, 0.75,
        K, N, code, flags, None, stream))
    assert torch.isfinite(apart).all() and torch.equal(together, apart)


@pytest.mark.parametrize("shape,dtype", [PAIRS[3], PAIRS[5], PAIRS[14], PAIRS[17]], ids=str)
def test_accumulating_into_an_fp32_gradient(shape, dtype):
    both, apart = _both_and_apart(shape, dtype, dhw_dtype=FP32, accumulate=True)
    for a, b in zip(both, apart):
        assert torch.equal(a, b)


# Windows of dHW whose operands' fragments are made beside the input-grad: its 32 x 128, 64, 128 and 256 x 128 tiles, complete and ragged
FRAGMENTS = [
    ((32, 10240, 10240, 6553600, 32, 64), BF16),
    ((19, 10232, 10240, 6553600, 32, 64), FP16),
    ((61, 3000, 4008, 750000, 32, 64), FP16),
    ((128, 4096, 4096, 700000, 32, 64), BF16),
    ((128, 10240, 10240, 6553600, 32, 64), BF16),
    ((96, 5000, 7000, 2200000, 32, 64), BF16),
    ((150, 3000, 5000, 937500, 32, 64), FP16),
    ((224, 10240, 10240, 6553600, 32, 64), BF16),
    ((61, 3001, 4008, 750000, 32, 64), FP16),      # rows that are not whole pieces: by a kernel of their own
]


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("shape,dtype", FRAGMENTS, ids=str)
def test_fragments_beside_the_input_grad(shape, dtype, accumulate):
    both, apart = _both_and_apart(shape, dtype, accumulate=accumulate)
    for name, a, b in zip(("dx", "dhw", "dbias"), both, apart):
        assert torch.isfinite(b.float()).all() and torch.equal(a, b), name


def test_an_input_grad_in_runs_goes_in_whole_tiles():
    # M = 1024, K = N = 10240: by itself in runs, whose parts are added up in fp32; the whole tiles' sums are in one piece.  Two
    # correctly accumulated results, each rounded once: they differ by an fp32 sum's error (10240 terms, < 1e-5 of the largest value)
    # and one unit in the last place of a bf16 value.
    shape = (1024, 10240, 10240, 6553600, 32, 64)
    both, apart = _both_and_apart(shape, BF16)
    assert torch.equal(both[1], apart[1]) and torch.equal(both[2], apart[2])
    a, b = both[0].double(), apart[0].double()
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-5 * b.abs().max()).all()


@pytest.mark.parametrize("shape,dtype", [PAIRS[0], PAIRS[3], PAIRS[5], PAIRS[11], FRAGMENTS[0], FRAGMENTS[5]], ids=str)
def test_captured_backward(shape, dtype):
    # (a cut input-grad has no counters under capture: a second kernel behind the common launch, the same bits)
    from rzlinear_amd import RzLinear
    M, K, N, H, BK, BN = shape
    (x, hw, dy), _ = make_inputs(M, K, N, H, dtype, seed=3)
    layer = RzLinear(K, N, hashed_weight=torch.nn.Parameter(hw), seed=1024, dtype=dtype, block_size_k=BK, block_size_n=BN).cuda()
    x.requires_grad_(True)

    def backward():
        return torch.autograd.grad(layer(x), (x, layer._hashed_weight, layer._bias), dy)

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        backward()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = backward()
    for i in range(3):
        with torch.no_grad():
            x.copy_(make_inputs(M, K, N, H, dtype, seed=20 + i)[0][0])
        graph.replay()
        eager = backward()
        torch.cuda.synchronize()
        for a, b in zip(captured, eager):
            assert torch.equal(a, b)
