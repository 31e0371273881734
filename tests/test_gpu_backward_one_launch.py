"""Input-grad and weight-grad of a backward pass in one launch, against the two by themselves."""
import pytest
import torch

from helpers import SEED_CONSTANTS, make_inputs

pytestmark = pytest.mark.gpu

R1024 = SEED_CONSTANTS[1024]
BF16, FP16, FP32 = torch.bfloat16, torch.float16, torch.float32

# (M, K, N, H, BK, BN), dtype, the form that it takes (_lib.backward_query): every pair of kernels, complete and ragged, at its smallest and around a
# round of workgroups
APART = (None, False, 0)
PAIRS = [
    ((96, 320, 192, 8192, 32, 64), BF16, ("64+64", False, 4)),        # a ragged M
    ((1, 8, 9, 4096, 32, 64), BF16, APART),                           # rows that are not whole pieces
    ((263, 286, 163, 8192, 64, 64), FP16, ("64+64", False, 4)),       # three slices of M
    ((128, 1024, 1024, 65536, 32, 64), BF16, ("64+64", True, 2)),     # more workgroups than compute units; stored tiles
    ((128, 256, 256, 16384, 32, 64), FP16, ("64+128", True)),
    ((160, 320, 1536, 8192, 64, 64), BF16, ("64+128", False)),        # the input-grad cut
    ((337, 885, 1501, 13268, 32, 64), FP16, ("64+128", False)),       # three slices of M
    ((62, 1001, 1203, 65536, 32, 64), BF16, ("64+128", False)),       # stored tiles
    ((1024, 1024, 1024, 65536, 64, 64), FP32, ("64+64", True, 2)),
    ((300, 135, 961, 16384, 64, 64), FP32, ("64+64", False, 2)),      # both cut
    ((61, 8384, 448, 234752, 64, 64), FP32, APART),                   # many more workgroups than compute units, of a short loop
    ((2048, 1024, 1024, 20000, 64, 64), BF16, ("128+128", True)),
    ((3738, 679, 525, 8192, 64, 64), FP16, ("128+128", False)),       # eight slices (whole ones to an XCD)
    ((3072, 2048, 2048, 31340, 64, 64), BF16, ("256x128+256", True)),
    ((3001, 2047, 1531, 31340, 64, 64), FP16, ("256x128+256", False)),   # nothing a multiple of anything
    ((6144, 2048, 1536, 31340, 64, 64), BF16, APART),
    ((6011, 2050, 1530, 31340, 64, 64), BF16, APART),
    ((14456, 556, 802, 27869, 64, 64), BF16, ("256+128", False)),     # seven slices
    ((5056, 2304, 256, 36864, 64, 64), FP16, APART),
    ((4288, 2304, 4544, 654336, 64, 64), BF16, APART),                # no compute unit would be done sooner
    ((513, 6143, 6145, 300000, 64, 64), BF16, APART),
    ((128, 2048, 4096, 400000, 32, 64), BF16, APART),                 # windows of dHW
    ((16384, 512, 1024, 5243, 64, 64), BF16, APART),                  # whole rounds of both
    ((5001, 1030, 1021, 20000, 64, 64), FP16, ("256x128+128", False)),
    ((2048, 4096, 1024, 262144, 32, 64), BF16, ("256x128+128", True)),   # stored tiles
    ((128, 192, 128, 8192, 32, 64), BF16, ("64+64", True, 4)),
    ((7, 4387, 161, 8192, 32, 64), FP16, ("64+64", False, 2)),
    ((320, 14336, 768, 110100, 32, 64), BF16, ("256x128+256", False)),
    ((768, 11008, 512, 8192, 32, 64), FP16, ("256+256", True)),
    ((1056, 7616, 704, 8192, 32, 64), BF16, ("256+256", False)),
    ((3584, 2816, 384, 16384, 64, 64), BF16, ("256+128", True)),
    ((3328, 1280, 256, 20480, 64, 64), FP16, ("256x128+128", True)),
    ((50, 1920, 192, 23040, 64, 64), FP32, ("64+64", False, 2)),      # fp32 images of dHW; weight-grad by four wavefronts apart
    ((512, 512, 512, 65536, 64, 64), FP32, ("64+64", True, 2)),
    ((1984, 320, 3008, 60160, 64, 64), FP32, APART),                  # as many rounds together as apart
    ((6688, 192, 12672, 24330, 64, 64), FP32, APART),                 # an image that takes the input-grad's neighbour
    ((9856, 192, 2688, 32256, 64, 64), BF16, APART),                  # ... the same in 16 bits
]
CODES = {FP32: 0, BF16: 1, FP16: 2}


def assert_form(shape, dtype, form):
    from rzlinear_amd import _lib
    q = _lib.backward_query(*shape, CODES[dtype])
    assert (q["pair"], q["full"], q["stages"])[:len(form)] == form, q


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


@pytest.mark.parametrize("shape,dtype,form", PAIRS, ids=str)
def test_same_bits_as_apart(shape, dtype, form):
    assert_form(shape, dtype, form)
    both, apart = _both_and_apart(shape, dtype)
    for name, a, b in zip(("dx", "dhw", "dbias"), both, apart):
        assert torch.isfinite(b.float()).all() and torch.equal(a, b), name


@pytest.mark.parametrize("shape,dtype", [p[:2] for p in PAIRS], ids=str)
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


@pytest.mark.parametrize("shape,dtype", [PAIRS[i][:2] for i in (3, 5, 14, 17)], ids=str)
def test_accumulating_into_an_fp32_gradient(shape, dtype):
    both, apart = _both_and_apart(shape, dtype, dhw_dtype=FP32, accumulate=True)
    for a, b in zip(both, apart):
        assert torch.equal(a, b)


# Windows of dHW whose operands' fragments are made beside the input-grad: by rows of its C tile (32, 64, 128, 256 x 128), complete and ragged
FRAGMENTS = [
    ((32, 10240, 10240, 6553600, 32, 64), BF16, (32, True)),
    ((19, 10232, 10240, 6553600, 32, 64), FP16, (32, False)),
    ((61, 3000, 4008, 750000, 32, 64), FP16, None),               # none are made
    ((128, 4096, 4096, 700000, 32, 64), BF16, "own"),             # no compute unit is idle: by a kernel of their own
    ((128, 10240, 10240, 6553600, 32, 64), BF16, (128, True)),
    ((96, 5000, 7000, 2200000, 32, 64), BF16, (128, False)),
    ((150, 3000, 5000, 937500, 32, 64), FP16, (128, False)),
    ((224, 10240, 10240, 6553600, 32, 64), BF16, (256, False)),
    ((61, 3001, 4008, 750000, 32, 64), FP16, "own"),              # rows that are not whole pieces
    ((256, 3328, 2048, 425984, 32, 64), BF16, (64, True)),
    ((5, 1344, 12736, 171171, 64, 64), FP16, (64, False)),
    ((256, 5888, 5120, 1884160, 64, 64), BF16, (256, True)),
    ((32, 10240, 10240, 6553600, 32, 64), FP32, "own"),
]


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("shape,dtype,beside", FRAGMENTS, ids=str)
def test_fragments_beside_the_input_grad(shape, dtype, beside, accumulate):
    from rzlinear_amd import _lib
    groups, *form = _lib.backward_query(*shape, CODES[dtype])["fragments"]
    assert (None if groups == 0 else "own" if groups < 0 else tuple(form)) == beside
    both, apart = _both_and_apart(shape, dtype, accumulate=accumulate)
    for name, a, b in zip(("dx", "dhw", "dbias"), both, apart):
        assert torch.isfinite(b.float()).all() and torch.equal(a, b), name


@pytest.mark.parametrize("shape,dtype,full", [
    ((1024, 10240, 10240, 6553600, 32, 64), BF16, True), ((2560, 3328, 7168, 23855, 32, 64), FP16, True), ((1044, 16012, 2555, 40910, 64, 64), FP16, False),
], ids=str)
def test_an_input_grad_in_runs_goes_in_whole_tiles(shape, dtype, full):
    # By itself in runs, whose parts are added up in fp32; the whole tiles' sums are in one piece.  Two correctly accumulated results,
    # each rounded once: they differ by an fp32 sum's error (at most 10240 terms, < 1e-5 of the largest value) and one unit in the last
    # place of the 16-bit value.
    from rzlinear_amd import _lib
    assert_form(shape, dtype, ("256+256", full))
    assert _lib.backward_query(*shape, CODES[dtype])["input_grad"] == "whole"
    both, apart = _both_and_apart(shape, dtype)
    assert torch.equal(both[1], apart[1]) and torch.equal(both[2], apart[2])
    a, b = both[0].double(), apart[0].double()
    assert ((a - b).abs() <= (2.0 ** -7 if dtype == BF16 else 2.0 ** -10) * b.abs() + 1e-5 * b.abs().max()).all()


@pytest.mark.parametrize("shape,dtype,with_bias", [
    ((1024, 10240, 10240, 6553600, 32, 64), BF16, False), ((3469, 5867, 14924, 5472443, 32, 64), FP16, False),
    ((5031, 4002, 6371, 1593546, 32, 64), BF16, False),
    ((15870, 1471, 4555, 418776, 64, 64), BF16, True), ((27152, 604, 3009, 113589, 64, 64), FP16, True),
], ids=str)
def test_an_input_grad_apart_stays_in_runs(shape, dtype, with_bias):
    # where the two ops share no launch (none does without a bias gradient) dX is the separate call's, by the same plan
    from rzlinear_amd import _lib
    from rzlinear_amd.impl.RzLinearBackward import backward_hashed, input_grad_hashed
    q = _lib.backward_query(*shape, CODES[dtype], with_dbias=with_bias)
    assert (q["pair"], q["input_grad"]) == (None, "runs")
    M, K, N, H, BK, BN = shape
    print(shape, dtype, flush=True)
    (x, hw, dy), _ = make_inputs(M, K, N, H, dtype, seed=5)
    R = _lib.hash_constants(*[R1024[7 - i] for i in range(8)])
    dx = backward_hashed(x, hw, dy, 0.75, M, K, N, H, R, BK, BN, with_bias_grad=with_bias)[0]
    assert torch.equal(dx, input_grad_hashed(dy, hw, 0.75, M, K, N, H, R, BK, BN, _lib.HASH_TWO_LEVEL))


@pytest.mark.parametrize("shape,dtype", [p[:2] for p in (PAIRS[0], PAIRS[3], PAIRS[5], PAIRS[11], FRAGMENTS[0], FRAGMENTS[5])], ids=str)
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
