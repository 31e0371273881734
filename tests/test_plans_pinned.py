"""The plan the library takes for every baseline configuration and for the reference's benchmark grid,
pinned: C tile, slices of the contracted dimension and the way the weight gradient reaches dHW, for
forward / input-grad / weight-grad.  The planner (rzlinear_amd/csrc/rz_launch.h) is a model fitted to
measurements; refitting it for one shape must not silently move another.  A deliberate change of plan
updates this table — together with the measurement that justifies it."""
import pytest

from rzlinear_amd import _lib

from helpers import stored_tile_bytes

F32, BF16, F16 = _lib.RZ_F32, _lib.RZ_BF16, _lib.RZ_F16

# name: ((M, K, N, H, BLOCK_K, BLOCK_N, dtype), [(tile, slices, mode) for forward, input-grad, weight-grad])
# (tile 32 = the 32 x 64 C tile of the fp32 kernels; 0 = the window kernel, which has no C tile)
PLANS = {
    "cpu_ref_1024 fp32": ((1024, 1024, 1024, 65536, 64, 64, F32), [(64, 1, "store"), (64, 1, "store"), (64, 1, "fold")]),
    "square1024 fp32": ((1024, 1024, 1024, 16384, 64, 64, F32), [(64, 1, "store"), (64, 1, "store"), (128, 4, "lds_image")]),
    "square1024 bf16": ((1024, 1024, 1024, 16384, 64, 64, BF16), [(64, 1, "store"), (64, 1, "store"), (128, 4, "lds_image")]),
    "square2048 fp32": ((2048, 2048, 2048, 16384, 64, 64, F32), [(128, 1, "store"), (128, 1, "store"), (256, 4, "lds_image")]),
    "square2048 bf16": ((2048, 2048, 2048, 16384, 64, 64, BF16), [(128, 1, "store"), (128, 1, "store"), (128, 1, "lds_image")]),
    "square4096 fp32": ((4096, 4096, 4096, 16778, 64, 64, F32), [(256, 1, "store"), (256, 1, "store"), (256, 1, "lds_image")]),
    "square4096 bf16": ((4096, 4096, 4096, 16778, 64, 64, BF16), [(256, 1, "store"), (256, 1, "store"), (256, 1, "lds_image")]),
    "square4096 fp16": ((4096, 4096, 4096, 16778, 64, 64, F16), [(256, 1, "store"), (256, 1, "store"), (256, 1, "lds_image")]),
    "rec_mlp bf16": ((16384, 512, 1024, 5243, 64, 64, BF16), [(256, 1, "store"), (128, 1, "store"), (128, 8, "lds_image")]),
    "ffn bf16": ((8192, 4096, 16384, 67109, 64, 64, BF16), [(256, 1, "store"), (256, 1, "store"), (256, 1, "fold")]),
    "collision fp32": ((32768, 2048, 2048, 32768, 64, 64, F32), [(256, 1, "store"), (256, 1, "store"), (256, 4, "lds_image")]),
    "grid_32_1024 fp32": ((32, 1024, 1024, 65536, 32, 64, F32), [(32, 6, "split"), (32, 6, "split"), (64, 1, "fold")]),
    "grid_32_1024 bf16": ((32, 1024, 1024, 65536, 32, 64, BF16), [(64, 1, "store"), (64, 1, "store"), (64, 1, "fold")]),
    "grid_32_10240 fp32": ((32, 10240, 10240, 6553600, 32, 64, F32), [(32, 3, "split"), (32, 3, "split"), (0, 1, "window")]),
    "grid_32_10240 bf16": ((32, 10240, 10240, 6553600, 32, 64, BF16), [(128, 3, "split"), (128, 3, "split"), (0, 1, "window")]),
    "grid_128_1024 fp32": ((128, 1024, 1024, 65536, 32, 64, F32), [(64, 6, "split"), (64, 6, "split"), (64, 1, "fold")]),
    "grid_128_1024 bf16": ((128, 1024, 1024, 65536, 32, 64, BF16), [(64, 1, "store"), (64, 1, "store"), (64, 1, "fold")]),
    "grid_128_10240 fp32": ((128, 10240, 10240, 6553600, 32, 64, F32), [(128, 3, "split"), (128, 3, "split"), (0, 1, "window")]),
    "grid_128_10240 bf16": ((128, 10240, 10240, 6553600, 32, 64, BF16), [(128, 3, "split"), (128, 3, "split"), (0, 1, "window")]),
    "grid_1024_1024 fp32": ((1024, 1024, 1024, 65536, 32, 64, F32), [(64, 1, "store"), (64, 1, "store"), (64, 1, "fold")]),
    "grid_1024_1024 bf16": ((1024, 1024, 1024, 65536, 32, 64, BF16), [(64, 1, "store"), (64, 1, "store"), (64, 1, "fold")]),
    "grid_1024_10240 fp32": ((1024, 10240, 10240, 6553600, 32, 64, F32), [(64, 1, "store"), (64, 1, "store"), (128, 1, "fold")]),
    "grid_1024_10240 bf16": ((1024, 10240, 10240, 6553600, 32, 64, BF16), [(256, 3, "split"), (256, 3, "split"), (256, 1, "fold")]),
}


@pytest.mark.parametrize("name", sorted(PLANS))
def test_plan_of_a_baseline_configuration_is_what_was_measured(name):
    (M, K, N, H, BK, BN, code), want = PLANS[name]
    got = []
    for op in (0, 1, 2):
        q = _lib.plan_query(op, M, K, N, H, BK, BN, code, planned=True)   # (as the launchers ask: with a layer plan)
        got.append((q["tile"], q["slices"], q["mode"]))
    assert got == want


def test_no_baseline_configuration_takes_the_atomic_scatter():
    """Global atomics — the one path that leaves the order of the additions open — serve none of the
    configurations above; the library keeps them for hashed tiles too large to fold (more than 16384
    elements) and for many small tiles under a batch of a few rows, where they are faster."""
    assert all(mode != "atomics" for _, plan in PLANS.values() for _, _, mode in plan)
    assert _lib.plan_query(2, 128, 2048, 1024, 1 << 20, 256, 128, BF16)["mode"] == "atomics"


@pytest.mark.parametrize("shape,code,bytes_of_each", [
    ((8192, 4096, 16384, 67109, 64, 64), BF16, 2), ((1024, 10240, 10240, 6553600, 32, 64), F16, 2),
    ((1024, 10240, 10240, 6553600, 32, 64), F32, 4), ((1024, 1024, 1024, 65536, 64, 64), F32, 4),
    ((96, 10240, 10240, 67109, 64, 64), BF16, 2),        # the 128 tile of a short batch, one slice
    ((20442, 6647, 591, 245486, 64, 64), BF16, 4),       # cut further than the plan by rate
    ((14592, 8448, 448, 236544, 64, 64), F16, 4),
    ((11552, 5632, 768, 270336, 64, 64), BF16, 4),       # added into an fp32 image by that plan
    ((4846, 519, 1167, 41000, 64, 64), BF16, 4), ((2322, 536, 3404, 91227, 64, 64), BF16, 4),
    ((1963, 1344, 3328, 279552, 64, 64), BF16, 4), ((1948, 2184, 1810, 197652, 64, 64), F16, 4),
], ids=str)
def test_width_of_the_stored_tiles(shape, code, bytes_of_each):
    """Tiles of a 16-bit layer are stored in its dtype where a stored value is a sum over M cut no further than by the plan by
    rate, and in fp32 where it is a partial sum of a further cut or would otherwise be added in fp32."""
    for planned in (False, True):
        assert stored_tile_bytes(shape, code, planned) == bytes_of_each
        assert stored_tile_bytes(shape, code, planned, _lib.WG_DHW_F32) == 4   # (an fp32 dHW never has them rounded)


@pytest.mark.parametrize("shape", [
    (96, 11712, 13760, 1611571, 32, 64), (93, 4672, 9344, 1309655, 32, 64), (127, 10560, 3904, 1236787, 32, 64),
    (158, 3520, 10368, 1094860, 32, 64), (61, 8192, 4608, 1282982, 32, 64), (91, 9088, 3648, 1170819, 64, 64),
    (72, 3648, 10048, 1249083, 64, 64),
], ids=str)
@pytest.mark.parametrize("code", [BF16, F16])
def test_a_short_batch_keeps_the_window_kernels_fp32_sums(shape, code):
    """The 128 tile that a short batch takes makes its fold cheaper; tiles stored in 16 bits must not win a call from the window
    kernel, which adds in fp32, by that.  (Each of these lies where the two tiles' prices fall on either side of the window kernel's.)"""
    assert _lib.plan_query(2, *shape, code, planned=True)["mode"] == "window"


@pytest.mark.parametrize("shape,mode", [
    ((1085, 4416, 1024, 282624, 64, 64), "atomics"), ((1124, 5844, 819, 299139, 32, 64), "atomics"), ((927, 393, 11100, 272643, 32, 64), "atomics"),
    ((1056, 1280, 4144, 265216, 64, 64), "atomics"), ((1655, 320, 16000, 320000, 32, 64), "atomics"),
    ((1963, 1344, 3328, 279552, 64, 64), "fold"), ((4070, 8148, 858, 436936, 32, 64), "fold"), ((11535, 5760, 768, 276480, 64, 64), "fold"),
], ids=str)
def test_slices_are_stored_in_place_of_atomics_only_where_that_pays_for_the_fold_kernel(shape, mode):
    """Measured (bf16): the first five are 3 to 12 % slower with stored slices, the others 3 to 60 % faster."""
    assert _lib.plan_query(2, *shape, BF16, planned=True)["mode"] == mode


@pytest.mark.parametrize("shape,tile", [
    ((36, 1863, 1524, 33541, 32, 64), 256), ((50, 704, 8704, 17299, 32, 64), 256), ((14, 2816, 1216, 33208, 32, 64), 256),
    ((23, 497, 8162, 29777, 32, 64), 256), ((11, 5952, 512, 29736, 64, 64), 256),
    ((19, 5120, 704, 8192, 32, 64), 128), ((18, 1368, 1112, 33794, 64, 64), 128), ((41, 8960, 704, 8192, 32, 64), 128),
    ((96, 8768, 2496, 8233, 32, 64), 128),
], ids=str)
def test_a_batch_below_the_fit_pays_for_the_images_of_the_128_tile(shape, tile):
    """Measured (bf16): the first five are 5 to 9 % slower with the 128 tile, the next three 12 to 60 % faster."""
    q = _lib.plan_query(2, *shape, BF16, planned=True)
    assert (q["mode"], q["tile"]) == ("lds_image", tile)


@pytest.mark.parametrize("op,shape,plan", [
    (0, (192, 3712, 1152, 267264, 32, 64), (64, 4)), (0, (640, 3072, 384, 16384, 64, 64), (64, 4)), (0, (101, 2233, 1012, 16384, 64, 64), (64, 4)),
    (1, (352, 896, 3328, 186368, 32, 64), (64, 3)), (1, (96, 1792, 2880, 322560, 64, 64), (64, 4)), (1, (274, 649, 3240, 131422, 64, 64), (64, 4)),
    (1, (224, 1024, 7296, 466944, 64, 64), (64, 4)), (0, (2368, 256, 13056, 33423, 32, 64), (256, 1)), (0, (12320, 256, 6080, 97280, 32, 64), (256, 1)),
], ids=str)
@pytest.mark.parametrize("code", [BF16, F16])
def test_16_bit_plans_that_a_second_kernel_or_ragged_tiles_make_slower(op, shape, plan, code):
    """Measured (bf16): other cuts, with a second kernel, or none, or the 128 tile for a few steps are 10 to 45 % slower here."""
    q = _lib.plan_query(op, *shape, code)
    assert (q["tile"], q["slices"]) == plan


@pytest.mark.parametrize("shape,code,mode", [
    ((2258, 14448, 12316, 4274303, 256, 128), F16, "atomics"), ((3090, 8935, 16125, 24837666, 256, 128), BF16, "atomics"),
    ((1735, 3163, 3873, 4012942, 256, 128), F16, "atomics"), ((13, 15569, 3913, 65536, 256, 128), F16, "atomics"),
    ((15, 2659, 3729, 65536, 256, 128), F16, "atomics"), ((12, 14806, 2030, 257201, 128, 128), F32, "fold"),
    ((751, 1861, 1542, 667316, 128, 64), BF16, "atomics"),
    ((128, 10240, 10240, 6553600, 32, 64), BF16, "window"), ((16, 2048, 8192, 1048576, 64, 64), BF16, "window"),
    ((10, 10240, 11648, 3028101, 128, 32), F32, "window"), ((64, 4096, 4096, 1048576, 128, 128), BF16, "window"),
], ids=str)
def test_windows_only_where_they_are_faster_whatever_the_hashed_tile(shape, code, mode):
    """Measured: the first seven take 1.4 to 5.2 times as long by windows, the others 0.4 to 0.9 times."""
    assert _lib.plan_query(2, *shape, code, planned=True)["mode"] == mode
