"""The tile hash takes remainders by multiplication with a precomputed inverse; the offsets must be those of
integer division for every divisor and up to the largest intermediates that the library accepts."""
import pytest

from rzlinear_amd import _lib

INT32_MAX = 2 ** 31 - 1


@pytest.mark.parametrize("R0", [1, 2, 3, 45007, 46340])   # 46340: R0 * R0 - 1 just fits 31 bits
@pytest.mark.parametrize("span", [1, 2, 3, 255, 65536, 16777213, INT32_MAX - 16 * 16])
@pytest.mark.parametrize("levels", [1, 2])
def test_offsets_are_those_of_integer_division(R0, span, levels):
    BK = BN = 16
    K, N, H = 40 * BK, 33 * BN, span + BK * BN
    # the largest constants that keep tk * R3 + tn * R2 + R1 (tk up to 40, tn up to 33) inside int32, and small ones
    for R in ([R0, 7, 3, 5, 11, 2, 0, 13], [R0, INT32_MAX - 40 * 29000000 - 33 * 29000000, 29000000, 29000000,
                                            INT32_MAX - 40 * 28999999 - 33 * 28999999, 28999999, 0, 28999999]):
        got = _lib.tile_offsets(K, N, H, BK, BN, R, hash_levels=levels)
        for tk in (0, 1, 17, 39):
            for tn in (0, 1, 16, 32):
                hi = (tk * R[3] + tn * R[2] + R[1]) % R[0]
                lo = (tk * R[7] + tn * R[5] + R[4]) % R[0]
                want = (hi if levels == 1 else hi * R[0] + lo) % span
                assert int(got[tk, tn]) == want, (tk, tn)
