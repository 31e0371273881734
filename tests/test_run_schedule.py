"""16-bit forward / input-grad in runs of equal length: the deal of a plan's tiles and R steps to the workgroups, restated
from the kernel's (rzlinear_amd/csrc/rz_gemm.h, run_all), covers every step of every tile once, and no tile has more parts than planes."""
import random

import pytest

from rzlinear_amd import _lib

CUS = 256


def deal(tiles, steps, groups, rounds, L):
    """[(tile, part, parts of the tile, first step, steps)] of every workgroup."""
    first = rounds * groups
    rest = tiles - first
    F = steps // L
    r = steps - F * L
    full = rest * F

    def parts(t):
        return F if r == 0 else F + 1 + (1 if ((t + 1) * r - 1) // L * L > t * r else 0)

    out = []
    for g in range(groups):
        items = [(k * groups + g, 0, 1, 0, steps) for k in range(rounds)]
        if g < full:
            items.append((first + g % rest, g // rest, parts(g % rest), g // rest * L, L))
        else:
            at = (g - full) * L
            end = min(at + L, rest * r)
            while at < end:
                t, o = at // r, at % r
                n = min(r - o, end - at)
                items.append((first + t, F + (1 if o else 0), parts(t), F * L + o, n))
                at += n
        out.append(items)
    return out


def check(op, M, K, N, code):
    q = _lib.plan_query(op, M, K, N, 1 << 20, 64, 64, code)
    if q["mode"] != "split" or q["windows"] == 0:
        return False
    J, R = (N, K) if op == 0 else (K, N)
    tiles, steps = -(-M // 256) * -(-J // q["tile"]), -(-R // 64)
    rounds = tiles // CUS
    assert q["workgroups"] <= CUS and (rounds == 0 or q["workgroups"] == CUS)
    assert 2 <= q["slices"] <= 4 and q["windows"] < steps
    seen = {}
    for items in deal(tiles, steps, q["workgroups"], rounds, q["windows"]):
        assert sum(n for *_, n in items) <= rounds * steps + q["windows"]
        for tile, part, parts, s0, n in items:
            assert n > 0
            seen.setdefault(tile, []).append((part, parts, s0, n))
    assert sorted(seen) == list(range(tiles))
    most = 1
    for items in seen.values():
        items.sort()
        at = 0
        for i, (part, parts, s0, n) in enumerate(items):
            assert (part, parts, s0) == (i, len(items), at)   # (in the order of R, none missing)
            at += n
        assert at == steps
        most = max(most, len(items))
    assert most <= q["slices"]   # (a plane for every part)
    return True


@pytest.mark.parametrize("op,shape", [
    (0, (1024, 10240, 10240)), (1, (1024, 10240, 10240)), (0, (3328, 7680, 10624)), (1, (5031, 4002, 6371)), (0, (8864, 9146, 934)),
    (1, (3744, 9622, 9701)), (0, (1286, 9678, 16359)), (1, (2163, 9063, 11174)), (0, (6072, 14309, 1473)),
], ids=str)
def test_a_plan_in_runs_covers_every_step_once(op, shape):
    assert check(op, *shape, _lib.RZ_BF16)   # (and these are dealt out in runs: 5 to 25 % faster, measured)


def test_drawn_plans_in_runs_cover_every_step_once():
    rng = random.Random(11)
    taken = 0
    for _ in range(3000):
        shape = (rng.randint(65, 12000), rng.randint(512, 16384), rng.randint(512, 16384))
        taken += check(rng.randint(0, 1), *shape, rng.choice([_lib.RZ_BF16, _lib.RZ_F16]))
    assert taken > 30


@pytest.mark.parametrize("tuning", [dict(tile=256), dict(tile=128), dict(split=-1), dict(split=3), dict(stages=1), dict(clamp=-1)], ids=str)
def test_an_override_is_never_dealt_out_in_runs(tuning):
    with _lib.tuning(**tuning):
        assert _lib.plan_query(0, 1024, 10240, 10240, 6553600, 32, 64, _lib.RZ_BF16)["windows"] == 0


def test_the_second_kernel_gets_the_plan_of_the_first():
    """finish=-1 promises the same bits: the same tile, slices and runs, whoever adds them up."""
    rng = random.Random(13)
    cut = runs = 0
    for _ in range(3000):
        code = rng.choice([_lib.RZ_F32, _lib.RZ_BF16, _lib.RZ_F16])
        call = (rng.randint(0, 1), int(2 ** rng.uniform(0, 13)), rng.randint(128, 12000), rng.randint(128, 12000), 1 << 20, 64, 64, code)
        q = _lib.plan_query(*call)
        with _lib.tuning(finish=-1):
            q2 = _lib.plan_query(*call)
        assert q2["shares"] == 0
        assert {**q, "shares": 0} == q2, call
        cut += q["mode"] == "split"
        runs += q["mode"] == "split" and q["windows"] > 0
    assert cut > 500 and runs > 10


@pytest.mark.parametrize("slices", [dict(tile=256, split=3), dict(tile=128, split=2)], ids=str)
def test_a_cut_that_is_asked_for_is_the_same_with_a_second_kernel(slices):
    for code in (_lib.RZ_F32, _lib.RZ_BF16):
        with _lib.tuning(**slices):
            q = _lib.plan_query(0, 512, 8192, 1024, 1 << 20, 64, 64, code)
        with _lib.tuning(finish=-1, **slices):
            assert _lib.plan_query(0, 512, 8192, 1024, 1 << 20, 64, 64, code) == {**q, "shares": 0}


@pytest.mark.parametrize("op,shape", [(1, (653, 11012, 6869)), (0, (317, 16216, 10935)), (1, (420, 11279, 13216)), (1, (578, 11175, 9098))], ids=str)
def test_planes_of_runs_stay_in_proportion_to_the_call(op, shape):
    """Planes of more than twice what the call reads and writes are not asked for where slices do without (these would have 90 to 104 MB
    beside 17 to 24 MB)."""
    lib = _lib.load()
    M, K, N = shape
    assert _lib.plan_query(op, *shape, 200000, 64, 64, _lib.RZ_BF16)["windows"] == 0
    need = lib.rz_forward_hashed_workspace_bytes if op == 0 else lib.rz_input_grad_hashed_workspace_bytes
    assert need(*shape, 200000, 64, 64, _lib.RZ_BF16, None) <= 4 * M * (K + N)


def test_a_backward_pass_takes_an_input_grad_out_of_its_runs_only_for_a_common_launch():
    lib, rng = _lib.load(), random.Random(17)
    runs = whole = 0
    for _ in range(6000):
        code = rng.choice([_lib.RZ_BF16, _lib.RZ_F16])
        call = (rng.randint(65, 16000), rng.randint(512, 16000), rng.randint(512, 16000), 300000, 64, 64, code)
        alone = _lib.plan_query(1, *call)
        in_runs = alone["mode"] == "split" and alone["windows"] > 0
        for with_dbias in (False, True):
            q = _lib.backward_query(*call, with_dbias=with_dbias)
            assert (q["input_grad"] == "plain") == (not in_runs), call
            assert (q["input_grad"] == "whole") == (in_runs and q["pair"] is not None), call
            assert with_dbias or q["pair"] is None
            # (planes are asked for where they are used: whole tiles need none)
            need = lib.rz_input_grad_hashed_workspace_bytes(*call, None)
            assert lib.rz_linear_backward_hashed_dx_workspace_bytes(*call, _lib.PLAN_WITH_LAYER_PLAN, int(with_dbias), None) == (
                0 if q["input_grad"] == "whole" else need), call
            runs += q["input_grad"] == "runs"
            whole += q["input_grad"] == "whole"
    assert runs > 50 and whole > 20
