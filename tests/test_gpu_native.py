"""The native host path of the layer (csrc/rz_torch.cpp) against the Python Function: the same bits for every
layout it accepts, and the same refusals — what the Function does not support, or would notice, the native
node must not let through."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch
from torch.autograd import forward_ad

from helpers import SEED_CONSTANTS

pytestmark = pytest.mark.gpu

K, N, H, TILE = 192, 320, 9000, (32, 64)
R = torch.tensor(SEED_CONSTANTS[1024], dtype=torch.int32)


def _functions():
    from rzlinear_amd.RzLinearFunction import RzLinearFunction

    class InPython(RzLinearFunction):   # (a subclass never takes the native path)
        pass

    return RzLinearFunction, InPython


def _call(function, x, hw, bias=None, fuse=False):
    return function.apply(x, hw, R, N, 1, 0.5, *TILE, bias, fuse)


def _inputs(dtype=torch.float32, M=37):
    g = torch.Generator().manual_seed(3)
    x = torch.randn((M, K), generator=g).to(dtype).cuda()
    hw = ((torch.rand((H,), generator=g) * 2 - 1) / K ** 0.5).to(dtype).cuda()
    bias = torch.randn((N,), generator=g).to(dtype).cuda()
    dy = torch.randn((M, N), generator=g).to(dtype).cuda()
    return x, hw, bias, dy


def _transposed(t):
    return t.t().contiguous().t()


def _pitched(t):
    wide = torch.zeros((t.shape[0], t.shape[1] + 5), dtype=t.dtype, device=t.device)
    wide[:, 3:3 + t.shape[1]] = t
    return wide[:, 3:3 + t.shape[1]]


def _every_other_row(t):
    wide = torch.zeros((2 * t.shape[0], t.shape[1]), dtype=t.dtype, device=t.device)
    wide[::2] = t
    return wide[::2]


def _one_row_repeated(t):
    return t[:1].expand(t.shape[0], t.shape[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("layout", [lambda t: t, _transposed, _pitched, _every_other_row, _one_row_repeated],
                         ids=["plain", "transposed", "pitched", "every_other_row", "expanded"])
def test_same_bits_as_the_python_function(dtype, layout):
    x, hw, bias, dy = _inputs(dtype)
    got = []
    for function in _functions():
        xs, hs, bs = layout(x).detach().requires_grad_(), hw.clone().requires_grad_(), bias.clone().requires_grad_()
        y = _call(function, xs, hs, bs)
        got.append((y,) + torch.autograd.grad(y, (xs, hs, bs), layout(dy)))
    for a, b in zip(*got):
        assert a.shape == b.shape and a.dtype == b.dtype
        np.testing.assert_array_equal(a.detach().float().cpu().numpy(), b.detach().float().cpu().numpy())


@pytest.mark.parametrize("wanted", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (0, 1, 1)])
@pytest.mark.parametrize("changed", ["x", "hw", "R"])
def test_a_change_in_place_before_the_backward_is_refused(wanted, changed):
    for function in _functions():
        x, hw, bias, dy = _inputs()
        for t, w in zip((x, hw, bias), wanted):
            t.requires_grad_(bool(w))
        r = R.clone()
        y = function.apply(x, hw, r, N, 1, 0.5, *TILE, bias, False)
        with torch.no_grad():
            {"x": x, "hw": hw, "R": r}[changed].add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.backward(dy)


@pytest.mark.parametrize("wanted", [(1, 0, 0), (0, 1, 0), (0, 0, 1)])
def test_a_second_backward_needs_retain_graph(wanted):
    for function in _functions():
        x, hw, bias, dy = _inputs()
        for t, w in zip((x, hw, bias), wanted):
            t.requires_grad_(bool(w))
        y = _call(function, x, hw, bias)
        y.backward(dy, retain_graph=True)
        y.backward(dy)
        with pytest.raises(RuntimeError, match="second time"):
            y.backward(dy)


@pytest.mark.parametrize("master", [False, True], ids=["grad", "main_grad"])
@pytest.mark.parametrize("returned", ["x", "bias", "x and bias", "all leaves"])
def test_a_fused_weight_gradient_is_added_whichever_gradients_the_backward_returns(returned, master):
    buffers = []
    for function in _functions():
        x, hw, bias, dy = _inputs()
        for t in (x, hw, bias):
            t.requires_grad_()
        if master:
            hw.main_grad = torch.zeros(H, device="cuda")
        for _ in range(2):
            y = _call(function, x, hw, bias, fuse=True)
            if returned == "all leaves":
                y.backward(dy)
            else:
                torch.autograd.grad(y, [t for n, t in (("x", x), ("bias", bias)) if n in returned.split()], dy)
        buffers.append(hw.main_grad if master else hw.grad)
        assert not master or hw.grad is None
    assert buffers[0].abs().sum() > 0 and torch.equal(*buffers)


@pytest.mark.parametrize("with_input", [False, True], ids=["weight", "weight and input"])
def test_a_backward_that_fails_leaves_no_fresh_gradient_buffer(with_input):
    """The buffer that a fused weight gradient makes for a parameter without one holds nothing until the kernels have filled it: after
    an error (here a refused override) the next backward must not add to it."""
    from rzlinear_amd import _lib
    for function in _functions():
        x, hw, bias, dy = _inputs()
        y = _call(function, x.requires_grad_(with_input), hw.requires_grad_(), bias, fuse=True)
        with _lib.tuning(tile=77), pytest.raises(_lib.RzLinearError):
            y.backward(dy, retain_graph=True)
        assert hw.grad is None
        y.backward(dy, retain_graph=True)
        once = hw.grad.clone()
        with _lib.tuning(tile=77), pytest.raises(_lib.RzLinearError):   # (one that was there before stays as it is)
            y.backward(dy, retain_graph=True)
        assert torch.equal(hw.grad, once)
        y.backward(dy)
        assert torch.allclose(hw.grad, 2 * once)


def test_no_fused_gradient_for_a_weight_that_needs_none():
    for function in _functions():
        x, hw, bias, dy = _inputs()
        hw.main_grad = torch.zeros(H, device="cuda")
        _call(function, x.requires_grad_(), hw, bias, fuse=True).backward(dy)
        assert hw.grad is None and not hw.main_grad.any()


@pytest.mark.parametrize("with_bias", [False, True])
def test_the_node_has_an_edge_and_a_gradient_for_every_tensor(with_bias):
    seen = []
    for function in _functions():
        x, hw, bias, dy = _inputs()
        for t in (x, hw, bias):
            t.requires_grad_()
        y = _call(function, x, hw, bias if with_bias else None)
        targets = [getattr(n, "variable", None) for n, _ in y.grad_fn.next_functions]
        assert [t is e for t, e in zip(targets, (x, hw, None, bias))] == [True] * (3 + with_bias)
        shapes = []
        y.grad_fn.register_hook(lambda ins, outs: shapes.append([None if g is None else tuple(g.shape) for g in ins + outs]))
        y.backward(dy)
        seen.append(shapes)
    assert seen[0] == seen[1] and len(seen[0]) == 1


def test_the_node_shows_what_it_has_saved():
    for function in _functions():
        x, hw, bias, dy = _inputs()
        y = _call(function, x, hw.requires_grad_(), bias)
        assert type(y.grad_fn).__name__ == y.grad_fn.name() == function.__name__ + "Backward"
        assert isinstance(y.grad_fn, torch.autograd.graph.Node)
        saved = y.grad_fn.saved_tensors
        assert type(saved) is tuple and [a is b for a, b in zip(saved, (x, hw, R))] == [True, True, True]
        y.backward(dy)
        with pytest.raises(RuntimeError, match="second time"):
            y.grad_fn.saved_tensors


def test_saved_tensor_hooks_see_what_the_function_saves():
    seen = []
    for function in _functions():
        x, hw, bias, dy = _inputs()
        hw.requires_grad_()
        shapes = []

        def pack(t):
            shapes.append(tuple(t.shape))
            return t.cpu()

        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t if t.dtype == torch.int32 else t.cuda()):
            y = _call(function, x, hw, bias)
        grad, = torch.autograd.grad(y, hw, dy)
        seen.append((shapes, grad.cpu()))
    assert seen[0][0] == seen[1][0]
    assert torch.equal(seen[0][1], seen[1][1])


@pytest.mark.parametrize("unpack", [lambda t: t.cpu(), lambda t: t.to(torch.int32 if t.dtype == torch.int32 else torch.float64),
                                    lambda t: t[:5]], ids=["cpu", "dtype", "shape"])
def test_what_a_hook_hands_back_is_checked_before_a_kernel_sees_it(unpack):
    function = _functions()[0]
    x, hw, bias, dy = _inputs()
    x.requires_grad_()
    hw.requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = _call(function, x, hw, bias)
    with pytest.raises((RuntimeError, TypeError, ValueError)):
        y.backward(dy)


_REFUSED = {   # name: (index of the argument of apply, what takes its place)
    "constants in two rows": (2, lambda t: t.view(2, 4)),
    "seven constants": (2, lambda t: t[:7]),
    "a negative constant": (2, lambda t: -t),
    "constants in a list": (2, lambda t: t.tolist()),
    "a batch of matrices": (0, lambda t: t[None]),
    "a vector": (0, lambda t: t[0]),
    "another input dtype": (0, lambda t: t.half()),
    "input on the host": (0, lambda t: t.cpu()),
    "a two-dimensional weight": (1, lambda t: t.view(9, -1)),
    "a weight of one tile": (1, lambda t: t[:TILE[0] * TILE[1]]),
    "weight on the host": (1, lambda t: t.cpu()),
    "a short bias": (8, lambda t: t[:-1]),
    "another bias dtype": (8, lambda t: t.half()),
    "no output columns": (3, lambda n: 0),
    "a fraction of columns": (3, lambda n: float(n)),
    "a tile of 24 rows": (6, lambda n: 24),
    "no scale": (5, lambda f: None),
}


@pytest.mark.parametrize("name", _REFUSED)
def test_what_the_function_refuses_is_refused_alike(name):
    at, change = _REFUSED[name]
    kinds = []
    for function in _functions():
        x, hw, bias, _ = _inputs()
        args = [x, hw, R, N, 1, 0.5, *TILE, bias, False]
        args[at] = change(args[at])
        with pytest.raises(Exception) as refused:
            function.apply(*args)
        kinds.append(refused.type)
    assert kinds[0] is kinds[1]


def test_forward_mode_is_refused():
    for function in _functions():
        for which in range(3):
            args = list(_inputs()[:3])
            with forward_ad.dual_level():
                args[which] = forward_ad.make_dual(args[which], torch.ones_like(args[which]))
                with pytest.raises((RuntimeError, NotImplementedError)):
                    _call(function, *args)


def test_vmap_and_batched_gradients_are_refused():
    for function in _functions():
        x, hw, bias, dy = _inputs()
        with pytest.raises(RuntimeError):
            torch.func.vmap(lambda v: _call(function, v, hw, bias))(torch.stack([x, x]))
        x.requires_grad_()
        y = _call(function, x, hw, bias)
        with pytest.raises(RuntimeError):
            torch.autograd.grad(y, x, torch.stack([dy, dy]), is_grads_batched=True)


_TRANSFORMS = {
    "vmap": lambda f, v: torch.func.vmap(f)(v),
    "grad": lambda f, v: torch.func.grad(lambda s: f(s).sum())(v[0]),
    "jvp": lambda f, v: torch.func.jvp(f, (v[0],), (v[0],)),
    "functionalize": lambda f, v: torch.func.functionalize(f)(v[0]),
}


@pytest.mark.parametrize("transform", _TRANSFORMS)
@pytest.mark.parametrize("constant", [True, False], ids=["constant_input", "transformed_input"])
def test_every_call_inside_a_transform_is_refused(transform, constant):
    """... whether or not the transform wraps one of its tensors; and taken again once the transform has ended."""
    for function in _functions():
        x, hw, bias, _ = _inputs()
        scale = torch.randn(3, device="cuda")
        before = _call(function, x, hw, bias)
        with pytest.raises(RuntimeError):
            _TRANSFORMS[transform](lambda s: _call(function, x if constant else x * s, hw, bias) * s, scale)
        assert torch.equal(_call(function, x, hw, bias), before)


@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("wanted", [(1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1), (0, 1, None), (1, 1, None)])
def test_compiled_autograd_takes_the_node_apart(wanted, fuse):
    from torch._dynamo import compiled_autograd
    got = []
    for function in _functions():
        x, hw, bias, dy = _inputs()
        leaves = (x, hw) if wanted[2] is None else (x, hw, bias)
        for t, w in zip(leaves, wanted):
            t.requires_grad_(bool(w))
        # (behind an operation and in front of one, so that edges of both kinds are met)
        y = _call(function, x * 2, hw, bias if wanted[2] is not None else None, fuse=fuse) * 3
        with compiled_autograd._enable(torch.compile(backend="eager")):
            y.backward(dy, retain_graph=True)
            y.backward(dy)
            with pytest.raises(RuntimeError, match="second time"):
                y.backward(dy)
        assert [t.grad is not None for t in leaves] == [bool(w) for w in wanted[:len(leaves)]]
        got.append([t.grad for t in leaves if t.grad is not None])
    assert all(torch.equal(a, b) for a, b in zip(*got))


def test_compiled_autograd_notices_a_change_in_place():
    from torch._dynamo import compiled_autograd
    for function in _functions():
        x, hw, bias, dy = _inputs()
        y = _call(function, x, hw.requires_grad_(), bias)
        x.add_(1)
        with compiled_autograd._enable(torch.compile(backend="eager")), pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.backward(dy)


@pytest.mark.parametrize("with_bias", [False, True])
def test_a_profiler_names_forward_and_backward(with_bias):
    seen = []
    for function in _functions():
        x, hw, bias, dy = _inputs()
        x.requires_grad_()
        for _ in range(2):   # (not the first call: that one also builds what it keeps)
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as profile:
                y = _call(function, x, hw, bias if with_bias else None)
                y.backward(dy)
        events = {e.name: e for e in profile.events()}
        forward, backward = events[function.__name__], events[function.__name__ + "Backward"]
        assert forward.sequence_nr == backward.sequence_nr >= 0
        seen.append((forward.input_shapes, backward.input_shapes))
    assert seen[0] == seen[1]


_ALLOCATOR = """
#include <hip/hip_runtime_api.h>
#include <sys/types.h>
extern "C" void* plain_alloc(ssize_t size, int, hipStream_t) {
  void* p = nullptr;
  return hipMalloc(&p, (size_t)size) == hipSuccess ? p : nullptr;
}
extern "C" void plain_free(void* p, ssize_t, int, hipStream_t) { (void)hipFree(p); }
"""

_UNDER_ANOTHER_ALLOCATOR = """
import sys
import torch
torch.cuda.memory.change_current_allocator(torch.cuda.memory.CUDAPluggableAllocator(sys.argv[1], "plain_alloc", "plain_free"))
from helpers import SEED_CONSTANTS
from rzlinear_amd import RzLinear, _lib
M, K, N = 1, 2048, 512
layer = RzLinear(K, N, hashed_weight=torch.nn.Parameter(torch.rand(20000).bfloat16()), dtype=torch.bfloat16).cuda()
x = torch.randn(M, K).bfloat16().cuda().requires_grad_()
assert _lib.load().rz_forward_hashed_workspace_bytes(M, K, N, 20000, 32, 64, _lib.RZ_BF16, None) > 0
got = []
for call in (layer, lambda v: type("InPython", (__import__("rzlinear_amd").RzLinearFunction,), {}).apply(
        v, layer._hashed_weight, layer._random_numbers, N, 1, 1.0, 32, 64, layer._bias, False)):
    y = call(x)
    got.append((y,) + torch.autograd.grad(y, (x, layer._hashed_weight, layer._bias), torch.ones_like(y)))
assert all(torch.equal(a, b) for a, b in zip(*got))
print("same", flush=True)
"""


def test_scratch_comes_from_the_allocator_in_force(tmp_path):
    """A program that has replaced torch's allocator has no caching allocator to take scratch memory from."""
    source, library = tmp_path / "allocator.cpp", tmp_path / "allocator.so"
    source.write_text(_ALLOCATOR)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-D__HIP_PLATFORM_AMD__", "-I%s/include" % rocm, "-shared", "-fPIC", str(source), "-o", str(library),
                    "-L%s/lib" % rocm, "-lamdhip64"], check=True)
    tests = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(tests), tests, os.environ.get("PYTHONPATH", "")]))
    child = subprocess.run([sys.executable, "-c", _UNDER_ANOTHER_ALLOCATOR, str(library)], env=env, capture_output=True, text=True, timeout=100)
    assert child.returncode == 0 and "same" in child.stdout, child.stdout + child.stderr
