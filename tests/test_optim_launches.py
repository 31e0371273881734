"""What FusedAdam hands to rz_adam_step_many, and when: a stand-in for the library records the launches (no GPU)."""
import weakref

import pytest
import torch

from rzlinear_amd import _lib, optim


class _Recorder:
    """rz_adam_step_many that notes (step, [(parameter's address, words of the tensor), ...]) of every launch."""

    def __init__(self):
        self.launches, self.fail_at = [], None

    def rz_adam_step_many(self, words, count, lr, b1, b2, eps, wd, decoupled, step, scale, stream):
        if self.fail_at == len(self.launches):
            self.fail_at = None
            return -8
        self.launches.append((step, [tuple(words[8 * i:8 * i + 8]) for i in range(count)]))
        return 0

    def rz_status_string(self, status):
        return b"refused by the stand-in"

    def order(self):
        return [[w[0] for w in words] for _, words in self.launches]


class _Stream:
    cuda_stream = 0


@pytest.fixture
def library(monkeypatch):
    rec = _Recorder()
    monkeypatch.setattr(_lib, "load", lambda: rec)
    monkeypatch.setattr(optim, "_check", lambda p, g: None)   # (which refuses CPU parameters)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: _Stream)
    return rec


def _params(n, dtype=torch.float32):
    out = [torch.nn.Parameter(torch.zeros(16, dtype=dtype)) for _ in range(n)]
    for p in out:
        p.grad = torch.ones_like(p)
    return out


def test_parameters_of_unequal_steps_keep_the_groups_order(library):
    """A, B and C, a view of B; B has no gradient in the first step, so that its count is one behind from then on."""
    a, b = _params(2)
    c = torch.nn.Parameter(b.detach()[4:12])
    c.grad = torch.ones_like(c)
    opt = optim.FusedAdam([a, b, c])
    b.grad = None
    opt.step()
    assert library.order() == [[a.data_ptr(), c.data_ptr()]]
    library.launches.clear()
    b.grad = torch.ones_like(b)
    opt.step()
    assert [p for launch in library.order() for p in launch] == [a.data_ptr(), b.data_ptr(), c.data_ptr()]
    assert [step for step, words in library.launches for _ in words] == [2, 1, 2]


class _MadeWhenAsked(torch.nn.Parameter):
    """A parameter whose main_grad has no owner but who asked for it."""

    @property
    def main_grad(self):
        g = torch.ones(self.shape)
        self.freed = []
        weakref.finalize(g, self.freed.append, True)
        return g


def test_a_gradient_is_held_until_its_launch(library):
    params = [_MadeWhenAsked(torch.zeros(16)) for _ in range(3)]
    launch = library.rz_adam_step_many
    alive = []

    def look(*args):
        alive.extend(not p.freed for p in params)
        return launch(*args)

    library.rz_adam_step_many = look
    optim.FusedAdam(params).step()
    assert alive == [True] * 3
    assert all(p.freed for p in params)   # (and no longer)


def test_a_launch_that_failed_is_not_made_again(library):
    """The second parameter's master copy forces a launch of the first; it fails, and its error is the one that is seen."""
    a, b = _params(2, torch.bfloat16)
    opt = optim.FusedAdam([a, b], master_weights=True)
    library.fail_at = 0
    with pytest.raises(_lib.RzLinearError, match="refused by the stand-in") as e:
        opt.step()
    assert library.launches == [] and e.value.__context__ is None
