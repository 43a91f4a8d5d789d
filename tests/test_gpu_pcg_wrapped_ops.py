"""Operators whose apply or preconditioner was replaced keep their own in every iteration of ``solve_pcg_batched`` (GPU).

Replaced on the class, or on a wrapper that hands every other name on to a plain operator: iterations as many as the
plain operator's, each with one call.
"""
import numpy as np
import pytest
import torch

import pgj

pytestmark = pytest.mark.gpu


def _problem():
    a = torch.tensor(np.exp(np.random.default_rng(1).uniform(-4, 0, (8, 8, 8))), device='cuda')
    op = pgj.set_alpha(pgj.build(a), .5)
    return op, op.compute_rhs(np.eye(6)[3])


@pytest.mark.parametrize('name', ['apply', 'green_precond'])
def test_methods_replaced_on_the_class_are_called(monkeypatch, name):
    print(f'class {name} replaced', flush=True)
    op, rhs = _problem()
    ref, it, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-8)
    calls = []
    method = getattr(pgj.Operator, name)
    monkeypatch.setattr(pgj.Operator, name, lambda self, *args: (calls.append(name), method(self, *args))[1])
    u, jt, _ = pgj.solve_pcg_batched(op, rhs, tol=1e-8)
    assert len(calls) == jt == it and float((u - ref).norm() / ref.norm()) < 1e-6


class _Shifted:
    """Hands everything on to an operator but its apply, which adds ``shift`` u."""

    def __init__(self, op, shift):
        self.op, self.shift, self.calls = op, shift, 0

    def __getattr__(self, name):
        return getattr(self.op, name)

    def apply(self, u):
        self.calls += 1
        return self.op.apply(u) + self.shift * u


def test_delegating_wrapper_solves_its_own_system():
    print('delegating wrapper', flush=True)
    op, rhs = _problem()
    wrapped = _Shifted(op, 1e-3)
    u, it, res = pgj.solve_pcg_batched(wrapped, rhs, tol=1e-8)
    assert wrapped.calls == it and float(res.max()) < 1e-8
    # the recurrence's residual is the true one up to rounding
    true = float((rhs - op.apply(u) - 1e-3 * u).norm() / rhs.norm())
    assert true < 2e-8
