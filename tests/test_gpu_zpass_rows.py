"""A radix plan set between the launches of a solve changes speed only (GPU).

The forms of the z pass leave different numbers of partial rows for the passes that sum r.z and the projection's means.
An iteration captured under one plan and a first direction formed under another must give the iterates of a solve under
one plan: four iterations agree to rounding (each pass rounds its sums differently, 1e-13 an iteration, amplified by the
step lengths: 1e-10).
"""
import numpy as np
import pytest
import torch

from oracle import design
from pgj import _lib
from pgj.batched import DesignGroup
from pgj.mixed import MixedResident

pytestmark = pytest.mark.gpu


def _plan_z(grid, es, plan):
    _lib.check(_lib.lib().pgj_fft_set_plan(grid, es, 1, plan))


def _captured(fn):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


# register-resident z pass by default, LDS form under plan 1 (64^3 FP64: the wide one at 12 loads)
@pytest.mark.parametrize('n, designs', [(16, 1), (32, 1), (64, 2), (128, 1)])
@pytest.mark.parametrize('captured, eager', [(-1, 1), (1, -1)])
def test_plan_between_capture_and_start(n, designs, captured, eager):
    print(f'plan between capture {captured} and start {eager}: FP64 {n}^3', flush=True)
    loads = np.eye(6) if n < 128 else np.eye(6)[[0, 4]]
    g = DesignGroup(n, designs, loads)
    a = torch.tensor(design.simp(design.filtered_noise(n, 5, 2), 1e-4), device='cuda')
    for d in range(designs):
        g.material(d, a)
        g.select(d, .5)

    def start():
        g.u.zero_()
        g.setup(1e-8)
        g.certify()
        g.initialize()
    try:
        start()
        g.iteration()
        ref = g.u.clone()
        _plan_z(g.op.grid, 8, captured)
        start()
        g.iteration()
        graph = _captured(g.iteration)
        _plan_z(g.op.grid, 8, eager)
        for _ in range(2):
            g.ws.fill_(255)      # rows that no pass of this solve wrote would be NaN
            start()
            graph.replay()
            assert not bool(g.bad.any())
            assert float((g.u - ref).abs().max()) < 1e-10 * float(ref.abs().max())
    finally:
        _plan_z(g.op.grid, 8, -1)


@pytest.mark.parametrize('n', [32, 64])
def test_plan_between_capture_and_start_fp32(n):
    """The FP32 inner solver: iterates of four iterations agree to FP32 rounding (1e-4 of max|d|)."""
    print(f'plan between capture and start: FP32 {n}^3', flush=True)
    m = MixedResident(n)
    m.material(0, torch.tensor(design.simp(design.filtered_noise(n, 5, 2), 1e-4), device='cuda'))
    m.select(0, .5)

    def start():
        m.u.zero_()
        m.setup(1e-8)
        m.certify()
        m.begin()
    try:
        start()
        m.iteration()
        ref = m.d.clone()
        graph = _captured(m.iteration)
        _plan_z(m.op.grid, 4, 1)
        m.ws32.fill_(255)
        start()
        graph.replay()
        assert not bool(m.bad32.any())
        assert float((m.d - ref).abs().max()) < 1e-4 * float(ref.abs().max())
    finally:
        _plan_z(m.op.grid, 4, -1)
