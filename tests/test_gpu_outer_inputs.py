"""What the outer loops take and hold whichever kernels they run (GPU)."""
import pytest
import torch

from pgj.outer import GaussianOuter, PaperOuter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rmin', [2.0, 4.5])
def test_physical_takes_a_strided_density(rmin):
    """A density of another memory order (assigned, not copied in) is filtered as its contiguous copy."""
    print(f'strided density rmin={rmin}', flush=True)
    x = torch.rand((9, 9, 9), generator=torch.Generator().manual_seed(3), dtype=torch.float64).cuda()
    out = []
    for strided in (False, True):
        o = PaperOuter(9, .3, rmin=rmin)
        assert o.fused == (rmin < 4)
        o.x = x.permute(2, 1, 0) if strided else x.permute(2, 1, 0).contiguous()
        o.physical()
        out.append([f.clone() for f in (o.t, o.ph, o.dp, o.a)])
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize('make, rest', [(lambda n: PaperOuter(n, .3), 2), (lambda n: GaussianOuter(n), 3)])
def test_fused_loops_hold_no_fields_they_do_not_use(make, rest):
    """At most the 11 fields of a design step and what the filter and the bisection need (root: two fields; tmp1, tmp2,
    gin) besides small workspaces."""
    print('outer fields', flush=True)
    n = 48
    make(8)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    o = make(n)
    assert o.fused
    assert torch.cuda.memory_allocated() - before < (11 + rest + .5) * n ** 3 * 8
