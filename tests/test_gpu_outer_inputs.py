"""What the outer loops take and hold whichever kernels they run (GPU)."""
import pytest
import torch

from pgj.outer import PaperOuter

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
