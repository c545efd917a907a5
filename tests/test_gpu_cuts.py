"""The forms that the rules of awfl_cut.hpp choose between: x lines of more than 512
cells, in segments and, updated in place, whole.  The sweeps against the oracle
with the tolerance of test_gpu_tiles.py, whose test they run at other boxes; the
in-place step against the other bit for bit, as the header promises."""
import pytest
import torch

from test_gpu_tiles import _state
from test_gpu_tiles import test_sweeps_match_oracle as sweeps_match_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,bc,og", [
    (513, 3, 2, (0, 0, 1), (5, 3)),
    (560, 2, 3, (1, 1, 1), (3, 2)),
    (700, 3, 2, (1, 0, 1), (5, 3)),
    (768, 2, 2, (0, 0, 0), (3, 2)),
    (1000, 1, 2, (1, 0, 1), (5, 3)),
])
def test_long_x_lines(nx, ny, nz, bc, og, figures):
    sweeps_match_oracle(nx, ny, nz, bc, og, figures)


@pytest.mark.parametrize("nx,bc,og", [(513, (0, 0, 1), (5, 3)), (700, (1, 1, 1), (5, 3)), (1000, (0, 0, 0), (5, 3)),
                                      (1023, (1, 0, 1), (3, 2))])
def test_whole_lines_in_place(nx, bc, og):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awflcloud_amd import Dycore
    D = Dycore(nx, 3, 2, bc=bc, ord=og[0], ngll=og[1])
    a = torch.from_numpy(_state((2, 3, nx), D.hs, 11)).cuda()
    b = a.clone()
    dt = 0.4 * min(D.dx, D.dy, D.dz) / 400.0
    for _ in range(2):                     # both orders of the splits
        ds = D.dim_switch
        D.time_step(a, dt)
        D.dim_switch = ds
        D.time_step_noalloc(b, dt)
    assert torch.isfinite(D.interior(a)).all()
    assert torch.equal(D.interior(a), D.interior(b))
