"""The fused sweep adjoint on long lines: two lines of up to 384 cells share a
work-group; it takes lines of up to 768 cells and no scratch per cell; longer ones
run as five kernels.  Tolerances as in
test_gpu_adjoint_tiles.py, whose test this is at other boxes."""
import pytest
import torch

from test_gpu_adjoint import _need_gpu, _setup
from test_gpu_adjoint_tiles import test_adjoint_of_sweeps as dot_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,bc,ord,ngll", [
    (682, 3, 2, (0, 1, 0), 3, 2),
    (3, 682, 2, (1, 0, 1), 3, 2),
    (2, 3, 682, (0, 1, 1), 3, 2),
    (768, 2, 3, (1, 0, 1), 5, 3),
    (2, 768, 3, (0, 0, 1), 5, 3),
    (2, 3, 768, (0, 0, 1), 3, 2),
    (257, 3, 87, (0, 0, 1), 5, 3),        # two lines to a group, the last group with one
    (20, 300, 13, (0, 1, 1), 3, 2),
    (9, 29, 384, (1, 0, 1), 5, 3),
    (7, 37, 321, (0, 0, 0), 3, 2),
    (384, 20, 13, (1, 1, 1), 3, 2),
    (769, 2, 3, (0, 0, 1), 3, 2),
    (2, 769, 3, (0, 1, 1), 5, 3),
    (2, 3, 769, (0, 0, 0), 3, 2),
])
def test_long_lines(nx, ny, nz, bc, ord, ngll):
    dot_product(nx, ny, nz, bc, ord, ngll)


@pytest.mark.parametrize("nx,ny,nz,d", [(682, 64, 40, 0), (64, 682, 40, 1), (64, 40, 682, 2), (768, 64, 40, 0)])
def test_no_scratch_per_cell(nx, ny, nz, d):
    """56 doubles per cell would be 780 MB here; the states are allocated before."""
    _need_gpu()
    D, st, dt = _setup(nx, ny, nz, ord=3, ngll=2)
    y, out = torch.ones_like(st), D.new_state()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    D.sweep_adjoint(st, y, dt, d, out)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 100e6
