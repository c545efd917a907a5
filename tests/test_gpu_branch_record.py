"""The upwind record of awfl_time_step_branches holds every face: of a periodic
line also the last one, in y and z by its own byte and in x, where it is the
first face, by the first's.  Lines whole and in segments."""
import pytest
import torch

from test_gpu_tiles import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(12, 10, 8), (1027, 3, 2), (5, 301, 3), (4, 3, 260)])
@pytest.mark.parametrize("bc", [(0, 0, 0), (0, 0, 1), (1, 1, 1)])
def test_record_holds_every_face(nx, ny, nz, bc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awflcloud_amd import Dycore
    D = Dycore(nx, ny, nz, bc=bc)
    base = torch.from_numpy(_state((nz, ny, nx), D.hs, 5)).cuda()
    dt = 0.4 * min(D.dx, D.dy, D.dz) / 400.0
    rec = D.new_branch_record().fill_(255)
    D.dim_switch = 1
    want = base.clone()
    D.time_step_branches(want, dt, rec, 1)
    n = (nx + 1) * (ny + 1) * (nz + 1)
    x = rec[:n][:nz * ny * (nx + 1)].view(nz, ny, nx + 1)
    y = rec[n:2 * n][:nz * (ny + 1) * nx].view(nz, ny + 1, nx)
    z = rec[2 * n:][:(nz + 1) * ny * nx].view(nz + 1, ny, nx)
    assert int(x[..., :nx if bc[0] == 0 else nx + 1].max()) <= 1
    assert int(y.max()) <= 1 and int(z.max()) <= 1
    if bc[1] == 0:
        assert torch.equal(y[:, 0], y[:, ny])
    if bc[2] == 0:
        assert torch.equal(z[0], z[nz])
    # a replay takes the last face of a periodic x line from the first's byte
    if bc[0] == 0:
        x[..., nx] = 1 - x[..., 0]
    D.dim_switch = 1
    got = base.clone()
    D.time_step_branches(got, dt, rec, 2)
    assert torch.equal(D.interior(got), D.interior(want))
