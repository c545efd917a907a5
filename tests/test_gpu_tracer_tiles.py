"""The tracer sweeps where their tiles and walkers can go wrong (awfl_tracers.hip:
k_tile_tr, k_walk_tr and the rule between them): lines as short as the stencil's
half width, one below, at and above whole waves, lines that share a work-group
unevenly, the longest line of a tile, lines that the walkers keep, one to eight
tracers, every boundary rule.  Updated state and tracers against the oracle.

Tolerance: a flux carries a few tens of roundings of the pressure (1e5) or of
the sound speed (350) times a tracer, and an update is a CFL number's worth of it:
0.8 / 350 * 1e5 * 64 eps = 3e-12 on momenta of 3 to 10, 1e-14 of a tracer.  1e-12
of the largest value of the field, as for the sweeps without tracers.  (Tendencies
themselves nearly cancel on some of these boxes and are no scale.)"""
import numpy as np
import pytest
import torch

from helpers import bubble_dicts
from test_gpu_tracers import P, _need_gpu, _spec_kw, _tracer_fields

pytestmark = pytest.mark.gpu

# nx, ny, nz, bc (0 periodic, 1 wall), positivity flags, ord, ngll
BOXES = [
    (2, 3, 2, (0, 0, 0), (1,), 5, 3),
    (3, 2, 7, (1, 1, 1), (1, 0), 5, 3),
    (7, 8, 9, (0, 1, 0), (0, 1, 1, 1), 3, 2),
    (63, 65, 33, (0, 1, 1), (1, 1, 0), 5, 3),
    (65, 64, 31, (1, 0, 0), (0,), 5, 3),
    (127, 40, 43, (0, 0, 1), (1, 1, 1, 0, 1), 5, 3),
    (86, 51, 26, (1, 1, 0), (0, 1, 1, 0, 1, 1, 1, 1), 3, 2),
    (257, 3, 64, (0, 0, 1), (1, 1), 5, 3),
    (6, 256, 100, (1, 0, 1), (0, 1, 1), 5, 3),      # y and z tiles of eight waves
    (6, 200, 3, (0, 0, 1), (0, 1, 1), 5, 3),        # y walker
    (8, 6, 180, (0, 1, 1), (0, 1, 1), 5, 3),        # z walkers
    (8, 6, 180, (0, 1, 0), (1, 0, 1, 1), 5, 3),
    (600, 3, 4, (1, 0, 1), (1, 1, 0), 5, 3),
    (1024, 2, 3, (0, 0, 1), (1,), 5, 3),
    (1030, 2, 3, (0, 0, 1), (1,), 5, 3),            # past a tile: the line kernel
]


@pytest.mark.parametrize("nx,ny,nz,bc,pos,ord,ngll", BOXES)
def test_sweeps_match_oracle(nx, ny, nz, bc, pos, ord, ngll):
    _need_gpu()
    from awflcloud_amd import Dycore, bubble_spec
    D = Dycore(nx, ny, nz, bc=bc, ord=ord, ngll=ngll)
    st = D.init_state(bubble_spec(bubble_dicts(), **_spec_kw(ny)))
    dt = D.compute_time_step(st, 0.8)
    D.set_tracers(pos)
    O = P.Oracle(nx, ny, nz, bc=bc, ord=ord, ngll=ngll)
    O.set_tracers(pos)
    O.set_dt_cache(dt)
    host = st.cpu().numpy().copy()
    fields = _tracer_fields(nx, ny, nz, O.dx, O.dy, O.dz, O.density(host))
    tr_host = np.zeros(O.tracer_shape())
    O.tracer_interior(tr_host)[...] = np.stack([fields[(t + 1) % 3] * (1.0 + 0.25 * t) for t in range(len(pos))])
    tr = torch.from_numpy(tr_host.copy()).cuda()
    D.dim_switch = 1
    for d in (0, 1, 2):
        tend = D.new_tend()
        ttend = torch.zeros(D.tracer_tend_shape, dtype=torch.float64, device="cuda")
        D.compute_tendencies_tracers(st, tr, tend, ttend, dt, d)
        otend, ottend = O.tendencies_dir_tr(host, tr_host, dt, d)
        out, tro = D.new_state(), D.new_tracers()
        D.sweep_tracers(st, tr, out, tro, dt, d)
        hs = D.hs
        inner = (slice(None),) + tuple(slice(hs, hs + m) for m in (nz, ny, nx))
        want, twant = host[inner] + dt * otend, O.tracer_interior(tr_host) + dt * ottend
        got, tgot = out.cpu().numpy()[inner], O.tracer_interior(tro.cpu().numpy())
        serr = float(np.abs(got - want).max() / np.abs(want).max())
        terr = max(float(np.abs(tgot[t] - twant[t]).max() / max(np.abs(twant[t]).max(), 1e-300)) for t in range(len(pos)))
        # the tendencies are the update's
        derr = float(np.abs(host[inner] + dt * tend.cpu().numpy() - got).max() / np.abs(want).max())
        g = ttend.cpu().numpy()
        uerr = max(float(np.abs(O.tracer_interior(tr_host)[t] + dt * g[t] - tgot[t]).max() /
                         max(np.abs(twant[t]).max(), 1e-300)) for t in range(len(pos)))
        print("dir %d  state %.2e  tracers %.2e  by tendencies %.2e %.2e" % (d, serr, terr, derr, uerr), flush=True)
        assert serr <= 1e-12
        assert terr <= 1e-12
        assert derr <= 1e-14
        assert uerr <= 1e-14
