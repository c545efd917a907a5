"""The FP64 sweep kernels at the edges of their cuts: lines of 1 cell, lines
shorter than a stencil, whole lines and segments (with the cells both
neighbours reconstruct), lines of more than 1024 cells, partly filled tiles
across the lines, periodic axes and walls; each direction against the oracle.

Tolerance: a sweep adds dt * tendency, whose rounding is a few ulp of the
1e5 Pa pressure (1.5e-11) times dt/dx (2e-3): some 1e-13 of momenta of order
10, and ulps of the full density and rho*theta.  1e-12 of each one's scale
leaves a factor of about ten.  The FP32 form against the FP64 sweeps: some
twenty roundings of 6e-8 in the weights and fluxes of rough data whose cell
differences are as large as the fields, 1e-5 of each field's maximum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# nx, ny, nz, bc (x, y, z), (ord, ngll)
BOXES = [
    (33, 1, 1, (0, 0, 1), (5, 3)),
    (5, 2, 3, (0, 0, 1), (5, 3)),
    (2, 3, 2, (0, 0, 0), (5, 3)),
    (3, 4, 5, (1, 1, 1), (5, 3)),
    (65, 17, 9, (1, 0, 1), (5, 3)),
    (100, 5, 66, (0, 0, 0), (5, 3)),
    (7, 131, 5, (0, 0, 1), (5, 3)),
    (7, 131, 5, (0, 1, 1), (5, 3)),
    (19, 70, 129, (0, 0, 1), (5, 3)),
    (6, 3, 301, (0, 0, 0), (5, 3)),
    (6, 3, 301, (0, 0, 1), (5, 3)),
    (1024, 2, 3, (0, 0, 1), (5, 3)),
    (1027, 2, 3, (0, 0, 1), (5, 3)),
    (1027, 2, 3, (1, 1, 1), (5, 3)),
    (37, 41, 23, (0, 0, 1), (3, 2)),
    (9, 150, 140, (1, 1, 0), (3, 2)),
]


def _state(shape, hs, seed):
    nz, ny, nx = shape
    rng = np.random.default_rng(seed)
    st = np.zeros((5, nz + 2 * hs, ny + 2 * hs, nx + 2 * hs))
    inner = st[:, hs:hs + nz, hs:hs + ny, hs:hs + nx]
    inner[0] = 1e-3 * rng.standard_normal((nz, ny, nx))
    inner[1:4] = 10.0 * rng.standard_normal((3, nz, ny, nx))
    inner[4] = 0.5 * rng.standard_normal((nz, ny, nx))
    return st


@pytest.mark.parametrize("nx,ny,nz,bc,og", BOXES)
def test_sweeps_match_oracle(nx, ny, nz, bc, og, figures):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pyoracle
    from awflcloud_amd import Dycore
    D = Dycore(nx, ny, nz, bc=bc, ord=og[0], ngll=og[1])
    O = pyoracle.Oracle(nx, ny, nz, bc=bc, ord=og[0], ngll=og[1])
    st = _state((nz, ny, nx), D.hs, 7)
    dt = 0.4 * min(D.dx, D.dz, D.dy if ny > 1 else D.dx) / 400.0
    full = [float(O.background(w)[D.hs:D.hs + nz].max()) for w in (0, 3)]
    scale = np.array([full[0], 10.0, 10.0, 10.0, full[1]])
    worst = []
    for d in (0, 1, 2):
        if d == 1 and ny == 1:
            continue
        ref = st.copy()
        O.sweep(ref, dt, d)
        out = torch.full(st.shape, np.nan, dtype=torch.float64, device="cuda")
        D.sweep(torch.from_numpy(st).cuda(), out, dt, d)
        got = D.interior(out).cpu().numpy()
        assert np.isfinite(got).all()
        worst.append(float((np.abs(got - O.interior(ref)).reshape(5, -1).max(1) / scale).max()))
        # tendencies and their application are the fused sweep bit for bit
        D.dim_switch = 1
        tend, two = D.new_tend(), torch.from_numpy(st).cuda()
        D.compute_tendencies(two, tend, dt, d)
        D.apply_tendencies(two, tend, dt, d)
        assert torch.equal(D.interior(two), D.interior(out))
    figures("sweeps vs oracle %s" % ["%.1e" % w for w in worst])
    assert max(worst) <= 1e-12


@pytest.mark.parametrize("nx,ny,nz,bc,og", BOXES)
def test_fp32_sweeps_match_fp64(nx, ny, nz, bc, og, figures):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awflcloud_amd import Dycore
    from awflcloud_amd.dycore import AWFL_FP32_PERT
    D = Dycore(nx, ny, nz, bc=bc, ord=og[0], ngll=og[1], precision=AWFL_FP32_PERT)
    st = torch.from_numpy(_state((nz, ny, nx), D.hs, 8)).cuda()
    s, c = D.to_f32(st)
    st = D.from_f32(s, c)
    dt = 0.4 * min(D.dx, D.dz, D.dy if ny > 1 else D.dx) / 400.0
    worst = []
    for d in (0, 1, 2):
        # across a periodic z boundary the FP32 form takes both sides' deviations
        # from the one background of the face, where the FP64 sweep sees the
        # background's own jump: another problem there
        if (d == 1 and ny == 1) or (d == 2 and bc[2] == 0):
            continue
        ref, so, co = D.new_state(), torch.zeros_like(s), torch.zeros_like(c)
        D.sweep(st, ref, dt, d)
        D.sweep_f32(s, c, so, co, dt, d)
        a, b = D.interior(D.from_f32(so, co)), D.interior(ref)
        scale = b.reshape(5, -1).abs().amax(1).clamp(min=1e-3)
        worst.append(float(((a - b).reshape(5, -1).abs().amax(1) / scale).max()))
    figures("FP32 sweeps vs FP64 %s" % ["%.1e" % w for w in worst])
    assert max(worst) <= 1e-5
