"""Both forms of the y and z sweeps, tiles and column walkers, wherever the rule
between them would go: the tests of test_gpu_tiles.py and test_gpu_tracer_tiles.py
with each form imposed, ragged widths (idle lanes of a walker's wave), lengths that
its segments do not divide, every boundary rule, and the forms against each other.

FP64 forms run the same statements with every multiply-add written out: equal bit
for bit.  FP32 forms and those with tracers are compiled with contraction, which may
fall differently in the two kernels: as far apart as a rounding each in weights and
fluxes, the bounds of test_gpu_tiles.py (1e-5 of a field, here also across periodic
z, where both see the same face backgrounds) and test_gpu_tracer_tiles.py (1e-12)."""
import pytest
import torch

import test_gpu_tiles as tiles
import test_gpu_tracer_tiles as tracer_tiles

pytestmark = pytest.mark.gpu

RAGGED = [
    (37, 45, 50, (0, 1, 0), (5, 3)),
    (65, 45, 50, (1, 0, 1), (3, 2)),
    (65, 33, 70, (1, 1, 1), (5, 3)),
    (37, 47, 66, (0, 0, 0), (3, 2)),
    (130, 70, 3, (0, 0, 1), (5, 3)),
]
BOXES = [b for b in tiles.BOXES if b[0] <= 100] + RAGGED
TR_BOXES = [b for b in tracer_tiles.BOXES if max(b[1], b[2]) >= 8]


@pytest.fixture
def impose(monkeypatch):
    """impose(form): Dycore objects made from here on take that form"""
    import awflcloud_amd

    def set_form(form):
        class Formed(awflcloud_amd.Dycore):
            def __init__(self, *a, **k):
                super().__init__(*a, **k)
                self.set_sweep_form(form)
        monkeypatch.setattr(awflcloud_amd, "Dycore", Formed)
    return set_form


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("nx,ny,nz,bc,og", BOXES)
def test_sweeps_match_oracle(nx, ny, nz, bc, og, form, impose, figures):
    impose(form)
    tiles.test_sweeps_match_oracle(nx, ny, nz, bc, og, figures)


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("nx,ny,nz,bc,og", BOXES)
def test_fp32_sweeps_match_fp64(nx, ny, nz, bc, og, form, impose, figures):
    if bc[2] == 0 and ny == 1:
        pytest.skip("no direction to compare")
    impose(form)
    tiles.test_fp32_sweeps_match_fp64(nx, ny, nz, bc, og, figures)


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("nx,ny,nz,bc,pos,ord,ngll", TR_BOXES)
def test_tracer_sweeps_match_oracle(nx, ny, nz, bc, pos, ord, ngll, form, impose):
    impose(form)
    tracer_tiles.test_sweeps_match_oracle(nx, ny, nz, bc, pos, ord, ngll)


@pytest.mark.parametrize("nx,ny,nz,bc,og", BOXES)
def test_forms_agree(nx, ny, nz, bc, og, figures):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awflcloud_amd import Dycore
    from awflcloud_amd.dycore import AWFL_FP32_PERT
    D = Dycore(nx, ny, nz, bc=bc, ord=og[0], ngll=og[1], precision=AWFL_FP32_PERT)
    st = torch.from_numpy(tiles._state((nz, ny, nx), D.hs, 9)).cuda()
    s, c = D.to_f32(st)
    dt = 0.4 * min(D.dx, D.dz, D.dy if ny > 1 else D.dx) / 400.0
    worst = []
    for d in (1, 2):
        if d == 1 and ny == 1:
            continue
        out = []
        for form in (1, 2):
            D.set_sweep_form(form)
            o = torch.full_like(st, float("nan"))
            D.sweep(st, o, dt, d)
            so, co = torch.zeros_like(s), torch.zeros_like(c)
            D.sweep_f32(s, c, so, co, dt, d)
            out.append((D.interior(o), D.interior(D.from_f32(so, co))))
        (a64, a32), (b64, b32) = out
        assert torch.isfinite(a64).all()
        assert torch.equal(a64, b64)
        scale = b32.reshape(5, -1).abs().amax(1).clamp(min=1e-3)
        worst.append(float(((a32 - b32).reshape(5, -1).abs().amax(1) / scale).max()))
    figures("FP32 forms apart %s" % ["%.1e" % w for w in worst])
    assert max(worst, default=0.0) <= 1e-5


def test_form_is_checked():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awflcloud_amd import Dycore
    from awflcloud_amd.dycore import AwflError
    D = Dycore(16, 16, 16)
    for form in (-1, 3):
        with pytest.raises(AwflError):
            D.set_sweep_form(form)
