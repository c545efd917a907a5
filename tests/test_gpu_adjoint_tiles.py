"""The fused sweep adjoint (k_adj_tile in awfl_adjoint.hip) where its lanes and
lines can go wrong: lines as short as the stencil's half width,
one below, at and above whole waves and the largest line of the kernel, lines
that share a work-group unevenly, every boundary rule.

<y, J x> of the tangent-linear sweep (dual numbers, kernels of its own) equals
<J^T y, x> of the adjoint.  Both sides are sums of products of FP64 results
whose relative errors are a few hundred roundings at most (3e-14 with growth
against cancelling terms); the bound 1e-11 of the sum of magnitudes is that of
the adjoint's other dot-product tests."""
import pytest
import torch

from test_gpu_adjoint import _interior_dot, _need_gpu, _rand_like_state, _setup

pytestmark = pytest.mark.gpu

# nx, ny, nz, bc (0 periodic, 1 wall), ord, ngll
BOXES = [
    (2, 2, 2, (0, 0, 0), 5, 3),
    (2, 2, 3, (1, 1, 1), 5, 3),
    (1, 2, 1, (0, 1, 1), 3, 2),
    (3, 2, 2, (1, 0, 1), 5, 3),
    (2, 3, 4, (0, 1, 0), 3, 2),
    (63, 65, 2, (0, 1, 1), 5, 3),
    (65, 3, 64, (1, 0, 1), 5, 3),
    (127, 86, 3, (0, 0, 0), 5, 3),
    (9, 51, 85, (1, 0, 0), 5, 3),
    (128, 31, 33, (0, 0, 1), 5, 3),
    (43, 129, 33, (1, 1, 1), 3, 2),
    (257, 3, 2, (0, 0, 1), 5, 3),
    (3, 256, 2, (0, 0, 1), 5, 3),
    (640, 2, 3, (1, 0, 1), 5, 3),
    (2, 640, 3, (0, 0, 1), 5, 3),
    (2, 3, 640, (0, 0, 1), 5, 3),
    (641, 2, 3, (0, 0, 1), 3, 2),
]


@pytest.mark.parametrize("nx,ny,nz,bc,ord,ngll", BOXES)
def test_adjoint_of_sweeps(nx, ny, nz, bc, ord, ngll):
    _need_gpu()
    D, st, dt = _setup(nx, ny, nz, bc=bc, ord=ord, ngll=ngll)
    for d in (0, 1, 2):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(77 + d)
        x, y = _rand_like_state(D, gen), _rand_like_state(D, gen)
        _, dout = D.sweep_tangent(st, x, dt, d)
        xb = D.sweep_adjoint(st, y, dt, d)
        lhs, rhs = _interior_dot(D, y, dout), _interior_dot(D, xb, x)
        scale = float((D.interior(y) * D.interior(dout)).abs().sum())
        print("dir %d  <y,Jx> %.15e  <J^T y,x> %.15e  rel %.2e" % (d, lhs, rhs, abs(lhs - rhs) / scale), flush=True)
        assert abs(lhs - rhs) <= 1e-11 * scale
        mask = torch.ones_like(xb, dtype=torch.bool)
        hs = D.hs
        mask[:, hs:hs + nz, hs:hs + ny, hs:hs + nx] = False
        assert float(xb[mask].abs().max()) == 0.0
