"""The Poisson pipeline on both sides of the line between one workgroup's
convolution (up to 256 points, no power of two) and the three launches: phi of a
smooth density within 1e-11 relative of the stencil's symbol (as test_gpu_moments),
h1 = phi - mean phi, and the residual norm, from a density and from a field.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [254, 255, 257, 258, 300, 320])
def test_poisson(nx, cuda):
    import torch
    from vivlasov1d_amd.core import Grid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, flush=True)
    L, nv = 4 * np.pi, 70
    g = Grid(nx, nv, L, 8.0, ht=0.05)
    ctx = Context(g, preconditioner='', charge=-1.0)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    x = np.arange(nx) * L / nx
    n = 1.0 + 0.3 * np.cos(0.5 * x) + 0.05 * np.sin(1.5 * x)
    sym = lambda k: (128 * np.sin(np.pi * k / nx) ** 2 - 20 * np.sin(2 * np.pi * k / nx) ** 2) / (12 * g.hx ** 2)
    ref = 0.3 * np.cos(0.5 * x) / sym(1) + 0.05 * np.sin(1.5 * x) / sym(3)
    phi, h1, nn = ctx.new_x(), ctx.new_x(), ctx.new_x()
    ctx.poisson_solve(T(n), phi)
    p = phi.cpu().numpy()
    assert np.abs((p - p.mean()) - ref).max() <= 1e-11 * np.abs(ref).max()
    f = np.full(nv, 1.0 / (nv * g.hv))[:, None] * n[None, :]       # the same density, from a field
    pres = ctx.moments(T(f), nn, phi, h1)
    p = phi.cpu().numpy()
    assert np.abs(nn.cpu().numpy() - n).max() <= 1e-13
    assert np.abs((p - p.mean()) - ref).max() <= 1e-11 * np.abs(ref).max()
    assert np.abs(h1.cpu().numpy() - (p - p.mean())).max() <= 1e-14 * np.abs(p).max()
    assert pres <= 1e-10 * np.linalg.norm(n - n.mean())
