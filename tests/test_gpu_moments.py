"""Column sums, the Poisson solve and the invariants at the edges of their
kernels' ranges: one and several chunks of rows (512 | 513), the FFT form of
the Poisson solve from the shortest to the longest x-grid with even and odd
log2, the one-workgroup convolution up to its limit (320) and the three-launch
form beyond it.

Bars: the sums of nv positive terms in any order differ by at most
nv eps relative, 1e-12 at nv = 4096; phi as in test_moments_and_poisson
(1e-11 relative); invariants 1e-11 relative (sums of up to 2^23 terms of one
sign in trees of depth < 2^9 a thread, the energies compared on their scale).
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu

GRIDS = [(8, 8), (9, 513), (64, 512), (65, 511), (128, 129), (320, 640), (321, 64), (512, 1025), (1000, 100),
         (2048, 513), (4096, 64), (16, 4096)]


@pytest.mark.parametrize("nx,nv", GRIDS)
def test_moments_poisson_invariants(nx, nv, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, flush=True)
    rng = np.random.default_rng(nx * 7 + nv)
    L = 4 * np.pi
    g = O.Grid(nx, nv, L, 8.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, L, 8.0, ht=0.05), preconditioner='', charge=-1.0)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    f = 0.5 + rng.random((nx, nv))
    fd = T(f.T)
    n_ref, u_ref, e_ref = O.density(f, g), O.velocity_density(f, g), O.energy_density(f, g)
    n, u, e, phi, h1 = (ctx.new_x() for _ in range(5))
    ctx.density(fd, n)
    ctx.velocity_moments(fd, u, e)
    assert np.abs(n.cpu().numpy() - n_ref).max() <= 1e-12 * n_ref.max()
    umax = (np.abs(g.v) * f).sum(axis=1).max() * g.hv
    assert np.abs(u.cpu().numpy() - u_ref).max() <= 1e-12 * umax
    assert np.abs(e.cpu().numpy() - e_ref).max() <= 1e-12 * e_ref.max()
    n2 = ctx.new_x()
    ctx.moments(fd, n2, phi, h1, want_norm=True)
    assert np.abs(n2.cpu().numpy() - n_ref).max() <= 1e-12 * n_ref.max()
    # a smooth density: phi well above the rounding of n
    x = np.arange(nx) * L / nx
    n_s = 1.0 + 0.3 * np.cos(0.5 * x) + 0.05 * np.sin(1.5 * x)
    # phi = (n - mean n) / lambda per mode, the stencil's symbol without the
    # cancellation of its cosine form (1.8e-11 relative at nx = 2048)
    sym = lambda k: (128 * np.sin(np.pi * k / nx) ** 2 - 20 * np.sin(2 * np.pi * k / nx) ** 2) / (12 * g.hx ** 2)
    phi_ref = 0.3 * np.cos(0.5 * x) / sym(1) + 0.05 * np.sin(1.5 * x) / sym(3)
    ctx.poisson_solve(T(n_s), phi)
    p = phi.cpu().numpy()
    assert np.abs((p - p.mean()) - (phi_ref - phi_ref.mean())).max() <= 1e-11 * np.abs(phi_ref).max()
    h0 = O.kinetic_hamiltonian(g)
    h1v, h2v = rng.standard_normal((2, nx))
    inv = ctx.invariants(fd, T(h0), T(h1v), T(h2v), phi)
    ref = O.invariants(f, h0, h1v, h2v, p, g, -1.0)
    scale = (f * (h0[None, :] + np.abs(h1v)[:, None] + np.abs(h2v)[:, None])).sum() * g.hx * g.hv
    for k in ('mass', 'l2', 'efield'):
        assert abs(inv[k] - ref[k]) <= 1e-11 * abs(ref[k]), k
    for k in ('energy', 'ekin', 'epot'):
        assert abs(inv[k] - ref[k]) <= 1e-11 * scale, k
