"""x-lengths whose transform is a single stage (primes; 9 and 15): P^-1 by the
direct real DFT, J u and the dots fused with the line sum up to 256 points and
2^25 products, separate launches beyond.  On both sides of each limit: the route
taken, P^-1 F, P^-1 J u, P^-1 in FP64 and FP32 (aligned and not) against the
oracle, and solves fused and separate, FP64, mixed and adjoint.

Bars as in test_gpu_rows: 1e-12 relative against the oracle, FP32 2e-6, solutions
1e-9 (rtol 1e-10; mixed 1e-8).
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu

# (nx, nv, whether the row blocks apply): 251^2 x 532 <= 2^25 < 251^2 x 533
GRIDS = [(9, 40, True), (15, 33, True), (11, 64, True), (53, 41, True), (251, 532, True), (251, 533, False),
         (257, 20, False), (499, 24, False), (1999, 12, False)]


def _setup(nx, nv, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    rng = np.random.default_rng(nx + 3 * nv)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.02)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.02), charge=-1.0)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    h0 = O.kinetic_hamiltonian(g)
    hs = [0.02 * rng.standard_normal(nx) for _ in range(4)]
    ctx.set_hamiltonian(T(h0), *[T(h) for h in hs])
    return g, ctx, O.h_average(h0, *hs), rng, T


@pytest.mark.parametrize("nx,nv,fused", GRIDS)
def test_callbacks_and_route(nx, nv, fused, cuda):
    import torch
    print("case", nx, nv, fused, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, cuda)
    pc = O.Preconditioner(g, 'lapack')
    f = rng.random((nx, nv))
    fh = f + 0.01 * rng.standard_normal((nx, nv))
    u = rng.standard_normal((nx, nv))
    y = ctx.new_field()
    ctx.function(T(f.T), T(fh.T), y)
    ref = pc.apply(O.residual('arakawaj4', f, fh, H, g))
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    ctx.profile(("jac_rfft", "jacobian", "rfft"))
    ctx.jacobian(T(u.T), y)
    n = {k: ctx.profile_read(k)[1] for k in ("jac_rfft", "jacobian", "rfft")}
    ctx.profile(())
    assert n == ({"jac_rfft": 1, "jacobian": 0, "rfft": 0} if fused else {"jac_rfft": 0, "jacobian": 1, "rfft": 1})
    ref = pc.apply(O.jacobian('arakawaj4', u, H, g))
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    ref = pc.apply(u)
    for off in (0, 1):                    # aligned for pairs, and not
        buf = torch.zeros(nx * nv + off, dtype=torch.float64, device=cuda)
        ctx.precond(T(u.T), buf[off:])
        assert np.abs(buf[off:].cpu().numpy().reshape(nv, nx).T - ref).max() <= 1e-12 * np.abs(ref).max()
    u32 = u.astype(np.float32)
    y32 = torch.empty(nv, nx, dtype=torch.float32, device=cuda)
    ctx.precond32(T(u32.T), y32)
    ref = pc.apply(u32.astype(np.float64))
    assert np.abs(y32.double().cpu().numpy().T - ref).max() <= 2e-6 * np.abs(ref).max()


@pytest.mark.parametrize("nx,nv,fused", GRIDS)
def test_solves(nx, nv, fused, cuda):
    print("case", nx, nv, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, cuda)
    f = np.exp(-0.5 * g.v ** 2)[None, :] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(nx) / nx))[:, None]
    b, fbar = T((f * np.sin(3 * g.v)[None, :]).T), T(f.T)
    out = []
    for on in (True, False):
        ctx.set_fusion(on)
        x, m, lam, mu = (ctx.new_field() for _ in range(4))
        r = ctx.ksp_solve(b, x, 1e-10, 1e-50, 1e5, 400)
        rm, _ = ctx.ksp_solve_mixed(b, m, 1e-10, 1e-50, 1e5, 800)
        ra = ctx.adjoint_step(b, lam, mu, 1e-10, 1e-50, 1e5, 400, fbar=fbar)
        assert r.reason > 0 and rm.reason > 0 and ra.reason > 0, (r, rm, ra)
        assert (x - m).norm().item() <= 1e-8 * x.norm().item()
        out.append((r, ra, x, lam, mu))
    for k in (0, 1):
        assert out[0][k].reason == out[1][k].reason and abs(out[0][k].its - out[1][k].its) <= 1
    for k in (2, 3, 4):
        assert (out[0][k] - out[1][k]).norm().item() <= 1e-9 * out[1][k].norm().item(), k


def test_potential_form_of_a_prime_length(cuda):
    """nv prime: the potential form's lines along v."""
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    nx, nv = 40, 251
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.02)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.02), preconditioner='tensor_potential')
    phi = 0.3 * np.cos(np.arange(nx) * 2 * np.pi / nx)
    ctx.precond_update(torch.from_numpy(phi).to(cuda))
    x = np.random.default_rng(2).standard_normal((nx, nv))
    ref = O.PotentialPreconditioner(g, phi, 'lapack').apply(x)
    y = ctx.new_field()
    ctx.precond(torch.from_numpy(np.ascontiguousarray(x.T)).to(cuda), y)
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
