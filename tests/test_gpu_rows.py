"""Row-block kernels (any x-length up to 2048) and the mixed-radix transform at
the edges of their ranges: row groups of short grids (8, 9, 85, 128, 129), one
strip and several (256 | 257, 500), primes (11, 211), long radices (201 = 3 x
67), the longest lines (1999 prime, 2000, 2047, 2048), ragged last blocks (odd
nv), pairs that end on an odd element (odd nx x odd nv).

Bars: P^-1 F, P^-1 J u within 1e-12 of the oracle as test_gpu_parity's, the
transform itself within 16 eps sqrt(sum of radices) of numpy's per the usual
growth of a direct sum, far inside 1e-12; GMRES solves fused and separate
within 1e-9 (rtol 1e-10).
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu

GRIDS = [(8, 9), (9, 9), (11, 33), (64, 128), (85, 67), (128, 256), (129, 35), (201, 101), (211, 40), (256, 61),
         (257, 64), (500, 33), (1999, 12), (2000, 64), (2047, 9), (2048, 35)]


def _nat(a):
    return np.ascontiguousarray(a.T)


def _setup(nx, nv, kind, cuda, restart=30, hx=None):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    rng = np.random.default_rng(nx + 3 * nv)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.05), bracket=kind, charge=-1.0, restart=restart)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    h0 = O.kinetic_hamiltonian(g)
    hs = [0.02 * rng.standard_normal(nx) for _ in range(4)]
    ctx.set_hamiltonian(T(h0), *[T(h) for h in hs])
    return g, ctx, O.h_average(h0, *hs), rng, T


@pytest.mark.parametrize("nx,nv", GRIDS)
def test_function_and_jacobian(nx, nv, cuda):
    kind = ['arakawaj1', 'arakawaj2', 'arakawaj4'][(nx + nv) % 3]
    print("case", nx, nv, kind, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, kind, cuda)
    pc = O.Preconditioner(g, 'lapack')
    f = rng.random((nx, nv))
    fh = f + 0.01 * rng.standard_normal((nx, nv))
    u = rng.standard_normal((nx, nv))
    y = ctx.new_field()
    ctx.function(T(_nat(f)), T(_nat(fh)), y)
    ref = pc.apply(O.residual(kind, f, fh, H, g))
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    ctx.jacobian(T(_nat(u)), y)
    ref = pc.apply(O.jacobian(kind, u, H, g))
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    ctx.precond(T(_nat(u)), y)
    ref = pc.apply(u)
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    # an output that is not aligned for pairs
    import torch
    buf = torch.zeros(nx * nv + 1, dtype=torch.float64, device=cuda)
    ctx.precond(T(_nat(u)), buf[1:])
    assert np.abs(buf[1:].cpu().numpy().reshape(nv, nx).T - ref).max() <= 1e-12 * np.abs(ref).max()
    assert buf[0].item() == 0.0


@pytest.mark.parametrize("nx,nv", GRIDS)
@pytest.mark.parametrize("coll", ['', 'collt', 'colle'])
def test_gmres_fused_and_separate(nx, nv, coll, cuda):
    """The same solve through the row blocks and through separate launches; a
    smooth right-hand side, so that both converge in a cycle or two."""
    import torch
    print("case", nx, nv, coll, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, 'arakawaj4', cuda)
    f = np.exp(-0.5 * g.v ** 2)[None, :] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(nx) / nx))[:, None]
    f[:, :2] = 0
    f[:, -2:] = 0
    if coll:
        n, U, e = O.density(f, g), O.velocity_density(f, g), O.energy_density(f, g)
        dev = [T(x) for x in (n, U, e, O.collision_factor(n, U, e))] * 2
        ctx.set_moments(*dev)
        ctx.set_dissipation(coll, 1e-3, 1.1, 0.9)
    b = T(_nat(f * np.sin(3 * g.v)[None, :]))
    out = []
    for on in (True, False):
        ctx.set_fusion(on)
        x = ctx.new_field()
        res = ctx.ksp_solve(b, x, 1e-10, 1e-50, 1e5, 300)
        out.append((res.its, res.reason, x))
    assert out[0][1] == out[1][1] and abs(out[0][0] - out[1][0]) <= 1, out[:2]
    if out[0][1] > 0:
        err = (out[0][2] - out[1][2]).norm().item() / out[1][2].norm().item()
        assert err <= 1e-9, err


@pytest.mark.parametrize("nx,nv", [(9, 9), (64, 128), (128, 50), (201, 101), (2048, 35)])
def test_fp32_preconditioner_and_cycle(nx, nv, cuda):
    """FP32 lines: P^-1 within the FP32 bar of test_gpu_general_grids (2e-6), and
    a mixed solve refined to the FP64 tolerance."""
    import torch
    print("case", nx, nv, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, 'arakawaj4', cuda)
    pc = O.Preconditioner(g, 'lapack')
    u = rng.standard_normal((nx, nv)).astype(np.float32).astype(np.float64)
    xf = T(_nat(u)).float()
    yf = torch.empty_like(xf)
    ctx.precond32(xf, yf)
    ref = pc.apply(u)
    assert np.abs(yf.double().cpu().numpy().T - ref).max() <= 2e-6 * np.abs(ref).max()
    f = np.exp(-0.5 * g.v ** 2)[None, :] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(nx) / nx))[:, None]
    b = T(_nat(f * np.sin(3 * g.v)[None, :]))
    x64, x32 = ctx.new_field(), ctx.new_field()
    r64 = ctx.ksp_solve(b, x64, 1e-10, 1e-50, 1e5, 300)
    r32, _ = ctx.ksp_solve_mixed(b, x32, 1e-10, 1e-50, 1e5, 600)
    assert r64.reason == r32.reason
    if r64.reason > 0:
        assert (x64 - x32).norm().item() <= 1e-8 * x64.norm().item()


def test_batched_equals_single(cuda):
    """Instances of a batched context on the row blocks: bit for bit the single
    instances', whatever rows a workgroup takes."""
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    nx, nv, B = 128, 256, 5
    rng = np.random.default_rng(3)
    Ls = [4 * np.pi / s for s in (1.0, 1.3, 0.7, 2.0, 1.1)]
    grids = [PGrid(nx, nv, L, 8.0, ht=0.05) for L in Ls]
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    h0 = T(0.5 * grids[0].v ** 2)
    h = [0.1 * rng.standard_normal((B, nx)) for _ in range(4)]
    prof = np.exp(-0.5 * grids[0].v ** 2) * np.sin(2 * grids[0].v)
    b = np.stack([prof[:, None] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(nx) / nx + q))[None, :] for q in range(B)])
    cb = Context(grids[0], hx=[g.hx for g in grids])
    cb.set_hamiltonian(h0, *[T(x) for x in h])
    xb = cb.new_field()
    rb = cb.ksp_solve(T(b), xb, 1e-10, 1e-50, 1e5, 200)
    for q in range(B):
        c1 = Context(grids[q])
        c1.set_hamiltonian(h0, *[T(x[q]) for x in h])
        x1 = c1.new_field()
        r1 = c1.ksp_solve(T(b[q]), x1, 1e-10, 1e-50, 1e5, 200)
        assert (rb[q].its, rb[q].reason) == (r1.its, r1.reason)
        assert torch.equal(xb[q], x1), q
