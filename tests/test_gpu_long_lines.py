"""Transforms of the longest power-of-two lines (2048 = 4 x 8 x 8 x 8, 4096 = 8 x 8 x
8 x 8; swizzled LDS) and spectra whose rows are padded: one and several row blocks,
a ragged last one, row counts around the padding (15 | 16 | 17, 32), and rows
per workgroup that are no power of two.

P^-1 x and P^-1 J u against the oracle, FP64 within 1e-12 and FP32 within 2e-6
relative as elsewhere.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


def _setup(nx, nv, cuda, **kw):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    rng = np.random.default_rng(nx + 3 * nv)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.05), charge=-1.0, **kw)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    h0 = O.kinetic_hamiltonian(g)
    hs = [0.02 * rng.standard_normal(nx) for _ in range(4)]
    ctx.set_hamiltonian(T(h0), *[T(h) for h in hs])
    return g, ctx, O.h_average(h0, *hs), rng, T


@pytest.mark.parametrize("nx,nv", [(2048, 15), (2048, 33), (4096, 9), (4096, 16), (4096, 17)])
def test_kinetic(nx, nv, cuda):
    import torch
    print("case", nx, nv, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, cuda)
    pc = O.Preconditioner(g, 'lapack')
    u = rng.standard_normal((nx, nv))
    y = ctx.new_field()
    ctx.precond(T(u.T), y)
    ref = pc.apply(u)
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    ctx.jacobian(T(u.T), y)
    ref = pc.apply(O.jacobian('arakawaj4', u, H, g))
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    u32 = u.astype(np.float32)
    y32 = torch.empty(nv, nx, dtype=torch.float32, device=cuda)
    ctx.precond32(T(u32.T), y32)
    ref = pc.apply(u32.astype(np.float64))
    assert np.abs(y32.double().cpu().numpy().T - ref).max() <= 2e-6 * np.abs(ref).max()


@pytest.mark.parametrize("nx,nv,rows", [(64, 31, 6), (256, 32, 10), (1024, 17, 6), (2048, 16, 2)])
def test_rows_per_workgroup(nx, nv, rows, cuda):
    print("case", nx, nv, rows, flush=True)
    g, ctx, H, rng, T = _setup(nx, nv, cuda)
    ctx.set_tuning(rows, 0)
    u = rng.standard_normal((nx, nv))
    y = ctx.new_field()
    ctx.precond(T(u.T), y)
    ref = O.Preconditioner(g, 'lapack').apply(u)
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
