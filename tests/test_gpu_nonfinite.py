"""An infinity or NaN reaches the points whose stencil holds it and no others:
the factored bracket (J u of the FP32 cycle, compared with the oracle's J u) for
each kind, one bad value of u or of the Hamiltonian's factors at a time, inside
a tile, at its edges and at the periodic seam.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


def _ctx(nx, nv, kind, hs, h0, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.05), bracket=kind)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    ctx.set_hamiltonian(T(h0), *[T(h) for h in hs])
    return ctx, T


def _finite(ctx, T, u, nx, nv, cuda):
    import torch
    y = torch.empty(nv, nx, dtype=torch.float32, device=cuda)
    ctx.jacobian_apply32(T(u.T).float(), y)
    return np.isfinite(y.cpu().numpy().T)


@pytest.mark.parametrize("kind", ['arakawaj1', 'arakawaj2', 'arakawaj4'])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_nonfinite_u(kind, bad, cuda):
    nx, nv = 70, 40
    print("case", kind, bad, flush=True)
    rng = np.random.default_rng(5)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    h0, hs = O.kinetic_hamiltonian(g), [0.3 * rng.standard_normal(nx) for _ in range(4)]
    ctx, T = _ctx(nx, nv, kind, hs, h0, cuda)
    H = O.h_average(h0, *hs)
    for i, j in [(20, 8), (63, 15), (64, 16), (0, 2), (69, 37), (1, 20), (30, 1)]:
        u = rng.standard_normal((nx, nv))
        u[i, j] = bad
        with np.errstate(invalid='ignore'):
            ref = np.isfinite(O.jacobian(kind, u, H, g))
        assert np.array_equal(_finite(ctx, T, u, nx, nv, cuda), ref), (i, j)


@pytest.mark.parametrize("kind", ['arakawaj1', 'arakawaj2', 'arakawaj4'])
def test_nonfinite_hamiltonian(kind, cuda):
    nx, nv = 70, 40
    print("case", kind, flush=True)
    rng = np.random.default_rng(6)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    u = rng.standard_normal((nx, nv))
    for where in [('x', 20), ('x', 63), ('x', 0), ('x', 69), ('v', 8), ('v', 15), ('v', 16), ('v', 37)]:
        h0, hs = O.kinetic_hamiltonian(g), [0.3 * rng.standard_normal(nx) for _ in range(4)]
        if where[0] == 'x':
            hs[1][where[1]] = np.nan
        else:
            h0[where[1]] = np.nan
        ctx, T = _ctx(nx, nv, kind, hs, h0, cuda)
        with np.errstate(invalid='ignore'):
            ref = np.isfinite(O.jacobian(kind, u, O.h_average(h0, *hs), g))
        assert np.array_equal(_finite(ctx, T, u, nx, nv, cuda), ref), where
