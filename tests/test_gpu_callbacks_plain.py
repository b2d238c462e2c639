"""Without a preconditioner P^-1 F and P^-1 J u are F and J u, and are returned in
the reference's operation order as residual and jacobian_apply return them: bit
for bit the oracle's, aliased output included.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nv", [(9, 9), (64, 128), (65, 17), (256, 33), (2048, 15)])
@pytest.mark.parametrize("kind", ['arakawaj1', 'arakawaj2', 'arakawaj4'])
def test_function_and_jacobian_without_preconditioner(nx, nv, kind, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, kind, flush=True)
    rng = np.random.default_rng(nx + nv)
    g = O.Grid(nx, nv, 4 * np.pi, 8.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 8.0, ht=0.05), bracket=kind, preconditioner=None)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    h0, hs = O.kinetic_hamiltonian(g), [0.3 * rng.standard_normal(nx) for _ in range(4)]
    ctx.set_hamiltonian(T(h0), *[T(h) for h in hs])
    H = O.h_average(h0, *hs)
    f, fh = rng.standard_normal((2, nx, nv))
    y = ctx.new_field()
    ctx.function(T(f.T), T(fh.T), y)
    ref = O.residual(kind, f, fh, H, g)
    assert np.array_equal(y.cpu().numpy().T, ref)
    w = T(f.T)
    ctx.function(w, T(fh.T), w)
    assert np.array_equal(w.cpu().numpy().T, ref)
    ref = O.jacobian(kind, f, H, g)
    ctx.jacobian(T(f.T), y)
    assert np.array_equal(y.cpu().numpy().T, ref)
    w = T(f.T)
    ctx.jacobian(w, w)
    assert np.array_equal(w.cpu().numpy().T, ref)
