"""A context after a solve that failed half way: a collision operator without
moments is an error once the first Arnoldi step needs them, with the cycle's
start already due.  What the context computes next is what a fresh one does, to
the bit: P^-1 J u, P^-1 F, and the same solve with the moments set.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


def _setup(nx, nv, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    rng = np.random.default_rng(nx + nv)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.05), charge=-1.0)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    ctx.set_hamiltonian(T(O.kinetic_hamiltonian(g)), *[T(0.02 * rng.standard_normal(nx)) for _ in range(4)])
    f = np.exp(-0.5 * g.v ** 2)[None, :] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(nx) / nx))[:, None]
    n, U, e = O.density(f, g), O.velocity_density(f, g), O.energy_density(f, g)
    mom = [T(x) for x in (n, U, e, O.collision_factor(n, U, e))] * 2
    return ctx, T(f.T), T((f * np.sin(3 * g.v)[None, :]).T), mom


@pytest.mark.parametrize("nx,nv", [(64, 96), (201, 101), (256, 64), (512, 33), (1024, 32)])
@pytest.mark.parametrize("solve", ['ksp', 'mixed'])
def test_context_after_a_failed_solve(nx, nv, solve, cuda):
    import torch
    from vivlasov1d_amd._lib import VVError
    print("case", nx, nv, solve, flush=True)
    ctx, f, b, mom = _setup(nx, nv, cuda)
    fresh = _setup(nx, nv, cuda)[0]
    args = (1e-10, 1e-50, 1e5, 300)
    ctx.set_dissipation('collt', 1e-3)
    with pytest.raises(VVError, match="set_moments"):
        if solve == 'ksp':
            ctx.ksp_solve(b, ctx.new_field(), *args)
        else:
            ctx.ksp_solve_mixed(b, ctx.new_field(), *args)
    ctx.set_dissipation(None)
    y, z = ctx.new_field(), ctx.new_field()
    ctx.jacobian(b, y)
    fresh.jacobian(b, z)
    assert torch.equal(y, z)
    ctx.function(f, b, y)
    fresh.function(f, b, z)
    assert torch.equal(y, z)
    for c in (ctx, fresh):
        c.set_moments(*mom)
        c.set_dissipation('collt', 1e-3)
    ctx.jacobian(b, y)
    fresh.jacobian(b, z)
    assert torch.equal(y, z)
    r, s = ctx.ksp_solve(b, y, *args), fresh.ksp_solve(b, z, *args)
    assert s.reason > 0 and (r.its, r.reason, r.rnorm) == (s.its, s.reason, s.rnorm)
    assert torch.equal(y, z)
