"""The right-hand side P^-1 F of a Newton step whose solve restarts: formed once
where the solve's start leaves it in its buffer (long and unfused transforms, no
preconditioner), and the step is the linear solve's with that right-hand side.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nv,pc,fuse,once", [(2048, 24, 'tensor_kinetic', True, True),
                                                (2500, 20, 'tensor_kinetic', True, True),
                                                (257, 24, 'tensor_kinetic', True, True),
                                                (64, 96, 'tensor_kinetic', False, True),
                                                (64, 96, None, True, True),
                                                (64, 128, 'tensor_potential', True, True),
                                                (64, 96, 'tensor_kinetic', True, False),
                                                (256, 64, 'tensor_kinetic', True, False)])
def test_right_hand_side(nx, nv, pc, fuse, once, cuda):
    import torch
    from vivlasov1d_amd.core import Grid, kinetic_hamiltonian
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, pc, fuse, flush=True)
    rng = np.random.default_rng(nx)
    ht = 0.002 if nx > 1024 else 0.02       # a few cycles of three steps
    g = Grid(nx, nv, 4 * np.pi, 6.0, ht=ht)
    ctx = Context(g, charge=-1.0, restart=3, preconditioner=pc)
    ctx.set_fusion(fuse)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    x, v = np.arange(nx) * 2 * np.pi / nx, np.asarray(g.v)
    ctx.set_hamiltonian(T(kinetic_hamiltonian(g)), *[T(0.02 * rng.standard_normal(nx)) for _ in range(4)])
    if pc == 'tensor_potential':
        ctx.precond_update(T(0.1 * np.cos(x)))
    f0 = np.exp(-0.5 * v * v)[:, None] * (1 + 0.1 * np.cos(x))[None, :]
    f, fh = T(f0), T(f0 * (1 + 0.01 * np.sin(2 * v))[:, None])
    b, d = ctx.new_field(), ctx.new_field()
    ctx.function(f, fh, b)
    rk = ctx.ksp_solve(b, d, 1e-9, 1e-50, 1e5, 400)
    ref = f - d
    ctx.profile(("residual",))
    rs = ctx.snes_ksponly(f, fh, 1e-9, 1e-50, 1e5, 400)
    n = ctx.profile_read("residual")[1]
    ctx.profile(())
    assert rk.reason > 0 and rk.its > 3, (rk.its, rk.reason)       # more than one cycle
    assert rs.reason == rk.reason and abs(rs.its - rk.its) <= 1
    assert (f - ref).norm().item() <= 1e-8 * d.norm().item()
    assert n == (1 if once else 2)
