"""Tridiagonal solves and the transposed operators at the edges of their
kernels' ranges.

* potential preconditioner: chunks of 2, 4, 8 rows a lane (128 | 129, 256 |
  257, 512) and the workgroup form beyond (513), the column transforms (even
  nx, aligned) and the transposing path (odd nx, a misaligned field);
* P^-T of the kinetic form from the forward pivots, one to sixteen rows a
  thread;
* the transposed linearisation's bracket pair on ragged tiles.

Bars: 1e-12 relative against the oracle (test_gpu_potential's); dot products
<P u, v> = <u, P^T v> and <A u, v> = <u, A^T v> to 1e-12 of the norms
(test_gpu_adjoint's).
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


def _nat(a):
    return np.ascontiguousarray(a.T)


def _ctx(nx, nv, cuda, precond='tensor_kinetic', kind='arakawaj4', hx=None):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    g = O.Grid(nx, nv, 4 * np.pi, 8.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 8.0, ht=0.05), bracket=kind, preconditioner=precond, charge=-1.0, hx=hx)
    return g, ctx, (lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda))


@pytest.mark.parametrize("nx,nv", [(8, 64), (9, 16), (64, 1024), (127, 32), (128, 8), (129, 64), (130, 2048),
                                   (256, 128), (257, 64), (512, 256), (512, 4096), (513, 32), (514, 64), (1030, 16)])
def test_potential_preconditioner(nx, nv, cuda):
    import torch
    print("case", nx, nv, flush=True)
    g, ctx, T = _ctx(nx, nv, cuda, 'tensor_potential')
    rng = np.random.default_rng(nx + nv)
    phi = 0.3 * np.cos(np.arange(nx) * 2 * np.pi / nx) + 0.02 * rng.standard_normal(nx)
    ctx.precond_update(T(phi))
    pc = O.PotentialPreconditioner(g, phi, 'lapack')
    x = rng.standard_normal((nx, nv))
    ref = pc.apply(x)
    y = ctx.new_field()
    ctx.precond(T(_nat(x)), y)
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    buf = torch.zeros(nx * nv + 1, dtype=torch.float64, device=cuda)
    buf[1:] = T(_nat(x)).reshape(-1)
    ctx.precond(buf[1:], buf[1:])                    # misaligned, in place
    assert np.abs(buf[1:].cpu().numpy().reshape(nv, nx).T - ref).max() <= 1e-12 * np.abs(ref).max()
    u, v = T(rng.standard_normal((nv, nx))), T(rng.standard_normal((nv, nx)))
    Pu, PTv = ctx.new_field(), ctx.new_field()
    ctx.precond(u, Pu)
    ctx.precond_t(v, PTv)
    assert abs((v * Pu).sum().item() - (PTv * u).sum().item()) <= 1e-12 * v.norm().item() * Pu.norm().item()


@pytest.mark.parametrize("nx,nv", [(8, 8), (64, 255), (64, 257), (32, 512), (100, 513), (16, 1025), (64, 2049),
                                   (16, 4096)])
def test_kinetic_transposed(nx, nv, cuda):
    print("case", nx, nv, flush=True)
    g, ctx, T = _ctx(nx, nv, cuda)
    rng = np.random.default_rng(nx * nv)
    u, v = T(rng.standard_normal((nv, nx))), T(rng.standard_normal((nv, nx)))
    Pu, PTv = ctx.new_field(), ctx.new_field()
    ctx.precond(u, Pu)
    ctx.precond_t(v, PTv)
    assert abs((v * Pu).sum().item() - (PTv * u).sum().item()) <= 1e-12 * v.norm().item() * Pu.norm().item()


@pytest.mark.parametrize("nx,nv", [(9, 9), (65, 33), (130, 50), (256, 100), (201, 41), (64, 16)])
@pytest.mark.parametrize("kind", ['arakawaj1', 'arakawaj2', 'arakawaj4'])
def test_transposed_linearisation(nx, nv, kind, cuda):
    import torch
    print("case", nx, nv, kind, flush=True)
    g, ctx, T = _ctx(nx, nv, cuda, kind=kind)
    rng = np.random.default_rng(nx + nv)
    h = [0.1 * rng.standard_normal(nx) for _ in range(4)]
    ctx.set_hamiltonian(T(O.kinetic_hamiltonian(g)), *[T(a) for a in h])
    u, v, fbar = (T(rng.standard_normal((nv, nx))) for _ in range(3))
    y, z = ctx.new_field(), ctx.new_field()
    for fwd, bwd in (('A', 'AT'), ('A0', 'A0T')):
        ctx.linear_apply(u, y, fwd, fbar)
        ctx.linear_apply(v, z, bwd, fbar)
        assert abs((v * y).sum().item() - (z * u).sum().item()) <= 1e-12 * v.norm().item() * y.norm().item()
    # the reverse step through the fused launches and through separate ones, a
    # right-hand side that GMRES solves in a few cycles
    f = np.exp(-0.5 * g.v ** 2)[:, None] * (1 + 0.1 * np.cos(2 * np.pi * np.arange(nx) / nx))[None, :]
    ctx.set_hamiltonian(T(O.kinetic_hamiltonian(g)), *[T(0.1 * a) for a in h])
    lam = T(f * np.sin(2 * g.v)[:, None])
    out = []
    for on in (True, False):
        ctx.set_fusion(on)
        lam0, mu = ctx.new_field(), ctx.new_field()
        r = ctx.adjoint_step(lam, lam0, mu, 1e-11, 1e-300, 1e5, 400, fbar=T(f))
        out.append((r.its, r.reason, lam0, mu))
    assert out[0][1] == out[1][1] and abs(out[0][0] - out[1][0]) <= 1, out
    if out[0][1] > 0:
        assert (out[0][2] - out[1][2]).norm().item() <= 1e-9 * out[1][2].norm().item()
        assert (out[0][3] - out[1][3]).norm().item() <= 1e-9 * out[1][3].norm().item()
