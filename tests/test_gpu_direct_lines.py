"""P^-1 on both sides of the lines between the direct real DFT and the row blocks
of composite lengths: 64 points (rFFT), 96 (irFFT), 2^23 products.  FP64 within
1e-12 and FP32 2e-6 of the oracle, aligned output and not, in place; the
potential form's lines along v; a batched context against single ones, to the bit.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


def _check(ctx, pc, nx, nv, cuda):
    import torch
    rng = np.random.default_rng(nx + nv)
    x = rng.standard_normal((nx, nv))
    ref = pc.apply(x)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a.T)).to(cuda)
    for off in (0, 1):
        buf = torch.zeros(nx * nv + off, dtype=torch.float64, device=cuda)
        buf[off:] = T(x).reshape(-1)
        ctx.precond(buf[off:], buf[off:])
        assert np.abs(buf[off:].cpu().numpy().reshape(nv, nx).T - ref).max() <= 1e-12 * np.abs(ref).max()
    y32 = torch.empty(nv, nx, dtype=torch.float32, device=cuda)
    ctx.precond32(T(x).float(), y32)
    assert np.abs(y32.double().cpu().numpy().T - ref).max() <= 2e-6 * np.abs(ref).max()


# 63^2 x 2113 <= 2^23 < 63^2 x 2114, 96^2 x 910 <= 2^23 < 96^2 x 911
@pytest.mark.parametrize("nx,nv", [(18, 40), (63, 41), (63, 2113), (63, 2114), (65, 41), (96, 40), (96, 910),
                                   (96, 911), (98, 41)])
def test_kinetic(nx, nv, cuda):
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, flush=True)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    _check(Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.05)), O.Preconditioner(g, 'lapack'), nx, nv, cuda)


@pytest.mark.parametrize("nx,nv", [(40, 63), (41, 66), (40, 96), (40, 98), (2114, 63)])
def test_potential(nx, nv, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, flush=True)
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 6.0, ht=0.05), preconditioner='tensor_potential')
    phi = 0.3 * np.cos(np.arange(nx) * 2 * np.pi / nx)
    ctx.precond_update(torch.from_numpy(phi).to(cuda))
    _check(ctx, O.PotentialPreconditioner(g, phi, 'lapack'), nx, nv, cuda)


@pytest.mark.parametrize("nx,nv,B", [(60, 256, 9), (60, 256, 10), (90, 64, 3)])
def test_batched(nx, nv, B, cuda):
    """60^2 x 256 x 9 <= 2^23 < 60^2 x 256 x 10: each instance within 1e-12 of its oracle."""
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, B, flush=True)
    Ls = [4 * np.pi * (1 + 0.1 * b) for b in range(B)]
    ctx = Context(PGrid(nx, nv, Ls[0], 6.0, ht=0.05), hx=[L / nx for L in Ls])
    x = np.random.default_rng(B).standard_normal((B, nv, nx))
    y = ctx.new_field()
    ctx.precond(torch.from_numpy(x).to(cuda), y)
    y = y.cpu().numpy()
    for b, L in enumerate(Ls):
        ref = O.Preconditioner(O.Grid(nx, nv, L, 6.0, ht=0.05), 'lapack').apply(x[b].T)
        assert np.abs(y[b].T - ref).max() <= 1e-12 * np.abs(ref).max(), b
