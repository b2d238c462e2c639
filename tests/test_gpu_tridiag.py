"""The kinetic preconditioner's pivoted solve at the edges of its forms: 64, 128
or 256 threads a mode, one to sixteen rows a thread, the last chunk full, with
one row, or empty; P^-1 and P^-T in FP64, P^-1 in FP32.

Bars: 1e-12 of the largest value against the LAPACK oracle (FP64: the systems
are diagonally dominant, so the rounding of nv-step recurrences does not grow);
FP32 2e-6 of it (the FP32 transforms' bar in the other tests, 2^-24 = 6e-8 times some tens of roundings).
P^-T: <P^-1 u, v> = <u, P^-T v> to 1e-12 of the norms.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv", [8, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047,
                                2048, 2049, 4095, 4096])
@pytest.mark.parametrize("nx", [16, 9])
def test_kinetic_solve(nx, nv, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, flush=True)
    g = O.Grid(nx, nv, 4 * np.pi, 8.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 8.0, ht=0.05))
    rng = np.random.default_rng(nx * nv)
    x = rng.standard_normal((nx, nv))
    ref = O.Preconditioner(g).apply(x)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a.T)).to(cuda)
    u, y = T(x), ctx.new_field()
    ctx.precond(u, y)
    assert np.abs(y.cpu().numpy().T - ref).max() <= 1e-12 * np.abs(ref).max()
    v, z = T(rng.standard_normal((nx, nv))), ctx.new_field()
    ctx.precond_t(v, z)
    assert abs((v * y).sum().item() - (z * u).sum().item()) <= 1e-12 * v.norm().item() * y.norm().item()
    y32 = torch.empty_like(u, dtype=torch.float32)
    ctx.precond32(u.float(), y32)
    assert np.abs(y32.double().cpu().numpy().T - ref).max() <= 2e-6 * np.abs(ref).max()
