"""The factored bracket in FP64 (SepWin, arakawa.h) against the stencils evaluated in
extended precision.  The transposed linearisation with f_bar = 0 has no coupling
left, so y = u/dt - 1/2 {u~, H} on all rows, u~ = u on rows 2..nv-3 and 0 elsewhere,
is what bracket_pair_kernel forms by row and column coefficients.  One tile and its
remainders (63 | 64 | 65 columns, 15 | 16 | 17 rows), grids narrower than a tile,
several tiles.

Bar as in test_gpu_sep_bracket: a coefficient is at most six roundings from exact, a
product and the sum of the eight add two and three more, a difference of F one: 12 eps
(2 max|u|) sum|coefficient|, sum|A| <= (4 c1 + 5 c2) max|H(2 cells) difference|; phi's
own rounding (4 eps max|phi| a difference) and u / dt, two roundings.
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu

LD = np.longdouble
GRIDS = [(8, 9), (9, 33), (63, 15), (64, 16), (65, 17), (130, 50), (512, 41), (1024, 20)]


def _bracket(kind, f, h, hx, hv):
    """{f, h} of (nx, nv) arrays, both axes wrapped (f is 0 on the first and last two rows)."""
    F = lambda i, j: np.roll(np.roll(f, -i, 0), -j, 1)
    H = lambda i, j: np.roll(np.roll(h, -i, 0), -j, 1)
    out = np.zeros_like(f)
    if kind != 'arakawaj2':
        t = ((F(1, 0) - F(-1, 0)) * (H(0, 1) - H(0, -1)) - (F(0, 1) - F(0, -1)) * (H(1, 0) - H(-1, 0))
             + F(1, 0) * (H(1, 1) - H(1, -1)) - F(-1, 0) * (H(-1, 1) - H(-1, -1))
             - F(0, 1) * (H(1, 1) - H(-1, 1)) + F(0, -1) * (H(1, -1) - H(-1, -1))
             + F(1, 1) * (H(0, 1) - H(1, 0)) - F(-1, -1) * (H(-1, 0) - H(0, -1))
             - F(-1, 1) * (H(0, 1) - H(-1, 0)) + F(1, -1) * (H(1, 0) - H(0, -1)))
        out += (2 if kind == 'arakawaj4' else 1) * t / (12 * hx * hv)
    if kind != 'arakawaj1':
        t = ((F(1, 1) - F(-1, -1)) * (H(-1, 1) - H(1, -1)) - (F(-1, 1) - F(1, -1)) * (H(1, 1) - H(-1, -1))
             + F(2, 0) * (H(1, 1) - H(1, -1)) - F(-2, 0) * (H(-1, 1) - H(-1, -1))
             - F(0, 2) * (H(1, 1) - H(-1, 1)) + F(0, -2) * (H(1, -1) - H(-1, -1))
             + F(1, 1) * (H(0, 2) - H(2, 0)) - F(-1, -1) * (H(-2, 0) - H(0, -2))
             - F(-1, 1) * (H(0, 2) - H(-2, 0)) + F(1, -1) * (H(2, 0) - H(0, -2)))
        out += (-1 if kind == 'arakawaj4' else 1) * t / (24 * hx * hv)
    return out


@pytest.mark.parametrize("nx,nv", GRIDS)
@pytest.mark.parametrize("kind", ['arakawaj1', 'arakawaj2', 'arakawaj4'])
def test_against_extended_precision(nx, nv, kind, cuda):
    import torch
    from vivlasov1d_amd.core import Grid as PGrid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, kind, flush=True)
    rng = np.random.default_rng(nx + 5 * nv)
    g = O.Grid(nx, nv, 4 * np.pi, 8.0, ht=0.05)
    ctx = Context(PGrid(nx, nv, 4 * np.pi, 8.0, ht=0.05), bracket=kind)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    h0 = O.kinetic_hamiltonian(g)
    hs = [0.3 * rng.standard_normal(nx) for _ in range(4)]
    ctx.set_hamiltonian(T(h0), *[T(h) for h in hs])
    phi = sum(LD(0.5) * h.astype(LD) for h in hs)
    u = rng.standard_normal((nx, nv))
    y = ctx.new_field()
    ctx.linear_apply(T(u.T), y, 'AT', ctx.new_field().zero_())
    um = u.astype(LD)
    um[:, :2] = 0
    um[:, -2:] = 0
    H = h0.astype(LD)[None, :] + phi[:, None]
    ref = u.astype(LD) / LD(g.ht) - LD(0.5) * _bracket(kind, um, H, LD(g.hx), LD(g.hv))
    eps, fmax = 2.0 ** -53, np.abs(u).max()
    c1 = (2 if kind == 'arakawaj4' else 1 if kind == 'arakawaj1' else 0) * 0.5 / (12 * g.hx * g.hv)
    c2 = (0 if kind == 'arakawaj1' else 1) * 0.5 / (24 * g.hx * g.hv)
    dv = np.abs(h0[2:] - h0[:-2]).max()
    dx = float(np.abs(np.roll(phi, -2) - phi).max()) + float(np.abs(np.roll(phi, -1) - phi).max())
    W = (4 * c1 + 5 * c2) * 2 * fmax
    bar = 12 * eps * W * (dv + dx) + W * 4 * eps * float(np.abs(phi).max()) + 2 * eps * 2 * fmax / g.ht
    err = np.abs(y.cpu().numpy().T - ref).max()
    assert err <= bar, (err, bar)
