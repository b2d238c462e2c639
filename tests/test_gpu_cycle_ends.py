"""Solves that converge at a given Arnoldi step, and solves that converge at all,
each asserted.

* Captured and eager Newton steps that converge at step k, for every k from 1 to
  14 (the captured cycle comes in parts of six steps: before, at and after a
  part's end), and past a restart: the tolerance is set just above the residual
  that a run stopped at k steps reports.  Iterations, reasons, norms and states
  are equal to the bit.
* Fused and separate launches at the edge sizes of the row blocks and strips:
  FP64, mixed and collisional solves that converge, reason > 0, iterations
  within 1 and solutions within 1e-9 (rtol 1e-10; mixed 1e-8).
"""

import numpy as np
import pytest

from oracle import vlasov_oracle as O

pytestmark = pytest.mark.gpu

LS = (4 * np.pi, 5 * np.pi, 3 * np.pi)


@pytest.mark.parametrize("nx,nv,ht", [(64, 96, 0.1), (129, 36, 0.05), (256, 64, 0.02), (1024, 64, 0.007)])
@pytest.mark.parametrize("B", [0, 3])
@pytest.mark.parametrize("restart", [30, 7])
def test_solves_that_end_at_a_given_step(nx, nv, ht, B, restart, cuda):
    import torch
    from vivlasov1d_amd.core import Grid, kinetic_hamiltonian
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, ht, B, restart, flush=True)
    rng = np.random.default_rng(nx)
    g = Grid(nx, nv, LS[0], 6.0, ht=ht)
    hx = [L / nx for L in LS[:B]] if B else None
    x, v = np.arange(nx) * 2 * np.pi / nx, np.asarray(g.v)
    f0 = np.exp(-0.5 * v * v)[:, None] * (1 + 0.3 * np.cos(x))[None, :]
    fh0 = f0 * (1 + 1e-2 * np.sin(3 * v))[:, None]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        rep = lambda a: np.ascontiguousarray(np.broadcast_to(a, (B,) + a.shape)) if B else a
        T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
        ce, cg = (Context(g, charge=-1.0, hx=hx, restart=restart, stream=stream.cuda_stream) for _ in range(2))
        hs = [T(rep(0.02 * rng.standard_normal(nx))) for _ in range(4)]
        for c in (ce, cg):
            c.set_hamiltonian(T(kinetic_hamiltonian(g)), *hs)
        cg.set_graph(True)
        start, fh = T(rep(f0)), T(rep(fh0))
        fe, fg = start.clone(), start.clone()
        one = lambda r: r[0] if B else r
        for k in range(1, 15):
            fe.copy_(start)
            r = one(ce.snes_ksponly(fe, fh, 1e-30, 1e-300, 1e5, k))
            assert r.its == k and r.reason == -3, (k, r.its, r.reason)
            rtol = 1.001 * r.rnorm / r.rnorm0
            out = []
            for c, f in ((ce, fe), (cg, fg)):
                f.copy_(start)
                rr = c.snes_ksponly(f, fh, rtol, 1e-300, 1e5, 200)
                out.append([(q.its, q.reason, q.rnorm) for q in (rr if B else [rr])])
            assert out[0][0][:2] == (k, 2), (k, out[0])
            assert out[0] == out[1], (k, out)
            assert torch.equal(fe, fg), k


GRIDS = [(8, 9), (9, 9), (11, 33), (64, 128), (85, 67), (128, 256), (129, 35), (201, 101), (256, 61), (257, 64),
         (500, 33), (512, 40), (1024, 40), (2000, 64), (2047, 9), (2048, 35)]


@pytest.mark.parametrize("nx,nv", GRIDS)
@pytest.mark.parametrize("coll", [None, 'collt', 'colle'])
def test_fused_and_separate_solves_converge(nx, nv, coll, cuda):
    from vivlasov1d_amd.core import Grid
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, coll, flush=True)
    rng = np.random.default_rng(nx + 3 * nv)
    ht = 0.05 if nx < 500 else 0.005
    g = O.Grid(nx, nv, 4 * np.pi, 6.0, ht=ht)
    ctx = Context(Grid(nx, nv, 4 * np.pi, 6.0, ht=ht), charge=-1.0)
    import torch
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    ctx.set_hamiltonian(T(O.kinetic_hamiltonian(g)), *[T(0.02 * rng.standard_normal(nx)) for _ in range(4)])
    f = np.exp(-0.5 * g.v ** 2)[None, :] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(nx) / nx))[:, None]
    if coll:
        n, U, e = O.density(f, g), O.velocity_density(f, g), O.energy_density(f, g)
        mom = [T(x) for x in (n, U, e, O.collision_factor(n, U, e))] * 2
        ctx.set_moments(*mom)
        ctx.set_dissipation(coll, 1e-3, 1.1, 0.9)
    b = T((f * np.sin(3 * g.v)[None, :]).T)
    out = []
    for on in (True, False):
        ctx.set_fusion(on)
        x, m = ctx.new_field(), ctx.new_field()
        r = ctx.ksp_solve(b, x, 1e-10, 1e-50, 1e5, 300)
        rm, _ = ctx.ksp_solve_mixed(b, m, 1e-10, 1e-50, 1e5, 600)
        assert r.reason > 0 and rm.reason > 0, (r.reason, r.its, rm.reason, rm.its)
        assert (x - m).norm().item() <= 1e-8 * x.norm().item()
        out.append((r, x))
    assert out[0][0].reason == out[1][0].reason and abs(out[0][0].its - out[1][0].its) <= 1
    assert (out[0][1] - out[1][1]).norm().item() <= 1e-9 * out[1][1].norm().item()
