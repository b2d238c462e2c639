"""The captured GMRES cycle in parts: cycles of one step, of less than a part, of
whole parts and one step more, and solves that end at each step around a part's
end, restarts included.  Replayed (twice from the captured parts, the later
parts first captured in a later solve) and eager solves run the same kernels in
the same order, so iterations, reasons, residual norms and states are equal to
the bit.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LS = (4 * np.pi, 5 * np.pi, 3 * np.pi)


@pytest.mark.parametrize("nx,nv", [(64, 96), (256, 64)])        # row blocks; strips
@pytest.mark.parametrize("restart", [1, 2, 5, 6, 7, 12, 13, 30, 64])
def test_parts(nx, nv, restart, cuda):
    import torch
    from vivlasov1d_amd.core import Grid, kinetic_hamiltonian
    from vivlasov1d_amd.solvers import Context
    print("case", nx, nv, restart, flush=True)
    rng = np.random.default_rng(nx + restart)
    g = Grid(nx, nv, LS[0], 8.0, ht=0.05)
    B = len(LS)
    x = np.arange(nx) * 2 * np.pi / nx
    v = np.asarray(g.v)
    f0 = np.stack([np.exp(-0.5 * v * v)[:, None] * (1 + a * np.cos(x))[None, :] for a in (0.01, 0.1, 0.3)])
    h1 = [0.1 * np.stack([np.cos(x + p) for p in rng.uniform(0, 6, B)]) for _ in range(4)]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
        ce, cg = (Context(g, charge=-1.0, hx=[L / nx for L in LS], restart=restart, stream=stream.cuda_stream)
                  for _ in range(2))
        h0 = T(kinetic_hamiltonian(g))
        for c in (ce, cg):
            c.set_hamiltonian(h0, *(T(h) for h in h1))
        cg.set_graph(True)
        fh = T(f0 * (1 + 1e-3 * rng.standard_normal(f0.shape)))
        fe, fg = T(f0), T(f0)
        its = set()
        for rtol in (1e-2, 1e-5, 1e-10, 1e-13, 1e-10, 1e-3, 1e-7):
            for _ in range(2):
                fe.copy_(T(f0))
                fg.copy_(T(f0))
                re = ce.snes_ksponly(fe, fh, rtol, 1e-50, 1e5, 200)
                rg = cg.snes_ksponly(fg, fh, rtol, 1e-50, 1e5, 200)
                assert [(r.its, r.reason, r.rnorm) for r in re] == [(r.its, r.reason, r.rnorm) for r in rg]
                assert torch.equal(fe, fg)
                its.update(r.its for r in re)
        print(sorted(its), flush=True)
