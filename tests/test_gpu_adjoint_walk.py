"""The reverse kick + drift takes every particle of a tile once, whatever
blocks its walk over a crowded tile is cut into: a container that repeats a few
particles many times against one that holds each of them once.

Tolerances: a particle's own adjoints are the same arithmetic (8 units of the
precision's epsilon).  The field adjoints are r times those of the single
particles: FP64 sums of n terms, up to 8 FP32 roundings where tiles meet and
their own rounding: 16 epsilon (FP32) or 64 n epsilon (FP64, for the order of
the sum) of the largest."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# one workgroup per CU and more, full and partial blocks, one pass, more passes than a block may have
@pytest.mark.parametrize("prec,N,r", [("mixed", 128, 1), ("mixed", 128, 173), ("mixed", 128, 1201), ("mixed", 64, 97),
                                      ("mixed", 32, 13), ("mixed", 32, 647), ("mixed", 16, 41), ("mixed", 4, 9),
                                      ("fp64", 64, 57), ("fp64", 64, 397), ("fp64", 32, 29), ("fp64", 32, 331),
                                      ("fp64", 8, 21), ("fp64", 4, 7)])
def test_repeated_particles(prec, N, r):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm as gp
    ctx = gp.Context(N, gp.GEV_FP64 if prec == "fp64" else gp.GEV_MIXED)
    rng = np.random.default_rng(N + r)
    m = 53
    cell = np.where(rng.random(m) < 0.9, rng.integers(0, 2, (3, m)), rng.integers(0, min(N, 8), (3, m)))
    pos = (cell + np.floor(rng.random((3, m)) * 2 ** 20) / 2 ** 20) / N
    q = rng.normal(0, 0.02, (3, m)).astype(np.float32).astype(np.float64)
    t = lambda c, s: (s * torch.from_numpy(rng.standard_normal((c, N, N, N)))).to(ctx.rdtype).cuda()
    phi, chi, B = t(1, 1e-3), t(1, 1e-3), t(3, 1e-5)
    lx0, lq0 = (torch.from_numpy(rng.standard_normal((3, m))).to(ctx.rdtype).cuda() for _ in range(2))

    def run(copies):
        n = m * copies
        who = rng.permutation(n) % m
        p = gp.Particles(ctx, n, 0.31 / n)
        p.load(pos[:, who], q[:, who], np.arange(n))
        w = torch.from_numpy(who).cuda()
        lx, lq = lx0[:, w].contiguous(), lq0[:, w].contiguous()
        f = [ctx.real(c) for c in (1, 1, 3)]
        p.adj_gr_kick_drift(phi, chi, B, lx, lq, *f, 3, 3, 0.1, 0.102, 0.015, 0.02)
        return w, lx.double(), lq.double(), [v.double() for v in f]

    w1, x1, q1, f1 = run(1)
    back = torch.argsort(w1)
    wr, xr, qr, fr = run(r)
    eps = 2.3e-16 if prec == "fp64" else 1.2e-7
    for one, many in ((x1[:, back], xr), (q1[:, back], qr)):
        assert float((many - one[:, wr]).abs().max()) <= 8 * eps * float(one.abs().max())
    tol = 16 * eps if prec == "mixed" else 64 * m * r * eps
    for one, many in zip(f1, fr):
        assert float((many - r * one).abs().max()) <= tol * r * float(one.abs().max())
