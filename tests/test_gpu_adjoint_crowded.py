"""The reverse GR particle kernels on crowded rows, where they hand
consecutive particles to different waves, against the same particles spread
over containers whose rows stay below that line: the field adjoints add up and
the per-particle ones are the same whichever container holds the particle.

Tolerances: sums are FP64 in LDS, rounded to the field's precision once per
tile and added there; with 40 containers that is 40 roundings per site against
one (FP32: 40 x 6e-8 of the largest partial sum; FP64 1e-16 likewise), and the
per-particle values are the same arithmetic."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm
    return gevpm


@pytest.mark.parametrize("prec,N,n,nf", [("mixed", 16, 1500, 3), ("mixed", 32, 2111, 3), ("mixed", 64, 3001, 3), ("mixed", 16, 777, 2),
                                         ("fp64", 16, 1000, 3), ("fp64", 8, 401, 3), ("mixed", 8, 401, 3)])
def test_crowded_rows_match_sparse_ones(gp, prec, N, n, nf):
    ctx = gp.Context(N, gp.GEV_FP64 if prec == "fp64" else gp.GEV_MIXED)
    rng = np.random.default_rng(n)
    # most particles in a few cells at the wrap of the mesh, offsets that both forms hold exactly
    cell = np.where(rng.random(n) < 0.8, rng.integers(0, 2, (3, n)) * (N - 1), rng.integers(0, N, (3, n)))
    pos = (cell + np.floor(rng.random((3, n)) * 2 ** 20) / 2 ** 20) / N
    q = rng.normal(0, 0.02, (3, n)).astype(np.float32).astype(np.float64)
    t = lambda c, s: (s * torch.from_numpy(rng.standard_normal((c, N, N, N)))).to(ctx.rdtype).cuda()
    phi, chi, B, lT00, lTij, lL = t(1, 1e-3), t(1, 1e-3), t(3, 1e-5), t(1, 1.0), t(6, 1.0), t(3, 1.0)
    lx0, lq0 = (torch.from_numpy(rng.standard_normal((3, n))).to(ctx.rdtype).cuda() for _ in range(2))

    def run(parts):
        out = [torch.zeros_like(lx0), torch.zeros_like(lq0)] + [ctx.real(c) for c in (1, 1, 3, 1)]
        for ids in parts:
            p = gp.Particles(ctx, len(ids), 0.31 / n)
            p.load(pos[:, ids], q[:, ids], np.arange(len(ids)))
            lx, lq = lx0[:, ids].contiguous(), lq0[:, ids].contiguous()
            p.adj_gr_kick_drift(phi, chi, B, lx, lq, out[2], out[3], out[4], nf, nf, 0.1, 0.102, 0.015, 0.02)
            p.adj_gr_deposit(phi, lT00, lTij, lL, lx, lq, out[5], 0.1, 0.7)
            out[0][:, ids], out[1][:, ids] = lx, lq
        return [o.double() for o in out]

    one = run([np.arange(n)])
    many = run(np.array_split(rng.permutation(n), 40))
    eps = 2.3e-16 if prec == "fp64" else 1.2e-7
    for a, b in zip(one[:2], many[:2]):
        assert float((a - b).abs().max()) <= 8 * eps * float(b.abs().max())
    for a, b in zip(one[2:], many[2:]):
        assert float((a - b).abs().max()) <= 40 * eps * float(b.abs().max())
