"""The mixed form's reverse GR particle kernels on 16^3 and 32^3 compute in FP64
from their FP32 operands: a particle's adjoints are those of the FP64 form on the
same inputs, rounded once.

Tolerance: half a unit in the last place of an FP32 result, 2^-24 of its
value, 1 % of that for what lies behind it, and 1e-12 of the largest for the
FP64 forms' own rounding.  FP32 arithmetic is 10 to 100 times that off.  The
fields' adjoints meet in FP32: up to 8 tiles at a site, each rounded and
added, 16 x 2^-24 of the largest."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,n", [(16, 1500), (32, 7001)])
def test_mixed_is_fp64_rounded_once(N, n):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm as gp
    rng = np.random.default_rng(n)
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    pos = (rng.integers(0, N, (3, n)) + np.floor(rng.random((3, n)) * 2 ** 16) / 2 ** 16) / N
    q = f32(rng.normal(0, 0.02, (3, n)))
    field = lambda c, s: f32(s * rng.standard_normal((c, N, N, N)))
    phi, chi, B, lT00, lTij, lL = (field(*a) for a in ((1, 1e-3), (1, 1e-3), (3, 1e-5), (1, 1.0), (6, 1.0), (3, 1.0)))
    l0 = [f32(rng.standard_normal((3, n))) for _ in range(2)]

    def run(prec):
        ctx = gp.Context(N, prec)
        t = lambda x: torch.from_numpy(x).to(ctx.rdtype).cuda()
        p = gp.Particles(ctx, n, 0.31 / n)
        p.load(pos, q, np.arange(n))
        kd = [t(x) for x in l0] + [ctx.real(c) for c in (1, 1, 3)]
        p.adj_gr_kick_drift(t(phi), t(chi), t(B), *kd, 3, 3, 0.1, 0.102, 0.015, 0.02)
        dep = [t(x) for x in l0] + [ctx.real(1)]
        p.adj_gr_deposit(t(phi), t(lT00), t(lTij), t(lL), *dep, 0.1, 0.7)
        return [x.double() for x in kd], [x.double() for x in dep]

    for mixed, exact in zip(run(gp.GEV_MIXED), run(gp.GEV_FP64)):
        for a, b in zip(mixed[:2], exact[:2]):
            assert bool(((a - b).abs() <= 1.01 * 2.0 ** -24 * b.abs() + 1e-12 * b.abs().max()).all())
        for a, b in zip(mixed[2:], exact[2:]):
            assert float((a - b).abs().max()) <= 16 * 2.0 ** -24 * float(b.abs().max())
