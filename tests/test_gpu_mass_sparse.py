"""The FP32 mass deposit of sparse meshes (64 x 8 x 4 tiles with 64-bit sums, N
>= 256 and fewer than one particle per two cells), uniform and in clumps, whose
tiles start their particles at different corners, written and accumulated.

Tolerance per site, in units of the mass: offsets are multiples of 2^-16 of a
cell, so a weight is rounded by its two products (2 x 2^-24 of it) and by the
fixed point (2^-31 per addition, at most 8 k with k in the fullest cell); the
sum's conversion, the scale and its product add 3 x 2^-24 of it, and an
accumulating store 2^-24 of the result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,n,clumped", [(256, 30001, 0.0), (256, 200003, 0.6), (256, 4000001, 0.3), (512, 150001, 0.9)])
@pytest.mark.parametrize("aligned,accumulate", [(True, False), (True, True), (False, True)])
def test_sparse_mass(N, n, clumped, aligned, accumulate):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm as gp
    ctx = gp.Context(N, gp.GEV_MIXED)
    rng = np.random.default_rng(N + n)
    x = rng.random((3, n))
    m = int(clumped * n)  # clumps of a few hundred within about a cell, the first at the corner of eight tiles
    if m:
        centre = rng.random((3, 1 + m // 300))
        centre[:, 0] = 0.0
        x[:, :m] = (centre[:, rng.integers(0, centre.shape[1], m)] + 0.6 / N * rng.standard_normal((3, m))) % 1.0
    u = np.floor(x * N * 2 ** 16) / 2 ** 16 % N
    p = gp.Particles(ctx, n, 1.0)
    p.load(u / N, np.zeros((3, n)), np.arange(n, dtype=np.int64))
    unit = float(N) ** 3  # project_mass with mass 1: density, one particle per cell = N^3
    buf = torch.full((N ** 3 + 1,), 3.0 * unit, dtype=torch.float32, device="cuda")
    out = (buf[:-1] if aligned else buf[1:]).view(1, N, N, N)
    p.project_mass(out, accumulate=accumulate)
    c = np.floor(u).astype(np.int64)
    d = u - c
    rho = np.zeros(N ** 3)
    for b in range(8):
        s = [b & 1, b >> 1 & 1, b >> 2]
        w = np.prod([d[i] if s[i] else 1 - d[i] for i in range(3)], axis=0)
        g = [(c[i] + s[i]) % N for i in range(3)]
        rho += np.bincount(g[0] + N * (g[1] + N * g[2]), w, N ** 3)
    k = np.bincount(c[0] + N * (c[1] + N * c[2])).max()
    tol = 8 * k * 2.0 ** -31 + 5 * 2.0 ** -24 * rho
    if accumulate:
        rho += 3.0
        tol += 2.0 ** -24 * rho
    got = out.cpu().numpy().astype(np.float64).ravel() / unit
    assert np.all(np.abs(got - rho) <= tol)
