"""FP32 mass deposit in long rows (N >= 256: 64 x 8 x 4 cells below one particle
per two cells, 16 x 8 x 8 from there and on smaller meshes), against
FP64 sums over the same positions.  Offsets are multiples of 2^-16 of a cell,
held exactly by FP32.  Bound per site, in units of the mass: every addition
rounds to half a unit of the tile's fixed point, cmax / 2^30, with at most 8 k
additions and cmax <= 36 k for a fullest cell of k particles; the weight's three
products, the scale's and the store's add 8 FP32 roundings of the sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,n", [(128, 300001), (256, 1), (256, 70001), (256, (1 << 23) - 1), (256, 1 << 23),
                                 (512, 200003)])
@pytest.mark.parametrize("aligned", [True, False])
def test_mass(N, n, aligned):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm as gp
    ctx = gp.Context(N, gp.GEV_MIXED)
    rng = np.random.default_rng(N + n)
    x = rng.random((3, n)) * np.where(rng.random(n) < 0.3, 0.25, 1.0)
    if n > 8:  # the tile's and the box's faces
        x[:, :8] = np.array([[0, 63 / N, 64 / N, 32 / N, 31 / N, 1 - 0.5 / N, 16 / N, 1 - 1 / N]] * 3)
    u = np.floor(x * N * 2 ** 16) / 2 ** 16
    p = gp.Particles(ctx, n, 1.0)
    p.load(u / N, np.zeros((3, n)), np.arange(n, dtype=np.int64))
    buf = torch.full((N ** 3 + 1,), 2.0, dtype=torch.float32, device="cuda")
    out = buf[:-1] if aligned else buf[1:]
    out = out.view(1, N, N, N)
    p.project_mass(out)
    c = np.floor(u).astype(np.int64)
    d = u - c
    rho = np.zeros(N ** 3)
    for b in range(8):
        s = [b & 1, b >> 1 & 1, b >> 2]
        w = np.prod([d[i] if s[i] else 1 - d[i] for i in range(3)], axis=0)
        g = [(c[i] + s[i]) % N for i in range(3)]
        rho += np.bincount(g[0] + N * (g[1] + N * g[2]), w, N ** 3)
    k = np.bincount(c[0] + N * (c[1] + N * c[2])).max()
    unit = float(N) ** 3  # project_mass with mass 1: density, one particle per cell = N^3
    tol = 8 * k * 36 * k / 2.0 ** 31 + 8 * 2.0 ** -24 * rho
    got = out.cpu().numpy().astype(np.float64).ravel() / unit
    assert np.all(np.abs(got - rho) <= tol)
