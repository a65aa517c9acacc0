"""Re-binning at the sizes where its form changes: the scan in one workgroup
(up to 4096 cells), with each workgroup adding up the chunks before it (up to
1024 chunks of 2048 cells), and with a pass of its own; the particles moved in
one pass below 2^20 and by a permutation and a gather from there.  Whole
numbers: everything is compared exactly."""
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


@pytest.mark.parametrize("prec,N,n", [("mixed", 4, 0), ("mixed", 4, 1), ("fp64", 8, 513), ("mixed", 16, 5000),
                                      ("fp64", 32, 33000), ("mixed", 64, (1 << 20) - 1), ("mixed", 64, 1 << 20),
                                      ("fp64", 64, (1 << 20) + 1), ("mixed", 128, 70001), ("mixed", 256, 65537)])
def test_cells_ids_and_offsets(gp, prec, N, n):
    ctx = gp.Context(N, gp.GEV_FP64 if prec == "fp64" else gp.GEV_MIXED)
    rng = np.random.default_rng(N + n)
    # half of the particles in a sixty-fourth of the box; offsets that both forms hold exactly
    x = rng.random((3, n)) * np.where(rng.random(n) < 0.5, 0.25, 1.0)
    pos = np.floor(x * N * 2 ** 16) / 2 ** 16 / N
    q = rng.normal(0, 1e-3, (3, n)).astype(np.float32).astype(np.float64)
    pid = rng.permutation(n).astype(np.int64)
    p = gp.Particles(ctx, max(n, 1), 1.0)
    p.load(pos, q, pid)
    if n:  # a second re-binning, by the drift's own counts, of a state at rest
        p.update_pos_newton(0.0, 1.0)
    c = np.floor(pos * N).astype(np.int64)
    key = c[0] + N * (c[1] + N * c[2])
    start = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=N ** 3))])
    assert np.array_equal(p.cell_start().cpu().numpy(), start)
    assert np.array_equal(p.cells().cpu().numpy(), np.sort(key))
    if n == 0:
        return  # store refuses an empty container
    gpos, gq, gid = (t.cpu().numpy() for t in p.store())
    o, go = np.argsort(pid), np.argsort(gid)
    assert np.array_equal(gid[go], pid[o]) and np.array_equal(gpos[:, go], pos[:, o])
    assert np.array_equal(gq[:, go], q[:, o])
