"""The plane transforms of 16 <= N <= 128 (x and y of a z plane in one
workgroup) at the edges of their range: several components per launch, past
the largest batch of one, inverse transforms of arrays that are not Hermitian,
and the fused solves with their sources formed in the planes, including the
source terms that meshes below 128 leave in place.

Tolerances: a transform of N^3 values in log2(N^3) <= 21 rounding stages is
within about 21 units of the precision's epsilon of the exact one, relative to
the array's rms (FP64 5e-15, FP32 3e-6); the solves run two of them and a
division, and compare two roundings of the same formulas: three times that.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = {"fp64": 5e-15, "mixed": 3e-6}


@pytest.fixture(scope="module")
def gp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm
    return gevpm


def make(gp, N, prec, *shapes, seed=1):
    ctx = gp.Context(N, gp.GEV_FP64 if prec == "fp64" else gp.GEV_MIXED)
    g = torch.Generator().manual_seed(seed * N)
    return (ctx,) + tuple(torch.randn((c, N, N, N), generator=g, dtype=torch.float64).to(ctx.rdtype).to(ctx.device)
                          for c in shapes)


def off(a, b):
    a, b = (torch.view_as_real(t) if t.is_complex() else t for t in (a, b))
    a, b = a.double(), b.double()
    return float((a - b).abs().max() / b.square().mean().sqrt())


@pytest.mark.parametrize("N,prec,ncomp", [(16, "fp64", 65), (16, "mixed", 3), (32, "mixed", 6), (64, "fp64", 2),
                                          (64, "mixed", 1), (128, "fp64", 2), (128, "mixed", 7)])
def test_components_forward_and_inverse(gp, N, prec, ncomp):
    """each component of a batched transform against torch.fft in FP64; padding columns zero; an inverse of data
    whose kx = 0 and kx = N/2 planes are not Hermitian keeps the real part on those two columns"""
    ctx, f = make(gp, N, prec, ncomp)
    F = ctx.fft_r2c(f)
    ref = torch.fft.rfftn(f.double(), dim=(1, 2, 3))
    assert off(ctx.unpad(F), ref) < 4 * TOL[prec]  # the largest of 1e5 .. 1e7 values
    assert not ctx.P > N // 2 + 1 or float(F[..., N // 2 + 1:].abs().max()) == 0.0
    assert off(ctx.fft_c2r(F) / N ** 3, f) < 8 * TOL[prec]
    _, re, im = make(gp, N, prec, ncomp, ncomp, seed=2)
    G = torch.complex(re, im)[..., : N // 2 + 1].contiguous()
    buf = ctx.fourier(ncomp)
    buf[..., : N // 2 + 1] = G
    buf[..., N // 2 + 1:] = 7.0  # ignored by the inverse
    g = torch.fft.ifftn(G.to(torch.complex128), dim=(1, 2), norm="forward")
    g[..., 0].imag.zero_()
    g[..., -1].imag.zero_()
    assert off(ctx.fft_c2r(buf), torch.fft.irfft(g, n=N, dim=3, norm="forward")) < 4 * TOL[prec]


@pytest.mark.parametrize("N,prec", [(16, "fp64"), (16, "mixed"), (32, "fp64"), (64, "mixed"), (128, "fp64"),
                                    (128, "mixed")])
def test_solves_against_unfused_sequences(gp, N, prec):
    """the phi, chi and B solves with the sources formed in the planes against the source kernels, the transforms
    and the k-space operators called one by one"""
    ctx, phi, chi, T00, Tij, L = make(gp, N, prec, 1, 1, 1, 6, 3)
    phi, chi, T00 = 1e-4 * phi, 1e-5 * chi, 1.0 + 0.3 * T00
    tol = 12 * TOL[prec]
    # phi: source, transform, k=0 mode, Poisson, inverse
    bg, c1, c2, c3, coeff, modif = 0.31, 2.3e-3, 4.1e-4, 7.7e-7, float(N * N), 0.21
    src, s0, s1 = ctx.prepare_source_T00(phi, chi, T00, bg, c1, c2, c3)
    F = ctx.fft_r2c(src)
    ctx.set_k0(F, s1)
    ref = ctx.fft_c2r(ctx.poisson(F, coeff, modif))
    t = T00.clone()
    got, (g0, g1) = ctx.solve_poisson_T00(phi, chi, t, bg, c1, c2, c3, coeff, modif, k0set=True)
    assert off(got, ref) < tol
    assert abs(g0 - s0) <= 1e-12 * abs(s0) and abs(g1 - s1) <= 1e-9 * max(1.0, abs(s1))
    assert torch.equal(t, T00) if N >= 128 else off(t, src) < TOL[prec]
    # chi
    S = ctx.prepare_source_Tij(phi, Tij, 0.7)
    ref = ctx.fft_c2r(ctx.project_ft_scalar(ctx.fft_r2c(S)))
    assert off(ctx.solve_chi(S), ref) < tol
    t = Tij.clone()
    assert off(ctx.solve_chi_Tij(phi, t, 0.7), ref) < tol
    assert torch.equal(t, Tij) if N >= 128 else off(t, S) < TOL[prec]
    # B
    V = torch.stack([L[i] * (1 + phi[0] + torch.roll(phi[0], -1, 2 - i)) for i in range(3)])
    ref = ctx.fft_c2r(ctx.project_ft_vector(ctx.fft_r2c(V), 0.25))
    assert off(ctx.solve_vector(V.clone(), 0.25), ref) < tol
    assert off(ctx.solve_vector_T0i_links(L.clone(), phi, 0.25), ref) < tol
