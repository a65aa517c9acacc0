"""The mixed form's scalar projection forms its weighted sums in FP64 up to
64^3: a Sij that is all trace (three equal diagonal components, whose
transforms are equal bit by bit) has no chi.

Tolerance: three FP64 weights that cancel, |w| <= 12 N^2 each, leave at most
4 units of 2^-53 of their largest product per mode, against a single
component's chi of the same modes; 1e-13 of the latter's largest value allows
for two hundred times that.  Weights rounded to FP32, or an FP32 sum, leave
about 1e-7."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N", [16, 32, 64])
def test_all_trace_has_no_chi(N):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm as gp
    ctx = gp.Context(N, gp.GEV_MIXED)
    g = torch.Generator().manual_seed(N)
    f = torch.randn((N, N, N), generator=g, dtype=torch.float64).to(ctx.rdtype).to(ctx.device)
    one, trace = ctx.real(6), ctx.real(6)
    one[0] = f
    for c in (0, 3, 5):
        trace[c] = f
    scale = float(ctx.solve_chi(one).abs().max())
    assert scale > 0.0
    assert float(ctx.solve_chi(trace).abs().max()) <= 1e-13 * scale
    phi = ctx.real(1)
    assert float(ctx.solve_chi_Tij(phi, trace.clone(), 1.0).abs().max()) <= 1e-13 * scale
    # and the whole projection is the k-space operator's on the six spectra, up to the transforms' rounding
    S = torch.randn((6, N, N, N), generator=g, dtype=torch.float64).to(ctx.rdtype).to(ctx.device)
    ref = ctx.fft_c2r(ctx.project_ft_scalar(ctx.fft_r2c(S))).double()
    assert float((ctx.solve_chi(S) - ref).abs().max() / ref.square().mean().sqrt()) < 9e-6
