"""The adjoint chi solve in both forms and at every kind of size (planes and
separate passes, the smallest and a large mesh, and 8^3 below the fused range)
against the transform, the k-space operator and the inverse transform called
one by one, and against the forward solve by a dot product.

Tolerance: a transform of N^3 <= 2^24 values is within about 24 units of the
precision's epsilon of the exact one relative to the array's rms (FP64 5e-15,
FP32 3e-6, as for the other solves); two transforms and the operator, in two
roundings of the same formulas, and the largest of up to 1e8 values against their rms:
twelve times that."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = {"fp64": 12 * 5e-15, "mixed": 12 * 3e-6}


@pytest.mark.parametrize("N,prec", [(8, "mixed"), (16, "fp64"), (16, "mixed"), (32, "mixed"), (64, "fp64"),
                                    (64, "mixed"), (128, "fp64"), (128, "mixed"), (256, "fp64"), (256, "mixed")])
def test_against_separate_operator(N, prec):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gevpm as gp
    from gevpm._lib import check, lib
    ctx = gp.Context(N, gp.GEV_FP64 if prec == "fp64" else gp.GEV_MIXED)
    g = torch.Generator(device="cuda").manual_seed(N)
    rand = lambda c: torch.randn((c, N, N, N), generator=g, dtype=torch.float64, device="cuda").to(ctx.rdtype)
    y, S = rand(1), rand(6)
    F, F6 = ctx.fft_r2c(y), ctx.fourier(6)
    check(lib.gev_adj_project_ft_scalar(ctx.handle, C.c_void_p(F.data_ptr()), C.c_void_p(F6.data_ptr())), "operator")
    ref = ctx.fft_c2r(F6).double()
    keep = y.clone()
    got = ctx.adj_solve_chi(y).double()
    assert torch.equal(y, keep)
    for a, b in zip(got, ref):
        assert float((a - b).abs().max()) <= TOL[prec] * float(b.square().mean().sqrt())
    chi = ctx.solve_chi(S.clone()).double()
    lhs, rhs = float((y.double() * chi).sum()), float((got * S.double()).sum())
    assert abs(lhs - rhs) <= TOL[prec] * float(y.double().norm() * chi.norm())
