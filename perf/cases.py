"""The work a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values; `kind` says which public entry points it
runs (all of them through the Python host layer gevpm):

  cycle    the main loop: main.cu's cycle with gevpm.step from a saved state
  update   one kick + drift + re-binning of a saved particle state
  grad     a differentiable run: forward and backward through torch.autograd
  adjoint  the particle kernels of one reverse GR cycle
  deposit  the CIC projections of one particle state
  density  the mass density of particles and its Fourier transform
  solve    the three metric solves (phi, chi, B) of one GR cycle

`mesh` is N of the N^3 mesh, `particles` the particle count, `fp64` the
precision form.  Meshes are 2.5 Mpc/h per cell, as the 256^3 and 512^3
workloads of the tests and the benchmark are.  Particle states are Zel'dovich
displacements (`disp`: rms in cells, per axis) of the cell-centred lattice, or
of uniformly drawn points where the count is not N^3, with a fraction `halos`
of the particles gathered into clumps of about a cell, as structure
formation leaves them at low redshift.

`exact` restates every kind in plain torch in FP64 on top of `_Mesh` below
(periodic fields as [z, y, x] tensors, particles as (3, n) positions in box
units); the gradients come from torch.autograd through that restatement.
"""
import math
import os
import sys

import torch
from torch.utils.checkpoint import checkpoint

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "gevolution-2.0_amd", "python"))

import gevpm  # noqa: E402
from gevpm.adjoint import PMRun, PMRunGR, pm_density, pm_density_gr  # noqa: E402

OM, OL = 0.31, 0.69     # Omega_m, Omega_Lambda
CELL = 2.5              # Mpc/h per mesh cell
DEV = "cuda"


def listed():
    return [
        # the headline run: the mixed-precision GR cycle at 512^3, mid-run (structure present, few crowded cells)
        dict(name="cycle_gr_mixed_512", kind="cycle", gr=True, fp64=False, mesh=512, particles=512 ** 3, z=3.0,
             disp=1.0, halos=0.05, cycles=4),
        # the FP64 GR run at 256^3 from early times
        dict(name="cycle_gr_fp64_256", kind="cycle", gr=True, fp64=True, mesh=256, particles=256 ** 3, z=50.0,
             disp=0.3, halos=0.0, cycles=3),
        # parameter scans and tests on small boxes: launches and host work count
        dict(name="cycle_gr_fp64_32", kind="cycle", gr=True, fp64=True, mesh=32, particles=32 ** 3, z=30.0, disp=0.4,
             halos=0.0, cycles=8),
        # Newtonian comparison runs, late and clustered, a particle number that is no cube
        dict(name="cycle_newton_mixed_128", kind="cycle", gr=False, fp64=False, mesh=128, particles=2000003, z=0.5,
             disp=1.5, halos=0.3, cycles=6),
        # gradient-based inference: the mixed GR run and its gradient, a checkpoint every second cycle
        dict(name="grad_gr_mixed_128", kind="grad", gr=True, fp64=False, mesh=128, steps=4, ckpt=2),
        # the Newtonian gradient on a small box in FP64
        dict(name="grad_newton_fp64_64", kind="grad", gr=False, fp64=True, mesh=64, steps=6, ckpt=1),
        # one late particle state projected for T00, Tij and the T0i links, the cycle's largest kernel after the kick
        dict(name="deposit_mixed_256", kind="deposit", links=True, fp64=False, mesh=256, particles=15485863, z=0.0,
             disp=1.5, halos=0.4),
        # one kick + drift of an FP64 state, fewer particles than cells
        dict(name="update_fp64_128", kind="update", gr=True, fp64=True, mesh=128, particles=1299709, z=1.0, disp=1.0,
             halos=0.2),
        # the reverse particle kernels of one GR cycle
        dict(name="adjoint_mixed_256", kind="adjoint", fp64=False, mesh=256, particles=256 ** 3, z=2.0, disp=0.8,
             halos=0.1),
        # the metric solves alone, large FP64 and small mixed
        dict(name="solve_fp64_512", kind="solve", fp64=True, mesh=512),
        dict(name="solve_mixed_64", kind="solve", fp64=False, mesh=64),
        # the density spectrum's input on the largest mesh, more cells than particles
        dict(name="density_mixed_1024", kind="density", fp64=False, mesh=1024, particles=99999989, z=1.0, disp=1.0,
             halos=0.1),
    ]


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["cycle", "cycle", "update", "grad", "adjoint", "deposit", "deposit", "density", "solve", "solve"])
    fp64 = rng.random() < 0.4
    c = dict(kind=kind, fp64=fp64)

    def size(lo, hi):  # powers of two only: what the library takes
        c["mesh"] = 1 << rng.randint(lo, hi)

    def state(most):
        cells = c["mesh"] ** 3
        if rng.random() < 0.4 and cells <= most:
            c["particles"] = cells
        else:
            n = int(cells * math.exp(rng.uniform(math.log(0.1), math.log(2.0))))
            c["particles"] = max(27, min(n, most)) | 1
        late = rng.random()
        c.update(z=round(50.0 * (1.0 - late) ** 2, 3), disp=round(0.2 + 1.4 * late, 3),
                 halos=round(max(0.0, 0.5 * (late - 0.2)), 3))

    if kind == "cycle":
        size(4, 8 if fp64 else 9)
        state(1 << 27)
        c.update(gr=rng.random() < 0.7, cycles=rng.randint(2, 3 if c["mesh"] >= 256 else 8))
    elif kind == "update":
        size(4, 8)
        state(1 << 25)
        c["gr"] = rng.random() < 0.7
    elif kind == "grad":
        size(4, 6 if fp64 else 7)
        c.update(gr=rng.random() < 0.6, steps=rng.randint(2, 5), ckpt=rng.randint(1, 3))
    elif kind == "adjoint":
        size(4, 8)
        state(1 << 24)
    elif kind == "deposit":
        size(4, 8)
        state(1 << 25)
        c["links"] = rng.random() < 0.5
    elif kind == "density":
        size(4, 9 if fp64 else 10)
        state(1 << 26)
    else:
        size(4, 8 if fp64 else 9)
        c["amp"] = round(rng.uniform(0.5, 2.0), 3)
    return c


# --------------------------------------------------------------- background --
def _fpg(N):
    return 1.5 * (CELL * N / 2997.92458) ** 2


def _hconf(a, fpg):
    return math.sqrt(2.0 * fpg / 3.0 * (OM / a + OL * a * a))


def _rk4(a, fpg, dtau):
    def f(x):
        return x * _hconf(x, fpg)
    k1 = f(a)
    k2 = f(a + 0.5 * dtau * k1)
    k3 = f(a + 0.5 * dtau * k2)
    k4 = f(a + dtau * k3)
    return a + dtau * (k1 + 2 * k2 + 2 * k3 + k4) / 6.0


def _horizon(a, fpg, panels=2000):
    # tau = int da / (a Hconf) in s = sqrt(a) by Simpson's rule, from 1e-7 of the upper limit as particleHorizon does
    # (background.hpp:268-290); s Hconf(s^2) is smooth down to s = 0
    hi = math.sqrt(a)
    lo = 1e-7 * hi
    h, tot = (hi - lo) / panels, 0.0
    for i in range(2 * panels + 1):
        w = 1 if i in (0, 2 * panels) else 4 if i % 2 else 2
        tot += w / math.sqrt(OM + OL * (lo + 0.5 * i * h) ** 6)
    return tot * 2.0 * h / 6.0 / math.sqrt(2.0 * fpg / 3.0)


def _dtau(fpg):
    """A hundredth of the conformal time from z = 100 to 0, the benchmark's step."""
    return 0.01 * (_horizon(1.0, fpg) - _horizon(1.0 / 101.0, fpg))


# ------------------------------------------------------------------- inputs --
def _smooth(N, gen, scale=4.0, slope=-1.0, count=1):
    """`count` real random fields (unit rms) with spectra ~ k^slope, cut off below `scale` cells."""
    out = torch.empty((count, N, N, N), dtype=torch.float64, device=DEV)
    k = torch.fft.fftfreq(N, 1.0 / N, device=DEV, dtype=torch.float64)
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, : N // 2 + 1] ** 2
    k2[0, 0, 0] = 1.0
    amp = k2 ** (0.5 * slope) * torch.exp(-0.5 * k2 * (scale / N) ** 2)
    amp[0, 0, 0] = 0.0
    for c in range(count):
        F = torch.fft.rfftn(torch.randn((N, N, N), generator=gen, dtype=torch.float64, device=DEV))
        f = torch.fft.irfftn(F.mul_(amp), s=(N, N, N))
        out[c] = f / f.std()
    return out


def _particles(case, gen):
    """(pos, q, id, phi): a displaced particle state and the potential that goes with it."""
    N, n = case["mesh"], case["particles"]
    fpg, a = _fpg(N), 1.0 / (1.0 + case["z"])
    psi = _smooth(N, gen, slope=-3.0)[0]
    # displacement -grad(psi), scaled to `disp` cells rms per axis
    d = torch.stack([0.5 * N * (torch.roll(psi, 1, 2 - i) - torch.roll(psi, -1, 2 - i)) for i in range(3)])
    s = case["disp"] / N / float(d.square().mean().sqrt())
    d *= s
    if n == N ** 3:
        x = (torch.arange(N, dtype=torch.float64, device=DEV) + 0.5) / N
        lag = torch.stack([x.expand(N, N, N), x[:, None].expand(N, N, N), x[:, None, None].expand(N, N, N)])
        lag, disp = lag.reshape(3, n), d.reshape(3, n)
    else:
        lag = torch.rand((3, n), generator=gen, dtype=torch.float64, device=DEV)
        ix = (lag * N).long().clamp_(0, N - 1)
        at = ix[0] + N * (ix[1] + N * ix[2])
        disp = torch.stack([d[i].reshape(-1)[at] for i in range(3)])
        del ix, at
    H = _hconf(a, fpg)
    f = (OM / (OM + OL * a ** 3)) ** 0.55
    q = (a * H * f) * disp
    pos = lag + disp
    del d, disp, lag
    m = int(case["halos"] * n)
    if m > 0:  # every so many particles go to a clump; a few clumps are much richer than the rest
        who = torch.randperm(n, generator=gen, device=DEV)[:m]
        nh = max(1, m // 150)
        centre = torch.rand((3, nh), generator=gen, dtype=torch.float64, device=DEV)
        which = (torch.rand(m, generator=gen, dtype=torch.float64, device=DEV) ** 1.3 * nh).long()
        pos[:, who] = centre[:, which] + torch.randn((3, m), generator=gen, dtype=torch.float64, device=DEV) * (0.6 / N)
        q[:, who] += torch.randn((3, m), generator=gen, dtype=torch.float64, device=DEV) * (2.0 * float(q.std()))
    pos -= torch.floor(pos)
    pos[pos >= 1.0] = 0.0
    phi = psi * (s * fpg * OM / a)
    return pos, q, torch.arange(n, device=DEV), phi.reshape(1, N, N, N)


def _metric(case, gen, phi):
    """chi and B of sizes that go with phi."""
    N, a = case["mesh"], 1.0 / (1.0 + case["z"])
    amp = float(phi.std())
    e = _smooth(N, gen, count=4)
    return e[:1] * (1e-3 * amp), e[1:] * (1e-2 * amp * a * a * N)


def _background(case):
    N = case["mesh"]
    fpg, a = _fpg(N), 1.0 / (1.0 + case["z"])
    dtau = _dtau(fpg)
    a_d = _rk4(a, fpg, 0.5 * dtau)
    return dict(fpg=fpg, a=a, a_d=a_d, dtau=dtau, bk=a * a * N, bd=a_d * a_d * N)


def _inputs(case, seed):
    """The inputs of a case by name, as FP64 tensors; those of a mixed-form case are values that its FP32 fields and
    cell offsets hold exactly."""
    x = _fp64_inputs(case, seed)
    if not case["fp64"]:
        for k in x:
            if k == "pos":
                grid = case["mesh"] * float(1 << 20)
                x[k].mul_(grid).floor_().div_(grid)
            elif k != "id":
                x[k] = x[k].float().double()
    return x


def _fp64_inputs(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    N, kind = case["mesh"], case["kind"]
    x = {}
    if kind == "grad":
        x["psi"] = _smooth(N, gen, scale=8.0, slope=-2.0) * (0.3 / N ** 2)
        x["g"] = _smooth(N, gen, scale=2.0)
        return x
    if kind == "solve":
        amp = 1e-5 * case.get("amp", 1.0)
        x["phi"] = _smooth(N, gen, slope=-3.0) * amp
        x["chi"] = _smooth(N, gen, slope=-2.0) * (1e-3 * amp)
        x["T00"] = OM * (1.0 + 0.5 * _smooth(N, gen, scale=2.0))
        x["Tij"] = 1e-5 * _smooth(N, gen, scale=2.0, count=6)
        x["L"] = 1e-3 * _smooth(N, gen, scale=2.0, count=3)
        return x
    x["pos"], x["q"], x["id"], x["phi"] = _particles(case, gen)
    if kind in ("update", "adjoint"):
        x["chi"], x["B"] = _metric(case, gen, x["phi"])
    if kind == "adjoint":
        n = case["particles"]
        for name in ("lx", "lq"):
            x[name] = torch.randn((3, n), generator=gen, dtype=torch.float64, device=DEV)
        for name, c in (("lphi", 1), ("lchi", 1), ("lT00", 1), ("lTij", 6), ("lL", 3)):
            x[name] = _smooth(N, gen, scale=2.0, count=c)
    return x


# ------------------------------------------------------------ the framework --
def _coefs(N, b, dtau_old):
    """The coefficients of one GR cycle's source and solves (main.cu:725-948)."""
    dx2, H = 1.0 / (N * N), _hconf(b["a"], b["fpg"])
    return dict(c1=3.0 * H * dx2 / dtau_old, c2=b["fpg"] * dx2 / b["a"], c3=3.0 * H * H * dx2, pcoeff=1.0 / dx2,
                modif=3.0 * H / dtau_old, ccoeff=2.0 * b["fpg"] * dx2 / b["a"], bcoeff=b["fpg"] * dx2)


def prepare(case, seed):
    N, kind = case["mesh"], case["kind"]
    prec = gevpm.GEV_FP64 if case["fp64"] else gevpm.GEV_MIXED
    s = dict(case=case)
    x = _inputs(case, seed)
    if kind == "grad":
        cls = PMRunGR if case["gr"] else PMRun
        run = cls(N, CELL * N, 50.0, 20.0, case["steps"], precision=prec, ckpt_every=case["ckpt"])
        s.update(run=run, psi=x["psi"].to(run.ctx.rdtype), g=x["g"].to(run.ctx.rdtype))
        return s
    ctx = s["ctx"] = gevpm.Context(N, prec)
    for name, v in x.items():
        if name not in ("pos", "q", "id"):
            s[name] = v.to(ctx.rdtype).contiguous()
    if kind == "solve":
        s["work"] = {c: ctx.fourier(c) for c in (1, 3, 6)}
        s["back"] = _background(dict(case, z=2.0))
        return s
    p = s["pcls"] = gevpm.Particles(ctx, case["particles"], OM / case["particles"])
    p.load(x["pos"], x["q"], x["id"])
    del x
    b = s["back"] = _background(case)
    if kind in ("cycle", "update"):
        s["saved"] = p.save()
    if kind == "cycle":
        s["fields"] = gevpm.Fields(ctx)
        s["state"] = gevpm.StepState(int(case["gr"]), b["fpg"], OM, OL, z_relax=100.0)
    if kind == "deposit":
        s["out"] = (ctx.real(1), ctx.real(6), ctx.real(3))
    if kind == "density":
        s["out"] = (ctx.real(1), ctx.fourier(1))
    return s


def _by_id(p):
    """Positions and momenta in ID order, in the precision of the run."""
    pos, q, pid = p.store()
    out = torch.empty((2,) + tuple(pos.shape), dtype=p.ctx.rdtype, device=pos.device)
    out[0][:, pid] = pos.to(out.dtype)
    out[1][:, pid] = q.to(out.dtype)
    return out[0], out[1]


def run(s):
    return _RUN[s["case"]["kind"]](s)


def _run_cycle(s):
    p, f, st, b = s["pcls"], s["fields"], s["state"], s["back"]
    p.restore(s["saved"])
    f.phi.copy_(s["phi"])
    f.chi.zero_()
    f.Bi.zero_()
    st.a, st.tau, st.dtau_old = b["a"], 0.0, b["dtau"]
    for _ in range(s["case"]["cycles"]):
        st.dtau = b["dtau"]
        gevpm.step(p, f, st)
    pos, q = _by_id(p)
    return dict(phi=f.phi, chi=f.chi, B=f.Bi, pos=pos, q=q)


def _run_update(s):
    p, b = s["pcls"], s["back"]
    p.restore(s["saved"])
    if s["case"]["gr"]:
        v2 = p.kick_drift(1, b["dtau"], b["dtau"], s["phi"], s["chi"], s["B"], 3, 3, b["a"], b["a_d"], b["bk"], b["bd"])
    else:
        v2 = p.kick_drift(0, b["dtau"], b["dtau"], s["phi"], None, None, 1, 0, b["a"], b["a_d"], 1.0, 1.0)
    pos, q = _by_id(p)
    return dict(pos=pos, q=q, v2=torch.tensor([v2], dtype=p.ctx.rdtype))


def _run_grad(s):
    psi = s["psi"].detach().requires_grad_(True)
    rho = (pm_density_gr if s["case"]["gr"] else pm_density)(psi, s["run"])
    rho.backward(s["g"])
    return dict(rho=rho.detach(), grad=psi.grad)


def _run_adjoint(s):
    p, b, ctx = s["pcls"], s["back"], s["ctx"]
    lx, lq, lphi, lchi = (s[k].clone() for k in ("lx", "lq", "lphi", "lchi"))
    lB, lold = ctx.real(3), ctx.real(1)
    p.adj_gr_kick_drift(s["phi"], s["chi"], s["B"], lx, lq, lphi, lchi, lB, 3, 3, b["a"], b["a_d"], b["dtau"], b["dtau"])
    p.adj_gr_deposit(s["phi"], s["lT00"], s["lTij"], s["lL"], lx, lq, lold, b["a"], 0.5)
    return dict(lx=lx, lq=lq, lphi=lphi, lchi=lchi, lB=lB, lold=lold)


def _run_deposit(s):
    p, a, (T00, Tij, v) = s["pcls"], s["back"]["a"], s["out"]
    if s["case"]["links"]:  # the GR cycle with the elliptic B
        p.project_T00_Tij_T0i_links(T00, Tij, v, a=a, phi=s["phi"])
    else:                   # the projections one by one, as main.cu calls them
        p.project_T00(T00, a=a, phi=s["phi"])
        p.project_Tij(Tij, a=a, phi=s["phi"])
        p.project_T0i(v, phi=s["phi"])
    return dict(T00=T00, Tij=Tij, T0i=v)


def _run_density(s):
    rho, F = s["out"]
    s["pcls"].project_mass(rho)
    s["ctx"].fft_r2c(rho, out=F)
    return dict(rho=rho, F=torch.view_as_real(s["ctx"].unpad(F)))


def _run_solve(s):
    ctx, N, w = s["ctx"], s["case"]["mesh"], s["work"]
    k = _coefs(N, s["back"], s["back"]["dtau"])
    B = s["L"].clone()
    if N >= 128:  # the sources formed inside the solves, as gevpm.step runs them
        phi, _ = ctx.solve_poisson_T00(s["phi"], s["chi"], s["T00"], OM, k["c1"], k["c2"], k["c3"], k["pcoeff"],
                                       k["modif"], k0set=not s["case"]["fp64"], work=w[1])
        chi = ctx.solve_chi_Tij(phi, s["Tij"], k["ccoeff"], work6=w[6], work1=w[1])
    else:
        src, _, k0 = ctx.prepare_source_T00(s["phi"], s["chi"], s["T00"], OM, k["c1"], k["c2"], k["c3"])
        phi = ctx.solve_poisson(src, k["pcoeff"], k["modif"], k0=None if s["case"]["fp64"] else k0, work=w[1])
        chi = ctx.solve_chi(ctx.prepare_source_Tij(phi, s["Tij"], k["ccoeff"]), work6=w[6], work1=w[1])
    ctx.solve_vector_T0i_links(B, phi, k["bcoeff"], 0.0, work=w[3])
    return dict(phi=phi, chi=chi, B=B)


_RUN = dict(cycle=_run_cycle, update=_run_update, grad=_run_grad, adjoint=_run_adjoint, deposit=_run_deposit,
            density=_run_density, solve=_run_solve)


def work(case):
    """Inputs read once and outputs written once, per cycle where the state passes through memory between cycles."""
    kind, N, R = case["kind"], case["mesh"], 8 if case["fp64"] else 4
    M = N ** 3
    n = case.get("particles", M)
    part = n * (6 * R + 12)               # positions, momenta, ID and cell of a particle
    fft = 2.5 * M * 3 * math.log2(N)      # one real transform
    if kind == "cycle":
        c = case["cycles"]
        if case["gr"]:
            return dict(bytes=c * (2 * part + 7 * M * R), flops=c * (900.0 * n + 15 * fft))
        return dict(bytes=c * (2 * part + 2 * M * R), flops=c * (150.0 * n + 2 * fft))
    if kind == "update":
        return dict(bytes=2 * part + (5 if case["gr"] else 1) * M * R, flops=(500.0 if case["gr"] else 120.0) * n)
    if kind == "grad":
        c = case["steps"]
        if case["gr"]:
            return dict(bytes=c * (6 * part + 30 * M * R), flops=c * (4000.0 * n + 42 * fft))
        return dict(bytes=c * (6 * part + 6 * M * R), flops=c * (900.0 * n + 6 * fft))
    if kind == "adjoint":
        return dict(bytes=part + n * 12 * R + M * R * 26, flops=2200.0 * n)
    if kind == "deposit":
        return dict(bytes=part + 11 * M * R, flops=400.0 * n)
    if kind == "density":
        return dict(bytes=n * (3 * R + 4) + 2 * M * R, flops=40.0 * n + fft)
    return dict(bytes=M * R * 17, flops=15 * fft)


# ---------------------------------------------------------- FP64 restatement --
_CORNERS = [(i, j, k) for i in (0, 1) for j in (0, 1) for k in (0, 1)]


def _sh(f, dx, dy, dz):
    """f at the site (x + dx, y + dy, z + dz); f ends in [z, y, x]."""
    return torch.roll(f, (-dz, -dy, -dx), (-3, -2, -1))


def _step(i):
    return tuple(int(j == i) for j in range(3))


class _Cells:
    """The cells of particles at pos (3, n) and their offsets r in them."""

    def __init__(self, pos, N):
        x = pos * N
        fl = torch.floor(x.detach())
        self.N, self.c, self.r = N, fl.long() & (N - 1), x - fl

    def at(self, d):
        N = self.N
        c = [(self.c[i] + d[i]) & (N - 1) for i in range(3)]
        return c[0] + N * (c[1] + N * c[2])

    def w(self, d, axes=(0, 1, 2)):
        out = None
        for i in axes:
            t = self.r[i] if d[i] else 1.0 - self.r[i]
            out = t if out is None else out * t
        return out

    def interp(self, f, axes=(0, 1, 2)):
        """f interpolated linearly along `axes`, taken at the cell's own site along the others"""
        f, out = f.reshape(-1), 0.0
        for d in _CORNERS:
            if all(d[i] == 0 or i in axes for i in range(3)):
                out = out + self.w(d, axes) * f[self.at(d)]
        return out


def _deposit(pos, q, phi, a, mass, N, phi_links=None, into=None):
    """T00, Tij (00, 01, 02, 11, 12, 22) and T0i's link sums (times 1 + phi_a + phi_b of phi_links when given)."""
    C, M = _Cells(pos, N), N ** 3
    m = mass * M
    q2 = (q * q).sum(0)
    e = torch.sqrt(q2 + a * a)
    f = 3.0 * e + q2 / e
    f2 = (0.5 * f * f + q2 / (1.0 + q2 / (a * a))) / e
    P = phi.reshape(-1)
    T00 = into[0] if into else torch.zeros(M, dtype=torch.float64, device=DEV)
    Tij = into[1] if into else [torch.zeros(M, dtype=torch.float64, device=DEV) for _ in range(6)]
    L = into[2] if into else [torch.zeros(M, dtype=torch.float64, device=DEV) for _ in range(3)]
    add = (lambda t, i, v: t.index_add_(0, i, v)) if into else (lambda t, i, v: t.index_add(0, i, v))
    tf = (1.0 + (4.0 + a * a / (e * e)) * C.interp(phi)) * (m / a) / e
    for d in _CORNERS:
        i, w = C.at(d), C.w(d)
        p = P[i]
        T00 = add(T00, i, w * (e + f * p + f2 * p * p) * (m / a))
        for ax, k in ((0, 0), (1, 3), (2, 5)):
            Tij[k] = add(Tij[k], i, w * tf * q[ax] * q[ax])
    for k, ax, by, along in ((1, 0, 1, 2), (2, 0, 2, 1), (4, 1, 2, 0)):
        for t in (0, 1):
            d = tuple(t * s for s in _step(along))
            Tij[k] = add(Tij[k], C.at(d), C.w(d, (along,)) * tf * q[ax] * q[by])
    for ax in range(3):
        across = tuple(i for i in range(3) if i != ax)
        for d in _CORNERS:
            if d[ax] == 0:
                v = C.w(d, across) * q[ax] * m
                if phi_links is not None:
                    far = tuple(d[i] + _step(ax)[i] for i in range(3))
                    v = v * (1.0 + phi_links.reshape(-1)[C.at(d)] + phi_links.reshape(-1)[C.at(far)])
                L[ax] = add(L[ax], C.at(d), v)
    return T00, Tij, L


def _mass(pos, mass, N, into=None):
    C = _Cells(pos, N)
    out = torch.zeros(N ** 3, dtype=torch.float64, device=DEV) if into is None else into
    for d in _CORNERS:
        v = C.w(d) * (mass * N ** 3)
        out = out.index_add(0, C.at(d), v) if into is None else out.index_add_(0, C.at(d), v)
    return out


def _kick_drift(pos, q, phi, chi, B, b, N, dtau_k, gr=True, mesh=None):
    """update_q and update_pos: new positions (not wrapped), new momenta, the kick's v^2/a^2.
    mesh: the gradient fields of _mesh_fields, when they are shared by several calls"""
    C = _Cells(pos, N)
    dphi, dB = mesh if mesh is not None else _mesh_fields(phi, B, gr)
    G2 = [C.interp(dphi[i]) for i in range(3)]
    a, ad = b["a"], b["a_d"]
    if not gr:
        qn = torch.stack([q[i] - dtau_k * a * N * G2[i] for i in range(3)])
        return pos + b["dtau"] / ad * qn, qn, (qn * qn).sum(0) / (a * a)
    q2 = (q * q).sum(0)
    e2 = q2 + a * a
    e = torch.sqrt(e2)
    Phi = C.interp(phi)
    fac = 4.0 * Phi / e2 * q2 + (1.0 + a * a * Phi / e2) * (q2 + e2) / e2
    qn = []
    for i in range(3):
        g = fac * G2[i] - C.interp(_sh(chi, *_step(i)) - chi, tuple(j for j in range(3) if j != i))
        pg = C.interp(dB[i][i]) * q[i]
        for j in range(3):
            if j != i:  # B_j along i, interpolated along the third axis
                pg = pg + C.interp(dB[j][i], (3 - i - j,)) * q[j]
        g = g + pg / (b["bk"] * e)
        qn.append(q[i] - dtau_k * e * N * g)
    qn = torch.stack(qn)
    w2 = (qn * qn).sum(0)
    f2 = w2 + ad * ad
    v = (1.0 + (3.0 - w2 / f2) * Phi - C.interp(chi)) / torch.sqrt(f2)
    new = [pos[i] + b["dtau"] * (qn[i] * v + C.interp(B[i], tuple(j for j in range(3) if j != i)) / b["bd"])
           for i in range(3)]
    return torch.stack(new), qn, w2 / (a * a)


def _mesh_fields(phi, B, gr):
    """central differences of phi; dB[j][i] the difference of B_j along i (backward for i = j, else forward)"""
    dphi = [0.5 * (_sh(phi, *_step(i)) - _sh(phi, *(-s for s in _step(i)))) for i in range(3)]
    if not gr:
        return dphi, None
    dB = [[(B[j] - _sh(B[j], *(-s for s in _step(i)))) if i == j else (_sh(B[j], *_step(i)) - B[j])
           for i in range(3)] for j in range(3)]
    return dphi, dB


def _kmesh(N):
    n = torch.arange(N, dtype=torch.float64, device=DEV)
    s = 2.0 * N * torch.sin(math.pi * n / N)
    ks = torch.polar(s.abs(), -math.pi * n / N)
    ks = [ks[None, None, : N // 2 + 1], ks[None, :, None], ks[:, None, None]]
    g = s * s
    g = [g[None, None, : N // 2 + 1], g[None, :, None], g[:, None, None]]
    kk = g[0] + g[1] + g[2]
    one = kk.clone()
    one[0, 0, 0] = 1.0
    return ks, g, kk, one


def _rf(f):
    return torch.fft.rfftn(f)


def _irf(F, N):
    return torch.fft.irfftn(F, s=(N, N, N), norm="forward")


def _solve_poisson(src, coeff, modif, N):
    _, _, kk, one = _kmesh(N)
    g = coeff / (-float(N) ** 3) / (kk + modif) if modif else torch.where(kk > 0, coeff / (-float(N) ** 3) / one, 0.0)
    return _irf(_rf(src) * g, N)


def _solve_chi(S, N):
    ks, g, kk, one = _kmesh(N)
    tot = 0.0
    for c, (i, j) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
        w = g[0] + g[1] + g[2] - 3.0 * g[i] if i == j else -6.0 * ks[i] * ks[j]
        tot = tot + w * _rf(S[c])
    return _irf(torch.where(kk > 0, tot / (2.0 * one * one * N), 0.0), N)


def _solve_vector(V, coeff, N):
    ks, _, kk, one = _kmesh(N)
    F = [_rf(v) for v in V]
    dot = (ks[0] * F[0] + ks[1] * F[1] + ks[2] * F[2]) / one
    return [_irf(torch.where(kk > 0, (F[i] - ks[i].conj() * dot) * (4.0 * coeff) / one, 0.0), N) for i in range(3)]


def _source_T00(phi, chi, T00, k):
    r = k["c2"] * (T00 - OM) * (1.0 - 2.0 * phi * (1.0 - phi))
    for i in range(3):
        r = r + 0.125 * (_sh(phi, *(-s for s in _step(i))) - _sh(phi, *_step(i))) ** 2
    return r + (k["c3"] * (1.0 - 3.0 * phi) - k["c1"]) * phi - k["c3"] * chi


def _source_Tij(phi, Tij, c):
    out = []
    for n, (i, j) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
        pi, pj = _sh(phi, *_step(i)), _sh(phi, *_step(j))
        if i == j:
            s = 0.5 * (pi - _sh(phi, *(-t for t in _step(i)))) ** 2
        else:
            pij = _sh(pi, *_step(j))
            s = pi * pj - phi * pij + 0.5 * (phi * phi - pi * pi - pj * pj + pij * pij)
        out.append(s + c * Tij[n])
    return out


def _metric_solves(phi, chi, T00, Tij, L, b, dtau_old, N):
    k = _coefs(N, b, dtau_old)
    phi = _solve_poisson(_source_T00(phi, chi, T00, k), k["pcoeff"], k["modif"], N)
    chi = _solve_chi(_source_Tij(phi, Tij, k["ccoeff"]), N)
    V = [L[i] * (1.0 + phi + _sh(phi, *_step(i))) for i in range(3)]
    return phi, chi, _solve_vector(V, k["bcoeff"], N)


def _chunks(n, size=1 << 23):
    return [slice(i, min(n, i + size)) for i in range(0, n, size)]


def _exact_cycle(case, x):
    N, n = case["mesh"], case["particles"]
    b, mass, M = _background(case), OM / n, N ** 3
    pos, q, phi = x["pos"], x["q"], x["phi"][0]
    chi = torch.zeros_like(phi)
    B = [torch.zeros_like(phi)] * 3
    for _ in range(case["cycles"]):
        if case["gr"]:
            into = tuple([torch.zeros(M, dtype=torch.float64, device=DEV) for _ in range(c)] for c in (1, 6, 3))
            for s in _chunks(n):
                _deposit(pos[:, s], q[:, s], phi, b["a"], mass, N, into=(into[0][0], into[1], into[2]))
            T00, Tij, L = (([t.reshape(N, N, N) for t in v]) for v in into)
            phi, chi, B = _metric_solves(phi, chi, T00[0], Tij, L, b, b["dtau"], N)
            del T00, Tij, L, into
        else:
            rho = torch.zeros(M, dtype=torch.float64, device=DEV)
            for s in _chunks(n):
                _mass(pos[:, s], mass, N, into=rho)
            phi = _solve_poisson(rho.reshape(N, N, N), b["fpg"] / b["a"], 0.0, N)
        mesh = _mesh_fields(phi, B, case["gr"])
        for s in _chunks(n):
            pos[:, s], q[:, s], _ = _kick_drift(pos[:, s], q[:, s], phi, chi, B, b, N, b["dtau"], case["gr"], mesh)
        pos -= torch.floor(pos)
        del mesh
        a = _rk4(b["a_d"], b["fpg"], 0.5 * b["dtau"])
        a_d = _rk4(a, b["fpg"], 0.5 * b["dtau"])
        b = dict(b, a=a, a_d=a_d, bk=a * a * N, bd=a_d * a_d * N)
    return dict(phi=phi[None], chi=chi[None], B=torch.stack(B), pos=pos, q=q)


def _exact_update(case, x):
    N, b = case["mesh"], _background(case)
    mesh = _mesh_fields(x["phi"][0], x["B"], case["gr"])
    pos, q, v2 = x["pos"], x["q"], 0.0
    for s in _chunks(case["particles"]):
        pos[:, s], q[:, s], v = _kick_drift(pos[:, s], q[:, s], x["phi"][0], x["chi"][0], x["B"], b, N, b["dtau"],
                                            case["gr"], mesh)
        v2 = max(v2, float(v.max()))
    pos -= torch.floor(pos)
    return dict(pos=pos, q=q, v2=torch.tensor([v2], dtype=torch.float64))


def _exact_grad(case, x):
    N, fpg = case["mesh"], _fpg(case["mesh"])
    n, mass = N ** 3, OM / N ** 3
    a = 1.0 / 51.0
    dtau = (_horizon(1.0 / 21.0, fpg) - _horizon(a, fpg)) / case["steps"]
    cq = a * (OM / (OM + OL * a ** 3)) ** 0.55 * _hconf(a, fpg)
    psi = x["psi"][0].requires_grad_(True)
    t = (torch.arange(N, dtype=torch.float64, device=DEV) + 0.5) / N
    lag = torch.stack([t.expand(N, N, N), t[:, None].expand(N, N, N), t[:, None, None].expand(N, N, N)]).reshape(3, n)
    C = _Cells(lag, N)
    g = torch.stack([C.interp(_sh(psi, *_step(i)) - psi, tuple(j for j in range(3) if j != i)) for i in range(3)])
    pos, q = lag + N * g, cq * N * g
    phi = chi = torch.zeros_like(psi)
    for k in range(case["steps"]):
        a_d = _rk4(a, fpg, 0.5 * dtau)
        b = dict(fpg=fpg, a=a, a_d=a_d, dtau=dtau, bk=a * a * N, bd=a_d * a_d * N)
        dtau_k = dtau if k else 0.5 * dtau

        def cycle(pos, q, phi, chi, b=b, dtau_k=dtau_k):
            pos = pos - torch.floor(pos.detach())
            if case["gr"]:
                T00, Tij, L = _deposit(pos, q, phi, b["a"], mass, N)
                phi, chi, B = _metric_solves(phi, chi, T00.reshape(N, N, N), [v.reshape(N, N, N) for v in Tij],
                                             [v.reshape(N, N, N) for v in L], b, dtau, N)
            else:
                phi = _solve_poisson(_mass(pos, mass, N).reshape(N, N, N), fpg / b["a"], 0.0, N)
                B = None
            pos, q, _ = _kick_drift(pos, q, phi, chi, B, b, N, dtau_k, case["gr"])
            return pos, q, phi, chi
        pos, q, phi, chi = checkpoint(cycle, pos, q, phi, chi, use_reentrant=False)
        a = _rk4(a_d, fpg, 0.5 * dtau)
    rho = _mass(pos - torch.floor(pos.detach()), mass, N).reshape(1, N, N, N)
    rho.backward(x["g"])
    return dict(rho=rho.detach(), grad=psi.grad[None])


def _exact_adjoint(case, x):
    N, n, b = case["mesh"], case["particles"], _background(case)
    mass = OM / n
    names = ("phi", "chi", "B0", "B1", "B2")
    f = {"phi": x["phi"][0], "chi": x["chi"][0], **{"B%d" % i: x["B"][i] for i in range(3)}}
    acc = {k: torch.zeros_like(v) for k, v in f.items()}
    lx, lq, lold = torch.zeros_like(x["pos"]), torch.zeros_like(x["q"]), torch.zeros_like(f["phi"])
    for s in _chunks(n, 1 << 20):
        leaf = {k: v.detach().requires_grad_(True) for k, v in f.items()}
        pos, q = (x[k][:, s].detach().requires_grad_(True) for k in ("pos", "q"))
        new, qn, _ = _kick_drift(pos, q, leaf["phi"], leaf["chi"], [leaf["B%d" % i] for i in range(3)], b, N, b["dtau"])
        got = torch.autograd.grad([new, qn], [pos, q] + [leaf[k] for k in names], [x["lx"][:, s], x["lq"][:, s]])
        lx[:, s], lq[:, s] = got[0], got[1]
        for k, v in zip(names, got[2:]):
            acc[k] += v
        old = f["phi"].detach().requires_grad_(True)
        T00, Tij, L = _deposit(pos, q, old, b["a"], mass, N)
        S = (T00 * x["lT00"].reshape(-1)).sum() + sum((L[i] * x["lL"][i].reshape(-1)).sum() for i in range(3)) \
            + sum(0.5 * (Tij[i] * x["lTij"][i].reshape(-1)).sum() for i in range(6))
        got = torch.autograd.grad(S, [pos, q, old])
        lx[:, s] += got[0]
        lq[:, s] += got[1]
        lold += got[2]
    return dict(lx=lx, lq=lq, lphi=(acc["phi"] + x["lphi"][0])[None], lchi=(acc["chi"] + x["lchi"][0])[None],
                lB=torch.stack([acc["B%d" % i] for i in range(3)]), lold=lold[None])


def _exact_deposit(case, x):
    N, n = case["mesh"], case["particles"]
    a, mass, M = 1.0 / (1.0 + case["z"]), OM / n, N ** 3
    into = tuple([torch.zeros(M, dtype=torch.float64, device=DEV) for _ in range(c)] for c in (1, 6, 3))
    for s in _chunks(n):
        _deposit(x["pos"][:, s], x["q"][:, s], x["phi"][0], a, mass, N, None if case["links"] else x["phi"][0],
                 into=(into[0][0], into[1], into[2]))
    return dict(zip(("T00", "Tij", "T0i"), (torch.stack(v).reshape(-1, N, N, N) for v in into)))


def _exact_density(case, x):
    N, n = case["mesh"], case["particles"]
    rho = torch.zeros(N ** 3, dtype=torch.float64, device=DEV)
    for s in _chunks(n):
        _mass(x["pos"][:, s], OM / n, N, into=rho)
    rho = rho.reshape(N, N, N)
    return dict(rho=rho[None], F=torch.view_as_real(_rf(rho))[None])


def _exact_solve(case, x):
    b = _background(dict(case, z=2.0))
    phi, chi, B = _metric_solves(x["phi"][0], x["chi"][0], x["T00"][0], x["Tij"], x["L"], b, b["dtau"], case["mesh"])
    return dict(phi=phi[None], chi=chi[None], B=torch.stack(B))


_EXACT = dict(cycle=_exact_cycle, update=_exact_update, grad=_exact_grad, adjoint=_exact_adjoint,
              deposit=_exact_deposit, density=_exact_density, solve=_exact_solve)


def exact(case, seed):
    return _EXACT[case["kind"]](case, _inputs(case, seed))
