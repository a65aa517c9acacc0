// gev_fft.hip -- 3D real<->complex FFT for CDNA4 as three LDS-staged pencil
// passes: x (real<->half-complex, contiguous lines), then y and z (complex,
// strided columns read as TX-wide coalesced row segments).  Radix-8/4/2
// Stockham stages in LDS, twiddles from a per-size table in global memory.
// For 16 <= N <= 128 (FP64: 64) the x and y passes are one kernel per plane
// (gev_fft_plane.hpp), all components of a field in one launch.
#include <algorithm>
#include <type_traits>

#include "gev_common.hpp"
#include "gev_fft_engine.hpp"
#include "gev_fft_plane.hpp"
#include "gev_kernels.hpp"
#include "gev_kops.hpp"

namespace gev {

// Stockham autosort stages over NLINES lines of length L stored in LDS with
// line pitch LDL.  tw = exp(-2 pi i m / (L*TWM)), m in [0, L*TWM).
template <typename T, int L, int NS, int NLINES, int NT, int LDL, int TWM>
__device__ __forceinline__ void fft_stages(cx<T> *buf, int dir, const cx<T> *__restrict__ tw)
{
    if constexpr (NS < L) {
        constexpr int REM = L / NS;
        constexpr int R = (REM >= 8) ? 8 : REM;
        constexpr int NB = L / R;
        constexpr int TOTAL = NB * NLINES;
        constexpr int PER = (TOTAL + NT - 1) / NT;
        cx<T> v[PER][R];
#pragma unroll
        for (int p = 0; p < PER; p++) {
            int b = threadIdx.x + p * NT;
            if (TOTAL % NT == 0 || b < TOTAL) {
                int line = b / NB, j = b % NB;
                int k = j % NS;
                const cx<T> *ln = buf + line * LDL;
#pragma unroll
                for (int r = 0; r < R; r++) v[p][r] = ln[j + r * NB];
                if constexpr (NS > 1) {
#pragma unroll
                    for (int r = 1; r < R; r++) {
                        cx<T> w = tw[(r * k * (L / (NS * R))) * TWM];
                        if (dir > 0) w.y = -w.y;
                        v[p][r] = v[p][r] * w;
                    }
                }
                dftR<T, R>(v[p], dir);
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PER; p++) {
            int b = threadIdx.x + p * NT;
            if (TOTAL % NT == 0 || b < TOTAL) {
                int line = b / NB, j = b % NB;
                int k = j % NS;
                cx<T> *ln = buf + line * LDL;
                int base = (j / NS) * NS * R + k;
#pragma unroll
                for (int r = 0; r < R; r++) ln[base + r * NS] = v[p][r];
            }
        }
        __syncthreads();
        fft_stages<T, L, NS * R, NLINES, NT, LDL, TWM>(buf, dir, tw);
    }
}

constexpr int FFT_NT = 256;

// pad a line so consecutive lines start in different LDS banks
template <typename T, int L> constexpr int ldl_of() { return L + (L >= 16 ? 1 : 0); }

// ------------------------------------------------------------ x pass r2c --
// NLINES consecutive (y,z) lines of N reals -> N/2+1 complex (pitch P).
template <typename T, int N, int NLINES>
__global__ __launch_bounds__(FFT_NT) void k_r2c_x(const T *__restrict__ in, cx<T> *__restrict__ out, int P,
                                                  int64_t nlines, const cx<T> *__restrict__ tw)
{
    constexpr int H = N / 2;
    constexpr int LDL = ldl_of<T, H>();
    __shared__ cx<T> buf[NLINES * LDL];
    const int64_t line0 = (int64_t)blockIdx.x * NLINES;
    const cx<T> *src = reinterpret_cast<const cx<T> *>(in) + line0 * H;
    for (int e = threadIdx.x; e < NLINES * H; e += FFT_NT) {
        int l = e / H, n = e % H;
        buf[l * LDL + n] = (line0 + l < nlines) ? src[e] : mk((T)0, (T)0);
    }
    __syncthreads();
    fft_stages<T, H, 1, NLINES, FFT_NT, LDL, 2>(buf, -1, tw);
    cx<T> *dst = out + line0 * P;
    for (int e = threadIdx.x; e < NLINES * P; e += FFT_NT) {
        int l = e / P, k = e % P;
        if (line0 + l >= nlines) continue;
        cx<T> X = mk((T)0, (T)0);
        if (k <= H) {
            cx<T> Zk = buf[l * LDL + (k % H)];
            cx<T> Zm = conj(buf[l * LDL + ((H - k) % H)]);
            cx<T> Fe = (Zk + Zm) * (T)0.5;
            cx<T> Fo = mul_i(Zk - Zm, -1) * (T)0.5;
            X = Fe + tw[k] * Fo;
        }
        dst[e] = X;
    }
}

// ------------------------------------------------------------ x pass c2r --
template <typename T, int N, int NLINES>
__global__ __launch_bounds__(FFT_NT) void k_c2r_x(const cx<T> *__restrict__ in, T *__restrict__ out, int P,
                                                  int64_t nlines, const cx<T> *__restrict__ tw)
{
    constexpr int H = N / 2;
    constexpr int LDL = ldl_of<T, H>();
    constexpr int LDX = H + 1;
    __shared__ cx<T> xin[NLINES * LDX];
    __shared__ cx<T> buf[NLINES * LDL];
    const int64_t line0 = (int64_t)blockIdx.x * NLINES;
    const cx<T> *src = in + line0 * P;
    for (int e = threadIdx.x; e < NLINES * P; e += FFT_NT) {
        int l = e / P, k = e % P;
        if (k <= H) xin[l * LDX + k] = (line0 + l < nlines) ? src[e] : mk((T)0, (T)0);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NLINES * H; e += FFT_NT) {
        int l = e / H, k = e % H;
        cx<T> Xk = xin[l * LDX + k];
        cx<T> Xm = xin[l * LDX + (H - k)];
        if (k == 0) { Xk.y = 0; Xm.y = 0; } /* DC and Nyquist are real on the x axis */
        cx<T> cm = conj(Xm);
        cx<T> E = Xk + cm;
        cx<T> O = (Xk - cm) * conj(tw[k]);
        buf[l * LDL + k] = E + mul_i(O, +1);
    }
    __syncthreads();
    fft_stages<T, H, 1, NLINES, FFT_NT, LDL, 2>(buf, +1, tw);
    cx<T> *dst = reinterpret_cast<cx<T> *>(out) + line0 * H;
    for (int e = threadIdx.x; e < NLINES * H; e += FFT_NT) {
        int l = e / H, n = e % H;
        if (line0 + l < nlines) dst[e] = buf[l * LDL + n];
    }
}

// ------------------------------------------------ y / z pass (complex) ----
// One workgroup = TX consecutive kx columns x the full line along y (axis 1)
// or z (axis 2) at a fixed other index.  In place.
template <typename T, int L, int TX>
__global__ __launch_bounds__(FFT_NT) void k_c2c_col(cx<T> *__restrict__ data, int P, int axis, int dir,
                                                    const cx<T> *__restrict__ tw)
{
    constexpr int LDL = L + 1;
    __shared__ cx<T> buf[TX * LDL];
    const int ntiles = P / TX;
    const int64_t b = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = (int)(b % ntiles);
    const int64_t o = b / ntiles;
    const int64_t stride = (axis == 1) ? (int64_t)P : (int64_t)P * L;
    const int64_t base = (int64_t)ct * TX + ((axis == 1) ? (int64_t)P * L * o : (int64_t)P * o);
    for (int e = threadIdx.x; e < TX * L; e += FFT_NT) {
        int j = e / TX, c = e % TX;
        buf[c * LDL + j] = data[base + j * stride + c];
    }
    __syncthreads();
    fft_stages<T, L, 1, TX, FFT_NT, LDL, 1>(buf, dir, tw);
    for (int e = threadIdx.x; e < TX * L; e += FFT_NT) {
        int j = e / TX, c = e % TX;
        data[base + j * stride + c] = buf[c * LDL + j];
    }
}

// ============================================ register-staged passes ====
template <typename T> constexpr int tx_of() { return sizeof(T) == 8 ? 8 : 16; }
template <typename T, int L> constexpr int col_tx() { return (tx_of<T>() * L / 8 > 1024) ? 8192 / L : tx_of<T>(); }
template <typename T, int N> constexpr int xlines() { return (sizeof(T) == 8 ? 4096 : 8192) / N; }

// y / z column pass, in place: TX adjacent kx columns x one full line; the
// grid covers one or several consecutive components.
template <typename T, int L, int TX>
__global__ __launch_bounds__(TX * L / 8) void k_col_reg(cx<T> *__restrict__ data, int P, int axis, int dir,
                                                        const cx<T> *__restrict__ tw)
{
    constexpr int NT = TX * L / 8;
    __shared__ cx<T> lds[TX * (L + 1)];
    __shared__ cx<T> twl[L];
    const TwiddleLoad<T, L, NT> twload(twl, tw);
    const int ntiles = P / TX;
    const int64_t b = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = (int)(b % ntiles);
    const int64_t o = b / ntiles;
    const int64_t stride = (axis == 1) ? (int64_t)P : (int64_t)P * L;
    cx<T> *base = data + (int64_t)ct * TX +
                  ((axis == 1) ? (int64_t)P * L * o : (int64_t)P * ((o & (L - 1)) + (int64_t)L * L * (o / L)));
    auto ld = [&](int line, int row) { return base[(int64_t)row * stride + line]; };
    auto st = [&](int line, int row, cx<T> v, int) { base[(int64_t)row * stride + line] = v; };
    reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, dir, ld, st, twload);
}

// Sources of the r2c x pass: the pair of reals (2n, 2n+1) of line L (= y + N z)
template <typename T, int N> struct SrcPlain {
    static constexpr bool kSums = false;
    const T *in;
    __device__ __forceinline__ cx<T> operator()(int64_t L, int n) const
    {
        return reinterpret_cast<const cx<T> *>(in)[L * (N / 2) + n];
    }
};
// component C of the Sij source of prepareFTsource_Tij (gevolution.hpp:64-107),
// computed from Tij and phi while the pass reads it (the same expressions as
// k_prepare_Tij); C: 0 xx, 1 xy, 2 xz, 3 yy, 4 yz, 5 zz
template <typename T, int N, int C> struct SrcSij {
    static constexpr bool kSums = false;
    const T *phi, *Tc;  // Tc: component C of Tij
    T coeff;
    __device__ __forceinline__ cx<T> operator()(int64_t L, int n) const
    {
        constexpr int lg = __builtin_ctz(N), M1 = N - 1;
        const int y = (int)(L & M1), z = (int)(L >> lg);
        const int x = 2 * n, xm = (x - 1) & M1, xp2 = (x + 2) & M1;
        auto row = [&](int dy, int dz) {
            return phi + (int64_t)((y + dy) & M1) * N + (int64_t)((z + dz) & M1) * N * N;
        };
        const cx<T> t = reinterpret_cast<const cx<T> *>(Tc + L * N)[n];
        const T *r0 = phi + L * N;
        const cx<T> pp = reinterpret_cast<const cx<T> *>(r0)[n];  // phi at x, x+1
        const T h = (T)0.5;
        cx<T> out;
        if constexpr (C == 0) {
            const T pm = r0[xm], p2 = r0[xp2];
            out.x = h * (pp.y - pm) * (pp.y - pm) + coeff * t.x;
            out.y = h * (p2 - pp.x) * (p2 - pp.x) + coeff * t.y;
        } else if constexpr (C == 3 || C == 5) {
            const T *ra = C == 3 ? row(1, 0) : row(0, 1), *rb = C == 3 ? row(-1, 0) : row(0, -1);
            const cx<T> a = reinterpret_cast<const cx<T> *>(ra)[n], b = reinterpret_cast<const cx<T> *>(rb)[n];
            out.x = h * (a.x - b.x) * (a.x - b.x) + coeff * t.x;
            out.y = h * (a.y - b.y) * (a.y - b.y) + coeff * t.y;
        } else if constexpr (C == 1 || C == 2) {
            // px py - p pxy + (p^2 - px^2 - py^2 + pxy^2)/2 with y -> z for C = 2
            const T *r1 = C == 1 ? row(1, 0) : row(0, 1);
            const cx<T> q = reinterpret_cast<const cx<T> *>(r1)[n];
            const T p2 = r0[xp2], q2 = r1[xp2];
            auto f = [&](T p, T px, T py, T pxy) { return px * py - p * pxy + h * (p * p - px * px - py * py + pxy * pxy); };
            out.x = f(pp.x, pp.y, q.x, q.y) + coeff * t.x;
            out.y = f(pp.y, p2, q.y, q2) + coeff * t.y;
        } else {
            // py pz - p pyz + (p^2 - py^2 - pz^2 + pyz^2)/2
            const cx<T> a = reinterpret_cast<const cx<T> *>(row(1, 0))[n], b = reinterpret_cast<const cx<T> *>(row(0, 1))[n],
                        d = reinterpret_cast<const cx<T> *>(row(1, 1))[n];
            auto f = [&](T p, T py, T pz, T pyz) { return py * pz - p * pyz + h * (p * p - py * py - pz * pz + pyz * pyz); };
            out.x = f(pp.x, a.x, b.x, d.x) + coeff * t.x;
            out.y = f(pp.y, a.y, b.y, d.y) + coeff * t.y;
        }
        return out;
    }
};

// component C of T0i from its link sums s (the particle parts of
// projection_T0i, gevolution.hpp:2031-2201) and the link factor
// 1 + phi(x) + phi(x + e_C) of the link from site x along axis C
template <typename T, int N, int C> struct SrcT0iLink {
    static constexpr bool kSums = false;
    const T *phi, *s;  // s: component C of the link sums
    __device__ __forceinline__ cx<T> operator()(int64_t L, int n) const
    {
        constexpr int lg = __builtin_ctz(N), M1 = N - 1;
        const int y = (int)(L & M1), z = (int)(L >> lg);
        const cx<T> sv = reinterpret_cast<const cx<T> *>(s + L * N)[n];
        const T *r0 = phi + L * N;
        const cx<T> p = reinterpret_cast<const cx<T> *>(r0)[n];  // phi at x, x+1
        cx<T> e;  // phi at the far end of the links from x and x+1
        if constexpr (C == 0) {
            e = mk(p.y, r0[(2 * n + 2) & M1]);
        } else {
            const int64_t row = C == 1 ? (int64_t)((y + 1) & M1) + (int64_t)z * N : (int64_t)y + (int64_t)((z + 1) & M1) * N;
            e = reinterpret_cast<const cx<T> *>(phi + row * N)[n];
        }
        return mk(sv.x * ((T)1 + p.x + e.x), sv.y * ((T)1 + p.y + e.y));
    }
};

// prepareFTsource's T00 form (gevolution.hpp:160-171, the same expressions as
// k_prepare_T00) evaluated while the Poisson solve's x pass reads it; every
// copy sums the source and the result it produced (FP64) for the k=0 mode
template <typename T, int N> struct SrcT00 {
    static constexpr bool kSums = true;
    const T *phi, *chi, *src;
    T bg, c1, c2, c3;
    double acc[2];
    __device__ __forceinline__ cx<T> operator()(int64_t L, int n)
    {
        constexpr int lg = __builtin_ctz(N), M1 = N - 1;
        const int y = (int)(L & M1), z = (int)(L >> lg);
        auto pair = [&](const T *f, int64_t line) { return reinterpret_cast<const cx<T> *>(f + line * N)[n]; };
        const int64_t ym = (int64_t)((y - 1) & M1) + (int64_t)z * N, yp = (int64_t)((y + 1) & M1) + (int64_t)z * N;
        const int64_t zm = (int64_t)y + (int64_t)((z - 1) & M1) * N, zp = (int64_t)y + (int64_t)((z + 1) & M1) * N;
        const T *r0 = phi + L * N;
        const cx<T> p = pair(phi, L), s = pair(src, L), ch = pair(chi, L);
        const cx<T> a = pair(phi, ym), b = pair(phi, yp), d = pair(phi, zm), e = pair(phi, zp);
        const T pm = r0[(2 * n - 1) & M1], p2 = r0[(2 * n + 2) & M1];
        auto res = [&](T sv, T pv, T xm, T xp, T ym_, T yp_, T zm_, T zp_, T cv) {
            T r = c2 * (sv - bg);
            r *= (T)1 - (T)2 * pv * ((T)1 - pv);
            const T d0 = xm - xp, d1 = ym_ - yp_, d2 = zm_ - zp_;
            r += (T)0.125 * d0 * d0;
            r += (T)0.125 * d1 * d1;
            r += (T)0.125 * d2 * d2;
            r += (c3 * ((T)1 - (T)3 * pv) - c1) * pv - c3 * cv;
            return r;
        };
        const T r0v = res(s.x, p.x, pm, p.y, a.x, b.x, d.x, e.x, ch.x);
        const T r1v = res(s.y, p.y, p.x, p2, a.y, b.y, d.y, e.y, ch.y);
        acc[0] += (double)s.x + (double)s.y;
        acc[1] += (double)r0v + (double)r1v;
        return mk(r0v, r1v);
    }
};

// x pass r2c: NL consecutive lines of N reals -> N/2+1 complex (pitch P)
template <typename T, int N, int NL, typename Src>
__global__ __launch_bounds__(NL * N / 16) void k_r2c_x_reg(Src src, cx<T> *__restrict__ out, int P, int64_t nlines,
                                                           const cx<T> *__restrict__ tw, double *partials)
{
    constexpr int H = N / 2, NT = NL * H / 8, LDL = H + 1;
    __shared__ cx<T> lds[NL * LDL];
    __shared__ cx<T> twl[N];
    const TwiddleLoad<T, N, NT> twload(twl, tw);
    const int64_t line0 = (int64_t)blockIdx.x * NL;
    Src sr = src;  // a source that sums keeps its sums per thread
    if constexpr (Src::kSums) sr.acc[0] = sr.acc[1] = 0.0;
    auto ld = [&](int line, int n) { return (line0 + line < nlines) ? sr(line0 + line, n) : mk((T)0, (T)0); };
    auto st = [&](int line, int k, cx<T> v, int) { lds[line * LDL + k] = v; };
    reg_fft<T, H, NL, false, 2, true, 1>(lds, twl, -1, ld, st, twload);
    if constexpr (Src::kSums) {
        // workgroup partials of the two sums, one slot pair per workgroup
        __shared__ double ws[NT / 64][2];
        double v0 = sr.acc[0], v1 = sr.acc[1];
        for (int o = 32; o > 0; o >>= 1) {
            v0 += __shfl_xor(v0, o, 64);
            v1 += __shfl_xor(v1, o, 64);
        }
        if ((threadIdx.x & 63) == 0) { ws[threadIdx.x >> 6][0] = v0; ws[threadIdx.x >> 6][1] = v1; }
        __syncthreads();
        if (threadIdx.x == 0) {
            double t0 = 0.0, t1 = 0.0;
            for (int w = 0; w < NT / 64; w++) { t0 += ws[w][0]; t1 += ws[w][1]; }
            partials[2 * (int64_t)blockIdx.x] = t0;
            partials[2 * (int64_t)blockIdx.x + 1] = t1;
        }
    }
    __syncthreads();
    cx<T> *dst = out + line0 * P;
    for (int e = threadIdx.x; e < NL * P; e += NT) {
        int l = e / P, k = e % P;
        if (line0 + l >= nlines) continue;
        cx<T> X = mk((T)0, (T)0);
        if (k <= H) {
            cx<T> Zk = lds[l * LDL + (k % H)];
            cx<T> Zm = conj(lds[l * LDL + ((H - k) % H)]);
            cx<T> Fe = (Zk + Zm) * (T)0.5;
            cx<T> Fo = mul_i(Zk - Zm, -1) * (T)0.5;
            X = Fe + twl[k] * Fo;
        }
        dst[e] = X;
    }
}

// x pass r2c of NC components of the same lines in one workgroup (out + c NK
// for component c): the sources of all components read the same phi rows,
// which the later components then find in the caches.  Src::get<C>(L, n)
// gives component C's pair n of line L.
template <typename T, int N, int NL, int NC, typename Src>
__global__ __launch_bounds__(NL * N / 16) void k_r2c_x_multi(Src src, cx<T> *__restrict__ out, int P, int64_t NK,
                                                             int64_t nlines, const cx<T> *__restrict__ tw)
{
    constexpr int H = N / 2, NT = NL * H / 8, LDL = H + 1;
    __shared__ cx<T> lds[NL * LDL];
    __shared__ cx<T> twl[N];
    const TwiddleLoad<T, N, NT> twload(twl, tw);
    const int64_t line0 = (int64_t)blockIdx.x * NL;
    auto comp = [&](auto cc) {
        constexpr int C = decltype(cc)::value;
        auto ld = [&](int line, int n) {
            return (line0 + line < nlines) ? src.template get<C>(line0 + line, n) : mk((T)0, (T)0);
        };
        auto st = [&](int line, int k, cx<T> v, int) { lds[line * LDL + k] = v; };
        if constexpr (C == 0) {
            reg_fft<T, H, NL, false, 2, true, 1>(lds, twl, -1, ld, st, twload);
        } else {
            __syncthreads();  // the previous component's stores have read lds
            reg_fft<T, H, NL, false, 2, true, 1>(lds, twl, -1, ld, st);
        }
        __syncthreads();
        cx<T> *dst = out + C * NK + line0 * P;
        for (int e = threadIdx.x; e < NL * P; e += NT) {
            int l = e / P, k = e % P;
            if (line0 + l >= nlines) continue;
            cx<T> X = mk((T)0, (T)0);
            if (k <= H) {
                cx<T> Zk = lds[l * LDL + (k % H)];
                cx<T> Zm = conj(lds[l * LDL + ((H - k) % H)]);
                cx<T> Fe = (Zk + Zm) * (T)0.5;
                cx<T> Fo = mul_i(Zk - Zm, -1) * (T)0.5;
                X = Fe + twl[k] * Fo;
            }
            dst[e] = X;
        }
    };
    comp(std::integral_constant<int, 0>{});
    if constexpr (NC > 1) comp(std::integral_constant<int, 1>{});
    if constexpr (NC > 2) comp(std::integral_constant<int, 2>{});
    if constexpr (NC > 3) comp(std::integral_constant<int, 3>{});
    if constexpr (NC > 4) comp(std::integral_constant<int, 4>{});
    if constexpr (NC > 5) comp(std::integral_constant<int, 5>{});
}

// projectFTscalar takes only the trace-free part of Sij, so two differences of
// the diagonal and the three off-diagonal components carry it:
//   0: S_xx - S_zz, 1: S_yy - S_zz, 2: S_xy, 3: S_xz, 4: S_yz
// (five half spectra to write, transform and read instead of six: 512^3 FP64
// phi + chi + B solves 20.48 -> 19.82 ms).  FP64 only.  In FP32 five gain 1 % of
// a 512^3 mixed cycle (meshes of 256^3 and more; smaller ones transform planes);
// six keep that cycle's chi as it is, where a last-bit change lets some particle
// cross a cell face a cycle earlier or later and moves its link deposits by a
// site (largest change of B 2e-3 to 3e-3, as between two runs of one build).
template <typename T> constexpr int sij_spectra() { return sizeof(T) == 8 ? 5 : 6; }
// From prepareFTsource(phi, Tij, coeff), Tij's component c at Tij + c M:
template <typename T, int N> struct SrcSijX {
    const T *phi, *Tij;
    int64_t M;
    T coeff;
    template <int C> __device__ __forceinline__ cx<T> get(int64_t L, int n) const
    {
        auto S = [&](auto cc) {
            constexpr int K = decltype(cc)::value;
            return SrcSij<T, N, K>{phi, Tij + K * M, coeff}(L, n);
        };
        if constexpr (sij_spectra<T>() == 6) return S(std::integral_constant<int, C>{});
        else if constexpr (C < 2)
            return S(std::integral_constant<int, C == 0 ? 0 : 3>{}) - S(std::integral_constant<int, 5>{});
        else return S(std::integral_constant<int, C == 2 ? 1 : C == 3 ? 2 : 4>{});
    }
};
// and from Sij itself
template <typename T, int N> struct SrcPlainX {
    const T *Sij;
    int64_t M;
    template <int C> __device__ __forceinline__ cx<T> get(int64_t L, int n) const
    {
        auto S = [&](int c) { return SrcPlain<T, N>{Sij + c * M}(L, n); };
        if constexpr (sij_spectra<T>() == 6) return S(C);
        else if constexpr (C < 2) return S(C == 0 ? 0 : 3) - S(5);
        else return S(C == 2 ? 1 : C == 3 ? 2 : 4);
    }
};

template <typename T, int N, int NC, typename Src>
static void launch_r2c_multi(const Src &src, cx<T> *out, int P, int64_t NK, int64_t nlines, const cx<T> *tw,
                             hipStream_t s)
{
    constexpr int NL = xlines<T, N>();
    int64_t nb = (nlines + NL - 1) / NL;
    hipLaunchKernelGGL((k_r2c_x_multi<T, N, NL, NC, Src>), dim3((unsigned)nb), dim3(NL * N / 16), 0, s, src, out, P, NK,
                       nlines, tw);
}

// x pass c2r: N/2+1 complex (pitch P) -> N reals; DC and Nyquist taken as real.
// The lines are staged in LDS with one coalesced read per element, the first
// stage pairs X[k] with X[H-k] from there, and the last stage's outputs go
// back through LDS so that the global stores are consecutive per lane group.
template <typename T, int N, int NL>
__global__ __launch_bounds__(NL * N / 16) void k_c2r_x_reg(const cx<T> *__restrict__ in, T *__restrict__ out, int P,
                                                           int64_t nlines, const cx<T> *__restrict__ tw)
{
    constexpr int H = N / 2, NT = NL * H / 8, LDL = H + 1;
    __shared__ cx<T> lds[NL * LDL];
    __shared__ cx<T> twl[N];
    const TwiddleLoad<T, N, NT> twload(twl, tw);
    const int64_t line0 = (int64_t)blockIdx.x * NL;
    const cx<T> *src = in + line0 * P;
    static_assert(LDL == H + 1, "a staged line holds X[0..H]");
    for (int e = threadIdx.x; e < NL * LDL; e += NT) {
        const int l = e / LDL;
        lds[e] = (line0 + l < nlines) ? src[(int64_t)l * P + (e - l * LDL)] : mk((T)0, (T)0);
    }
    twload();
    __syncthreads();
    auto ld = [&](int line, int k) {
        const cx<T> *row = lds + line * LDL;
        cx<T> Xk = row[k];
        cx<T> Xm = row[H - k];
        if (k == 0) { Xk.y = 0; Xm.y = 0; }
        cx<T> cm = conj(Xm);
        cx<T> E = Xk + cm;
        cx<T> O = (Xk - cm) * conj(twl[k]);
        return E + mul_i(O, +1);
    };
    cx<T> *dst = reinterpret_cast<cx<T> *>(out) + line0 * H;
    auto st = [&](int line, int n, cx<T> v, int) { lds[line * LDL + n] = v; };
    reg_fft<T, H, NL, false, 2, true, 1>(lds, twl, +1, ld, st);
    __syncthreads();
    for (int e = threadIdx.x; e < NL * H; e += NT) {
        const int l = e / H;
        if (line0 + l < nlines) dst[e] = lds[l * LDL + (e - l * H)];
    }
}

// ---------------------------------------------------------- dispatchers ---

template <typename T, int N, typename Src>
static void launch_r2c_src(const Src &src, cx<T> *out, int P, int64_t nlines, const cx<T> *tw, hipStream_t s,
                           double *partials = nullptr)
{
    constexpr int NL = xlines<T, N>();
    int64_t nb = (nlines + NL - 1) / NL;
    hipLaunchKernelGGL((k_r2c_x_reg<T, N, NL, Src>), dim3((unsigned)nb), dim3(NL * N / 16), 0, s, src, out, P, nlines,
                       tw, partials);
}

template <typename T, int N>
static void launch_r2c(const T *in, cx<T> *out, int P, int64_t nlines, const cx<T> *tw, hipStream_t s)
{
    if constexpr (N >= 128) {
        launch_r2c_src<T, N>(SrcPlain<T, N>{in}, out, P, nlines, tw, s);
    } else {
        static_assert(N <= 8, "16 <= N <= 64 transforms whole planes");
        constexpr int NLINES = 4096 / N > 1024 ? 1024 : 4096 / N;
        int64_t nb = (nlines + NLINES - 1) / NLINES;
        hipLaunchKernelGGL((k_r2c_x<T, N, NLINES>), dim3((unsigned)nb), dim3(FFT_NT), 0, s, in, out, P, nlines, tw);
    }
}

template <typename T, int N>
static void launch_c2r(const cx<T> *in, T *out, int P, int64_t nlines, const cx<T> *tw, hipStream_t s)
{
    if constexpr (N >= 128) {
        constexpr int NL = xlines<T, N>();
        int64_t nb = (nlines + NL - 1) / NL;
        hipLaunchKernelGGL((k_c2r_x_reg<T, N, NL>), dim3((unsigned)nb), dim3(NL * N / 16), 0, s, in, out, P, nlines,
                           tw);
    } else {
        static_assert(N <= 8, "16 <= N <= 64 transforms whole planes");
        constexpr int NLINES = 4096 / N > 1024 ? 1024 : 4096 / N;
        int64_t nb = (nlines + NLINES - 1) / NLINES;
        hipLaunchKernelGGL((k_c2r_x<T, N, NLINES>), dim3((unsigned)nb), dim3(FFT_NT), 0, s, in, out, P, nlines, tw);
    }
}

// axis 1 (y) or 2 (z) of ncomp consecutive components
template <typename T, int N>
static void launch_col(cx<T> *data, int P, int axis, int dir, const cx<T> *tw, hipStream_t s, int ncomp = 1)
{
    if constexpr (N >= 16) {
        constexpr int TX = col_tx<T, N>();
        int64_t nb = (int64_t)(P / TX) * N * ncomp;
        hipLaunchKernelGGL((k_col_reg<T, N, TX>), dim3((unsigned)nb), dim3(TX * N / 8), 0, s, data, P, axis, dir, tw);
    } else {
        constexpr int TX = tx_of<T>();
        int64_t nb = (int64_t)(P / TX) * N;
        for (int c = 0; c < ncomp; c++)
            hipLaunchKernelGGL((k_c2c_col<T, N, TX>), dim3((unsigned)nb), dim3(FFT_NT), 0, s,
                               data + (int64_t)c * P * N * N, P, axis, dir, tw);
    }
}

// the sources of the plane transforms' components (k_fwd_plane)
template <typename T, int N> struct CompPlain {
    const T *in;
    int64_t M;
    template <class F> __device__ __forceinline__ void with(int c, F f) const { f(SrcPlain<T, N>{in + c * M}); }
};

// FP64 planes of N = 128 fill the LDS (one workgroup per CU, 64 to 128 of the
// 256 CUs) and lose to the separate passes: 128^3 FP64 GR cycles 936 against
// 903 us each; FP32 ones gain (see gev_fft_plane.hpp)
template <typename T> constexpr bool plane_size(int N) { return N >= 16 && (N <= 64 || (N == 128 && sizeof(T) == 4)); }

// forward x and y passes of ncomp components (r2c without the z pass) from
// plane sources, and the inverse y and x passes
template <typename T, int N, class Comp>
static void launch_fwd_plane(gev_ctx *c, const Comp &comp, cx<T> *out, int ncomp, const cx<T> *tw,
                             double *partials = nullptr)
{
    hipLaunchKernelGGL((k_fwd_plane<T, N, Comp>), dim3(N / plane_np<N>(), ncomp), dim3(plane_nt<N>()), 0, c->stream,
                       comp, out, c->NK, tw, partials);
}
template <typename T, int N> static void fwd_xy(gev_ctx *c, const T *in, cx<T> *out, int ncomp, const cx<T> *tw)
{
    if constexpr (plane_size<T>(N)) {
        launch_fwd_plane<T, N>(c, CompPlain<T, N>{in, c->M}, out, ncomp, tw);
    } else {
        for (int i = 0; i < ncomp; i++) {
            launch_r2c<T, N>(in + i * c->M, out + i * c->NK, c->P, (int64_t)N * N, tw, c->stream);
            launch_col<T, N>(out + i * c->NK, c->P, 1, -1, tw, c->stream);
        }
    }
}
template <typename T, int N> static void inv_yx(gev_ctx *c, cx<T> *in, T *out, int ncomp, const cx<T> *tw)
{
    if constexpr (plane_size<T>(N)) {
        hipLaunchKernelGGL((k_inv_plane<T, N>), dim3(N / plane_np<N>(), ncomp), dim3(plane_nt<N>()), 0, c->stream, in,
                           out, c->NK, c->M, tw);
    } else {
        for (int i = 0; i < ncomp; i++) {
            launch_col<T, N>(in + i * c->NK, c->P, 1, +1, tw, c->stream);
            launch_c2r<T, N>(in + i * c->NK, out + i * c->M, c->P, (int64_t)N * N, tw, c->stream);
        }
    }
}

#define GEV_FOR_FUSED_N(X) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)
#define GEV_FOR_EACH_N(X) X(4) X(8) GEV_FOR_FUSED_N(X)

// components at a time: all of them where a component is small (launches and
// latency count); one by one on large meshes, whose passes then find the
// component just written in the Infinity Cache
template <typename T, int N> constexpr int fft_batch() { return plane_size<T>(N) ? 64 : 1; }

template <typename T>
int fft_r2c_impl(gev_ctx *ctx, const T *in, cx<T> *out, int ncomp, const cx<T> *tw)
{
    const int64_t M = ctx->M, NK = ctx->NK;
    switch (ctx->N) {
#define X(n)                                                                        \
    case n:                                                                         \
        for (int c = 0; c < ncomp; c += fft_batch<T, n>()) {                           \
            const int m = std::min(ncomp - c, fft_batch<T, n>());                      \
            fwd_xy<T, n>(ctx, in + c * M, out + c * NK, m, tw);                     \
            launch_col<T, n>(out + c * NK, ctx->P, 2, -1, tw, ctx->stream, m);      \
        }                                                                           \
        break;
        GEV_FOR_EACH_N(X)
#undef X
    default: gev_set_error("unsupported N"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

template <typename T>
int fft_c2r_impl(gev_ctx *ctx, cx<T> *in, T *out, int ncomp, const cx<T> *tw)
{
    const int64_t M = ctx->M, NK = ctx->NK;
    switch (ctx->N) {
#define X(n)                                                                        \
    case n:                                                                         \
        for (int c = 0; c < ncomp; c += fft_batch<T, n>()) {                           \
            const int m = std::min(ncomp - c, fft_batch<T, n>());                      \
            launch_col<T, n>(in + c * NK, ctx->P, 2, +1, tw, ctx->stream, m);       \
            inv_yx<T, n>(ctx, in + c * NK, out + c * M, m, tw);                     \
        }                                                                           \
        break;
        GEV_FOR_EACH_N(X)
#undef X
    default: gev_set_error("unsupported N"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

// ===================================== z pass fused with a k-space solve ====
// Forward z transforms of the NIN input components of TX adjacent kx columns
// (one ky), the per-mode operator applied in registers, inverse z transforms
// of the NOUT outputs.  Replaces [z pass, k-space kernel, inverse z pass]:
// every mode is read once and written once instead of three times each.
// In place (in == out) is allowed: a workgroup reads all its columns before
// writing them and no two workgroups share a column.
// ZOP_SCALAR: projectFTscalar, every weight of which is linear in the kz
// factors g2 = gk2[kz] and k2 = ks[kz], so three combinations of the six Sij
// components carry it through the z transform:
//   A = (g1 - 2 g0) S_xx - 6 k0 k1 S_xy + (g0 - 2 g1) S_yy + (g0 + g1) S_zz
//   B = S_xx + S_yy - 2 S_zz,   C = -6 (k0 S_xz + k1 S_yz)
// ZOP_SCALAR3: the same from the three groups that k_col_comb forms in the y
// pass (below) instead of the six components
// ZOP_ADJ_SCALAR: projectFTscalar's adjoint, one component in and the six
// conj(w_c) lchi / (2 k^4 N) out
enum { ZOP_POISSON = 0, ZOP_SCALAR = 1, ZOP_VECTOR = 2, ZOP_SCALAR3 = 3, ZOP_ADJ_SCALAR = 4 };

struct ZParams {
    const double *gk2;
    const cx<double> *ks;
    double coeff, modif;  // Poisson: coeff pre-scaled by -1/N^3; vector: as projectFTvector
    double k0re, k0im;    // Poisson: value taken for the k=0 mode when k0set
    int k0set;
    // Poisson with the source formed in the x pass: the pass's workgroup sums
    // (nparts pairs), reduced by the workgroup that holds the k=0 mode into
    // sums[0], sums[1]; the real part of that mode is then sums[1] when k0set
    const double *parts;
    int nparts;
    double *sums;
};

// ============================ y pass of Sij forming the groups of the z solve ==
// The y transforms of the six Sij components, or in FP64 the five trace-free
// combinations of SrcSijX (x-transformed, at data + c NK), of TX adjacent kx
// columns and one z, each
// output mode added with its (kx, ky) weight of projectFTscalar into the three
// groups that the z solve transforms (gevolution.hpp:317-323 with g = gridk2,
// k = kshift; U = S_xx - S_zz, V = S_yy - S_zz):
//   A = (g1 - 2 g0) S_xx - 6 k0 k1 S_xy + (g0 - 2 g1) S_yy + (g0 + g1) S_zz
//     = (g1 - 2 g0) U + (g0 - 2 g1) V - 6 k0 k1 S_xy
//   B = S_xx + S_yy - 2 S_zz = U + V,   C = -6 (k0 S_xz + k1 S_yz)
// written over components 0..2 (every column of the workgroup is read before
// any is written; no other workgroup touches them).  Padding columns
// (kx > N/2) get 0.  Replaces six y passes and the z solve's reads of six
// components by reads of three.
template <typename T, int L, int TX>
__global__ __launch_bounds__(TX * L / 8) void k_col_comb(cx<T> *data, int P, int64_t NK, const cx<T> *__restrict__ tw,
                                                         const double *__restrict__ gk2, const cx<double> *__restrict__ ks)
{
    constexpr int NIN = sij_spectra<T>();
    constexpr int NT = TX * L / 8;
    __shared__ cx<T> lds[TX * (L + 1)];
    __shared__ cx<T> twl[L];
    // the k tables in the transform's precision (the weights are applied in it)
    __shared__ T gkl[L];
    __shared__ cx<T> ksl[L];
    auto tables = [&]() {
        for (int m = threadIdx.x; m < L; m += NT) {
            twl[m] = tw[m];
            gkl[m] = (T)gk2[m];
            ksl[m] = mk((T)ks[m].x, (T)ks[m].y);
        }
    };
    const int ntiles = P / TX;
    const int64_t b = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = (int)(b % ntiles);
    const int64_t z = b / ntiles;
    cx<T> *base = data + (int64_t)ct * TX + (int64_t)P * L * z;
    // byte offset of (row, column) inside a component's (kx, y) plane of this
    // z: 32 bits, so every access takes the workgroup's base from scalar
    // registers instead of a 64-bit address per element
    auto boff = [&](int row, int ln) -> uint32_t { return ((uint32_t)row * (uint32_t)P + (uint32_t)ln) * (uint32_t)sizeof(cx<T>); };
    const int line = threadIdx.x % TX;  // the column every slot of this thread lands in
    const int kx = ct * TX + line;
    const bool valid = kx <= L / 2;
    const T g0 = valid ? (T)gk2[kx] : (T)0;
    const cx<T> k0 = valid ? mk((T)ks[kx].x, (T)ks[kx].y) : mk((T)0, (T)0);
    const cx<T> k0m = k0 * (T)-6;
    cx<T> A[8], B[8], C[8], v[8];
    int rows[8];
    auto comp = [&](auto cc) {
        constexpr int c = decltype(cc)::value;
        const cx<T> *src = base + c * NK;
        auto ld = [&](int ln, int row) { return *reinterpret_cast<const cx<T> *>(reinterpret_cast<const char *>(src) + boff(row, ln)); };
        auto st = [&](int, int row, cx<T> val, int slot) {
            if constexpr (c == 0) rows[slot] = row;
            v[slot] = val;
        };
        if constexpr (c == 0) {
            reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, -1, ld, st, tables);
        } else {
            __syncthreads();  // the previous transform is done with lds
            reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, -1, ld, st);
        }
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int row = rows[s];
            if constexpr (NIN == 6) {
                if constexpr (c == 0) {
                    A[s] = v[s] * (gkl[row] - (T)2 * g0);
                    B[s] = v[s];
                } else if constexpr (c == 1) {
                    A[s] = A[s] + (k0m * ksl[row]) * v[s];
                } else if constexpr (c == 2) {
                    C[s] = k0m * v[s];
                } else if constexpr (c == 3) {
                    A[s] = A[s] + v[s] * (g0 - (T)2 * gkl[row]);
                    B[s] = B[s] + v[s];
                } else if constexpr (c == 4) {
                    C[s] = C[s] + (ksl[row] * (T)-6) * v[s];
                } else {
                    A[s] = A[s] + v[s] * (g0 + gkl[row]);
                    B[s] = B[s] - v[s] * (T)2;
                }
            } else if constexpr (c == 0) {
                A[s] = v[s] * (gkl[row] - (T)2 * g0);
                B[s] = v[s];
            } else if constexpr (c == 1) {
                A[s] = A[s] + v[s] * (g0 - (T)2 * gkl[row]);
                B[s] = B[s] + v[s];
            } else if constexpr (c == 2) {
                A[s] = A[s] + (k0m * ksl[row]) * v[s];
            } else if constexpr (c == 3) {
                C[s] = k0m * v[s];
            } else {
                C[s] = C[s] + (ksl[row] * (T)-6) * v[s];
            }
        }
    };
    comp(std::integral_constant<int, 0>{});
    comp(std::integral_constant<int, 1>{});
    comp(std::integral_constant<int, 2>{});
    comp(std::integral_constant<int, 3>{});
    comp(std::integral_constant<int, 4>{});
    if constexpr (NIN == 6) comp(std::integral_constant<int, 5>{});
    // (selects on the scalar parts: a select of whole structs becomes a select
    // of their addresses, which keeps the arrays out of registers)
    auto put = [&](cx<T> *dst, int s, cx<T> val) {
        *reinterpret_cast<cx<T> *>(reinterpret_cast<char *>(dst) + boff(rows[s], line)) =
            mk(valid ? val.x : (T)0, valid ? val.y : (T)0);
    };
#pragma unroll
    for (int s = 0; s < 8; s++) {
        put(base, s, A[s]);
        put(base + NK, s, B[s]);
        put(base + 2 * NK, s, C[s]);
    }
}

template <typename T, int L> constexpr int comb_tx() { return 4096 / L < 8 ? 4096 / L : 8; }

template <typename T, int N>
static void launch_col_comb(cx<T> *data, int P, int64_t NK, const cx<T> *tw, const ZParams &zp, hipStream_t s)
{
    constexpr int TX = comb_tx<T, N>();
    const int64_t nb = (int64_t)(P / TX) * N;
    hipLaunchKernelGGL((k_col_comb<T, N, TX>), dim3((unsigned)nb), dim3(TX * N / 8), 0, s, data, P, NK, tw, zp.gk2,
                       zp.ks);
}

// FP32 vector projection from L = 128 up: 4 waves per SIMD (two workgroups
// per CU) at the price of a spill of up to 56 bytes, 4.5 -> 4.1 ms for the
// 512^3 B solve; the scalar projection and FP64 measured no better that way
template <typename T, int L, int OP> constexpr int zs_waves() { return (OP == ZOP_VECTOR && sizeof(T) == 4 && L >= 128) ? 4 : 1; }

// The type of ZOP_SCALAR's weights and group sums.  Up to L = 64 FP64 in both
// forms, as k_project_ft_scalar's: these meshes are bound by latency and FP64
// costs no time there (mixed chi solves of 16^3, 32^3, 64^3 14.6, 15.7, 20.9 us
// with FP32 sums, 14.5, 15.3, 21.0 with FP64 ones), and a Sij that is all trace
// then gives nothing instead of 1e-8 to 1e-7 of its single components' chi.  At
// 128 it costs 1 % (56.8, 57.4 us): the transform's precision, as k_col_comb.
template <typename T, int L> using scalar_weight_t = std::conditional_t<(L <= 64), double, T>;

template <typename T, int L, int TX, int OP>
__global__ __launch_bounds__(TX * L / 8, (zs_waves<T, L, OP>())) void k_zsolve(const cx<T> *in, cx<T> *out, int P, int64_t NK,
                                                       const cx<T> *__restrict__ tw, ZParams zp)
{
    constexpr int NT = TX * L / 8, LDL = L + 1, NW = (NT + 63) / 64;
    constexpr int NV = OP == ZOP_VECTOR ? 3 : 1;  // values per mode held at once
    __shared__ cx<T> lds[TX * LDL];
    __shared__ cx<T> twl[L];
    const TwiddleLoad<T, L, NT> twload(twl, tw);
    const int ntiles = P / TX;
    const int64_t b = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = (int)(b % ntiles);
    const int ky = (int)(b / ntiles);
    const int64_t stride = (int64_t)P * L;
    const int64_t off = (int64_t)ct * TX + (int64_t)P * ky;
    const int H = L / 2;
    int lines[8], poss[8];
    cx<T> vin[NV][8];
    const double gy = zp.gk2[ky];
    const cx<double> kyv = zp.ks[ky];
    __shared__ double k0src;  // the k=0 value summed here (Poisson)
    if constexpr (OP == ZOP_POISSON) {
        if (zp.parts && ct == 0 && ky == 0) {
            // fixed order: per thread, per wave, then the waves in turn
            __shared__ double ws[NW][2];
            double v0 = 0.0, v1 = 0.0;
            for (int j = threadIdx.x; j < zp.nparts; j += NT) {
                v0 += zp.parts[2 * j];
                v1 += zp.parts[2 * j + 1];
            }
            for (int o = NT < 64 ? NT / 2 : 32; o > 0; o >>= 1) {
                v0 += __shfl_xor(v0, o, 64);
                v1 += __shfl_xor(v1, o, 64);
            }
            if ((threadIdx.x & 63) == 0) { ws[threadIdx.x >> 6][0] = v0; ws[threadIdx.x >> 6][1] = v1; }
            __syncthreads();
            if (threadIdx.x == 0) {
                double t0 = 0.0, t1 = 0.0;
                for (int w = 0; w < NW; w++) { t0 += ws[w][0]; t1 += ws[w][1]; }
                zp.sums[0] = t0;
                zp.sums[1] = t1;
                k0src = t1;
            }
        }
    }
    // forward z transform of component c, read by the transform's first stage
    // straight from memory; every output mode goes to st(line, kz, value, slot)
    auto forward = [&](auto comp, auto &st) {
        constexpr int c = decltype(comp)::value;
        const cx<T> *src = in + c * NK + off;
        auto ld = [&](int line, int row) { return src[(int64_t)row * stride + line]; };
        if constexpr (c == 0) {
            reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, -1, ld, st, twload);
        } else {
            __syncthreads();  // previous transform done with lds
            reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, -1, ld, st);
        }
    };
    // inverse z transform of component j of the output from vin[held]
    auto inverse = [&](int j, auto held) {
        constexpr int CH = decltype(held)::value;
        __syncthreads();  // previous transform done with lds
#pragma unroll
        for (int s = 0; s < 8; s++) lds[lines[s] * LDL + poss[s]] = vin[CH][s];
        __syncthreads();
        cx<T> *dst = out + j * NK + off;
        auto ld2 = [&](int line, int row) { return lds[line * LDL + row]; };
        auto st2 = [&](int line, int row, cx<T> v, int) { dst[(int64_t)row * stride + line] = v; };
        reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, +1, ld2, st2);
    };
    if constexpr (OP == ZOP_POISSON) {
        auto st = [&](int ln, int row, cx<T> v, int slot) {
            lines[slot] = ln;
            poss[slot] = row;
            vin[0][slot] = v;
        };
        forward(std::integral_constant<int, 0>{}, st);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int kx = ct * TX + lines[s], kz = poss[s];
            const bool zero_mode = (kx == 0 && ky == 0 && kz == 0);
            cx<double> r = mk(0.0, 0.0);
            if (kx <= H) {
                cx<double> sv = mk((double)vin[0][s].x, (double)vin[0][s].y);
                if (zero_mode && zp.k0set) sv = mk(zp.parts ? k0src : zp.k0re, zp.k0im);
                if (!(zero_mode && zp.modif == 0.0))
                    r = kop_poisson(sv, zp.gk2[kx] + gy + zp.gk2[kz], zp.coeff, zp.modif);
            }
            vin[0][s] = mk((T)r.x, (T)r.y);
        }
        inverse(0, std::integral_constant<int, 0>{});
    } else if constexpr (OP == ZOP_VECTOR) {
        // the projection applied per mode when the last component arrives, so
        // no operator loop holds eight modes' FP64 values (1.31 against
        // 1.34 ms at 512^3 for loading all operands first, spill 56 against 80)
        auto fwd = [&](auto held) {
            constexpr int CH = decltype(held)::value;
            auto st = [&](int ln, int row, cx<T> v, int slot) {
                lines[slot] = ln;
                poss[slot] = row;
                if constexpr (CH < 2) {
                    vin[CH][slot] = v;
                } else {
                    const int kx = ct * TX + ln;
                    cx<double> bo[3] = {mk(0.0, 0.0), mk(0.0, 0.0), mk(0.0, 0.0)};
                    if (kx <= H && !(kx == 0 && ky == 0 && row == 0)) {
                        const cx<double> sv[3] = {mk((double)vin[0][slot].x, (double)vin[0][slot].y),
                                                  mk((double)vin[1][slot].x, (double)vin[1][slot].y),
                                                  mk((double)v.x, (double)v.y)};
                        kop_vector(sv, zp.gk2[kx] + gy + zp.gk2[row], zp.ks[kx], kyv, zp.ks[row], zp.coeff, zp.modif,
                                   bo);
                    }
#pragma unroll
                    for (int j = 0; j < 3; j++) vin[j][slot] = mk((T)bo[j].x, (T)bo[j].y);
                }
            };
            forward(held, st);
        };
        fwd(std::integral_constant<int, 0>{});
        fwd(std::integral_constant<int, 1>{});
        fwd(std::integral_constant<int, 2>{});
        inverse(0, std::integral_constant<int, 0>{});
        inverse(1, std::integral_constant<int, 1>{});
        inverse(2, std::integral_constant<int, 2>{});
    } else if constexpr (OP == ZOP_ADJ_SCALAR) {
        // the one forward transform stays in registers; every component's
        // modes go through LDS to its inverse transform
        __shared__ double gkd[L];
        __shared__ cx<double> ksd[L];
        for (int m = threadIdx.x; m < L; m += NT) {
            gkd[m] = zp.gk2[m];
            ksd[m] = zp.ks[m];
        }
        auto st = [&](int ln, int row, cx<T> v, int slot) {
            lines[slot] = ln;
            poss[slot] = row;
            vin[0][slot] = v;
        };
        forward(std::integral_constant<int, 0>{}, st);
        auto component = [&](auto cc) {
            constexpr int C = decltype(cc)::value;
            __syncthreads();  // previous transform done with lds
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int kx = ct * TX + lines[s], kz = poss[s];
                cx<double> r = mk(0.0, 0.0);
                if (kx <= H && !(kx == 0 && ky == 0 && kz == 0)) {
                    const cx<double> w = conj(kop_scalar_weight(C, gkd[kx], gy, gkd[kz], ksd[kx], kyv, ksd[kz]));
                    r = (w * mk((double)vin[0][s].x, (double)vin[0][s].y)) * kop_scalar_norm(gkd[kx] + gy + gkd[kz], L);
                }
                lds[lines[s] * LDL + kz] = mk((T)r.x, (T)r.y);
            }
            __syncthreads();
            cx<T> *dst = out + C * NK + off;
            auto ld2 = [&](int line, int row) { return lds[line * LDL + row]; };
            auto st2 = [&](int line, int row, cx<T> v, int) { dst[(int64_t)row * stride + line] = v; };
            reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, +1, ld2, st2);
        };
        component(std::integral_constant<int, 0>{});
        component(std::integral_constant<int, 1>{});
        component(std::integral_constant<int, 2>{});
        component(std::integral_constant<int, 3>{});
        component(std::integral_constant<int, 4>{});
        component(std::integral_constant<int, 5>{});
    } else {
        // chi = sum_c w_c S_c from the three kz groups:
        //   sum_c w_c S_c = FFT_z(A) + g2 FFT_z(B) + k2 FFT_z(C)
        // so only the FP64 sums stay live between the transforms.  The k
        // tables are read per mode from LDS (FP64).
        __shared__ double gkd[L];
        __shared__ cx<double> ksd[L];
        for (int m = threadIdx.x; m < L; m += NT) {
            gkd[m] = zp.gk2[m];
            ksd[m] = zp.ks[m];
        }
        if constexpr (OP == ZOP_SCALAR) __syncthreads();  // read by the first loads
        cx<double> acc[8];
        auto group = [&](auto kind) {
            constexpr int K = decltype(kind)::value;
            auto st = [&](int ln, int row, cx<T> v, int slot) {
                lines[slot] = ln;
                poss[slot] = row;
                const cx<double> d = mk((double)v.x, (double)v.y);
                if constexpr (K == 0) {
                    acc[slot] = d;
                } else if constexpr (K == 1) {
                    acc[slot] = acc[slot] + d * gkd[row];
                } else {
                    // the last group completes the mode: the operator here,
                    // so each slot's FP64 sum dies at once (eight of them
                    // held through an operator loop doubled the registers)
                    const cx<double> sum = acc[slot] + ksd[row] * d;
                    const int kx = ct * TX + ln;
                    cx<double> r = mk(0.0, 0.0);
                    if (kx <= H && !(kx == 0 && ky == 0 && row == 0))
                        r = sum * kop_scalar_norm(gkd[kx] + gy + gkd[row], L);
                    vin[0][slot] = mk((T)r.x, (T)r.y);
                }
            };
            if constexpr (OP == ZOP_SCALAR3) {
                forward(kind, st);
            } else {
                // from the six components, each group formed in the loads of
                // its transform (the formulas of k_col_comb) and rounded once
                const cx<T> *src = in + off;
                auto ld = [&](int line, int row) {
                    const int kx = ct * TX + line;
                    const bool valid = kx <= H;  // padding columns give 0 above
                    const cx<T> *e = src + (int64_t)row * stride + line;
                    using W = scalar_weight_t<T, L>;
                    auto at = [&](int c) { return mk((W)e[c * NK].x, (W)e[c * NK].y); };
                    const W g0 = valid ? (W)gkd[kx] : (W)0, g1 = (W)gy;
                    const cx<W> k0 = valid ? mk((W)ksd[kx].x, (W)ksd[kx].y) : mk((W)0, (W)0);
                    const cx<W> k1 = mk((W)kyv.x, (W)kyv.y);
                    cx<W> r;
                    if constexpr (K == 0)
                        r = at(0) * (g1 - (W)2 * g0) + ((k0 * (W)-6) * k1) * at(1) + at(3) * (g0 - (W)2 * g1) +
                            at(5) * (g0 + g1);
                    else if constexpr (K == 1)
                        r = at(0) + at(3) - at(5) * (W)2;
                    else
                        r = (k0 * (W)-6) * at(2) + (k1 * (W)-6) * at(4);
                    return mk((T)r.x, (T)r.y);
                };
                if constexpr (K == 0) {
                    reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, -1, ld, st, twload);
                } else {
                    __syncthreads();  // previous transform done with lds
                    reg_fft<T, L, TX, true, 1, false, 1>(lds, twl, -1, ld, st);
                }
            }
        };
        group(std::integral_constant<int, 0>{});
        group(std::integral_constant<int, 1>{});
        group(std::integral_constant<int, 2>{});
        inverse(0, std::integral_constant<int, 0>{});
    }
}

// the vector and scalar operators keep 3 x 8 values per thread in registers:
// at most 512 threads per workgroup there; Poisson takes 512 too up to L = 512
// (three workgroups per CU instead of one, 4 % faster at L = 512)
// threads per workgroup of the scalar-projection and vector z solves: the
// scalar one (150+ registers, one 512-thread workgroup per CU) runs three
// 256-thread workgroups per CU (0.90 against 1.02 ms at 512^3, FP32); the
// vector one measured slower that way (1.75 against 1.34 ms)
template <typename T, int L, int OP> constexpr int zs_tx()
{
    constexpr bool narrow = OP != ZOP_POISSON || L <= 512;
    constexpr int tx = (narrow && col_tx<T, L>() * L / 8 > 512) ? 4096 / L : col_tx<T, L>();
    constexpr int cap = OP == ZOP_SCALAR3 ? 256 : (OP == ZOP_VECTOR ? 512 : 1 << 30);
    return (tx * L / 8 > cap && cap * 8 / L >= 1) ? cap * 8 / L : tx;
}

template <typename T, int N, int OP>
static void launch_zsolve(const cx<T> *in, cx<T> *out, int P, int64_t NK, const cx<T> *tw, const ZParams &zp,
                          hipStream_t s)
{
    constexpr int TX = zs_tx<T, N, OP>();
    const int64_t nb = (int64_t)(P / TX) * N;
    hipLaunchKernelGGL((k_zsolve<T, N, TX, OP>), dim3((unsigned)nb), dim3(TX * N / 8), 0, s, in, out, P, NK, tw, zp);
}

template <typename T> static const cx<T> *twiddles_of(gev_ctx *c)
{
    if constexpr (sizeof(T) == 8) return c->tw64;
    else return c->tw32;
}

template <typename T, int N>
static void zsolve_chain(gev_ctx *c, int op, const T *rin, int nin, cx<T> *ftin, cx<T> *ftout, T *rout, int nout,
                         const ZParams &zp)
{
    const cx<T> *tw = twiddles_of<T>(c);
    if (op == ZOP_SCALAR && !plane_size<T>(N)) {
        // x passes, then the y pass that forms the three groups of projectFTscalar
        if constexpr (!plane_size<T>(N)) {
            launch_r2c_multi<T, N, sij_spectra<T>()>(SrcPlainX<T, N>{rin, c->M}, ftin, c->P, c->NK, (int64_t)N * N, tw, c->stream);
            launch_col_comb<T, N>(ftin, c->P, c->NK, tw, zp, c->stream);
            launch_zsolve<T, N, ZOP_SCALAR3>(ftin, ftout, c->P, c->NK, tw, zp, c->stream);
        }
    } else {
        fwd_xy<T, N>(c, rin, ftin, nin, tw);
        if (op == ZOP_POISSON)
            launch_zsolve<T, N, ZOP_POISSON>(ftin, ftout, c->P, c->NK, tw, zp, c->stream);
        else if (op == ZOP_VECTOR)
            launch_zsolve<T, N, ZOP_VECTOR>(ftin, ftout, c->P, c->NK, tw, zp, c->stream);
        else if constexpr (plane_size<T>(N))
            launch_zsolve<T, N, ZOP_SCALAR>(ftin, ftout, c->P, c->NK, tw, zp, c->stream);
    }
    inv_yx<T, N>(c, ftout, rout, nout, tw);
}

template <typename T>
static int zsolve_dispatch(gev_ctx *c, int op, const T *rin, int nin, cx<T> *ftin, cx<T> *ftout, T *rout, int nout,
                           const ZParams &zp)
{
    switch (c->N) {
#define X(n) case n: zsolve_chain<T, n>(c, op, rin, nin, ftin, ftout, rout, nout, zp); break;
        GEV_FOR_FUSED_N(X)
#undef X
    default: gev_set_error("fused z-pass solve needs 16 <= N <= 1024"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

bool zsolve_supported(const gev_ctx *c) { return c->N >= 16 && c->N <= 1024; }

// pot = c2r(poisson(r2c(src))) with the k=0 mode optionally replaced first
template <typename T>
int solve_poisson_fused_impl(gev_ctx *c, const T *src, T *pot, cx<T> *work, double coeff, double modif, int k0set,
                             double k0re)
{
    ZParams zp{c->gk2, c->kshift, coeff / -((double)c->N * (double)c->N * (double)c->N), modif, k0re, 0.0, k0set,
               nullptr, 0, nullptr};
    return zsolve_dispatch<T>(c, ZOP_POISSON, src, 1, work, work, pot, 1, zp);
}

// A source written back over its input as it is formed (meshes below 128,
// where gev_solve_poisson_T00 and gev_solve_chi_Tij leave the source terms in
// place): each pair is read and written by the one thread that forms it.
template <typename T, int N, class S> struct SrcPut : S {
    T *dst;
    __device__ __forceinline__ SrcPut(const S &s, T *d) : S(s), dst(d) {}
    __device__ __forceinline__ cx<T> operator()(int64_t L, int n)
    {
        const cx<T> v = S::operator()(L, n);
        reinterpret_cast<cx<T> *>(dst)[L * (N / 2) + n] = v;
        return v;
    }
};

template <typename T, int N> struct CompT00 {
    SrcT00<T, N> s;
    T *put;  // the source, written back
    template <class F> __device__ __forceinline__ void with(int, F f) const
    {
        static_assert(N < 128, "the T00 source is formed in planes up to 64^3 only");
        f(SrcPut<T, N, SrcT00<T, N>>(s, put));
    }
};

// pot = c2r(poisson(r2c(prepareFTsource_T00(phi, chi, src)))) with the source
// formed inside the x pass; its workgroup sums go to ctx->red + 64 and are
// reduced inside the z pass to ctx->red[0] (source) and ctx->red[1] (result),
// which is the k=0 mode when zp.k0set
template <typename T, int N>
static void poisson_T00_chain(gev_ctx *c, const SrcT00<T, N> &src, T *put, T *pot, cx<T> *work, ZParams zp)
{
    const cx<T> *tw = twiddles_of<T>(c);
    zp.parts = c->red + 64;
    zp.sums = c->red;
    // at N = 128 one component is 128 planes: half the CUs, each with the nine
    // phi rows of its source to fetch (25.9 us, FP32), against 14.9 + 6.9 us for
    // the two passes
    if constexpr (N <= 64) {
        zp.nparts = N / plane_np<N>();
        launch_fwd_plane<T, N>(c, CompT00<T, N>{src, put}, work, 1, tw, c->red + 64);
    } else {
        constexpr int NL = xlines<T, N>();
        const int64_t nl = (int64_t)N * N;
        zp.nparts = (int)((nl + NL - 1) / NL);
        launch_r2c_src<T, N>(src, work, c->P, nl, tw, c->stream, c->red + 64);
        launch_col<T, N>(work, c->P, 1, -1, tw, c->stream);
    }
    launch_zsolve<T, N, ZOP_POISSON>(work, work, c->P, c->NK, tw, zp, c->stream);
    inv_yx<T, N>(c, work, pot, 1, tw);
}

template <typename T>
int solve_poisson_T00_fused_impl(gev_ctx *c, const T *phi, const T *chi, T *src, double bg, double c1, double c2,
                                 double c3, T *pot, cx<T> *work, double coeff, double modif, int k0set)
{
    ZParams zp{c->gk2, c->kshift, coeff / -((double)c->N * (double)c->N * (double)c->N), modif, 0.0, 0.0, k0set,
               nullptr, 0, nullptr};
    switch (c->N) {
#define X(n)                                                                                                     \
    case n:                                                                                                      \
        poisson_T00_chain<T, n>(c, SrcT00<T, n>{phi, chi, src, (T)bg, (T)c1, (T)c2, (T)c3, {0.0, 0.0}}, src, pot, \
                                work, zp);                                                                       \
        break;
        GEV_FOR_FUSED_N(X)
#undef X
    default: gev_set_error("prepareFTsource T00 inside the Poisson solve needs 16 <= N <= 1024"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

// chi = c2r(projectFTscalar(r2c(Sij)))
template <typename T> int solve_chi_fused_impl(gev_ctx *c, const T *Sij, T *chi, cx<T> *SijFT, cx<T> *chiFT)
{
    ZParams zp{c->gk2, c->kshift, 0.0, 0.0, 0.0, 0.0, 0, nullptr, 0, nullptr};
    return zsolve_dispatch<T>(c, ZOP_SCALAR, Sij, 6, SijFT, chiFT, chi, 1, zp);
}

template <typename T, int N> struct CompSij {
    const T *phi;
    T *Tij;
    int64_t M;
    T coeff;
    template <class F> __device__ __forceinline__ void with(int c, F f) const
    {
        auto one = [&](auto cc) {
            constexpr int C = decltype(cc)::value;
            const SrcSij<T, N, C> s{phi, Tij + C * M, coeff};
            if constexpr (N < 128) f(SrcPut<T, N, SrcSij<T, N, C>>(s, Tij + C * M));
            else f(s);
        };
        switch (c) {
        case 0: one(std::integral_constant<int, 0>{}); break;
        case 1: one(std::integral_constant<int, 1>{}); break;
        case 2: one(std::integral_constant<int, 2>{}); break;
        case 3: one(std::integral_constant<int, 3>{}); break;
        case 4: one(std::integral_constant<int, 4>{}); break;
        default: one(std::integral_constant<int, 5>{}); break;
        }
    }
};

// chi from Tij: the x passes compute Sij = prepareFTsource(phi, Tij, coeff)
// on the fly (and write it over Tij below N = 128)
template <typename T, int N>
static void chi_from_Tij_chain(gev_ctx *c, const T *phi, T *Tij, T coeff, cx<T> *SijFT, cx<T> *chiFT, T *chi)
{
    const int64_t nl = (int64_t)N * N;
    const cx<T> *tw = twiddles_of<T>(c);
    ZParams zp{c->gk2, c->kshift, 0.0, 0.0, 0.0, 0.0, 0, nullptr, 0, nullptr};
    if constexpr (plane_size<T>(N)) {
        launch_fwd_plane<T, N>(c, CompSij<T, N>{phi, Tij, c->M, coeff}, SijFT, 6, tw);
        launch_zsolve<T, N, ZOP_SCALAR>(SijFT, chiFT, c->P, c->NK, tw, zp, c->stream);
    } else {
        launch_r2c_multi<T, N, sij_spectra<T>()>(SrcSijX<T, N>{phi, Tij, c->M, coeff}, SijFT, c->P, c->NK, nl, tw, c->stream);
        launch_col_comb<T, N>(SijFT, c->P, c->NK, tw, zp, c->stream);
        launch_zsolve<T, N, ZOP_SCALAR3>(SijFT, chiFT, c->P, c->NK, tw, zp, c->stream);
    }
    inv_yx<T, N>(c, chiFT, chi, 1, tw);
}

bool fused_sources_supported(const gev_ctx *c) { return c->N >= 16 && c->N <= 1024; }

template <typename T>
int solve_chi_Tij_fused_impl(gev_ctx *c, const T *phi, T *Tij, double coeff, T *chi, cx<T> *SijFT, cx<T> *chiFT)
{
    switch (c->N) {
#define X(n) case n: chi_from_Tij_chain<T, n>(c, phi, Tij, (T)coeff, SijFT, chiFT, chi); break;
        GEV_FOR_FUSED_N(X)
#undef X
    default: gev_set_error("chi from Tij needs 16 <= N <= 1024"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

// lS[c] = c2r(conj(w_c) r2c(lchi) / (2 k^4 N)): the adjoint of solve_chi.  The
// weights are applied between the forward and the six inverse z transforms,
// so no Fourier component passes through memory in between (the operator's
// own kernel and six z passes before: at 128^3 FP32 13.7 + 44 us of the adjoint
// chi solve)
template <typename T, int N>
static void adj_chi_chain(gev_ctx *c, const T *lchi, T *lS, cx<T> *work1, cx<T> *work6)
{
    const cx<T> *tw = twiddles_of<T>(c);
    ZParams zp{c->gk2, c->kshift, 0.0, 0.0, 0.0, 0.0, 0, nullptr, 0, nullptr};
    fwd_xy<T, N>(c, lchi, work1, 1, tw);
    launch_zsolve<T, N, ZOP_ADJ_SCALAR>(work1, work6, c->P, c->NK, tw, zp, c->stream);
    inv_yx<T, N>(c, work6, lS, 6, tw);
}

template <typename T>
int adj_solve_chi_fused_impl(gev_ctx *c, const T *lchi, T *lS, cx<T> *work1, cx<T> *work6)
{
    switch (c->N) {
#define X(n) case n: adj_chi_chain<T, n>(c, lchi, lS, work1, work6); break;
        GEV_FOR_FUSED_N(X)
#undef X
    default: gev_set_error("the fused adjoint chi solve needs 16 <= N <= 1024"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

// Bi = c2r(projectFTvector(r2c(Bi))), in place on Bi
template <typename T> int solve_vector_fused_impl(gev_ctx *c, T *Bi, cx<T> *BiFT, double coeff, double modif)
{
    ZParams zp{c->gk2, c->kshift, coeff, modif, 0.0, 0.0, 0, nullptr, 0, nullptr};
    return zsolve_dispatch<T>(c, ZOP_VECTOR, Bi, 3, BiFT, BiFT, Bi, 3, zp);
}

template <typename T, int N> struct CompLink {
    const T *phi, *L;
    int64_t M;
    template <class F> __device__ __forceinline__ void with(int c, F f) const
    {
        if (c == 0) f(SrcT0iLink<T, N, 0>{phi, L});
        else if (c == 1) f(SrcT0iLink<T, N, 1>{phi, L + M});
        else f(SrcT0iLink<T, N, 2>{phi, L + 2 * M});
    }
};

// the same from T0i link sums: the x passes apply the link factor with phi
template <typename T, int N>
static void vector_from_links_chain(gev_ctx *c, T *Bi, const T *phi, cx<T> *BiFT, const ZParams &zp)
{
    const cx<T> *tw = twiddles_of<T>(c);
    if constexpr (plane_size<T>(N)) {
        launch_fwd_plane<T, N>(c, CompLink<T, N>{phi, Bi, c->M}, BiFT, 3, tw);
    } else {
        const int64_t nl = (int64_t)N * N, M = c->M;
        auto xy = [&](const auto &src, int i) {
            launch_r2c_src<T, N>(src, BiFT + i * c->NK, c->P, nl, tw, c->stream);
            launch_col<T, N>(BiFT + i * c->NK, c->P, 1, -1, tw, c->stream);
        };
        xy(SrcT0iLink<T, N, 0>{phi, Bi}, 0);
        xy(SrcT0iLink<T, N, 1>{phi, Bi + M}, 1);
        xy(SrcT0iLink<T, N, 2>{phi, Bi + 2 * M}, 2);
    }
    launch_zsolve<T, N, ZOP_VECTOR>(BiFT, BiFT, c->P, c->NK, tw, zp, c->stream);
    inv_yx<T, N>(c, BiFT, Bi, 3, tw);
}

// the link factor alone, in place (meshes below the fused chain's range)
template <typename T> __global__ void k_t0i_link_factor(T *Bi, const T *__restrict__ phi, int N, int64_t M)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    const int lg = __builtin_ctz(N), M1 = N - 1;
    const int x = (int)(i & M1), y = (int)((i >> lg) & M1), z = (int)(i >> (2 * lg));
    const T p = phi[i];
    Bi[i] *= (T)1 + p + phi[site(N, x + 1, y, z)];
    Bi[M + i] *= (T)1 + p + phi[site(N, x, y + 1, z)];
    Bi[2 * M + i] *= (T)1 + p + phi[site(N, x, y, z + 1)];
}

template <typename T> int t0i_link_factor_impl(gev_ctx *c, T *Bi, const T *phi)
{
    hipLaunchKernelGGL((k_t0i_link_factor<T>), dim3((unsigned)((c->M + 255) / 256)), dim3(256), 0, c->stream, Bi, phi,
                       c->N, c->M);
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

template <typename T>
int solve_vector_links_fused_impl(gev_ctx *c, T *Bi, const T *phi, cx<T> *BiFT, double coeff, double modif)
{
    ZParams zp{c->gk2, c->kshift, coeff, modif, 0.0, 0.0, 0, nullptr, 0, nullptr};
    switch (c->N) {
#define X(n) case n: vector_from_links_chain<T, n>(c, Bi, phi, BiFT, zp); break;
        GEV_FOR_FUSED_N(X)
#undef X
    default: gev_set_error("B from T0i links needs 16 <= N <= 1024"); return GEV_ERR_ARG;
    }
    GEV_HIP(hipGetLastError());
    return GEV_OK;
}

#define INSTZ(T)                                                                                       \
    template int solve_chi_Tij_fused_impl<T>(gev_ctx *, const T *, T *, double, T *, cx<T> *, cx<T> *);  \
    template int solve_poisson_fused_impl<T>(gev_ctx *, const T *, T *, cx<T> *, double, double, int, double); \
    template int solve_chi_fused_impl<T>(gev_ctx *, const T *, T *, cx<T> *, cx<T> *);                  \
    template int adj_solve_chi_fused_impl<T>(gev_ctx *, const T *, T *, cx<T> *, cx<T> *);               \
    template int solve_vector_fused_impl<T>(gev_ctx *, T *, cx<T> *, double, double);                    \
    template int solve_vector_links_fused_impl<T>(gev_ctx *, T *, const T *, cx<T> *, double, double);    \
    template int t0i_link_factor_impl<T>(gev_ctx *, T *, const T *);                                      \
    template int solve_poisson_T00_fused_impl<T>(gev_ctx *, const T *, const T *, T *, double, double, double, \
                                                 double, T *, cx<T> *, double, double, int);
INSTZ(double)
INSTZ(float)
#undef INSTZ

template int fft_r2c_impl<double>(gev_ctx *, const double *, cx<double> *, int, const cx<double> *);
template int fft_r2c_impl<float>(gev_ctx *, const float *, cx<float> *, int, const cx<float> *);
template int fft_c2r_impl<double>(gev_ctx *, cx<double> *, double *, int, const cx<double> *);
template int fft_c2r_impl<float>(gev_ctx *, cx<float> *, float *, int, const cx<float> *);

}  // namespace gev
