// gev_fft_plane.hpp -- x and y transforms of a whole z plane in one workgroup
// (16 <= N <= 128 in FP32, up to 64 in FP64).
//
// The half spectrum of such a plane fits the LDS with room for a second
// workgroup (N (N/2 + 1) complex values: 66 KB at N = 128 in FP32),
// so the plane is read once, transformed along x and along y in LDS and
// written once; all components of a field go in one launch.  At these sizes
// the transforms are bound by launches and by the latency of each pass, not by
// memory.  Per component, separate x and y passes took 7.7 + 7.4 us at 128^3
// (FP32), 7.9 + 3.6 us at 64^3 (FP32) and 7.4 + 3.1 us at 32^3 (FP64), twelve
// launches for a symmetric tensor; the plane kernels take 10.1, 6.5 and 4-6 us
// forward and 10.1, 4.6 and 4.4 us back, one launch for all components (the
// phi, chi and B solves of a 64^3 FP32 cycle 213 -> 76 us of kernel time, a
// 32^3 FP64 GR cycle 2.0x).  Above 128 a plane does not fit.
//
// The x transform of real lines is the packed complex one of length H = N/2;
// its post-twiddle happens in the loads of the y transform.  X[0] and X[H] of
// a real line are real, so the two columns travel as one complex column
// X[0] + i X[H] through the y transform and H columns suffice (N H / 8
// threads, radix-8 stages in registers).
#pragma once
#include "gev_fft_engine.hpp"

namespace gev {

template <int N> constexpr int plane_np() { return N >= 32 ? 1 : 4; }                 // planes per workgroup
template <int N> constexpr int plane_nt() { return plane_np<N>() * N * N / 16; }       // threads per workgroup
// kx pitch, as gev_ctx_create sets it
template <typename T, int N> constexpr int plane_pitch()
{
    return (N / 2 + 1 + 64 / (int)sizeof(T) - 1) / (64 / (int)sizeof(T)) * (64 / (int)sizeof(T));
}

// [plane][y][kx] with row pitch H + 1; line = plane * H + column
template <int N> struct ColAddr {
    static constexpr int H = N / 2, PT = H + 1;
    __device__ __forceinline__ int operator()(int line, int pos) const
    {
        return (line / H) * (N * PT) + pos * PT + line % H;
    }
};

template <typename T, int N, class Src>
__device__ __forceinline__ void fwd_plane(Src &src, cx<T> *out, const cx<T> *__restrict__ tw, cx<T> *lds, cx<T> *twl,
                                          cx<T> *c0)
{
    constexpr int H = N / 2, PT = H + 1, NP = plane_np<N>(), NT = plane_nt<N>(), P = plane_pitch<T, N>();
    const int t = threadIdx.x;
    const int z0 = blockIdx.x * NP;
    out += (int64_t)P * N * z0;
    {
        const TwiddleLoad<T, N, NT> twload(twl, tw);
        auto ld = [&](int line, int n) { return src((int64_t)z0 * N + line, n); };
        auto st = [&](int line, int k, cx<T> v, int) { lds[line * PT + k] = v; };
        reg_fft_at<T, H, NP * N, false, 2, true, 1>(lds, twl, -1, LineAddr<PT>{}, ld, st, twload);
    }
    __syncthreads();
    // column c of row y after the x transform: the post-twiddle of the packed
    // transform, column 0 holding X[0] + i X[H] (both real)
    auto ld = [&](int line, int y) {
        const int c = line % H;
        const cx<T> *row = lds + (line / H) * (N * PT) + y * PT;
        const cx<T> Zk = row[c], Zm = conj(row[c ? H - c : 0]);
        const cx<T> Fe = (Zk + Zm) * (T)0.5, Fo = mul_i(Zk - Zm, -1) * (T)0.5;
        const cx<T> X = Fe + twl[c] * Fo;  // no branch: its waits would serialise the eight reads
        return mk(c ? X.x : Zk.x + Zk.y, c ? X.y : Zk.x - Zk.y);
    };
    auto st = [&](int line, int ky, cx<T> v, int) {
        const int c = line % H, pl = line / H;
        if (c == 0) c0[pl * N + ky] = v;
        else out[c + P * (pl * N + ky)] = v;
    };
    reg_fft_at<T, N, NP * H, true, 1, false, 1>(lds, twl, -1, ColAddr<N>{}, ld, st, NoHook{});
    __syncthreads();
    // columns 0 and H from the packed one, and the zero padding columns
    constexpr int W = P - H + 1;
    for (int e = t; e < NP * N * W; e += NT) {
        const int row = e / W, j = e - row * W, pl = row / N, ky = row % N;
        const cx<T> a = c0[row], b = conj(c0[pl * N + ((N - ky) & (N - 1))]);
        cx<T> *dst = out + P * row;
        if (j == W - 1) dst[0] = (a + b) * (T)0.5;
        else dst[H + j] = j == 0 ? mul_i(a - b, -1) * (T)0.5 : mk((T)0, (T)0);
    }
}

template <typename T, int N>
__device__ __forceinline__ void inv_plane(const cx<T> *in, T *out, const cx<T> *__restrict__ tw, cx<T> *lds,
                                          cx<T> *twl, cx<T> *ca, cx<T> *cb)
{
    constexpr int H = N / 2, PT = H + 1, NP = plane_np<N>(), NT = plane_nt<N>(), P = plane_pitch<T, N>();
    const int t = threadIdx.x;
    const int z0 = blockIdx.x * NP;
    in += (int64_t)P * N * z0;
    const TwiddleLoad<T, N, NT> twload(twl, tw);
    for (int e = t; e < NP * N; e += NT) {
        ca[e] = in[P * e];
        cb[e] = in[P * e + H];
    }
    {
        // columns 0 and H enter as one: after the y transform only the real
        // parts of both are kept, and Re(IFFT(X)) is the IFFT of X's Hermitian
        // part, so the packed column is herm(X[0]) + i herm(X[H]) (from LDS,
        // selected without a branch, so that the eight loads stay in flight
        // together: 14.4 -> 10.1 us at 128^3 in FP32)
        auto ld = [&](int line, int ky) {
            const int c = line % H, p0 = (line / H) * N, k = p0 + ky, km = p0 + ((N - ky) & (N - 1));
            const cx<T> v = in[c + P * k];
            const cx<T> ha = (ca[k] + conj(ca[km])) * (T)0.5, hb = (cb[k] + conj(cb[km])) * (T)0.5;
            return mk(c ? v.x : ha.x - hb.y, c ? v.y : ha.y + hb.x);
        };
        auto st = [&](int line, int y, cx<T> v, int) { lds[ColAddr<N>{}(line, y)] = v; };
        __syncthreads();  // ca, cb
        reg_fft_at<T, N, NP * H, true, 1, true, 1>(lds, twl, +1, ColAddr<N>{}, ld, st, twload);
    }
    __syncthreads();
    auto ld = [&](int line, int k) {
        const cx<T> *row = lds + line * PT;
        const cx<T> Xk = row[k], cm = conj(row[k ? H - k : 0]);
        const cx<T> Z = (Xk + cm) + mul_i((Xk - cm) * conj(twl[k]), +1);
        return mk(k ? Z.x : Xk.x + Xk.y, k ? Z.y : Xk.x - Xk.y);
    };
    cx<T> *dst = reinterpret_cast<cx<T> *>(out) + (int64_t)z0 * N * H;
    auto st = [&](int line, int n, cx<T> v, int) { dst[line * H + n] = v; };
    reg_fft_at<T, H, NP * N, false, 2, false, 1>(lds, twl, +1, LineAddr<PT>{}, ld, st, NoHook{});
}

// grid (planes / NP, components); Comp::with(c, f) calls f with component c's
// source of the pair of reals (2n, 2n + 1) of line y + N z.  A source that sums
// (Src::kSums) leaves its workgroup's two sums in partials[2 b], [2 b + 1].
template <typename T, int N, class Comp>
__global__ __launch_bounds__(plane_nt<N>()) void k_fwd_plane(Comp comp, cx<T> *out, int64_t NK,
                                                             const cx<T> *__restrict__ tw, double *partials)
{
    constexpr int PT = N / 2 + 1, NP = plane_np<N>(), NT = plane_nt<N>();
    __shared__ cx<T> lds[NP * N * PT];
    __shared__ cx<T> twl[N];
    __shared__ cx<T> c0[NP * N];
    comp.with((int)blockIdx.y, [&](auto src) {
        fwd_plane<T, N>(src, out + blockIdx.y * NK, tw, lds, twl, c0);
        if constexpr (decltype(src)::kSums) {
            __shared__ double ws[NT / 64][2];
            const double v0 = wave_sum(src.acc[0]), v1 = wave_sum(src.acc[1]);
            if ((threadIdx.x & 63) == 0) { ws[threadIdx.x >> 6][0] = v0; ws[threadIdx.x >> 6][1] = v1; }
            __syncthreads();
            if (threadIdx.x == 0) {
                double t0 = 0.0, t1 = 0.0;
                for (int w = 0; w < NT / 64; w++) { t0 += ws[w][0]; t1 += ws[w][1]; }
                partials[2 * blockIdx.x] = t0;
                partials[2 * blockIdx.x + 1] = t1;
            }
        }
    });
}

template <typename T, int N>
__global__ __launch_bounds__(plane_nt<N>()) void k_inv_plane(const cx<T> *__restrict__ in, T *__restrict__ out,
                                                             int64_t NK, int64_t M, const cx<T> *__restrict__ tw)
{
    constexpr int PT = N / 2 + 1, NP = plane_np<N>();
    __shared__ cx<T> lds[NP * N * PT];
    __shared__ cx<T> twl[N];
    __shared__ cx<T> ca[NP * N], cb[NP * N];
    inv_plane<T, N>(in + blockIdx.y * NK, out + blockIdx.y * M, tw, lds, twl, ca, cb);
}

}  // namespace gev
