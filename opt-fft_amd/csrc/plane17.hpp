// 17^3 with a workgroup per output x-plane, for batches too small to fill the device with a
// volume per workgroup: there one CU runs three passes of 17-point lines one after the other,
// which is latency.
// Workgroup (v, k), 289 of its 320 threads a (y, z) point each:
//   x:  X_k = x_0 + sum_j (u_j cos + S i v_j sin), u_j = x_j + x_{17-j}, v_j = x_j - x_{17-j},
//       j = 1..8, straight from HBM (every workgroup of a volume reads all of it, from the L2
//       of the XCD they share after the first), to LDS plane 0;
//   z, y: thread (pair p, line l) takes outputs p and 17 - p of line l (p = 0: output 0), with
//       the same cosines and sines in both passes, so a line is spread over nine threads;
//       plane 0 -> plane 1 -> HBM, runs of 17 elements.
// A workgroup an output plane reads the volume 17 times (from L2) and spends about four times the
// arithmetic of whole lines, so the volume kernel takes over when its workgroups begin to fill
// the device (us a launch back to back, this kernel / the quickest volume kernel, over 64 MB of
// buffers in turn; 3.3 is the host's issue).  Times step where another round of workgroups
// begins, past 8, 24 and 32 volumes in complex128:
//   x 1 3.9 / 6.8   x 8 4.1 / 7.1   x 24 5.5 / 8.0   x 32 7.4 / 8.2   x 36 8.1 / 8.2   x 48 9.6 / 8.3
//   over 1 GB: x 1 4.5 / 7.2   x 24 6.8 / 8.5   x 32 8.4 / 8.7   x 36 9.4 / 8.8   x 48 11.3 / 8.9
//   complex64: x 1 3.8 / 5.7   x 24 4.5 / 6.4   x 40 5.4 / 6.5   x 48 6.2 / 6.5   x 64 7.0 / 6.6
//   over 1 GB: x 1 3.8 / 5.8   x 24 5.1 / 6.7   x 40 6.3 / 6.9   x 48 7.1 / 7.0   x 64 8.2 / 7.2
// and waited for one by one: complex128 x 24 16.5 / 18.0, x 32 18.3 / 18.1; complex64 x 40 16.3 /
// 16.8, x 48 17.5 / 17.2;
// hence TINY, 32 and 48 volumes on 256 CUs.
#pragma once
#include "codelets.hpp"
#include "registry.hpp"

namespace fx {

template <typename T_, int S_>
struct Plane17Cfg {
    using T = T_;
    static constexpr int S = S_, NT = 320, L = 17, PLANE = 289, V = 4913;
    static constexpr int LDS = 2 * PLANE;   // elements
    static constexpr int kXcds = 8;
    static constexpr int TINY = sizeof(T) == 8 ? 32 : 48;   // KernelDesc::tiny
};

template <class C>
struct Plane17 {
    using T = typename C::T;
    // Cosines and sines of the thread's pair: index j - 1.
    struct Regs {
        T c[8], s[8];
    };

    // Workgroup g -> (volume, output plane): a volume's workgroups follow one another on one XCD.
    static FX_HD void task(long g, long& v, int& k)
    {
        const long x = g % C::kXcds, i = g / C::kXcds;
        v = i / C::L * C::kXcds + x;
        k = (int)(i % C::L);
    }
    static FX_HD long grid(long nvol) { return (nvol + C::kXcds - 1) / C::kXcds * C::kXcds * C::L; }

    static FX_HD int pair_of(int tid) { return tid / C::L; }
    static FX_HD int line_of(int tid) { return tid % C::L; }
    static FX_HD bool has_pair(int tid) { return tid < 9 * C::L; }

    static FX_HD void xpass(int tid, long v, int k, const cx<T>* __restrict__ in, cx<T>* sm, Regs& R,
                            const Bank<T>* __restrict__ bk)
    {
        const int q = tid < C::PLANE ? tid : C::PLANE - 1;
        const cx<T>* __restrict__ src = in + v * (long)C::V + q;
        cx<T> x[C::L];
#pragma unroll
        for (int j = 0; j < C::L; ++j) x[j] = src[j * C::PLANE];
        const int p = has_pair(tid) ? pair_of(tid) : 0;
#pragma unroll
        for (int j = 1; j <= 8; ++j) {
            const int m = (j * p) % C::L;
            R.c[j - 1] = bk->cos17[m];
            R.s[j - 1] = bk->sin17[m];
        }
        cx<T> A = x[0], B = {T(0), T(0)};
#pragma unroll
        for (int j = 1; j <= 8; ++j) {
            const int m = (j * k) % C::L;
            const T c = bk->cos17[m], s = bk->sin17[m];
            const cx<T> u = x[j] + x[C::L - j], w = x[j] - x[C::L - j];
            A.r += c * u.r;
            A.i += c * u.i;
            B.r += s * w.r;
            B.i += s * w.i;
        }
        if (tid < C::PLANE) sm[tid] = A + mul_si<C::S>(B);
    }
    // Outputs p and 17 - p of the line whose point j is at t[j * st].
    static FX_HD void pair_dft(const cx<T>* t, int st, const Regs& R, cx<T>& lo, cx<T>& hi)
    {
        cx<T> x[C::L];
#pragma unroll
        for (int j = 0; j < C::L; ++j) x[j] = t[j * st];
        cx<T> A = x[0], B = {T(0), T(0)};
#pragma unroll
        for (int j = 1; j <= 8; ++j) {
            const cx<T> u = x[j] + x[C::L - j], w = x[j] - x[C::L - j];
            A.r += R.c[j - 1] * u.r;
            A.i += R.c[j - 1] * u.i;
            B.r += R.s[j - 1] * w.r;
            B.i += R.s[j - 1] * w.i;
        }
        const cx<T> b = mul_si<C::S>(B);
        lo = A + b;
        hi = A - b;
    }
    static FX_HD void zpass(int tid, cx<T>* sm, const Regs& R)
    {
        if (!has_pair(tid)) return;
        const int p = pair_of(tid), l = line_of(tid);
        cx<T> lo, hi;
        pair_dft(sm + l * C::L, 1, R, lo, hi);
        cx<T>* d = sm + C::PLANE + l * C::L;
        d[p] = lo;
        if (p > 0) d[C::L - p] = hi;
    }
    static FX_HD void ypass(int tid, long v, int k, const cx<T>* sm, cx<T>* __restrict__ out,
                            const Regs& R, T scl)
    {
        if (!has_pair(tid)) return;
        const int p = pair_of(tid), l = line_of(tid);
        cx<T> lo, hi;
        pair_dft(sm + C::PLANE + l, C::L, R, lo, hi);
        // Always scaled: a product by 1 is exact.
        cx<T>* __restrict__ d = out + v * (long)C::V + (long)k * C::PLANE + l;
        st_hint<0>(d + p * C::L, scale(lo, scl));
        if (p > 0) st_hint<0>(d + (C::L - p) * C::L, scale(hi, scl));
    }
};

template <class C>
__global__ void __launch_bounds__(C::NT)
    k_plane17(const cx<typename C::T>* __restrict__ in, cx<typename C::T>* __restrict__ out, long nvol,
              const Bank<typename C::T>* __restrict__ bk, typename C::T scl)
{
    using K = Plane17<C>;
    __shared__ cx<typename C::T> sm[C::LDS];
    long v;
    int k;
    K::task(blockIdx.x, v, k);
    if (v >= nvol) return;   // uniform over the workgroup, before any barrier
    const int tid = threadIdx.x;
    typename K::Regs R;
    K::xpass(tid, v, k, in, sm, R, bk);
    __syncthreads();
    K::zpass(tid, sm, R);
    __syncthreads();
    K::ypass(tid, v, k, sm, out, R, scl);
}

}  // namespace fx

#include <fx_plane17_launch.hpp>
