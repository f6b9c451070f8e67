// Single-pass kernel for volumes larger than a CU holds (36^3 complex128, 746 KB; 24x24x48
// complex128, 442 KB; also 24^3 complex128 and the complex64 36^3 and 24x24x48): the x DFT
// split by output residue.  With N0 = R * M, output x-plane R q + h of
// X[k] = sum_j x[j] W^(j k) is
//
//   X[R q + h] = sum_{n < M} W_M^(n q) * ( W_N0^(n h) * sum_{m < R} x[n + M m] W_R^(m h) ),
//
// so a workgroup (v, h) reads all N0 x-planes of volume v, forms the M sums of residue h in
// registers (a thread per (y, z) point, every load instruction of a wave 64 consecutive
// elements), and an M-point DFT over n gives the x transform of its M output planes.  Those
// M planes (N1 x N2, rows padded by PZ) are held in LDS, z lines and then y lines are
// transformed there, and the y pass writes planes R q + h to HBM.  Every element is written
// once; it is read R times, by the R workgroups of its volume, which are consecutive
// workgroups of one XCD (an 8-XCD part dispatches workgroup g to XCD g mod 8), so they run
// together and most reads of a line after the first are served by that XCD's L2.  The
// inputs are therefore read with plain loads, the outputs stored nontemporal (HS = 1).
//
// The x pass is one stream of groups of M loads (M planes at one point) with PF groups in
// flight across the points of a thread, its order pinned by sched_fence: left to itself the
// compiler waits for all loads of a point before it issues the next ones (14, 13 and 9 at a
// time at 36^3), and recomputes 64-bit addresses for each.  Against that form 24^3 x 365
// takes 36.7 us instead of 39.9 (r3), 24x24x48 complex64 x 300 36.7 instead of 40.6 (r3),
// 36^3 x 64 33.4 instead of 35.0 (r6).  At 36^3 x 128 it gains nothing (56.3 against 56.9):
// the rate at which a CU reads from L2 bounds that x pass, whatever is in flight (PF = 2 .. 6
// 56.3-57.3 us).  A probe that only reads (R = 6, every workgroup all of its volume) gets
// 62-75 GB/s a CU there, 108 from an L2 that already holds the volumes.
#pragma once

#include "kernels.hpp"

namespace fx {

// OR: order of the x pass's points.  0: every workgroup of a volume walks the plane from
// point 0, so the R of them request the same lines together; 1: residue h starts at its
// thread block h mod PPT (the blocks of NT points taken in rotated order); 2: residue h
// starts at point h * PLANE / R (the plane walked with a wrap).  1 and 2 spread the R
// workgroups' requests over different lines (and L2 channels) at the price of keeping each
// line in L2 longer.  PF: groups of M loads in flight (24-32 loads; 12 where a 48-point line
// sets the VGPRs: PF = 4 took 17.1 us at 24x24x48 x 64, PF = 2 16.7).
template <int N0_, int N1_, int N2_, typename T_, int S_, int R_, int NT_, int OR_ = 0,
          int PF_ = 4, int PZ_ = 1, int HS_ = 1, int ALG_ = 0>
struct XResCfg {
    using T = T_;
    static constexpr int N0 = N0_, N1 = N1_, N2 = N2_, S = S_, R = R_, NT = NT_, PZ = PZ_;
    static constexpr int OR = OR_, PF = PF_;
    static constexpr int PPT = (N1 * N2 + NT - 1) / NT;   // (y, z) points per thread
    static constexpr int HS = HS_, ALG = ALG_, V17 = ALG_, VPW = 1, P = 0;
    static_assert(N0 % R == 0, "the residues split the x-planes evenly");
    static constexpr int M = N0 / R;       // x-planes per workgroup
    static constexpr int V = N0 * N1 * N2;
    static constexpr int PLANE = N1 * N2;
    static constexpr int YS = N2 + PZ;     // LDS pitch between z rows
    static constexpr int SS = N1 * YS;     // LDS pitch between x-planes
    static constexpr int LDS = M * SS;     // elements
    static constexpr int WPE = waves_per_eu(LDS * (int)sizeof(cx<T>), NT, 0);
    static constexpr int kXcds = 8;
};

template <class C>
struct XRes {
    using T = typename C::T;

    // Workgroup g -> (volume v, residue h): g = kXcds * i + x, volume kXcds * (i / R) + x,
    // residue i mod R.
    static FX_HD void task(long g, long& v, int& h)
    {
        const long x = g % C::kXcds, i = g / C::kXcds;
        const long vq = i / C::R;
        h = (int)(i - vq * C::R);
        v = vq * C::kXcds + x;
    }
    static FX_HD long grid(long nvol) { return (nvol + C::kXcds - 1) / C::kXcds * C::kXcds * C::R; }

    // W_N0^e with the transform's sign.
    static FX_HD cx<T> w0(int e, const Bank<T>* __restrict__ bk)
    {
        cx<T> w = bk->w[woff(C::N0) + e];
        if constexpr (C::S > 0) w.i = -w.i;
        return w;
    }

    // Phase 1: residue h of the x DFT of volume v, HBM -> VGPRs -> LDS planes 0 .. M-1.
    static FX_HD void xpass(int tid, long v, int h, const cx<T>* __restrict__ in, cx<T>* sm,
                            const Bank<T>* __restrict__ bk)
    {
        // Waves whose points of the last block all lie past the plane leave it out.
        const bool last = wave_first(tid) + (C::PPT - 1) * C::NT < C::PLANE;
        if (C::PPT == 1 || last) xrun<C::PPT>(tid, v, h, in, sm, bk);
        else xrun<C::PPT == 1 ? 1 : C::PPT - 1>(tid, v, h, in, sm, bk);
    }
    // Point of the kk-th of NK thread blocks, or PLANE and above past the end.
    template <int NK>
    static FX_HD int point(int tid, int h, int kk)
    {
        if constexpr (C::OR == 1) return tid + ((kk + h) % NK) * C::NT;
        const int p = tid + kk * C::NT;
        if constexpr (C::OR == 2) {
            if (p >= C::PLANE) return p;
            const int w = p + h * (C::PLANE / C::R);
            return w < C::PLANE ? w : w - C::PLANE;
        }
        return p;
    }
    // First thread of tid's wave.
    static FX_HD int wave_first(int tid)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return __builtin_amdgcn_readfirstlane(tid & ~63);
#else
        return tid & ~63;
#endif
    }
    // NK blocks of points as one stream of NK * R groups of M loads (group (kk, m): planes
    // M m .. M m + M - 1 at point kk), PF groups in flight.
    template <int NK>
    static FX_HD void xrun(int tid, long v, int h, const cx<T>* __restrict__ in, cx<T>* sm,
                           const Bank<T>* __restrict__ bk)
    {
        constexpr int E = (int)sizeof(cx<T>), NG = NK * C::R;
        constexpr int PF = C::PF < NG ? C::PF : NG;
        const Window<T> win(in + v * (long)C::V, C::V);
        cx<T> wr[C::R], tw[C::M];
#pragma unroll
        for (int m = 1; m < C::R; ++m) wr[m] = w0(C::M * ((m * h) % C::R), bk);
#pragma unroll
        for (int n = 1; n < C::M; ++n) tw[n] = w0(n * h, bk);
        unsigned off[NK];
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
            const int p = point<NK>(tid, h, kk);
            off[kk] = p < C::PLANE ? (unsigned)(p * E) : Window<T>::kNone;
        }
        cx<T> buf[PF][C::M], a[C::M];
#pragma unroll
        for (int g = 0; g < PF; ++g)
#pragma unroll
            for (int n = 0; n < C::M; ++n)
                buf[g][n] = win.ld(off[g / C::R], (unsigned)((n + C::M * (g % C::R)) * C::PLANE * E));
        sched_fence();
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int m = g % C::R, f = g + PF;
#pragma unroll
            for (int n = 0; n < C::M; ++n)
                a[n] = m == 0 ? buf[g % PF][n] : a[n] + cmul(buf[g % PF][n], wr[m]);
            if (m > 0) {
#pragma unroll
                for (int n = 0; n < C::M; ++n) settle(a[n]);
            }
            if (f < NG) {
#pragma unroll
                for (int n = 0; n < C::M; ++n)
                    buf[f % PF][n] =
                        win.ld(off[f / C::R], (unsigned)((n + C::M * (f % C::R)) * C::PLANE * E));
            }
            if (m == C::R - 1) {
#pragma unroll
                for (int n = 1; n < C::M; ++n) a[n] = cmul(a[n], tw[n]);
                dft<C::M, C::S, T, C::ALG>(a, bk);
                const int p = (int)(off[g / C::R] / E);
                if (p < C::PLANE) {
                    const int y = p / C::N2;
                    const int z = p - y * C::N2;
#pragma unroll
                    for (int q = 0; q < C::M; ++q) sm[q * C::SS + y * C::YS + z] = a[q];
                }
            }
            sched_fence();
        }
    }
    // Phase 2: z lines (plane s, y).
    static FX_HD void zpass(int tid, cx<T>* sm, const Bank<T>* __restrict__ bk)
    {
        lds_pass<C::N2, 1, C::S, C::ALG, C::NT>(
            tid, sm, C::M * C::N1,
            [](int l) {
                const int s = l / C::N1;
                const int y = l - s * C::N1;
                return s * C::SS + y * C::YS;
            },
            bk);
    }
    // Phase 3: y lines (plane s, z), LDS -> output x-plane R s + h (coalesced across z).
    static FX_HD void ypass(int tid, long v, int h, const cx<T>* sm, cx<T>* __restrict__ out,
                            const Bank<T>* __restrict__ bk, T scl)
    {
        cx<T>* __restrict__ dst = out + v * (long)C::V;
        for (int l = tid; l < C::M * C::N2; l += C::NT) {
            const int s = l / C::N2;
            const int z = l - s * C::N2;
            cx<T> t[C::N1];
#pragma unroll
            for (int j = 0; j < C::N1; ++j) t[j] = sm[s * C::SS + j * C::YS + z];
            dft<C::N1, C::S, T, C::ALG>(t, bk);
            cx<T>* __restrict__ o = dst + (long)(C::R * s + h) * C::PLANE + z;
            if (scl != T(1)) {
#pragma unroll
                for (int k = 0; k < C::N1; ++k) st_hint<C::HS>(o + k * C::N2, scale(t[k], scl));
            } else {
#pragma unroll
                for (int k = 0; k < C::N1; ++k) st_hint<C::HS>(o + k * C::N2, t[k]);
            }
        }
    }
};

template <class C>
__global__ void __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::WPE, 8)))
    k_xres(const cx<typename C::T>* __restrict__ in, cx<typename C::T>* __restrict__ out,
           long nvol, const Bank<typename C::T>* __restrict__ bk, typename C::T scl)
{
    using K = XRes<C>;
    __shared__ cx<typename C::T> sm[C::LDS];
    long v;
    int h;
    K::task(blockIdx.x, v, h);
    if (v >= nvol) return;   // uniform over the workgroup, before any barrier
    const int tid = threadIdx.x;
    K::xpass(tid, v, h, in, sm, bk);
    __syncthreads();
    K::zpass(tid, sm, bk);
    __syncthreads();
    K::ypass(tid, v, h, sm, out, bk, scl);
}

}  // namespace fx

#include <fx_xres_launch.hpp>
