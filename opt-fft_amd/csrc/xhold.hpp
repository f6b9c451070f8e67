// Residue-split single pass with most of a workgroup's planes in registers: the x DFT split
// over R workgroups (xres.hpp has the arithmetic), each of which keeps its N0 / R output
// planes on its CU, PR at a time in LDS and the rest in VGPRs.
//
//   x pass: as in XRes, a thread per (y, z) point and PPT points per thread, M = N0 / R planes
//     of the output in registers; planes 0 .. PR-1 go to LDS, the rest stays (H);
//   rounds: z lines and then y lines of the PR planes in LDS, the y pass storing to HBM; the
//     next PR planes go from H to LDS while those stores drain.
//
// Why: XRes at 36^3 complex128 needs R = 6 for its planes to fit in LDS, and is bound by the
// six reads of every element from L2 (its x passes alone take 36 of 57 us at x 128).  The 18
// planes of R = 2 (373 KB) fit in a CU's 160 KB of LDS and 512 KB of VGPRs together: 256
// threads, one wave per SIMD, 12 planes held, whole 36-point lines in registers beside them.
//   36^3 x 128, r2h6   56.8 -> 40.5 us (4.7 TB/s); x 300 125.3 -> 108.7, x 512 219 -> 158
//   36^3 x 64, r4h6    33.4 -> 26.4 us (448 threads, 9 planes, 3 held; r2 34.0)
//   24x24x48 x 300     74.7 -> 66.4 us (r2h8); x 64 20.5 against 16.4 us for XRes, whose four
//                      workgroups a volume fill the device there
//   24^3 x 365, r2h8   36.7 -> 32.4 us (two workgroups per CU, 4 of 12 planes held)
//   24x24x48 complex64 x 256, r1h12  28.9 -> 24.6 us (a volume per workgroup)
//   24^3 complex64 x 678, r1h8l  37.4 (LDS-resident, one volume a CU) -> 30.9 us with four
//                      workgroups per CU; x 1989 102.7 -> 88.0
//   36^3 complex64 x 255, r1h12l  45.8 (split-resident) -> 40.8 us, x 589 123.3 -> 108.6;
//                      r2h9l x 128 37.3 -> 25.5 us
// At R = 2 a copy with the same reads, the same stores and no arithmetic takes 37.5 us at
// 36^3 x 128: reads and stores come in turns, since the one round of workgroups walks in step.
// The two workgroups of a volume walk it in the same order (19.6 us for the reads alone);
// starts a plane part apart, which XRes needs at R = 6, read it at 29.4.
// Stores are nontemporal: with plain ones 36^3 x 128 takes 50.8 us.  PR = 7 (42.5-43.0 us) and
// 5 (41.2) against 6; 27 loads in flight, 18-36 being within 1%.
//
// LIN = 1: the y pass writes its lines back to LDS and a copy stores the planes, 16 bytes a
// lane, where rows are not whole 128-byte lines and an element is 8 bytes: stores of 288-byte
// rows at 36^3 complex64 took 27 us for 95 MB (49.0 us in all), the copy's 40.8.  With rows of
// 576 (36^3 complex128: 44.7 against 40.5 us) or 384 bytes (24x24x48 complex64: 27.2 against
// 24.6) the extra LDS round trip costs more than it gains; at 24^3 complex64 (192) it gains
// from about 500 volumes on, 30.9 against 33.1 us at x 678, and loses at x 300, 22.1 against
// 20.1, so both are raced.
#pragma once

#include <type_traits>
#include <utility>

#include "xres.hpp"

namespace fx {

// GS: planes per group of loads; PF: groups in flight during the x pass; LIN: see above.
template <int N0_, int N1_, int N2_, typename T_, int S_, int R_, int NT_, int PR_, int GS_, int PF_,
          int LIN_ = 0, int HS_ = 1, int PZ_ = 1, int ALG_ = 0>
struct XHoldCfg {
    using T = T_;
    static constexpr int N0 = N0_, N1 = N1_, N2 = N2_, S = S_, R = R_, NT = NT_, PR = PR_;
    static constexpr int GS = GS_, PF = PF_, LIN = LIN_, HS = HS_, PZ = PZ_, ALG = ALG_, V17 = ALG_;
    static constexpr int M = N0 / R;                    // output x-planes per workgroup
    static constexpr int V = N0 * N1 * N2;
    static constexpr int PLANE = N1 * N2;
    static constexpr int PPT = (PLANE + NT - 1) / NT;   // (y, z) points per thread
    static constexpr int RD = (M + PR - 1) / PR;        // rounds
    static constexpr int YS = N2 + PZ;                  // LDS pitch between z rows
    static constexpr int SS = N1 * YS;                  // LDS pitch between planes
    static constexpr int LDS = PR * SS;                 // elements
    static constexpr int WPE = waves_per_eu(LDS * (int)sizeof(cx<T>), NT, 0);
    static constexpr int kXcds = 8;
    static_assert(N0 % R == 0 && M % GS == 0 && NT % 64 == 0, "whole groups of planes, whole waves");
    static_assert(PR < M, "with every plane in LDS this is XRes");
    static_assert(LDS * (int)sizeof(cx<T>) <= 163840, "the planes of a round fit in LDS");
};

// f(std::integral_constant<int, i>{}) for i = 0 .. N-1: indices constant from the front end on,
// so the arrays they select stay in registers however long the body.
template <typename F, int... I>
FX_HD void static_for(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
FX_HD void static_for(F&& f)
{
    static_for(f, std::make_integer_sequence<int, N>{});
}

template <class C>
struct XHold {
    using T = typename C::T;
    using Regs = cx<T>[C::PPT][C::M - C::PR];

    // Planes of round rd.
    static constexpr int planes(int rd) { return C::M - rd * C::PR < C::PR ? C::M - rd * C::PR : C::PR; }

    static FX_HD void task(long g, long& v, int& h) { XRes<C>::task(g, v, h); }
    static FX_HD long grid(long nvol) { return XRes<C>::grid(nvol); }

    // x pass: groups of GS loads in the order (point, planes c GS .., m), PF of them in flight.
    static FX_HD void xpass(int tid, long v, int h, const cx<T>* __restrict__ in, cx<T>* sm, Regs& H,
                            const Bank<T>* __restrict__ bk)
    {
        constexpr int E = (int)sizeof(cx<T>), NC = C::M / C::GS, GP = NC * C::R;  // groups per point
        constexpr int NG = C::PPT * GP;
        const Window<T> win(in + v * (long)C::V, C::V);
        unsigned off[C::PPT];
#pragma unroll
        for (int kk = 0; kk < C::PPT; ++kk) {
            const int p = tid + kk * C::NT;
            off[kk] = p < C::PLANE ? (unsigned)(p * E) : Window<T>::kNone;
        }
        cx<T> buf[C::PF][C::GS], a[C::M];
        auto load = [&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value, kk = g / GP, c = g % GP / C::R, m = g % C::R;
            static_for<C::GS>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, plane = c * C::GS + i + C::M * m;
                buf[g % C::PF][i] = win.ld(off[kk], (unsigned)(plane * C::PLANE * E));
            });
        };
        static_for<C::PF>(load);
        sched_fence();
        static_for<NG>([&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value, kk = g / GP, c = g % GP / C::R, m = g % C::R;
            static_for<C::GS>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, n = c * C::GS + i;
                const cx<T> b = buf[g % C::PF][i];
                if constexpr (m == 0) a[n] = b;
                else if constexpr (C::R == 2) a[n] = a[n] + scale(b, h ? T(-1) : T(1));
                else a[n] = a[n] + cmul(b, XRes<C>::w0(C::M * ((m * h) % C::R), bk));
                if constexpr (m > 0) settle(a[n]);
            });
            if constexpr (g + C::PF < NG) load(std::integral_constant<int, g + C::PF>{});
            if constexpr (g % GP == GP - 1) {
                static_for<C::M>([&](auto nc) __attribute__((always_inline)) {
                    constexpr int n = decltype(nc)::value;
                    if constexpr (n > 0 && C::R > 1) a[n] = cmul(a[n], XRes<C>::w0(n * h, bk));
                });
                dft<C::M, C::S, T, C::ALG>(a, bk);
                const int p = tid + kk * C::NT;
                if (p < C::PLANE) {
                    const int y = p / C::N2;
                    const int z = p - y * C::N2;
                    static_for<C::PR>([&](auto qc) __attribute__((always_inline)) {
                        constexpr int q = decltype(qc)::value;
                        sm[q * C::SS + y * C::YS + z] = a[q];
                    });
                }
                static_for<C::M - C::PR>([&](auto qc) __attribute__((always_inline)) {
                    constexpr int q = decltype(qc)::value;
                    H[kk][q] = a[q + C::PR];
                    settle(H[kk][q]);
                });
            }
            sched_fence();
        });
    }
    // Planes of round rd >= 1 from registers to LDS.
    template <int rd>
    static FX_HD void put(int tid, const Regs& H, cx<T>* sm)
    {
#pragma unroll
        for (int kk = 0; kk < C::PPT; ++kk) {
            const int p = tid + kk * C::NT;
            if (p < C::PLANE) {
                const int y = p / C::N2;
                const int z = p - y * C::N2;
#pragma unroll
                for (int q = 0; q < planes(rd); ++q)
                    sm[q * C::SS + y * C::YS + z] = H[kk][(rd - 1) * C::PR + q];
            }
        }
    }
    template <int rd>
    static FX_HD void zpass(int tid, cx<T>* sm, const Bank<T>* __restrict__ bk)
    {
        lds_pass<C::N2, 1, C::S, C::ALG, C::NT>(
            tid, sm, planes(rd) * C::N1,
            [](int l) {
                const int s = l / C::N1;
                const int y = l - s * C::N1;
                return s * C::SS + y * C::YS;
            },
            bk);
    }
    // y lines, LDS -> output x-planes R (rd PR + s) + h (rows of N2 elements, in order); LIN = 1:
    // back to LDS, for copy.
    template <int rd>
    static FX_HD void ypass(int tid, long v, int h, cx<T>* sm, cx<T>* __restrict__ out,
                            const Bank<T>* __restrict__ bk, T scl)
    {
        cx<T>* __restrict__ dst = out + v * (long)C::V + (long)(C::R * rd * C::PR + h) * C::PLANE;
        for (int l = tid; l < planes(rd) * C::N2; l += C::NT) {
            const int s = l / C::N2;
            const int z = l - s * C::N2;
            cx<T>* t0 = sm + s * C::SS + z;
            cx<T> t[C::N1];
#pragma unroll
            for (int j = 0; j < C::N1; ++j) t[j] = t0[j * C::YS];
            dft<C::N1, C::S, T, C::ALG>(t, bk);
            cx<T>* __restrict__ o = dst + s * (C::R * C::PLANE) + z;
            // Always scaled: a product by 1 is exact.
#pragma unroll
            for (int k = 0; k < C::N1; ++k) {
                if constexpr (C::LIN) t0[k * C::YS] = scale(t[k], scl);
                else st_hint<C::HS>(o + k * C::N2, scale(t[k], scl));
            }
        }
    }
    // LIN = 1: the round's planes LDS -> HBM, 16 bytes a lane and consecutive lanes adjacent.
    template <int rd>
    static FX_HD void copy(int tid, long v, int h, const cx<T>* sm, cx<T>* __restrict__ out)
    {
        constexpr int W = 16 / (int)sizeof(cx<T>);   // elements per lane
        static_assert(C::N2 % W == 0, "a lane's elements lie in one row");
        cx<T>* __restrict__ dst = out + v * (long)C::V + (long)(C::R * rd * C::PR + h) * C::PLANE;
#pragma unroll 4
        for (int e = tid; e < planes(rd) * C::PLANE / W; e += C::NT) {
            const int s = e / (C::PLANE / W);
            const int q = (e - s * (C::PLANE / W)) * W;
            const int y = q / C::N2;
            const cx<T>* t = sm + s * C::SS + y * C::YS + (q - y * C::N2);
            st_wide<C::HS>(dst + s * (C::R * C::PLANE) + q, t);
        }
    }
};

template <class C, int rd = 0>
__device__ __forceinline__ void xhold_rounds(int tid, long v, int h, const typename XHold<C>::Regs& H,
                                             cx<typename C::T>* sm, cx<typename C::T>* __restrict__ out,
                                             const Bank<typename C::T>* __restrict__ bk, typename C::T scl)
{
    using K = XHold<C>;
    if constexpr (rd > 0) {
        __syncthreads();
        K::template put<rd>(tid, H, sm);
    }
    __syncthreads();
    K::template zpass<rd>(tid, sm, bk);
    __syncthreads();
    K::template ypass<rd>(tid, v, h, sm, out, bk, scl);
    if constexpr (C::LIN) {
        __syncthreads();
        K::template copy<rd>(tid, v, h, sm, out);
    }
    if constexpr (rd + 1 < C::RD) xhold_rounds<C, rd + 1>(tid, v, h, H, sm, out, bk, scl);
}

template <class C>
__global__ void __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
    k_xhold(const cx<typename C::T>* __restrict__ in, cx<typename C::T>* __restrict__ out, long nvol,
            const Bank<typename C::T>* __restrict__ bk, typename C::T scl)
{
    using K = XHold<C>;
    __shared__ cx<typename C::T> sm[C::LDS];
    long v;
    int h;
    K::task(blockIdx.x, v, h);
    if (v >= nvol) return;   // uniform over the workgroup, before any barrier
    const int tid = threadIdx.x;
    typename K::Regs H;
    K::xpass(tid, v, h, in, sm, H, bk);
    xhold_rounds<C>(tid, v, h, H, sm, out, bk, scl);
}

}  // namespace fx

#include <fx_xhold_launch.hpp>
