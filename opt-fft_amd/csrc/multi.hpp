// One persistent launch over a mixed batch: several items, each a batch of volumes of one
// of the fused geometries (6^3, 8^3, 12^3, 17^3, 8x8x16) in either direction.
//
// The host cuts every item into blocks (VPW volumes, the tile the preset gives that
// geometry), sorts the blocks heaviest first into a task list, and launches one grid of
// resident workgroups that take tasks from a claim counter (claim_block).  A task runs the pipelined fused
// pass structure of its geometry (x from HBM into VGPRs, z in LDS, y from LDS to HBM) out
// of one LDS buffer sized for the largest block.  The backward direction reuses the forward
// code: conj(DFT(conj(x))) is the unnormalised backward DFT, and both conjugations are sign
// flips folded into the load and the store.
#pragma once
#include "kernels.hpp"

namespace fx {

constexpr int kMultiMaxItems = 16;
constexpr int kMultiGeoms = 5;   // 6^3, 8^3, 12^3, 17^3, 8x8x16
constexpr int kMultiShape[kMultiGeoms][3] = {{6, 6, 6}, {8, 8, 8}, {12, 12, 12}, {17, 17, 17},
                                             {8, 8, 16}};

template <typename T>
struct MultiItem {
    const cx<T>* in;
    cx<T>* out;
    long nvol;
    int code;    // index into kMultiShape
    int conj;    // 1 for the backward direction
    T scale;
};

template <typename T>
struct MultiArgs {
    MultiItem<T> item[kMultiMaxItems];
};

// Tile presets: workgroup size and volumes per block for each geometry code.
template <typename T, int PRESET>
struct MultiPreset;
// 320 threads: 90-100% of the lanes busy in every line pass.
template <typename T>
struct MultiPreset<T, 0> {
    static constexpr int NT = 320;
    static constexpr int HN = 0;  // streaming hints (FusedCfg::HN): none
    using G0 = FusedCfg<6, 6, 6, T, -1, 8, NT, 1, 0, 1>;
    using G1 = FusedCfg<8, 8, 8, T, -1, 5, NT, 1, 0, 1>;
    using G2 = FusedCfg<12, 12, 12, T, -1, 2, NT, 1, 0, 1>;
    using G3 = FusedCfg<17, 17, 17, T, -1, 1, NT, 0, 0, 1>;
    using G4 = FusedCfg<8, 8, 16, T, -1, 2, NT, 1, 0, 1>;
};
// 640 threads: twice the volumes per block.
template <typename T>
struct MultiPreset<T, 1> {
    static constexpr int NT = 640;
    static constexpr int HN = 0;
    using G0 = FusedCfg<6, 6, 6, T, -1, 16, NT, 1, 0, 1>;
    using G1 = FusedCfg<8, 8, 8, T, -1, 10, NT, 1, 0, 1>;
    using G2 = FusedCfg<12, 12, 12, T, -1, 4, NT, 1, 0, 1>;
    using G3 = FusedCfg<17, 17, 17, T, -1, 2, NT, 0, 0, 1>;
    using G4 = FusedCfg<8, 8, 16, T, -1, 5, NT, 1, 0, 1>;
};

// 640 threads, every geometry's block sized to the LDS the two 17^3 volumes need (78.6 KB
// at complex64): the small geometries move 2-4x the bytes per task of preset 1, in the same
// two resident workgroups per CU.
template <typename T>
struct MultiPreset<T, 2> {
    static constexpr int NT = 640;
    static constexpr int HN = 0;
    using G0 = FusedCfg<6, 6, 6, T, -1, 38, NT, 1, 0, 1>;
    using G1 = FusedCfg<8, 8, 8, T, -1, 17, NT, 1, 0, 1>;
    using G2 = FusedCfg<12, 12, 12, T, -1, 5, NT, 1, 0, 1>;
    using G3 = FusedCfg<17, 17, 17, T, -1, 2, NT, 0, 0, 1>;
    using G4 = FusedCfg<8, 8, 16, T, -1, 9, NT, 1, 0, 1>;
};
// 320 threads, every geometry's block sized to the LDS of one 17^3 volume (39.3 KB at
// complex64, 78.6 KB at complex128): four (complex64) or two (complex128) resident
// workgroups per CU, each with a whole block of its own.
template <typename T>
struct MultiPreset<T, 3> {
    static constexpr int NT = 320;
    static constexpr int HN = 0;
    using G0 = FusedCfg<6, 6, 6, T, -1, 19, NT, 1, 0, 1>;
    using G1 = FusedCfg<8, 8, 8, T, -1, 8, NT, 1, 0, 1>;
    using G2 = FusedCfg<12, 12, 12, T, -1, 2, NT, 1, 0, 1>;
    using G3 = FusedCfg<17, 17, 17, T, -1, 1, NT, 0, 0, 1>;
    using G4 = FusedCfg<8, 8, 16, T, -1, 4, NT, 1, 0, 1>;
};
// Presets 3 and 1 with linear stores (FusedCfg LIN; L6: 6^3 too).  In one launch the passes' own
// runs are shorter still, since the block order of the y pass decides them: the complex64 mix
// below 165.6 -> 159.0 us as preset 4 (items interleaved 168.4 -> 157.3), 6^3 x 65536 alone 50.1
// -> 46.1 and 12^3 x 8192 46.4 -> 43.9.  Complex128, as preset 5: 17^3 x 1000 43.3 -> 40.5, 12^3 x
// 4000 52.5 -> 50.4, 8^3 x 16000 57.6 -> 55.7; 6^3 x 30000 went from 45.9 to 50.5, so it keeps
// its own stores there.
template <typename T, int B, int L6>
struct LinPreset {
    using Q = MultiPreset<T, B>;
    static constexpr int NT = Q::NT, HN = 0;
    template <class G, int LIN = 1>
    using L = FusedCfg<G::N0, G::N1, G::N2, T, -1, G::VPW, NT, G::PZ, 0, 1, G::IX, LIN>;
    using G0 = L<typename Q::G0, L6>;
    using G1 = L<typename Q::G1>;
    using G2 = L<typename Q::G2>;
    using G3 = L<typename Q::G3>;
    using G4 = L<typename Q::G4>;
};
template <typename T>
struct MultiPreset<T, 4> : LinPreset<T, 3, 1> {};
template <typename T>
struct MultiPreset<T, 5> : LinPreset<T, 1, 0> {};
// Small blocks, sized without regard to 17^3: 192 threads and one 12^3 volume (30 KB at
// complex128), or 320 / 384 and two of complex64.  These presets have a second kernel for
// launches without 17^3 items, whose LDS and registers are those of the other geometries: at
// complex128 five workgroups a CU (88 VGPRs) where 17^3 allows two (184), at complex64 five of
// 320-384 threads instead of four.  Against the best earlier preset (us):
//   complex128, 7:  12^3 x 2401 with 6^3 x 40  33.5 -> 27.4; 6^3 x 2842, 8^3 x 8442  36.3 -> 31.0;
//                   6^3 x 20000, 8^3 x 8000, 12^3 x 3000  86.1 -> 78.8; a hundredth of it 9.1 -> 8.3
//   complex64, 8/9: the same 17.9 -> 12.4 / 13.6; 19.9 -> 17.0 / 16.8; 43.7 -> 40.0 / 40.3; 6.4 -> 6.1
// With 17^3 in the mix (289 lines on 192 threads) preset 6 is ahead at complex128 where the
// small geometries hold most of the bytes, 6^3 x 10000, 8^3 x 4000, 12^3 x 1500, 17^3 x 500
// 65.7 -> 61.2, and 9 at complex64, 12^3 x 4854 with 17^3 x 258 36.3 -> 35.7; 8x8x16 x 6000 with
// 17^3 x 100 takes 58.2 (54.4 as preset 3).  Not registered: 6 and 7 with the items interleaved
// (127-140 us in place of 61-68 at the mix above), 5 interleaved (behind t640_mix or a 192-thread
// preset in each of eleven mixes, 66.7 to 61.9 at the same one, 17^3 x 1000 with 8^3 x 16000 91.7 to
// 81.9), 9 at complex128 (two workgroups a CU: 42.0
// to 31.0 at 6^3 with 8^3), 192 threads at complex64 (within 2% of 8).
template <typename T>
struct MultiPreset<T, 6> {
    static constexpr int NT = 192;
    static constexpr int HN = 0;
    using G0 = FusedCfg<6, 6, 6, T, -1, 5, NT, 1, 0, 1>;
    using G1 = FusedCfg<8, 8, 8, T, -1, 3, NT, 1, 0, 1>;
    using G2 = FusedCfg<12, 12, 12, T, -1, 1, NT, 1, 0, 1>;
    using G3 = FusedCfg<17, 17, 17, T, -1, 1, NT, 0, 0, 1>;
    using G4 = FusedCfg<8, 8, 16, T, -1, 1, NT, 1, 0, 1>;
};
template <typename T>
struct MultiPreset<T, 7> : LinPreset<T, 6, 1> {};
template <typename T>
struct MultiPreset<T, 8> : LinPreset<T, 0, 1> {};
template <typename T>
struct MultiPreset<T, 10> {   // the blocks of preset 9
    static constexpr int NT = 384;
    static constexpr int HN = 0;
    using G0 = FusedCfg<6, 6, 6, T, -1, 10, NT, 1, 0, 1>;
    using G1 = FusedCfg<8, 8, 8, T, -1, 6, NT, 1, 0, 1>;
    using G2 = FusedCfg<12, 12, 12, T, -1, 2, NT, 1, 0, 1>;
    using G3 = FusedCfg<17, 17, 17, T, -1, 1, NT, 0, 0, 1>;
    using G4 = FusedCfg<8, 8, 16, T, -1, 3, NT, 1, 0, 1>;
};
template <typename T>
struct MultiPreset<T, 9> : LinPreset<T, 10, 1> {};
template <int PRESET>
constexpr bool kMultiSmall = PRESET >= 6;   // has the second kernel
// The staged task structure (block HBM -> LDS in one grouped read, z and y in LDS, x pass
// LDS -> HBM with whole-line stores; the per-geometry plans of 6^3, 8^3 and 12^3 complex64
// race to it) was built on presets 0 and 3 and measured slower in one launch: 213-228 us on
// the mix below against 164.5 us for preset 0, and alone 69.8 us at 6^3 x 65536 against
// 50.6 us (the per-geometry staged kernel: 40.0 us at six workgroups per CU; here four, and a
// staged task computes nothing until its whole block has landed).  Not built.
// Measured on the complex64 mix 6^3 x 65536, 8^3 x 32768, 12^3 x 8192, 17^3 x 2048 (not
// built): preset 3 with the items interleaved and nontemporal stores 168.6 us, with
// nontemporal loads, or loads and stores, 174.0 us, against 168.9 us plain on one device;
// preset 2 with nontemporal loads, or loads and stores, 207.8 us against 186.8 us plain.
// (The same blocks on 1024 threads, 32 waves per CU, spill at the 64-VGPR cap: not built.)

constexpr int cmax(int a, int b) { return a > b ? a : b; }

// G17: 17^3 items may occur.  Without them the workgroup's LDS and registers are those of the
// other geometries.
template <typename T, int PRESET, bool G17 = true>
struct MultiCfg {
    using P = MultiPreset<T, PRESET>;
    static constexpr int NT = P::NT;
    static constexpr bool LIN = P::G1::LIN != 0;   // some geometry stores in phase 3
    static constexpr int LDS =
        cmax(cmax(cmax(P::G0::LDS, P::G1::LDS), cmax(P::G2::LDS, G17 ? P::G3::LDS : 0)), P::G4::LDS);
    static constexpr int WPE = waves_per_eu(LDS * (int)sizeof(cx<T>), NT, 0);
    static constexpr int vpw(int code)
    {
        return code == 0 ? P::G0::VPW : code == 1 ? P::G1::VPW : code == 2 ? P::G2::VPW
             : code == 3 ? P::G3::VPW : P::G4::VPW;
    }
};

// Phase `ph` (0: x from HBM, 1: z, 2: y to HBM, or to LDS for 3: copy to HBM, where the block's
// configuration has LIN) of one block of one item.  Phases are
// separated by workgroup barriers; no register state crosses a barrier.
template <class C, int HN>
FX_HD void multi_phase(int ph, int tid, long b, const MultiItem<typename C::T>& it,
                       cx<typename C::T>* sm, const Bank<typename C::T>* __restrict__ bk)
{
    using K = FusedPipe<HintCfg<C, HN>>;
    if (ph == 0) {
        typename K::Regs R;
        K::load_x(tid, b, it.nvol, it.in, R);
        if (it.conj) {
#pragma unroll
            for (int i = 0; i < K::LPT; ++i)
#pragma unroll
                for (int j = 0; j < C::N0; ++j) R[i][j].i = -R[i][j].i;
        }
        K::xpass(tid, b, it.nvol, R, sm, bk);
    } else if (ph == 1) {
        K::zpass(tid, b, it.nvol, sm, bk);
    } else if (ph == 2) {
        K::ypass(tid, b, it.nvol, sm, it.out, bk, it.scale, it.conj != 0);
    } else if constexpr (C::LIN) {
        Fused<C>::copy(tid, b, it.nvol, sm, it.out);
    }
}

template <typename T, int PRESET, bool G17 = true>
FX_HD void multi_task_phase(int ph, int tid, int2 task, const MultiArgs<T>& a, cx<T>* sm,
                            const Bank<T>* __restrict__ bk)
{
    using P = MultiPreset<T, PRESET>;
    const MultiItem<T>& it = a.item[task.x];
    switch (it.code) {
    case 0: multi_phase<typename P::G0, P::HN>(ph, tid, task.y, it, sm, bk); break;
    case 1: multi_phase<typename P::G1, P::HN>(ph, tid, task.y, it, sm, bk); break;
    case 2: multi_phase<typename P::G2, P::HN>(ph, tid, task.y, it, sm, bk); break;
    case 3:
        if constexpr (G17) multi_phase<typename P::G3, P::HN>(ph, tid, task.y, it, sm, bk);
        break;
    default: multi_phase<typename P::G4, P::HN>(ph, tid, task.y, it, sm, bk); break;
    }
}

// Walk the task list: the first task is blockIdx.x, the next ones are claimed from `work`
// (NULL: a fixed stride of gridDim.x).  The claim is issued before phase 0 and published to
// the workgroup at the first barrier.
template <typename T, int PRESET, bool G17 = true>
__device__ __forceinline__ void multi_walk(const MultiArgs<T>& a, const int2* __restrict__ tasks,
                                           int ntasks, const Bank<T>* __restrict__ bk,
                                           unsigned* work, cx<T>* sm, long* s_next)
{
    const int tid = threadIdx.x;
    long t = blockIdx.x;
    while (t < ntasks) {
        long claim = 0;
        if (tid == 0) claim = claim_block(work, ntasks, t);
        const int2 task = tasks[t];
        multi_task_phase<T, PRESET, G17>(0, tid, task, a, sm, bk);
        if (tid == 0) *s_next = claim;
        __syncthreads();
        const long nt = *s_next;
        multi_task_phase<T, PRESET, G17>(1, tid, task, a, sm, bk);
        __syncthreads();
        multi_task_phase<T, PRESET, G17>(2, tid, task, a, sm, bk);
        __syncthreads();
        if constexpr (MultiCfg<T, PRESET>::LIN) {
            multi_task_phase<T, PRESET, G17>(3, tid, task, a, sm, bk);
            __syncthreads();
        }
        t = nt;
    }
}

template <typename T, int PRESET, bool G17 = true>
__global__ void __launch_bounds__((MultiCfg<T, PRESET, G17>::NT))
    __attribute__((amdgpu_waves_per_eu(MultiCfg<T, PRESET, G17>::WPE, 8)))
    k_multi(const MultiArgs<T> a, const int2* __restrict__ tasks, int ntasks,
            const Bank<T>* __restrict__ bk, unsigned* __restrict__ work)
{
    using M = MultiCfg<T, PRESET, G17>;
    __shared__ cx<T> sm[M::LDS];
    __shared__ long s_next;
    multi_walk<T, PRESET, G17>(a, tasks, ntasks, bk, work, sm, &s_next);
}

// Same kernel with the items, the task count and the task list read from device memory, so a
// launch can be captured once in a hipGraph and replayed with new descriptors (serving).
// `work`: the launch's claim counters (kClaimWords, zero before the first launch and left
// at zero by every launch, claim_block), owned by whoever owns the descriptor.
template <typename T>
struct MultiDescriptor {
    MultiArgs<T> args;
    int ntasks;
    int2 tasks[1];  // ntasks entries follow
};

template <typename T, int PRESET>
__global__ void __launch_bounds__((MultiCfg<T, PRESET>::NT))
    __attribute__((amdgpu_waves_per_eu(MultiCfg<T, PRESET>::WPE, 8)))
    k_multi_dev(MultiDescriptor<T>* __restrict__ d, const Bank<T>* __restrict__ bk,
                unsigned* __restrict__ work)
{
    using M = MultiCfg<T, PRESET>;
    __shared__ cx<T> sm[M::LDS];
    __shared__ long s_next;
    const int ntasks = d->ntasks;
    multi_walk<T, PRESET>(d->args, d->tasks, ntasks, bk, ntasks >= 2L * gridDim.x ? work : nullptr,
                          sm, &s_next);
}

// Does any item of a launch hold 17^3 volumes?
template <typename T>
bool multi_has17(const MultiArgs<T>& a)
{
    for (const MultiItem<T>& it : a.item)
        if (it.code == 3 && it.nvol > 0) return true;
    return false;
}

// Registry entry of a multi kernel.
// `work`: claim counter as for LaunchFn (registry.hpp).
typedef hipError_t (*MultiLaunchFn)(const void* args, const int2* tasks, int ntasks,
                                    const void* bank, unsigned* work, hipStream_t stream);
// Launch of the descriptor-reading form on `grid` workgroups with claim counters `work`.
typedef hipError_t (*MultiDevLaunchFn)(const void* descriptor, const void* bank, unsigned* work,
                                       int grid, hipStream_t stream);
struct MultiDesc {
    int prec;
    int preset;
    int nthreads;
    int vpw[kMultiGeoms];
    size_t lds_bytes;
    const char* name;
    MultiLaunchFn launch;
    MultiDevLaunchFn launch_dev;  // NULL: no descriptor form
    int (*resident_grid)();  // persistent grid of the descriptor form on the current device
    int algo = 0;            // as KernelDesc::algo: 0 FFT, 1 / 2 matrix-core bf16 / fp16
    // Workgroups `launch` starts for ntasks, of items with or without 17^3.
    long (*launch_grid)(long ntasks, bool g17) = nullptr;
    int order = 0;  // task order (multi_tasks): 0 heaviest first, 1 items interleaved
};

void register_multi(std::vector<MultiDesc>& r);
const std::vector<MultiDesc>& multi_registry();

}  // namespace fx

#include <fx_multi_launch.hpp>
