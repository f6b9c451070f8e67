// Device launchers and registry descriptors for the kernel templates of kernels.hpp.
// Included at the end of kernels.hpp through the include path.
#pragma once
namespace fx {

// Compute units of the current device (cached per device ordinal).
inline int cu_count()
{
    static int cache[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    if (!cache[dev]) {
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            c < 1)
            c = 1;
        cache[dev] = c;
    }
    return cache[dev];
}

// Workgroups of kernel `f` (nt threads) resident per CU.  Launchers keep it in a static of
// their own instantiation: looked up by kernel address in a locked map on every launch, it was
// a tenth of a small persistent launch (12^3 complex128 x 1, back to back: 4.15 us a launch
// against 3.76 with the static).
template <typename F>
int resident_per_cu(F f, int nt)
{
    int o = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&o, reinterpret_cast<const void*>(f), nt, 0) !=
            hipSuccess || o < 1)
        o = 1;
    return o;
}

// Grid of a persistent kernel with `per` resident workgroups per CU: at most `cap` per CU, never
// more than nblocks.
inline long persistent_grid(int per, int cap, long nblocks)
{
    const long g = (long)(per < cap ? per : cap) * cu_count();
    return g < nblocks ? g : nblocks;
}

// Dynamic block claiming pays when workgroups walk several blocks each; when the grid
// covers (nearly) every block, the one-per-workgroup failing claims would only queue on a
// single address, so those launches walk a fixed stride instead.
inline unsigned* claim_counter(unsigned* work, long grid, long nblocks)
{
    return nblocks >= 2 * grid ? work : nullptr;
}

template <class C>
hipError_t launch_fused(const void* in, void* out, long nvol, const void* bank, double scl,
                        unsigned*, hipStream_t stream)
{
    using T = typename C::T;
    if (nvol <= 0) return hipSuccess;
    const long grid = (nvol + C::VPW - 1) / C::VPW;
    hipLaunchKernelGGL((k_fused<C>), dim3((unsigned)grid), dim3(C::NT), 0, stream,
                       (const cx<T>*)in, (cx<T>*)out, nvol, (const Bank<T>*)bank, (T)scl);
    return hipGetLastError();
}

template <class C, int PERSIST, int ST = 0, int HN = 3>
hipError_t launch_fpipe(const void* in, void* out, long nvol, const void* bank, double scl,
                        unsigned* work, hipStream_t stream)
{
    using T = typename C::T;
    if (nvol <= 0) return hipSuccess;
    const long nblocks = (nvol + C::VPW - 1) / C::VPW;
    if (nblocks >= (1L << 31)) return hipErrorInvalidValue;
    using P = PipeCfg<C, PERSIST, ST, HN>;
    long grid = nblocks;
    if constexpr (PERSIST > 0) {
        static const int per = resident_per_cu(k_fpipe<P>, C::NT);
        grid = persistent_grid(per, PERSIST, nblocks);
    }
    hipLaunchKernelGGL((k_fpipe<P>), dim3((unsigned)grid), dim3(C::NT), 0, stream,
                       (const cx<T>*)in, (cx<T>*)out, nvol, nblocks, (const Bank<T>*)bank,
                       (T)scl, claim_counter(work, grid, nblocks));
    return hipGetLastError();
}

template <class C>
hipError_t launch_pencil(const void* in, void* out, long nvol, const void* bank, double scl,
                         unsigned* work, hipStream_t stream)
{
    using T = typename C::T;
    if (nvol <= 0) return hipSuccess;
    const long chunk = C::CHUNK > 0 ? C::CHUNK : nvol;
    for (long v0 = 0; v0 < nvol; v0 += chunk) {
        const long nv = (nvol - v0) < chunk ? (nvol - v0) : chunk;
        const cx<T>* src = (const cx<T>*)in + v0 * C::V;
        cx<T>* dst = (cx<T>*)out + v0 * C::V;
        const long nslab = nv * C::N0;
        const long nblocks = (nslab + C::SPW - 1) / C::SPW;
        if constexpr (C::PIPE > 0) {
            static const int per = resident_per_cu(k_spipe<C>, C::NT);
            const long ga = persistent_grid(per, C::PIPE, nblocks);
            if (nblocks >= (1L << 31)) return hipErrorInvalidValue;
            hipLaunchKernelGGL((k_spipe<C>), dim3((unsigned)ga), dim3(C::NT), 0, stream, src,
                               dst, nslab, nblocks, (const Bank<T>*)bank,
                               claim_counter(work, ga, nblocks));
        } else {
            hipLaunchKernelGGL((k_slab<C>), dim3((unsigned)nblocks), dim3(C::NT), 0, stream,
                               src, dst, nslab, (const Bank<T>*)bank);
        }
        const long nlines = nv * C::PLANE;
        const long gb = (nlines + C::NTB - 1) / C::NTB;
        hipLaunchKernelGGL((k_xline<C>), dim3((unsigned)gb), dim3(C::NTB), 0, stream, dst,
                           nlines, (const Bank<T>*)bank, (T)scl);
    }
    return hipGetLastError();
}

template <class C>
KernelDesc fused_desc(const char* name)
{
    return KernelDesc{C::N0, C::N1, C::N2, prec_of<typename C::T>(), C::S, kFused, C::VPW,
                      C::NT, C::V17, 0, sizeof(cx<typename C::T>) * (size_t)C::LDS, name,
                      &launch_fused<C>};
}

template <class C, int PERSIST, int ST = 0, int HN = 3>
KernelDesc fpipe_desc(const char* name)
{
    return KernelDesc{C::N0, C::N1, C::N2, prec_of<typename C::T>(), C::S, kFused, C::VPW,
                      C::NT, C::V17, PERSIST, sizeof(cx<typename C::T>) * (size_t)C::LDS, name,
                      &launch_fpipe<C, PERSIST, ST, HN>};
}

template <class C>
KernelDesc pencil_desc(const char* name)
{
    return KernelDesc{C::N0, C::N1, C::N2, prec_of<typename C::T>(), C::S, kPencil, C::SPW,
                      C::NT, 0, C::PIPE, sizeof(cx<typename C::T>) * (size_t)C::LDS, name,
                      &launch_pencil<C>};
}

}  // namespace fx
