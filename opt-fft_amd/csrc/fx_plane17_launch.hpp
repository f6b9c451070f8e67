// Device launcher and registry descriptor of the plane-per-workgroup 17^3 kernel (plane17.hpp).
#pragma once

namespace fx {

template <class C>
hipError_t launch_plane17(const void* in, void* out, long nvol, const void* bank, double scl,
                          unsigned*, hipStream_t stream)
{
    using T = typename C::T;
    if (nvol <= 0) return hipSuccess;
    if (nvol >= (1L << 31) / C::L - C::kXcds) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_plane17<C>), dim3((unsigned)Plane17<C>::grid(nvol)), dim3(C::NT), 0, stream,
                       (const cx<T>*)in, (cx<T>*)out, nvol, (const Bank<T>*)bank, (T)scl);
    return hipGetLastError();
}

template <class C>
KernelDesc plane17_desc(const char* name)
{
    return KernelDesc{C::L, C::L, C::L, prec_of<typename C::T>(), C::S, kFused, 1, C::NT, 1, 0,
                      sizeof(cx<typename C::T>) * (size_t)C::LDS, name, &launch_plane17<C>, 0,
                      C::TINY};
}

}  // namespace fx
