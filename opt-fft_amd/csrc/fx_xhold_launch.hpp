// Device launcher and registry descriptor of the register-holding residue-split kernel (xhold.hpp).
#pragma once

namespace fx {

template <class C>
hipError_t launch_xhold(const void* in, void* out, long nvol, const void* bank, double scl,
                       unsigned*, hipStream_t stream)
{
    using T = typename C::T;
    if (nvol <= 0) return hipSuccess;
    const long grid = XHold<C>::grid(nvol);
    if (grid >= (1L << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_xhold<C>), dim3((unsigned)grid), dim3(C::NT), 0, stream,
                       (const cx<T>*)in, (cx<T>*)out, nvol, (const Bank<T>*)bank, (T)scl);
    return hipGetLastError();
}

// Compute units that launch_rounds (xrounds.hpp) plans for.
inline int rounds_cus() { return cu_count(); }

template <class C>
KernelDesc xhold_desc(const char* name)
{
    return KernelDesc{C::N0, C::N1, C::N2, prec_of<typename C::T>(), C::S, kFused, 1, C::NT,
                      C::V17, 0, sizeof(cx<typename C::T>) * (size_t)C::LDS, name,
                      &launch_xhold<C>};
}

}  // namespace fx
