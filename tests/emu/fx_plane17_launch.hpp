// TEST INFRASTRUCTURE: host emulation of the plane-per-workgroup 17^3 kernel (plane17.hpp) with
// the same phase functions, each thread keeping its own cosines and sines.
#pragma once
#include <vector>

namespace fx {

template <class C>
hipError_t launch_plane17(const void* in, void* out, long nvol, const void* bank, double scl,
                          unsigned*, hipStream_t)
{
    using T = typename C::T;
    using K = Plane17<C>;
    if (nvol <= 0) return hipSuccess;
    const Bank<T>* bk = (const Bank<T>*)bank;
    EmuLds<T> lds(C::LDS);
    std::vector<typename K::Regs> R(C::NT);
    const long grid = K::grid(nvol);
    for (long g = 0; g < grid; ++g) {
        long v;
        int k;
        K::task(g, v, k);
        if (v >= nvol) continue;
        lds.poison();
        cx<T>* sm = lds.data();
        emu_threads(C::NT, [&](int t) { K::xpass(t, v, k, (const cx<T>*)in, sm, R[t], bk); });
        emu_threads(C::NT, [&](int t) { K::zpass(t, sm, R[t]); });
        emu_threads(C::NT, [&](int t) { K::ypass(t, v, k, sm, (cx<T>*)out, R[t], (T)scl); });
        if (!lds.guards_ok() && g_emu_bad_block < 0) g_emu_bad_block = g;
    }
    return hipSuccess;
}

template <class C>
KernelDesc plane17_desc(const char* name)
{
    return KernelDesc{C::L, C::L, C::L, prec_of<typename C::T>(), C::S, kFused, 1, C::NT, 1, 0,
                      sizeof(cx<typename C::T>) * (size_t)C::LDS, name, &launch_plane17<C>, 0,
                      C::TINY};
}

}  // namespace fx
