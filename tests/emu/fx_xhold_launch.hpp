// TEST INFRASTRUCTURE: host emulation of the register-holding residue-split kernel (xhold.hpp)
// with the same phase functions, each thread keeping its own held planes; the LDS is
// re-poisoned before every round's planes are put.
#pragma once
#include <vector>

namespace fx {

template <class C, int rd, typename Box>
void emu_xhold_round(long v, int h, std::vector<Box>& H, EmuLds<typename C::T>& lds,
                     cx<typename C::T>* dst, const Bank<typename C::T>* bk, typename C::T scl)
{
    using K = XHold<C>;
    cx<typename C::T>* sm = lds.data();
    if constexpr (rd > 0) {
        lds.poison();
        emu_threads(C::NT, [&](int t) { K::template put<rd>(t, H[t].r, sm); });
    }
    emu_threads(C::NT, [&](int t) { K::template zpass<rd>(t, sm, bk); });
    emu_threads(C::NT, [&](int t) { K::template ypass<rd>(t, v, h, sm, dst, bk, scl); });
    if constexpr (C::LIN) emu_threads(C::NT, [&](int t) { K::template copy<rd>(t, v, h, sm, dst); });
    if (!lds.guards_ok() && g_emu_bad_block < 0) g_emu_bad_block = v;
    if constexpr (rd + 1 < C::RD) emu_xhold_round<C, rd + 1>(v, h, H, lds, dst, bk, scl);
}

template <class C>
hipError_t launch_xhold(const void* in, void* out, long nvol, const void* bank, double scl,
                        unsigned*, hipStream_t)
{
    using T = typename C::T;
    using K = XHold<C>;
    struct Box {
        typename K::Regs r;
    };
    if (nvol <= 0) return hipSuccess;
    const Bank<T>* bk = (const Bank<T>*)bank;
    const cx<T>* src = (const cx<T>*)in;
    cx<T>* dst = (cx<T>*)out;
    EmuLds<T> lds(C::LDS);
    std::vector<Box> H(C::NT);
    const long grid = K::grid(nvol);
    for (long g = 0; g < grid; ++g) {
        long v;
        int h;
        K::task(g, v, h);
        if (v >= nvol) continue;
        lds.poison();
        emu_threads(C::NT, [&](int t) { K::xpass(t, v, h, src, lds.data(), H[t].r, bk); });
        emu_xhold_round<C, 0>(v, h, H, lds, dst, bk, (T)scl);
    }
    return hipSuccess;
}

// Compute units that launch_rounds (xrounds.hpp) plans for; tests set it.
extern int g_emu_cus;
inline int rounds_cus() { return g_emu_cus; }

template <class C>
KernelDesc xhold_desc(const char* name)
{
    return KernelDesc{C::N0, C::N1, C::N2, prec_of<typename C::T>(), C::S, kFused, 1, C::NT,
                      C::V17, 0, sizeof(cx<typename C::T>) * (size_t)C::LDS, name,
                      &launch_xhold<C>};
}

}  // namespace fx
