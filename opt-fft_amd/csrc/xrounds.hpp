// Residue-split launch by rounds.  A form (a residue-split kernel with R workgroups a volume)
// takes about as long for one volume as for a round of them, and as long again for the next one:
// 36^3 complex128 in two workgroups a volume takes 27.7 us for 1 volume, 41.5 for 128 (one round
// of 256 workgroups), 70.4 for 150 and 80.0 for 256.  Fewer
// volumes than a round go faster through a form with more workgroups a volume, as long as
// those run in one round themselves.  So a batch runs its full rounds in the last form of the
// list, and what remains in the first form (R descending) that holds it in one round, as a
// second launch on the same stream:
//   36^3 complex128, 2 / 4 / 6 / 12 workgroups a volume, rounds of 128 / 64 / 40 / 16 volumes:
//   16 volumes 32.1 / 22.0 / 14.8 / 13.5 us, 32 volumes 32.6 / 22.7 / 17.4 / 24.4,
//   64 volumes 34.3 / 26.7 / 33.2 / 35.7, 128 volumes 41.5 / 51.9 / 57.1 / 69.7.
// W of a form is the number of workgroups a CU that its round is counted with, where its time was
// measured to step: not its occupancy, which is higher for most (LDS alone would let two
// workgroups of 24^3 complex128 r4 share a CU, but 80 volumes take 14.4 us to the 8.9 of 64; 40
// volumes of r6 7.1 us, 56 12.4).  24^3 complex64 r1h8 steps after 512 volumes, W = 2 (22.6 us; 600
// 31.4), and the same form with linear stores is ahead from there on (23.9 and 30.0): it ends the
// list with the four workgroups that fit on a CU.
// Where the last form has several workgroups on a CU (W > 1) its rounds overlap, and a batch of
// more than one of them runs in that form alone: 24^3 complex64 x 1200 took 56.6 us in two
// launches and 55.5 in one, 24^3 complex128 x 340 35.9 and 31.5.
// A round counts per XCD: a volume's workgroups share one, volumes go to the XCDs in turn, so a
// form's round is 8 floor(CUs / 8 * W / R) volumes.
#pragma once

#include "xhold.hpp"

namespace fx {

constexpr int kXcds = 8;

// Volumes of one round of R workgroups a volume, counted with W workgroups a CU.
inline long round_volumes(int cus, int R, int W) { return (long)(cus / kXcds * W / R) * kXcds; }

template <class C_, int W_>
struct ResForm {
    using C = C_;
    static constexpr int W = W_;
    static hipError_t launch(const void* in, void* out, long nvol, const void* bank, double scl,
                             hipStream_t s)
    {
        return launch_xres<C>(in, out, nvol, bank, scl, nullptr, s);
    }
};
template <class C_, int W_>
struct HoldForm {
    using C = C_;
    static constexpr int W = W_;
    static hipError_t launch(const void* in, void* out, long nvol, const void* bank, double scl,
                             hipStream_t s)
    {
        return launch_xhold<C>(in, out, nvol, bank, scl, nullptr, s);
    }
};

// `rem` volumes in the first form that holds them in one round; the last form takes any number.
template <class F, class... Fs>
hipError_t launch_remainder(const void* in, void* out, long rem, const void* bank, double scl,
                            int cus, hipStream_t s)
{
    if constexpr (sizeof...(Fs) > 0) {
        if (rem > round_volumes(cus, F::C::R, F::W))
            return launch_remainder<Fs...>(in, out, rem, bank, scl, cus, s);
    }
    return F::launch(in, out, rem, bank, scl, s);
}

template <class... Fs>
struct LastForm;
template <class F>
struct LastForm<F> {
    using type = F;
};
template <class F, class G, class... Fs>
struct LastForm<F, G, Fs...> {
    using type = typename LastForm<G, Fs...>::type;
};

// True when the last form is the one launch_remainder would take for `rem`.
template <class F, class... Fs>
bool remainder_is_last(long rem, int cus)
{
    if constexpr (sizeof...(Fs) == 0) return true;
    else return rem > round_volumes(cus, F::C::R, F::W) && remainder_is_last<Fs...>(rem, cus);
}

template <class... Fs>
hipError_t launch_rounds(const void* in, void* out, long nvol, const void* bank, double scl,
                         unsigned*, hipStream_t s)
{
    using M = typename LastForm<Fs...>::type;
    using C = typename M::C;
    if (nvol <= 0) return hipSuccess;
    const int cus = rounds_cus();
    const long round = round_volumes(cus, C::R, M::W);
    long full = round > 0 ? nvol / round * round : nvol;
    const long rem = nvol - full;
    if (rem > 0 && ((full > 0 && M::W > 1) || remainder_is_last<Fs...>(rem, cus))) full = nvol;
    if (full > 0) {
        const hipError_t e = M::launch(in, out, full, bank, scl, s);
        if (e != hipSuccess || full == nvol) return e;
    }
    const size_t off = sizeof(cx<typename C::T>) * (size_t)C::V * (size_t)full;
    return launch_remainder<Fs...>((const char*)in + off, (char*)out + off, nvol - full, bank, scl,
                                   cus, s);
}

template <class... Fs>
KernelDesc rounds_desc(const char* name)
{
    using C = typename LastForm<Fs...>::type::C;
    return KernelDesc{C::N0, C::N1, C::N2, prec_of<typename C::T>(), C::S, kFused, 1, C::NT,
                      C::V17, 0, sizeof(cx<typename C::T>) * (size_t)C::LDS, name,
                      &launch_rounds<Fs...>};
}

}  // namespace fx
