// Matrix fragments of the matrix-core kernels (mfma.hpp), made on the host at plan time in the
// order the lanes load them and uploaded behind the constant bank: per line form the high and
// low halves of every matrix tile, 64 lanes of Q values each, so that a wave fetches an operand
// with one load of 8 or 16 bytes a lane.  Deriving the entries in the kernel (a bank gather,
// index arithmetic mod N and the split, per entry and wave) cost more than the products in the
// forms that run one block per workgroup, and set the latency of small batches: the mix 6^3 x
// 65536, 8^3 x 32768, 12^3 x 8192, 17^3 x 2048 in one launch went from 190.4 to 174.1 us (bf16x3)
// and from 214.0 to 198.5 (fp16x3), 17^3 x 50 from 11.7 to 9.6, 12^3 x 144 from 6.8 to 5.4, and
// 6^3 x 200 with 12^3 x 50 and 17^3 x 30 from 12.1 to 10.1.
#pragma once
#include "cx.hpp"

namespace fx {

struct FragForm {
    int n;      // line length
    int kw;     // instruction K
    int fold;   // 17 points by the conjugate-pair fold: its P and M matrices as two tiles
};
constexpr FragForm kFragForms[] = {{6, 16, 0},  {8, 16, 0},  {12, 16, 0}, {12, 32, 0}, {16, 16, 0},
                                   {16, 32, 0}, {17, 16, 0}, {17, 32, 0}, {17, 32, 1}};
constexpr int kNumFragForms = sizeof(kFragForms) / sizeof(kFragForms[0]);

constexpr int frag_tiles_m(const FragForm& f) { return f.fold ? 2 : (2 * f.n + 15) / 16; }
constexpr int frag_tiles_k(const FragForm& f) { return f.fold ? 1 : (2 * f.n + f.kw - 1) / f.kw; }
// Bytes of one half (high or low) of one tile: 64 lanes of kw / 4 16-bit values.
constexpr int frag_half_bytes(const FragForm& f) { return 64 * (f.kw / 4) * 2; }
constexpr int frag_bytes(const FragForm& f)
{
    return frag_tiles_m(f) * frag_tiles_k(f) * 2 * frag_half_bytes(f);
}
// Offset of form (n, kw, fold) in a set; the set's size for a form that is not in the list.
constexpr int frag_off(int n, int kw, int fold)
{
    int off = 0;
    for (int k = 0; k < kNumFragForms; ++k) {
        if (kFragForms[k].n == n && kFragForms[k].kw == kw && kFragForms[k].fold == fold) return off;
        off += frag_bytes(kFragForms[k]);
    }
    return off;
}
constexpr int kFragSet = frag_off(0, 0, 0);
// One set per direction S and split (0 bf16, 1 fp16), behind the bank on a 256-byte boundary.
constexpr int kFragBase = ((int)sizeof(Bank<float>) + 255) / 256 * 256;
constexpr int frag_set(int S, int split) { return kFragBase + kFragSet * ((S > 0 ? 2 : 0) + split); }
constexpr int kFragEnd = kFragBase + 4 * kFragSet;

}  // namespace fx
