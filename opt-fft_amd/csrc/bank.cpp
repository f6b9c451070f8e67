// Plan-time constant bank, computed on the host in long double (no device calls here).
//   * W_N^m = exp(-2 pi i m/N) for every line length in kLens, with the quarter-turn
//     entries written exactly;
//   * the Rader-17 spectra Bhat = DFT16(b')/16, b'[q] = W17^(3^-q mod 17), for both
//     directions (bench/geom/strategies/L17_rader.md:21-55), with Bhat[0] = -1/16 and
//     Bhat[8] = sqrt(17)/16 written in closed form;
//   * cos and sin of 2 pi m/17 for the folded-dense 17-point line;
//   * behind it, for plans of the matrix-core kernels, their matrix fragments (mfma_frag.hpp).
#include <cmath>
#include <cstring>
#include <vector>

#include "cx.hpp"
#include "mfma_frag.hpp"
#include "plan_internal.hpp"
#include "registry.hpp"

namespace fx {

typedef long double ld;
static const ld kTwoPi = 6.283185307179586476925286766559005768L;

template <typename T>
static void build_bank(Bank<T>& b)
{
    std::memset(&b, 0, sizeof b);
    for (int k = 0; k < kNumLens; ++k) {
        const int n = kLens[k], off = woff(n);
        for (int m = 0; m < n; ++m) {
            ld c, s;
            if (m == 0) { c = 1; s = 0; }
            else if (4 * m == n) { c = 0; s = -1; }
            else if (2 * m == n) { c = -1; s = 0; }
            else if (4 * m == 3 * n) { c = 0; s = 1; }
            else { const ld a = kTwoPi * (ld)m / (ld)n; c = cosl(a); s = -sinl(a); }
            b.w[off + m].r = (T)c;
            b.w[off + m].i = (T)s;
        }
    }
    // Rader-17 spectra.  perm[u] = 3^u mod 17; b'[q] = W17^(3^-q mod 17), 3^-1 = 6 mod 17.
    for (int d = 0; d < 2; ++d) {
        const ld sign = d == 0 ? -1.0L : 1.0L;
        ld br[16], bi[16];
        int p = 1;
        for (int q = 0; q < 16; ++q) {
            const ld a = kTwoPi * (ld)p / 17.0L;
            br[q] = cosl(a);
            bi[q] = sign * sinl(a);
            p = (p * 6) % 17;
        }
        for (int s = 0; s < 16; ++s) {
            ld ar = 0, ai = 0;
            for (int q = 0; q < 16; ++q) {
                const int m = (s * q) % 16;
                const ld c = cosl(kTwoPi * (ld)m / 16.0L), sn = -sinl(kTwoPi * (ld)m / 16.0L);
                ar += br[q] * c - bi[q] * sn;
                ai += br[q] * sn + bi[q] * c;
            }
            b.rader17[d][s].r = (T)(ar / 16.0L);
            b.rader17[d][s].i = (T)(ai / 16.0L);
        }
        // Closed forms: the 16 nontrivial 17th roots sum to -1; index 8 is the quadratic
        // Gauss sum, real and equal to sqrt(17) for p = 1 mod 4, in either direction.
        b.rader17[d][0].r = (T)(-1.0L / 16.0L);
        b.rader17[d][0].i = (T)0;
        b.rader17[d][8].r = (T)(sqrtl(17.0L) / 16.0L);
        b.rader17[d][8].i = (T)0;
    }
    for (int m = 0; m < 17; ++m) {
        const ld a = kTwoPi * (ld)m / 17.0L;
        b.cos17[m] = (T)cosl(a);
        b.sin17[m] = (T)sinl(a);
    }
}

void bank_host_image(int prec, std::vector<unsigned char>& img)
{
    if (prec == kC128) {
        Bank<double> b;
        build_bank(b);
        img.assign((unsigned char*)&b, (unsigned char*)&b + sizeof b);
    } else {
        Bank<float> b;
        build_bank(b);
        img.assign((unsigned char*)&b, (unsigned char*)&b + sizeof b);
    }
}

// ------------------------------------------------- matrix fragments (mfma_frag.hpp)
// A float rounded to nearest even to bf16 (split 0) or fp16 (1, subnormals kept), |x| <= 1.
static uint16_t half_bits(float x, int split)
{
    uint32_t u;
    std::memcpy(&u, &x, 4);
    if (split == 0) return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
    const uint32_t sign = (u >> 16) & 0x8000u;
    const float a = std::fabs(x);
    if (a < 0x1p-14f) return (uint16_t)(sign | (uint32_t)std::nearbyint(a * 0x1p24f));
    u &= 0x7FFFFFFFu;
    return (uint16_t)(sign | ((u + 0xFFFu + ((u >> 13) & 1u) - (112u << 23)) >> 13));
}
static float half_value(uint16_t h, int split)
{
    if (split == 0) {
        const uint32_t u = (uint32_t)h << 16;
        float x;
        std::memcpy(&x, &u, 4);
        return x;
    }
    const int e = (h >> 10) & 31, m = h & 0x3FF;
    const float a = e ? std::ldexp((float)(1024 + m), e - 25) : std::ldexp((float)m, -24);
    return (h & 0x8000) ? -a : a;
}

// A[m][k] of the real block matrix of an n-point line, rows and columns interleaved (re, im)
// per point; zero past 2n.
static float dft_entry(const Bank<float>& b, int n, int S, int m, int k)
{
    const int o = m >> 1, j = k >> 1;
    if (o >= n || j >= n) return 0.f;
    const cx<float> w = b.w[woff(n) + (o * j) % n];
    const float wr = w.r, wi = S < 0 ? w.i : -w.i;
    if ((m & 1) == 0) return (k & 1) == 0 ? wr : -wi;
    return (k & 1) == 0 ? wi : wr;
}
// Fold form: row m (output point m/2 + 1, re/im), column c (a or b of point (c % 16)/2 + 1,
// re/im) of the P (minus = 0) or M matrix.
static float fold_entry(const Bank<float>& b, int S, int m, int c, int minus)
{
    const int k = m / 2 + 1, j = (c % 16) / 2 + 1;
    const cx<float> w = b.w[woff(17) + (j * k) % 17];   // exp(-2 pi i jk/17)
    const float cs = w.r, sn = (S < 0 ? w.i : -w.i) * (minus ? -1.f : 1.f);   // S sin
    const bool re_out = (m & 1) == 0, re_in = (c & 1) == 0;
    if (c < 16) return re_out == re_in ? cs : 0.f;          // a_j c
    if (re_out) return re_in ? 0.f : -sn;                    // Re(i b s) = -Im(b) s
    return re_in ? sn : 0.f;                                 // Im(i b s) =  Re(b) s
}

static std::vector<unsigned char> build_frags()
{
    Bank<float> b;
    build_bank(b);
    std::vector<unsigned char> img(kFragEnd, 0);
    std::memcpy(img.data(), &b, sizeof b);
    for (int S = -1; S <= 1; S += 2)
        for (int split = 0; split < 2; ++split)
            for (const FragForm& f : kFragForms) {
                unsigned char* p = img.data() + frag_set(S, split) + frag_off(f.n, f.kw, f.fold);
                const int Q = f.kw / 4;
                for (int mt = 0; mt < frag_tiles_m(f); ++mt)
                    for (int kt = 0; kt < frag_tiles_k(f); ++kt, p += 2 * frag_half_bytes(f))
                        for (int lane = 0; lane < 64; ++lane)
                            for (int q = 0; q < Q; ++q) {
                                const int r = lane % 16, c = f.kw * kt + Q * (lane / 16) + q;
                                const float a = f.fold ? fold_entry(b, S, r, c, mt)
                                                       : dft_entry(b, f.n, S, 16 * mt + r, c);
                                const uint16_t hi = half_bits(a, split);
                                const uint16_t lo = half_bits(a - half_value(hi, split), split);
                                std::memcpy(p + 2 * (lane * Q + q), &hi, 2);
                                std::memcpy(p + frag_half_bytes(f) + 2 * (lane * Q + q), &lo, 2);
                            }
            }
    return img;
}

void bank_device_image(int prec, int algo, std::vector<unsigned char>& img)
{
    if (algo == 0 || prec != kC64) {
        bank_host_image(prec, img);
        return;
    }
    static const std::vector<unsigned char> all = build_frags();
    img = all;
}

size_t elem_bytes(int prec) { return prec == kC128 ? 16 : 8; }

}  // namespace fx
