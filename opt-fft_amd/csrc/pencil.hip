// Two-pass pencil kernels for volumes that exceed LDS at complex128 (L = 24, 36 and
// 24x24x48) and their complex64 counterparts.  Names: s<SPW> slabs per workgroup,
// t<NT> threads, b<NTB> threads of the x-line pass, c<CHUNK> volumes per launch pair
// (0 = whole batch), p<P> persistent pipelined pass A with at most P workgroups per CU,
// "_st" pass A with staggered HBM traffic (PencilCfg ST = 1).  Also the residue-split
// single-pass kernels of the same geometries (xres.hpp): "xres_..._v1r<R>t<NT>".
#include "kernels.hpp"
#include "xhold.hpp"
#include "xres.hpp"
#include "xrounds.hpp"

namespace fx {

#define FX_P(N0, N1, N2, T, S, SPW, NT, PZ, NTB, CH, PIPE, NAME) \
    r.push_back(pencil_desc<PencilCfg<N0, N1, N2, T, S, SPW, NT, PZ, NTB, CH, PIPE>>(NAME))
#define FX_P_BOTH(N0, N1, N2, T, TAG, SPW, NT, PZ, NTB, CH, PIPE)                                \
    FX_P(N0, N1, N2, T, -1, SPW, NT, PZ, NTB, CH, PIPE,                                          \
         "pencil_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_s" #SPW "t" #NT "b" #NTB "c" #CH "p" #PIPE); \
    FX_P(N0, N1, N2, T, +1, SPW, NT, PZ, NTB, CH, PIPE,                                          \
         "pencil_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_s" #SPW "t" #NT "b" #NTB "c" #CH "p" #PIPE)

#define FX_PS(N0, N1, N2, T, S, SPW, NT, PZ, NTB, CH, PIPE, NAME) \
    r.push_back(pencil_desc<PencilCfg<N0, N1, N2, T, S, SPW, NT, PZ, NTB, CH, PIPE, 1>>(NAME))
#define FX_PS_BOTH(N0, N1, N2, T, TAG, SPW, NT, PZ, NTB, CH, PIPE)                                \
    FX_PS(N0, N1, N2, T, -1, SPW, NT, PZ, NTB, CH, PIPE,                                          \
         "pencil_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_s" #SPW "t" #NT "b" #NTB "c" #CH "p" #PIPE "_st"); \
    FX_PS(N0, N1, N2, T, +1, SPW, NT, PZ, NTB, CH, PIPE,                                          \
         "pencil_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_s" #SPW "t" #NT "b" #NTB "c" #CH "p" #PIPE "_st")

// Radix order ("_r1": the line factors in the other order, PencilCfg ALG = 1).
#define FX_PR(N0, N1, N2, T, S, SPW, NT, PZ, NTB, CH, PIPE, ST, NAME) \
    r.push_back(pencil_desc<PencilCfg<N0, N1, N2, T, S, SPW, NT, PZ, NTB, CH, PIPE, ST, 1>>(NAME))
#define FX_PR_BOTH(N0, N1, N2, T, TAG, SPW, NT, PZ, NTB, CH, PIPE, ST, SUF)                      \
    FX_PR(N0, N1, N2, T, -1, SPW, NT, PZ, NTB, CH, PIPE, ST,                                      \
          "pencil_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_s" #SPW "t" #NT "b" #NTB "c" #CH "p" #PIPE SUF "_r1"); \
    FX_PR(N0, N1, N2, T, +1, SPW, NT, PZ, NTB, CH, PIPE, ST,                                      \
          "pencil_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_s" #SPW "t" #NT "b" #NTB "c" #CH "p" #PIPE SUF "_r1")

// Residue-split single pass (xres.hpp): "xres_<shape>_<prec>_<dir>_v1r<R>t<NT>", R workgroups
// per volume, each holding N0 / R x-planes in LDS; PF groups of loads in flight.
#define FX_X(N0, N1, N2, T, S, R, NT, OR, PF, NAME) \
    r.push_back(xres_desc<XResCfg<N0, N1, N2, T, S, R, NT, OR, PF>>(NAME))
#define FX_X_BOTH(N0, N1, N2, T, TAG, R, NT, PF)                                                  \
    FX_X(N0, N1, N2, T, -1, R, NT, 0, PF, "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_v1r" #R "t" #NT); \
    FX_X(N0, N1, N2, T, +1, R, NT, 0, PF, "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_v1r" #R "t" #NT)
// "o<OR>": the x pass's point order (XResCfg OR: 1 rotated thread blocks, 2 offset starts).
#define FX_XO_BOTH(N0, N1, N2, T, TAG, R, NT, OR, PF)                                           \
    FX_X(N0, N1, N2, T, -1, R, NT, OR, PF,                                                      \
         "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_v1r" #R "t" #NT "o" #OR);                   \
    FX_X(N0, N1, N2, T, +1, R, NT, OR, PF,                                                      \
         "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_v1r" #R "t" #NT "o" #OR)
// The same with most of the planes in registers (xhold.hpp): "...h<PR>", PR planes in LDS at a
// time, PF groups of GS loads in flight.
#define FX_XH(N0, N1, N2, T, S, R, NT, PR, GS, PF, NAME) \
    r.push_back(xhold_desc<XHoldCfg<N0, N1, N2, T, S, R, NT, PR, GS, PF>>(NAME))
#define FX_XH_BOTH(N0, N1, N2, T, TAG, R, NT, PR, GS, PF)                                        \
    FX_XH(N0, N1, N2, T, -1, R, NT, PR, GS, PF,                                                  \
          "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_v1r" #R "t" #NT "h" #PR);                    \
    FX_XH(N0, N1, N2, T, +1, R, NT, PR, GS, PF,                                                  \
          "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_v1r" #R "t" #NT "h" #PR)

// "...h<PR>l": stored by a copy of 16 bytes a lane out of LDS (XHoldCfg LIN).
#define FX_XHL(N0, N1, N2, T, S, R, NT, PR, GS, PF, NAME) \
    r.push_back(xhold_desc<XHoldCfg<N0, N1, N2, T, S, R, NT, PR, GS, PF, 1>>(NAME))
#define FX_XHL_BOTH(N0, N1, N2, T, TAG, R, NT, PR, GS, PF)                                       \
    FX_XHL(N0, N1, N2, T, -1, R, NT, PR, GS, PF,                                                 \
           "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_v1r" #R "t" #NT "h" #PR "l");               \
    FX_XHL(N0, N1, N2, T, +1, R, NT, PR, GS, PF,                                                 \
           "xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_v1r" #R "t" #NT "h" #PR "l")

// Launches by rounds (xrounds.hpp): forms with R descending, the last one for full rounds.
#define FX_R_BOTH(N0, N1, N2, TAG, FORMS)                                                        \
    r.push_back(rounds_desc<FORMS(-1)>("xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_fwd_v1rounds"));    \
    r.push_back(rounds_desc<FORMS(+1)>("xres_" #N0 "x" #N1 "x" #N2 "_" TAG "_bwd_v1rounds"))
#define FX_R36D(S)                                                                               \
    ResForm<XResCfg<36, 36, 36, double, S, 12, 256, 1, 4>, 1>,                                   \
        ResForm<XResCfg<36, 36, 36, double, S, 6, 512, 2, 4>, 1>,                                \
        HoldForm<XHoldCfg<36, 36, 36, double, S, 4, 448, 6, 9, 2>, 1>,                           \
        HoldForm<XHoldCfg<36, 36, 36, double, S, 2, 256, 6, 9, 3>, 1>
#define FX_R48D(S)                                                                               \
    ResForm<XResCfg<24, 24, 48, double, S, 8, 256, 1, 4>, 1>,                                    \
        ResForm<XResCfg<24, 24, 48, double, S, 4, 384, 1, 2>, 1>,                                \
        HoldForm<XHoldCfg<24, 24, 48, double, S, 2, 256, 8, 6, 4>, 1>
#define FX_R24D(S)                                                                               \
    ResForm<XResCfg<24, 24, 24, double, S, 6, 192, 0, 4>, 1>,                                    \
        ResForm<XResCfg<24, 24, 24, double, S, 4, 192, 0, 4>, 1>,                                \
        ResForm<XResCfg<24, 24, 24, double, S, 3, 256, 1, 3>, 2>
#define FX_R36F(S)                                                                               \
    ResForm<XResCfg<36, 36, 36, float, S, 12, 256, 1, 4>, 1>,                                    \
        ResForm<XResCfg<36, 36, 36, float, S, 6, 448, 2, 4>, 1>,                                 \
        ResForm<XResCfg<36, 36, 36, float, S, 3, 512, 2, 2>, 1>,                                 \
        HoldForm<XHoldCfg<36, 36, 36, float, S, 2, 448, 9, 9, 3, 1>, 1>,                         \
        HoldForm<XHoldCfg<36, 36, 36, float, S, 1, 448, 12, 9, 4, 1>, 1>
#define FX_R48F(S)                                                                               \
    ResForm<XResCfg<24, 24, 48, float, S, 6, 192, 0, 4>, 1>,                                     \
        ResForm<XResCfg<24, 24, 48, float, S, 3, 256, 0, 3>, 1>,                                 \
        ResForm<XResCfg<24, 24, 48, float, S, 2, 384, 0, 3>, 1>,                                 \
        HoldForm<XHoldCfg<24, 24, 48, float, S, 1, 384, 12, 6, 4>, 1>
#define FX_R24F(S)                                                                               \
    ResForm<XResCfg<24, 24, 24, float, S, 6, 192, 0, 6>, 1>,                                     \
        ResForm<XResCfg<24, 24, 24, float, S, 3, 192, 0, 4>, 1>,                                 \
        ResForm<XResCfg<24, 24, 24, float, S, 2, 320, 0, 2>, 1>,                                 \
        HoldForm<XHoldCfg<24, 24, 24, float, S, 1, 192, 8, 6, 4>, 2>,                            \
        HoldForm<XHoldCfg<24, 24, 24, float, S, 1, 192, 8, 6, 4, 1>, 4>

// (Pass B with plain stores, PencilCfg XH = 1, measured 8% slower at 36^3 x 128 and 1% at
// 24x24x48 x 64 than with nontemporal ones: not registered.)

void register_pencil(std::vector<KernelDesc>& r)
{
    // L = 36: slab 36x36 = 20.7 KB complex128.  The race keeps an earlier variant unless a
    // later one is 1.5% and 0.1 us faster: at batch 128 s7t256p1 staggered (71 us), then unstaggered
    // (73 us), ahead of s3t128p2 (73-74 us).
    FX_PS_BOTH(36, 36, 36, double, "c128", 7, 256, 1, 128, 0, 1);
    FX_P_BOTH(36, 36, 36, double, "c128", 7, 256, 1, 128, 0, 1);
    FX_P_BOTH(36, 36, 36, double, "c128", 3, 128, 1, 128, 0, 2);
    FX_P_BOTH(36, 36, 36, double, "c128", 3, 128, 1, 128, 0, 0);
    FX_P_BOTH(36, 36, 36, double, "c128", 7, 256, 1, 128, 0, 0);
    FX_PR_BOTH(36, 36, 36, double, "c128", 7, 256, 1, 128, 0, 1, 1, "_st");
    FX_P_BOTH(36, 36, 36, float, "c64", 7, 256, 1, 128, 0, 1);
    FX_P_BOTH(36, 36, 36, float, "c64", 3, 128, 1, 128, 0, 4);
    // L = 24: slab 24x24 = 9.2 KB complex128.
    FX_P_BOTH(24, 24, 24, double, "c128", 8, 192, 1, 128, 0, 2);
    FX_P_BOTH(24, 24, 24, double, "c128", 8, 192, 1, 128, 0, 0);
    FX_P_BOTH(24, 24, 24, double, "c128", 16, 384, 1, 128, 0, 0);
    FX_P_BOTH(24, 24, 24, float, "c64", 16, 384, 1, 128, 0, 2);
    FX_P_BOTH(24, 24, 24, float, "c64", 16, 384, 1, 128, 0, 0);
    // 24 x 24 x 48: slab 24x48 = 18.4 KB complex128; z lines 48-point, y and x 24-point.
    // Two slabs per 128-thread block first (768 blocks at batch 64, ~3 resident per CU, so
    // blocks in different phases overlap): 26.6 us against 27.9 us for four slabs.
    FX_P_BOTH(24, 24, 48, double, "c128", 2, 128, 1, 128, 0, 0);
    FX_P_BOTH(24, 24, 48, double, "c128", 4, 128, 1, 128, 0, 0);
    FX_P_BOTH(24, 24, 48, double, "c128", 8, 256, 1, 128, 0, 0);
    FX_PR_BOTH(24, 24, 48, double, "c128", 2, 128, 1, 128, 0, 0, 0, "");
    FX_PR_BOTH(24, 24, 24, double, "c128", 8, 192, 1, 128, 0, 2, 0, "");
    FX_P_BOTH(24, 24, 48, float, "c64", 8, 384, 1, 128, 0, 2);
    FX_P_BOTH(24, 24, 48, float, "c64", 8, 256, 1, 128, 0, 0);
    // Residue-split single pass (forced by name, over 1 GB of buffers in turn).  24x24x48 x 64: r4
    // (112.9 KB) 16.6-16.8 us with 384 threads, 17.2 with 256, r8 18.8, against 22.5 us for the best
    // pencil; 24^3 x 512: r3 (76.8 KB, two per CU) 45.6 us with 256 threads, 46.2 with 192, r4 52.6,
    // against 53.2 us for the split-resident kernel; x 64 r4 8.9, r3 9.1 against 15.7 us for the
    // pencil, x 8 r6 6.0, r4 6.6, r3 7.0.  36^3 x 128: r6 (127.9 KB, one workgroup per CU) 55.6 us,
    // r12 (63.9 KB, 12 reads of every element from L2) 68.4, against 67.0 us for the best pencil
    // and 40.3 with held planes (xhold.hpp).  Thread counts keep every variant within its VGPR
    // budget without scratch (a 48-point complex128 line takes ~200 VGPRs).  Point order
    // of the x pass: 36^3 x 128 r6 57.4 us with offset starts (o2), 55.6 with rotated
    // blocks (o1), 64.0 from point 0, x 1024 426 / 417 / 468; 36^3 complex64 x 64 r3 19.6 (o2) against
    // 20.0; 24x24x48 x 64 16.9 / 16.6 / 16.8; 24^3 x 512 47.2 (o1) against 45.6, but x 64 9.2 both.
    // Not kept, before the x pass was pipelined (xres.hpp): a persistent form at 36^3 that computes
    // the next task's x pass into registers during the
    // LDS passes (256 threads, 486 VGPRs) ran at 165 us: at that register pressure its loads
    // were issued one or two at a time, and issuing them together spilled.  A second form
    // (512 threads, 169 VGPRs: two-stage 4 x 9 line passes, loads six at a time, offset
    // starts) ran without scratch but took 69.8 us at x 128 and 251.4 at x 512 against 57.0 /
    // 225.3 us for the one-task form.
    // By rounds, ahead of the single forms so that a plan that ties takes the launch that also
    // fits its smaller executes (single form -> by rounds, us):
    //   36^3              x 1 27.7 -> 11.3, x 64 34.2 -> 26.4, x 150 70.0 -> 57.0, x 258 107 -> 92
    //   24x24x48          x 1 16.5 -> 8.6, x 64 20.5 -> 16.3, x 150 42.8 -> 35.4
    //   36^3 complex64    x 1 27.1 -> 10.4, x 64 30.8 -> 19.4, x 300 68.3 -> 56.7
    //   24x24x48 complex64 x 1 15.4 -> 7.9, x 128 18.4 -> 14.9, x 300 40.4 -> 35.9
    //   24^3 complex64    x 1 9.2 (LDS-resident) -> 5.0, x 85 10.3 -> 8.0, x 1024 53.4 -> 44.0
    // 24^3 complex128 ends in r3: r2h8 is 3% faster at x 256 and 5% at x 192, and 11% slower
    // at x 400.
    FX_R_BOTH(36, 36, 36, "c128", FX_R36D);
    FX_R_BOTH(24, 24, 48, "c128", FX_R48D);
    FX_R_BOTH(24, 24, 24, "c128", FX_R24D);
    FX_R_BOTH(36, 36, 36, "c64", FX_R36F);
    FX_R_BOTH(24, 24, 48, "c64", FX_R48F);
    FX_R_BOTH(24, 24, 24, "c64", FX_R24F);
    FX_XO_BOTH(36, 36, 36, double, "c128", 6, 512, 2, 4);
    FX_XO_BOTH(36, 36, 36, double, "c128", 6, 512, 1, 4);
    FX_X_BOTH(36, 36, 36, double, "c128", 6, 512, 4);
    FX_X_BOTH(36, 36, 36, double, "c128", 6, 256, 4);
    FX_XO_BOTH(24, 24, 48, double, "c128", 4, 384, 1, 2);
    FX_XO_BOTH(24, 24, 48, double, "c128", 4, 384, 2, 2);
    FX_X_BOTH(24, 24, 48, double, "c128", 4, 384, 2);
    FX_X_BOTH(24, 24, 48, double, "c128", 4, 256, 2);
    FX_XO_BOTH(24, 24, 24, double, "c128", 3, 256, 1, 3);
    FX_X_BOTH(24, 24, 24, double, "c128", 3, 256, 3);
    FX_X_BOTH(24, 24, 24, double, "c128", 3, 192, 4);
    FX_X_BOTH(24, 24, 24, double, "c128", 4, 192, 4);
    FX_X_BOTH(24, 24, 24, double, "c128", 6, 192, 4);
    // complex64: 24x24x48 x 256 r2 (12 planes, 112.9 KB) 28.8 us and r3 31.6 us against 42.0 us
    // for the best pencil (x 64: 12.6 / 14.0 against 17.1 us); 36^3 x 512 r3 125.7 us against
    // 94.0 us for the split-resident kernel (r4 161.3, r6 134.6), but at x 64 r3 20.5 against
    // 21.6 us for the pencil.
    // Small batches, where a workgroup's x pass (all of its volume from L2, at up to 108 GB/s a
    // CU) and its line passes are latencies in a row: more residues shorten the line passes.
    // 36^3 x 5 r12 11.4 us (r9 12.1, r6 12.8, pencil 11.9), x 16 13.4 against 15.6 (pencil);
    // 24x24x48 x 8 r8 8.8 us (r4 10.5, pencil 10.0), x 32 11.2 against 13.0 (r4).
    FX_XO_BOTH(36, 36, 36, double, "c128", 12, 256, 1, 4);
    FX_XO_BOTH(24, 24, 48, double, "c128", 8, 256, 1, 4);
    FX_X_BOTH(24, 24, 48, float, "c64", 2, 384, 3);
    FX_X_BOTH(24, 24, 48, float, "c64", 3, 256, 3);
    FX_XO_BOTH(36, 36, 36, float, "c64", 3, 512, 2, 2);
    FX_X_BOTH(36, 36, 36, float, "c64", 3, 512, 2);
    // Small batches again: 36^3 complex64 x 8 r12 10.7 us (r6 11.2, pencil 11.5), x 32 r6 13.7
    // (r3 15.9); 24x24x48 complex64 x 9 r6 8.2 (r3 9.6), x 32 10.3 (11.2).  24^3 complex64
    // against the LDS-resident kernel (one 576-thread workgroup a volume, one per CU): x 18
    // r6 5.4 against 9.8 us, x 90 r2 8.1 against 10.3, x 300 r3 18.9 against 22.5; x 180, one
    // volume for most CUs, 12.9 against 11.4.
    FX_XO_BOTH(36, 36, 36, float, "c64", 6, 448, 2, 4);
    FX_XO_BOTH(36, 36, 36, float, "c64", 12, 256, 1, 4);
    FX_X_BOTH(24, 24, 48, float, "c64", 6, 192, 4);
    FX_X_BOTH(24, 24, 24, float, "c64", 2, 320, 2);
    FX_X_BOTH(24, 24, 24, float, "c64", 3, 192, 4);
    FX_X_BOTH(24, 24, 24, float, "c64", 6, 192, 6);
    FX_XH_BOTH(36, 36, 36, double, "c128", 2, 256, 6, 9, 3);
    FX_XH_BOTH(36, 36, 36, double, "c128", 4, 448, 6, 9, 2);
    FX_XH_BOTH(24, 24, 48, double, "c128", 2, 256, 8, 6, 4);
    FX_XH_BOTH(24, 24, 24, double, "c128", 2, 256, 8, 6, 4);
    FX_XH_BOTH(24, 24, 48, float, "c64", 1, 384, 12, 6, 4);
    FX_XH_BOTH(24, 24, 24, float, "c64", 1, 192, 8, 6, 4);
    FX_XHL_BOTH(24, 24, 24, float, "c64", 1, 192, 8, 6, 4);
    FX_XHL_BOTH(36, 36, 36, float, "c64", 1, 448, 12, 9, 4);
    // 256 threads, 6 planes in LDS and 12 held: ahead of the other single forms at 36^3 complex64 x
    // 300-384 (66.8-68.4 us; r1h12l 69.2-72.2, r2h9l 70.2-73.6) and nowhere the quickest, since the
    // rounds take 58.4-66.5 there; between 40 and 256 volumes r2h9l or r1h12l is 10% ahead.
    FX_XHL_BOTH(36, 36, 36, float, "c64", 2, 256, 6, 9, 4);
    FX_XHL_BOTH(36, 36, 36, float, "c64", 2, 448, 9, 9, 3);
}

}  // namespace fx
