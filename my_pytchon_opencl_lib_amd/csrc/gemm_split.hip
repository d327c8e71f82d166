// Tiled fp32 GEMM for gfx950 on the bf16 matrix cores: C = op(A) op(B) (+ bias) with every
// fp32 operand value split exactly into three bf16 parts (gemm_split.h).
//
// What bounds a large product on the fp32 MFMA is its rate: 157.3 TFLOP/s, of which
// gemm_direct_kernel reaches 94-95 % at 4096^3. The bf16 MFMA is 16 times as fast, and an
// fp32 value is the sum of three bf16 values, x = h + m + l (8 significand bits each, rounded
// to nearest, so the next part carries the signed remainder; bit for bit equal to x). Six of the nine products of the parts are computed, the smallest first, into
// one fp32 accumulator per output:
//   a b = ah bl + al bh + am bm + am bh + ah bm + ah bh;
// the three left out (am bl, al bm, al bl) are below 2^-26 of |a b|, a quarter of the
// rounding of one fp32 product. The accumulator is rounded 12 times per 16 k against 16 on
// the fp32 MFMA. Normwise error against fp64, this kernel / the fp32 MFMA chain: N(0,1)
// operands K = 256 2.4e-7 / 2.9e-7, 1024 4.9e-7 / 5.7e-7, 4096 1.00e-6 / 1.14e-6, 12000
// 1.77e-6 / 1.95e-6; U[0,1) K = 4096 5.3e-7 / 8.5e-7, 12000 1.05e-6 / 1.66e-6. (Parts cut off
// instead of rounded leave a one-sided error: 1.05e-5 at U[0,1), K = 4096.)
//
// The kernel:
//  * A k-tile of 16 goes global memory -> registers -> split -> LDS once per work-group, so
//    the split's 13 vector instructions per pair of values are shared by every wavefront that
//    reads the tile. Its steps run between the MFMAs of the k-tile before (one step of 6-8
//    instructions behind an MFMA), and the loads of the k-tile after are issued as soon as
//    the registers are free. Two LDS stages, one barrier per k-tile.
//  * 8 wavefronts (two per SIMD): 256x256 tiles (64x128 outputs per wavefront, one
//    work-group per CU), 256x128 (64x64) and 128x128 (32x64, two work-groups per CU).
//  * Loads are 16 bytes per lane for a K-contiguous operand and 4 bytes, adjacent lanes
//    adjacent rows, for an I-contiguous one; neither needs alignment, so odd leading
//    dimensions and sizes run the same code. The last k-tile of K % 16 != 0 is read from
//    k = K - 16 on with the shared k cleared.
//  * Operand values are scaled by 2^23 while they are split and the sums by 2^-46 at the end:
//    the parts of every fp32 value, subnormal ones too, are then normal bf16 numbers, and no
//    tile is computed in another way for its small values (4096^3 with one value of 1e-35 in
//    every row of A, us: tiles with values below 2^-110 a second time in fp32 1698, so 601;
//    without such values 619 and 599).
//  * Values the parts cannot carry: an infinity, a NaN or a value of 4.04e31 or more leaves
//    its outputs not finite, and so does a sum of 4.83e24 or more. A work-group that meets one
//    computes its tile once more with v_mfma_f32_32x32x2_f32, so these give what the fp32
//    kernels give (such a tile costs about 2.5 times an ordinary one).
//
// Measured (events around 10 launches, N(0,1) operands, us, this kernel / the fp32 choice):
// 4096^3 NN 650 / 910, NT 605 / 908, TN 610 / 906 (211-227 TFLOP/s); 12000 x 500 x 6565
// 487 / 640; 6400 x 512 x 4096 165 / 211; 2048^3 100 / 118; 1000 x 777 x 3000 41 / 41.
// At 4096^3 the MFMA is busy 65 % of the cycles at a clock of 1.69 GHz: the card's power
// limit sets the clock (all-zero operands run at 302 TFLOP/s), so what is left is energy per
// product, not issue slots.
#include "gemm_split.h"

#include <math.h>

namespace migemm {

namespace {

// Estimated time of `t` x 256 tiles (us per k-tile of 16, without the tiles' fixed part).
// A work-group that has its CU to itself takes `full` us per k-tile when every CU works (the
// power limit) and `alone` when few do; a last, partial round lies between. 128x128 tiles
// run two to a CU: up to 8 rounds each CU's share is a whole number of them, beyond that
// they even out.
struct SplitFit {
    int bm, bn;
    double full, alone, over;  // over: us per tile and CU for first loads, C store, launch
};
// Fitted on one box (events around 10 launches; estimate / measured, us): 4096^3 256x256
// 627 / 605-650; 6400 x 2048 x 4096 256x256 613 / 584, 128x128 653 / 611; 2048^3 128x128
// 103 / 100; 1000 x 777 x 3000 128x128 42 / 41; 500 x 12000 x 6565 TN in 6 ranges 256x128
// 505 / 488, 128x128 459 / 490, in 5 ranges 582 / 564, 547 / 534.
constexpr SplitFit kSplitFit[3] = {
    {256, 256, 2.35, 1.75, 20.0}, {256, 128, 1.29, 1.05, 11.0}, {128, 128, 0.70, 0.58, 3.5}};
constexpr double kSplitLaunch = 5.0;        // us: start of the grid
constexpr double kSplitPartialBytes = 6e6;  // partial sums' HBM traffic, bytes per us
// C rows off 64-byte boundaries: us more per tile and CU (12000 x 500 x 6565 against x 6560:
// 256x256 532 / 474, 128x128 508 / 486)
constexpr double kSplitOddRows[3] = {11.0, 5.0, 1.2};

double split_rounds(const SplitFit &f, double t) {
    const double whole = floor(t), part = t - whole;
    if (f.bn == 128 && f.bm == 128)
        return t <= 1 ? f.alone + 0.12 * t : (t <= 8 ? ceil(t) : t + 0.3) * f.full;
    return whole * f.full + (part > 0 ? f.alone + (f.full - f.alone) * part : 0.0);
}

}  // namespace

SplitPlan plan_split(const GemmDesc &d, int plan_splits) {
    SplitPlan best = {0, 0, 1, 1e300};
    // A k-long sum's error grows as the root of its k range and is 0.83-0.91 of the fp32
    // MFMA's here, so no fewer ranges than the fp32 plan has keep it no larger: the LSTM input
    // gradient 6400 x 4096 x 512 (3 ranges in fp32, 6.6e-7) has 1.0e-6 in one range, 5.8e-7 in
    // three.
    const int least = plan_splits;
    const int most = plan_splits > 8 ? plan_splits : 8;
    const int nk = (d.K + SBK - 1) / SBK;
    const bool odd = d.ldc % 16 != 0 || ((uintptr_t)d.C & 63) != 0 ||
                     (d.batch > 1 && d.sC % 16 != 0);
    for (int i = 0; i < 3; ++i) {
        const SplitFit &f = kSplitFit[i];
        const double tiles =
            (double)((d.M + f.bm - 1) / f.bm) * ((d.N + f.bn - 1) / f.bn) * d.batch;
        for (int s = least; s <= most; ++s) {
            const double partial = s > 1 ? (double)s * d.batch * d.M * d.N * 4.0 : 0.0;
            // ranges beyond the fp32 plan's only while their partial sums fit the
            // no-allocation entry's scratch, so that every entry decides alike
            if (s > plan_splits && partial > (double)MIGEMM_NOALLOC_SCRATCH_BYTES) break;
            const double ks = (double)((nk + s - 1) / s);
            if (s > 1 && ks < 16) break;
            const double t = tiles * s / 256.0;
            const double over = f.over + (odd && s == 1 ? kSplitOddRows[i] : 0.0);
            const double us = ks * split_rounds(f, t) +
                              (f.bm == 256 ? ceil(t) : fmax(t, 1.0)) * over + kSplitLaunch +
                              (s > 1 ? (2.0 * partial + 4.0 * d.batch * d.M * d.N) /
                                               kSplitPartialBytes + 4.0
                                     : 0.0);
            if (us < best.us) best = {f.bm, f.bn, s, us};
        }
    }
    return best;
}

int launch_gemm_split(hipStream_t stream, TiledArgs &a, const SplitPlan &plan, bool akc,
                      bool bkc) {
    a.splits = plan.splits;
    if (plan.bn == 256) return launch_split_256(stream, a, akc, bkc);
    if (plan.bm == 256) return launch_split_256x128(stream, a, akc, bkc);
    return launch_split_128(stream, a, akc, bkc);
}

}  // namespace migemm
