// Tiled fp32 GEMM for gfx950 on the bf16 matrix cores: C = op(A) op(B) (+ bias) with every
// fp32 operand value split exactly into three bf16 parts (gemm_split.h).
//
// What bounds a large product on the fp32 MFMA is its rate: 157.3 TFLOP/s, of which
// gemm_direct_kernel reaches 94-95 % at 4096^3. The bf16 MFMA is 16 times as fast, and an
// fp32 value is the sum of three bf16 values, x = h + m + l (8 significand bits each, rounded
// to nearest, so the next part carries the signed remainder; bit for bit equal to x). Six of
// the nine products of the parts are computed, into two fp32 sums per output that are added
// at the end:
//   low  += ah bl + al bh + am bm + am bh + ah bm   (the smallest first)
//   high += ah bh.
//  * What is left out (am bl, al bm, al bl) is at most (1 + 2^-10) 2^-24 |a b|, since |m| <=
//    2^-8 |x| and |l| <= 2^-17 |x| (checked over every significand), about one rounding of an
//    fp32 product; root mean square 0.1 x 2^-24 over N(0,1) pairs. It is zero where a b has no
//    more than 24 significant bits. Eight products (am bl and al bm too) leave every dense
//    error below as it is to three digits and take 755-791 us at 4096^3.
//  * The high sum is rounded twice per 16 k against 16 times on the fp32 MFMA, and only where
//    a product is not zero; the low one's roundings weigh 2^-7 as much. In one sum the high
//    product and the five others round it 12 times per 16 k, six times around a product whose
//    neighbours are zero: sparse operands then lose up to half of their accuracy.
//  * Normwise error against fp64 over the fp32 MFMA chain's (in brackets: all six in one sum),
//    K = 1009, n values of each row of A not zero. N(0,1): n = 1 1.02 (1.36), 2 0.84 (1.67), 4
//    0.68 (1.88), 16 0.47 (2.03), 256 0.36 (1.46), 512 0.35 (1.14), all 0.33 (0.86); U[0,1): 1
//    1.02 (1.25), 4 0.73 (1.74), 256 0.51 (1.33), all 0.37 (0.70). Dense N(0,1): K = 512
//    1.3e-7 / 4.1e-7, 2048 2.7e-7 / 8.1e-7, 4096 4.0e-7 / 1.15e-6. So from two products per sum
//    on the error is below the fp32 kernels'; a sum of a single product has 1.02-1.05 times
//    their error, at most 1.9 x 2^-24 of the product against 1.0. MIGEMM_TUNE_DIRECT = 2 keeps
//    every product on the fp32 MFMA.
//  * Parts cut off instead of rounded leave a one-sided error: 1.05e-5 at U[0,1), K = 4096.
//
// The kernel:
//  * A k-tile of 16 goes global memory -> registers -> split -> LDS once per work-group, so
//    the split's 13 vector instructions per pair of values are shared by every wavefront that
//    reads the tile. Its steps run between the MFMAs of the k-tile before (one step of 6-8
//    instructions behind an MFMA), and the loads of the k-tile after are issued as soon as
//    the registers are free. Two LDS stages, one barrier per k-tile.
//  * 8 wavefronts: 256x128 tiles (64x64 outputs per wavefront, one work-group per CU: 226-228
//    registers) and 128x128 (32x64, two work-groups per CU: 128). Two sums of 256x256 tiles do
//    not fit in the registers.
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
//    kernels give (such a tile costs 2.2-2.6 times an ordinary one: 4096^3 1777, in fp32 910).
//
// Measured (events around 10 launches, N(0,1) operands, us, this kernel / the fp32 choice):
// 4096^3 NN 673 / 916, NT 667 / 912, TN 692 / 916 (199-206 TFLOP/s; one sum in 256x256 tiles
// 608, 602, 624, in 256x128 tiles 670, 667, 693); 12000 x 500 x 6565 504 / 646; 6400 x 512 x
// 4096 167 / 225; 6400 x 2048 x 4096 599 / 783; 2048^3 100 / 128; 1000 x 777 x 3000 40 / 43.
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
// Estimate / measured (events around 10 launches, us): 4096^3 256x128 688 / 671, 128x128 736 /
// 711; 6400 x 2048 x 4096 683 / 641, 654 / 599; 12000 x 500 x 6565 574 / 529, 529 / 484; 2500 x
// 4096 x 2500 in 2 ranges 369 / 316, 399 / 341; 500 x 12000 x 6565 TN in 6 ranges 537 / 492,
// 492 / 465; 6400 x 4096 x 512 NT in 5 189 / 156, 192 / 161; 2048^3 128x128 98 / 98; 1000 x 777
// x 3000 128x128 43 / 41. Of 22 such products the pick was the slower tile in two, by 1 %.
constexpr SplitFit kSplitFit[2] = {{256, 128, 1.29, 1.05, 11.0}, {128, 128, 0.70, 0.58, 3.5}};
constexpr double kSplitLaunch = 5.0;        // us: start of the grid
constexpr double kSplitPartialBytes = 6e6;  // partial sums' HBM traffic, bytes per us
// C rows off 64-byte boundaries: us more per tile and CU (12000 x 500 x 6565 against x 6560:
// 128x128 508 / 486)
constexpr double kSplitOddRows[2] = {5.0, 1.2};

double split_rounds(const SplitFit &f, double t) {
    const double whole = floor(t), part = t - whole;
    if (f.bm == 128)
        return t <= 1 ? f.alone + 0.12 * t : (t <= 8 ? ceil(t) : t + 0.3) * f.full;
    return whole * f.full + (part > 0 ? f.alone + (f.full - f.alone) * part : 0.0);
}

}  // namespace

SplitPlan plan_split(const GemmDesc &d, int plan_splits) {
    SplitPlan best = {0, 0, 1, 1e300};
    // No fewer ranges than the fp32 plan has: a k-long sum's error grows as the root of its k
    // range, so this keeps the ratios above.
    const int least = plan_splits;
    const int most = plan_splits > 8 ? plan_splits : 8;
    const int nk = (d.K + SBK - 1) / SBK;
    const bool odd = d.ldc % 16 != 0 || ((uintptr_t)d.C & 63) != 0 ||
                     (d.batch > 1 && d.sC % 16 != 0);
    for (int i = 0; i < 2; ++i) {
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
    if (plan.bm == 256) return launch_split_256x128(stream, a, akc, bkc);
    return launch_split_128(stream, a, akc, bkc);
}

}  // namespace migemm
