// Kernel template and launch helpers of gemm_split_kernel, shared by the translation units
// that instantiate it per tile shape (gemm_split.hip describes the kernel and holds the rule
// that picks it).
#pragma once

#include <utility>

#include "tiled_common.h"

namespace migemm {

// Per tile shape: launches gemm_split_kernel for the operand layouts (akc, bkc).
int launch_split_256x128(hipStream_t stream, TiledArgs &a, bool akc, bool bkc);
int launch_split_128(hipStream_t stream, TiledArgs &a, bool akc, bool bkc);

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int SBK = 16;  // k per k-tile: one 32x32x16 MFMA step

// Operand values are scaled by 2^23 before they are split, and the sums by 2^-46 after the k
// loop, both exact: a multiple of fp32's least subnormal 2^-149 becomes one of 2^-126, so that
// every part of every value is a normal bf16 number or zero.
constexpr float kSplitScale = 0x1p+23f;
constexpr float kSplitUnscale = 0x1p-46f;

template <typename F, int... I>
__device__ __forceinline__ void unroll_impl(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
// f(0), f(1), ... f(N - 1), each index a compile-time constant.
template <int N, typename F>
__device__ __forceinline__ void unroll(F f) {
    unroll_impl(f, std::make_integer_sequence<int, N>{});
}

// LDS layout of one k-tile of an operand of T rows: three planes (high, mid, low) of two
// chunks of 8 k; a chunk holds its 8 bf16 of every row, 16 bytes a row. A fragment read of 16
// lanes covers 256 contiguous bytes. The chunks of a plane are 128 bytes off a multiple of
// 256, so that the lanes of a row, which write both chunks at once, fall on different banks.
template <int T>
struct SplitLds {
    static constexpr int CHUNK = T * 4 + 32;  // dwords
    static constexpr int PLANE = 2 * CHUNK;
    static constexpr int STAGE = 3 * PLANE;
};

// One operand of a T-row x 16-k tile, fetched into registers by NT threads: a thread holds
// E (8 or 4) consecutive k of one row. K-contiguous (KC): the 16 / E lanes of a row read its
// 64 bytes of the k-tile. I-contiguous: the lanes read adjacent rows, one k-row at a time.
// Loads address memory as a wave-uniform base plus a 32-bit byte offset per lane (the
// launcher checks that it fits). Rows beyond the operand read the last one; their outputs
// are not stored. The last k-tile of an operand with K % 16 != 0 is fetched from k = K - 16
// on, and the k that the tile before it holds are set to zero: every load is whole and in
// bounds (K >= 16).
template <int NT, bool KC, int T>
struct SplitOperand {
    static constexpr int E = T * SBK / NT;  // consecutive k per thread
    static constexpr int LPR = SBK / E;     // lanes per row
    static_assert((E == 8 || E == 4) && E * NT == T * SBK, "one row per thread");
    float v[E];
    const char *base;    // wave-uniform: element (i0, k 0)
    int64_t ld;
    uint32_t voff;       // this lane's byte offset from `base` at k-tile 0
    int row;             // row of the tile this thread holds
    int k0;              // its first k of the k-tile

    __device__ __forceinline__ void init(const float *op, int64_t ld_, int i0, int extent,
                                         int tid) {
        ld = ld_;
        base = reinterpret_cast<const char *>(op + (KC ? (int64_t)i0 * ld : (int64_t)i0));
        row = KC ? tid / LPR : tid % T;
        k0 = E * (KC ? tid % LPR : tid / T);
        const uint32_t r = (uint32_t)min(row, extent - i0 - 1);
        voff = (KC ? r * (uint32_t)ld + k0 : (uint32_t)k0 * (uint32_t)ld + r) * 4;
    }

    // The 16 k from kt on, all below K.
    __device__ __forceinline__ void fetch(int kt) {
        if constexpr (KC) {
            const char *tb = base + (int64_t)kt * 4;
#pragma unroll
            for (int q = 0; q < E; q += 4) __builtin_memcpy(&v[q], tb + voff + 4 * q, 16);
        } else {
            const char *tb = base + (int64_t)kt * ld * 4;
#pragma unroll
            for (int k = 0; k < E; ++k)
                v[k] = *reinterpret_cast<const float *>(tb + (int64_t)k * ld * 4 + voff);
        }
    }

    // Clears the first `dup` k of a fetched k-tile, which the tile before it holds.
    __device__ __forceinline__ void drop(int dup) {
#pragma unroll
        for (int k = 0; k < E; ++k) v[k] = k0 + k >= dup ? v[k] : 0.f;
    }

    // Splitting and storing the k-tile in STEPS steps, two for each pair of values: a value x
    // becomes high + mid + low, each a bf16 rounded to nearest, which is x (scaled) bit for bit
    // below bf16's rounding overflow (|x| < 4.04e31): 24 significand bits in three of 8 bits.
    // The last step stores the three parts into `stage`. As volatile assembly the steps stay
    // where the k loop places them, between MFMAs; as ordinary code the compiler gathers them
    // in one stretch under no MFMA. A step scales one value of the next pair: scaled in the
    // step that splits them, they lengthen its chain (4096^3 NN / NT / TN 616 / 624 / 624 us,
    // this way 603 / 597 / 606).
    static constexpr int STEPS = E;
    typedef uint32_t Part __attribute__((ext_vector_type(E / 2)));
    Part h, m, l;
    static __device__ __forceinline__ void scale(float &x) {
        asm volatile("v_mul_f32 %0, %1, %0" : "+v"(x) : "s"(kSplitScale));
    }
    template <int S>
    __device__ __forceinline__ void split_step(uint32_t *stage) {
        constexpr int q = S / 2;
        uint32_t t0, t1;
        if constexpr (S % 2 == 0) {
            uint32_t a;
            if constexpr (S == 0) {
                scale(v[0]);
                scale(v[1]);
            }
            asm volatile(
                "v_cvt_pk_bf16_f32 %[a], %[x0], %[x1]\n\t"
                "v_lshlrev_b32 %[t0], 16, %[a]\n\t"
                "v_and_b32 %[t1], 0xffff0000, %[a]\n\t"
                "v_sub_f32 %[x0], %[x0], %[t0]\n\t"
                "v_sub_f32 %[x1], %[x1], %[t1]"
                : [a] "=&v"(a), [t0] "=&v"(t0), [t1] "=&v"(t1), [x0] "+v"(v[2 * q]),
                  [x1] "+v"(v[2 * q + 1]));
            if constexpr (S + 2 < STEPS) scale(v[2 * q + 2]);
            h[q] = a;
        } else {
            uint32_t b, c;
            asm volatile(
                "v_cvt_pk_bf16_f32 %[b], %[x0], %[x1]\n\t"
                "v_lshlrev_b32 %[t0], 16, %[b]\n\t"
                "v_and_b32 %[t1], 0xffff0000, %[b]\n\t"
                "v_sub_f32 %[x0], %[x0], %[t0]\n\t"
                "v_sub_f32 %[x1], %[x1], %[t1]\n\t"
                "v_cvt_pk_bf16_f32 %[c], %[x0], %[x1]"
                : [b] "=&v"(b), [c] "=&v"(c), [t0] "=&v"(t0), [t1] "=&v"(t1),
                  [x0] "+v"(v[2 * q]), [x1] "+v"(v[2 * q + 1]));
            if constexpr (S + 1 < STEPS) scale(v[2 * q + 3]);
            m[q] = b;
            l[q] = c;
        }
        if constexpr (S == STEPS - 1) {
            typedef SplitLds<T> L;
            uint32_t *o = stage + (k0 >> 3) * L::CHUNK + row * 4 + (k0 & 7) / 2;
            *reinterpret_cast<Part *>(o) = h;
            *reinterpret_cast<Part *>(o + L::PLANE) = m;
            *reinterpret_cast<Part *>(o + 2 * L::PLANE) = l;
        }
    }

    // The fp32 values into `stage`: [4 k][row].
    __device__ __forceinline__ void put_f32(float *stage) {
#pragma unroll
        for (int q = 0; q < E; q += 4)
            *reinterpret_cast<f4 *>(stage + ((k0 + q) / 4 * T + row) * 4) =
                f4{v[q], v[q + 1], v[q + 2], v[q + 3]};
    }
};

template <int BM, int BN, int WM, int WN, bool AKC, bool BKC>
__global__ void __launch_bounds__(WM *WN * 64)
    __attribute__((amdgpu_waves_per_eu(BM * BN <= 128 * 128 ? 4 : 2)))  // work-groups per CU: 2, 1
gemm_split_kernel(TiledArgs p) {
    constexpr int NT = WM * WN * 64;
    constexpr int WTM = BM / WM;
    constexpr int WTN = BN / WN;
    constexpr int FM = WTM / 32;
    constexpr int FN = WTN / 32;
    static_assert(FN % 2 == 0, "column blocks in pairs");
    typedef SplitOperand<NT, AKC, BM> OpA;
    typedef SplitOperand<NT, BKC, BN> OpB;
    constexpr int A_W = SplitLds<BM>::STAGE;
    constexpr int B_W = SplitLds<BN>::STAGE;
    __shared__ __attribute__((aligned(16))) uint32_t lds_a[2 * A_W];
    __shared__ __attribute__((aligned(16))) uint32_t lds_b[2 * B_W];
    __shared__ int lds_flag;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int lo = lane & 31;
    const int hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN;
    const int wn = wave % WN;

    TileCoord tc = tile_coord<BM, BN>(p, blockIdx.x);
    tc.split = __builtin_amdgcn_readfirstlane(tc.split);
    tc.b = __builtin_amdgcn_readfirstlane(tc.b);
    tc.m0 = __builtin_amdgcn_readfirstlane(tc.m0);
    tc.n0 = __builtin_amdgcn_readfirstlane(tc.n0);

    OpA opa;
    OpB opb;
    opa.init(p.A + (int64_t)tc.b * p.sA, p.lda, tc.m0, p.M, tid);
    opb.init(p.B + (int64_t)tc.b * p.sB, p.ldb, tc.n0, p.N, tid);

    f16 acc[FM][FN], low[FM][FN];  // sums of the high parts' products, of the others
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.f;
    };
    clear();
    if (tid == 0) lds_flag = 0;

    const int K = p.K;
    const int kt0 = tc.split * p.kt_per_split;
    const int kt1 = min((K + SBK - 1) / SBK, kt0 + p.kt_per_split);
    // k-tile kt from its first k on (past the range's end: its last k-tile again, which is
    // then not multiplied), and the k it shares with the tile before it
    auto first_k = [&](int kt) { return min(min(kt, kt1 - 1) * SBK, K - SBK); };
    auto drop = [&](int kt) {
        const int dup = kt * SBK - (K - SBK);
        if (kt < kt1 && dup > 0) {
            opa.drop(dup);
            opb.drop(dup);
        }
    };
    // Step s of splitting the k-tile in registers into stage st, A's steps before B's; each
    // operand's next k-tile (first k: next) is fetched behind its last step.
    constexpr int STEPS = OpA::STEPS + OpB::STEPS;
    auto split_step = [&](auto s, int st, int next) {
        constexpr int S = decltype(s)::value;
        if constexpr (S < OpA::STEPS) {
            opa.template split_step<S>(lds_a + st * A_W);
            if constexpr (S == OpA::STEPS - 1) opa.fetch(next);
        } else if constexpr (S < STEPS) {
            opb.template split_step<S - OpA::STEPS>(lds_b + st * B_W);
            if constexpr (S == STEPS - 1) opb.fetch(next);
        }
    };

    // The products of two parts (0 high, 1 mid, 2 low), the smallest first (gemm_split.hip: what
    // the three that are left out amount to, and why the last has a sum of its own).
    constexpr int PA[6] = {0, 2, 1, 1, 0, 0};
    constexpr int PB[6] = {2, 0, 1, 0, 1, 0};
    bf8 fa[3][FM], fb[3][2];
    auto read_a = [&](int st, int pl) {
        typedef SplitLds<BM> L;
#pragma unroll
        for (int i = 0; i < FM; ++i)
            __builtin_memcpy(&fa[pl][i], lds_a + st * A_W + pl * L::PLANE + hi * L::CHUNK +
                                             (wm * WTM + 32 * i + lo) * 4, 16);
    };
    auto read_b = [&](int st, int j0, int pl) {
        typedef SplitLds<BN> L;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            __builtin_memcpy(&fb[pl][j], lds_b + st * B_W + pl * L::PLANE + hi * L::CHUNK +
                                             (wn * WTN + 32 * (j0 + j) + lo) * 4, 16);
    };
    // k-tile kt out of stage ST while k-tile kt + 1 (in registers) is split into the other
    // stage and k-tile kt + 2 is fetched. MFMA n is followed by split step n / SPREAD. A part
    // of the next two column blocks is read once its last product is issued.
    constexpr int MFMAS = 6 * FM * FN;
    constexpr int SPREAD = MFMAS * 3 / 4 / STEPS > 1 ? MFMAS * 3 / 4 / STEPS : 1;
    auto step = [&](int kt, auto stage) {
        constexpr int ST = decltype(stage)::value;
        drop(kt + 1);
        const int next = first_k(kt + 2);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            read_a(ST, PA[q]);
            read_b(ST, 0, PB[q]);
        }
        unroll<MFMAS>([&](auto n) {
            constexpr int N = decltype(n)::value;
            constexpr int j0 = N / (12 * FM) * 2, q = N / (2 * FM) % 6;
            constexpr int i = N / 2 % FM, j = N % 2;
            __builtin_amdgcn_sched_barrier(0);
            f16 &c = q == 5 ? acc[i][j0 + j] : low[i][j0 + j];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[PA[q]][i], fb[PB[q]][j], c, 0, 0, 0);
            // (an MFMA has no side effect: without a use here it is moved down)
            asm volatile("" : "+v"(c));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (i == FM - 1 && j == 1 && j0 + 2 < FN) {
                if constexpr (q == 0) read_b(ST, j0 + 2, 2);
                if constexpr (q == 4) read_b(ST, j0 + 2, 1);
                if constexpr (q == 5) read_b(ST, j0 + 2, 0);
            }
            if constexpr (N % SPREAD == 0 && N / SPREAD < STEPS)
                split_step(std::integral_constant<int, N / SPREAD>{}, ST ^ 1, next);
        });
        __syncthreads();
    };

    opa.fetch(first_k(kt0));
    opb.fetch(first_k(kt0));
    drop(kt0);
    unroll<STEPS>([&](auto s) { split_step(s, 0, first_k(kt0 + 1)); });
    __syncthreads();
    for (int kt = kt0; kt < kt1; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        if (kt + 1 < kt1) step(kt + 1, std::integral_constant<int, 1>{});
    }

    // An output that is not finite (an infinity, NaN or value of 4.04e31 or more among the
    // operands, which the parts do not carry, or a sum of 4.83e24 or more, which overflows
    // scaled): the tile again in fp32, on the fp32 MFMA.
    bool bad = false;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] += low[i][j][r];
                bad |= !(__builtin_fabsf(acc[i][j][r]) < __builtin_inff());
                acc[i][j][r] *= kSplitUnscale;
            }
    if (bad) lds_flag = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(lds_flag) != 0) {
        clear();
        float *pa = reinterpret_cast<float *>(lds_a);
        float *pb = reinterpret_cast<float *>(lds_b);
        for (int kt = kt0; kt < kt1; ++kt) {
            opa.fetch(first_k(kt));
            opb.fetch(first_k(kt));
            drop(kt);
            __syncthreads();
            opa.put_f32(pa);
            opb.put_f32(pb);
            __syncthreads();
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                f4 xa[FM], xb[FN];
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    xa[i] = *reinterpret_cast<const f4 *>(
                        pa + ((2 * g + hi) * BM + wm * WTM + 32 * i + lo) * 4);
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    xb[j] = *reinterpret_cast<const f4 *>(
                        pb + ((2 * g + hi) * BN + wn * WTN + 32 * j + lo) * 4);
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                xa[i][s], xb[j][s], acc[i][j], 0, 0, 0);
            }
        }
    }
    store_tile<FM, FN>(p, tc, tc.m0 + wm * WTM, tc.n0 + wn * WTN, lane, acc);
}

template <int BM, int BN, int WM, int WN, bool AKC, bool BKC>
int launch_split(hipStream_t s, TiledArgs &a) {
    a.tiles_m = (a.M + BM - 1) / BM;
    a.tiles_n = (a.N + BN - 1) / BN;
    const int nk = (a.K + SBK - 1) / SBK;
    const int want = a.splits < nk ? a.splits : nk;
    a.kt_per_split = (nk + want - 1) / want;
    a.splits = (nk + a.kt_per_split - 1) / a.kt_per_split;
    const int64_t total = (int64_t)a.tiles_m * a.tiles_n * a.batch * a.splits;
    if (total > INT32_MAX)
        return set_error(MIGEMM_ERR_UNSUPPORTED, "gemm: %lld tiles exceed one launch",
                         (long long)total);
    a.total = (int)total;
    if (const int rc = check_partials(a)) return rc;
    set_tile_divisors(a);
    MIGEMM_LAUNCH((gemm_split_kernel<BM, BN, WM, WN, AKC, BKC>), dim3(a.total),
                  dim3(WM * WN * 64), 0, s, a);
    return launch_status("gemm_split_kernel launch");
}

template <int BM, int BN, int WM, int WN>
int launch_split_layouts(hipStream_t s, TiledArgs &a, bool akc, bool bkc) {
    if (akc && bkc) return launch_split<BM, BN, WM, WN, true, true>(s, a);
    if (akc) return launch_split<BM, BN, WM, WN, true, false>(s, a);
    if (!bkc) return launch_split<BM, BN, WM, WN, false, false>(s, a);
    return launch_split<BM, BN, WM, WN, false, true>(s, a);
}

}  // namespace

}  // namespace migemm
