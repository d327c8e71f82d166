// Layout and reduction kernels of the matmul path:
//  * tensor permute (cl_kernels/permute.cl:11-50): through LDS tiles when the source's
//    contiguous axis moves (the [0,2,1] / [1,0] forms that BmmOp.Backward and the Python
//    Linear use among them), else a generic <=10-D gather;
//  * column sums (cs/cl_kernels/linear.cl:149-168 linear_bias_backward and
//    cs/cl_kernels/reduce_sum_axis.cl:3-24 reduce_sum_axis): each output is summed over
//    the reduced axis in ascending order from +0.0f, exactly as the reference kernels do,
//    so these results are bit-identical to the reference's.
#include "migemm_internal.h"

namespace migemm {
namespace {

constexpr int MAXD = 10;

// FastDiv / make_fastdiv / fast_div: migemm_internal.h.
struct PermuteArgs {
    const float *src;
    float *dst;
    int64_t total;
    int ndim;
    int narrow;  // total < 2^31: every index and offset fits 32 bits
    int64_t dst_dims[MAXD];
    int64_t src_stride_of_dst_axis[MAXD];  // stride in src of the axis placed at dst axis i
    FastDiv div[MAXD];                     // dst_dims as invariant divisors (narrow only)
};

// dst[t] = src[offset of t's destination coordinates], coordinates from the last axis
// (permute.cl:2-8,11-50), on the canonical form built by launch_permute. Element t is a
// group of VW floats (VW = 4 when the innermost destination axis is contiguous in the source
// too); total, dims and strides are in those units. Tensors under 2^31 elements unpack t
// with 32-bit invariant divisions: with one 64-bit division and remainder per axis per
// element the kernel was bound by integer arithmetic, not by memory.
template <int VW>
__global__ void __launch_bounds__(256) permute_gather_kernel(PermuteArgs a) {
    typedef float vec __attribute__((ext_vector_type(VW)));
    const vec *src = reinterpret_cast<const vec *>(a.src);
    vec *dst = reinterpret_cast<vec *>(a.dst);
    if (a.narrow) {
        const uint32_t total = (uint32_t)a.total;
        const uint32_t step = gridDim.x * blockDim.x;
        for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += step) {
            uint32_t rem = t;
            uint32_t off = 0;
            for (int i = a.ndim - 1; i >= 0; --i) {
                const uint32_t q = fast_div(rem, a.div[i]);
                off += (rem - q * a.div[i].d) * (uint32_t)a.src_stride_of_dst_axis[i];
                rem = q;
            }
            dst[t] = src[off];
        }
        return;
    }
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < a.total; t += step) {
        int64_t rem = t;
        int64_t off = 0;
        for (int i = a.ndim - 1; i >= 0; --i) {
            const int64_t d = a.dst_dims[i];
            const int64_t c = rem % d;
            rem /= d;
            off += c * a.src_stride_of_dst_axis[i];
        }
        dst[t] = src[off];
    }
}

// dst[o][c][r] = src[row_offset(o, r) + c]: every permutation whose source-contiguous axis (c)
// is not its innermost one. r runs over the destination axes behind c, merged (R of them,
// contiguous in dst), o over those before it; row_offset unpacks both by invariant divisions.
// A batched transpose is the case of one axis behind c.
//  * HBM-bound: 64x64 tiles through LDS, 16 bytes per lane on both sides (no alignment
//    needed), so a row of the tile is 256 contiguous bytes read and 256 written. LDS rows of
//    65 floats keep the scalar writes and reads on distinct banks. Matrices that a tile of
//    32x32 holds or that fill only half of a 64-wide one take 32x32 tiles (launch_permute).
//  * Consecutive work-groups of an XCD step along r, in groups of 32 tiles: where dst rows do
//    not start on 128-byte lines, neighbouring tiles share lines, and L2 merges the two parts
//    before the line goes to HBM. Whole columns of tiles would touch every page of a large
//    source at once (46342 x 46342: 7036 us, in groups 6300).
// Measured (us per call, 3 rotating inputs, 32x32 tiles with 4-byte accesses or, for the
// reversed axes, the gather kernel / this): 4096 x 4096 25.3 / 21.9 (6.1 TB/s), 4095 x 4097
// 36.9 / 23.4, 64 x 600 x 600 by (0, 2, 1) 51.0 / 33.9, by (2, 1, 0) 175.9 / 38.4, 32 x 500
// x 16 x 64 by (0, 2, 3, 1) 24.6 / 22.2.
struct TransposeArgs {
    const float *src;
    float *dst;
    uint32_t R, C;
    uint32_t tiles_r;
    uint32_t total;  // work-groups
    FastDiv by_rc;       // tiles_r * tiles_c
    FastDiv in_group;    // TR_GROUP * tiles_c
    FastDiv last_group;  // tiles of r in the last group
    // source axes of r (innermost first) and of o (innermost first)
    int nr, no;
    FastDiv rdiv[MAXD], odiv[MAXD];
    uint64_t rstride[MAXD], ostride[MAXD];
};

// Work-groups of 256 threads that one launch can hold: a grid has fewer than 2^32 threads.
constexpr int64_t kMaxGroups = ((int64_t)1 << 24) - 1;

constexpr int TR_GROUP = 32;  // tiles of r rastered together

__device__ __forceinline__ uint64_t unpack_offset(uint32_t t, int n, const FastDiv *div,
                                                  const uint64_t *stride) {
    uint64_t off = 0;
    for (int i = 0; i + 1 < n; ++i) {
        const uint32_t q = fast_div(t, div[i]);
        off += (t - q * div[i].d) * stride[i];
        t = q;
    }
    return off + t * stride[n - 1];
}

template <int TR>  // tile edge
__global__ void __launch_bounds__(256) transpose_kernel(TransposeArgs a) {
    typedef float vec __attribute__((ext_vector_type(4)));
    __shared__ float tile[TR][TR + 1];
    uint32_t pid = blockIdx.x;
    pid = (a.total & 7) == 0 ? (pid & 7) * (a.total >> 3) + (pid >> 3) : pid;
    const uint32_t o = fast_div(pid, a.by_rc);
    const uint32_t t = pid - o * a.by_rc.d;
    const uint32_t first = fast_div(t, a.in_group) * TR_GROUP;
    const uint32_t tg = t - first / TR_GROUP * a.in_group.d;
    uint32_t tc, tr;
    if (a.tiles_r - first >= TR_GROUP) {
        tc = tg / TR_GROUP;
        tr = first + tg % TR_GROUP;
    } else {
        tc = fast_div(tg, a.last_group);
        tr = first + tg - tc * a.last_group.d;
    }
    const uint32_t r0 = tr * TR;
    const uint32_t c0 = tc * TR;
    const uint64_t obase = a.no > 0 ? unpack_offset(o, a.no, a.odiv, a.ostride) : 0;
    const uint32_t lane4 = 4 * (threadIdx.x % (TR / 4));  // this thread's 4 columns (rows of dst)
    const uint32_t line = threadIdx.x / (TR / 4);   // and its line of each LINES
    const uint32_t nr = min((uint32_t)TR, a.R - r0), nc = min((uint32_t)TR, a.C - c0);
    const float *s = a.src + obase + c0;
    constexpr int LINES = 1024 / TR, PASSES = TR / LINES;
    vec v[PASSES];
#pragma unroll
    for (int j = 0; j < PASSES; ++j) {
        const uint32_t r = line + LINES * j;
        if (r < nr) {
            const float *q = s + unpack_offset(r0 + r, a.nr, a.rdiv, a.rstride) + lane4;
            if (lane4 + 4 <= nc) {
                __builtin_memcpy(&v[j], q, sizeof(vec));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[j][e] = lane4 + e < nc ? q[e] : 0.0f;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < PASSES; ++j) {
        const uint32_t r = line + LINES * j;
        if (r < nr)
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[r][lane4 + e] = v[j][e];
    }
    __syncthreads();
    float *d = a.dst + ((size_t)o * a.C + c0) * a.R + r0;
#pragma unroll
    for (int j = 0; j < PASSES; ++j) {
        const uint32_t c = line + LINES * j;
        if (c < nc) {
            vec x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = tile[lane4 + e][c];
            float *q = d + (size_t)c * a.R + lane4;
            if (lane4 + 4 <= nr) {
                __builtin_memcpy(q, &x, sizeof(vec));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (lane4 + e < nr) q[e] = x[e];
            }
        }
    }
}

// Sum over the middle axis of X[outer][axis][inner], in chunks of `rows` consecutive a:
//   out[c][o][i] = sum over a in [c*rows, min((c+1)*rows, axis)), ascending from +0.0f,
//                  of X[(o*axis + a)*inner + i].
// The reference kernels (cs/cl_kernels/reduce_sum_axis.cl:3-27, linear.cl:149-168) run one
// ascending chain per output over the whole axis: a single dependent chain per column,
// which at 12000 rows leaves the GPU waiting on one load at a time. With one chunk (axis <=
// rows) this is exactly the reference's order; otherwise the chunk sums are added in
// chunk order by reduce_slices_kernel (deterministic, and within the blocked-summation
// error bound (rows - 1 + chunks - 1) * 2^-24 * sum |x|). Each thread owns VW consecutive i
// (128-bit loads when VW = 4) and keeps CS_INFLIGHT rows of loads in flight. With
// `accumulate` (one chunk only) the sum is added to the output's value: out += sum.
constexpr int CS_INFLIGHT = 16;

template <int VW>
__global__ void __launch_bounds__(256) column_sum_kernel(const float *__restrict__ X,
                                                           float *__restrict__ out, int outer,
                                                           int axis, int inner, int rows,
                                                           int accumulate) {
    typedef float vec __attribute__((ext_vector_type(VW)));
    const int vecs = (inner + VW - 1) / VW;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)outer * vecs) return;
    // 32-bit division where it fits (a 64-bit one is a long software sequence)
    const int o = t <= INT32_MAX ? (int)((uint32_t)t / (uint32_t)vecs) : (int)(t / vecs);
    const int i0 = (int)(t - (int64_t)o * vecs) * VW;
    const int cnt = inner - i0 < VW ? inner - i0 : VW;
    const int c = blockIdx.y;
    const int a0 = c * rows;
    const int a1 = axis - a0 < rows ? axis : a0 + rows;
    const float *x = X + ((int64_t)o * axis + a0) * inner + i0;
    vec sum = {};
    if (cnt == VW) {
        for (int a = a0; a < a1; a += CS_INFLIGHT) {
            vec v[CS_INFLIGHT];
#pragma unroll
            for (int g = 0; g < CS_INFLIGHT; ++g)
                if (a + g < a1)
                    __builtin_memcpy(&v[g], x + (int64_t)(a - a0 + g) * inner, sizeof(vec));
#pragma unroll
            for (int g = 0; g < CS_INFLIGHT; ++g)
                if (a + g < a1) sum += v[g];
        }
    } else {
        for (int e = 0; e < cnt; ++e) {
            float s = 0.0f;
            for (int a = a0; a < a1; ++a) s += x[(int64_t)(a - a0) * inner + e];
            sum[e] = s;
        }
    }
    float *y = out + ((int64_t)c * outer + o) * inner + i0;
#pragma unroll
    for (int e = 0; e < VW; ++e)
        if (e < cnt) y[e] = accumulate ? y[e] + sum[e] : sum[e];
}

// Row sums (inner = 1): out[o] = sum over a of X[o][a], in column_sum_kernel's order (chunks
// of CS_ROWS ascending from +0.0f, the chunk sums added in chunk order), so the bits are the
// same. There every thread walked a row of its own, 4 bytes at a time at a stride of the row
// length: 64000 rows of 513 (131 MB) took 135 us + 4.7 us for the chunk sums. Here a
// wavefront owns a chunk of 64 rows and moves it through LDS in tiles of 64 columns: 16
// loads of 16 bytes per lane cover 4 rows x 256 contiguous bytes each, the next tile's are in
// flight while the lane of a row adds this tile's 64 values, 4 per LDS read (a row stride of
// 68 floats keeps 16 lanes on distinct banks). The 4 wavefronts of a work-group take 4
// consecutive chunks at a time and wavefront 0 adds their sums in order, so one launch does
// all of it: 149 -> 28.9 us per call, 4.5 TB/s (4096 x 4096: 37 -> 17 us; 100 x 100000:
// 42 -> 29). With few rows and many chunks (PARTIAL) each work-group takes
// one group of 4 chunks and writes their sums [chunk][row] for reduce_slices_kernel.
constexpr int CS_ROWS = 256;  // rows of the reduced axis per chunk
constexpr int RS_TILE = 64;   // columns per tile (and rows per wavefront)
constexpr int RS_LD = 68;

template <bool PARTIAL>
__global__ void __launch_bounds__(256) row_sum_kernel(const float *__restrict__ X,
                                                      float *__restrict__ out, int outer,
                                                      int axis) {
    typedef float vec __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) float tiles[4][RS_TILE * RS_LD];
    __shared__ float sums[4][RS_TILE];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int o0 = blockIdx.x * RS_TILE;
    const int chunks = (axis + CS_ROWS - 1) / CS_ROWS;
    const int g0 = PARTIAL ? blockIdx.y * 4 : 0;
    const int g1 = PARTIAL ? min(chunks, g0 + 4) : chunks;
    float *tile = tiles[w];
    // this lane's loads: 4 columns from 4 (lane % 16) of rows lane / 16 + 4 j
    const int lc = 4 * (lane & 15);
    const int lr = lane >> 4;
    vec v[16];
    auto fetch = [&](int c0, int c1) {  // columns c0 .. c0 + 63, those from c1 on zero
        const bool whole = c0 + RS_TILE <= c1;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float *q = X + (int64_t)min(o0 + lr + 4 * j, outer - 1) * axis + c0 + lc;
            if (whole) {
                __builtin_memcpy(&v[j], q, sizeof(vec));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[j][e] = c0 + lc + e < c1 ? q[e] : 0.0f;
            }
        }
    };
    float total = 0.0f;
    for (int g = g0; g < g1; g += 4) {
        const int c = g + w;  // this wavefront's chunk
        if (c < g1) {
            const int a0 = c * CS_ROWS;
            const int a1 = min(axis, a0 + CS_ROWS);
            float sum = 0.0f;
            fetch(a0, a1);
            for (int a = a0; a < a1; a += RS_TILE) {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    *reinterpret_cast<vec *>(tile + (lr + 4 * j) * RS_LD + lc) = v[j];
                // (the wavefront's own LDS accesses complete in order; this keeps the compiler
                // from moving them across)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (a + RS_TILE < a1) fetch(a + RS_TILE, a1);
#pragma unroll
                for (int q = 0; q < RS_TILE; q += 4) {
                    const vec x = *reinterpret_cast<const vec *>(tile + lane * RS_LD + q);
                    sum += x[0];
                    sum += x[1];
                    sum += x[2];
                    sum += x[3];
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            if constexpr (PARTIAL) {
                if (o0 + lane < outer) out[(int64_t)c * outer + o0 + lane] = sum;
            } else {
                sums[w][lane] = sum;
            }
        }
        if constexpr (!PARTIAL) {
            __syncthreads();
            if (w == 0) {
                const int n = min(4, g1 - g);
                total = g == 0 ? sums[0][lane] : total + sums[0][lane];
                for (int q = 1; q < n; ++q) total += sums[q][lane];
            }
            __syncthreads();
        }
    }
    if constexpr (!PARTIAL) {
        const int o = o0 + lane;
        if (w == 0 && o < outer) out[o] = total;
    }
}

// Hp[t][h] = H[t - 1][h] when step t % seq_len > 0 of its sequence, else 0: the previous
// hidden state of the same sequence, the left operand of grad_U += H_prev^T * grad_gates
// (cs/cl_kernels/lstm.cl:582-590, tokens ordered [batch][seq_len]). VW consecutive h per
// thread (hidden % VW == 0).
template <int VW>
__global__ void __launch_bounds__(256) shift_rows_kernel(const float *__restrict__ H,
                                                           float *__restrict__ Hp,
                                                           int64_t total, int seq_len,
                                                           int hidden) {
    typedef float vec __attribute__((ext_vector_type(VW)));
    const int64_t step = (int64_t)gridDim.x * blockDim.x * VW;
    for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * VW; i < total;
         i += step) {
        // token index, by 32-bit division where it fits
        const int64_t t = i <= INT32_MAX ? (int64_t)((uint32_t)i / (uint32_t)hidden) : i / hidden;
        const int step_in_seq = t <= INT32_MAX ? (int)((uint32_t)t % (uint32_t)seq_len)
                                               : (int)(t % seq_len);
        vec v = {};
        if (step_in_seq != 0) __builtin_memcpy(&v, H + i - hidden, sizeof(vec));
        __builtin_memcpy(Hp + i, &v, sizeof(vec));
    }
}

// The streaming-read reference of the HBM-bound kernels (the GEMV of BASELINE config 5b):
// reads n4 float4 once, each work-group a contiguous range, every lane RS_U 16-byte
// non-temporal loads in flight, and writes one sum per work-group so the loads stay live.
// What it reaches is the read rate a kernel that only streams can get on the box.
constexpr int RS_U = 16;
__global__ void __launch_bounds__(256) stream_read_kernel(const float4 *__restrict__ src,
                                                          int64_t n4, int64_t per,
                                                          float *__restrict__ sums) {
    typedef float vec __attribute__((ext_vector_type(4)));
    const int64_t lo = (int64_t)blockIdx.x * per;
    const int64_t hi = lo + per < n4 ? lo + per : n4;
    const vec *s = reinterpret_cast<const vec *>(src);
    vec acc = vec{0.f, 0.f, 0.f, 0.f};
    for (int64_t i = lo + threadIdx.x; i < hi; i += 256 * RS_U) {
        vec v[RS_U];
#pragma unroll
        for (int u = 0; u < RS_U; ++u) {
            const int64_t j = i + (int64_t)u * 256;
            v[u] = j < hi ? __builtin_nontemporal_load(s + j) : vec{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < RS_U; ++u) acc += v[u];
    }
    __shared__ float part[256];
    part[threadIdx.x] = acc[0] + acc[1] + acc[2] + acc[3];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = part[0];
}

}  // namespace

int launch_stream_read(hipStream_t stream, const float *src, int64_t n4, float *sums,
                       int blocks) {
    const int64_t per = (n4 + blocks - 1) / blocks;
    MIGEMM_LAUNCH(stream_read_kernel, dim3(blocks), dim3(256), 0, stream,
                  reinterpret_cast<const float4 *>(src), n4, per, sums);
    return launch_status("stream_read_kernel launch");
}

int launch_permute(hipStream_t stream, const float *src, float *dst, const int *src_dims,
                   const int *axes, int num_dims, int64_t total) {
    // Canonical form: size-1 axes dropped, and each run of destination axes that lie
    // consecutively and in order in the source merged into one axis (the outer one's source
    // stride is the inner one's stride times its size). [32,128,16,64] by (0,2,1,3) stays
    // 4-D; [B,R,C] by (0,2,1) is a batched transpose; an identity permutation is one axis.
    int64_t src_strides[MAXD];
    int64_t st = 1;
    for (int i = num_dims - 1; i >= 0; --i) {
        src_strides[i] = st;
        st *= src_dims[i];
    }
    int64_t cd[MAXD], cs[MAXD];
    int nd = 0;
    for (int i = 0; i < num_dims; ++i) {
        const int64_t d = src_dims[axes[i]];
        const int64_t str = src_strides[axes[i]];
        if (d == 1) continue;
        if (nd > 0 && cs[nd - 1] == str * d) {
            cd[nd - 1] *= d;
            cs[nd - 1] = str;
        } else {
            cd[nd] = d;
            cs[nd] = str;
            ++nd;
        }
    }
    if (nd == 0) {  // a single element
        cd[0] = 1;
        cs[0] = 1;
        nd = 1;
    }
    // The source's contiguous axis (C elements) is not the innermost destination axis: through
    // LDS tiles where these are full enough. A 64x64 tile takes about 1.0 ns of the chip, a
    // 32x32 one 0.6, an element of the gather kernel 2.2 ps and up, and the memory 1.3 ps an
    // element. So the tiles are 32x32 for C <= 32 unless R leaves over a quarter of several
    // tiles empty (us of 2^24 elements as outer x R x C, 64x64 / 32x32: 24 x 24 35.0 / 24.5, 512
    // x 32 25.8 / 21.0, 130 x 16 35.3 / 30.4; 40 x 32 23.6 / 26.5, 16 x 130 28.9 / 32.2), and
    // tiles with fewer than `full` elements are left to the gather kernel (tiles / gather: 8 x 130
    // 48.6 / 37.4, 16 x 16 43.9 / 41.0, 8388608 x 2 134 / 37, 4194304 x 4 71 / 50; 8 x 64 38.0 /
    // 37.6, 16 x 20 37.9 / 39.4, 64 x 7 51.4 / 39.4, 64 x 8 44.2 / 42.6, 1000 x 7 40.9 / 61.3,
    // 2097152 x 8 38 / 84).
    int jc = 0;  // its place
    while (cs[jc] != 1) ++jc;
    const int64_t C = cd[jc];
    int64_t R = 1;
    for (int i = jc + 1; i < nd; ++i) R *= cd[i];
    const int64_t outer = total / (R * C);
    const bool small = C <= 32 && (R <= 32 || 4 * R >= 3 * 32 * ((R + 31) / 32));
    const int TR = small ? 32 : 64;
    const int full = !small ? 512 : R <= 32 ? 320 : R <= 128 ? 256 : 224;
    const int64_t tiles_r = (R + TR - 1) / TR, tiles_c = (C + TR - 1) / TR;
    if (jc < nd - 1 && R * C >= full * tiles_r * tiles_c && R <= INT32_MAX && C <= INT32_MAX &&
        outer * tiles_r * tiles_c <= kMaxGroups && TR_GROUP * tiles_c <= INT32_MAX) {
        TransposeArgs a;
        a.src = src;
        a.dst = dst;
        a.nr = a.no = 0;
        for (int i = nd - 1; i > jc; --i, ++a.nr) {
            a.rdiv[a.nr] = make_fastdiv((uint32_t)cd[i]);
            a.rstride[a.nr] = (uint64_t)cs[i];
        }
        for (int i = jc - 1; i >= 0; --i, ++a.no) {
            a.odiv[a.no] = make_fastdiv((uint32_t)cd[i]);
            a.ostride[a.no] = (uint64_t)cs[i];
        }
        a.R = (uint32_t)R;
        a.C = (uint32_t)C;
        a.tiles_r = (uint32_t)tiles_r;
        a.in_group = make_fastdiv((uint32_t)(TR_GROUP * tiles_c));
        a.last_group = make_fastdiv((uint32_t)(tiles_r % TR_GROUP));
        a.by_rc = make_fastdiv((uint32_t)(tiles_r * tiles_c));
        a.total = (uint32_t)(outer * tiles_r * tiles_c);
        if (small)
            MIGEMM_LAUNCH(transpose_kernel<32>, dim3(a.total), dim3(256), 0, stream, a);
        else
            MIGEMM_LAUNCH(transpose_kernel<64>, dim3(a.total), dim3(256), 0, stream, a);
        record_plan(PlanRecord{"transpose", TR, TR, 1, 16, (int)a.R, (int)a.C, 0, (int)outer,
                               false, false});
        return launch_status("transpose_kernel launch");
    }
    // 16-byte elements when the innermost destination axis is the source's contiguous one
    // and holds whole groups of 4 (every other stride is then a multiple of 4 as well)
    const int vw = (cs[nd - 1] == 1 && cd[nd - 1] % 4 == 0 && ((uintptr_t)src & 15) == 0 &&
                    ((uintptr_t)dst & 15) == 0)
                       ? 4
                       : 1;
    PermuteArgs a;
    a.src = src;
    a.dst = dst;
    a.total = total / vw;
    a.ndim = nd;
    a.narrow = a.total <= INT32_MAX;
    for (int i = 0; i < MAXD; ++i) {
        a.dst_dims[i] = i < nd ? (i == nd - 1 ? cd[i] / vw : cd[i]) : 1;
        // in units of vw floats; with vw = 4 the innermost axis is contiguous (stride 1)
        a.src_stride_of_dst_axis[i] = i < nd ? cs[i] / (i == nd - 1 ? 1 : vw) : 0;
        a.div[i] = make_fastdiv(a.narrow ? (uint32_t)a.dst_dims[i] : 1u);
    }
    int64_t blocks = (a.total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (vw == 4)
        MIGEMM_LAUNCH(permute_gather_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, stream,
                           a);
    else
        MIGEMM_LAUNCH(permute_gather_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, stream,
                           a);
    record_plan(PlanRecord{"permute_gather", 0, 0, 1, 4 * vw, 0, 0, 0, nd, false, false});
    return launch_status("permute_gather_kernel launch");
}

int launch_column_sum(hipStream_t stream, const float *X, float *Y, int outer, int axis,
                      int inner, bool accumulate) {
    // Chunks of 256 rows: 12000 x 6565 (the Linear(500 -> 6565) bias gradient) is 47 chunks
    // of 7 work-groups, each thread with 16 rows of 128-bit loads in flight.
    int rows = CS_ROWS;
    if ((axis + rows - 1) / rows > 65535) rows = (axis + 65534) / 65535;
    const int chunks = (axis + rows - 1) / rows;
    // row_sum_kernel: not for rows shorter than 16 (two lanes' worth of a tile) or fewer than
    // 64 (lanes of every tile idle). With 512 or more work-groups of rows, or one group of
    // chunks, a work-group takes whole rows, and there are no chunk sums to keep.
    const int64_t blocks = ((int64_t)outer + RS_TILE - 1) / RS_TILE;
    const bool by_row = inner == 1 && !accumulate && rows == CS_ROWS && outer >= 64 &&
                        axis >= 16 && blocks <= kMaxGroups;
    const bool whole = by_row && (chunks <= 4 || blocks >= 512);
    float *dst = Y;
    if (chunks > 1 && !whole) {
        int st = MIGEMM_OK;
        dst = static_cast<float *>(
            workspace(stream, (size_t)chunks * outer * inner * sizeof(float), &st));
        if (dst == nullptr) return st;
    }
    if (by_row) {
        if (whole)
            MIGEMM_LAUNCH(row_sum_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, stream, X,
                          Y, outer, axis);
        else
            MIGEMM_LAUNCH(row_sum_kernel<true>,
                          dim3((unsigned)blocks, (unsigned)((chunks + 3) / 4)), dim3(256), 0,
                          stream, X, dst, outer, axis);
        const int rc = launch_status("row_sum_kernel launch");
        record_plan(PlanRecord{"row_sum", rows, RS_TILE, whole ? 1 : chunks, 16, outer, inner,
                               axis, 1, false, false});
        if (rc != MIGEMM_OK || whole) return rc;
        return launch_reduce_slices(stream, dst, chunks, outer, 1, inner, nullptr, Y, inner,
                                    inner);
    }
    const bool vec = inner % 4 == 0;
    const int64_t threads = (int64_t)outer * (vec ? inner / 4 : inner);
    const dim3 grid((unsigned)((threads + 255) / 256), (unsigned)chunks);
    if (vec)
        MIGEMM_LAUNCH(column_sum_kernel<4>, grid, dim3(256), 0, stream, X, dst, outer,
                           axis, inner, rows, (int)(accumulate && chunks == 1));
    else
        MIGEMM_LAUNCH(column_sum_kernel<1>, grid, dim3(256), 0, stream, X, dst, outer,
                           axis, inner, rows, (int)(accumulate && chunks == 1));
    const int rc = launch_status("column_sum_kernel launch");
    record_plan(PlanRecord{"column_sum", rows, vec ? 4 : 1, chunks, 0, outer, inner, axis, 1,
                           false, false});
    if (rc != MIGEMM_OK || chunks == 1) return rc;
    return launch_reduce_slices(stream, dst, chunks, outer, 1, inner, nullptr, Y, inner, inner,
                                accumulate);
}

int launch_shift_rows(hipStream_t stream, const float *H, float *Hp, int total_tokens,
                      int seq_len, int hidden) {
    const int64_t total = (int64_t)total_tokens * hidden;
    const bool vec = hidden % 4 == 0;
    int64_t blocks = ((vec ? total / 4 : total) + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (vec)
        MIGEMM_LAUNCH(shift_rows_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, stream, H,
                           Hp, total, seq_len, hidden);
    else
        MIGEMM_LAUNCH(shift_rows_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, stream, H,
                           Hp, total, seq_len, hidden);
    return launch_status("shift_rows_kernel launch");
}

}  // namespace migemm
