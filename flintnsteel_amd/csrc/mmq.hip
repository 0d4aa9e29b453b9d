// mmq.hip - prefill / batched expert GEMM (MMQ) over GGUF K-quant weights for MI355X gfx950: expert-id compaction,
// split Q8_1 activation images, and an f16-MFMA grouped GEMM with the SwiGLU + Q8_1 of act fused into the gate/up pass.
//
// Reference semantics: src/ggml/ggml_mmq.cu:74-129 (mmq_q8_1_bytes, mmq, mmq_experts: mm_ids_helper sorts the
// (token, slot) pairs by expert, the activations are quantised once per source row, the GEMM writes each row back to
// its (token, slot) position), include/fns/ggml_kernels.h:50-69. This is a new CDNA4 design, not ggml's mmq.cuh:
//
//   * Two forms of the GEMM. Types whose scales change every 32 columns (Q4_K, Q5_K, Q8_0, IQ4_XS, IQ3_XXS, IQ3_S) run on
//     int8 MFMA, one exact integer dot per sub-block and a convert + scale + fma per output (fns_mmq_i8.hpp). The others
//     (Q6_K and Q3_K scale every 16 columns, IQ2_S every 16) run the split form of this file, to which the points below
//     apply:
//   * In the split form the scales are folded into the operands instead, exactly: A = q8 * d8 as two f16 halves (hi + lo, see the image
//     layout below), B = integer code * integer sub-block scale as f16 (|B| <= 2048: exact; Q6_K's 8-bit scales are
//     split in two operands). v_mfma_f32_32x32x16_f16 then accumulates a whole 256-column superblock, and only the
//     superblock's float scales d (and dmin times one more MFMA of the min term) touch the accumulators.
//     Every product is exact; the sums are fp32.
//   * A = 32 activation rows (tokens) x 16 columns, B = 16 columns x 32 weight rows: the lane that owns output
//     (token i, weight row j) holds weight row j = lane % 32 for 16 tokens and decodes row j's codes and scales
//     itself. The 32x32 shape moves half the operand bytes (LDS reads, decode VALU) per product of the 16x16 one.
//   * A workgroup (4 waves) owns two 32-row weight streams per wave - gate and up of the same 128 rows (GLU), or 256
//     rows - and up to 64 of the expert's routed activation rows (2 tiles of 32): each weight byte is read from HBM
//     once per 64 routed rows. Activations are staged per half superblock in LDS by LDS-DMA, double-buffered (66 KB:
//     two workgroups per CU); weights go straight to VGPRs, half a superblock ahead.
//   * Gate/up: both matrices in one pass, then act = up * silu(gate) and its Q8_1 blocks (32 consecutive rows = 32
//     consecutive act columns) written straight into the split image rows the down pass reads.
//
// Outputs match the float64 oracle (oracle/fns_oracle.c) on the same Q8_1 activations within the fp32 tolerance of
// the tests.
#include <algorithm>
#include "fns_block.hpp"
#include "fns_common.hpp"
#include "fns_host.hpp"
#include "fns_internal.hpp"
#include "fns_lanes.hpp"
#include "fns_q8x8.hpp"
#include "fns_quarter.hpp"
#include "fns_router_gemm.hpp"

#include "fns/ggml_kernels.h"

namespace fns {

using namespace fns::dev;

namespace {

constexpr int kMmqThreads = 256;   // 4 waves
constexpr int kMmqWaves = kMmqThreads / 64;
constexpr int kMmqRows = 64;       // row granularity of the weight matrices
constexpr int kMmqTok = 64;        // activation rows per workgroup (2 MFMA tiles of 32)
constexpr int kCompactThreads = 1024;

// ---- scratch layout of the expert path --------------------------------------------------------------------------
// bounds[n_expert + 1] (sorted-row offset of each expert); the GEMM's group prefixes gprefix[2][n_expert + 1]: the
// 64-row groups of each expert (n_e / 64 full ones, and the remainder if it is > 32 rows; two 32-row MFMA tiles), and
// the remainder groups of <= 32 rows (one tile).
inline size_t bounds_bytes(int64_t n_expert) { return (size_t) 3 * (n_expert + 1) * 4; }
inline size_t gprefix_bytes(int64_t n_expert) { return (size_t) 2 * (n_expert + 1) * 4; }

// ---- compaction (ggml mm_ids_helper semantics, stable) ------------------------------------------------------------
// ids [n_tok][k] -> pairs p = t k + j sorted by expert, ties in p order: ids_dst[q] = p, ids_src1[q] = the activation
// row of p (t when x_rows_per_tok = 1, p when x_rows_per_tok = k), bounds[e] = first sorted position of expert e.
// Workgroup b owns the 1024-pair pieces [b per_wg, (b + 1) per_wg) and needs no other workgroup: each reads every id
// (they sit in the L2) into two LDS histograms - the pairs before its own, and the rest - which give every expert's
// first position and how many of its rows earlier workgroups place. Its own pieces are then ranked in order: the lanes
// that share an expert by ballots on the id bits, the waves by a prefix of their counts. One workgroup walking all
// pairs took 47 us at 32768 pairs and 7.8 us at 4096.
// Workgroup barrier for LDS data only: no global memory is produced and consumed inside the compaction kernel, so its
// barriers need not wait for the id loads and the output stores still in flight (__syncthreads' fence would).
__device__ __forceinline__ void lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// Exclusive prefix of the per-expert counts cnt[0..ne) (ne <= 256) by one wave (lane = its lane): cnt[e] becomes the
// expert's first sorted position; bounds[0..ne], and the group prefixes gprefix[0..ne] of the 64-row groups
// (n_e / 64 full ones, and the remainder if it is > 32 rows) and gprefix[ne + 1 .. 2 ne + 1] of the <= 32-row
// remainders are written (bounds null: none are). 4 experts per lane, then a lane scan.
__device__ __forceinline__ void expert_prefix_wave(int lane, int *cnt, int ne, int32_t *bounds, int32_t *gprefix) {
    int v[4], g[4], g2[4], s = 0, sg = 0, sg2 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = 4 * lane + j, r = (e < ne ? cnt[e] : 0) % kMmqTok;
        v[j] = e < ne ? cnt[e] : 0;
        g[j] = v[j] / kMmqTok + (r > kMmqTok / 2);
        g2[j] = r > 0 && r <= kMmqTok / 2;
        s += v[j];
        sg += g[j];
        sg2 += g2[j];
    }
    int incl = s, inclg = sg, inclg2 = sg2;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64), tg = __shfl_up(inclg, o, 64), tg2 = __shfl_up(inclg2, o, 64);
        if (lane >= o) {
            incl += t;
            inclg += tg;
            inclg2 += tg2;
        }
    }
    int run = incl - s, rung = inclg - sg, rung2 = inclg2 - sg2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = 4 * lane + j;
        if (e < ne) {
            cnt[e] = run;  // the expert's first sorted position (its count is no longer needed)
            if (bounds) {
                bounds[e] = run;
                gprefix[e] = rung;
                gprefix[ne + 1 + e] = rung2;
            }
        }
        run += v[j];
        rung += g[j];
        rung2 += g2[j];
    }
    if (lane == 63 && bounds) {
        bounds[ne] = incl;
        gprefix[ne] = inclg;
        gprefix[2 * ne + 1] = inclg2;
    }
}

__global__ __launch_bounds__(kCompactThreads) void k_mmq_compact(const int32_t *__restrict__ ids, int n, int k, int ne,
                                                                 int x_rows_per_tok, int32_t *__restrict__ ids_src1,
                                                                 int32_t *__restrict__ ids_dst, int32_t *bounds,
                                                                 int32_t *gprefix, int32_t *gdone, int n_gdone,
                                                                 int per_wg) {
    constexpr int NW = kCompactThreads / kWave, NT = kCompactThreads;
    __shared__ int pos[256], rest[256], cnt[256];
    __shared__ int wpos[NW][256];  // a piece's per-wave counts, then each wave's first sorted position per expert
    PF_MARK(2, 0);
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    const int n_it = (n + NT - 1) / NT, it0 = blockIdx.x * per_wg, it1 = min(n_it, it0 + per_wg);
    // this workgroup's first piece, in flight beside the histogram's loads
    const int own = n > 0 ? ids[min(it0 * NT + tid, n - 1)] : -1;
    for (int i = tid; i < NW * 256; i += NT) (&wpos[0][0])[i] = 0;
    if (tid < 256) pos[tid] = rest[tid] = 0;
    for (int i = blockIdx.x * NT + tid; i < n_gdone; i += gridDim.x * NT) gdone[i] = 0;  // the fused GEMM launch's arrivals
    lds_sync();
    PF_MARK(2, 2);
    // a piece's lanes with the same expert id: intersect the ballots of each id bit (and of liveness); the lane's rank
    // among them, and the wave's count of the expert
    auto rank_piece = [&](int e, bool live) __attribute__((always_inline)) {
        uint64_t same = __ballot(live);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t m = __ballot(live && ((e >> b) & 1));
            same &= ((e >> b) & 1) ? m : ~m;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1ull));
        if (live && rank == 0) wpos[wave][e] = __popcll(same);
        return rank;
    };
    int e = it0 * NT + tid < n ? own : -1;
    bool live = e >= 0 && e < ne;
    int rank = rank_piece(e, live);
    if (n_it > 1) {
        // clamped, unconditional loads, eight in flight
        constexpr int U = 8;
        for (int it = 0; it < n_it; it += U) {
            int v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = ids[min((it + u) * NT + tid, n - 1)];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if ((it + u) * NT + tid < n && v[u] >= 0 && v[u] < ne) atomicAdd(it + u < it0 ? &pos[v[u]] : &rest[v[u]], 1);
        }
    }
    lds_sync();
    PF_MARK(2, 3);
    if (tid < ne) {
        int c = pos[tid] + rest[tid];
        if (n_it <= 1)  // one piece: its counts are the waves'
            for (int w = 0; w < NW; ++w) c += wpos[w][tid];
        cnt[tid] = c;
    }
    lds_sync();
    if (wave == 0) expert_prefix_wave(lane, cnt, ne, blockIdx.x == 0 ? bounds : nullptr, gprefix);
    lds_sync();
    PF_MARK(2, 5);
    if (tid < ne) pos[tid] += cnt[tid];  // where this workgroup's first row of the expert goes
    for (int it = it0; it < it1; ++it) {
        if (it > it0) {
            lds_sync();
            for (int i = tid; i < NW * 256; i += NT) (&wpos[0][0])[i] = 0;
            lds_sync();
            e = it * NT + tid < n ? ids[it * NT + tid] : -1;
            live = e >= 0 && e < ne;
            rank = rank_piece(e, live);
            lds_sync();
        }
        if (tid < ne) {  // the piece's rows of the expert, split over the waves in wave order
            int q = pos[tid];
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int c = wpos[w][tid];
                wpos[w][tid] = q;
                q += c;
            }
            pos[tid] = q;
        }
        lds_sync();
        if (live) {
            const int p = it * NT + tid, q = wpos[wave][e] + rank;
            ids_dst[q] = p;
            ids_src1[q] = x_rows_per_tok == 1 ? p / k : p;
        }
    }
    PF_MARK(2, 1);
}

// ---- split activation images --------------------------------------------------------------------------------------
// The GEMM's A operand is the Q8_1 activation q8 * d8 as an exact pair of halves (hi = f16(q8 d8), lo = f16(q8 d8 - hi):
// a 7-bit integer times an f16 scale has at most 18 significant bits, two halves hold 22). Row layout, per 256-column
// superblock kb: 1024 bytes at kb * 1024, two 128-column halves of [hi 128 f16][lo 128 f16]; then at nb * 1024 + 32 kb
// the min-term sums [S_hi 8 f16][S_lo 8 f16], S_s = d8_s * sum(q8 of sub-block s). Within every 8 columns (and every
// 4 sums) the stored order is 0 2 1 3 4 6 5 7: the order in which the weight decoders below emit their B operand.
// Magnitudes are those of the reference's f16 Q8_1 fields (|q8 d8| <= amax, S within the f16 sum's range). A block of
// nothing but NaNs is stored as zeros in either form of image.
constexpr int kSbMain = 1024, kSbMin = 32;
__host__ __device__ constexpr int64_t split_row_bytes(int64_t ncols) { return ncols / 256 * (kSbMain + kSbMin); }
__device__ __forceinline__ int perm8(int k) { return (k & ~3) | ((k & 1) << 1) | ((k >> 1) & 1); }

// The split of eight codes of a block (four lanes per 32-value block, all active) with scale dh (an f16 value): lane
// q = 0 of the block also stores its min-term sums.
struct Q8Split {
    _Float16 hi[8], lo[8];  // in the stored order
    _Float16 shi, slo;      // the block's min-term sum (lane q = 0 of the block stores it)
};
__device__ __forceinline__ Q8Split q8_split_of(const int (&q)[8], float dh) {
    Q8Split r;
    int qsum = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        qsum += q[k];
        const float x = (float) q[k] * dh;  // exact
        const _Float16 h = (_Float16) x;
        r.hi[perm8(k)] = h;
        r.lo[perm8(k)] = (_Float16) (x - (float) h);
    }
    qsum = lanes_sum_i<4>(qsum);
    const float sv = dh * (float) qsum;  // exact in fp32
    r.shi = (_Float16) sv;
    r.slo = (_Float16) (sv - (float) r.shi);
    return r;
}
// byte offsets within an image row of the 8 columns at col (hi; lo at + 256) and of the block's min-term sums (hi;
// lo at + 16)
__device__ __forceinline__ uint32_t img_col_off(int col) {
    return (uint32_t) ((col >> 8) * kSbMain + ((col >> 7) & 1) * 512 + ((col & 127) >> 3) * 16);
}
__device__ __forceinline__ uint32_t img_sum_off(int ncols, int col) {
    return (uint32_t) ((ncols >> 8) * kSbMain + (col >> 8) * kSbMin + 2 * perm8((col >> 5) & 7));
}

// ---- int8 images (the int8 form of the GEMM, fns_mmq_i8.hpp) ---------------------------------------------------------
// Row layout, per 256-column superblock kb at kb * 320: the 256 int8 codes, the 8 block scales d8 (f32, f16 values), the
// min-term sums of the split image (same order). A row's codes, scales and sums define its split row and the other way
// round.
enum : int { kImgSplit = 0, kImgI8 = 1 };
constexpr int kI8Sb = 320, kI8Scale = 256, kI8Sum = 288;
__host__ __device__ constexpr int img_sb_bytes(int form) { return form == kImgI8 ? kI8Sb : kSbMain + kSbMin; }

// The scale as the images store it: rounded to f16, 0 for NaN.
__device__ __forceinline__ float image_scale(float d) { return half_to_float(float_to_half(fmaxf(d, 0.0f))); }

// The lane's part of a quantised block (8 codes at column col, a multiple of 8; all four lanes of the block active):
// put(byte offset within the row, value); the block's first lane also stores the scale and the sums.
template <class Put> __device__ __forceinline__ void i8_put(const Q8x8 &r, int col, Put put) {
    const uint32_t sb = (uint32_t) (col >> 8) * kI8Sb;
    uint32_t w[2] = {0, 0};
    int qsum = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        w[k / 4] |= (uint32_t) (uint8_t) (int8_t) r.q[k] << (8 * (k % 4));
        qsum += r.q[k];
    }
    put(sb + (col & 255), make_uint2(w[0], w[1]));
    qsum = lanes_sum_i<4>(qsum);
    if ((col & 31) == 0) {
        const int s = (col >> 5) & 7;
        const float dh = image_scale(r.d), sv = dh * (float) qsum;  // exact in fp32
        const _Float16 hi = (_Float16) sv, lo = (_Float16) (sv - (float) hi);
        put(sb + kI8Scale + 4 * s, __builtin_bit_cast(uint32_t, dh));
        put(sb + kI8Sum + 2 * perm8(s), __builtin_bit_cast(uint16_t, hi));
        put(sb + kI8Sum + 16 + 2 * perm8(s), __builtin_bit_cast(uint16_t, lo));
    }
}
template <class Put> __device__ __forceinline__ void split_put(const Q8x8 &q, int ncols, int col, Put put) {
    const Q8Split r = q8_split_of(q.q, image_scale(q.d));
    const uint32_t o = img_col_off(col);
    put(o, __builtin_bit_cast(uint4, r.hi));
    put(o + 256, __builtin_bit_cast(uint4, r.lo));
    if ((col & 31) == 0) {
        const uint32_t m = img_sum_off(ncols, col);
        put(m, __builtin_bit_cast(uint16_t, r.shi));
        put(m + 16, __builtin_bit_cast(uint16_t, r.slo));
    }
}
__device__ __forceinline__ void image_store(int form, const Q8x8 &q, uint8_t *row, int ncols, int col) {
    auto put = [&](uint32_t o, auto v) __attribute__((always_inline)) { *(decltype(v) *) (row + o) = v; };
    if (form == kImgI8) i8_put(q, col, put);
    else split_put(q, ncols, col, put);
}

// x [rows][ncols] f32 -> image rows with the reference's Q8_1 arithmetic; grid (rows, ceil(ncols / 2048)), 256 threads
// of 8 columns each (ncols % 256 == 0, so a block's 4 lanes are all in or all out).
__device__ __forceinline__ void quant_image8(const float *__restrict__ x, int ncols, int row, int col, int form,
                                             uint8_t *__restrict__ out, int64_t img_row_bytes) {
    const float *src = x + (size_t) row * ncols + col;
    const float4 x0 = *(const float4 *) src, x1 = *(const float4 *) (src + 4);
    const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    image_store(form, q8_1_x8(v), out + (size_t) row * img_row_bytes, ncols, col);
}
__global__ __launch_bounds__(256) void k_quant_image(const float *__restrict__ x, int ncols, int form,
                                                     uint8_t *__restrict__ out, int64_t img_row_bytes) {
    const int row = blockIdx.x, col = (blockIdx.y * 256 + threadIdx.x) * 8;
    if (col < ncols) quant_image8(x, ncols, row, col, form, out, img_row_bytes);
}

// RMSNorm of a row of at most 2048 C columns (fns_q8x8.hpp) with its Q8_1 blocks (xq null: none) and its image row, as
// rms_norm_q8_1 and k_quant_image give them, in one pass over x.
template <int C>
__global__ __launch_bounds__(256) void k_rms_norm_image(const float *__restrict__ x, const float *__restrict__ w,
                                                        float *__restrict__ out, uint8_t *__restrict__ xq, int n,
                                                        float eps, int64_t row_bytes, int form, uint8_t *__restrict__ img,
                                                        int64_t img_row_bytes) {
    __shared__ __align__(16) float xs[2048 * C];
    const size_t r = blockIdx.x;
    uint8_t *row = img + r * img_row_bytes;
    rms_norm_row<C>(x + r * n, w, out + r * n, xq ? xq + r * row_bytes : nullptr, n, eps, xs,
                    [&](const Q8x8 &q, int col) { image_store(form, q, row, n, col); });
}

// F16 guard of the act rows (reference src/kernels.cu:534-577), one wave per row of n columns (n % 256 == 0): the scale
// from the row's maximum, and only where it is not 1 the division in place and the row's image again (the GEMM epilogue
// has written the image of the undivided values, which is the same when it is 1). Bound by reading the rows once; the
// scale and the image were two launches (9.9 + 5.2 us at 6126 rows of 512).
__global__ __launch_bounds__(256) void k_guard_image(float *__restrict__ act, float *__restrict__ escale, int n, int rows,
                                                     int form, uint8_t *__restrict__ out, int64_t img_row_bytes) {
    const int row = blockIdx.x * (256 / kWave) + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (row >= rows) return;
    float *r = act + (size_t) row * n;
    float m = 0.0f;
#pragma unroll 2
    for (int i = 4 * lane; i < n; i += 4 * kWave) {
        const float4 v = *(const float4 *) (r + i);
        m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    }
    const float e = guard_scale(lanes_max<64>(m));
    if (lane == 0) escale[row] = e;
    if (e == 1.0f) return;  // (the whole wave)
    for (int i = 8 * lane; i < n; i += 8 * kWave) {  // a block's four lanes are all in or all out
        const float4 x0 = *(const float4 *) (r + i), x1 = *(const float4 *) (r + i + 4);
        const float v[8] = {x0.x / e, x0.y / e, x0.z / e, x0.w / e, x1.x / e, x1.y / e, x1.z / e, x1.w / e};
        *(float4 *) (r + i) = make_float4(v[0], v[1], v[2], v[3]);
        *(float4 *) (r + i + 4) = make_float4(v[4], v[5], v[6], v[7]);
        image_store(form, q8_1_x8(v), out + (size_t) row * img_row_bytes, n, i);
    }
}

// Router GEMM tiles and the split activation image of the same rows in one launch (the two only read x): workgroups
// [0, n_rt) are router tiles (tile (id % tiles_x, id / tiles_x)), the rest quantise two 2048-column pieces of x each,
// as k_quant_image does, so the image is built on the CUs the router tiles leave free.
template <bool BF16, bool TILE32>
__global__ __launch_bounds__(512) void k_router_image(const void *__restrict__ w, const float *__restrict__ bias,
                                                      const float *__restrict__ x, float *__restrict__ y, int ncols,
                                                      int nrows, int n_tok, int tiles_x, int n_rt,
                                                      int form, uint8_t *__restrict__ img, int64_t img_row_bytes,
                                                      int nxb) {
    PF_MARK(0, 0);
    const int id = blockIdx.x;
    if (id < n_rt) {
        if constexpr (TILE32) router_gemm_tile32<BF16>(w, bias, x, y, ncols, nrows, n_tok, id % tiles_x, id / tiles_x);
        else router_gemm_tile<BF16, true>(w, bias, x, y, ncols, nrows, n_tok, id % tiles_x, id / tiles_x);
        PF_MARK(0, 1);
        return;
    }
    const int item = 2 * (id - n_rt) + (int) threadIdx.x / 256;
    const int row = item / nxb, col = ((item % nxb) * 256 + (int) threadIdx.x % 256) * 8;
    if (item < nxb * n_tok && col < ncols) quant_image8(x, ncols, row, col, form, img, img_row_bytes);
    PF_MARK(0, 1);
}

// ---- grouped GEMM -------------------------------------------------------------------------------------------------
struct MmqArgs {
    const char *const *table;  // expert pointer table (null: dense, w_dense)
    const uint8_t *w_dense;
    int64_t off_a, off_b;      // byte offsets of the (gate) matrix and of the up matrix (GLU)
    int ncols, nrows;          // K (columns of W) and N (rows of W)
    int n_expert;
    const uint8_t *xpack;      // split activation image rows
    int64_t x_img;             // bytes per activation image row
    const int32_t *bounds;     // [n_expert + 1] (null: dense)
    const int32_t *gprefix;    // [2][n_expert + 1] group prefixes: 64-row groups, then the <= 32-row remainders
    int n_groups, n_cb;        // launch: groups (dense); weight row blocks per group
    const int32_t *src;        // sorted position -> activation image row (null: identity, dense only)
    const int32_t *dst_rows;   // sorted position -> output row (null: identity)
    int half;                  // item: 0 / 1 = that 32-row half of a 64-row group of the list, -1: the whole group
    int n_rows;                // dense: number of activation rows
    int dense_small;           // dense: 1 = groups of 32 activation rows (one tile), 0 = of 64
    int rows_first;            // dense: 1 = row blocks over the XCDs, all groups of a block in turn; 0 = groups over them
    int ksplit;                // dense, non-GLU: > 1 = the K range split into ksplit parts (blockIdx.y), part p's
    int64_t part_stride;       //   partial sums written at dst + p * part_stride floats
    float *dst;                // [out row][nrows] f32 (non-GLU)
    uint8_t *out_pack;         // GLU: act split image rows (by output row)
    int64_t out_img;
    int out_form;              // GLU: the form of the act image rows (kImg*)
    float *act_out;            // GLU: optional f32 act [out row][nrows]
    int *gdone;                // fused launch: per-group arrival counts (zeroed by the compaction kernel)
    int slot;                  // fused launch: the item's group's count
    int gwait;                 // fused launch: arrivals a down item waits for (its group's gate/up items)
    int spin_limit;            // fused launch: polls before a down item gives up (its outputs are then NaN)
    uint32_t *status;          // fused launch: sticky status word, kStatusTimeout once a wait gave up
};

// One dense matrix that rides in the expert launch (a layer's shared expert, of the routed experts' type): its groups
// of 64 activation rows x row blocks take the first workgroups of the grid. n_rows = 0: none.
struct MmqShared {
    const uint8_t *w;
    int64_t off_b;             // GLU: the up matrix from w (the gate)
    int ncols, nrows, n_rows;
    const uint8_t *xpack;      // activation image rows (x_img bytes each), row t of every group in order
    int64_t x_img;
    float *dst;                // non-GLU
    uint8_t *out_pack;         // GLU
    int64_t out_img;
    int out_form;
    int n_cb, items;           // launch: row blocks per group; workgroups of the grid it takes (a multiple of kXcds)
    int may_halve;             // launch (with or without such a matrix): the device looks whether it runs in halves
};

// Weight fragments of one 256-value block for one lane: the header (scales, d) and the codes of column groups
// kg = 2 h and 2 h + 1 (h = lane / 32) of every sub-block - 16 contiguous bytes per code array, one load each.
template <int T> struct WFrag;
template <> struct WFrag<T_Q4_K> { uint4 h; uint4 q[4]; };
template <> struct WFrag<T_Q5_K> { uint4 h; uint4 q[4]; uint4 qh; };
template <> struct WFrag<T_Q6_K> { uint4 ql[4]; uint4 qh[2]; uint4 sc; uint32_t d; };
template <> struct WFrag<T_Q3_K> { uint4 qs[2]; uint4 hm; uint4 tail; };
// Q8_0 (8 blocks of 34 bytes per 256 values): the 16 code bytes of column groups 2 h, 2 h + 1 and the f16 d of
// every block (low 16 bits)
template <> struct WFrag<T_Q8_0> { uint4 q[8]; uint32_t d[8]; };
// IQ formats (lane half h, its two column groups of every 32-value sub-block; see decode):
//   IQ4_XS : header (d, scales_h, scales_l) and qs bytes 8 h .. 8 h + 7 of each sub-block
//   IQ3_XXS: d, index bytes 4 h .. 4 h + 3 of each sub-block, the sub-block's aux word (signs, scale)
//   IQ3_S  : d, qh (8 bytes), scales (4 bytes), index bytes 4 h .. 4 h + 3 and sign bytes 2 h, 2 h + 1 per sub-block
//   IQ2_S  : d, qh, scales, the 16 index bytes and 16 sign bytes of each half block (lanes use 2 of every 4)
template <> struct WFrag<T_IQ4_XS> { uint2 h; uint2 q[8]; };
template <> struct WFrag<T_IQ3_XXS> { uint32_t d; uint32_t idx[8]; uint4 aux[2]; };
template <> struct WFrag<T_IQ3_S> { uint32_t d, sc; uint2 qh; uint32_t idx[8], sg[8]; };
template <> struct WFrag<T_IQ2_S> { uint32_t d; uint2 qh, sc; uint4 idx[2], sg[2]; };

// Buffer loads: a uniform base in a resource (SGPRs), a 32-bit per-lane offset and a uniform offset - no 64-bit
// address arithmetic per load. (Unaligned dword access is enabled on the platform, as for the plain global loads.)
// A resource reaches kRsrcBytes from its base (a read past that gives zeros), so one launch's scattered image rows lie
// within that many bytes (image_tokens), image rows in order are read from their group's first and weight rows from the
// workgroup's first.
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int64_t kRsrcBytes = 0x7FFFFFFF;
__device__ __forceinline__ Rsrc rsrc_of(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int) kRsrcBytes, 0x00020000);
}
// Activation image rows of a group whose first sorted row is seg: a.src names them from the image's start; without it they
// are rows seg, seg + 1, ... and are counted from seg.
__device__ __forceinline__ Rsrc image_rsrc(const uint8_t *img, int64_t row_bytes, bool listed, int seg) {
    return rsrc_of(listed ? img : img + seg * row_bytes);
}
__device__ __forceinline__ uint4 bload16(Rsrc r, uint32_t vo, uint32_t so) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint2 bload8(Rsrc r, uint32_t vo, uint32_t so) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0);
    return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ uint32_t bload4(Rsrc r, uint32_t vo, uint32_t so) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0);
}
__device__ __forceinline__ uint32_t bload2(Rsrc r, uint32_t vo, uint32_t so) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, vo, so, 0);
}

// Part P (compile time) of the fragment of the block at (vo + so) from r; vc = vo + 16 h selects the lane's code
// bytes. Part 0: the header and the codes of sub-blocks 0-3; part 1: the codes of sub-blocks 4-7.
template <int T, int P>
__device__ __forceinline__ void wfrag_load(Rsrc r, uint32_t vo, uint32_t vc, uint32_t so, WFrag<T> &f) {
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        constexpr int qoff = T == T_Q4_K ? 16 : 48;
        if constexpr (P == 0) {
            f.h = bload16(r, vo, so);
            if constexpr (T == T_Q5_K) f.qh = bload16(r, vc, so + 16);
        }
#pragma unroll
        for (int g = 2 * P; g < 2 * P + 2; ++g) f.q[g] = bload16(r, vc, so + qoff + 32 * g);
    } else if constexpr (T == T_Q6_K) {
        f.ql[2 * P] = bload16(r, vc, so + 64 * P);
        f.ql[2 * P + 1] = bload16(r, vc, so + 64 * P + 32);
        f.qh[P] = bload16(r, vc, so + 128 + 32 * P);
        if constexpr (P == 0) {
            f.sc = bload16(r, vo, so + 192);
            f.d = __builtin_amdgcn_raw_buffer_load_b16(r, vo, so + 208, 0);
        }
    } else if constexpr (T == T_Q3_K) {
        if constexpr (P == 0) {
            f.hm = bload16(r, vc, so);
            f.tail = bload16(r, vo, so + 94);  // scales[12] at +2, d at +14
        }
        f.qs[P] = bload16(r, vc, so + 32 + 32 * P);
    } else if constexpr (T == T_Q8_0) {  // block s at 34 s: d @0, qs @2 (vc - vo = 16 h selects the lane's 16 bytes)
#pragma unroll
        for (int b = 4 * P; b < 4 * P + 4; ++b) {
            f.q[b] = bload16(r, vc, so + 34 * b + 2);
            f.d[b] = bload2(r, vo, so + 34 * b);
        }
    } else if constexpr (T == T_IQ4_XS) {  // d @0, scales_h @2, scales_l @4, qs @8 (16 per sub-block)
        const uint32_t vq = vo + ((vc - vo) >> 1);  // + 8 h
        if constexpr (P == 0) f.h = bload8(r, vo, so);
#pragma unroll
        for (int ib = 4 * P; ib < 4 * P + 4; ++ib) f.q[ib] = bload8(r, vq, so + 8 + 16 * ib);
    } else if constexpr (T == T_IQ3_XXS) {  // d @0, index bytes @2 (8 per sub-block), aux words @66
        const uint32_t vq = vo + ((vc - vo) >> 2);  // + 4 h
        if constexpr (P == 0) f.d = bload2(r, vo, so);
#pragma unroll
        for (int ib = 4 * P; ib < 4 * P + 4; ++ib) f.idx[ib] = bload4(r, vq, so + 2 + 8 * ib);
        f.aux[P] = bload16(r, vo, so + 66 + 16 * P);
    } else if constexpr (T == T_IQ3_S) {  // d @0, qs @2 (8 per sub-block), qh @66, signs @74 (4 per sub-block), scales @106
        const uint32_t vq = vo + ((vc - vo) >> 2), vs = vo + ((vc - vo) >> 3);  // + 4 h, + 2 h
        if constexpr (P == 0) {
            f.d = bload2(r, vo, so);
            f.qh = bload8(r, vo, so + 66);
            f.sc = bload4(r, vo, so + 106);
        }
#pragma unroll
        for (int ib = 4 * P; ib < 4 * P + 4; ++ib) {
            f.idx[ib] = bload4(r, vq, so + 2 + 8 * ib);
            f.sg[ib] = bload2(r, vs, so + 74 + 4 * ib);
        }
    } else {  // IQ2_S: d @0, index bytes @2 (4 per sub-block), sign bytes @34 (4 per sub-block), qh @66, scales @74
        if constexpr (P == 0) {
            f.d = bload2(r, vo, so);
            f.qh = bload8(r, vo, so + 66);
            f.sc = bload8(r, vo, so + 74);
        }
        f.idx[P] = bload16(r, vo, so + 2 + 16 * P);
        f.sg[P] = bload16(r, vo, so + 34 + 16 * P);
    }
}
// vector loads issued by part P of wfrag_load for one stream
template <int T, int P> constexpr int wfrag_loads() {
    return T == T_Q4_K    ? (P ? 2 : 3)
           : T == T_Q5_K  ? (P ? 2 : 4)
           : T == T_Q6_K  ? (P ? 3 : 5)
           : T == T_Q3_K  ? (P ? 1 : 3)
           : T == T_Q8_0  ? 8
           : T == T_IQ4_XS ? (P ? 4 : 5)
           : T == T_IQ3_XXS ? (P ? 5 : 6)
           : T == T_IQ3_S ? (P ? 8 : 11)
                          : (P ? 2 : 5);  // IQ2_S
}
// the 8 code bytes of column group 2 h + p (p compile time) from a 16-byte code array
__device__ __forceinline__ uint2 half8(const uint4 &v, int p) { return p ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y); }

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2 splat(_Float16 v) { return h2{v, v}; }
// bytes b0..b3 (< 1024 each) of w -> halves (1024 + b0, 1024 + b2) and (1024 + b1, 1024 + b3): 0x6400 is 1024.0
__device__ __forceinline__ h2 biased02(uint32_t w) { return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04020400u)); }
__device__ __forceinline__ h2 biased13(uint32_t w) { return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04030401u)); }
__device__ __forceinline__ h2 fma2(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ v8h cat4(h2 a, h2 b, h2 c, h2 d) {
    return __builtin_bit_cast(v8h, make_uint4(as_u(a), as_u(b), as_u(c), as_u(d)));
}
// codes bytes (x = columns 0-3, y = columns 4-7 of the lane) times a scale: exact products (|code * scale| <= 2048)
__device__ __forceinline__ v8h scaled8(uint32_t x, uint32_t y, h2 sc, h2 bias) {  // (1024 + c) sc + bias, bias = -1024 sc
    return cat4(fma2(biased02(x), sc, bias), fma2(biased13(x), sc, bias), fma2(biased02(y), sc, bias),
                fma2(biased13(y), sc, bias));
}
__device__ __forceinline__ v8h centred8(uint32_t x, uint32_t y, h2 off, h2 sc) {  // ((1024 + c) - off) * sc
    return cat4((biased02(x) - off) * sc, (biased13(x) - off) * sc, (biased02(y) - off) * sc,
                (biased13(y) - off) * sc);
}

// B operand(s) of sub-block s, column group kg = 2 h + p (s, p compile time) for this lane: B[k][row] = integer code x
// integer scale as f16 (Q6_K: two operands, scale split as 16 (sc >> 4) + (sc & 15), each product exact). The block's
// float scale d (and dmin) are applied per superblock. on = (d != 0): a block with d = 0 contributes d * (...) = 0
// whatever its codes.
template <int T> constexpr int kNumB = T == T_Q6_K || T == T_IQ4_XS || T == T_Q8_0 ? 2 : 1;
template <int T> struct BOp { v8h b[kNumB<T>]; };
template <int T>
__device__ __forceinline__ BOp<T> decode(const WFrag<T> &f, int s, int p, int h, bool on, const uint32_t *grid);

// (sc_s, sc_s) as f16 and its bias -1024 sc_s for sub-block s (compile time) of a Q4_K / Q5_K block; on = 0: zeros.
// The 6-bit scales are unpacked four at a time (ggml get_scale_min_k4), byte s placed twice next to 0x64 (1024.0).
__device__ __forceinline__ void k4_scale2(const uint4 &h, int s, bool on, h2 &s2, h2 &bias) {
    const uint32_t w = s < 4 ? (h.y & 0x3F3F3F3Fu) : ((h.w & kLo4) | ((h.y >> 2) & 0x30303030u));
    const uint32_t i = (uint32_t) (s & 3);
    s2 = as_h2(__builtin_amdgcn_perm(0x64646464u, on ? w : 0u, 0x04000400u | (i << 16) | i)) - splat((_Float16) 1024.0f);
    bias = s2 * splat((_Float16) -1024.0f);
}
template <> __device__ __forceinline__ BOp<T_Q4_K> decode<T_Q4_K>(const WFrag<T_Q4_K> &f, int s, int p, int, bool on, const uint32_t *) {
    const uint2 q = half8(f.q[s >> 1], p);
    const int sh = 4 * (s & 1);
    h2 s2, bias;
    k4_scale2(f.h, s, on, s2, bias);
    BOp<T_Q4_K> r;
    r.b[0] = scaled8((q.x >> sh) & kLo4, (q.y >> sh) & kLo4, s2, bias);
    return r;
}
template <> __device__ __forceinline__ BOp<T_Q5_K> decode<T_Q5_K>(const WFrag<T_Q5_K> &f, int s, int p, int, bool on, const uint32_t *) {
    const uint2 q = half8(f.q[s >> 1], p), qh = half8(f.qh, p);
    const int sh = 4 * (s & 1);
    h2 s2, bias;
    k4_scale2(f.h, s, on, s2, bias);
    BOp<T_Q5_K> r;
    r.b[0] = scaled8(((q.x >> sh) & kLo4) | (((qh.x >> s) & 0x01010101u) << 4),
                     ((q.y >> sh) & kLo4) | (((qh.y >> s) & 0x01010101u) << 4), s2, bias);
    return r;
}
// Q6_K sub-block s: n = s / 4, qq = s % 4: ql[64 n + 32 (qq & 1) + l] nibble qq >> 1, qh[32 n + l] bits 2 qq,
// value - 32; int8 scale of group 8 n + 2 qq + (l >= 16), i.e. + h for column groups 2 h, 2 h + 1.
template <> __device__ __forceinline__ BOp<T_Q6_K> decode<T_Q6_K>(const WFrag<T_Q6_K> &f, int s, int p, int h, bool on, const uint32_t *) {
    const int n = s >> 2, qq = s & 3;
    const uint2 ql = half8(f.ql[2 * n + (qq & 1)], p), qh = half8(f.qh[n], p);
    const int shl = 4 * (qq >> 1), shh = 2 * qq;
    const uint32_t x = ((ql.x >> shl) & kLo4) | (((qh.x >> shh) & 0x03030303u) << 4);
    const uint32_t y = ((ql.y >> shl) & kLo4) | (((qh.y >> shh) & 0x03030303u) << 4);
    const int g0 = 8 * n + 2 * qq;  // even: both groups in one word
    const uint32_t w0 = word(f.sc, g0 >> 2);
    const int sc = on ? (int) (int8_t) ((w0 >> (8 * ((g0 & 3) + h))) & 0xffu) : 0;
    const h2 off = splat((_Float16) 1056.0f);
    BOp<T_Q6_K> r;
    r.b[0] = centred8(x, y, off, splat((_Float16) (16 * (sc >> 4))));
    r.b[1] = centred8(x, y, off, splat((_Float16) (sc & 15)));
    return r;
}
// Q3_K sub-block s: n = s / 4, j = s % 4: qs[32 n + l] bits 2 j, hmask[l] bit 4 n + j (clear: -4); scale groups
// 8 n + 2 j + (l >= 16), 6-bit value - 32 (low nibbles in scales[0..7], high bit pairs in scales[8..11]).
template <> __device__ __forceinline__ BOp<T_Q3_K> decode<T_Q3_K>(const WFrag<T_Q3_K> &f, int s, int p, int h, bool on, const uint32_t *) {
    const int n = s >> 2, j = s & 3;
    const uint2 q = half8(f.qs[n], p), hm = half8(f.hm, p);
    const int hs = 4 * n + j;
    const uint32_t x = ((q.x >> (2 * j)) & 0x03030303u) | (((hm.x >> hs) & 0x01010101u) << 2);
    const uint32_t y = ((q.y >> (2 * j)) & 0x03030303u) | (((hm.y >> hs) & 0x01010101u) << 2);
    // tail = block bytes 94..109: scales[i] is tail byte 2 + i
    const uint32_t hi_w = (f.tail.z >> 16) | (f.tail.w << 16);  // scales[8..11]
    int scv[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int g = 8 * n + 2 * j + u;
        const int lb = (g & 7) + 2;  // tail byte of scales[g & 7]
        const uint32_t lw = lb < 4 ? f.tail.x : lb < 8 ? f.tail.y : f.tail.z;
        const uint32_t b = (lw >> (8 * (lb & 3))) & 0xffu;
        const uint32_t lo4 = g < 8 ? (b & 0xFu) : (b >> 4);
        const uint32_t hi2 = (((hi_w >> (8 * (g & 3))) & 0xffu) >> (2 * (g >> 2))) & 3u;
        scv[u] = (int) (lo4 | (hi2 << 4)) - 32;
    }
    const int sc = on ? (h == 0 ? scv[0] : scv[1]) : 0;
    BOp<T_Q3_K> r;
    r.b[0] = centred8(x, y, splat((_Float16) 1028.0f), splat((_Float16) sc));
    return r;
}

// IQ formats: B = signed codebook value x integer sub-block scale, exact in f16 (|B| <= 2048, or split in two
// operands), the rest of the float scale in blk_d: IQ4_XS kv * (ls - 32) (split as 4 (s >> 2) + (s & 3)) with d;
// IQ3_XXS g * (2 ls + 1) with d / 4; IQ3_S g * (2 sc + 1) with d; IQ2_S g * (2 ls + 1) with d / 8 - the products of
// the dequantisers' scales (ggml-quants.c dequantize_row_iq*). Codebook entries come from the LDS copy `grid` of the
// format's table. Signed values are biased by 128 (byte ^ 0x80) for the 1024 + byte conversion.
__device__ __forceinline__ v8h signed_scaled8(uint32_t x, uint32_t y, int sc, bool on) {  // x, y: 4 int8 each
    const _Float16 s = (_Float16) (on ? sc : 0);
    return scaled8(x ^ 0x80808080u, y ^ 0x80808080u, splat(s), splat((_Float16) -1152.0f * s));
}
template <> __device__ __forceinline__ BOp<T_IQ4_XS> decode<T_IQ4_XS>(const WFrag<T_IQ4_XS> &f, int s, int p, int,
                                                                      bool on, const uint32_t *) {
    // column group p: the low (p = 0) or high (p = 1) nibbles of the lane's 8 bytes, values 8 h .. 8 h + 7 (+ 16 p)
    const uint32_t x = iq4nl_values((f.q[s].x >> (4 * p)) & kLo4), y = iq4nl_values((f.q[s].y >> (4 * p)) & kLo4);
    const int ls = (int) (((f.h.y >> (4 * s)) & 0xfu) | (((f.h.x >> (16 + 2 * s)) & 3u) << 4)) - 32;
    BOp<T_IQ4_XS> r;
    r.b[0] = signed_scaled8(x, y, 4 * (ls >> 2), on);
    r.b[1] = signed_scaled8(x, y, ls & 3, on);
    return r;
}
template <> __device__ __forceinline__ BOp<T_IQ3_XXS> decode<T_IQ3_XXS>(const WFrag<T_IQ3_XXS> &f, int s, int p, int h,
                                                                        bool on, const uint32_t *grid) {
    const int g = 2 * h + p;  // column group: index bytes 2 g, 2 g + 1; signs (aux >> 7 g) & 127
    const uint32_t aux = word(f.aux[s >> 2], s & 3), idx = f.idx[s] >> (16 * p);
    const uint32_t sg = ksigns((aux >> (7 * g)) & 127u);
    const int x = signed_grid(grid[idx & 0xffu], spread4(sg & 0xfu));
    const int y = signed_grid(grid[(idx >> 8) & 0xffu], spread4(sg >> 4));
    BOp<T_IQ3_XXS> r;
    r.b[0] = signed_scaled8((uint32_t) x, (uint32_t) y, 2 * (int) (aux >> 28) + 1, on);
    return r;
}
template <> __device__ __forceinline__ BOp<T_IQ3_S> decode<T_IQ3_S>(const WFrag<T_IQ3_S> &f, int s, int p, int h,
                                                                    bool on, const uint32_t *grid) {
    const int g = 2 * h + p;  // codebook entries 2 g, 2 g + 1 of the sub-block (9-bit indices), sign byte g
    const uint32_t qh = (s < 4 ? f.qh.x : f.qh.y) >> (8 * (s & 3)), idx = f.idx[s] >> (16 * p);
    const uint32_t i0 = (idx & 0xffu) | (((qh >> (2 * g)) & 1u) << 8);
    const uint32_t i1 = ((idx >> 8) & 0xffu) | (((qh >> (2 * g + 1)) & 1u) << 8);
    const uint32_t sb = (f.sg[s] >> (8 * p)) & 0xffu;
    const int x = signed_grid(grid[i0], spread4(sb & 0xfu)), y = signed_grid(grid[i1], spread4(sb >> 4));
    BOp<T_IQ3_S> r;
    r.b[0] = signed_scaled8((uint32_t) x, (uint32_t) y, 2 * (int) ((f.sc >> (4 * s)) & 0xfu) + 1, on);
    return r;
}
template <> __device__ __forceinline__ BOp<T_IQ2_S> decode<T_IQ2_S>(const WFrag<T_IQ2_S> &f, int s, int p, int h,
                                                                    bool on, const uint32_t *grid) {
    const int g = 2 * h + p;  // codebook entry g of the sub-block (10-bit index, 8 values), sign byte g
    const uint32_t idx = word(f.idx[s >> 2], s & 3), sgw = word(f.sg[s >> 2], s & 3);
    const uint32_t qh = (s < 4 ? f.qh.x : f.qh.y) >> (8 * (s & 3)), sc = (s < 4 ? f.sc.x : f.sc.y) >> (8 * (s & 3));
    const uint32_t gi = ((idx >> (8 * g)) & 0xffu) | (((qh >> (2 * g)) & 3u) << 8);
    const uint32_t sb = (sgw >> (8 * g)) & 0xffu;
    const int x = signed_grid(grid[2 * gi], spread4(sb & 0xfu)), y = signed_grid(grid[2 * gi + 1], spread4(sb >> 4));
    BOp<T_IQ2_S> r;
    r.b[0] = signed_scaled8((uint32_t) x, (uint32_t) y, 2 * (int) ((sc >> (4 * h)) & 0xfu) + 1, on);
    return r;
}

// Q8_0: B = code * d split into two f16 operands, hi = f16(code d) and lo = f16(code d - hi) (an fma in f16): code d
// has at most 19 significant bits and hi + lo holds 22, so the pair is the product exactly when lo is a normal f16
// (|code d| >= 2^-3); for smaller products lo is rounded to a multiple of 2^-24 (an absolute error of at most 2^-25
// per weight). The block scale is then inside the operands and the superblock unit is 1. Codes are signed bytes:
// (1024 + (c ^ 0x80)) - 1152. Weights must stay below the f16 range (|code d| <= 65504), as they do in a Q8_0 block.
template <> __device__ __forceinline__ BOp<T_Q8_0> decode<T_Q8_0>(const WFrag<T_Q8_0> &f, int s, int p, int, bool, const uint32_t *) {
    const uint2 q = half8(f.q[s], p);
    const uint32_t x = q.x ^ 0x80808080u, y = q.y ^ 0x80808080u;
    const h2 off = splat((_Float16) 1152.0f), d2 = as_h2((f.d[s] & 0xffffu) * 0x10001u);
    const h2 c[4] = {biased02(x) - off, biased13(x) - off, biased02(y) - off, biased13(y) - off};
    h2 hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        hi[i] = c[i] * d2;
        lo[i] = fma2(c[i], d2, -hi[i]);
    }
    BOp<T_Q8_0> r;
    r.b[0] = cat4(hi[0], hi[1], hi[2], hi[3]);
    r.b[1] = cat4(lo[0], lo[1], lo[2], lo[3]);
    return r;
}

// Per-superblock float scales of this lane's row: d, and dmin for Q4_K / Q5_K.
template <int T> __device__ __forceinline__ float blk_d(const WFrag<T> &f) {
    if constexpr (T == T_Q4_K || T == T_Q5_K) return half_to_float(f.h.x & 0xffffu);
    else if constexpr (T == T_Q8_0) return 1.0f;  // the block scales are inside the B operands
    else if constexpr (T == T_Q6_K) return half_to_float(f.d);
    else if constexpr (T == T_Q3_K) return half_to_float(f.tail.w >> 16);
    else if constexpr (T == T_IQ4_XS) return half_to_float(f.h.x & 0xffffu);
    else if constexpr (T == T_IQ3_XXS) return 0.25f * half_to_float(f.d & 0xffffu);
    else if constexpr (T == T_IQ3_S) return half_to_float(f.d & 0xffffu);
    else return 0.125f * half_to_float(f.d & 0xffffu);  // IQ2_S
}
// The A piece (8 columns, 16 bytes of a half-superblock chunk row) of step i for lane half hh: sub-block i / 2,
// column group 2 hh + i % 2 (the decoders above emit those), or for IQ4_XS group 2 (i % 2) + hh (its lane half reads
// 8 bytes of both nibbles: values 8 hh .. 8 hh + 7 and 16 + 8 hh ..).
template <int T> __device__ __forceinline__ int a_piece(int i, int hh) {
    return T == T_IQ4_XS ? 4 * (i >> 1) + 2 * (i & 1) + hh : 4 * (i >> 1) + 2 * hh + (i & 1);
}
// LDS words of the format's codebook (IQ2_S: two words per entry)
template <int T> constexpr int kGridWords = T == T_IQ3_XXS ? 256 : T == T_IQ3_S ? 512 : T == T_IQ2_S ? 2048 : 0;
// Q4_K / Q5_K min term operand: B[k][row] = m_s against the A operand [S_hi 8 | S_lo 8] (lane half h holds k = 8 h ..
// 8 h + 7), both halves the 8 mins in the stored sum order 0 2 1 3 4 6 5 7.
template <int T> __device__ __forceinline__ v8h min_b(const WFrag<T> &f) {
    const uint32_t m_lo = f.h.z & 0x3F3F3F3Fu;                                         // m[0..3]
    const uint32_t m_hi = ((f.h.w >> 4) & kLo4) | ((f.h.z >> 2) & 0x30303030u);       // m[4..7]
    const h2 off = splat((_Float16) 1024.0f);
    return cat4(biased02(m_lo) - off, biased13(m_lo) - off, biased02(m_hi) - off, biased13(m_hi) - off);
}

// LDS of one workgroup (static, distinct objects, so the compiler can tell the chunk being filled by LDS-DMA from the
// one being read and puts no wait between them): the half-superblock activation chunks [rows][512] (hi, lo)
// double-buffered, with the 16-byte pieces of row r stored at piece index p ^ (r % 16) so that the 16 rows of an
// A-fragment read quarter hit distinct banks; the superblock min-term sums [rows][32]. 66 KB for 64 rows: two
// workgroups per CU.
constexpr int kRowA = 512, kRowS = 32;

// 1 / (1 + e^-g); 0 for g -> -inf (the exponential saturates to +inf), 1 for g -> +inf
__device__ __forceinline__ float silu_rcp(float g) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * 1.4426950408889634f));
}

__device__ __forceinline__ v16f mfma32(v8h a, v8h b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Workgroup barrier for LDS filled by LDS-DMA: the DMA data is complete once this wave's vmcnt wait before it retires
// (waits placed by the caller: __syncthreads' fence would also wait for the weight loads still in flight). This
// wave's own LDS reads must have returned (lgkmcnt 0) before the next DMA into the buffer may start, and the asm's
// memory clobber keeps the compiler from moving LDS accesses across it (the s_barrier builtin is not a memory op).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef __attribute__((address_space(3))) void *LdsPtr;
// 16 bytes per lane from r at (vo + so) into LDS at dst + 16 lane (dst wave-uniform); CPOL: cache-policy bits
template <int CPOL = 0>
__device__ __forceinline__ void dma16(Rsrc r, void *dst, uint32_t vo, uint32_t so) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsPtr) dst, 16, vo, so, 0, CPOL);
}

// ---- the fused gate/up + down launch: per-group arrivals --------------------------------------------------------
// A gate/up item stores its act image rows device-coherent (sc1: written through to memory, so no other XCD's L2 can
// serve an older copy), waits for the stores to complete and then counts its arrival on the group's counter; a down
// item of the group polls the counter (device-scope loads) until every gate/up item of the group has arrived and then
// reads the act rows with device-scope (sc1) loads. No fence is involved: the order comes from the completed stores
// before the arrival, as in the decode layer's exchange.
constexpr int kCpolDevice = 16;           // sc1
constexpr uint32_t kStatusTimeout = 1u;   // FNS_STATUS_EXCHANGE_TIMEOUT
__device__ __forceinline__ void image_store_dev(int form, const float (&v)[8], Rsrc r, uint32_t row_off, int ncols, int col,
                                                bool store) {
    const Q8x8 q = q8_1_x8(v);
    if (!store) return;
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    auto put = [&](uint32_t o, auto w) __attribute__((always_inline)) {
        const uint32_t at = row_off + o;
        if constexpr (sizeof w == 16) __builtin_amdgcn_raw_buffer_store_b128(v4u{w.x, w.y, w.z, w.w}, r, at, 0, kCpolDevice);
        else if constexpr (sizeof w == 8) __builtin_amdgcn_raw_buffer_store_b64(v2u{w.x, w.y}, r, at, 0, kCpolDevice);
        else if constexpr (sizeof w == 4) __builtin_amdgcn_raw_buffer_store_b32(w, r, at, 0, kCpolDevice);
        else __builtin_amdgcn_raw_buffer_store_b16(w, r, at, 0, kCpolDevice);
    };
    if (form == kImgI8) i8_put(q, col, put);
    else split_put(q, ncols, col, put);
}
// thread 0 polls the group's arrival count (bounded); true for every thread when the wait gave up
__device__ __forceinline__ bool wait_group(const MmqArgs &a, int slot, int *flag) {
    if (threadIdx.x == 0) {
        int spins = 0, fail = 0;
        while (__hip_atomic_load(a.gdone + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < a.gwait) {
            if (++spins > a.spin_limit) {
                fail = 1;
                __hip_atomic_fetch_or(a.status, kStatusTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        *flag = fail;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*flag) != 0;
}

// One workgroup = 4 waves x two 32-row weight streams x up to 32 NT routed activation rows of one expert (NT = 2: the
// 64-row groups and remainders > 32 rows; NT = 1: remainders <= 32 rows). GLU: stream 0 is the gate row, stream 1 the
// same up row (128 rows per workgroup); otherwise the streams are rows r and r + 128 (256).
// v_mfma_f32_32x32x16_f16: A = 32 activation rows x 16 columns, B = 16 columns x 32 weight rows; the lane that owns
// weight row j = lane % 32 decodes row j's codes and scales itself (column groups 2 h, 2 h + 1 of each sub-block,
// h = lane / 32), and holds the outputs of row j for 16 of the 32 tokens.
// LDS of one workgroup, sized for the 64-row groups (the 32-row groups use the first half of each array).
struct MmqLds {
    uint8_t (&a0)[kMmqTok * kRowA];
    uint8_t (&a1)[kMmqTok * kRowA];
    uint8_t (&s)[kMmqTok * kRowS];
    int (&src)[kMmqTok];
    int (&dst)[kMmqTok];
    int (&grp)[4];  // the group's expert, first sorted row and row count
    uint32_t *grid;  // IQ3_XXS / IQ3_S / IQ2_S: the codebook (kGridWords words)
};

// Expert e, first sorted row seg and row count cnt (1 .. 32 NT) of group g; false: the group does not exist.
template <int NT>
__device__ __forceinline__ bool group_rows(const MmqArgs &a, int g, int (&grp)[4], int &e, int &seg, int &cnt) {
    const int tid = threadIdx.x;
    // which expert / rows of activations: thread t < n_expert tests whether group g is expert t's (gp[t] <= g <
    // gp[t + 1]); all the prefix loads are independent, one round trip, and the one match publishes through LDS
    e = seg = cnt = 0;
    if (a.bounds) {
        const bool rest = NT == 1 && a.half < 0;  // the list of the <= 32-row remainders
        const int32_t *gp = rest ? a.gprefix + a.n_expert + 1 : a.gprefix;
        if (g >= gp[a.n_expert]) return false;
        if (tid < a.n_expert) {
            const int g0 = gp[tid], g1 = gp[tid + 1], b0 = a.bounds[tid], b1 = a.bounds[tid + 1];
            if (g0 <= g && g < g1) {
                int c, sg;
                if (rest) {  // the expert's last rows: n_e % 64 of them
                    c = (b1 - b0) % kMmqTok;
                    sg = b1 - c;
                } else {  // a group, or 32 rows of it
                    sg = b0 + (g - g0) * kMmqTok + (NT == 1 ? 32 * a.half : 0);
                    c = min(32 * NT, b1 - sg);
                }
                grp[0] = tid;
                grp[1] = sg;
                grp[2] = c;
            }
        }
        __syncthreads();
        e = __builtin_amdgcn_readfirstlane(grp[0]);
        seg = __builtin_amdgcn_readfirstlane(grp[1]);
        cnt = __builtin_amdgcn_readfirstlane(grp[2]);
    } else {
        seg = g * 32 * NT;
        cnt = min(32 * NT, a.n_rows - seg);
    }
    return cnt > 0;
}

// The matrix of expert e (or the dense one), as a scalar, so the weight buffer resources stay in SGPRs.
__device__ __forceinline__ const uint8_t *expert_base(const MmqArgs &a, int e) {
    const uint64_t w = (uint64_t) (a.table ? (const uint8_t *) gload<const char *>((const uint8_t *) (a.table + e)) : a.w_dense);
    return (const uint8_t *) (((uint64_t) __builtin_amdgcn_readfirstlane((uint32_t) (w >> 32)) << 32) |
                              (uint32_t) __builtin_amdgcn_readfirstlane((uint32_t) w));
}

// Output rows of a finished group: (token i, weight row row0 and row0 + 128) of acc[t][m][r], i = 32 t + 8 (r / 4) + 4 hh + r % 4
template <int NT>
__device__ __forceinline__ void store_group(const MmqArgs &a, const v16f (&acc)[NT][2], const int *dst, int cnt, int row0,
                                            int hh, int part, bool failed) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = t * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
            if (i < cnt) {
                float *o = a.dst + (size_t) part * a.part_stride + (size_t) dst[i] * a.nrows;
                if (row0 < a.nrows) o[row0] = failed ? __builtin_nanf("") : acc[t][0][r];
                if (row0 + 128 < a.nrows) o[row0 + 128] = failed ? __builtin_nanf("") : acc[t][1][r];
            }
        }
}

// act = up * silu(gate) of a finished GLU group (reference src/ggml/ggml_mmvq.cu:240-247 epilogue with zero biases;
// silu(g) = g / (1 + e^-g) from the hardware exp2 and reciprocal, about 2 ulp) into LDS as [token][64 rows] f32 per wave
// pair: waves 0-1 in t0, waves 2-3 in t1, row stride kActRow floats (16-byte aligned rows).
constexpr int kActRow = 68;
template <int NT>
__device__ __forceinline__ void act_to_lds(const v16f (&acc)[NT][2], float *t0, float *t1, int wave, int jl, int hh) {
    float *act = wave < 2 ? t0 : t1;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = t * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
            const float g = acc[t][0][r] + 0.0f;
            act[i * kActRow + (wave & 1) * 32 + jl] = (acc[t][1][r] + 0.0f) * (g * silu_rcp(g));
        }
}
// Then the Q8_1 blocks (token, 32 rows), 4 lanes per block and 8 values per lane: sink(i, col, live, v) for token i and
// act column col; the 4 lanes of a block are live together. The f32 act rows too when act_out asks for them.
template <class Sink>
__device__ __forceinline__ void act_blocks(const MmqArgs &a, const float *t0, const float *t1, const int *dst, int cnt, int wb,
                                           int wave, int lane, Sink sink) {
    for (int p0 = wave * 16; p0 < 4 * cnt; p0 += 16 * kMmqWaves) {  // wave-uniform trip count
        const int p = p0 + lane / 4, q = lane % 4;
        const int i = p < 4 * cnt ? p / 4 : 0, blk = p % 4;
        const int col = wb * 128 + 32 * blk + 8 * q;
        const bool live = p < 4 * cnt && col < a.nrows;  // the same for the 4 lanes of a block
        const float *src = (blk < 2 ? t0 : t1) + i * kActRow + 32 * (blk & 1) + 8 * q;
        const float4 x0 = *(const float4 *) src, x1 = *(const float4 *) (src + 4);
        const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        sink(i, col, live, v);
        if (live && a.act_out) {
            float *ao = a.act_out + (size_t) dst[i] * a.nrows + col;
            *(float4 *) ao = x0;
            *(float4 *) (ao + 4) = x1;
        }
    }
}

// Group g of the launch's list (NT = 2: the 64-row groups and remainders > 32 rows; NT = 1: the expert's <= 32-row
// remainder), weight row block wb. DEV: an item of the fused launch (gate/up items count their arrival, down items
// wait for their group's).
template <int T, bool GLU, int NT, bool DEV>
__device__ __forceinline__ void mmq_group(const MmqArgs &a, int g, int wb, const MmqLds &L) {
    constexpr int ROWS = 32 * NT;  // activation rows of the workgroup
    constexpr int WROWS = GLU ? 128 : 256;  // weight rows of the workgroup
    auto &sh_a0 = L.a0;
    auto &sh_a1 = L.a1;
    auto &sh_s = L.s;
    auto &sh_src = L.src;
    auto &sh_dst = L.dst;
    constexpr int BB = Traits<T>::bytes, NB = kNumB<T>;
    constexpr bool MIN = T == T_Q4_K || T == T_Q5_K;
    // (the wave index as a scalar: the LDS-DMA destinations derived from it are wave-uniform M0 values)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int hh = lane / 32, jl = lane % 32;

    if constexpr (kGridWords<T> > 0) {  // the codebook into LDS (visible after the barriers below)
        const uint4 *src = (const uint4 *) (T == T_IQ3_XXS ? (const void *) g_iq_grids.iq3xxs
                                            : T == T_IQ3_S ? (const void *) g_iq_grids.iq3s
                                                           : (const void *) g_iq_grids.iq2s);
        for (int i = tid; i < kGridWords<T> / 4; i += kMmqThreads) ((uint4 *) L.grid)[i] = src[i];
    }
    int e, seg, cnt;
    if (!group_rows<NT>(a, g, L.grp, e, seg, cnt)) return;
    MMQ_MARK(0);
    MMQ_NOTE(NT * 1000 + cnt);
    for (int i = tid; i < ROWS; i += kMmqThreads) {
        const int q = seg + min(i, cnt - 1);
        sh_src[i] = a.src ? a.src[q] : q - seg;
        sh_dst[i] = a.dst_rows ? a.dst_rows[q] : q;
    }

    const int nb = a.ncols / 256;
    const int64_t row_bytes = (int64_t) nb * BB;
    const uint8_t *wbase = expert_base(a, e) + wb * WROWS * row_bytes;  // the workgroup's first weight row
    // weight rows past nrows (nrows % WROWS != 0) are computed from the last row and not stored
    const int row0 = wb * WROWS + wave * 32 + jl;
    const int ra = min(row0, a.nrows - 1), rb = GLU ? ra : min(row0 + 128, a.nrows - 1);
    const Rsrc r0 = rsrc_of(wbase + a.off_a), r1 = rsrc_of(wbase + (GLU ? a.off_b : a.off_a)), rx = image_rsrc(a.xpack, a.x_img, a.src, seg);
    const uint32_t v0 = (uint32_t) ((ra - wb * WROWS) * row_bytes), v1 = (uint32_t) ((rb - wb * WROWS) * row_bytes);
    const uint32_t c0 = v0 + 16 * hh, c1 = v1 + 16 * hh;
    __syncthreads();  // sh_src / sh_dst

    // LDS-DMA of chunk (kb, h) - columns 256 kb + 128 h .. + 127, hi and lo: 512 bytes per row - by instruction u of
    // wave w: rows 8 u + 2 w, + 1 (one per 32 lanes; lane piece i of row r reads image piece i ^ (r % 16))
    constexpr int NU = ROWS / 8;
    uint32_t qo[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int r = 8 * u + 2 * wave + lane / 32;
        qo[u] = (uint32_t) ((size_t) sh_src[r] * a.x_img + 16 * ((lane % 32) ^ (r % 16)));
    }
    // min-term sums of superblock kb: rows 32 w' + lane / 2 (2 pieces per row), w' = wave % (ROWS / 32)
    const int srow = 32 * (wave % (ROWS / 32));
    const uint32_t so = (uint32_t) ((size_t) sh_src[srow + lane / 2] * a.x_img + (size_t) nb * kSbMain + 16 * (lane & 1));
    // (unconditional: a fixed number of loads in flight keeps the compiler's wait counts exact; rows past cnt read
    // the last routed row again)
    constexpr int CPOL = DEV && !GLU ? kCpolDevice : 0;  // the fused down items read this launch's act rows
    auto dma_chunk = [&](uint8_t *buf, int kb, int h) __attribute__((always_inline)) {
        const uint32_t soff = (uint32_t) (kb * kSbMain + h * 512);
#pragma unroll
        for (int u = 0; u < NU; ++u) dma16<CPOL>(rx, buf + (8 * u + 2 * wave) * kRowA, qo[u], soff);
    };
    auto dma_sums = [&](int kb) __attribute__((always_inline)) {  // the waves past ROWS / 32 repeat the first ones
        if constexpr (MIN) dma16<CPOL>(rx, sh_s + srow * kRowS, so, (uint32_t) (kb * kSbMin));
    };

    // the superblocks [kb0, kb_end) of this item: all of them, or part blockIdx.y of a split K range
    int kb0 = 0, kb_end = nb, part = 0;
    if constexpr (!GLU && !DEV) {
        if (a.ksplit > 1) {
            part = (int) blockIdx.y;
            kb0 = part * nb / a.ksplit;
            kb_end = (part + 1) * nb / a.ksplit;
        }
    }
    WFrag<T> f0, f1, n0, n1;
    bool failed = false;
    if constexpr (DEV && !GLU) {  // the first weights in flight, then the wait for the group's act rows
        wfrag_load<T, 0>(r0, v0, c0, 0, f0);
        wfrag_load<T, 0>(r1, v1, c1, 0, f1);
        failed = wait_group(a, a.slot, &L.grp[3]);
        dma_chunk(sh_a0, 0, 0);
        dma_sums(0);
    } else {
        dma_chunk(sh_a0, kb0, 0);
        dma_sums(kb0);
        wfrag_load<T, 0>(r0, v0, c0, (uint32_t) (kb0 * BB), f0);
        wfrag_load<T, 0>(r1, v1, c1, (uint32_t) (kb0 * BB), f1);
    }
    dma_wait();
    lds_barrier();
    MMQ_MARK(1);

    // acc[t][m] is kept in units of the current superblock's d (per lane: its row's d, 1 if d = 0), so the MFMAs
    // accumulate into it directly; between superblocks it is rescaled and the min term added (fp32 rounding).
    // All tiles are computed whatever cnt (rows past it hold stale LDS data and are never stored).
    v16f acc[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][0][r] = acc[t][1][r] = 0.0f;
    float ds0 = blk_d<T>(f0), ds1 = blk_d<T>(f1);
    bool on0 = ds0 != 0.0f, on1 = ds1 != 0.0f;
    ds0 = on0 ? ds0 : 1.0f;
    ds1 = on1 ? ds1 : 1.0f;

    // eight 16-column steps of one half from LDS chunk buf (step i: sub-block 4 h + i / 2, column group 2 hh + i % 2):
    // acc[t][m] += A (hi, lo) x B (integer-scaled codes). Software-pipelined: while the MFMAs of step i issue, the A
    // fragments of step i + 1 are read from LDS and its B operands decoded (VALU); the compiler interleaves them
    // (pinning one MFMA to a fixed number of VALU instructions with scheduling-group barriers measured 2% slower).
    auto load_a = [&](const uint8_t *buf, int i, v8h (&av)[2][NT]) __attribute__((always_inline)) {
        const int piece = a_piece<T>(i, hh);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint8_t *ap = buf + (t * 32 + jl) * kRowA;
            av[0][t] = *(const v8h *) (ap + 16 * (piece ^ (jl & 15)));
            av[1][t] = *(const v8h *) (ap + 16 * ((16 + piece) ^ (jl & 15)));
        }
    };
    auto load_a1 = [&](const uint8_t *buf, int i, int x, v8h (&av)[NT]) __attribute__((always_inline)) {
        const int piece = 16 * x + a_piece<T>(i, hh);
#pragma unroll
        for (int t = 0; t < NT; ++t) av[t] = *(const v8h *) (buf + (t * 32 + jl) * kRowA + 16 * (piece ^ (jl & 15)));
    };
    auto half_pass = [&](const uint8_t *buf, auto hc, const WFrag<T> &f0, const WFrag<T> &f1) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        v8h av[2][NT];
        const uint32_t *grid = L.grid;
        BOp<T> b0 = decode<T>(f0, 4 * h, 0, hh, on0, grid), b1 = decode<T>(f1, 4 * h, 0, hh, on1, grid), d0, d1;
        load_a(buf, 0, av);
        if constexpr (NB == 1) {
            // One B operand per stream: the hi fragments of step i + 1 are read into the registers of step i's as soon
            // as its hi MFMAs have issued, the lo ones after its lo MFMAs (no second set of A registers).
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                if (i < 7) {
                    d0 = decode<T>(f0, 4 * h + (i + 1) / 2, (i + 1) & 1, hh, on0, grid);
                    d1 = decode<T>(f1, 4 * h + (i + 1) / 2, (i + 1) & 1, hh, on1, grid);
                }
#pragma unroll
                for (int x = 0; x < 2; ++x) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        acc[t][0] = mfma32(av[x][t], b0.b[0], acc[t][0]);
                        acc[t][1] = mfma32(av[x][t], b1.b[0], acc[t][1]);
                    }
                    if (i < 7) load_a1(buf, i + 1, x, av[x]);
                }
                if (i < 7) {
                    b0 = d0;
                    b1 = d1;
                }
            }
        } else {
            v8h an[2][NT];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                if (i < 7) {
                    load_a(buf, i + 1, an);
                    d0 = decode<T>(f0, 4 * h + (i + 1) / 2, (i + 1) & 1, hh, on0, grid);
                    d1 = decode<T>(f1, 4 * h + (i + 1) / 2, (i + 1) & 1, hh, on1, grid);
                }
                // hi for every (tile, stream), then lo: dependent MFMAs 2 NT issues apart
#pragma unroll
                for (int g = 0; g < NB; ++g)
#pragma unroll
                    for (int x = 0; x < 2; ++x)
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            acc[t][0] = mfma32(av[x][t], b0.b[g], acc[t][0]);
                            acc[t][1] = mfma32(av[x][t], b1.b[g], acc[t][1]);
                        }
                if (i < 7) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        av[0][t] = an[0][t];
                        av[1][t] = an[1][t];
                    }
                    b0 = d0;
                    b1 = d1;
                }
            }
        }
    };

    // The scheduling barriers (sched_barrier 0) between the phases below are load-bearing: they keep the compiler from
    // moving instructions across the explicit vmcnt waits that stand for the DMA and fragment loads (removing them
    // all fails the GEMM tests).
    // one superblock with fragments f0, f1 (current; their first part loaded) and n0, n1 (next, first part loaded here)
    auto superblock = [&](int kb, WFrag<T> &f0, WFrag<T> &f1, WFrag<T> &n0, WFrag<T> &n1)
                          __attribute__((always_inline)) {
        const bool more = kb + 1 < kb_end;
        const int kn = more ? kb + 1 : kb;  // the last superblock reloads itself: same load count every iteration
        dma_chunk(sh_a1, kb, 1);
        __builtin_amdgcn_sched_barrier(0);
        // Weights one half superblock ahead: this block's second-half codes now, the next block's header and
        // first-half codes during the second half. Each part has half a superblock of compute to land, and only
        // about one and a half fragments per stream are live at a time.
        wfrag_load<T, 1>(r0, v0, c0, kb * BB, f0);
        wfrag_load<T, 1>(r1, v1, c1, kb * BB, f1);
        __builtin_amdgcn_sched_barrier(0);
        half_pass(sh_a0, std::integral_constant<int, 0>{}, f0, f1);
        __builtin_amdgcn_sched_barrier(0);
        // chunk (kb, 1) landed (only the weight loads issued after it may still be in flight)
        constexpr int kPend = 2 * wfrag_loads<T, 1>();  // s_waitcnt vmcnt(kPend): vmcnt bits 3:0 and 15:14
        __builtin_amdgcn_s_waitcnt(0x0F70 | (kPend & 0xF) | ((kPend >> 4) << 14));
        lds_barrier();  // chunk (kb, 1) visible; chunk buffer 0 free

        dma_chunk(sh_a0, kn, 0);
        wfrag_load<T, 0>(r0, v0, c0, kn * BB, n0);
        wfrag_load<T, 0>(r1, v1, c1, kn * BB, n1);
        __builtin_amdgcn_sched_barrier(0);
        half_pass(sh_a1, std::integral_constant<int, 1>{}, f0, f1);
        __builtin_amdgcn_sched_barrier(0);
        // superblock done: acc <- (acc ds - dmin (m . S)) / ds_next, ds_next = 1 after the last superblock
        float nd0 = 1.0f, nd1 = 1.0f;
        bool non0 = true, non1 = true;
        dma_wait();  // the next weights (and chunk (kb + 1, 0))
        if (more) {
            nd0 = blk_d<T>(n0);
            nd1 = blk_d<T>(n1);
            non0 = nd0 != 0.0f;
            non1 = nd1 != 0.0f;
            nd0 = non0 ? nd0 : 1.0f;
            nd1 = non1 ? nd1 : 1.0f;
        }
        const float inv0 = __builtin_amdgcn_rcpf(nd0), inv1 = __builtin_amdgcn_rcpf(nd1);
        const float k0 = ds0 * inv0, k1 = ds1 * inv1;
        float km0 = 0.0f, km1 = 0.0f;
        v8h bm0, bm1;
        if constexpr (MIN) {
            km0 = -half_to_float(f0.h.x >> 16) * inv0;
            km1 = -half_to_float(f1.h.x >> 16) * inv1;
            bm0 = min_b<T>(f0);
            bm1 = min_b<T>(f1);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if constexpr (MIN) {
                // one min-term product at a time (each is 16 registers)
                v16f z;
#pragma unroll
                for (int r = 0; r < 16; ++r) z[r] = 0.0f;
                const v8h am = *(const v8h *) (sh_s + (t * 32 + jl) * kRowS + 16 * hh);
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const v16f mt = mfma32(am, m ? bm1 : bm0, z);
                    const float k = m ? k1 : k0, km = m ? km1 : km0;
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[t][m][r] = fmaf_(acc[t][m][r], k, km * mt[r]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[t][0][r] *= k0;
                    acc[t][1][r] *= k1;
                }
            }
        }
        ds0 = nd0;
        ds1 = nd1;
        on0 = non0;
        on1 = non1;
        lds_barrier();  // chunk (kb + 1, 0) visible; chunk buffer 1 and the sums free
        dma_sums(kn);  // read at the end of superblock kb + 1, after its first barrier
        MMQ_MARK(2 + kb);
    };
    // the fragment sets swap roles every superblock
    for (int kb = kb0; kb < kb_end; kb += 2) {
        superblock(kb, f0, f1, n0, n1);
        if (kb + 1 < kb_end) superblock(kb + 1, n0, n1, f0, f1);
    }

    dma_wait();  // the last (unused) sums load
    if constexpr (!GLU) {
        store_group<NT>(a, acc, sh_dst, cnt, row0, hh, part, failed);
    } else {
        static_assert(ROWS * kActRow * 4 <= ROWS * kRowA, "act tile fits a chunk buffer");
        act_to_lds<NT>(acc, (float *) sh_a0, (float *) sh_a1, wave, jl, hh);
        __syncthreads();
        // the reference's Q8_1 arithmetic (q = roundf(v / d), IEEE division): the same codes as the quantiser of the f32
        // act rows would give, written straight into the act split image rows
        act_blocks(a, (const float *) sh_a0, (const float *) sh_a1, sh_dst, cnt, wb, wave, lane,
                   [&](int i, int col, bool live, const float (&v)[8]) {
                       if constexpr (DEV)
                           image_store_dev(a.out_form, v, rsrc_of(a.out_pack), (uint32_t) ((size_t) sh_dst[i] * a.out_img),
                                           a.nrows, col, live);
                       else if (const Q8x8 q = q8_1_x8(v); live)
                           image_store(a.out_form, q, a.out_pack + (size_t) sh_dst[i] * a.out_img, a.nrows, col);
                   });
        if constexpr (DEV) {  // every act store of the workgroup has completed: count the arrival
            dma_wait();
            __syncthreads();
            if (tid == 0)
                __hip_atomic_fetch_add(a.gdone + a.slot, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    MMQ_MARK(12);
}

// One launch runs both lists, the 64-row groups first and then the experts' <= 32-row remainders, so the
// smaller workgroups fill the machine while the last large ones finish. The grid is one-dimensional and XCD-aware:
// workgroup L runs on XCD L % 8 (the hardware's round-robin dispatch), and the n_cb weight row blocks of a group are
// consecutive items of one XCD, so the group's activation rows are fetched into that XCD's L2 once, not once per
// row block; groups go to the XCDs in turn (group u on XCD u % 8) in increasing order.
// (SPX mode: one partition of all 8 XCDs. In a partitioned mode the mapping is a performance assumption only.)
constexpr int kXcds = 8;  // MI355X: 8 XCDs, each with its own L2
// A launch of the int8 form whose items leave CUs idle runs its 64-row groups as two items of 32 rows: its time is that of
// one item, which is half, for the same sums (200 tokens to 4 of 16 experts, Q4_K, 2048 / 768: 81 -> 64 us, where the
// split form takes 70). The rule: at most one item per CU, the groups counted as halves and the shared expert's too.
constexpr int kHalvesMax = 256;
__host__ __device__ constexpr int xcd_items(int groups, int n_cb) { return n_cb * kXcds * ((groups + kXcds - 1) / kXcds); }
__host__ __device__ constexpr int groups32(int rows) { return (rows + 31) / 32; }

// Item j of the two lists (nm 64-row groups, then the remainders): its group g, half, and whether it is one token tile.
__device__ __forceinline__ void list_item(int j, int nm, bool halves, int &g, int &half, bool &one) {
    half = -1;
    one = true;
    if (halves && j < 2 * nm) {
        g = j >> 1;
        half = j & 1;
    } else {
        g = halves ? j - nm : j;
        one = g >= nm;
        if (one) g -= nm;
    }
}

// Workgroup -> its arguments, group g, weight row block wb and whether the group is one token tile (at most 32 rows);
// false: nothing to do. I8: a launch of the int8 form.
template <bool I8>
__device__ __forceinline__ bool mmq_item(const MmqArgs &m, const MmqShared &sh, MmqArgs &a, int &g, int &wb, bool &one) {
    a = m;
    a.half = -1;
    int nm, nr, sh_items = sh.items;
    bool halves = false;
    // expert path: the groups that exist in this call (the device-side counts of the 64-row list and of the remainder
    // list) take the first workgroups; the rest of the grid (sized for the upper bound) returns at once
    auto counts = [&] { nm = m.gprefix[m.n_expert], nr = m.gprefix[2 * (m.n_expert + 1) - 1]; };
    if (I8 && sh.may_halve) {
        counts();
        halves = (2 * nm + nr) * m.n_cb + groups32(sh.n_rows) * sh.n_cb <= kHalvesMax;
        if (halves) sh_items = xcd_items(groups32(sh.n_rows), sh.n_cb);
    }
    const bool shared = (int) blockIdx.x < sh_items;
    const int lid = shared ? (int) blockIdx.x : (int) blockIdx.x - sh_items, r = lid / kXcds;
    const int n_cb = shared ? sh.n_cb : m.n_cb;
    const int j = (r / n_cb) * kXcds + lid % kXcds, wbj = r % n_cb;
    one = false;
    g = j;
    wb = wbj;
    if (shared) {
        a.table = nullptr;
        a.w_dense = sh.w;
        a.off_a = 0;
        a.off_b = sh.off_b;
        a.ncols = sh.ncols;
        a.nrows = sh.nrows;
        a.xpack = sh.xpack;
        a.x_img = sh.x_img;
        a.bounds = a.src = a.dst_rows = nullptr;
        a.n_rows = sh.n_rows;
        a.dst = sh.dst;
        a.out_pack = sh.out_pack;
        a.out_img = sh.out_img;
        a.out_form = sh.out_form;
        a.act_out = nullptr;
        if (halves) {
            one = true;
            return 32 * j < sh.n_rows;
        }
        if (kMmqTok * j >= sh.n_rows) return false;
        one = sh.n_rows - kMmqTok * j <= kMmqTok / 2;
        if (one) g = 2 * j;
    } else if (m.bounds) {
        if (!(I8 && sh.may_halve)) counts();
        if (j >= (halves ? 2 * nm : nm) + nr) return false;
        list_item(j, nm, halves, g, a.half, one);
    } else {
        if (m.rows_first) {
            wb = (r / m.n_groups) * kXcds + lid % kXcds;
            g = r % m.n_groups;
            if (wb >= n_cb) return false;
        } else if (j >= m.n_groups) {
            return false;
        }
        one = m.dense_small != 0;
    }
    return true;
}

template <int T, bool GLU>
__global__ __launch_bounds__(kMmqThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void k_mmq(const MmqArgs m,
                                                                                            const MmqShared sh) {
    __shared__ __align__(16) uint8_t sh_a0[kMmqTok * kRowA];
    __shared__ __align__(16) uint8_t sh_a1[kMmqTok * kRowA];
    __shared__ __align__(16) uint8_t sh_s[(T == T_Q4_K || T == T_Q5_K) ? kMmqTok * kRowS : 16];
    __shared__ __align__(16) uint32_t sh_grid[kGridWords<T> > 0 ? kGridWords<T> : 4];
    __shared__ int sh_src[kMmqTok], sh_dst[kMmqTok], sh_grp[4];
    const MmqLds L{sh_a0, sh_a1, *(uint8_t (*)[kMmqTok * kRowS]) sh_s, sh_src, sh_dst, sh_grp, sh_grid};
    MmqArgs a;
    int g, wb;
    bool one;
    if (!mmq_item<false>(m, sh, a, g, wb, one)) return;
    if (one) mmq_group<T, GLU, 1, false>(a, g, wb, L);
    else mmq_group<T, GLU, 2, false>(a, g, wb, L);
}

}  // namespace
}  // namespace fns
#include "fns_mmq_i8.hpp"
namespace fns {
namespace {

// Gate/up (with SwiGLU and the Q8_1 of act) and down of the expert path in one launch. The gate/up items come first,
// in the order and XCD mapping of k_mmq (group g's weight row blocks on XCD g % 8), then the down items with the same
// mapping; a down item first waits for its group's gate/up items (arrival counts, see above). Workgroups are
// dispatched in index order on each XCD and every gate/up item precedes every down item, so a waiting down item never
// holds a slot that a gate/up item it waits for still needs: the wait always ends. The gate/up tail and the first
// down items overlap instead of being separated by a launch. (A persistent variant that takes items from per-XCD
// queues measured no faster.)
struct MoeArgs {
    const char *const *table;
    int64_t gate_off, up_off, down_off;
    int hidden, inter, n_expert, n_main;  // n_main: the 64-row list's upper bound
    int n_cb_gu, n_cb_dn, gwait, spin_limit;
    const uint8_t *ximg;                  // x images [n_tok][x_img]
    uint8_t *aimg;                        // act images [n_tok * k][a_img]
    int64_t x_img, a_img;
    const int32_t *bounds, *gprefix, *src1, *dstr;
    float *dexp;
    int *gdone;
    uint32_t *status;
};
// Each GEMM reads the form of image that is the faster one for its type (GU8, DN8: int8), so a pair whose types take
// different forms is one launch as well.
template <int TGU, bool GU8, int TDN, bool DN8>
__global__ __launch_bounds__(kMmqThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void k_mmq_moe(const MoeArgs m) {
    constexpr bool ANY8 = GU8 || DN8;
    constexpr int kSplitBuf = kMmqTok * kRowA, kBuf = GU8 && DN8 ? kI8Buf : kSplitBuf;
    static_assert(kI8Buf <= kSplitBuf, "the split form's buffers hold the int8 form's");
    __shared__ __align__(16) uint8_t sh_a0[kBuf];
    __shared__ __align__(16) uint8_t sh_a1[kBuf];
    __shared__ __align__(16) float sh_d[2][8][ANY8 ? kMmqTok : 4];
    __shared__ __align__(16) uint8_t sh_s[2][kMmqTok * kRowS];
    __shared__ int sh_src[kMmqTok], sh_dst[kMmqTok], sh_grp[4];
    PF_MARK(3, 0);
    // The groups that exist in this call (the device-side counts of the two lists: the 64-row groups, then the <= 32-row
    // remainders) are numbered j = 0 .. R - 1 and take the first workgroups of the grid; the workgroups past them (the
    // grid is sized for the upper bound) return at once, after every real item has been dispatched.
    const int nm = m.gprefix[m.n_expert], nr = m.gprefix[2 * (m.n_expert + 1) - 1];
    const bool halves_gu = GU8 && (2 * nm + nr) * m.n_cb_gu <= kHalvesMax, halves_dn = DN8 && (2 * nm + nr) * m.n_cb_dn <= kHalvesMax;
    const int items_gu = xcd_items((halves_gu ? 2 * nm : nm) + nr, m.n_cb_gu);  // a multiple of kXcds
    const bool is_gu = (int) blockIdx.x < items_gu, halves = is_gu ? halves_gu : halves_dn;
    const int cb = is_gu ? m.n_cb_gu : m.n_cb_dn;
    const int lid = is_gu ? (int) blockIdx.x : (int) blockIdx.x - items_gu, r = lid / kXcds;
    const int j = (r / cb) * kXcds + lid % kXcds, wb = r % cb;
    if (j >= (halves ? 2 * nm : nm) + nr) return;
    MmqArgs a{};
    int g;
    bool one;
    list_item(j, nm, halves, g, a.half, one);
    const bool rest = one && a.half < 0;
    a.slot = rest ? m.n_main + g : g;
    auto run = [&](auto glu) __attribute__((always_inline)) {
        constexpr bool GLU = decltype(glu)::value;
        constexpr int T = GLU ? TGU : TDN;
        if constexpr (GLU ? GU8 : DN8) {
            const MmqI8Lds L{(uint8_t (&)[kI8Buf]) sh_a0, (uint8_t (&)[kI8Buf]) sh_a1, (float (&)[2][8][kMmqTok]) sh_d, sh_s,
                             sh_src, sh_dst, sh_grp, nullptr};
            if (one) mmq_group_i8<T, GLU, 1, true>(a, g, wb, L);
            else mmq_group_i8<T, GLU, 2, true>(a, g, wb, L);
        } else {
            const MmqLds L{(uint8_t (&)[kSplitBuf]) sh_a0, (uint8_t (&)[kSplitBuf]) sh_a1, sh_s[0], sh_src, sh_dst, sh_grp, nullptr};
            if (one) mmq_group<T, GLU, 1, true>(a, g, wb, L);
            else mmq_group<T, GLU, 2, true>(a, g, wb, L);
        }
    };
    a.table = m.table;
    a.n_expert = m.n_expert;
    a.bounds = m.bounds;
    a.gprefix = m.gprefix;
    a.dst_rows = m.dstr;
    a.gdone = m.gdone;
    if (is_gu) {
        a.off_a = m.gate_off;
        a.off_b = m.up_off;
        a.ncols = m.hidden;
        a.nrows = m.inter;
        a.xpack = m.ximg;
        a.x_img = m.x_img;
        a.src = m.src1;
        a.out_pack = m.aimg;
        a.out_img = m.a_img;
        a.out_form = DN8 ? kImgI8 : kImgSplit;
        run(std::true_type{});
    } else {
        a.off_a = m.down_off;
        a.ncols = m.inter;
        a.nrows = m.hidden;
        a.xpack = m.aimg;
        a.x_img = m.a_img;
        a.src = m.dstr;
        a.dst = m.dexp;
        a.gwait = m.gwait + (halves_gu && !rest ? m.n_cb_gu : 0);  // both halves of a group arrive at its count
        a.spin_limit = m.spin_limit;
        a.status = m.status;
        run(std::false_type{});
    }
    PF_MARK(3, 1);
}

// the split form: the types without an int8 form, mmq and mmq_experts over the caller's split image (Q8_0 takes the int8
// form there), and gate/up beside a shared expert that reads the split image of x
const void *mmq_kernel(int type, bool glu) {
    switch (type) {
        case T_Q3_K: return glu ? (const void *) k_mmq<T_Q3_K, true> : (const void *) k_mmq<T_Q3_K, false>;
        case T_Q6_K: return glu ? (const void *) k_mmq<T_Q6_K, true> : (const void *) k_mmq<T_Q6_K, false>;
        case T_IQ2_S: return glu ? (const void *) k_mmq<T_IQ2_S, true> : (const void *) k_mmq<T_IQ2_S, false>;
        case T_Q4_K: return glu ? (const void *) k_mmq<T_Q4_K, true> : (const void *) k_mmq<T_Q4_K, false>;
        case T_Q5_K: return glu ? (const void *) k_mmq<T_Q5_K, true> : (const void *) k_mmq<T_Q5_K, false>;
        case T_IQ4_XS: return glu ? (const void *) k_mmq<T_IQ4_XS, true> : (const void *) k_mmq<T_IQ4_XS, false>;
        case T_IQ3_XXS: return glu ? (const void *) k_mmq<T_IQ3_XXS, true> : (const void *) k_mmq<T_IQ3_XXS, false>;
        case T_IQ3_S: return glu ? (const void *) k_mmq<T_IQ3_S, true> : (const void *) k_mmq<T_IQ3_S, false>;
        case T_Q8_0: return glu ? (const void *) k_mmq<T_Q8_0, true> : nullptr;
    }
    return nullptr;
}

// the most items that n_cb row blocks of halves take, where 64-row groups and remainders are at most total
int64_t halves_items(int total, int n_cb) { return xcd_items(std::min(2 * total, kHalvesMax / n_cb), n_cb); }

// groups: upper bound of the 64-row list; expert path: of the 64-row list and the <= 32-row remainders together (the
// workgroups past the device-side counts return at once)
// sh: a dense matrix of the same type whose groups come first in the grid (expert path only); form: of the activations
int launch_mmq(int type, bool glu, const MmqArgs &a, int groups, hipStream_t st, const MmqShared *sh = nullptr,
               int form = kImgSplit) {
    const void *fn = form == kImgI8 ? (glu ? mmq_i8_kernel<true>(type) : mmq_i8_kernel<false>(type)) : mmq_kernel(type, glu);
    if (!fn) return host::set_error(host::ERR_TYPE, "mmq: type %d not supported", type);
    if (groups <= 0) return host::OK;
    MmqArgs arg = a;
    // expert path: n_expert + ceil(pairs / 64) (the 64-row list's bound) bounds both lists together, as expert e
    // has ceil(n_e / 64) groups in all
    int total = groups;
    MmqShared shared{};
    void *args[] = {&arg, &shared};
    const int rows = glu ? 128 : 256;  // weight rows per workgroup
    int64_t sh_items = 0;
    if (sh && a.bounds) {
        shared = *sh;
        shared.n_cb = (sh->nrows + rows - 1) / rows;
        sh_items = xcd_items((sh->n_rows + kMmqTok - 1) / kMmqTok, shared.n_cb);
    }
    arg.n_cb = (a.nrows + rows - 1) / rows;
    // dense: when even twice the workgroups of the 64-row groups fit one per CU, groups of 32 rows (one token tile:
    // more B decode per MFMA, but twice the workgroups; measured faster for 64 -> 128 workgroups, slower for
    // 192 -> 384)
    arg.dense_small = 0;
    const int ks = !glu && !a.bounds && a.ksplit > 1 ? a.ksplit : 1;
    if (ks > 1 && (a.ncols / 256 < ks || ks > 8)) return host::set_error(host::ERR_SHAPE, "mmq: bad K split");
    arg.ksplit = ks;
    if (!a.bounds && (a.n_rows <= 32 || (int64_t) 2 * groups * arg.n_cb * ks <= 256)) {
        arg.dense_small = 1;
        total = (a.n_rows + 31) / 32;
    }
    arg.n_groups = total;
    arg.rows_first = form != kImgSplit && !a.bounds && (arg.n_cb % kXcds == 0 || arg.n_cb >= 4 * kXcds);
    int64_t items = sh_items + (arg.rows_first ? (int64_t) total * kXcds * ((arg.n_cb + kXcds - 1) / kXcds)
                                               : (int64_t) arg.n_cb * kXcds * ((total + kXcds - 1) / kXcds));
    // Halves where the rows allow them (an item takes at most 32 of the more than 64 (groups - n_expert - 1) rows), so that
    // the first workgroups of a larger launch, the shared expert's, need not wait for the counts (1021-token block: 1 us).
    const int sh32 = groups32(shared.n_rows);
    shared.may_halve = form == kImgI8 && a.bounds &&
                       (int64_t) std::max(1, 2 * (groups - a.n_expert) - 1) * arg.n_cb + sh32 * shared.n_cb <= kHalvesMax;
    if (shared.may_halve)
        items = std::max<int64_t>(items, xcd_items(sh32, shared.n_cb) + halves_items(total, arg.n_cb));
    if (items > INT32_MAX) return host::set_error(host::ERR_SHAPE, "mmq: grid too large");
    shared.items = (int) sh_items;
    const hipError_t e = hipLaunchKernel(fn, dim3((unsigned) items, (unsigned) ks), dim3(kMmqThreads), args, 0, st);
    if (e != hipSuccess) return host::set_error(host::ERR_LAUNCH, "mmq: %s", hipGetErrorString(e));
    return host::check_launch("mmq");
}

// The fused kernel of a pair of {Q3_K, Q4_K} and the forms of the x and act images; the other pairs take two launches (the
// Q5_K and Q6_K decoders push the combined kernel past 256 registers).
template <int TGU, bool GU8> const void *mmq_moe_kernel_dn(int tdn, int act_form) {
    if (tdn == T_Q4_K) return act_form == kImgI8 ? (const void *) k_mmq_moe<TGU, GU8, T_Q4_K, true> : nullptr;
    return tdn == T_Q3_K && act_form == kImgSplit ? (const void *) k_mmq_moe<TGU, GU8, T_Q3_K, false> : nullptr;
}
const void *mmq_moe_kernel(int tgu, int tdn, int x_form, int act_form) {
    if (tgu == T_Q4_K)
        return x_form == kImgI8 ? mmq_moe_kernel_dn<T_Q4_K, true>(tdn, act_form) : mmq_moe_kernel_dn<T_Q4_K, false>(tdn, act_form);
    return tgu == T_Q3_K && x_form == kImgSplit ? mmq_moe_kernel_dn<T_Q3_K, false>(tdn, act_form) : nullptr;
}

// The fused launch (the arrival counters zero: the compaction kernel clears them).
int launch_mmq_moe(int tgu, int tdn, int x_form, int act_form, MoeArgs m, hipStream_t st) {
    const void *fn = mmq_moe_kernel(tgu, tdn, x_form, act_form);
    if (!fn) return host::set_error(host::ERR_TYPE, "mmq: types %d / %d not supported", tgu, tdn);
    if (m.n_main <= 0) return host::OK;
    m.n_cb_gu = (m.inter + 127) / 128;
    m.n_cb_dn = (m.hidden + 255) / 256;
    m.gwait += m.n_cb_gu;
    // n_main = n_expert + ceil(pairs / 64) bounds both lists together: expert e has ceil(n_e / 64) groups in all
    const int total = m.n_main;
    auto part = [&](int n_cb, bool i8) {
        const int64_t whole = (int64_t) n_cb * kXcds * ((total + kXcds - 1) / kXcds);
        return i8 ? std::max(whole, halves_items(total, n_cb)) : whole;
    };
    const int64_t items = part(m.n_cb_gu, x_form == kImgI8) + part(m.n_cb_dn, act_form == kImgI8);
    if (items > INT32_MAX) return host::set_error(host::ERR_SHAPE, "mmq: grid too large");
    void *args[] = {&m};
    const hipError_t e = hipLaunchKernel(fn, dim3((unsigned) items), dim3(kMmqThreads), args, 0, st);
    if (e != hipSuccess) return host::set_error(host::ERR_LAUNCH, "mmq: %s", hipGetErrorString(e));
    return host::check_launch("mmq (gate/up + down)");
}

int check_mmq_shape(int type, int64_t ncols, int64_t nrows) {
    if (!host::is_kquant(type) && !host::is_iq(type) && type != T_Q8_0)
        return host::set_error(host::ERR_TYPE, "mmq: type %d not supported", type);
    if (host::iq_needs_grid(type) && !host::iq_grids_ready())
        return host::set_error(host::ERR_TYPE, "mmq: type %d needs the IQ codebooks (fns_hip_set_iq_grids)", type);
    if (ncols <= 0 || ncols % 256 || nrows <= 0 || nrows % kMmqRows || ncols > 65536)
        return host::set_error(host::ERR_SHAPE, "mmq: ncols must be a positive multiple of 256, nrows of 64");
    return host::OK;
}
}  // namespace

namespace impl {

// This translation unit's copy of the IQ codebooks (fns_quarter.hpp g_iq_grids), on the current device.
int iq_grids_upload_mmq(const void *grids) {
    const hipError_t e = dev::upload_iq_grids((const dev::IqGrids *) grids);
    return e == hipSuccess ? host::OK : host::set_error(host::ERR_LAUNCH, "set_iq_grids: %s", hipGetErrorString(e));
}

size_t mmq_image_bytes(int64_t ncols) { return (size_t) split_row_bytes(ncols); }
size_t mmq_q8_1_bytes(int64_t ncols, int64_t nrows) { return (size_t) nrows * mmq_image_bytes(ncols) + 4096; }
size_t mmq_bounds_bytes(int64_t n_expert) { return bounds_bytes(n_expert); }

size_t mmq_form_bytes(int form, int64_t ncols) { return (size_t) (ncols / 256) * img_sb_bytes(form); }
int mmq_form(int type) { return mmq_i8_kernel<false>(type) ? kImgI8 : kImgSplit; }

int mmq_quant_image(const float *x, int64_t ncols, int64_t rows, int form, void *ximg, hipStream_t st) {
    if (!x || !ximg || ncols <= 0 || ncols % 256 || ncols > 65536 || rows < 0 || rows > INT32_MAX)
        return host::set_error(host::ERR_SHAPE, "mmq quantize: bad arguments");
    if (rows == 0) return host::OK;
    hipLaunchKernelGGL(k_quant_image, dim3((unsigned) rows, (unsigned) ((ncols + 2047) / 2048)), dim3(256), 0, st, x,
                       (int) ncols, form, (uint8_t *) ximg, (int64_t) mmq_form_bytes(form, ncols));
    return host::check_launch("mmq quantize");
}

// RMSNorm of x (f32 [rows][n]) into out, its Q8_1 blocks into xq (null: none) and its image rows into ximg, for rows
// that mmq_rms_norm_image_fits: at most 8192 columns, 16-byte aligned arrays.
bool mmq_rms_norm_image_fits(const float *x, const float *w, const float *out, int64_t n) {
    return n > 0 && n % 256 == 0 && n <= 8192 && (((uintptr_t) x | (uintptr_t) w | (uintptr_t) out) & 15) == 0;
}
int mmq_rms_norm_image(const float *x, const float *w, float *out, void *xq, int n, float eps, int rows, int form,
                       void *ximg, hipStream_t st) {
    if (!x || !w || !out || !ximg || rows < 0 || !mmq_rms_norm_image_fits(x, w, out, n))
        return host::set_error(host::ERR_SHAPE, "mmq rms_norm: bad arguments");
    if (rows == 0) return host::OK;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned) rows), dim3(256), 0, st, x, w, out, (uint8_t *) xq, n, eps,
                           host::q8_1_row_bytes(n), form, (uint8_t *) ximg, (int64_t) mmq_form_bytes(form, n));
    };
    if (n <= 2048) go(k_rms_norm_image<1>);
    else if (n <= 4096) go(k_rms_norm_image<2>);
    else go(k_rms_norm_image<4>);
    return host::check_launch("mmq rms_norm");
}

int mmq_guard_image(float *act, float *escale, int64_t ncols, int64_t rows, int form, void *img, int64_t stride,
                    hipStream_t st) {
    if (!act || !escale || !img || ncols <= 0 || ncols % 256 || ncols > 65536 || rows < 0 || rows > INT32_MAX - 3)
        return host::set_error(host::ERR_SHAPE, "mmq guard: bad arguments");
    if (rows == 0) return host::OK;
    hipLaunchKernelGGL(k_guard_image, dim3((unsigned) ((rows + 3) / 4)), dim3(256), 0, st, act, escale, (int) ncols,
                       (int) rows, form, (uint8_t *) img, stride);
    return host::check_launch("mmq guard");
}

int mmq_compact(const int32_t *ids, int64_t n_tok, int64_t k, int64_t n_expert, int64_t x_rows_per_tok,
                int32_t *ids_src1, int32_t *ids_dst, int32_t *bounds, int32_t *gprefix, hipStream_t st, int32_t *gdone,
                int n_gdone) {
    // an empty batch (n_tok = 0) may pass null id arrays: it only writes zero bounds
    const bool any = n_tok > 0;
    if ((any && (!ids || !ids_src1 || !ids_dst)) || !bounds || !gprefix || n_tok < 0 || k < 1 || n_expert < 1 || n_expert > 256 ||
        n_tok * k > (1 << 20) || (x_rows_per_tok != 1 && x_rows_per_tok != k))
        return host::set_error(host::ERR_SHAPE, "mmq compaction: bad arguments");
    // at most 64 workgroups (every one reads all ids), one 1024-pair piece each up to 65536 pairs
    const int64_t pieces = (n_tok * k + kCompactThreads - 1) / kCompactThreads;
    const int per_wg = (int) std::max<int64_t>(1, (pieces + 63) / 64);
    const unsigned wgs = (unsigned) std::max<int64_t>(1, (pieces + per_wg - 1) / per_wg);
    hipLaunchKernelGGL(k_mmq_compact, dim3(wgs), dim3(kCompactThreads), 0, st, ids, (int) (n_tok * k), (int) k,
                       (int) n_expert, (int) x_rows_per_tok, ids_src1, ids_dst, bounds, gprefix, gdone, gdone ? n_gdone : 0,
                       per_wg);
    return host::check_launch("mmq compaction");
}

// Bytes per act image row in the prefill workspace: the image rounded up to whole 128-byte lines, so that no cache
// line holds parts of two rows. The fused launch depends on it: rows of different groups are written and read by
// different workgroups at different times, and a line read for one row must never carry another row's older bytes.
int64_t act_stride(int64_t ncols, int form = kImgSplit) { return ((int64_t) mmq_form_bytes(form, ncols) + 127) / 128 * 128; }

// Tokens of one expert launch, whose tokens' image rows (row_bytes a token) a buffer resource has to reach: all of a call
// whose images are below 2 GiB, otherwise ranges of tokens one after another.
int64_t image_tokens(int64_t n_tok, int64_t row_bytes) {
    return std::min(n_tok, std::max<int64_t>(1, kRsrcBytes / std::max<int64_t>(1, row_bytes)));
}

// the 64-row list's upper bound for n_pairs sorted rows over n_expert experts: sum_e (n_e / 64 + (n_e % 64 > 32))
int64_t main_groups(int64_t n_expert, int64_t n_pairs) { return n_expert + (n_pairs + kMmqTok - 1) / kMmqTok; }

// x_stride / out_stride: bytes per activation / act image row (0: the image's own size)
int expert_args(int type, const char *const *table, size_t off_a, size_t off_b, bool glu, int64_t ncols,
                int64_t nrows, int64_t n_expert, const void *xpack, const int32_t *ids_src1, const int32_t *ids_dst,
                const int32_t *bounds, const int32_t *gprefix, float *dst, void *out_pack, float *act_out, MmqArgs &a,
                int64_t x_stride = 0, int64_t out_stride = 0) {
    FNS_TRY(check_mmq_shape(type, ncols, nrows));
    if (!table || !xpack || !bounds || !gprefix || (!glu && !dst) || (glu && !out_pack) || n_expert < 1 || n_expert > 256)
        return host::set_error(host::ERR_SHAPE, "mmq_experts: bad arguments");
    a = MmqArgs{};
    a.table = table;
    a.off_a = (int64_t) off_a;
    a.off_b = (int64_t) off_b;
    a.ncols = (int) ncols;
    a.nrows = (int) nrows;
    a.n_expert = (int) n_expert;
    a.xpack = (const uint8_t *) xpack;
    a.x_img = x_stride ? x_stride : (int64_t) mmq_image_bytes(ncols);
    a.bounds = bounds;
    a.gprefix = gprefix;
    a.src = ids_src1;
    a.dst_rows = ids_dst;
    a.dst = dst;
    a.out_pack = (uint8_t *) out_pack;
    a.out_img = out_stride ? out_stride : (int64_t) mmq_image_bytes(nrows);
    a.act_out = act_out;
    return host::OK;
}

// Q8_0 (the reference's dense and output-head type, src/ggml/ggml_mmq.cu:59) takes the int8 form of the GEMM, and for
// row counts that are not a multiple of 64 the GEMV kernels, a few token columns per weight pass. The K-quants and IQ
// types read the split image here and in mmq_experts; nothing in these calls forbids the int8 form, which has not been
// measured for them.
int mmq(int type, const void *w, int64_t ncols, int64_t nrows, const float *x, int64_t n_tok, void *xq, float *dst,
        hipStream_t st) {
    if (type == T_Q8_0 && nrows % kMmqRows) {  // the GEMV kernels (any row count), a few token columns per pass
        if (!w || !x || !xq || !dst || n_tok < 0 || ncols <= 0 || ncols % 256 || nrows <= 0)
            return host::set_error(host::ERR_SHAPE, "mmq: bad arguments");
        if (n_tok == 0) return host::OK;
        FNS_TRY(quantize_q8_1(x, xq, ncols, n_tok, st));
        return mmvq(type, w, ncols, nrows, xq, dst, n_tok, st);
    }
    FNS_TRY(check_mmq_shape(type, ncols, nrows));
    if (!w || !x || !xq || !dst || n_tok < 0 || n_tok > 65535) return host::set_error(host::ERR_SHAPE, "mmq: bad arguments");
    if (n_tok == 0) return host::OK;
    const int form = type == T_Q8_0 ? kImgI8 : kImgSplit;
    FNS_TRY(mmq_quant_image(x, ncols, n_tok, form, xq, st));
    MmqArgs a{};
    a.w_dense = (const uint8_t *) w;
    a.ncols = (int) ncols;
    a.nrows = (int) nrows;
    a.xpack = (const uint8_t *) xq;
    a.x_img = (int64_t) mmq_form_bytes(form, ncols);
    a.n_rows = (int) n_tok;
    a.dst = dst;
    return launch_mmq(type, false, a, (int) ((n_tok + kMmqTok - 1) / kMmqTok), st, nullptr, form);
}

int mmq_experts(int type, const char *const *table, size_t off, int64_t ncols, int64_t nrows, int64_t n_expert,
                const float *x, int64_t x_rows_per_tok, int64_t n_tok, const int32_t *ids, int64_t n_used,
                int32_t *ids_src1, int32_t *ids_dst, int32_t *bounds, void *xq, float *dst, hipStream_t st) {
    if (type == T_Q8_0 && nrows % kMmqRows) {  // the GEMV over every (token, slot), as mmq above; the sort is still written
        if (!x || !xq || !table || !ids || !dst || n_used < 1 || n_tok < 0 || ncols <= 0 || ncols % 256 ||
            (x_rows_per_tok != 1 && x_rows_per_tok != n_used))
            return host::set_error(host::ERR_SHAPE, "mmq_experts: bad arguments");
        if (n_tok == 0) return host::OK;
        const int64_t rows = n_tok * x_rows_per_tok;
        int32_t *gprefix = (int32_t *) ((uint8_t *) xq + (size_t) rows * host::q8_1_row_bytes(ncols));
        FNS_TRY(mmq_compact(ids, n_tok, n_used, n_expert, x_rows_per_tok, ids_src1, ids_dst, bounds, gprefix, st));
        FNS_TRY(quantize_q8_1(x, xq, ncols, rows, st));
        return mmvq_experts_div(type, table, off, ncols, nrows, xq, rows, x_rows_per_tok == 1 ? n_used : 1, ids,
                                n_tok * n_used, dst, st);
    }
    FNS_TRY(check_mmq_shape(type, ncols, nrows));
    if (!x || !xq || n_used < 1 || n_tok < 0 || n_tok * x_rows_per_tok > 65535)
        return host::set_error(host::ERR_SHAPE, "mmq_experts: bad arguments");
    if (n_tok == 0) return host::OK;
    // bounds holds n_expert + 1 ints (the reference's MmqIdsScratch sizing); the tile-group prefix of the GEMM goes in
    // the slack that mmq_q8_1_bytes adds after the activation images (4096 bytes >= 257 ints)
    const int64_t rows = n_tok * x_rows_per_tok;
    int32_t *gprefix = (int32_t *) ((uint8_t *) xq + (size_t) rows * mmq_image_bytes(ncols));
    const int form = type == T_Q8_0 ? kImgI8 : kImgSplit;
    const int64_t img = (int64_t) mmq_form_bytes(form, ncols);
    FNS_TRY(mmq_compact(ids, n_tok, n_used, n_expert, x_rows_per_tok, ids_src1, ids_dst, bounds, gprefix, st));
    FNS_TRY(mmq_quant_image(x, ncols, rows, form, xq, st));
    const int64_t step = image_tokens(n_tok, x_rows_per_tok * img);
    for (int64_t t = 0; t < n_tok; t += step) {
        const int64_t n = std::min(step, n_tok - t);
        if (step < n_tok)
            FNS_TRY(mmq_compact(ids + t * n_used, n, n_used, n_expert, x_rows_per_tok, ids_src1, ids_dst, bounds, gprefix, st));
        MmqArgs a;
        FNS_TRY(expert_args(type, table, off, 0, false, ncols, nrows, n_expert, (uint8_t *) xq + t * x_rows_per_tok * img,
                            ids_src1, ids_dst, bounds, gprefix, dst + t * n_used * nrows, nullptr, nullptr, a, img));
        FNS_TRY(launch_mmq(type, false, a, (int) main_groups(n_expert, n * n_used), st, nullptr, form));
    }
    // the sort that the caller's arrays are left with is the whole call's
    if (step < n_tok)
        FNS_TRY(mmq_compact(ids, n_tok, n_used, n_expert, x_rows_per_tok, ids_src1, ids_dst, bounds, gprefix, st));
    return host::OK;
}

// ---- prefill MoE layer ----------------------------------------------------------------------------------------
// The MoE section of the reference's Engine::prefill_chunk (src/engine.cu:340-357: gemm_bf16_batch, route_topk_batch,
// mmq_experts for gate and up, swiglu, amax_guard, mmq_experts for down, moe_combine_batch) for n_tok tokens, with the
// activations quantised once per token, gate and up in one pass with the SwiGLU and the Q8_1 of act fused, and the
// expert sort shared by both GEMMs.
namespace {
constexpr int kPrefillSections = 15;
void prefill_sizes(const FnsMoeLayer *L, int64_t T, size_t *sz) {
    const int64_t P = T * L->k;
    sz[0] = (size_t) T * L->n_expert * 4;                 // logits
    sz[1] = (size_t) P * 4;                               // ids
    sz[2] = (size_t) P * 4;                               // w
    sz[3] = (size_t) T * mmq_image_bytes(L->hidden);      // x images
    sz[4] = (size_t) P * act_stride(L->inter);            // act images
    sz[5] = (size_t) P * L->hidden * 4;                   // per-(token, slot) down outputs
    sz[6] = (size_t) P * 4;                               // ids_src1
    sz[7] = (size_t) P * 4;                               // ids_dst
    // bounds + group prefix, arrival counters, status word
    sz[8] = bounds_bytes(L->n_expert) + 4 * (size_t) (main_groups(L->n_expert, P) + L->n_expert) + 4;
    sz[9] = L->guard ? (size_t) P * L->inter * 4 : 0;     // f32 act (F16 guard only)
    sz[10] = (size_t) P * 4;                              // escale
    const int64_t fs = L->shexp_inter > 0 ? L->shexp_inter : 0;
    sz[11] = L->ffn_norm ? (size_t) T * L->hidden * 4 : 0;                         // RMSNorm output h
    sz[12] = L->ffn_norm ? (size_t) T * host::q8_1_row_bytes(L->hidden) : 0;      // its Q8_1 blocks (for inspection)
    sz[13] = fs ? (size_t) T * mmq_image_bytes(fs) : 0;                            // shared-expert act images
    sz[14] = fs ? (size_t) T * L->hidden * 4 : 0;                                  // shared-expert output
}
}  // namespace

int moe_prefill_section(const FnsMoeLayer *L, int64_t n_tok, int section, size_t *offset, size_t *bytes) {
    FNS_TRY(moe_prefill_workspace(L, n_tok, nullptr, nullptr));
    if (section < 0 || section >= kPrefillSections) return host::set_error(host::ERR_SHAPE, "moe_prefill: no section %d", section);
    size_t sz[kPrefillSections], off = 0;
    prefill_sizes(L, n_tok, sz);
    for (int i = 0; i < section; ++i) off += (sz[i] + 255) / 256 * 256;
    if (offset) *offset = off;
    if (bytes) *bytes = sz[section];
    return host::OK;
}

int moe_prefill_workspace(const FnsMoeLayer *L, int64_t n_tok, size_t *offsets, size_t *total) {
    if (!L || n_tok < 1 || n_tok * L->k > 65536)
        return host::set_error(host::ERR_SHAPE, "moe_prefill: 1 <= n_tok, n_tok * k <= 65536");
    size_t sz[kPrefillSections], off = 0;
    prefill_sizes(L, n_tok, sz);
    for (int i = 0; i < kPrefillSections; ++i) {
        if (offsets && i < 6) offsets[i] = off;
        off += (sz[i] + 255) / 256 * 256;
    }
    if (total) *total = off + 4096;
    return host::OK;
}

// The shared expert over the n_tok split-image rows of h: gate and up, SwiGLU and the Q8_1 of act into act_img (gu),
// then down into sh [n_tok][hidden] (dn). Both are the grouped GEMM over one dense matrix; with the routed experts'
// type they ride in the routed launch (its workgroups are few: 8 at 37 tokens of the reference model's block, 25.5 +
// 15.9 us as launches of their own, against nothing beside the routed 149 experts'), otherwise mmq_dense_shared
// launches them.
MmqShared shared_gate_up(const FnsMoeLayer *L, const void *ximg, int x_form, int64_t n_tok, void *act_img, int act_form) {
    MmqShared g{};
    g.w = (const uint8_t *) L->shexp_gate;
    g.off_b = (const uint8_t *) L->shexp_up - (const uint8_t *) L->shexp_gate;
    g.ncols = L->hidden;
    g.nrows = L->shexp_inter;
    g.n_rows = (int) n_tok;
    g.xpack = (const uint8_t *) ximg;
    g.x_img = (int64_t) mmq_form_bytes(x_form, L->hidden);
    g.out_pack = (uint8_t *) act_img;
    g.out_img = (int64_t) mmq_form_bytes(act_form, L->shexp_inter);
    g.out_form = act_form;
    return g;
}
MmqShared shared_down(const FnsMoeLayer *L, const void *act_img, int act_form, int64_t n_tok, float *sh) {
    MmqShared d{};
    d.w = (const uint8_t *) L->shexp_down;
    d.ncols = L->shexp_inter;
    d.nrows = L->hidden;
    d.n_rows = (int) n_tok;
    d.xpack = (const uint8_t *) act_img;
    d.x_img = (int64_t) mmq_form_bytes(act_form, L->shexp_inter);
    d.dst = sh;
    return d;
}
int mmq_dense_shared(int type, bool glu, int form, const MmqShared &s, hipStream_t st) {
    MmqArgs a{};
    a.w_dense = s.w;
    a.off_b = s.off_b;
    a.ncols = s.ncols;
    a.nrows = s.nrows;
    a.xpack = s.xpack;
    a.x_img = s.x_img;
    a.n_rows = s.n_rows;
    a.dst = s.dst;
    a.out_pack = s.out_pack;
    a.out_img = s.out_img;
    a.out_form = s.out_form;
    return launch_mmq(type, glu, a, (s.n_rows + kMmqTok - 1) / kMmqTok, st, nullptr, form);
}

// Dense GEMMs on activation images already built (the dense FFN block): gate/up in one GLU launch (SwiGLU and the
// Q8_1 of act in the epilogue, act images out), and a plain launch whose K range may be split into ksplit parts
// (dst then holds ksplit partial sums, part_stride floats apart). x_form, act_form: the forms of the activation image
// read and of the act image written.
bool mmq_tiled(int type, int64_t ncols, int64_t nrows) {
    const bool t = host::is_kquant(type) || type == T_Q8_0 || (host::is_iq(type) && (!host::iq_needs_grid(type) ||
                                                                                      host::iq_grids_ready()));
    return t && ncols > 0 && ncols % 256 == 0 && ncols <= 65536 && nrows > 0 && nrows % kMmqRows == 0;
}

int mmq_dense_glu(int type, const void *gate, const void *up, int64_t ncols, int64_t nrows, const void *ximg,
                  int64_t n_tok, void *act_img, int x_form, int act_form, hipStream_t st) {
    FNS_TRY(check_mmq_shape(type, ncols, nrows));
    MmqArgs g{};
    g.w_dense = (const uint8_t *) gate;
    g.off_a = 0;
    g.off_b = (const uint8_t *) up - (const uint8_t *) gate;
    g.ncols = (int) ncols;
    g.nrows = (int) nrows;
    g.xpack = (const uint8_t *) ximg;
    g.x_img = (int64_t) mmq_form_bytes(x_form, ncols);
    g.n_rows = (int) n_tok;
    g.out_pack = (uint8_t *) act_img;
    g.out_img = (int64_t) mmq_form_bytes(act_form, nrows);
    g.out_form = act_form;
    return launch_mmq(type, true, g, (int) ((n_tok + kMmqTok - 1) / kMmqTok), st, nullptr, x_form);
}

int mmq_dense_parts(int type, const void *w, int64_t ncols, int64_t nrows, const void *ximg, int64_t n_tok, float *dst,
                    int ksplit, int x_form, hipStream_t st) {
    FNS_TRY(check_mmq_shape(type, ncols, nrows));
    MmqArgs d{};
    d.w_dense = (const uint8_t *) w;
    d.ncols = (int) ncols;
    d.nrows = (int) nrows;
    d.xpack = (const uint8_t *) ximg;
    d.x_img = (int64_t) mmq_form_bytes(x_form, ncols);
    d.n_rows = (int) n_tok;
    d.dst = dst;
    d.ksplit = ksplit;
    d.part_stride = n_tok * nrows;
    return launch_mmq(type, false, d, (int) ((n_tok + kMmqTok - 1) / kMmqTok), st, nullptr, x_form);
}

namespace {
__global__ void k_zero_word(uint32_t *w) { *w = 0; }
}  // namespace

// The sticky status word of a prefill workspace (after the fused launch's arrival counters in section 8), read after
// the stream's work so far has completed; clear: zero it afterwards (a kernel on `st`).
int moe_prefill_status(const FnsMoeLayer *L, int64_t n_tok, void *ws, int clear, uint32_t *status, hipStream_t st) {
    if (!ws || !status) return host::set_error(host::ERR_SHAPE, "moe_prefill_status: null argument");
    size_t off;
    FNS_TRY(moe_prefill_section(L, n_tok, 8, &off, nullptr));
    const int64_t words = 3 * (L->n_expert + 1) + main_groups(L->n_expert, n_tok * L->k) + L->n_expert;
    uint32_t *word = (uint32_t *) ((uint8_t *) ws + off) + words;
    if (hipMemcpyAsync(status, word, 4, hipMemcpyDeviceToHost, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
        return host::set_error(host::ERR_LAUNCH, "moe_prefill_status: reading the status word failed");
    if (clear) {
        hipLaunchKernelGGL(k_zero_word, dim3(1), dim3(1), 0, st, word);
        FNS_TRY(host::check_launch("moe_prefill_status: clearing"));
    }
    return host::OK;
}

int moe_prefill_status_collect(const FnsMoeLayer *L, int64_t n_tok, void *ws, uint32_t *dst, hipStream_t st) {
    if (!ws || !dst) return host::set_error(host::ERR_SHAPE, "moe_prefill_status_collect: null argument");
    size_t off;
    FNS_TRY(moe_prefill_section(L, n_tok, 8, &off, nullptr));
    const int64_t words = 3 * (L->n_expert + 1) + main_groups(L->n_expert, n_tok * L->k) + L->n_expert;
    return status_collect((uint32_t *) ((uint8_t *) ws + off) + words, dst, st);
}

// The forms of a layer's activation images: int8 where every matrix that reads the image has the int8 form (x: the routed
// and the shared gate/up). They follow from the types alone, so a token's result has the same bits in a call of any
// length. (In calls whose items leave CUs idle the split form was the faster one for Q4_K and Q5_K, 70 against 81 us for
// 200 tokens to 4 of 16 experts; the int8 form's halves and its groups of few rows made up for that: 64.)
namespace {
struct PrefillForms { int x, act, sh; };
PrefillForms prefill_forms(const FnsMoeLayer *L) {
    const bool has_sh = L->shexp_inter > 0;
    const int sgt = has_sh && L->shexp_gu_type ? L->shexp_gu_type : L->gu_type;
    const int sdt = has_sh && L->shexp_down_type ? L->shexp_down_type : L->down_type;
    return {std::min(mmq_form(L->gu_type), mmq_form(sgt)), mmq_form(L->down_type), mmq_form(sdt)};
}
}  // namespace

int moe_prefill_image(const FnsMoeLayer *L, int section, int *form, size_t *row_stride) {
    if (!L || !form || !row_stride) return host::set_error(host::ERR_SHAPE, "moe_prefill_image: null argument");
    const PrefillForms f = prefill_forms(L);
    switch (section) {
        case 3: *form = f.x, *row_stride = mmq_form_bytes(f.x, L->hidden); return host::OK;
        case 4: *form = f.act, *row_stride = (size_t) act_stride(L->inter, f.act); return host::OK;
        case 13: *form = f.sh, *row_stride = mmq_form_bytes(f.sh, L->shexp_inter); return host::OK;
    }
    return host::set_error(host::ERR_SHAPE, "moe_prefill_image: section %d holds no image", section);
}

int moe_prefill(const FnsMoeLayer *L, const float *x, const float *x_resid, float *out, int64_t n_tok, void *ws,
                size_t ws_bytes, hipStream_t st) {
    if (!L || !x || !out || !ws || !L->router_w || !L->table) return host::set_error(host::ERR_SHAPE, "moe_prefill: null argument");
    size_t total;
    FNS_TRY(moe_prefill_workspace(L, n_tok, nullptr, &total));
    if (ws_bytes < total) return host::set_error(host::ERR_NOMEM, "moe_prefill: workspace %zu < %zu bytes", ws_bytes, total);
    if (L->k < 1 || L->k > 16 || L->k > L->n_expert || L->n_expert > 256)
        return host::set_error(host::ERR_SHAPE, "moe_prefill: 1 <= k <= min(16, n_expert), n_expert <= 256");
    FNS_TRY(check_mmq_shape(L->gu_type, L->hidden, L->inter));
    FNS_TRY(check_mmq_shape(L->down_type, L->inter, L->hidden));
    if (L->shexp_inter < 0 || (L->shexp_inter > 0 && (!L->shexp_gate || !L->shexp_up || !L->shexp_down)))
        return host::set_error(host::ERR_SHAPE, "moe_prefill: shared expert: gate, up and down given");
    size_t sz[kPrefillSections];
    prefill_sizes(L, n_tok, sz);
    uint8_t *sec[kPrefillSections];
    size_t off = 0;
    for (int i = 0; i < kPrefillSections; ++i) {
        sec[i] = (uint8_t *) ws + off;
        off += (sz[i] + 255) / 256 * 256;
    }
    float *logits = (float *) sec[0], *w = (float *) sec[2], *dexp = (float *) sec[5], *act = (float *) sec[9];
    float *escale = (float *) sec[10];
    int32_t *ids = (int32_t *) sec[1], *src1 = (int32_t *) sec[6], *dstr = (int32_t *) sec[7], *bounds = (int32_t *) sec[8];
    const int64_t P = n_tok * L->k;
    const char *const *table = (const char *const *) L->table;

    const bool has_sh = L->shexp_inter > 0;
    const int sgt = has_sh && L->shexp_gu_type ? L->shexp_gu_type : L->gu_type;
    const int sdt = has_sh && L->shexp_down_type ? L->shexp_down_type : L->down_type;
    const PrefillForms forms = prefill_forms(L);
    const int x_form = forms.x, act_form = forms.act, sh_form = forms.sh;
    const int64_t x_img = (int64_t) mmq_form_bytes(x_form, L->hidden);

    // RMSNorm first when the layer has one: the router and the experts read h (reference src/engine.cu:331)
    bool have_img = false;  // the RMSNorm kernel has built the activation image
    if (L->ffn_norm) {
        float *h = (float *) sec[11];
        have_img = mmq_rms_norm_image_fits(x, L->ffn_norm, h, L->hidden);
        if (have_img)
            FNS_TRY(mmq_rms_norm_image(x, L->ffn_norm, h, sec[12], (int) L->hidden, L->norm_eps, (int) n_tok, x_form,
                                       sec[3], st));
        else
            FNS_TRY(rms_norm_q8_1(x, L->ffn_norm, h, sec[12], (int) L->hidden, L->norm_eps, (int) n_tok, st));
        x = h;
    }
    // the router GEMM and the activation image (unless the RMSNorm built it) in one launch when the GEMM takes its unguarded path (whole 64-column
    // chunks, aligned rows, 32-bit offsets), else as two launches
    const int H = (int) L->hidden, NE = (int) L->n_expert;
    const bool bf = L->router_dtype == T_BF16;
    const bool one = (bf || L->router_dtype == 0) && H % 64 == 0 && (int64_t) H * std::max<int64_t>(n_tok, NE) < INT32_MAX &&
                     ((uintptr_t) x & 15) == 0 && ((uintptr_t) L->router_w & (bf ? 7 : 15)) == 0;
    if (one) {
        const bool t32 = (n_tok + 31) / 32 * ((NE + 31) / 32) >= kRouterTile32Min;
        const int side = t32 ? 32 : 16, tiles_x = (int) ((n_tok + side - 1) / side), n_rt = tiles_x * ((NE + side - 1) / side);
        const int nxb = (H + 2047) / 2048;
        const int64_t n_img = have_img ? 0 : (nxb * n_tok + 1) / 2;
        if (n_rt + n_img > INT32_MAX) return host::set_error(host::ERR_SHAPE, "prefill: grid too large");
        const dim3 g((unsigned) (n_rt + n_img));
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, g, dim3(512), 0, st, L->router_w, L->router_bias, x, logits, H, NE, (int) n_tok, tiles_x,
                               n_rt, x_form, (uint8_t *) sec[3], x_img, nxb);
        };
        if (bf) t32 ? go(k_router_image<true, true>) : go(k_router_image<true, false>);
        else t32 ? go(k_router_image<false, true>) : go(k_router_image<false, false>);
        FNS_TRY(host::check_launch("prefill router + image"));
    } else {
        FNS_TRY(gemm_router_bias(L->router_dtype, L->router_w, L->router_bias, x, logits, L->hidden, L->n_expert,
                                 (int) n_tok, st));
        if (!have_img) FNS_TRY(mmq_quant_image(x, L->hidden, n_tok, x_form, sec[3], st));
    }
    FNS_TRY(route_topk(logits, ids, w, L->n_expert, L->k, (int) n_tok, L->gating, L->norm_w, st));
    // gate/up (SwiGLU and the Q8_1 of act fused) and down: act image rows padded to whole cache lines; one launch
    // unless the F16 guard's whole-row amax has to sit between them (or the type pair has no fused kernel)
    const int64_t astride = act_stride(L->inter, act_form);
    int32_t *gprefix = bounds + L->n_expert + 1, *gdone = bounds + 3 * (L->n_expert + 1);
    uint32_t *status = (uint32_t *) (gdone + main_groups(L->n_expert, P) + L->n_expert);
    const bool fused = !L->guard && mmq_moe_kernel(L->gu_type, L->down_type, x_form, act_form);
    if (has_sh) {
        FNS_TRY(check_mmq_shape(sgt, L->hidden, L->shexp_inter));
        FNS_TRY(check_mmq_shape(sdt, L->shexp_inter, L->hidden));
    }
    const int64_t sh_img = has_sh ? (int64_t) mmq_form_bytes(sh_form, L->shexp_inter) : 0;
    float *sh = has_sh ? (float *) sec[14] : nullptr;
    // tokens [t, t + n): all of them unless an image has 2 GiB or more (image_tokens)
    const int64_t step = image_tokens(n_tok, std::max(x_img, L->k * astride));
    for (int64_t t = 0; t < n_tok; t += step) {
        const int64_t n = std::min(step, n_tok - t), p0 = t * L->k, np = n * L->k;
        const int groups = (int) main_groups(L->n_expert, np);
        const uint8_t *ximg = sec[3] + t * x_img;
        uint8_t *aimg = sec[4] + p0 * astride, *shimg = has_sh ? sec[13] + t * sh_img : nullptr;
        FNS_TRY(mmq_compact(ids + p0, n, L->k, L->n_expert, 1, src1 + p0, dstr + p0, bounds, gprefix, st,
                            fused ? gdone : nullptr, groups + (int) L->n_expert));
        // down: one act row per (token, slot), in the same expert order as gate/up: the sorted rows are the pairs
        // themselves (activation row = output row = p), so the gate/up sort is reused with ids_dst as the source list
        MmqArgs gu, dn;
        FNS_TRY(expert_args(L->gu_type, table, L->gate_off, L->up_off, true, L->hidden, L->inter, L->n_expert, ximg,
                            src1 + p0, dstr + p0, bounds, gprefix, nullptr, aimg,
                            L->guard ? act + p0 * L->inter : nullptr, gu, x_img, astride));
        gu.out_form = act_form;
        FNS_TRY(expert_args(L->down_type, table, L->down_off, 0, false, L->inter, L->hidden, L->n_expert, aimg, dstr + p0,
                            dstr + p0, bounds, gprefix, dexp + p0 * L->hidden, nullptr, nullptr, dn, astride));
        // the shared expert (reference src/engine.cu:351-355): in the routed launches where the types agree
        MmqShared sgu{}, sdn{};
        if (has_sh) {
            sgu = shared_gate_up(L, ximg, x_form, n, shimg, sh_form);
            sdn = shared_down(L, shimg, sh_form, n, sh + t * L->hidden);
        }
        const bool ride_gu = has_sh && !fused && sgt == L->gu_type, ride_dn = has_sh && !fused && sdt == L->down_type;
        if (has_sh && !ride_gu) FNS_TRY(mmq_dense_shared(sgt, true, x_form, sgu, st));
        if (fused) {
            MoeArgs m{};
            m.table = table;
            m.gate_off = (int64_t) L->gate_off;
            m.up_off = (int64_t) L->up_off;
            m.down_off = (int64_t) L->down_off;
            m.hidden = (int) L->hidden;
            m.inter = (int) L->inter;
            m.n_expert = (int) L->n_expert;
            m.n_main = groups;
            m.ximg = ximg;
            m.x_img = x_img;
            m.aimg = aimg;
            m.a_img = astride;
            m.bounds = bounds;
            m.gprefix = gprefix;
            m.src1 = src1 + p0;
            m.dstr = dstr + p0;
            m.dexp = dexp + p0 * L->hidden;
            m.gdone = gdone;
            m.status = status;
            moe_test_hooks(&m.spin_limit, &m.gwait);  // withheld arrivals; + the gate/up row blocks per group
            FNS_TRY(launch_mmq_moe(L->gu_type, L->down_type, x_form, act_form, m, st));
        } else {
            FNS_TRY(launch_mmq(L->gu_type, true, gu, groups, st, ride_gu ? &sgu : nullptr, x_form));
            // whole-row amax: a second pass over the f32 act rows (reference src/kernels.cu:534-552)
            if (L->guard)
                FNS_TRY(mmq_guard_image(act + p0 * L->inter, escale + p0, L->inter, np, act_form, aimg, astride, st));
            FNS_TRY(launch_mmq(L->down_type, false, dn, groups, st, ride_dn ? &sdn : nullptr, act_form));
        }
        if (has_sh && !ride_dn) FNS_TRY(mmq_dense_shared(sdt, false, sh_form, sdn, st));
    }
    return moe_combine(dexp, L->guard ? escale : nullptr, w, sh, x_resid, out, L->hidden, L->k, (int) n_tok, st);
}

}  // namespace impl

// ---- C++ API (reference names; abort on error) ----
size_t mmq_q8_1_bytes(int64_t ncols, int64_t nrows) { return impl::mmq_q8_1_bytes(ncols, nrows); }
size_t mmq_bounds_bytes(int64_t n_expert) { return impl::mmq_bounds_bytes(n_expert); }

void mmq(ggml_type type, const void *w, int64_t ncols, int64_t nrows, const float *x, int64_t n_tok, void *xq,
         float *dst, hipStream_t stream) {
    host::abort_on_error(impl::mmq(type, w, ncols, nrows, x, n_tok, xq, dst, stream), "mmq");
}

void mmq_experts(ggml_type type, const char *const *table, size_t off, int64_t ncols, int64_t nrows, int64_t n_expert,
                 const float *x, int64_t x_rows_per_tok, int64_t n_tok, const int32_t *ids, int64_t n_used,
                 MmqIdsScratch &s, float *dst, hipStream_t stream) {
    host::abort_on_error(impl::mmq_experts(type, table, off, ncols, nrows, n_expert, x, x_rows_per_tok, n_tok, ids,
                                           n_used, s.ids_src1, s.ids_dst, s.expert_bounds, s.xq, dst, stream),
                         "mmq_experts");
}

}  // namespace fns
