// fns_mmq_i8.hpp - the grouped GEMM on int8 MFMA, for the types whose scales change every 32 columns (Q8_0, Q4_K, Q5_K,
// IQ4_XS, IQ3_XXS, IQ3_S: a sub-block is exactly one v_mfma_i32_32x32x32_i8). Included by mmq.hip, whose group lists,
// epilogues and weight fragments it shares.
//
// Per sub-block s the MFMA gives the exact integer dot I of 32 codes; the output takes I * (d8[token] * dw[row]) with
// dw = the row's sub-block scale (block d times the integer scale, exact in fp32). The scale product d8 dw is rounded to fp32
// once per sub-block (relative 2^-24; exact for Q8_0). Convert, scale product and fma are 48 VALU instructions per 32x32x32
// step against one 32-cycle MFMA, decode, addresses and waits about 6 more, so the kernel is bound by VALU issue: at 4096
// tokens (Q4_K gate/up) 54.5 instructions of 4 cycles in 234 cycles a step, 93 % of the launch, the matrix pipe busy for
// 14 %. The f16 form spends four MFMAs (128 cycles; eight for Q8_0 and IQ4_XS, whose operands are
// split in two) plus the B decode on the same step, and its activations are 4.125 bytes a value against 1.25 here: less
// than a third of the LDS-DMA traffic, one barrier instead of two, and no f16 decode of the codes.
// Measured against the f16 form (us): Q8_0 dense block (2048 / 6144) of 512 tokens 251 -> 140, of 40 tokens 173 -> 62; Q4_K
// gate/up of 4096 tokens to 8 of 128 experts 452 -> 400; Q4_K dense block of 2048 tokens 343 -> 275. Tried and slower:
// scales fetched a sub-block ahead (spills: a Q8_0 block 140 -> 167), v_dot4 for groups of at most 8 rows (512 tokens
// 150 -> 175, an LDS round trip per row and sub-block), the f16 codes with d8 applied after each sub-block (418-449
// against 400). Registers: 216 to 252, Q8_0 256 with 6 (GLU) and 14 (plain) spilled.
#pragma once

namespace fns {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// ---- weight fragments ---------------------------------------------------------------------------------------------
// The types of the f16 form keep their fragments (WFrag). Q8_0 (blocks of 34 bytes, f16 d then 32 codes): blocks e = 2 p
// and e + 1 start at 68 p, a multiple of four; lane half h reads the even block's 16 codes as the 20 aligned bytes at
// 68 p + 16 h (they start two bytes in) and the odd block's 16 at 68 p + 36 + 16 h. The two d lie in those bytes, the
// even block's in the first dword of half 0, the odd block's in the last of half 1: one exchange between the halves.
// (16 bytes at 2-byte addresses and a 2-byte load per d, as the f16 form had, were half of that kernel's time.)
template <int T> struct I8Frag { WFrag<T> f; };
template <> struct I8Frag<T_Q8_0> { uint4 e[4], o[4]; uint32_t x[4]; };
template <int T, int P>
__device__ __forceinline__ void i8frag_load(Rsrc r, uint32_t vo, uint32_t vc, uint32_t so, I8Frag<T> &f) {
    if constexpr (T == T_Q8_0) {
#pragma unroll
        for (int p = 2 * P; p < 2 * P + 2; ++p) {
            f.e[p] = bload16(r, vc, so + 68 * p);
            f.x[p] = bload4(r, vc, so + 68 * p + 16);
            f.o[p] = bload16(r, vc, so + 68 * p + 36);
        }
    } else {
        wfrag_load<T, P>(r, vo, vc, so, f.f);
    }
}
// Sub-block s (compile time): the lane's 16 codes as signed bytes (columns 16 h .. 16 h + 15 of the sub-block; IQ4_XS:
// 8 h .. 8 h + 7 and 16 + 8 h ..) and the row's scale of the sub-block.
template <int T>
__device__ __forceinline__ v4i i8_codes(const I8Frag<T> &f, int s, int h, const uint32_t *grid) {
    if constexpr (T == T_Q8_0) {
        const int p = s >> 1;
        if (s & 1) return v4i{(int) f.o[p].x, (int) f.o[p].y, (int) f.o[p].z, (int) f.o[p].w};
        return v4i{(int) __builtin_amdgcn_alignbit(f.e[p].y, f.e[p].x, 16),
                   (int) __builtin_amdgcn_alignbit(f.e[p].z, f.e[p].y, 16),
                   (int) __builtin_amdgcn_alignbit(f.e[p].w, f.e[p].z, 16),
                   (int) __builtin_amdgcn_alignbit(f.x[p], f.e[p].w, 16)};
    } else if constexpr (T == T_Q4_K || T == T_Q5_K) {
        const uint4 q = f.f.q[s >> 1];
        const int sh = 4 * (s & 1);
        uint32_t w[4] = {(q.x >> sh) & kLo4, (q.y >> sh) & kLo4, (q.z >> sh) & kLo4, (q.w >> sh) & kLo4};
        if constexpr (T == T_Q5_K) {
            const uint4 qh = f.f.qh;
            w[0] |= ((qh.x >> s) & 0x01010101u) << 4;
            w[1] |= ((qh.y >> s) & 0x01010101u) << 4;
            w[2] |= ((qh.z >> s) & 0x01010101u) << 4;
            w[3] |= ((qh.w >> s) & 0x01010101u) << 4;
        }
        return v4i{(int) w[0], (int) w[1], (int) w[2], (int) w[3]};
    } else if constexpr (T == T_IQ4_XS) {
        const uint2 q = f.f.q[s];
        return v4i{(int) iq4nl_values(q.x & kLo4), (int) iq4nl_values(q.y & kLo4), (int) iq4nl_values((q.x >> 4) & kLo4),
                   (int) iq4nl_values((q.y >> 4) & kLo4)};
    } else if constexpr (T == T_IQ3_XXS) {
        const uint32_t aux = word(f.f.aux[s >> 2], s & 3), idx = f.f.idx[s];
        v4i r;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t sg = ksigns((aux >> (7 * (2 * h + p))) & 127u);
            r[2 * p] = signed_grid(grid[(idx >> (16 * p)) & 0xffu], spread4(sg & 0xfu));
            r[2 * p + 1] = signed_grid(grid[(idx >> (16 * p + 8)) & 0xffu], spread4(sg >> 4));
        }
        return r;
    } else {
        static_assert(T == T_IQ3_S, "a type of the int8 form");
        const uint32_t qh = (s < 4 ? f.f.qh.x : f.f.qh.y) >> (8 * (s & 3)), idx = f.f.idx[s];
        v4i r;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int g = 2 * h + p;
            const uint32_t sb = (f.f.sg[s] >> (8 * p)) & 0xffu;
            r[2 * p] = signed_grid(grid[((idx >> (16 * p)) & 0xffu) | (((qh >> (2 * g)) & 1u) << 8)], spread4(sb & 0xfu));
            r[2 * p + 1] =
                signed_grid(grid[((idx >> (16 * p + 8)) & 0xffu) | (((qh >> (2 * g + 1)) & 1u) << 8)], spread4(sb >> 4));
        }
        return r;
    }
}
template <int T> __device__ __forceinline__ float i8_scale(const I8Frag<T> &f, int s, int h) {
    if constexpr (T == T_Q8_0) {
        const int p = s >> 1;
        const uint32_t own = h ? f.x[p] >> 16 : f.e[p].x & 0xffffu;  // half 0: the even block's d, half 1: the odd one's
        const uint32_t other = (uint32_t) xor_lane_i<32>((int) own);
        return half_to_float((s & 1) == h ? own : other);
    } else if constexpr (T == T_Q4_K || T == T_Q5_K) {
        const uint4 hd = f.f.h;
        const uint32_t w = s < 4 ? (hd.y & 0x3F3F3F3Fu) : ((hd.w & kLo4) | ((hd.y >> 2) & 0x30303030u));
        return half_to_float(hd.x & 0xffffu) * (float) ((w >> (8 * (s & 3))) & 0xffu);
    } else if constexpr (T == T_IQ4_XS) {
        const int ls = (int) (((f.f.h.y >> (4 * s)) & 0xfu) | (((f.f.h.x >> (16 + 2 * s)) & 3u) << 4)) - 32;
        return half_to_float(f.f.h.x & 0xffffu) * (float) ls;
    } else if constexpr (T == T_IQ3_XXS) {
        return 0.25f * half_to_float(f.f.d & 0xffffu) * (float) (2 * (int) (word(f.f.aux[s >> 2], s & 3) >> 28) + 1);
    } else {
        return half_to_float(f.f.d & 0xffffu) * (float) (2 * (int) ((f.f.sc >> (4 * s)) & 0xfu) + 1);
    }
}

// ---- one group ----------------------------------------------------------------------------------------------------
// LDS: the superblock's codes [rows][256] and scales [8][rows], double-buffered (the 16-byte pieces of row r at piece
// p ^ (r % 16), so an operand read touches distinct banks), and its min-term sums. 43.5 KB for 64 rows (39.4 without the
// sums, 1 or 2 KB more with a codebook); the registers allow two workgroups per CU.
constexpr int kI8Buf = kMmqTok * kActRow * 4;  // a code buffer, sized for the GLU epilogue's act tile (17 KB)
struct MmqI8Lds {
    uint8_t (&q0)[kI8Buf];
    uint8_t (&q1)[kI8Buf];
    float (&d)[2][8][kMmqTok];
    uint8_t (&s)[2][kMmqTok * kRowS];
    int (&src)[kMmqTok];
    int (&dst)[kMmqTok];
    int (&grp)[4];
    uint32_t *grid;
};

// the type's codebook into LDS (visible after the barriers that follow)
template <int T> __device__ __forceinline__ void grid_to_lds(const MmqI8Lds &L) {
    if constexpr (kGridWords<T> > 0) {
        const uint4 *src = (const uint4 *) (T == T_IQ3_XXS ? (const void *) g_iq_grids.iq3xxs : (const void *) g_iq_grids.iq3s);
        for (int i = threadIdx.x; i < kGridWords<T> / 4; i += kMmqThreads) ((uint4 *) L.grid)[i] = src[i];
    }
}
// Rows seg .. seg + cnt - 1 of expert e, weight row block wb: as mmq_group (4 waves, two 32-row weight streams each, 32 NT
// activation rows; DEV: an item of the fused launch). LIVE: the rows of a tile whose products are scaled, all 32 or
// (NT = 1, see mmq_group_i8) as many as the group has; the others are not stored.
template <int T, bool GLU, int NT, int LIVE, bool DEV>
__device__ __forceinline__ void mmq_rows_i8(const MmqArgs &a, int wb, int e, int seg, int cnt, const MmqI8Lds &L) {
    constexpr int ROWS = 32 * NT, WROWS = GLU ? 128 : 256, BB = Traits<T>::bytes;
    constexpr bool MIN = T == T_Q4_K || T == T_Q5_K;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int hh = lane / 32, jl = lane % 32;
    int *const sh_src = L.src, *const sh_dst = L.dst;
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

    // LDS-DMA of a superblock's codes: instruction u of wave w takes rows 16 u + 4 w .. + 3, 16 lanes per row
    constexpr int CPOL = DEV && !GLU ? kCpolDevice : 0;  // the fused down items read this launch's act rows
    constexpr int NU = ROWS / 16;
    uint32_t qo[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int r = 16 * u + 4 * wave + lane / 16;
        qo[u] = (uint32_t) ((size_t) sh_src[r] * a.x_img + 16 * ((lane % 16) ^ (r % 16)));
    }
    const int srow = 32 * (wave % NT);
    const uint32_t so = (uint32_t) ((size_t) sh_src[srow + lane / 2] * a.x_img + kI8Sum + 16 * (lane & 1));
    // scales: thread t < 2 ROWS reads four of row t / 2 and stores them transposed
    const bool dthr = tid < 2 * ROWS;
    const uint32_t dof = (uint32_t) ((size_t) sh_src[(tid / 2) % ROWS] * a.x_img + kI8Scale + 16 * (tid & 1));
    auto dma_sb = [&](uint8_t *buf, int sb, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NU; ++u) dma16<CPOL>(rx, buf + (16 * u + 4 * wave) * 256, qo[u], (uint32_t) (kb * kI8Sb));
        if constexpr (MIN) dma16<CPOL>(rx, L.s[sb] + srow * kRowS, so, (uint32_t) (kb * kI8Sb));
    };
    auto load_d = [&](int kb) __attribute__((always_inline)) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rx, dof, (uint32_t) (kb * kI8Sb), CPOL);
        return make_uint4(v[0], v[1], v[2], v[3]);
    };
    auto store_d = [&](int sb, const uint4 &v) __attribute__((always_inline)) {
        if (dthr) {
            const int r = tid / 2, s = 4 * (tid & 1);
            L.d[sb][s][r] = __builtin_bit_cast(float, v.x);
            L.d[sb][s + 1][r] = __builtin_bit_cast(float, v.y);
            L.d[sb][s + 2][r] = __builtin_bit_cast(float, v.z);
            L.d[sb][s + 3][r] = __builtin_bit_cast(float, v.w);
        }
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
    I8Frag<T> f0, f1, n0, n1;
    bool failed = false;
    if constexpr (DEV && !GLU) {  // the first weights in flight, then the wait for the group's act rows
        i8frag_load<T, 0>(r0, v0, c0, 0, f0);
        i8frag_load<T, 0>(r1, v1, c1, 0, f1);
        failed = wait_group(a, a.slot, &L.grp[3]);
        dma_sb(L.q0, 0, 0);
        store_d(0, load_d(0));
    } else {
        dma_sb(L.q0, 0, kb0);
        const uint4 dv = load_d(kb0);
        i8frag_load<T, 0>(r0, v0, c0, (uint32_t) (kb0 * BB), f0);
        i8frag_load<T, 0>(r1, v1, c1, (uint32_t) (kb0 * BB), f1);
        store_d(0, dv);
    }
    dma_wait();
    lds_barrier();

    v16f acc[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][0][r] = acc[t][1][r] = 0.0f;

    // The codes of step i (sub-block i / NT, token tile i % NT) of the superblock in LDS buffer buf, and the scales d8 of
    // the 16 tokens of the tile that this lane holds.
    auto load_step = [&](const uint8_t *buf, int i) __attribute__((always_inline)) {
        const int s = i / NT, t = i % NT, r = t * 32 + jl;
        const uint8_t *row = buf + r * 256;
        if constexpr (T == T_IQ4_XS) {
            const uint2 lo = *(const uint2 *) (row + 8 * hh + 16 * ((2 * s) ^ (r & 15)));
            const uint2 hi = *(const uint2 *) (row + 8 * hh + 16 * ((2 * s + 1) ^ (r & 15)));
            return v4i{(int) lo.x, (int) lo.y, (int) hi.x, (int) hi.y};
        } else {
            return *(const v4i *) (row + 16 * ((2 * s + hh) ^ (r & 15)));
        }
    };
    auto load_scales = [&](int sb, int i, float (&d)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < LIVE / 8; ++q) {
            const float4 v = *(const float4 *) &L.d[sb][i / NT][(i % NT) * 32 + 8 * q + 4 * hh];
            d[4 * q] = v.x, d[4 * q + 1] = v.y, d[4 * q + 2] = v.z, d[4 * q + 3] = v.w;
        }
    };
    // Four sub-blocks 4 P .. 4 P + 3, one step at a time (the scheduling barrier keeps the compiler from hoisting the
    // operands of many steps, which spills); a step's codes are read during the step before it. (The scales too: 16 more
    // registers, and 465 us against 384 for a 2048-token Q8_0 dense FFN block.)
    auto half_pass = [&](const uint8_t *buf, int sb, auto pc, const I8Frag<T> &f0, const I8Frag<T> &f1) __attribute__((always_inline)) {
        constexpr int P = decltype(pc)::value;
        v4i cur = load_step(buf, 4 * P * NT), nxt;
        v4i b0, b1;
        float w0, w1;
#pragma unroll
        for (int i = 4 * P * NT; i < (4 * P + 4) * NT; ++i) {
            const int s = i / NT, t = i % NT;
            __builtin_amdgcn_sched_barrier(0);
            if (t == 0) {
                b0 = i8_codes<T>(f0, s, hh, L.grid), b1 = i8_codes<T>(f1, s, hh, L.grid);
                w0 = i8_scale<T>(f0, s, hh), w1 = i8_scale<T>(f1, s, hh);
            }
            float d8[16];
            load_scales(sb, i, d8);
            if (i + 1 < (4 * P + 4) * NT) nxt = load_step(buf, i + 1);
            const v16i z = {};
            const v16i i0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur, b0, z, 0, 0, 0);
            const v16i i1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur, b1, z, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < LIVE / 2; ++q) {
                acc[t][0][q] = fmaf_((float) i0[q], d8[q] * w0, acc[t][0][q]);
                acc[t][1][q] = fmaf_((float) i1[q], d8[q] * w1, acc[t][1][q]);
            }
            // (pins this step's sums here: instruction selection is free to sink them past the scheduling barriers)
            asm volatile("" : "+v"(acc[t][0]), "+v"(acc[t][1]));
            cur = nxt;
        }
    };
    auto superblock = [&](int kb, int sb, uint8_t *buf, uint8_t *nbuf, I8Frag<T> &f0, I8Frag<T> &f1, I8Frag<T> &n0,
                          I8Frag<T> &n1) __attribute__((always_inline)) {
        const int kn = kb + 1 < kb_end ? kb + 1 : kb;  // the last superblock reloads itself: the same loads every time
        dma_sb(nbuf, sb ^ 1, kn);
        const uint4 dn = load_d(kn);
        i8frag_load<T, 1>(r0, v0, c0, (uint32_t) (kb * BB), f0);
        i8frag_load<T, 1>(r1, v1, c1, (uint32_t) (kb * BB), f1);
        __builtin_amdgcn_sched_barrier(0);
        half_pass(buf, sb, std::integral_constant<int, 0>{}, f0, f1);
        __builtin_amdgcn_sched_barrier(0);
        i8frag_load<T, 0>(r0, v0, c0, (uint32_t) (kn * BB), n0);
        i8frag_load<T, 0>(r1, v1, c1, (uint32_t) (kn * BB), n1);
        __builtin_amdgcn_sched_barrier(0);
        half_pass(buf, sb, std::integral_constant<int, 1>{}, f0, f1);
        if constexpr (MIN) {  // the min term: acc -= dmin (m . S)
            const float m0 = -half_to_float(f0.f.h.x >> 16), m1 = -half_to_float(f1.f.h.x >> 16);
            const v8h bm0 = min_b<T>(f0.f), bm1 = min_b<T>(f1.f);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                v16f z;
#pragma unroll
                for (int r = 0; r < 16; ++r) z[r] = 0.0f;
                const v8h am = *(const v8h *) (L.s[sb] + (t * 32 + jl) * kRowS + 16 * hh);
                const v16f t0 = mfma32(am, bm0, z), t1 = mfma32(am, bm1, z);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[t][0][r] = fmaf_(m0, t0[r], acc[t][0][r]);
                    acc[t][1][r] = fmaf_(m1, t1[r], acc[t][1][r]);
                }
            }
        }
        store_d(sb ^ 1, dn);
        __builtin_amdgcn_sched_barrier(0);
        dma_wait();     // the next superblock's codes and sums (and the next weights)
        lds_barrier();  // visible to every wave; this superblock's buffers are free
    };
    for (int kb = kb0; kb < kb_end; kb += 2) {
        superblock(kb, 0, L.q0, L.q1, f0, f1, n0, n1);
        if (kb + 1 < kb_end) superblock(kb + 1, 1, L.q1, L.q0, n0, n1, f0, f1);
    }
    if constexpr (!GLU) {
        store_group<NT>(a, acc, sh_dst, cnt, row0, hh, part, failed);
    } else {
        float *t0 = (float *) L.q0, *t1 = (float *) L.q1;
        act_to_lds<NT>(acc, t0, t1, wave, jl, hh);
        __syncthreads();
        act_blocks(a, t0, t1, sh_dst, cnt, wb, wave, lane, [&](int i, int col, bool live, const float (&v)[8]) {
            if constexpr (DEV)
                image_store_dev(a.out_form, v, rsrc_of(a.out_pack), (uint32_t) ((size_t) sh_dst[i] * a.out_img), a.nrows, col, live);
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
}

// Group g, weight row block wb. The scaling of a tile is what bounds a group, so one of at most 8 or 16 rows leaves out that of
// the rows it does not have: 1 token to 8 of 128 experts (Q4_K, 2048 / 768) 51.0 -> 40.8 us, 12 tokens through a dense
// Q4_K block (2048 / 6144) 49.5 -> 40.1; a 37-token block (256 experts, one or two rows each) 135 -> 124. (The same as a
// branch per 8 rows inside the tile: 24 rows a group 252 -> 266 us; as two copies inside a superblock: Q5_K and IQ spill.)
template <int T, bool GLU, int NT, bool DEV>
__device__ __forceinline__ void mmq_group_i8(const MmqArgs &a, int g, int wb, const MmqI8Lds &L) {
    grid_to_lds<T>(L);
    int e, seg, cnt;
    if (!group_rows<NT>(a, g, L.grp, e, seg, cnt)) return;
    if constexpr (NT == 1) {
        if (cnt <= 8) return mmq_rows_i8<T, GLU, 1, 8, DEV>(a, wb, e, seg, cnt, L);
        if (cnt <= 16) return mmq_rows_i8<T, GLU, 1, 16, DEV>(a, wb, e, seg, cnt, L);
    }
    mmq_rows_i8<T, GLU, NT, 32, DEV>(a, wb, e, seg, cnt, L);
}

// Grid as k_mmq's for the expert lists and the shared expert. Dense: the row blocks go to the XCDs in turn and an XCD
// takes every row group of one block before the next, so each weight byte enters one XCD's L2 and the (small) activation
// images all eight; with few row blocks (rows_first = 0) the groups go to the XCDs instead, as in k_mmq.
template <int T, bool GLU>
__global__ __launch_bounds__(kMmqThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void k_mmq_i8(const MmqArgs m,
                                                                                               const MmqShared sh) {
    __shared__ __align__(16) uint8_t sh_q0[kI8Buf];
    __shared__ __align__(16) uint8_t sh_q1[kI8Buf];
    __shared__ __align__(16) float sh_d[2][8][kMmqTok];
    __shared__ __align__(16) uint8_t sh_s[2][(T == T_Q4_K || T == T_Q5_K) ? kMmqTok * kRowS : 16];
    __shared__ __align__(16) uint32_t sh_grid[kGridWords<T> > 0 ? kGridWords<T> : 4];
    __shared__ int sh_src[kMmqTok], sh_dst[kMmqTok], sh_grp[4];
    const MmqI8Lds L{sh_q0, sh_q1, sh_d, *(uint8_t (*)[2][kMmqTok * kRowS]) sh_s, sh_src, sh_dst, sh_grp, sh_grid};
    MmqArgs a;
    int g, wb;
    bool one;
    if (!mmq_item<true>(m, sh, a, g, wb, one)) return;
    if (one) mmq_group_i8<T, GLU, 1, false>(a, g, wb, L);
    else mmq_group_i8<T, GLU, 2, false>(a, g, wb, L);
}

template <bool GLU> const void *mmq_i8_kernel(int type) {
    switch (type) {
        case T_Q8_0: return (const void *) k_mmq_i8<T_Q8_0, GLU>;
        case T_Q4_K: return (const void *) k_mmq_i8<T_Q4_K, GLU>;
        case T_Q5_K: return (const void *) k_mmq_i8<T_Q5_K, GLU>;
        case T_IQ4_XS: return (const void *) k_mmq_i8<T_IQ4_XS, GLU>;
        case T_IQ3_XXS: return (const void *) k_mmq_i8<T_IQ3_XXS, GLU>;
        case T_IQ3_S: return (const void *) k_mmq_i8<T_IQ3_S, GLU>;
    }
    return nullptr;
}
}  // namespace
}  // namespace fns
