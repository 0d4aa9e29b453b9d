// fns_q8x8.hpp - Q8_1 of eight consecutive values per lane, and the RMSNorm of a row built on it.
//
// A 32-value block lies on four lanes of a quad (lane q = lane % 4 holds values 8 q .. 8 q + 7), so the block's max and
// sums take two quad exchanges per value instead of the five row exchanges of the one-value-per-lane form
// (fns_lanes.hpp): a row of 2048 columns is one 256-thread workgroup with 8 values a thread, all of its loads in flight
// together. The f32 sum keeps the one-value form's order - butterfly offsets 16, 8 (across lanes), then 4, 2, 1 (inside
// a lane) - so the blocks are the same bit for bit.
#pragma once

#include "fns_common.hpp"

namespace fns::dev {

struct Q8x8 {
    int q[8];
    float d, sum;  // the block's d = amax / 127 and the f32 sum of its values (every lane of the quad)
};
// All four lanes of a block must be active.
__device__ __forceinline__ Q8x8 q8_1_x8(const float (&v)[8]) {
    Q8x8 r;
    float amax = fabsf(v[0]), s[8];  // (not from 0: a block of NaNs keeps a NaN scale, as in the one-value form)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        amax = fmaxf(amax, fabsf(v[k]));
        s[k] = v[k] + xor_lane<2>(v[k]);  // offset 16
    }
    amax = lanes_max<4>(amax);
#pragma unroll
    for (int k = 0; k < 8; ++k) s[k] += xor_lane<1>(s[k]);  // offset 8
    r.sum = ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
    r.d = amax / 127.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) r.q[k] = amax == 0.0f ? 0 : (int) (int8_t) roundf(v[k] / r.d);
    return r;
}
// The lane's part of the reference's 36-byte block at column col (a multiple of 8) of the row y.
__device__ __forceinline__ void q8_1_store_x8(const Q8x8 &r, uint8_t *y, int col) {
    uint32_t *b = (uint32_t *) (y + (size_t) (col / 32) * 36);
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k / 4] |= (uint32_t) (uint8_t) (int8_t) r.q[k] << (8 * (k % 4));
    const int q = (col / 8) % 4;
    b[1 + 2 * q] = w[0];
    b[2 + 2 * q] = w[1];
    if (q == 0) b[0] = float_to_half(r.d) | (float_to_half(r.sum) << 16);
}

// RMSNorm of one row (n a multiple of 32, n <= 2048 C, x, w and out 16-byte aligned) by 256 threads, then its Q8_1
// blocks into y (padded to 512 columns with zeros; null: none) and sink(v, q, col) for every column group below n. xs: 2048 C
// floats of LDS. The sum of squares keeps the order of the row walked 256 columns at a time (thread t sums columns t,
// t + 256, ...), which the eight-column loads would change: the row goes through LDS once. Columns past n are zeros
// and add nothing.
template <int C, class Sink>
__device__ __forceinline__ void rms_norm_row(const float *__restrict__ xr, const float *__restrict__ w,
                                             float *__restrict__ out, uint8_t *__restrict__ y, int n, float eps,
                                             float *xs, Sink sink) {
    __shared__ float red[4];
    const int tid = threadIdx.x;
    float v[C][8], wv[C][8];
#pragma unroll
    for (int c = 0; c < C; ++c) {  // clamped, unconditional loads: all in flight together
        const int col = min((256 * c + tid) * 8, n - 8);
        const float4 a0 = *(const float4 *) (xr + col), a1 = *(const float4 *) (xr + col + 4);
        const float4 b0 = *(const float4 *) (w + col), b1 = *(const float4 *) (w + col + 4);
        v[c][0] = a0.x, v[c][1] = a0.y, v[c][2] = a0.z, v[c][3] = a0.w;
        v[c][4] = a1.x, v[c][5] = a1.y, v[c][6] = a1.z, v[c][7] = a1.w;
        wv[c][0] = b0.x, wv[c][1] = b0.y, wv[c][2] = b0.z, wv[c][3] = b0.w;
        wv[c][4] = b1.x, wv[c][5] = b1.y, wv[c][6] = b1.z, wv[c][7] = b1.w;
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int col = (256 * c + tid) * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k) v[c][k] = col < n ? v[c][k] : 0.0f;
        *(float4 *) (xs + col) = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
        *(float4 *) (xs + col + 4) = make_float4(v[c][4], v[c][5], v[c][6], v[c][7]);
    }
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 8 * C; ++j) {
        const float x = xs[tid + 256 * j];
        s += x * x;
    }
    s = lanes_sum<64>(s);
    if (tid % 64 == 0) red[tid / 64] = s;
    __syncthreads();
    s = (red[0] + red[1]) + (red[2] + red[3]);
    const float scale = 1.0f / sqrtf(s / n + eps);
    const int npad = (n + 511) / 512 * 512;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int col = (256 * c + tid) * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k) v[c][k] = col < n ? scale * v[c][k] * wv[c][k] : 0.0f;
        const Q8x8 q = q8_1_x8(v[c]);
        if (col < n) {
            *(float4 *) (out + col) = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
            *(float4 *) (out + col + 4) = make_float4(v[c][4], v[c][5], v[c][6], v[c][7]);
            sink(q, col);
        }
        if (y && col < npad) q8_1_store_x8(q, y, col);
    }
}

}  // namespace fns::dev
