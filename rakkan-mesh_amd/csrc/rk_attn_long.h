// rk_attn_long.h — softmax and weighted values of a position that sees more
// than kVrMaxCtx positions: the body of att_values_long_kernel
// (rk_attn_long.hip says what bounds it), for gfx950.
#pragma once

#include "rk_attn_reg.h"

namespace rk {

constexpr int kLongThreads = 512;  // waves 0-3 (0 adds), waves 4-7 load and multiply
constexpr int kLongWaves = kLongThreads / 64;
constexpr int kLongSlice = 32;     // elements a workgroup
constexpr int kLongChunk = 256;    // positions a product tile

// Softmax and weighted values of a 32-element slice of one head (workgroup
// x of token y): Go max, e_t = Exp32(s_t - max), the sum, inv = Recip32(sum),
// then out_i = Σ_t (e_t·inv)·v_t,i in t order from +0. Chunk c's products
// stand transposed and swizzled in tile c mod 2 while wave 0 adds them; waves
// 4-7 meanwhile write chunk c+1's from registers and request chunk c+3.
// (T > kVrMaxCtx.)
__device__ __forceinline__ void att_values_long_body(const float *att, int32_t att_stride, const float *vals,
                                                     float *out, const int32_t *ctl, const AttBatch &bt, int kv_mul,
                                                     int hs, int kv_dim, int nsl, int ctx_pad, int8_t *qx, float *xs,
                                                     int32_t *xsum) {
    extern __shared__ __align__(16) float smem[];
    __shared__ float s_red[kLongWaves];
    __shared__ float s_inv;
    __shared__ __align__(16) float s_res[kLongSlice];
    float *sa = smem;               // [ctx_pad] scores -> e_t
    float *tiles = smem + ctx_pad;  // [2][32][kLongChunk] products, swizzled rows
    const int z = blockIdx.y;
    const int T = att_position(ctl, bt, z) + 1;
    const int nch = (T + kLongChunk - 1) / kLongChunk;
    const int h = blockIdx.x / nsl, e0 = (blockIdx.x % nsl) * kLongSlice;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int u = tid - 256, fq = u & 7, pq = u >> 3;  // waves 4-7: float4 column, position quads pq and pq + 32
    const float *vb = vals + att_cache(bt, z) + (int64_t)(h / kv_mul) * hs + e0 + 4 * fq;
    float4 va[2][4], vc[2][4];  // even and odd chunks on their way: [quad][position in it]
    // positions past T - 1 load T - 1's values (their products are never summed)
    auto load = [&](float4 (&v)[2][4], int c) {
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                v[q][j] = *reinterpret_cast<const float4 *>(
                    vb + (int64_t)min(c * kLongChunk + 4 * (pq + 32 * q) + j, T - 1) * kv_dim);
    };
    // the head's scores, eight in flight a thread; the first before the values
    // (loads arrive in order)
    const float *ah = att + (int64_t)z * bt.att_stride + (int64_t)h * att_stride;
    float sv[8];
    auto scores = [&](int t0) {
#pragma unroll
        for (int k = 0; k < 8; k++) sv[k] = ah[min(t0 + tid + k * kLongThreads, T - 1)];
    };
    scores(0);
    if (wave >= 4) {
        load(va, 0);
        load(vc, 1);
    }
    float m = sv[0];
    for (int t0 = 0;;) {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int t = t0 + tid + k * kLongThreads;
            if (t < T) {
                sa[t] = sv[k];
                m = gomax(m, sv[k]);
            }
        }
        t0 += 8 * kLongThreads;
        if (t0 >= T) break;
        scores(t0);
    }
    m = wave_gomax(m);
    if (lane == 0) s_red[wave] = m;
    __syncthreads();
    m = s_red[0];
#pragma unroll
    for (int w = 1; w < kLongWaves; w++) m = gomax(m, s_red[w]);
    for (int t = tid; t < T; t += kLongThreads) sa[t] = exp32(sa[t] - m);
    __syncthreads();
    if (tid == 0) s_inv = recip32(lds_chain_sum(sa, T, 0.0f));
    __syncthreads();
    const float inv = s_inv;

    auto products = [&](const float4 (&v)[2][4], int c) {
        float *tile = tiles + (c & 1) * (kLongSlice * kLongChunk);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int qd = pq + 32 * q;  // the quad within the chunk
            const float4 e4 = *reinterpret_cast<const float4 *>(sa + min(c * kLongChunk + 4 * qd, ctx_pad - 4));
            const float4 a4 = make_float4(e4.x * inv, e4.y * inv, e4.z * inv, e4.w * inv);
            const float4 p[4] = {make_float4(a4.x * v[q][0].x, a4.y * v[q][1].x, a4.z * v[q][2].x, a4.w * v[q][3].x),
                                 make_float4(a4.x * v[q][0].y, a4.y * v[q][1].y, a4.z * v[q][2].y, a4.w * v[q][3].y),
                                 make_float4(a4.x * v[q][0].z, a4.y * v[q][1].z, a4.z * v[q][2].z, a4.w * v[q][3].z),
                                 make_float4(a4.x * v[q][0].w, a4.y * v[q][1].w, a4.z * v[q][2].w, a4.w * v[q][3].w)};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = 4 * fq + j;
                reinterpret_cast<float4 *>(tile + i * kLongChunk)[qd ^ vr_swz(i)] = p[j];
            }
        }
    };
    float acc = 0.0f;
    auto sums = [&](int c) {
        if (lane < kLongSlice)
            acc = swz_chain_sum(tiles + (c & 1) * (kLongSlice * kLongChunk) + lane * kLongChunk,
                                min(kLongChunk, T - c * kLongChunk), vr_swz(lane), acc);
    };
    // Each role has a loop of its own, nch barriers each: with both in one, the
    // loaded values meet at its joins and are copied there, which waits for
    // loads just issued. While five chunks are left the loads stand without a
    // test (it would make the compiler wait too); the last chunks load nothing
    // that nobody reads, for a launch ends when its loads have. (nch >= 5.)
    if (wave >= 4) {
        products(va, 0);
        load(va, 2);
        __syncthreads();
        int c = 0;
        for (; c + 4 < nch; c += 2) {
            products(vc, c + 1);
            __builtin_amdgcn_sched_barrier(0);  // the loads into the registers just read, not into others
            load(vc, c + 3);
            __syncthreads();
            products(va, c + 2);
            __builtin_amdgcn_sched_barrier(0);
            load(va, c + 4);
            __syncthreads();
        }
        const bool four = nch - c > 3;  // three or four chunks are left
        products(vc, c + 1);
        if (four) load(vc, c + 3);
        __syncthreads();
        products(va, c + 2);
        __syncthreads();
        if (four) {
            products(vc, c + 3);
            __syncthreads();
        }
        return;
    }
    for (int c = 0; c < nch; c++) {
        __syncthreads();
        if (wave == 0) sums(c);
    }
    if (wave != 0) return;
    const int64_t base = (int64_t)z * bt.out_stride + (int64_t)h * hs + e0;
    if (lane < kLongSlice) out[base + lane] = acc;
    if (qx) {
        // the slice is one Q8_0 block of the next input: lanes 0-7 take
        // four values each
        if (lane < kLongSlice) s_res[lane] = acc;
        const float4 v4 = reinterpret_cast<const float4 *>(s_res)[min(lane, 7)];
        float d;
        int cs;
        const uint32_t pk = quantize_group(v4.x, v4.y, v4.z, v4.w, d, cs);
        if (lane < 8) {
            reinterpret_cast<uint32_t *>(qx + base)[lane] = pk;
            if (lane == 0) {
                xs[base >> 5] = d;
                xsum[base >> 5] = cs;
            }
        }
    }
}

}  // namespace rk
