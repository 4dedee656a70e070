// rk_attn_reg.h — softmax and weighted values of a position that sees at most
// kVrMaxCtx positions, the values held in registers, for gfx950: the body of
// att_values_reg_kernel and of the longer contexts' kernel at such positions.
#pragma once

#include "rk_dev.h"
#include "rk_fused.h"
#include "rk_sync.h"

namespace rk {

constexpr int kValSlice = 32;  // elements of a head a values workgroup forms

// Every position's values of the slice are in registers from the start. Waves
// 0-3 take the scores and the softmax as att_values_kernel does (lane 0 of wave 0 adds the
// e_t); waves 4-7 load the slice's values of chunks of kVrChunk positions
// (two position quads of one float4 column a thread a chunk, loads only
// for chunks below T) and, once inv is known, write a chunk's products
// a_t·v_t,i transposed into a tile while wave 0 adds the previous chunk's
// (lane i < 32: its element's products in position order). Tile row i
// keeps logical float4 q of the row at q ^ vr_swz(i): with that swizzle
// both the products' 16-byte writes (eight lanes: eight rows 4 apart, one
// column) and the sums' reads (eight lanes: eight consecutive rows, one
// logical column) touch 32 distinct banks.
constexpr int kVrThreads = 512;
constexpr int kVrChunk = 256;
constexpr int kVrMaxChunks = 4;
constexpr int kVrMaxCtx = kVrChunk * kVrMaxChunks;

// The body of att_values_reg_kernel for workgroup bx of token z. SIG: the
// values launch that also runs the Wo product (att_values_wo_kernel): the
// slice's Q8_0 block is stored through to the device's coherence point and
// the workgroup then counts itself done in `sync` (sync_signal_done).
template <bool SIG>
__device__ __forceinline__ void att_values_reg_body(const float *att, int32_t att_stride, const float *vals,
                                                    float *out, const int32_t *ctl, const AttBatch &bt, int kv_mul,
                                                    int hs, int kv_dim, int nsl, int ctx_pad, int8_t *qx, float *xs,
                                                    int32_t *xsum, int bx, int z, unsigned long long *sync, int na) {
    extern __shared__ __align__(16) float smem[];
    __shared__ float s_red[4];
    __shared__ float s_inv;
    __shared__ __align__(16) float s_res[kValSlice];
    float *sa = smem;               // [ctx_pad] scores -> e_t
    float *tiles = smem + ctx_pad;  // [2][32][kVrChunk] products, swizzled rows
    const int T = att_position(ctl, bt, z) + 1;
    const int nch = (T + kVrChunk - 1) / kVrChunk;
    att += (int64_t)z * bt.att_stride;
    out += (int64_t)z * bt.out_stride;
    vals += att_cache(bt, z);
    if (qx) {
        qx += (int64_t)z * bt.out_stride;
        xs += (int64_t)z * (bt.out_stride >> 5);
        xsum += (int64_t)z * (bt.out_stride >> 5);
    }
    const int h = bx / nsl, e0 = (bx % nsl) * kValSlice;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // waves 4-7: float4 column fq (elements 4fq..4fq+3) and position quads
    // pq, pq + 32 of each chunk
    const int u = tid - 256, fq = u & 7, pq = u >> 3;
    float4 vr[kVrMaxChunks][2][4];  // [chunk][quad][position in the quad]
    float sc[4];
    if (wave < 4) {
        const float *ah = att + (int64_t)h * att_stride;
#pragma unroll
        for (int k = 0; k < 4; k++) sc[k] = ah[min(tid + 256 * k, T - 1)];
        float m = sc[0];
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (tid + 256 * k < T) m = gomax(m, sc[k]);
        m = wave_gomax(m);
        if (lane == 0) s_red[wave] = m;
    } else {
        // positions past T-1 load T-1's values (their products are never summed)
        const float *vb = vals + (int64_t)(h / kv_mul) * hs + e0 + 4 * fq;
#pragma unroll
        for (int c = 0; c < kVrMaxChunks; c++)
            if (c < nch) {  // uniform
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int t = min(c * kVrChunk + 4 * (pq + 32 * q) + j, T - 1);
                        vr[c][q][j] = *reinterpret_cast<const float4 *>(vb + (int64_t)t * kv_dim);
                    }
            }
    }
    __syncthreads();
    if (wave < 4) {
        float m = s_red[0];
#pragma unroll
        for (int w = 1; w < 4; w++) m = gomax(m, s_red[w]);
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (tid + 256 * k < T) sa[tid + 256 * k] = exp32(sc[k] - m);
    }
    __syncthreads();
    if (tid == 0) s_inv = recip32(lds_chain_sum(sa, T, 0.0f));
    __syncthreads();
    const float inv = s_inv;

    // chunk c's products into tile c mod 2 (waves 4-7); positions past T
    // take a clamped weight and give products that are never summed
    auto products = [&](int c) {
        float *tile = tiles + (c & 1) * (kValSlice * kVrChunk);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int qd = pq + 32 * q;  // the quad within the chunk
            const float4 e4 = *reinterpret_cast<const float4 *>(sa + min(c * kVrChunk + 4 * qd, ctx_pad - 4));
            const float4 a4 = make_float4(e4.x * inv, e4.y * inv, e4.z * inv, e4.w * inv);
            const float4(&v)[4] = vr[c][q];
            const float4 p[4] = {make_float4(a4.x * v[0].x, a4.y * v[1].x, a4.z * v[2].x, a4.w * v[3].x),
                                 make_float4(a4.x * v[0].y, a4.y * v[1].y, a4.z * v[2].y, a4.w * v[3].y),
                                 make_float4(a4.x * v[0].z, a4.y * v[1].z, a4.z * v[2].z, a4.w * v[3].z),
                                 make_float4(a4.x * v[0].w, a4.y * v[1].w, a4.z * v[2].w, a4.w * v[3].w)};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = 4 * fq + j;
                reinterpret_cast<float4 *>(tile + i * kVrChunk)[qd ^ vr_swz(i)] = p[j];
            }
        }
    };
    if (wave >= 4) products(0);
    __syncthreads();
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < kVrMaxChunks; c++) {
        if (c < nch) {  // uniform
            if (wave == 0) {
                if (lane < kValSlice)
                    acc = swz_chain_sum(tiles + (c & 1) * (kValSlice * kVrChunk) + lane * kVrChunk,
                                        min(kVrChunk, T - c * kVrChunk), vr_swz(lane), acc);
            } else if (wave >= 4 && c + 1 < nch) {
                products(c + 1);
            }
            __syncthreads();
        }
    }
    if (wave != 0) return;
    if (lane < kValSlice) out[(int64_t)h * hs + e0 + lane] = acc;
    if (qx) {
        // the slice is one Q8_0 block of the next input: lanes 0-7 take
        // four values each
        if (lane < kValSlice) s_res[lane] = acc;
        const int q = min(lane, 7);
        const float4 v4 = reinterpret_cast<const float4 *>(s_res)[q];
        float d;
        int cs;
        const uint32_t pk = quantize_group(v4.x, v4.y, v4.z, v4.w, d, cs);
        const int64_t base = (int64_t)h * hs + e0;
        if (SIG) {
            // agent-scope stores (written through to where every XCD's
            // loads of that scope look), complete before the count
            if (lane < 8) {
                __hip_atomic_store(reinterpret_cast<uint32_t *>(qx + base) + lane, pk, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                if (lane == 0) {
                    __hip_atomic_store(xs + (base >> 5), d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    xsum[base >> 5] = cs;
                }
            }
            sync_signal_done(sync, na);
        } else if (lane < 8) {
            reinterpret_cast<uint32_t *>(qx + base)[lane] = pk;
            if (lane == 0) {
                xs[base >> 5] = d;
                xsum[base >> 5] = cs;
            }
        }
    }
}

}  // namespace rk
