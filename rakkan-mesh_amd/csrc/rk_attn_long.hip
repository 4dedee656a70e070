// rk_attn_long.hip — decode attention over contexts past kAttLongCtx
// positions (internal/llm/model.go:575-591): the same scores, softmax and
// value sums, in the same order, as the shorter contexts' kernels.
//
// What bounds a long context: two chains of T dependent float32 adds, the
// softmax's sum and then each output element's (about 8.7 cycles an add: 22
// us each at 6000 positions). So nothing else may stand in their way:
//  * The scores of a kv head's query heads share a workgroup, which holds 64
//    positions' keys in registers: each key row is read once, not once a
//    query head (6000 positions, 28 heads on 4: 13.4 -> 5.4 us).
//  * Four waves load the values two chunks ahead and multiply one ahead, one
//    wave only adds (the sums 25.5 us of a launch; the launch 65.9 -> 54).
// Forming the softmax's sum in parallel (exactly: the sum as an integer on
// its binade's grid, each thread's terms as how far they move an even and an
// odd one, a scan, again after each thread that leaves the binade) measured
// slower: 2.7 us a scan, and rows whose terms grow towards the last position
// leave a binade every few threads (35-56 us against the chain's 22).
#include <algorithm>
#include <mutex>

#include "rk_attn_reg.h"
#include "rk_dev.h"
#include "rk_fused.h"

namespace rk {

namespace {

constexpr int kLongHs = 128;       // head size of the scores kernel
constexpr int kLongTile = 64;      // positions a scores workgroup
constexpr int kLongMaxMul = 16;    // query heads a kv head
constexpr int kLongSplitLog2 = 2;  // four scores workgroups a kv head and tile, or one
constexpr int kLongWgs = 512;      // scores workgroups that keep the chip busy
constexpr int kLongThreads = 512;  // values: waves 0-3 (0 adds), waves 4-7 load and multiply
constexpr int kLongWaves = kLongThreads / 64;
constexpr int kLongSlice = 32;     // elements a workgroup
constexpr int kLongChunk = 256;    // positions a product tile

}  // namespace

// Scores of kLongTile positions for query heads of one kv head (size 128):
// thread (position tid/4, part tid%4) keeps its key's elements 8·part .. +7 of
// each 32-element step in registers and runs the heads over them, as
// quad_dot32 (the running sums j = 8·part .. +7, combined by DPP). A kv head's
// 2^split_log2 workgroups share its query heads while the positions so far leave
// workgroups of the chip idle; from there on the first takes them all.
__global__ __launch_bounds__(256) void att_scores_long_kernel(const float *q, const float *keys, float *att,
                                                              int32_t att_stride, const int32_t *ctl, AttBatch bt,
                                                              int kv_heads, int kv_mul, int split_log2, int kv_dim,
                                                              float inv_sqrt) {
    __shared__ __align__(16) float sq[kLongMaxMul * kLongHs];
    const int z = (int)blockIdx.z >> split_log2;
    const int T = att_position(ctl, bt, z) + 1;
    const int t0 = blockIdx.y * kLongTile;
    if (t0 >= T) return;
    const int g = blockIdx.x;
    int m0 = 0, m1 = kv_mul;  // the workgroup's query heads of the kv head's
    if (split_log2) {         // uniform (the divisions take 0.5 us)
        // the shares lie in z, so that the first ones alone go round the XCDs
        const int split = 1 << split_log2, part_of = (int)blockIdx.z & (split - 1);
        // workgroups with one a kv head and tile
        const int whole = kv_heads * ((T + kLongTile - 1) / kLongTile) * ((int)gridDim.z >> split_log2);
        const int parts = min(split, max(1, kLongWgs / whole));
        const int share = (kv_mul + parts - 1) / parts;
        m0 = part_of * share;
        m1 = min(kv_mul, m0 + share);
        if (m0 >= kv_mul) return;
    }
    const int h0 = g * kv_mul;
    const int part = threadIdx.x & 3, t = t0 + (threadIdx.x >> 2);
    const float *kt = keys + att_cache(bt, z) + (int64_t)min(t, T - 1) * kv_dim + (int64_t)g * kLongHs + 8 * part;
    float4 k0[kLongHs / 32], k1[kLongHs / 32];
#pragma unroll
    for (int st = 0; st < kLongHs / 32; st++) {
        k0[st] = *reinterpret_cast<const float4 *>(kt + 32 * st);
        k1[st] = *reinterpret_cast<const float4 *>(kt + 32 * st + 4);
    }
    const float *qh = q + (int64_t)z * bt.q_stride + (int64_t)h0 * kLongHs;
    for (int i = m0 * (kLongHs / 4) + threadIdx.x; i < m1 * (kLongHs / 4); i += 256)
        reinterpret_cast<float4 *>(sq)[i] = reinterpret_cast<const float4 *>(qh)[i];
    __syncthreads();
    att += (int64_t)z * bt.att_stride;
    for (int m = m0; m < m1; m++) {
        float s[8];
#pragma unroll
        for (int k = 0; k < 8; k++) s[k] = 0.0f;
#pragma unroll
        for (int st = 0; st < kLongHs / 32; st++) {
            const float *qp = sq + m * kLongHs + 32 * st + 8 * part;
            const float4 q0 = *reinterpret_cast<const float4 *>(qp), q1 = *reinterpret_cast<const float4 *>(qp + 4);
            s[0] += q0.x * k0[st].x;
            s[1] += q0.y * k0[st].y;
            s[2] += q0.z * k0[st].z;
            s[3] += q0.w * k0[st].w;
            s[4] += q1.x * k1[st].x;
            s[5] += q1.y * k1[st].y;
            s[6] += q1.z * k1[st].z;
            s[7] += q1.w * k1[st].w;
        }
        float e[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float u = s[k] + dppf_x1(s[k]);
            e[k] = u + dppf_x2(u);
        }
        const float dot = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
        if (part == 0 && t < T) att[(int64_t)(h0 + m) * att_stride + t] = dot * inv_sqrt;
    }
}

// Softmax and weighted values of a 32-element slice of one head (workgroup
// x of token y): Go max, e_t = Exp32(s_t - max), the sum, inv = Recip32(sum),
// then out_i = Σ_t (e_t·inv)·v_t,i in t order from +0. Chunk c's products
// stand transposed and swizzled in tile c mod 2 while wave 0 adds them; waves
// 4-7 meanwhile write chunk c+1's from registers and request chunk c+3. A
// position that sees at most kVrMaxCtx takes att_values_reg_body (position 50
// of a context of 8192: 7.0 us here, 4.9 there).
__global__ __launch_bounds__(kLongThreads) void att_values_long_kernel(const float *att, int32_t att_stride,
                                                                       const float *vals, float *out,
                                                                       const int32_t *ctl, AttBatch bt, int kv_mul,
                                                                       int hs, int kv_dim, int nsl, int ctx_pad,
                                                                       int8_t *qx, float *xs, int32_t *xsum) {
    extern __shared__ __align__(16) float smem[];
    __shared__ float s_red[kLongWaves];
    __shared__ float s_inv;
    __shared__ __align__(16) float s_res[kLongSlice];
    float *sa = smem;               // [ctx_pad] scores -> e_t
    float *tiles = smem + ctx_pad;  // [2][32][kLongChunk] products, swizzled rows
    const int z = blockIdx.y;
    const int T = att_position(ctl, bt, z) + 1;
    if (T <= kVrMaxCtx) {  // uniform
        att_values_reg_body<false>(att, att_stride, vals, out, ctl, bt, kv_mul, hs, kv_dim, nsl, ctx_pad, qx, xs, xsum,
                                   blockIdx.x, z, nullptr, 0);
        return;
    }
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

bool launch_att_scores_long(const float *q, const float *keys, float *att, int32_t att_stride, const int32_t *ctl,
                            const AttBatch &bt, int ctx, int heads, int kv_heads, int hs, int kv_dim, float inv_sqrt,
                            hipStream_t s) {
    const int kv_mul = heads / kv_heads;
    if (ctx <= kAttLongCtx || hs != kLongHs || kv_mul < 2 || kv_mul > kLongMaxMul || kv_dim % 4 != 0 ||
        bt.q_stride % 4 != 0 || ((reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(q)) & 15) != 0 ||
        bt.cache_stride % 4 != 0)
        return false;
    const int npos = att_positions(ctl, bt, ctx);
    const int tokens = ctl ? 1 : bt.tokens, tiles = (npos + kLongTile - 1) / kLongTile;
    // More than four query heads in turn take longer than a launch's start and
    // end (16 of one kv head, positions up to 4000: 6.5-7.3 us, shared by four
    // workgroups 3.8-4.1; 7 of one 4.1-4.7 and 3.9-4.1), but workgroups that
    // exit at once cost too (32768 of them 9 us more than 8192).
    const int64_t wgs = (int64_t)kv_heads * tokens * tiles;
    const int split_log2 = kv_mul > 4 && wgs <= 1024 ? kLongSplitLog2 : 0;
    const dim3 grid(kv_heads, tiles, tokens << split_log2);
    RK_LAUNCH(att_scores_long_kernel, grid, dim3(256), 0, s, q, keys, att, att_stride, ctl, bt, kv_heads, kv_mul,
              split_log2, kv_dim, inv_sqrt);
    return true;
}

bool launch_att_values_long(const float *att, int32_t att_stride, const float *vals, float *out, const int32_t *ctl,
                            const AttBatch &bt, int ctx, int heads, int kv_heads, int hs, int kv_dim, int8_t *qx,
                            float *xs, int32_t *xsum, hipStream_t s) {
    const int ctx_pad = (ctx + 3) & ~3;
    const size_t lds = ((size_t)ctx_pad + 2 * kLongSlice * kLongChunk) * 4;
    if (ctx <= kAttLongCtx || hs % kLongSlice != 0 || kv_dim % 4 != 0 || bt.cache_stride % 4 != 0 ||
        (reinterpret_cast<uintptr_t>(vals) & 15) != 0 || lds > kMaxLdsBytes - 2048)
        return false;
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute((const void *)att_values_long_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)(kMaxLdsBytes - 2048));
    });
    const int nsl = hs / kLongSlice;
    RK_LAUNCH(att_values_long_kernel, dim3(heads * nsl, ctl ? 1 : bt.tokens), dim3(kLongThreads), lds, s, att,
              att_stride, vals, out, ctl, bt, heads / kv_heads, hs, kv_dim, nsl, ctx_pad, qx, xs, xsum);
    return true;
}

}  // namespace rk
