// rk_attn_long.hip — decode attention over contexts past kAttLongCtx
// positions (internal/llm/model.go:575-591): the same scores, softmax and
// value sums, in the same order, as the shorter contexts' kernels: the scores
// here, the values in rk_attn_long.h.
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

#include "rk_dev.h"
#include "rk_fused.h"

namespace rk {

namespace {

constexpr int kLongHs = 128;       // head size of the scores kernel
constexpr int kLongTile = 64;      // positions a scores workgroup
constexpr int kLongMaxMul = 16;    // query heads a kv head
constexpr int kLongSplitLog2 = 2;  // four scores workgroups a kv head and tile, or one
constexpr int kLongWgs = 512;      // scores workgroups that keep the chip busy

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

}  // namespace rk
