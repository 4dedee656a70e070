// rk_tensor.hip — the rakkan_tensor_v1 operators on this path
// (internal/sandbox/tensor.go): matmul / matmul_t in f32 and i8, and the
// quantize / scale that produce and consume the i8 form.
//
// f32 (tensor.go:318-327): c_ij = Canonical(acc), acc += float32(a_ip·b_pj)
// for p = 0..k-1 from +0, a sequential sum per output. The products of a
// 16x16 tile at one position are an outer product: v_mfma_f32_16x16x1 with a
// zero accumulator gives four positions' rounded products at once (a K = 1
// result is one product plus +0: only the sign of a zero is lost, and a sum
// that starts at +0 never is -0, so adding either zero leaves it), and the
// vector ALU does the adds alone, in order. What bounds it: an add and a
// product a position, 16 adds (2.3 cycles each) and one matrix instruction
// (34 cycles) per 1024 products, which measured one after the other on
// MI355X, not together: 24.5 us of a 1024 x 784 x 1024 product. It takes 35-36
// us (two outputs a side a thread from LDS, products on the vector ALU: 64,
// and 82 with inputs not in the caches): operand reads, tests and the loads'
// latency are the rest.
//
// i8 (tensor.go:328-335): c_ij = Σ int32(a_ip)·int32(b_pj) with Go's int32
// wraparound. Integer sums are exact in any order, so the sums run on int8
// MFMA (v_mfma_i32_16x16x64_i8, accumulator chained); the accumulator
// restarts every 65536 positions (|partial| <= 2^30, no overflow inside the
// matrix core) and the partials are added with wrapping integer adds. What
// bounds it: LDS reads and the staging of slices (16 bytes a lane and row;
// b[k][n] turned in registers, 4x4 bytes at a time, so that both operands
// read 16 positions of a row or column as one LDS load). 2048^3: 22-23 us, 380
// TMAC/s (20 us with b[n][k]), against 221 us with byte loads, 8-byte LDS
// reads and no load in flight during the sums.
//
// Both load the next slice while this one is summed (two LDS slices, one
// barrier a slice). A slice that is whole takes no tests: a test around a
// load makes the compiler wait for it there.
#include <algorithm>
#include <mutex>

#include "rk_dev.h"
#include "rk_kernels.h"
#include "rk_runtime.h"

namespace rk {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int rk_i2 __attribute__((ext_vector_type(2)));

constexpr int kTileRow = 1 << 20;  // workgroups of a grid row (tile_grid)

// Tile order: workgroup ids (tile_grid's rows one after the other, each a
// multiple of 8) go round the 8 XCDs, so id mod 8 picks a contiguous run of
// tiles (along n first): an XCD's workgroups then share rows of a and columns
// of b in its own L2. -1: past the last tile.
__device__ __forceinline__ int64_t xcd_tile(int64_t tiles) {
    const int64_t id = (int64_t)blockIdx.y * kTileRow + blockIdx.x;
    const int64_t per = (tiles + 7) >> 3, t = (id & 7) * per + (id >> 3);
    return (id >> 3) < per && t < tiles ? t : -1;
}

// ---- f32 ----
constexpr int kTfTile = 32;    // outputs per side of a workgroup: 16 per side a wave
constexpr int kTfChunk = 64;   // positions per staged slice
constexpr int kTfPitch = kTfChunk + 4;
constexpr int kTfLoads = kTfTile * kTfChunk / 4 / 256;  // 16-byte loads a thread and operand

typedef float v16f __attribute__((ext_vector_type(16)));

// Four floats from `at` of an array of `total` (>= 4), zeros past the first
// `valid`: near the array's end the load moves back into it and what
// precedes `at` is dropped.
__device__ __forceinline__ float4 tf_edge4(const float *x, int64_t at, int64_t total, int64_t valid) {
    const int64_t q = min(at, total - 4);
    const int o = (int)min(at - q, (int64_t)4);
    float4 v;
    __builtin_memcpy(&v, x + q, 16);
    if (o & 1) v = make_float4(v.y, v.z, v.w, 0.0f);
    if (o & 2) v = make_float4(v.z, v.w, 0.0f, 0.0f);
    if (o & 4) v.x = 0.0f;
    return make_float4(valid > 0 ? v.x : 0.0f, valid > 1 ? v.y : 0.0f, valid > 2 ? v.z : 0.0f, valid > 3 ? v.w : 0.0f);
}

template <bool TRANS>
__global__ __launch_bounds__(256, 4) void tensor_mm_f32_kernel(const float *a, const float *b, float *c, int64_t m,
                                                               int64_t k, int64_t n) {
    __shared__ __align__(16) float sa[2][kTfTile][kTfPitch];  // rows of a
    __shared__ __align__(16) float sb[2][kTfTile][kTfPitch];  // columns of b
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lq = lane >> 4, ln = lane & 15;
    const int64_t tn = (n + kTfTile - 1) / kTfTile;
    const int64_t t = xcd_tile((m + kTfTile - 1) / kTfTile * tn);
    if (t < 0) return;  // uniform
    const int64_t i0 = t / tn * kTfTile, j0 = t % tn * kTfTile;
    // a slice's loads; rows past m and columns past n repeat others (never
    // stored); positions past k are zeros, whose products add +0. Whole
    // slices (all but the last; b[k][n]'s last columns read on into the next
    // row, so there whole slices end before the last row) take no tests.
    float4 va[kTfLoads], vb[kTfLoads];
    const float *ra[kTfLoads], *rb[kTfLoads];
#pragma unroll
    for (int e = 0; e < kTfLoads; e++) {
        const int u = tid + 256 * e, r = u / (kTfChunk / 4), p = 4 * (u % (kTfChunk / 4));
        ra[e] = a + min(i0 + r, m - 1) * k + p;
        const int64_t j = j0 + 4 * (u % (kTfTile / 4));
        rb[e] = TRANS ? b + min(j0 + r, n - 1) * k + p : b + (u / (kTfTile / 4)) * n + (j < n ? j : 0);
    }
    const int64_t whole = TRANS || n % 4 == 0 ? k : k - 4;
    auto load = [&](int64_t p0) {
        if (p0 + kTfChunk <= whole) {  // uniform
#pragma unroll
            for (int e = 0; e < kTfLoads; e++) {
                __builtin_memcpy(&va[e], ra[e] + p0, 16);
                __builtin_memcpy(&vb[e], rb[e] + (TRANS ? p0 : p0 * n), 16);
            }
        } else {
#pragma unroll
            for (int e = 0; e < kTfLoads; e++) {
                const int u = tid + 256 * e, p = 4 * (u % (kTfChunk / 4));
                va[e] = tf_edge4(a, ra[e] - a + p0, m * k, k - p0 - p);
                if constexpr (TRANS)
                    vb[e] = tf_edge4(b, rb[e] - b + p0, n * k, k - p0 - p);
                else
                    vb[e] = tf_edge4(b, rb[e] - b + p0 * n, n * k, p0 + u / (kTfTile / 4) < k ? 4 : 0);
            }
        }
    };
    const int ar = 16 * (wave >> 1) + ln, bc = 16 * (wave & 1) + ln;  // the wave's row of a, column of b
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    load(0);
    int s = 0;
    auto store = [&]() {
#pragma unroll
        for (int e = 0; e < kTfLoads; e++) {
            const int u = tid + 256 * e, r = u / (kTfChunk / 4), p = 4 * (u % (kTfChunk / 4));
            *reinterpret_cast<float4 *>(&sa[s][r][p]) = va[e];
            if constexpr (TRANS) {
                *reinterpret_cast<float4 *>(&sb[s][r][p]) = vb[e];
            } else {
                const int q = u / (kTfTile / 4), j = 4 * (u % (kTfTile / 4));
                sb[s][j][q] = vb[e].x;
                sb[s][j + 1][q] = vb[e].y;
                sb[s][j + 2][q] = vb[e].z;
                sb[s][j + 3][q] = vb[e].w;
            }
        }
        __syncthreads();
    };
    auto four = [&](int p) {
        // block q of the matrix core's four takes position p + q: its four
        // results are elements 4q .. 4q + 3
        const v16f z = {};
        const v16f d = __builtin_amdgcn_mfma_f32_16x16x1f32(sa[s][ar][p + lq], sb[s][bc][p + lq], z, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] += d[4 * q + e];
    };
    int64_t p0 = 0;
    for (; p0 + kTfChunk <= k; p0 += kTfChunk, s ^= 1) {
        store();
        if (p0 + kTfChunk < k) load(p0 + kTfChunk);
#pragma unroll 4
        for (int p = 0; p < kTfChunk; p += 4) four(p);
    }
    // A last, partial slice: its positions only, up to a whole four. (Summing
    // all 64 positions of it: 2048 x 8 x 2048 19.7 us against 12.3, 100000 x 16
    // x 32 16.3 against 11.4. In the loop above, as a second case, it slowed
    // the whole slices: 2048^3 333 against 317 us.)
    if (p0 < k) {
        store();
        for (int p = 0; p < (int)(k - p0); p += 4) four(p);
    }
    // the 16x16 result layout: lane holds column ln, rows 4·lq + e
    const int64_t j = j0 + 16 * (wave & 1) + ln;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int64_t i = i0 + 16 * (wave >> 1) + 4 * lq + e;
        if (i < m && j < n) c[i * n + j] = canonical(acc[e]);
    }
}

// ---- i8 ----
constexpr int64_t kTiRestart = 65536;   // positions per matrix-core accumulation

// 16 bytes from `at` of an array of `total` (>= 16), zeros past the first
// `valid` (any alignment); near the array's end as tf_edge4.
__device__ __forceinline__ v4i ti_edge16(const int8_t *x, int64_t at, int64_t total, int64_t valid) {
    const int64_t q = min(at, total - 16);
    const int o = (int)min(at - q, (int64_t)16), keep = (int)max(min(valid, (int64_t)16), (int64_t)0);
    unsigned __int128 w;
    __builtin_memcpy(&w, x + q, 16);
    w = o < 16 ? w >> (8 * o) : 0;
    w = keep == 16 ? w : w & (((unsigned __int128)1 << (8 * keep)) - 1);
    v4i v;
    __builtin_memcpy(&v, &w, 16);
    return v;
}

// Four bytes from `at`, zeros unless `valid`, likewise.
__device__ __forceinline__ int ti_edge4(const int8_t *x, int64_t at, int64_t total, bool valid) {
    const int64_t q = min(at, total - 4);
    const int o = (int)min(at - q, (int64_t)4);
    uint32_t v;
    __builtin_memcpy(&v, x + q, 4);
    return valid && o < 4 ? (int)(v >> (8 * o)) : 0;
}

// A workgroup of four waves forms TM x TN outputs from slices of KC
// positions: WM x WN waves side by side, WK waves sharing each part's
// positions (their integer partials added at the end).
template <int TM, int TN, int KC, int WM, int WN, int WK, bool TRANS>
__global__ __launch_bounds__(256) void tensor_mm_i8_kernel(const int8_t *a, const int8_t *b, int32_t *c, int64_t m,
                                                           int64_t k, int64_t n) {
    constexpr int PITCH = KC + 16;    // bytes: 16 rows at one offset in distinct banks
    constexpr int NA = TM * KC / 16 / 256, NB = TN * KC / 16 / 256;  // 16-byte loads a thread
    constexpr int RM = TM / WM / 16, RN = TN / WN / 16;              // 16x16 results a wave
    // b[k][n]: a thread takes 8 positions of 4 columns and turns them; its
    // low lane bits spread over columns and positions so that the turned
    // columns' stores fall in distinct banks
    constexpr int CG = TN / 4, KG = 256 / CG, NU = KC / 8 / KG;
    static_assert(WM * WN * WK == 4 && NA >= 1 && NB >= 1 && NU >= 1 && CG >= 8, "four waves, whole loads");
    extern __shared__ __align__(16) int8_t ti_lds[];
    int8_t *sa = ti_lds, *sb = ti_lds + 2 * TM * PITCH;  // rows of a, columns of b, two slices each
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lq = lane >> 4, ln = lane & 15;
    const int wk = wave % WK, wn = wave / WK % WN, wm = wave / WK / WN;
    const int64_t tn = (n + TN - 1) / TN;
    const int64_t t = xcd_tile((m + TM - 1) / TM * tn);
    if (t < 0) return;  // uniform
    const int64_t i0 = t / tn * TM, j0 = t % tn * TN;
    const int cg = (tid & 3) | (tid >> 5) % (CG / 4) * 4, kg = (tid >> 2 & 7) | (tid >> 5) / (CG / 4) * 8;
    const int64_t jc = j0 + 4 * cg < n ? j0 + 4 * cg : 0;
    // as in the f32 kernel: rows and columns past the end repeat others,
    // positions past k are zeros, whole slices take no tests
    v4i va[NA], vb[NB];
    int vc[NU][8];
    const int8_t *ra[NA], *rb[NB];
#pragma unroll
    for (int e = 0; e < NA; e++) {
        const int u = tid + 256 * e;
        ra[e] = a + min(i0 + u / (KC / 16), m - 1) * k + 16 * (u % (KC / 16));
    }
#pragma unroll
    for (int e = 0; e < NB; e++) {
        const int u = tid + 256 * e;
        rb[e] = b + min(j0 + u / (KC / 16), n - 1) * k + 16 * (u % (KC / 16));
    }
    const int64_t whole = TRANS || n % 4 == 0 ? k : k - 4;
    auto load = [&](int64_t p0) {
        if (p0 + KC <= whole) {  // uniform
#pragma unroll
            for (int e = 0; e < NA; e++) __builtin_memcpy(&va[e], ra[e] + p0, 16);
            if constexpr (TRANS) {
#pragma unroll
                for (int e = 0; e < NB; e++) __builtin_memcpy(&vb[e], rb[e] + p0, 16);
            } else {
#pragma unroll
                for (int u = 0; u < NU; u++) {
                    const int8_t *q = b + (p0 + 8 * (kg + KG * u)) * n + jc;
#pragma unroll
                    for (int e = 0; e < 8; e++, q += n) __builtin_memcpy(&vc[u][e], q, 4);
                }
            }
        } else {
            const int p = 16 * (tid % (KC / 16));  // the same for each e (256 threads are whole rows)
#pragma unroll
            for (int e = 0; e < NA; e++) va[e] = ti_edge16(a, ra[e] - a + p0, m * k, k - p0 - p);
            if constexpr (TRANS) {
#pragma unroll
                for (int e = 0; e < NB; e++) vb[e] = ti_edge16(b, rb[e] - b + p0, n * k, k - p0 - p);
            } else {
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const int64_t q = p0 + 8 * (kg + KG * u) + e;
                        vc[u][e] = ti_edge4(b, q * n + jc, n * k, q < k);
                    }
            }
        }
    };
    auto store = [&](int s) {
#pragma unroll
        for (int e = 0; e < NA; e++) {
            const int u = tid + 256 * e;
            *reinterpret_cast<v4i *>(sa + (s * TM + u / (KC / 16)) * PITCH + 16 * (u % (KC / 16))) = va[e];
        }
        if constexpr (TRANS) {
#pragma unroll
            for (int e = 0; e < NB; e++) {
                const int u = tid + 256 * e;
                *reinterpret_cast<v4i *>(sb + (s * TN + u / (KC / 16)) * PITCH + 16 * (u % (KC / 16))) = vb[e];
            }
        } else {
#pragma unroll
            for (int u = 0; u < NU; u++) {
                rk_i2 col[4];
#pragma unroll
                for (int h = 0; h < 2; h++) {  // a 4x4 turn of bytes
                    const int *x = vc[u] + 4 * h;
                    const uint32_t l01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400);
                    const uint32_t h01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602);
                    const uint32_t l23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400);
                    const uint32_t h23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602);
                    col[0][h] = (int)__builtin_amdgcn_perm(l23, l01, 0x05040100);
                    col[1][h] = (int)__builtin_amdgcn_perm(l23, l01, 0x07060302);
                    col[2][h] = (int)__builtin_amdgcn_perm(h23, h01, 0x05040100);
                    col[3][h] = (int)__builtin_amdgcn_perm(h23, h01, 0x07060302);
                }
#pragma unroll
                for (int e = 0; e < 4; e++)
                    *reinterpret_cast<rk_i2 *>(sb + (s * TN + 4 * cg + e) * PITCH + 8 * (kg + KG * u)) = col[e];
            }
        }
    };
    for (int64_t k0 = 0; k0 < k; k0 += kTiRestart) {  // uniform; one pass up to 65536 positions
        const int64_t k1 = min(k, k0 + kTiRestart);
        v4i d[RM][RN];
#pragma unroll
        for (int r = 0; r < RM; r++)
#pragma unroll
            for (int q = 0; q < RN; q++) d[r][q] = v4i{0, 0, 0, 0};
        load(k0);
        int s = 0;
        for (int64_t p0 = k0; p0 < k1; p0 += KC, s ^= 1) {
            store(s);
            __syncthreads();
            if (p0 + KC < k1) load(p0 + KC);
#pragma unroll
            for (int ks = 0; ks < KC / WK; ks += 64) {
                const int at = wk * (KC / WK) + ks + 16 * lq;
                v4i fa[RM], fb[RN];
#pragma unroll
                for (int r = 0; r < RM; r++)
                    fa[r] = *reinterpret_cast<const v4i *>(sa + (s * TM + (wm * RM + r) * 16 + ln) * PITCH + at);
#pragma unroll
                for (int q = 0; q < RN; q++)
                    fb[q] = *reinterpret_cast<const v4i *>(sb + (s * TN + (wn * RN + q) * 16 + ln) * PITCH + at);
#pragma unroll
                for (int r = 0; r < RM; r++)
#pragma unroll
                    for (int q = 0; q < RN; q++)
                        d[r][q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[r], fb[q], d[r][q], 0, 0, 0);
            }
        }
        __syncthreads();  // the slices are read before they are written again
        if constexpr (WK > 1) {
            // the waves' partials through LDS, wrapping adds
            int32_t *red = reinterpret_cast<int32_t *>(ti_lds);  // [WK][TM][TN]: within the slices
#pragma unroll
            for (int r = 0; r < RM; r++)
#pragma unroll
                for (int q = 0; q < RN; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        red[(wk * TM + (wm * RM + r) * 16 + 4 * lq + e) * TN + (wn * RN + q) * 16 + ln] = d[r][q][e];
            __syncthreads();
            for (int o = tid; o < TM * TN; o += 256) {
                uint32_t v = 0;
#pragma unroll
                for (int w = 0; w < WK; w++) v += (uint32_t)red[w * TM * TN + o];
                const int64_t i = i0 + o / TN, j = j0 + o % TN;
                if (i < m && j < n) c[i * n + j] = (int32_t)(k0 ? (uint32_t)c[i * n + j] + v : v);
            }
            __syncthreads();
        } else {
            // the 16x16 result layout: lane holds column ln, rows 4·lq + e
#pragma unroll
            for (int r = 0; r < RM; r++)
#pragma unroll
                for (int q = 0; q < RN; q++) {
                    const int64_t j = j0 + (wn * RN + q) * 16 + ln;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int64_t i = i0 + (wm * RM + r) * 16 + 4 * lq + e;
                        const uint32_t v = (uint32_t)d[r][q][e];
                        if (i < m && j < n) c[i * n + j] = (int32_t)(k0 ? (uint32_t)c[i * n + j] + v : v);
                    }
                }
        }
    }
}

// Operands smaller than a load (fewer than 4 floats or 16 bytes, so k < 16):
// a thread an output.
template <typename T, typename R>
__global__ __launch_bounds__(256) void tensor_mm_small_kernel(const T *a, const T *b, R *c, int64_t m, int64_t k,
                                                              int64_t n, int transposed) {
    for (int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x; o < m * n; o += (int64_t)gridDim.x * 256) {
        const int64_t i = o / n, j = o % n;
        R v = 0;
        for (int64_t p = 0; p < k; p++) v += (R)a[i * k + p] * (R)b[transposed ? j * k + p : p * n + j];
        if constexpr (sizeof(T) == 4) v = canonical(v);
        c[o] = v;
    }
}

// ---- elementwise ----
// tensor.go:445-461: q = int8(max(-127, min(127, float32(RoundToEven(v/k)))))
// with v/k the correctly rounded f32 quotient; NaN quotients give 0 (Go's
// conversion of NaN on amd64 takes the low byte of 0x80000000).
__global__ void tensor_quantize_kernel(const float *a, int8_t *q, int64_t n, float k) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float r = __builtin_rintf(a[i] / k);
        q[i] = (int8_t)(r != r ? 0 : (r > 127.0f ? 127 : (r < -127.0f ? -127 : (int)r)));
    }
}

// tensor.go:366-387: out = Canonical(float32(v)·k), v f32 or i32.
__global__ void tensor_scale_kernel(const void *a, int i32, float *out, int64_t n, float k) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float v = i32 ? (float)static_cast<const int32_t *>(a)[i] : static_cast<const float *>(a)[i];
        out[i] = canonical(v * k);
    }
}

}  // namespace

static unsigned elem_grid(int64_t n) { return (unsigned)std::min<int64_t>((n + 255) / 256, 65536); }

static int64_t tiles_of(int64_t m, int64_t n, int tm, int tn) { return ((m + tm - 1) / tm) * ((n + tn - 1) / tn); }

// One workgroup a tile, the count padded to whole rounds of the 8 XCDs
// (xcd_tile), in rows of kTileRow: a grid dimension takes fewer than 2^32
// threads, 2^24 of these workgroups (2^34 float32 outputs, 64 GiB).
static dim3 tile_grid(int64_t m, int64_t n, int tm, int tn) {
    const int64_t ids = (tiles_of(m, n, tm, tn) + 7) / 8 * 8, row = std::min<int64_t>(ids, kTileRow);
    return dim3((unsigned)row, (unsigned)((ids + row - 1) / row));
}

template <int TM, int TN, int KC, int WM, int WN, int WK, bool TRANS>
static void launch_tensor_i8_t(const int8_t *a, const int8_t *b, int32_t *c, int64_t m, int64_t k, int64_t n,
                               hipStream_t s) {
    constexpr int lds = 2 * (TM + TN) * (KC + 16);
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute((const void *)tensor_mm_i8_kernel<TM, TN, KC, WM, WN, WK, TRANS>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    });
    RK_LAUNCH((tensor_mm_i8_kernel<TM, TN, KC, WM, WN, WK, TRANS>), tile_grid(m, n, TM, TN), dim3(256), lds, s, a, b, c,
              m, k, n);
}

template <bool TRANS>
static void launch_tensor_i8(const int8_t *a, const int8_t *b, int32_t *c, int64_t m, int64_t k, int64_t n,
                             hipStream_t s) {
    // The largest tile that still gives the chip's 256 CUs a workgroup or two
    // each; below 128 tiles of 64 the 32 x 32 one, whose four waves share a
    // slice of 512 positions, unless k would leave most of that slice empty.
    // Measured (us, k x n operand b; 128 x 64, 64 x 64, 32 x 32): 2048^3 22.8,
    // 33.5, 105; 1024^3 9.7, 7.4, 16.4; 256 x 2048 x 256 15.2, 11.1, 6.4;
    // 118 x 45 x 279 6.3, 4.9, 6.2.
    if (tiles_of(m, n, 128, 64) >= 256)
        launch_tensor_i8_t<128, 64, 128, 2, 2, 1, TRANS>(a, b, c, m, k, n, s);
    else if (tiles_of(m, n, 64, 64) >= 128 || k < 512)
        launch_tensor_i8_t<64, 64, 128, 2, 2, 1, TRANS>(a, b, c, m, k, n, s);
    else
        launch_tensor_i8_t<32, 32, 512, 1, 1, 4, TRANS>(a, b, c, m, k, n, s);
}

int enqueue_tensor_matmul(rk_device *d, int32_t dtype, int32_t transposed, int64_t m, int64_t k, int64_t n,
                          const void *a, const void *b, void *c, hipStream_t s) {
    const int64_t least = std::min(m, n) * k;  // the smaller operand's elements
    if (dtype == RK_TENSOR_F32) {
        ProfScope p(d, s, "tensor_matmul_f32");
        const float *fa = static_cast<const float *>(a), *fb = static_cast<const float *>(b);
        float *fc = static_cast<float *>(c);
        const dim3 grid = tile_grid(m, n, kTfTile, kTfTile);
        if (least < 4)
            RK_LAUNCH((tensor_mm_small_kernel<float, float>), dim3(elem_grid(m * n)), dim3(256), 0, s, fa, fb, fc, m, k,
                      n, transposed);
        else if (transposed)
            RK_LAUNCH(tensor_mm_f32_kernel<true>, grid, dim3(256), 0, s, fa, fb, fc, m, k, n);
        else
            RK_LAUNCH(tensor_mm_f32_kernel<false>, grid, dim3(256), 0, s, fa, fb, fc, m, k, n);
    } else {
        ProfScope p(d, s, "tensor_matmul_i8");
        const int8_t *ia = static_cast<const int8_t *>(a), *ib = static_cast<const int8_t *>(b);
        int32_t *ic = static_cast<int32_t *>(c);
        if (least < 16)
            RK_LAUNCH((tensor_mm_small_kernel<int8_t, int32_t>), dim3(elem_grid(m * n)), dim3(256), 0, s, ia, ib, ic, m,
                      k, n, transposed);
        else if (transposed)
            launch_tensor_i8<true>(ia, ib, ic, m, k, n, s);
        else
            launch_tensor_i8<false>(ia, ib, ic, m, k, n, s);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(d, e, "tensor matmul launch");
    return RK_OK;
}

int enqueue_tensor_quantize(rk_device *d, const float *a, int8_t *q, int64_t n, float k, hipStream_t s) {
    ProfScope p(d, s, "tensor_quantize");
    RK_LAUNCH(tensor_quantize_kernel, dim3(elem_grid(n)), dim3(256), 0, s, a, q, n, k);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? RK_OK : hip_fail(d, e, "tensor quantize launch");
}

int enqueue_tensor_scale(rk_device *d, int32_t dtype, const void *a, float *out, int64_t n, float k, hipStream_t s) {
    ProfScope p(d, s, "tensor_scale");
    RK_LAUNCH(tensor_scale_kernel, dim3(elem_grid(n)), dim3(256), 0, s, a, dtype == RK_TENSOR_I32 ? 1 : 0, out, n, k);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? RK_OK : hip_fail(d, e, "tensor scale launch");
}

}  // namespace rk

using namespace rk;

namespace {

// Shape and type checks of tenMatmul (tensor.go:287-300): the same dtype on
// both sides, not i32; dimensions within the tensor table's 2^24 limit
// (tensor.go:60).
int check_tensor_matmul(rk_device *d, int32_t dtype, int64_t m, int64_t k, int64_t n) {
    if (!d) return RK_ERR_ARGS;
    if (dtype != RK_TENSOR_F32 && dtype != RK_TENSOR_I8)
        return fail(d, RK_ERR_ARGS, "rk_tensor_matmul: dtype %d (f32 or i8 only)", dtype);
    const int64_t lim = (int64_t)1 << 24;
    if (m <= 0 || k <= 0 || n <= 0 || m > lim || k > lim || n > lim)
        return fail(d, RK_ERR_ARGS, "rk_tensor_matmul: shape %lldx%lld by %lld", (long long)m, (long long)k,
                    (long long)n);
    return RK_OK;
}

size_t dsize(int32_t dtype) { return dtype == RK_TENSOR_I8 ? 1 : 4; }

}  // namespace

extern "C" {

int rk_tensor_matmul(rk_device *d, int32_t dtype, int32_t transposed, int64_t m, int64_t k, int64_t n, const void *a,
                     const void *b, void *c) {
    int rc = check_tensor_matmul(d, dtype, m, k, n);
    if (rc) return rc;
    if (!a || !b || !c) return fail(d, RK_ERR_ARGS, "rk_tensor_matmul: null buffer");
    Hold hold(d->gate);
    HIP_TRY(d, hipSetDevice(d->index), "hipSetDevice");
    if (d->capturing) return fail(d, RK_ERR_ARGS, "rk_tensor_matmul waits for its result: it cannot be recorded");
    const size_t ab = (size_t)(m * k) * dsize(dtype), bb = (size_t)(k * n) * dsize(dtype), cb = (size_t)(m * n) * 4;
    void *da = nullptr, *db = nullptr, *dc = nullptr;
    if ((rc = dev_alloc(d, &da, ab, "tensor a")) || (rc = dev_alloc(d, &db, bb, "tensor b")) ||
        (rc = dev_alloc(d, &dc, cb, "tensor c"))) {
        (void)hipFree(da);
        (void)hipFree(db);
        return rc;
    }
    hipStream_t s = d->stream;
    hipError_t e = hipMemcpyAsync(da, a, ab, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(db, b, bb, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) rc = enqueue_tensor_matmul(d, dtype, transposed, m, k, n, da, db, dc, s);
    if (e == hipSuccess && !rc) e = hipMemcpyAsync(c, dc, cb, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && !rc) e = hipStreamSynchronize(s);
    (void)hipFree(da);
    (void)hipFree(db);
    (void)hipFree(dc);
    if (rc) return rc;
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return hip_fail(d, e, "rk_tensor_matmul");
    }
    return RK_OK;
}

int rk_tensor_matmul_device(rk_device *d, int32_t dtype, int32_t transposed, int64_t m, int64_t k, int64_t n,
                            const void *d_a, const void *d_b, void *d_c, void *stream) {
    int rc = check_tensor_matmul(d, dtype, m, k, n);
    if (rc) return rc;
    if (!d_a || !d_b || !d_c) return fail(d, RK_ERR_ARGS, "rk_tensor_matmul_device: null buffer");
    Hold hold(d->gate);
    HIP_TRY(d, hipSetDevice(d->index), "hipSetDevice");
    hipStream_t s = stream ? (hipStream_t)stream : d->stream;
    if (d->capturing && s != d->stream)
        return fail(d, RK_ERR_ARGS, "while recording a graph, work goes on the device's stream");
    return enqueue_tensor_matmul(d, dtype, transposed, m, k, n, d_a, d_b, d_c, s);
}

int rk_tensor_quantize(rk_device *d, const float *a, int8_t *q, int64_t n, float k) {
    if (!d) return RK_ERR_ARGS;
    if (!(k > 0.0f) || n < 0 || (n > 0 && (!a || !q))) return fail(d, RK_ERR_ARGS, "rk_tensor_quantize: bad arguments");
    if (n == 0) return RK_OK;
    Hold hold(d->gate);
    HIP_TRY(d, hipSetDevice(d->index), "hipSetDevice");
    if (d->capturing) return fail(d, RK_ERR_ARGS, "rk_tensor_quantize waits for its result: it cannot be recorded");
    float *da = nullptr;
    int8_t *dq = nullptr;
    int rc;
    if ((rc = dev_alloc(d, (void **)&da, (size_t)n * 4, "tensor")) || (rc = dev_alloc(d, (void **)&dq, (size_t)n, "tensor"))) {
        (void)hipFree(da);
        return rc;
    }
    hipStream_t s = d->stream;
    hipError_t e = hipMemcpyAsync(da, a, (size_t)n * 4, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) rc = enqueue_tensor_quantize(d, da, dq, n, k, s);
    if (e == hipSuccess && !rc) e = hipMemcpyAsync(q, dq, (size_t)n, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && !rc) e = hipStreamSynchronize(s);
    (void)hipFree(da);
    (void)hipFree(dq);
    if (rc) return rc;
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return hip_fail(d, e, "rk_tensor_quantize");
    }
    return RK_OK;
}

int rk_tensor_scale(rk_device *d, int32_t dtype, const void *a, float *out, int64_t n, float k) {
    if (!d) return RK_ERR_ARGS;
    if ((dtype != RK_TENSOR_F32 && dtype != RK_TENSOR_I32) || n < 0 || (n > 0 && (!a || !out)))
        return fail(d, RK_ERR_ARGS, "rk_tensor_scale: bad arguments (f32 or i32 input)");
    if (n == 0) return RK_OK;
    Hold hold(d->gate);
    HIP_TRY(d, hipSetDevice(d->index), "hipSetDevice");
    if (d->capturing) return fail(d, RK_ERR_ARGS, "rk_tensor_scale waits for its result: it cannot be recorded");
    void *da = nullptr;
    float *dout = nullptr;
    int rc;
    if ((rc = dev_alloc(d, &da, (size_t)n * 4, "tensor")) || (rc = dev_alloc(d, (void **)&dout, (size_t)n * 4, "tensor"))) {
        (void)hipFree(da);
        return rc;
    }
    hipStream_t s = d->stream;
    hipError_t e = hipMemcpyAsync(da, a, (size_t)n * 4, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) rc = enqueue_tensor_scale(d, dtype, da, dout, n, k, s);
    if (e == hipSuccess && !rc) e = hipMemcpyAsync(out, dout, (size_t)n * 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && !rc) e = hipStreamSynchronize(s);
    (void)hipFree(da);
    (void)hipFree(dout);
    if (rc) return rc;
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return hip_fail(d, e, "rk_tensor_scale");
    }
    return RK_OK;
}

}  // extern "C"
