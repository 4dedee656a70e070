// rk_dense.hip — float32 and bfloat16 matrix-vector products in the Dot32
// order (internal/num/matvec.go:32-67 Dot32 / DotBF16 / combine,
// :106-123 MatVec32 / MatVecBF16), for gfx950.
//
// Dot32 of a row: element i goes into running sum i mod 32, in order of i,
// each product rounded before it is added; then e_j = (s_j + s_j+8) +
// (s_j+16 + s_j+24) and ((e0+e1)+(e2+e3))+((e4+e5)+(e6+e7)). A bfloat16
// weight converts to float32 exactly, so DotBF16 is Dot32 of the converted
// row.
//
// Layout: rows padded with zeros to a multiple of 32 elements on upload
// (rk_matrix_upload). A padded element adds the product +0·+0 = +0 to its
// running sum, which leaves the sum unchanged: a sum starts at +0 and can
// never become -0 (x + y is -0 only when both are), so s + (+0) == s, NaN
// payloads included.
//
// Work layout: 32 lanes per row, two rows a wave; lane l of a row keeps the
// running sum l and takes element 32m + l of row step m. A wave's rows come
// by direct-to-LDS loads, 1 KiB of one row an instruction, into a ring of
// its own of kDenseRing parts of 16 steps: the bytes in flight need no
// registers, many waves fit a CU, and a part is waited for by count, without
// a barrier. The input is staged in LDS the same way (kDenseX elements at a
// time for wider rows). Up to three matrices of one input share a launch.
// Narrow rows: dense_narrow_kernel.
//
// What bounds it: HBM, then the launch and the input's way into LDS for the
// smaller ones. MI355X, bfloat16 (us, weights past the MALL; before: rows
// loaded a step an instruction into registers, a launch a matrix):
// 2048 + 512 + 512 x 2048 5.3 (24.3), 8192 + 8192 x 2048 12.9, 5.2 TB/s
// (21.5), 2048 x 8192 9.7 (21.4), 4096 x 4096 8.7 (12.0), 14336 + 14336 x
// 4096 41.3, 5.7 TB/s (57.0); float32 23.2 (29.9), 15.1 (18.3), 13.3 (15.1)
// and 72.0, 6.5 TB/s (80.5) for the last four. Rings of 3, 4 and 8 parts
// were slower (8192 + 8192: 14.0, 14.9, 20.1: fewer waves fit), as were two
// sums a lane, four rows a wave (15.5) and 1, 2 and 8 waves a workgroup.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "rk_dense.h"
#include "rk_dev.h"
#include "rk_kernels.h"

namespace rk {

namespace {

constexpr int kDensePart = 512;  // elements of a row (16 steps) in a ring part
constexpr int kDenseX = 8192;    // input elements staged at a time
constexpr int kDenseRing = 2;    // parts of a wave's ring

typedef float rk_v2f __attribute__((ext_vector_type(2)));

struct DenseArgs {
    DenseMat m[kDenseMats];
    int64_t first[kDenseMats];  // a matrix's first wave
    const float *x;
    int64_t row_elems;
    int32_t cols, waves;        // waves a workgroup
    int32_t groups;             // dense_narrow_kernel: groups of four rows a wave
};

__device__ __forceinline__ uint32_t lds_off(void *p) { return (uint32_t)(uintptr_t)lds_ptr(p); }

// 16 bytes a lane from global memory into LDS at `to` + 16·lane.
__device__ __forceinline__ void load_lds16(const uint8_t *from, uint8_t *to) {
    __builtin_amdgcn_global_load_lds(from, lds_ptr(to), 16, 0, kAuxStream);
}

// Waits for the wave's loads, except (more) the NI of the ring's other part.
template <int NI>
__device__ __forceinline__ void wait_part(bool more) {
    static_assert(kDenseRing == 2, "one part in flight past the one waited for");
    if (more)  // uniform
        __builtin_amdgcn_s_waitcnt(vmcnt_wait(NI));
    else
        __builtin_amdgcn_s_waitcnt(vmcnt_wait(0));
    asm volatile("" ::: "memory");
}

// A part's 16 steps of a lane from LDS: weights at byte wa (step stride 64 or
// 128), input at byte xa (step stride 128). The reads and their wait are one
// block, so no output is seen before it has arrived (and the compiler, which
// cannot tell the ring's parts apart, adds no wait for the loads in flight).
template <bool BF>
struct DensePart;
template <>
struct DensePart<true> {
    int w[16];
    rk_v2f x[8];
    __device__ __forceinline__ void read(uint32_t wa, uint32_t xa) {
        asm volatile(
            "ds_read_u16 %0, %24\n\tds_read_u16 %1, %24 offset:64\n\tds_read2_b32 %16, %25 offset0:0 offset1:32\n\t"
            "ds_read_u16 %2, %24 offset:128\n\tds_read_u16 %3, %24 offset:192\n\tds_read2_b32 %17, %25 offset0:64 offset1:96\n\t"
            "ds_read_u16 %4, %24 offset:256\n\tds_read_u16 %5, %24 offset:320\n\tds_read2_b32 %18, %25 offset0:128 offset1:160\n\t"
            "ds_read_u16 %6, %24 offset:384\n\tds_read_u16 %7, %24 offset:448\n\tds_read2_b32 %19, %25 offset0:192 offset1:224\n\t"
            "ds_read_u16 %8, %24 offset:512\n\tds_read_u16 %9, %24 offset:576\n\tds_read2_b32 %20, %26 offset0:0 offset1:32\n\t"
            "ds_read_u16 %10, %24 offset:640\n\tds_read_u16 %11, %24 offset:704\n\tds_read2_b32 %21, %26 offset0:64 offset1:96\n\t"
            "ds_read_u16 %12, %24 offset:768\n\tds_read_u16 %13, %24 offset:832\n\tds_read2_b32 %22, %26 offset0:128 offset1:160\n\t"
            "ds_read_u16 %14, %24 offset:896\n\tds_read_u16 %15, %24 offset:960\n\tds_read2_b32 %23, %26 offset0:192 offset1:224\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7]),
              "=&v"(w[8]), "=&v"(w[9]), "=&v"(w[10]), "=&v"(w[11]), "=&v"(w[12]), "=&v"(w[13]), "=&v"(w[14]),
              "=&v"(w[15]), "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]),
              "=&v"(x[7])
            : "v"(wa), "v"(xa), "v"(xa + 1024)
            : "memory");
    }
    __device__ __forceinline__ float weight(int m) const { return __int_as_float(w[m] << 16); }
    __device__ __forceinline__ float input(int m) const { return x[m >> 1][m & 1]; }
};
template <>
struct DensePart<false> {
    rk_v2f w[8], x[8];
    __device__ __forceinline__ void read(uint32_t wa, uint32_t xa) {
        asm volatile(
            "ds_read2_b32 %0, %16 offset0:0 offset1:32\n\tds_read2_b32 %8, %18 offset0:0 offset1:32\n\t"
            "ds_read2_b32 %1, %16 offset0:64 offset1:96\n\tds_read2_b32 %9, %18 offset0:64 offset1:96\n\t"
            "ds_read2_b32 %2, %16 offset0:128 offset1:160\n\tds_read2_b32 %10, %18 offset0:128 offset1:160\n\t"
            "ds_read2_b32 %3, %16 offset0:192 offset1:224\n\tds_read2_b32 %11, %18 offset0:192 offset1:224\n\t"
            "ds_read2_b32 %4, %17 offset0:0 offset1:32\n\tds_read2_b32 %12, %19 offset0:0 offset1:32\n\t"
            "ds_read2_b32 %5, %17 offset0:64 offset1:96\n\tds_read2_b32 %13, %19 offset0:64 offset1:96\n\t"
            "ds_read2_b32 %6, %17 offset0:128 offset1:160\n\tds_read2_b32 %14, %19 offset0:128 offset1:160\n\t"
            "ds_read2_b32 %7, %17 offset0:192 offset1:224\n\tds_read2_b32 %15, %19 offset0:192 offset1:224\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7]),
              "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7])
            : "v"(wa), "v"(wa + 1024), "v"(xa), "v"(xa + 1024)
            : "memory");
    }
    __device__ __forceinline__ float weight(int m) const { return w[m >> 1][m & 1]; }
    __device__ __forceinline__ float input(int m) const { return x[m >> 1][m & 1]; }
};

template <bool BF>
struct DenseShape {
    static constexpr int RPW = 2;  // rows a wave
    static constexpr int ES = BF ? 2 : 4, SB = 32 * ES;  // bytes an element, a row step
    static constexpr int PB = kDensePart * ES;           // bytes of a row in a part
    // rows of a part lie PB + pad apart, so a step's pieces fall in distinct banks
    static constexpr int PITCH = PB + (BF ? 64 : 128), PART = RPW * PITCH;
    static constexpr int NI = RPW * (PB / 1024);         // loads a part
};

template <bool BF>
__global__ __launch_bounds__(256) void dense_matvec_kernel(DenseArgs a) {
    typedef DenseShape<BF> D;
    constexpr int S = kDenseRing;
    extern __shared__ __align__(16) uint8_t dense_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 31, g = lane >> 5;
    const int re = (int)a.row_elems;
    const int xe = min(re, kDenseX);  // input elements staged at a time
    float *sx = reinterpret_cast<float *>(dense_lds);
    uint8_t *ring = dense_lds + 4 * ((xe + kDensePart - 1) / kDensePart * kDensePart) + wv * S * D::PART;
    // the wave's matrix and rows; past the end it repeats the last row
    // (never stored) and takes part in the barriers
    const int64_t gw = (int64_t)blockIdx.x * a.waves + wv;
    const int mi = (gw >= a.first[1] ? 1 : 0) + (gw >= a.first[2] ? 1 : 0);
    const uint8_t *w = static_cast<const uint8_t *>(a.m[mi].w);
    const int64_t rows = a.m[mi].rows, r0 = (gw - a.first[mi]) * D::RPW;
    const int64_t rb = (int64_t)re * D::ES;
    const int parts = (re + kDensePart - 1) / kDensePart;
    // part c into its place in the ring; past the row's end the last 16
    // bytes again (never added)
    auto fetch = [&](int c) {
        uint8_t *to = ring + (c % S) * D::PART;
#pragma unroll
        for (int r = 0; r < D::RPW; r++) {
            const uint8_t *row = w + min(r0 + r, rows - 1) * rb;
#pragma unroll
            for (int h = 0; h < D::PB / 1024; h++)
                load_lds16(row + min((int64_t)c * D::PB + 1024 * h + 16 * lane, rb - 16), to + r * D::PITCH + 1024 * h);
        }
    };
    // input elements c0 .. c0 + n, zeros past cols
    const bool a16 = ((uintptr_t)a.x & 15) == 0;
    auto stage = [&](int c0) {
        const int n = min(xe, re - c0), have = max(0, min(n, a.cols - c0)), m16 = a16 ? have & ~255 : 0;
        const float *x = a.x + c0;
        for (int p = 256 * wv; p < m16; p += 256 * a.waves)
            __builtin_amdgcn_global_load_lds(x + p + 4 * lane, lds_ptr(sx + p), 16, 0, 0);
        for (int p = m16 + 64 * wv; p + 64 <= have; p += 64 * a.waves)
            __builtin_amdgcn_global_load_lds(x + p + lane, lds_ptr(sx + p), 4, 0, 0);
        const int t = (have & ~63) + lane;  // fewer than 64 left, then zeros
        if (wv == 0 && t < n) sx[t] = t < have ? x[t] : 0.0f;
    };
    stage(0);
    const int ahead = min(S, parts);
    for (int c = 0; c < ahead; c++) fetch(c);
    // the input is there once only the weights' loads are in flight
    static_assert(S * D::NI <= 63, "the counter's range");
    if (ahead == S)
        __builtin_amdgcn_s_waitcnt(vmcnt_wait(S * D::NI));
    else
        __builtin_amdgcn_s_waitcnt(vmcnt_wait(0));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const uint32_t wo = lds_off(ring) + g * D::PITCH + l * D::ES, xo = lds_off(sx) + 4 * l;
    float acc = 0.0f;
    for (int c = 0; c < parts; c++) {
        const int e0 = c * kDensePart, c0 = e0 % kDenseX;
        if (c0 == 0 && c > 0) {  // the next elements of a wide row's input
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();  // every wave is done with the last ones
            stage(e0);
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
        }
        wait_part<D::NI>(c + 1 < parts);
        DensePart<BF> t;
        t.read(wo + (c % S) * D::PART, xo + 4 * c0);
        if (c + S < parts) fetch(c + S);  // into the part just read
        if (e0 + kDensePart <= re) {
#pragma unroll
            for (int m = 0; m < 16; m++) acc += t.weight(m) * t.input(m);
        } else {
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (e0 + 32 * m < re) acc += t.weight(m) * t.input(m);  // uniform
        }
    }
    // Dot32's combine, s_j in lane j of the row: s_j + s_j+8 (lanes of j <
    // 8), then + (s_j+16 + s_j+24) gives e_j; then
    // ((e0+e1)+(e2+e3))+((e4+e5)+(e6+e7)).
    const float v = acc + __shfl_down(acc, 8, 32);
    const float e = v + __shfl_down(v, 16, 32);
    const float p = e + __shfl_down(e, 1, 32);  // lanes 0, 2, 4, 6
    const float q = p + __shfl_down(p, 2, 32);  // lanes 0, 4
    const float res = q + __shfl_down(q, 4, 32);
    if (l == 0 && r0 + g < rows) a.m[mi].out[r0 + g] = res;
}

// v of the lane N up in its row of 16 (the last N lanes: another's).
template <int N>
__device__ __forceinline__ float row_up(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + N, 0xf, 0xf, true));
}

// Rows of at most ST steps (narrow ones): lane l of the 16 of a row keeps the
// running sums 2l and 2l + 1, four rows a wave, and holds the row and its own
// input elements in registers; a wave takes a.groups groups of four rows, the
// next one's loads in flight during the sums. The ring above reads whole parts
// of 512 elements and a wave ends after two rows: bounded by latency and by
// the number of waves. Measured (us, ring and this): bfloat16 32000 x 288 9.8
// and 5.3, 16000 x 384 6.3 and 4.5, 1000000 x 32 201 and 23, float32 32000 x
// 288 12.7 and 7.1, 128000 x 32 34.7 and 8.0.
template <bool BF, int ST>
__global__ __launch_bounds__(256) void dense_narrow_kernel(DenseArgs a) {
    typedef typename std::conditional<BF, uint32_t, float2>::type W;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int l = lane & 15, g = lane >> 4;
    const int steps = (int)a.row_elems >> 5;
    const int64_t gw = (int64_t)blockIdx.x * a.waves + wv;
    const int mi = (gw >= a.first[1] ? 1 : 0) + (gw >= a.first[2] ? 1 : 0);
    const int64_t rows = a.m[mi].rows, r0 = (gw - a.first[mi]) * (4 * a.groups);
    if (r0 >= rows) return;
    const int64_t rw = a.row_elems * (BF ? 2 : 4) / (int64_t)sizeof(W);  // a row's loads
    const W *w = static_cast<const W *>(a.m[mi].w) + l;
    const int ng = (int)min((int64_t)a.groups, (rows - r0 + 3) >> 2);
    W wc[ST];
    auto load = [&](int64_t r) {
        const W *p = w + min(r + g, rows - 1) * rw;
#pragma unroll
        for (int m = 0; m < ST; m++) wc[m] = p[16 * min(m, steps - 1)];
    };
    load(r0);
    // the lane's input elements, zeros past cols (odd widths in the last step
    // alone: a lane there reads the last pair of the input)
    float2 x[ST];
    if (a.cols == a.row_elems) {  // uniform
#pragma unroll
        for (int m = 0; m < ST; m++) __builtin_memcpy(&x[m], a.x + 32 * min(m, steps - 1) + 2 * l, 8);
    } else {
        const int i = 32 * (steps - 1) + 2 * l, o = min(i, a.cols - 2);
        float2 v = {0.0f, a.x[0]};
        if (a.cols > 1) __builtin_memcpy(&v, a.x + o, 8);
        if (steps > 1)
#pragma unroll
            for (int m = 0; m < ST - 1; m++) __builtin_memcpy(&x[m], a.x + 32 * min(m, steps - 2) + 2 * l, 8);
        const float2 t = {i == o ? v.x : i == o + 1 ? v.y : 0.0f, i == o ? v.y : 0.0f};
#pragma unroll
        for (int m = 0; m < ST; m++)
            if (m == steps - 1) x[m] = t;
    }
    for (int i = 0; i < ng; i++) {
        W wt[ST];
#pragma unroll
        for (int m = 0; m < ST; m++) wt[m] = wc[m];
        const int64_t r = r0 + 4 * i;
        if (i + 1 < ng) load(r + 4);
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int m = 0; m < ST; m++)
            if (m < steps) {  // uniform
                if constexpr (BF) {
                    s0 += __uint_as_float(wt[m] << 16) * x[m].x;
                    s1 += __uint_as_float(wt[m] & 0xffff0000u) * x[m].y;
                } else {
                    s0 += wt[m].x * x[m].x;
                    s1 += wt[m].y * x[m].y;
                }
            }
        const float v0 = s0 + row_up<4>(s0), v1 = s1 + row_up<4>(s1);
        const float e0 = v0 + row_up<8>(v0), e1 = v1 + row_up<8>(v1);
        const float p = e0 + e1;
        const float q = p + row_up<1>(p);
        const float res = q + row_up<2>(q);
        if (l == 0 && r + g < rows) a.m[mi].out[r + g] = res;
    }
}

template <bool BF, int ST>
void launch_narrow_t(DenseArgs a, int n, hipStream_t s) {
    int64_t groups = 0, waves = 0;
    for (int i = 0; i < n; i++) groups += (a.m[i].rows + 3) / 4;
    // up to four groups a wave while 2048 waves are left (32000 x 288: one 7.4
    // us, two 5.8, four 5.3), more once 8192 are (1000000 x 32: 8192 waves 23,
    // 2048 waves 54)
    a.groups = (int)std::max<int64_t>((groups + 8191) / 8192, std::min<int64_t>(4, (groups + 2047) / 2048));
    for (int i = 0; i < kDenseMats; i++) {
        a.first[i] = i < n ? waves : INT64_MAX;
        if (i < n) waves += (a.m[i].rows + 4 * a.groups - 1) / (4 * a.groups);
    }
    a.waves = (int)std::min<int64_t>(4, std::max<int64_t>(1, waves / 256));
    RK_LAUNCH((dense_narrow_kernel<BF, ST>), dim3((unsigned)((waves + a.waves - 1) / a.waves)),
              dim3((unsigned)(64 * a.waves)), 0, s, a);
}

template <bool BF>
void launch_dense_t(DenseArgs a, int n, hipStream_t s) {
    // Wider float32 rows hold too many registers for it (4000 x 512 4.3 us, by
    // the ring 3.7; 24000 x 512 10.3 and 10.0).
    constexpr int widest = BF ? 16 : 14;  // steps
    if (a.row_elems <= 32 * widest) {
        if (a.row_elems <= 128)
            launch_narrow_t<BF, 4>(a, n, s);
        else if (a.row_elems <= 288)
            launch_narrow_t<BF, 9>(a, n, s);
        else if (a.row_elems <= 384)
            launch_narrow_t<BF, 12>(a, n, s);
        else
            launch_narrow_t<BF, widest>(a, n, s);
        return;
    }
    typedef DenseShape<BF> D;
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute((const void *)dense_matvec_kernel<BF>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  4 * kDenseX + 4 * kDenseRing * D::PART);
    });
    int64_t waves = 0;
    for (int i = 0; i < kDenseMats; i++) {
        a.first[i] = i < n ? waves : INT64_MAX;
        if (i < n) waves += (a.m[i].rows + D::RPW - 1) / D::RPW;
    }
    // four waves a workgroup once that leaves every CU a workgroup
    a.waves = (int)std::min<int64_t>(4, std::max<int64_t>(1, waves / 256));
    const int64_t xe = (std::min<int64_t>(a.row_elems, kDenseX) + kDensePart - 1) / kDensePart * kDensePart;
    const size_t lds = (size_t)(4 * xe + a.waves * kDenseRing * D::PART);
    RK_LAUNCH(dense_matvec_kernel<BF>, dim3((unsigned)((waves + a.waves - 1) / a.waves)),
              dim3((unsigned)(64 * a.waves)), lds, s, a);
}

}  // namespace

int64_t dense_row_elems(int64_t cols) { return (cols + 31) & ~(int64_t)31; }

void launch_dense_matvecs(bool bf16, const DenseMat *m, int n, int64_t cols, const float *x, hipStream_t s) {
    DenseArgs a{};
    a.x = x;
    a.row_elems = dense_row_elems(cols);
    a.cols = (int32_t)cols;
    for (int i = 0; i < n; i++) a.m[i] = m[i];
    if (bf16)
        launch_dense_t<true>(a, n, s);
    else
        launch_dense_t<false>(a, n, s);
}

}  // namespace rk
