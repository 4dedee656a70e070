// rk_dense.h — launchers of the float32 / bfloat16 products (rk_dense.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rk {

// Elements per row of an uploaded float32 / bfloat16 matrix: cols rounded
// up to a multiple of 32, the padding zero.
int64_t dense_row_elems(int64_t cols);

// One product of a launch: out[r] = Dot32(row r, x) for r < rows
// (internal/num/matvec.go:106-123 MatVec32 / MatVecBF16); w holds rows of
// dense_row_elems(cols) float32 or bfloat16 values, device buffers.
struct DenseMat {
    const void *w;
    float *out;
    int64_t rows;
};
constexpr int kDenseMats = 3;  // matrices of a launch

// n (<= kDenseMats) matrices of one format times x (cols device floats).
void launch_dense_matvecs(bool bf16, const DenseMat *m, int n, int64_t cols, const float *x, hipStream_t s);

}  // namespace rk
