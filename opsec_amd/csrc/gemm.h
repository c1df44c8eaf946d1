// MFMA GEMM building blocks for gfx950 (wave64).
//
// Operand sources of the eigen-solver's GEMMs: workgroup tile 128 x 128 x 16,
// 256 threads = 4 waves, each wave owning a 64 x 64 sub-tile as 4 x 4 MFMA
// fragments of 16 x 16, operand tiles staged through LDS k-major (As[k][m],
// Bs[k][n]) so that the 16 lanes of a fragment row read consecutive words.
// (The projection's GEMM is in nt_gemm.h.)
//
// Fragment layouts (measured with an in-bounds probe on gfx950):
//   f64 16x16x4:    A lane l -> A[l%16][l/16],  B lane l -> B[l/16][l%16],
//                   D lane l, item r -> D[l/16 + 4r][l%16]
//   f32 16x16x4:    A, B as f64;                D lane l, item r -> D[4(l/16)+r][l%16]
//   bf16 16x16x32:  A lane l -> A[l%16][8(l/16)+e], B lane l -> B[8(l/16)+e][l%16],
//                   D as f32.
#pragma once

#include <cstdint>

#include "common.h"

namespace opsec {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

constexpr int GT_M = 128, GT_N = 128, GT_THREADS = 256;

// Row (within a 16 x 16 output fragment) of accumulator item r of `lane`.
template <typename T>
__device__ __forceinline__ int acc_row(int lane, int r) {
    return 4 * (lane >> 4) + r;
}
template <>
__device__ __forceinline__ int acc_row<double>(int lane, int r) {
    return (lane >> 4) + 4 * r;
}

// ---- operand sources -------------------------------------------------------
// Each source exposes  T get(m_or_n, k)  with bounds handled by the caller,
// and a flag telling which index is contiguous in memory.

struct SrcDenseRowMajor {      // X[i][k] = p[i*ld + k]   (k contiguous)
    const double* p;
    size_t ld;
    static constexpr bool k_contig = true;
    __device__ __forceinline__ double get(int i, int k) const { return p[(size_t)i * ld + k]; }
};

struct SrcDenseColMajor {      // X[i][k] = p[k*ld + i]   (i contiguous)
    const double* p;
    size_t ld;
    static constexpr bool k_contig = false;
    __device__ __forceinline__ double get(int i, int k) const { return p[(size_t)k * ld + i]; }
};

struct SrcKColMajor {          // X[i][k] = p[i*ld + k], i.e. a column-major K x N operand read as [n][k]
    const double* p;
    size_t ld;
    static constexpr bool k_contig = true;
    __device__ __forceinline__ double get(int i, int k) const { return p[(size_t)i * ld + k]; }
};

}  // namespace opsec
