/*
 * mfma64.h -- the FP64 MFMA building block shared by the GEMM kernels and the
 * Lagrange iteration: v_mfma_f64_16x16x4_f64.
 *
 * Instruction layout (measured on gfx950): A lane l = A[l%16][l/16], B lane
 * l = B[l/16][l%16], D register r of lane l = D[4r + l/16][l%16].  Each element
 * of D is C plus its four products added by fused multiply-adds in the order
 * of k (measured bit for bit), so a sum formed by these instructions over
 * increasing k is the sequential FMA chain, whatever the tiling.
 *
 * The instruction sustains 77.8 TFLOP/s (nominal 78.6) from one wave per SIMD
 * up, provided its accumulators stay in place: a kernel that may use more
 * than 256 registers per lane (__launch_bounds__(256) and no minimum of
 * waves) gets them copied between the two register files around every loop
 * and drops to 37-51, so the GEMM kernels are bounded to 256 or fewer.  The
 * Lagrange and carried-overlap kernels are not bound by the instruction (it
 * keeps the matrix cores busy 0.05 of k_lagrange_str's time): of them only
 * k_lagrange_res is bounded.
 */
#pragma once
#include <hip/hip_runtime.h>

typedef double mfma_d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ mfma_d4 mfma16(double a, double b, mfma_d4 c)
{
   return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

/* row of a 16 x 16 tile that D register r of this lane holds */
__device__ __forceinline__ int mfma16_row(int r, int lane) { return 4 * r + (lane >> 4); }
