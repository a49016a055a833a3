// Internal launcher of the batched INT4 projection (w4_mfma.hip): FP32 MFMA up
// to 16 rows, the f16-limb kernel (qgemm.hip) from 17.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace tb {

struct MfmaParams {
    const float *x;      // [m, k] activations
    const uint8_t *w0;   // [n, k/2] packed nibbles (gate when dual)
    const float *s0;     // [n, k/group] scales
    const float *b0;     // [n] bias or null
    const uint8_t *w1;   // up projection of a SwiGLU pair, or null
    const float *s1;
    const float *b1;
    const float *res;    // [m, n] residual (EPI_RESID)
    float *y;            // [m, n]
    int m, n, k;
    int gshift;          // log2(group_size)
    int scale_mode;      // 0: grouped [n, k/group]; 1: one scale per row; 2: one scalar
    int v2;              // 1: w0 / w1 are v2 streams of 34-byte group-64 blocks
                         // (f16 scales inside, s0 / s1 unused)
};

// Scratch of the fastest form for this shape (dual = SwiGLU pair).
size_t w4_mfma_scratch_bytes(int m, int n, int k, bool dual, bool v2 = false,
                             bool grouped = true);

// Scratch that serves every row count from 1 to m (v1 weights): below its own
// fastest plan a call takes one that fits.
size_t w4_mfma_scratch_upto(int m, int n, int k, bool dual);

// y = epilogue(x . deq(w)^T) for any m >= 1.  epi: EPI_PLAIN, EPI_RESID, or
// EPI_SWIGLU when w1 is set.  part: cap bytes of device scratch, 256-byte
// aligned: w4_mfma_scratch_bytes(), or less (fewer K splits, or the FP32-MFMA
// form where the f16 limbs of x do not fit).  Shapes validated by the caller
// (K % 32 == 0, K % group == 0, 16-byte aligned rows).
int w4_mfma(const MfmaParams &p, int epi, float *part, size_t cap, hipStream_t st);

}  // namespace tb
