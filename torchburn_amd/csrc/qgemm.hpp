// Internal launcher of the batched quantized projection on f16 MFMA (qgemm.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace tb {

enum QFmt { Q_W4 = 0, Q_V2 = 1, Q_W8 = 2 };

struct QGemmParams {
    const float *x;        // [m, k] activations
    const void *w0;        // [n, k/2] nibbles, v2 blocks or [n, k] int8 (gate of a pair)
    const float *s0;       // scales of w0 (null for v2)
    const float *b0;       // [n] bias or null
    const void *w1;        // up projection of a SwiGLU pair, or null
    const float *s1;
    const float *b1;
    const float *res;      // [m, n] residual or null (single projection); may be y
    float *y;              // [m, n]; silu(gate) * up for a pair
    int m, n, k;
    int fmt;               // QFmt
    int grouped;           // 1: INT4 scales [n, k >> gshift] (or v2); 0: a scale per row / scalar
    int gshift;            // log2(group), >= 5 (grouped)
    int s0_len, s1_len;    // 1 or n scales (not grouped)
};

// Shapes the kernel takes: m >= 1, k a multiple of 32 (v2: of 64) up to 2^24.
bool qgemm_shape_ok(int64_t m, int64_t n, int64_t k, int fmt);

// Scratch of one call's fastest plan: the split activations and the split-K
// partial sums.  A plan takes any `cap` that holds at least the activations
// (qgemm_fits).
size_t qgemm_scratch_bytes(int m, int n, int k, int fmt, bool grouped, bool pair);
bool qgemm_fits(int64_t m, int64_t n, int64_t k, int fmt, bool grouped, bool pair, size_t cap);

// scratch: cap bytes, 256-byte aligned.
int qgemm(const QGemmParams &p, void *scratch, size_t cap, hipStream_t st);

}  // namespace tb
