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

// Whether INT8 rows go to this kernel rather than to GEMV passes of 2 rows that
// re-read the weights (elems of them): from 5 rows, or 3 on weights of 32 Mi
// elements (us, passes against batched: 4096 x 4096 at 3 rows 12.2 / 13.6 and
// at 5 17 / 14; 14336 x 4096 at 2 rows 14.0 / 22.7 and at 3 25.4 / 23.5; 4864 x
// 896 at 4 rows 9.3 / 11.1).
inline bool qgemm_w8_wins(int64_t m, int64_t elems) {
    return m >= 5 || (m >= 3 && elems >= (int64_t)1 << 25);
}

// Scratch of one call's fastest plan: the split activations and the split-K
// partial sums.  A plan takes any `cap` that holds at least the activations
// (qgemm_fits).
size_t qgemm_scratch_bytes(int m, int n, int k, int fmt, bool grouped, bool pair);
bool qgemm_fits(int64_t m, int64_t n, int64_t k, int fmt, bool grouped, bool pair, size_t cap);

// scratch: cap bytes, 256-byte aligned.
int qgemm(const QGemmParams &p, void *scratch, size_t cap, hipStream_t st);

}  // namespace tb
