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

// Shapes the kernel takes: k a multiple of 32 (v2: of 64) up to 2^30, m below 2^24.
bool qgemm_shape_ok(int64_t m, int64_t n, int64_t k, int fmt);

// Whether INT8 rows go to this kernel rather than to GEMV passes of 2 rows that
// re-read the weights (elems of them): from 4 rows, or 3 on weights of 32 Mi
// elements (us, passes / batched: 4096 x 4096 at 3 rows 12.3 / 12.5, 14336 x 4096
// at 2 rows 14.0 / 22.7 and at 3 25.4 / 23.5, 4864 x 896 at 4 rows 9.4 / 9.2).
inline bool qgemm_w8_wins(int64_t m, int64_t elems) {
    return m >= 4 || (m >= 3 && elems >= (int64_t)1 << 25);
}

// Whether 3..16 INT4 rows with K % 128 == 0 stay on the small-batch kernel of
// w4_limb.hip, which reads large weights faster (us, it / this one: 8 rows,
// 14336 x 4096 17.9 / 20.3 and 4096 x 14336 16.8 / 21.5; at 4096 x 4096 12.7 / 13.0;
// with its record and reduce kernels it is behind on smaller ones: 4 rows, 4864 x
// 896 11.5 / 9.2, and 16 rows, 4096 x 4096 15.4 / 13.9).
inline bool limb_wins(int64_t elems) { return elems > (int64_t)1 << 24; }

// How a call runs: the block's tile, the K split and whether the blocks build
// the activations' limbs themselves.
struct QPlan {
    int mt, nt, mz, nbx, splits, slen, slabs, groups;
    bool direct;
    size_t bytes;   // scratch: the activations' limbs and the split-K partial sums
    double us;      // the cost model's time
};

// The fastest plan whose scratch is at most cap bytes (one with none exists).
QPlan qgemm_plan(int m, int n, int k, int fmt, bool grouped, bool pair, size_t cap = SIZE_MAX);

inline QPlan qgemm_plan(const QGemmParams &p, size_t cap = SIZE_MAX) {
    return qgemm_plan(p.m, p.n, p.k, p.fmt, p.grouped != 0, p.w1 != nullptr, cap);
}

// y = epilogue(x . deq(w)^T): + bias (+ residual), or silu(x w0^T + b0) *
// (x w1^T + b1) for a pair.  scratch: pl.bytes, 256-byte aligned.
int qgemm(const QGemmParams &p, const QPlan &pl, void *scratch, hipStream_t st);

}  // namespace tb
