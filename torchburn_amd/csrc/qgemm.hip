// Batched quantized projection Y[M, N] = X[M, K] . deq(W)^T on f16 MFMA
// (v_mfma_f32_32x32x16_f16) for INT4 (v1 nibbles, v2 blocks) and INT8 weights.
//
// Replaces the M > 1 path of the reference's w4a32_grouped_linear
// (src/quantization/packed_v2.rs:557-624 -> gemm_w4a32_grouped,
// src/quantization/gemv.rs:1690-1725), w8a32_linear (gemv.rs:974-1061) and the
// batched SwiGLU of fused_swiglu_mlp_batched_w4a32
// (src/quantization/fused_ops.rs:1267-1319), which run one GEMV per activation
// row; here a weight byte is read once per block of activation rows.
//
// Arithmetic.  A stored weight is a small integer, exact in f16: the nibble q
// becomes (1024 + q) - 1032, at bits 4-7 of its byte (64 + q) - 72 (one AND-OR
// and half a packed subtraction), an INT8 code b becomes (1024 + b + 128) - 1152.
// An activation is scaled by a power of two 2^e (the largest magnitude of its
// row in the block's K range lands in [2^14, 2^15)) and split into two f16 limbs,
// x 2^e = h1 + h2 + r with |r| <= 2^-22 |x 2^e| (or 2^-25 absolute, 2^-39 of the
// row's largest).  Both limbs accumulate in one f32 MFMA chain over 32 elements,
// smaller limb first; the chain's result takes the group scale and is added in
// f32, and the row's 2^-e is applied once at the end.
//
// Rows of wide range.  Elements below 2^-17 of the row's largest keep fewer than
// 22 bits, and where the large ones meet zero codes nothing else is left of the
// sum.  A row in whose K range more than one in 16 nonzero elements is that small
// and fewer than 8 lie between them and 2^-10 of the largest, or whose largest is
// past 2^100, is marked by a negative 2^-e, and its slab of 32 rows is multiplied
// from the f32 activations on three bf16 limbs, which hold an f32 whole (wide_slab).
// Rows of N(0, 1) with one channel of 1e3 to 1e9 on zero codes are off by 0.8e-7 to
// 1.4e-7 of their 2-norm throughout, K from 512 to 14336, INT4 and INT8, as without
// the channel (two limbs alone, INT4: 1.5e-6 at 1e6, 1.6e-3 at 1e9).  The gap tells
// such rows from those of silu(g) u with large g, most of whose elements all but
// vanish beside the others (511 rows of 14336, a few hundred of them within 2^-17: a
// prompt of synthetic weights 30.4 ms with such rows marked, not marked 20.1).
// Counting takes 0 to 0.3 us of a call (37 x 4805 x 1600 in v2 14.6 -> 14.9 us,
// 64 x 14336 x 4096 31.2 -> 31.3).
//
// Inf and NaN travel through the first limb, as in the reference's
// unpack-and-fma.  An MFMA step rounds its sum down, which over a long row adds
// up (a mean error of 1.3e-7 of the results' size at K = 14336): the records
// hold every other group negated and its chain is subtracted, so that one
// group's bias cancels another's (negated()).
//
// Why two limbs on f16: f32 MFMA runs at 1/16 of the f16 rate, three int8
// limbs at twice the f16 rate would need an integer-to-float conversion per
// result and group, and one exponent per row instead of one per 64 elements
// leaves a single multiply-add per result and group on the vector ALUs.
//
// Tiling.  A block is four waves side by side along N, each 32 MT activation
// rows x 32 NT weight rows.  The limbs of the block's rows go to LDS by direct
// global-to-LDS loads, one K stage (SG groups of 32) ahead, and are read by
// all four waves; a lane's weights (one 16-byte chunk per 32 rows x 64 K) and
// scales go straight to registers, one stage ahead, and are expanded there.
// Lane (i, h) = (l % 32, l / 32) loads group 2 j + h of weight row i;
// v_permlane32_swap then leaves dwords 2 h and 2 h + 1 of each group in half
// h, so K slot (u, h, e) of a group (step u of two) is element
// 16 h + 8 u + e, and the records hold x in that order.
//
// Bound, from 256 rows: 950-1020 TFLOP/s of MFMA work (a large library product in
// bf16 runs at 1.2 PFLOP/s, half the nominal rate), with the matrix cores busy 0.49
// of the time and the waves waiting 0.43 of theirs.  Measured on whole calls, against the kernel on fixed-point
// limbs with an exponent per 64 elements and two more MFMAs per group for the
// -8 of the weights that this one replaced:
//   Llama-3-8B gate/up pair, 512 rows, group 32    251 us, 479 TFLOP/s (958 in
//                                                  MFMA work)
//   Llama-3-8B MLP, 512 rows, group 64             942 -> 393 us
//   64 rows, N = 14336, K = 4096, group 32         54.0 -> 31.1 us
//   Llama-3-8B MLP in INT8, 128 rows               2559 -> 151 us, against GEMV
//                                                  passes of 2 rows each
// The error against 64 bits went from 6.2e-7 to 1.4e-7 for INT4 (activations
// with large channels: the limbs follow each element's own size) and from
// 2.3e-7 to 2.1e-7 for the INT8 MLP.
#include <math.h>

#include <algorithm>

#include "gemv_common.hpp"
#include "qgemm.hpp"
#include "tb_common.hpp"

namespace tb {

using namespace gemv;

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kSlab = 32;            // activation rows of one MFMA tile
constexpr int kGroupBytes = 4096;    // one slab x 32 K: 2 steps x 2 limbs x 1 KiB
constexpr int kRun = 512;            // K per level of the row-scale sums
constexpr int kDirectGroups = 12;    // k_qdirect: K range of a block, 48 KiB of limbs
constexpr int kPad = 128;            // K is padded to whole stages in the records

// K slot e of a step's 8 holds element slot_elem(e): the order in which a dword
// of nibbles expands.
__host__ __device__ constexpr int slot_elem(int e) { return (e >> 1) | ((e & 1) << 2); }

// The groups held negated: every other one, starting anew each 4 groups (so
// that large channels a power of two apart meet both signs).
__host__ __device__ constexpr bool negated(int g) { return ((g ^ (g >> 2)) & 1) != 0; }

// The nibble masks, in registers: behind a literal the compiler takes an AND
// and an OR instead of one v_and_or_b32.  The f16 numbers that the nibbles are
// put into, in both halves: 1024 (a unit in the last place of 1) for bits 0-3,
// 64 (of 1/16) for bits 4-7.
struct Masks {
    uint32_t lo, hi, f_lo, f_hi;
};
__device__ __forceinline__ Masks nibble_masks() {
    Masks k = {0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm("" : "+v"(k.lo), "+v"(k.hi), "+s"(k.f_lo), "+s"(k.f_hi));
    return k;
}

__device__ __forceinline__ h8 expand_w4(uint32_t d, const Masks &k) {
    const uint32_t u = d >> 8;
    const u32x4 v = {(d & k.lo) | k.f_lo, (d & k.hi) | k.f_hi, (u & k.lo) | k.f_lo,
                     (u & k.hi) | k.f_hi};
    const _Float16 a = (_Float16)-1032.f, b = (_Float16)-72.f;
    return __builtin_bit_cast(h8, v) + h8{a, a, b, b, a, a, b, b};
}

__device__ __forceinline__ h8 expand_w8(uint32_t d0, uint32_t d1) {
    const uint32_t a = d0 ^ 0x80808080u, b = d1 ^ 0x80808080u, o = 0x64646464u;
    const u32x4 v = {__builtin_amdgcn_perm(a, o, 0x00050004u), __builtin_amdgcn_perm(a, o, 0x00070006u),
                     __builtin_amdgcn_perm(b, o, 0x00050004u), __builtin_amdgcn_perm(b, o, 0x00070006u)};
    const _Float16 m = (_Float16)-1152.f;
    return __builtin_bit_cast(h8, v) + h8{m, m, m, m, m, m, m, m};
}

struct QArgs {
    const float *x;        // activations (k_qdirect, wide_slab)
    const uint8_t *rec;    // split activations
    const float *inv;      // [splits][slabs * 32] 2^-e, negative for rows of wide range
    const uint8_t *w0, *w1;
    const float *s0, *s1, *b0, *b1, *res;
    float *y;              // [m, n], or the partials [splits][pair ? 2 : 1][m][n]
    int m, n, k;
    int scols, gshift, s0_len, s1_len;
    int slabs, groups;     // 32-row slabs, padded 32-K groups of the records
    int mz, nbx, splits, slen;   // row blocks, column blocks, K splits, groups per split
};

// SM: 0 a scale per 32-element group, 1 per 64 or more, 2 one per row (applied
// in the epilogue).
template <int FMT, int MT, int NT, int SM, bool PAIR>
struct QTile {
    static constexpr int SG = FMT == Q_W8 || MT == 4 ? 2 : 4;   // groups per stage
    static constexpr int LD = FMT == Q_W8 ? SG : SG / 2;   // 16-byte chunks per lane and column tile
    static constexpr int NDW = FMT == Q_V2 ? 5 : 4;
    static constexpr int NS = SM == 0 ? SG : SG / 2;       // scales per column tile and stage

    struct Stage {
        uint32_t q[NT][LD][NDW];
        float s[NT][NS];
    };

    const QArgs &a;
    int lane, wave, i, h;
    const uint8_t *wp[NT];   // the lane's weight row
    const float *sp[NT];
    uint32_t vrow[NT];       // byte offset of the lane's row (v2)
    int chunks;              // 32-element chunks of a row
    Masks msk;

    __device__ __forceinline__ QTile(const QArgs &aa) : a(aa) {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        i = lane & 31;
        h = lane >> 5;
        chunks = a.k >> 5;
        msk = nibble_masks();
    }

    __device__ __forceinline__ int col(int bx, int nt) const {
        return PAIR ? bx * 128 + 32 * wave + i : bx * (128 * NT) + 32 * (NT * wave + nt) + i;
    }

    __device__ __forceinline__ void rows(int bx) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int c = col(bx, nt);
            const size_t row = c < a.n ? c : 0;   // rows past n read row 0, never stored
            const bool second = PAIR && nt == 1;
            const uint8_t *w = second ? a.w1 : a.w0;
            vrow[nt] = (uint32_t)row * (uint32_t)((a.k >> 6) * kV2Block);
            wp[nt] = FMT == Q_V2 ? w : w + row * (size_t)(FMT == Q_W8 ? a.k : a.k >> 1);
            sp[nt] = SM == 2 || FMT == Q_V2
                         ? nullptr
                         : (second ? a.s1 : a.s0) + row * (size_t)a.scols;
        }
    }

    // Weights and scales of the stage at group g0.  Chunks past the row (K not
    // a multiple of the stage) re-read its last chunk: their activations are 0.
    __device__ __forceinline__ void load(int g0, Stage &st) const {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
            for (int j = 0; j < LD; ++j) {
                if constexpr (FMT == Q_W8) {
                    const int c = min(g0 + j, chunks - 1);
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(wp[nt] + 32 * (size_t)c + 16 * h);
                    st.q[nt][j][0] = v.x; st.q[nt][j][1] = v.y; st.q[nt][j][2] = v.z; st.q[nt][j][3] = v.w;
                } else if constexpr (FMT == Q_V2) {
                    const int c = min(g0 + 2 * j + h, chunks - 1);
                    const uint32_t o = vrow[nt] + (uint32_t)(c >> 1) * kV2Block + (uint32_t)(c & 1) * 16u;
                    const uint32_t *p = reinterpret_cast<const uint32_t *>(wp[nt] + (o & ~3u));
#pragma unroll
                    for (int d = 0; d < 5; ++d) st.q[nt][j][d] = p[d];
                } else {
                    const int c = min(g0 + 2 * j + h, chunks - 1);
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(wp[nt] + 16 * (size_t)c);
                    st.q[nt][j][0] = v.x; st.q[nt][j][1] = v.y; st.q[nt][j][2] = v.z; st.q[nt][j][3] = v.w;
                }
            }
            if constexpr (FMT == Q_V2) {
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    const int b = min((g0 >> 1) + j, (chunks >> 1) - 1);
                    st.s[nt][j] = __uint_as_float((uint32_t)*reinterpret_cast<const uint16_t *>(
                        wp[nt] + vrow[nt] + (uint32_t)b * kV2Block + 32u));
                }
            } else if constexpr (SM == 0) {
                typedef float fvu __attribute__((ext_vector_type(NS), aligned(4)));
                if (g0 + NS <= chunks) {
                    const fvu v = *reinterpret_cast<const fvu *>(sp[nt] + g0);
#pragma unroll
                    for (int t = 0; t < NS; ++t) st.s[nt][t] = v[t];
                } else {
#pragma unroll
                    for (int t = 0; t < NS; ++t)
                        st.s[nt][t] = g0 + t < chunks ? sp[nt][g0 + t] : 0.f;
                }
            } else if constexpr (SM == 1) {
#pragma unroll
                for (int t = 0; t < NS; ++t)
                    st.s[nt][t] = g0 + 2 * t < chunks ? sp[nt][(32 * (g0 + 2 * t)) >> a.gshift] : 0.f;
            }
        }
    }

    // The two B operands (steps u = 0, 1) of group g of the stage.
    __device__ __forceinline__ void expand(const Stage &st, int nt, int g, int g0, h8 (&B)[2]) const {
        if constexpr (FMT == Q_W8) {
            const uint32_t *q = st.q[nt][g];
            B[0] = expand_w8(q[0], q[1]);
            B[1] = expand_w8(q[2], q[3]);
        } else {
            const int j = g >> 1;
            uint32_t d[4];
            if constexpr (FMT == Q_V2) {
                const int c = min(g0 + 2 * j + h, chunks - 1);
                const uint32_t o = vrow[nt] + (uint32_t)(c >> 1) * kV2Block;
                const uint32_t sh = (o & 2u) * 8u;
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    d[t] = __builtin_amdgcn_alignbit(st.q[nt][j][t + 1], st.q[nt][j][t], sh);
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) d[t] = st.q[nt][j][t];
            }
            const auto s0 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
            B[0] = expand_w4((g & 1) ? s0[1] : s0[0], msk);
            B[1] = expand_w4((g & 1) ? s1[1] : s1[0], msk);
        }
    }

    __device__ __forceinline__ float scale(const Stage &st, int nt, int g) const {
        if (SM == 0) return st.s[nt][g];
        if (FMT == Q_V2) return f16_bits_to_f32(__float_as_uint(st.s[nt][g >> 1]));
        return SM == 1 ? st.s[nt][g >> 1] : 1.0f;
    }

    // One stage, a fresh chain per 32 K.  With group scales acc += scale *
    // chain; with one scale per row (SM 2) run += chain, and flush() adds run
    // to acc every kRun elements: two levels of sums keep a long row as exact
    // as the GEMV's lane tree (INT8, K = 4096, error against 64 bits: 1.3e-7
    // there; a chain that runs on for 128 K 1.5e-7, for 1024 K 3e-7; two levels
    // 1.1e-7).
    __device__ __forceinline__ void compute(const uint8_t *lds, int g0, const Stage &st,
                                            f32x16 (&acc)[MT][NT], f32x16 (&run)[MT][NT]) const {
        const float sgn = negated(g0) ? -1.f : 1.f;   // g0 is even: group g's is that of g & 1
#pragma unroll
        for (int g = 0; g < SG; ++g) {
            h8 B[NT][2];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) expand(st, nt, g, g0, B[nt]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                h8 A[2][2];   // [step][limb]
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int l = 0; l < 2; ++l)
                        A[u][l] = *reinterpret_cast<const h8 *>(
                            lds + (mt * SG + g) * kGroupBytes + (2 * u + l) * 1024 + lane * 16);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    f32x16 D = {};
#pragma unroll
                    for (int l = 1; l >= 0; --l)
#pragma unroll
                        for (int u = 0; u < 2; ++u)
                            D = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[u][l], B[nt][u], D, 0, 0, 0);
                    const float s = (g & 1) ? -sgn * scale(st, nt, g) : sgn * scale(st, nt, g);
                    if constexpr (SM == 2) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) run[mt][nt][r] = fmaf(D[r], s, run[mt][nt][r]);
                    } else {
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[mt][nt][r] = fmaf(D[r], s, acc[mt][nt][r]);
                    }
                }
            }
        }
    }

    // Group g of the stage at g0 for one slab (MT 1) on three bf16 limbs: x is the
    // lane's half of the group (elements 16 h .. 16 h + 15 of its row), up its 2^e.
    __device__ __forceinline__ void compute_wide(const f32x4 (&x)[4], float up, int g, int g0,
                                                 const Stage &st, f32x16 (&acc)[1][NT],
                                                 f32x16 (&run)[1][NT]) const {
        const float sgn = negated(g0 + g) ? -1.f : 1.f;
        h8 H[NT][2];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) expand(st, nt, g, g0, H[nt]);
        f32x16 D[NT] = {};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            b8 A[3];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int el = 8 * u + (FMT == Q_W8 ? e : slot_elem(e));
                const float v = x[el >> 2][el & 3] * (sgn * up);
                const float r1 = fabsf(v) < INFINITY ? v - (float)(__bf16)v : 0.f;
                A[0][e] = (__bf16)v;
                A[1][e] = (__bf16)r1;
                A[2][e] = (__bf16)(r1 - (float)(__bf16)r1);
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                b8 B;
#pragma unroll
                for (int e = 0; e < 8; ++e) B[e] = (__bf16)(float)H[nt][u][e];
#pragma unroll
                for (int l = 2; l >= 0; --l)
                    D[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[l], B, D[nt], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);   // one step's limbs in registers at a time
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const float s = sgn * scale(st, nt, g);
            f32x16 &to = SM == 2 ? run[0][nt] : acc[0][nt];
#pragma unroll
            for (int r = 0; r < 16; ++r) to[r] = fmaf(D[nt][r], s, to[r]);
        }
    }

    __device__ __forceinline__ static void flush(f32x16 (&acc)[MT][NT], f32x16 (&run)[MT][NT]) {
        if constexpr (SM == 2) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    acc[mt][nt] += run[mt][nt];
                    run[mt][nt] = f32x16{};
                }
        }
    }
};

// The sum over 8 consecutive lanes.
__device__ __forceinline__ float sum8(float v) {
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) v += shfl_xor_u(v, o);
    return v;
}

// Consecutive tiles (row blocks of the same columns first) on one XCD: blocks
// go to the 8 XCDs round robin, the grid is a multiple of 8.
__device__ __forceinline__ int block_tile() {
    const int per = gridDim.x >> 3;
    return (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
}

// The limbs of 8 consecutive elements a, b of a row, scaled by sc (2^e, negated
// for the groups negated() names), W4: slots in nibble order.  `lack` sums 15 for
// an element that keeps fewer than 22 bits, or is zero, and -1 for another: ordinary
// rows keep it negative in every wave, so that only others pay for a closer look
// (Spread).
template <bool W4>
__device__ __forceinline__ void limbs8(const f32x4 &a, const f32x4 &b, float sc, h8 &l1, h8 &l2,
                                       int &lack) {
    int full = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int el = W4 ? slot_elem(j) : j;
        const float s = (el < 4 ? a[el & 3] : b[el & 3]) * sc;
        const _Float16 u = (_Float16)s;
        l1[j] = u;
        l2[j] = fabsf(s) < INFINITY ? (_Float16)(s - (float)u) : (_Float16)0.f;
        full += fabsf(s) >= 0.25f;   // h2's last place is 2^-24 or more
    }
    lack += 15 * 8 - 16 * full;
    asm("" : "+v"(lack));   // summed here, not kept as 8 flags for later
}

// What decides on a row whose lack is positive: its zeros, and the elements from
// 2^-17 to 2^-10 of the largest (scaled: 2^-2 to 2^5).
struct Spread {
    int zeros = 0, mid = 0;
    __device__ __forceinline__ void add(const f32x4 &a, const f32x4 &b, float sc) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = fabsf((e < 4 ? a : b)[e & 3]);
            zeros += v == 0.f;
            mid += v * sc >= 0.25f && v * sc < 32.f;
        }
    }
};

// The largest finite magnitude of a, b and mx.
__device__ __forceinline__ float max_finite(float mx, const f32x4 &a, const f32x4 &b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float u = fabsf(a[e]), v = fabsf(b[e]);
        mx = fmaxf(mx, u < INFINITY ? u : 0.f);
        mx = fmaxf(mx, v < INFINITY ? v : 0.f);
    }
    return mx;
}

// e of a row whose largest finite magnitude is mx: mx 2^e in [2^14, 2^15), past
// 2^100 (a row of wide range) in [2^99, 2^100).
constexpr float kLargest = 0x1p100f;
__device__ __forceinline__ int row_exp(float mx) {
    int E = 0;
    (void)frexpf(mx, &E);   // mx = f 2^E, f in [0.5, 1)
    return mx > kLargest ? 100 - E : mx > 0.f ? min(15 - E, 126) : 0;
}

// 2^-e as stored: negative for a row of wide range, which has more than one short
// element in 16 (lack, over the nonzero ones, positive) and a gap above them.
__device__ __forceinline__ float row_inv(float mx, float lack = 0.f, float mid = 0.f) {
    const float v = ldexpf(1.f, -row_exp(mx));
    return mx > kLargest || (lack > 0.f && mid < 8.f) ? -v : v;
}

// The block's results, scaled by their rows' 2^-e (inv: of slab0's first row
// on), to y or the split's partials.  Register r of lane (i, h) is row
// 8 (r / 4) + 4 h + r % 4 of weight row i.  Slabs with a row of wide range are
// left out (unless WIDE) and returned, a bit each.
template <bool WIDE, int FMT, int MT, int NT, int SM, bool PAIR>
__device__ __forceinline__ int store_tile(const QArgs &a, const QTile<FMT, MT, NT, SM, PAIR> &t,
                                          const f32x16 (&acc)[MT][NT], int bx, int split,
                                          int slab0, const float *inv) {
    int left = 0;
    const bool split_k = a.splits > 1;
    const size_t plane = (size_t)a.m * a.n;
    float *y = a.y + (split_k ? (size_t)split * (PAIR ? 2 : 1) * plane : 0);
    auto row_scale = [&](const float *s, int len, int c) {
        return SM == 2 ? s[len > 1 ? c : 0] : 1.0f;
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int slab = slab0 + mt;
        if (slab >= a.slabs) break;
        f32x4 f[4];
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
            f[r4] = *reinterpret_cast<const f32x4 *>(inv + mt * kSlab + 8 * r4 + 4 * t.h);
        float least = f[0][0];
#pragma unroll
        for (int r = 1; r < 16; ++r) least = fminf(least, f[r >> 2][r & 3]);
        if (!WIDE && __any(least < 0.f)) {
            left |= 1 << mt;
            continue;
        }
#pragma unroll
        for (int nt = 0; nt < (PAIR ? 1 : NT); ++nt) {
            const int c = t.col(bx, nt);
            if (c >= a.n) continue;
            const float rs0 = row_scale(a.s0, a.s0_len, c);
            const float rs1 = PAIR ? row_scale(a.s1, a.s1_len, c) : 1.0f;
            const float b0 = !split_k && a.b0 ? a.b0[c] : 0.f;
            const float b1 = PAIR && !split_k && a.b1 ? a.b1[c] : 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = slab * kSlab + 8 * (r >> 2) + 4 * t.h + (r & 3);
                if (row >= a.m) continue;
                const size_t o = (size_t)row * a.n + c;
                const float fr = fabsf(f[r >> 2][r & 3]);
                const float g = acc[mt][nt][r] * fr * rs0;
                if constexpr (PAIR) {
                    const float u = acc[mt][NT - 1][r] * fr * rs1;
                    if (split_k) {
                        y[o] = g;
                        y[plane + o] = u;
                    } else {
                        y[o] = silu(g + b0) * (u + b1);
                    }
                } else {
                    float v = g;
                    if (!split_k) {
                        if (a.b0) v += b0;
                        if (a.res) v += a.res[o];
                    }
                    y[o] = v;
                }
            }
        }
    }
    return left;
}

// The results of one slab with rows of wide range, on three bf16 limbs: K range and
// columns as the block's, 6 MFMAs per group in place of 4.  The waves read the
// activations themselves, one group ahead, and split them: bound by those reads and
// the splitting.  Only such slabs pay for it, after the block's other work.  us for
// INT4, group 32, without such rows / with one / all of them: 64 x 14336 x 4096 34 /
// 100 / 99, 512 rows 137 / 290 / 452 (on 16 f32 MFMAs per group, without reading
// ahead: 126 / 125 and 478 / 814).
template <int FMT, int NT, int SM, bool PAIR>
__device__ __forceinline__ void wide_slab(const QArgs &a, int bx, int split, int slab,
                                          const float *inv) {
    using T = QTile<FMT, 1, NT, SM, PAIR>;
    constexpr int SG = T::SG;
    const int gb = split * a.slen, ge = min(gb + a.slen, a.groups);
    T t(a);
    t.rows(bx);
    // rows past m repeat the last one and are not stored, groups past K the last one
    // and are not added
    const float *xr = a.x + (size_t)min(slab * kSlab + t.i, a.m - 1) * a.k + 16 * t.h;
    auto fetch = [&](int g, f32x4 (&v)[4]) {
        const f32x4 *p = reinterpret_cast<const f32x4 *>(xr + 32 * (size_t)min(g, t.chunks - 1));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = p[j];
    };
    const float up = 1.0f / fabsf(inv[t.i]);   // a power of two
    f32x16 acc[1][NT] = {}, run[1][NT] = {};
    f32x4 xa[4], xb[4];
    typename T::Stage st;
    fetch(gb, xa);
#pragma unroll 1
    for (int g = gb; g < ge; g += SG) {
        t.load(g, st);
#pragma unroll
        for (int j = 0; j < SG; j += 2) {
            fetch(g + j + 1, xb);
            if (g + j < t.chunks) t.compute_wide(xa, up, j, g, st, acc, run);
            fetch(g + j + 2, xa);
            if (g + j + 1 < t.chunks) t.compute_wide(xb, up, j + 1, g, st, acc, run);
        }
        if (((g - gb) & (kRun / 32 - 1)) == kRun / 32 - SG) T::flush(acc, run);
    }
    T::flush(acc, run);
    store_tile<true>(a, t, acc, bx, split, slab, inv);
}

template <int FMT, int MT, int NT, int SM, bool PAIR>
__global__ __launch_bounds__(256, 2) void k_qgemm(QArgs a) {
    using T = QTile<FMT, MT, NT, SM, PAIR>;
    constexpr int SG = T::SG;
    constexpr int kStage = MT * SG * kGroupBytes;
    static_assert(!PAIR || NT == 2, "a pair's column tiles are gate and up");
    __shared__ __align__(16) uint8_t lds0[kStage];
    __shared__ __align__(16) uint8_t lds1[kStage];
    const int tile = block_tile();
    if (tile >= a.mz * a.nbx * a.splits) return;
    const int mz = tile % a.mz, rest = tile / a.mz;
    const int bx = rest % a.nbx, split = rest / a.nbx;
    const int gb = split * a.slen, ge = min(gb + a.slen, a.groups);

    T t(a);
    t.rows(bx);
    const int slab0 = mz * MT;

    auto stage_x = [&](uint8_t *lds, int g0) {
        constexpr int kChunks = MT * SG * 4;   // KiB pieces of a stage
#pragma unroll
        for (int c0 = 0; c0 < kChunks; c0 += 4) {
            const int c = c0 + t.wave, mt = c / (SG * 4), o = c - mt * (SG * 4);
            const int slab = min(slab0 + mt, a.slabs - 1);   // slabs past the last are not stored
            const uint8_t *src = a.rec + ((size_t)slab * a.groups + g0) * kGroupBytes + o * 1024 +
                                 t.lane * 16;
            __builtin_amdgcn_global_load_lds(src, lds + c * 1024, 16, 0, 0);
        }
    };
    auto landed = [&] {   // this wave's copies landed, then everybody's
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));   // vmcnt(0)
        __syncthreads();
    };

    f32x16 acc[MT][NT] = {}, run[MT][NT] = {};

    typename T::Stage sa, sb;
    stage_x(lds0, gb);
    t.load(gb, sa);
    landed();
    for (int g = gb; g < ge; g += 2 * SG) {
        if (g + SG < ge) {
            stage_x(lds1, g + SG);
            t.load(g + SG, sb);
        }
        t.compute(lds0, g, sa, acc, run);
        landed();
        if (g + SG >= ge) break;
        if (g + 2 * SG < ge) {
            stage_x(lds0, g + 2 * SG);
            t.load(g + 2 * SG, sa);
        }
        t.compute(lds1, g + SG, sb, acc, run);
        if (((g - gb) & (kRun / 32 - 1)) == kRun / 32 - 2 * SG) T::flush(acc, run);
        landed();
    }
    T::flush(acc, run);

    const float *inv = a.inv + ((size_t)split * a.slabs + slab0) * kSlab;
    const int left = store_tile<false>(a, t, acc, bx, split, slab0, inv);
#pragma unroll 1
    for (int mt = 0; left >> mt; ++mt)
        if ((left >> mt) & 1)
            wide_slab<FMT, NT, SM, PAIR>(a, bx, split, slab0 + mt, inv + mt * kSlab);
}

// The same projection for few rows: the block builds the limbs of its 32 rows
// itself, straight into LDS and while its first weights are on their way, 12
// groups at a time, and needs no record kernel before it.  Up to 12 groups per
// split x is read once and the loop has no barrier; a longer range (LONG) reads x
// once more before, for the rows' maxima.
// Wave w converts rows 8 w .. 8 w + 7, eight lanes each.  Small calls are bound
// by their launches: 41 x 904 x 1088 takes 8.9 us here, 12.4 with the record
// kernel (FP32 MFMA with split K, which this replaced: 9.8), 16 x 4096 x 4096
// 13.9 / 14.8 (14.7), 37 x 4805 x 1600 in v2 15.2 / 16.6 (19.3), 13 x 4605 x 1984
// in INT8 12.5 / 13.8 (35 as GEMV passes).
// (Three blocks a CU, as many as their LDS allows, where the registers do; the LONG
// form spills at three: 20 rows, N 2048, K 8192 13.4 us against 12.2.)
template <int FMT, int NT, int SM, bool PAIR, bool LONG>
__global__ __launch_bounds__(
    256, NT == 1 && !LONG && (FMT == Q_W8 || (FMT == Q_W4 && SM != 2)) ? 3 : 2)
    void k_qdirect(QArgs a) {
    using T = QTile<FMT, 1, NT, SM, PAIR>;
    constexpr int SG = T::SG, PC = kDirectGroups * 32 / 64;   // pieces of 8 per lane
    extern __shared__ __align__(16) uint8_t lds[];             // min(slen, 12) groups
    __shared__ float inv[kSlab];
    const int tile = block_tile();
    if (tile >= a.mz * a.nbx * a.splits) return;
    const int mz = tile % a.mz, rest = tile / a.mz;
    const int bx = rest % a.nbx, split = rest / a.nbx;
    const int gb = split * a.slen, ge = min(gb + a.slen, a.groups);

    T t(a);
    t.rows(bx);
    const int r = 8 * t.wave + (t.lane >> 3), row = mz * kSlab + r, c0 = t.lane & 7;
    const float *xr = a.x + (size_t)min(row, a.m - 1) * a.k;
    f32x4 xa[PC], xb[PC];
    auto piece = [&](int kk, f32x4 &va, f32x4 &vb) {
        va = vb = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row < a.m && kk < min(ge * 32, a.k)) {
            va = *reinterpret_cast<const f32x4 *>(xr + kk);
            vb = *reinterpret_cast<const f32x4 *>(xr + kk + 4);
        }
    };
    auto fetch = [&](int g0) {   // the lane's pieces of groups g0 .. g0 + 11
#pragma unroll
        for (int c = 0; c < PC; ++c) piece(g0 * 32 + 8 * (c0 + 8 * c), xa[c], xb[c]);
    };
    float mx = 0.f;
    for (int g = gb + kDirectGroups; LONG && g < ge; g += kDirectGroups) {
        fetch(g);
#pragma unroll
        for (int c = 0; c < PC; ++c) mx = max_finite(mx, xa[c], xb[c]);
    }
    fetch(gb);
    typename T::Stage sa, sb;
    t.load(gb, sa);
#pragma unroll
    for (int c = 0; c < PC; ++c) mx = max_finite(mx, xa[c], xb[c]);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) mx = fmaxf(mx, shfl_xor_u(mx, o));
    const float up = ldexpf(1.f, row_exp(mx));
    int lack = 0;
    f32x16 acc[1][NT] = {}, run[1][NT] = {};
    for (int g0 = gb; g0 < (LONG ? ge : gb + 1); g0 += kDirectGroups) {
        const int g1 = LONG ? min(g0 + kDirectGroups, ge) : ge;
        if (LONG && g0 > gb) {
            fetch(g0);
            __syncthreads();   // the last chunk's readers are done
        }
#pragma unroll
        for (int c = 0; c < PC; ++c) {
            const int p = c0 + 8 * c, g = p >> 2, q = p & 3;
            if (g0 + g < g1) {
                h8 l1, l2;
                limbs8<FMT != Q_W8>(xa[c], xb[c], negated(g0 + g) ? -up : up, l1, l2, lack);
                if (32 * g0 + 8 * p >= a.k) lack -= 15 * 8;   // padding
                uint8_t *d = lds + g * kGroupBytes + (q & 1) * 2048 + ((q >> 1) * 32 + r) * 16;
                *reinterpret_cast<h8 *>(d) = l1;
                *reinterpret_cast<h8 *>(d + 1024) = l2;
            }
        }
        __syncthreads();
        for (int g = g0; g < g1; g += 2 * SG) {
            if (g + SG < ge) t.load(g + SG, sb);
            t.compute(lds + (g - g0) * kGroupBytes, g, sa, acc, run);
            if (g + SG >= g1) {   // an odd number of stages: the next chunk's first is in sb
                if (LONG) sa = sb;
                break;
            }
            if (g + 2 * SG < ge) t.load(g + 2 * SG, sa);
            t.compute(lds + (g + SG - g0) * kGroupBytes, g + SG, sb, acc, run);
        }
        T::flush(acc, run);
    }
    float sc = row < a.m ? (float)lack : 0.f, mid = 0.f;
    sc = sum8(sc);
    if (__any(sc > 0.f)) {
        Spread sp;
#pragma unroll 1
        for (int kk = gb * 32 + 8 * c0; kk < min(ge * 32, a.k); kk += 64) {
            f32x4 va, vb;
            piece(kk, va, vb);
            sp.add(va, vb, up);
        }
        sc -= 15.f * sum8((float)sp.zeros);
        mid = sum8((float)sp.mid);
    }
    if (c0 == 0) inv[r] = row_inv(mx, sc, mid);
    __syncthreads();
    if (store_tile<false>(a, t, acc, bx, split, mz, inv))
        wide_slab<FMT, NT, SM, PAIR>(a, bx, split, mz, inv);
}

// The limbs of x [m, k] for one K split of R rows: slab s, group g at
// rec + (s groups + g) 4096, then [step][limb][lane (i, h)][8 slots].  A thread
// takes pieces of 8 elements of row t % R; rows past m and K past k are 0.
// Bound by how many CUs take part (a row's largest magnitude ties its K range to
// one block) against the length of the stores (16 R bytes).  us at 8 / 4 / 2 rows:
// 64 x 4096 5.7 / 4.9 / 4.1, 128 rows of 4096 and 14336 8.2 / 6.4 / 6.4 on average,
// 512 rows 11.6 / 9.6 / 12.4 (without the count of short elements; with it, at the
// chosen rows, 4.5, 5.9 and 9.8).
template <bool W4, int R>
__global__ __launch_bounds__(1024, 8) void k_qsplit(const float *__restrict__ x,
                                                 uint8_t *__restrict__ rec,
                                                 float *__restrict__ inv, int m, int k, int slabs,
                                                 int groups, int slen) {
    constexpr int PC = 4;   // pieces kept in registers
    __shared__ float red[16][R], mids[16][R];
    __shared__ int any_short;
    const int t = threadIdx.x, tpr = blockDim.x / R, p0 = t / R;
    const int row = blockIdx.x * R + t % R, split = blockIdx.y;
    const int k0 = split * slen * 32, k1 = min(k0 + slen * 32, groups * 32);
    const int pieces = (k1 - k0) >> 3;
    const float *xr = x + (size_t)row * k;
    auto fetch = [&](int p, f32x4 &a, f32x4 &b) {
        const int kk = k0 + 8 * p;
        a = b = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row < m && kk < k) {
            a = *reinterpret_cast<const f32x4 *>(xr + kk);
            b = *reinterpret_cast<const f32x4 *>(xr + kk + 4);
        }
    };
    float mx = 0.f;
    f32x4 ra[PC], rb[PC];
#pragma unroll
    for (int c = 0; c < PC; ++c) {
        const int p = p0 + c * tpr;
        ra[c] = rb[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (p < pieces) fetch(p, ra[c], rb[c]);
    }
#pragma unroll
    for (int c = 0; c < PC; ++c) mx = max_finite(mx, ra[c], rb[c]);
    for (int p = p0 + PC * tpr; p < pieces; p += tpr) {
        f32x4 a, b;
        fetch(p, a, b);
        mx = max_finite(mx, a, b);
    }
#pragma unroll
    for (int o = R; o < 64; o <<= 1) mx = fmaxf(mx, shfl_xor_u(mx, o));
    if ((t & 63) < R) red[t >> 6][t % R] = mx;
    if (t == 0) any_short = 0;
    __syncthreads();
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) mx = fmaxf(mx, red[w][t % R]);
    const int e = row_exp(mx);
    const float up = ldexpf(1.f, e);
    if (t < R) inv[(size_t)split * slabs * kSlab + row] = row_inv(mx);
    int lack = 0;
    auto put = [&](int p, const f32x4 &a, const f32x4 &b) {
        const int kk = k0 + 8 * p, g = kk >> 5, q = (kk >> 3) & 3;
        h8 l1, l2;
        limbs8<W4>(a, b, negated(g) ? -up : up, l1, l2, lack);
        if (kk >= k) lack -= 15 * 8;   // padding
        uint8_t *d = rec + ((size_t)(row >> 5) * groups + g) * kGroupBytes +
                     (size_t)(q & 1) * 2048 + (size_t)((q >> 1) * 32 + (row & 31)) * 16;
        *reinterpret_cast<h8 *>(d) = l1;
        *reinterpret_cast<h8 *>(d + 1024) = l2;
    };
#pragma unroll
    for (int c = 0; c < PC; ++c) {
        const int p = p0 + c * tpr;
        if (p < pieces) put(p, ra[c], rb[c]);
    }
    for (int p = p0 + PC * tpr; p < pieces; p += tpr) {
        f32x4 a, b;
        fetch(p, a, b);
        put(p, a, b);
    }
    float sc = row < m ? (float)lack : 0.f;
#pragma unroll
    for (int o = R; o < 64; o <<= 1) sc += shfl_xor_u(sc, o);
    if (sc > 0.f) any_short = 1;
    __syncthreads();
    if (!any_short) return;
    mx = 0.f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) mx = fmaxf(mx, red[w][t % R]);
    __syncthreads();
    Spread sp;
    const float scale = ldexpf(1.f, row_exp(mx));
#pragma unroll 1
    for (int p = p0; p < pieces; p += tpr) {
        f32x4 a, b;
        fetch(p, a, b);
        if (k0 + 8 * p < k) sp.add(a, b, scale);
    }
    float zc = (float)sp.zeros, mc = (float)sp.mid;
#pragma unroll
    for (int o = R; o < 64; o <<= 1) {
        zc += shfl_xor_u(zc, o);
        mc += shfl_xor_u(mc, o);
    }
    if ((t & 63) < R) {
        red[t >> 6][t % R] = sc - 15.f * zc;
        mids[t >> 6][t % R] = mc;
    }
    __syncthreads();
    if (t >= R) return;
    sc = mc = 0.f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
        sc += red[w][t];
        mc += mids[w][t];
    }
    inv[(size_t)split * slabs * kSlab + row] = row_inv(mx, sc, mc);
}

// Sum of the split-K partials in split order, then the epilogue.  res may be y
// (each element is read before the same thread writes it).
template <bool PAIR, int VEC>
__global__ __launch_bounds__(256) void k_qreduce(const float *__restrict__ part, int splits,
                                                 int m, int n, const float *__restrict__ b0,
                                                 const float *__restrict__ b1, const float *res,
                                                 float *y) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    const size_t plane = (size_t)m * n, total = plane / VEC;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const size_t o = e * VEC;
        const int c = (int)(o % (size_t)n);
        vec g = {}, u = {}, r = {}, bg = {}, bu = {};
        if (res) r = *reinterpret_cast<const vec *>(res + o);
        if (b0) bg = *reinterpret_cast<const vec *>(b0 + c);
        if (PAIR && b1) bu = *reinterpret_cast<const vec *>(b1 + c);
#pragma unroll 4
        for (int s = 0; s < splits; ++s) {
            g += *reinterpret_cast<const vec *>(part + (size_t)s * (PAIR ? 2 : 1) * plane + o);
            if (PAIR) u += *reinterpret_cast<const vec *>(part + (size_t)(2 * s + 1) * plane + o);
        }
        vec v;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            if (PAIR) {
                v[j] = silu(g[j] + bg[j]) * (u[j] + bu[j]);
            } else {
                float w = g[j];
                if (b0) w += bg[j];
                if (res) w += r[j];
                v[j] = w;
            }
        }
        *reinterpret_cast<vec *>(y + o) = v;
    }
}

constexpr int kCUs = 256;
constexpr int kMaxSplits = 16;

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t rec_bytes(const QPlan &pl) { return (size_t)pl.slabs * pl.groups * kGroupBytes; }
size_t inv_bytes(const QPlan &pl, int splits) {
    return up256((size_t)splits * pl.slabs * kSlab * sizeof(float));
}
size_t scratch_of(const QPlan &pl, int splits, bool direct, int m, int n, bool pair) {
    return (direct ? 0 : rec_bytes(pl) + inv_bytes(pl, splits)) +
           (splits > 1 ? (size_t)splits * (pair ? 2 : 1) * (size_t)m * n * sizeof(float) : 0);
}

// What a tile costs, in us per 128 K: `busy` of a CU's time when other blocks
// hide its waits, `alone` by itself; `grain` is how finely a last, partly
// filled round of blocks is paid for (blocks per CU).
struct Tile {
    int mt, nt;
    double busy, alone, grain;
};
constexpr Tile kTiles[] = {{1, 1, 0.77, 1.35, 0.25}, {1, 2, 1.95, 1.0, 0.5}, {2, 1, 1.2, 1.95, 1.0},
                           {2, 2, 2.15, 2.85, 1.0}, {4, 2, 3.9, 7.0, 1.0}};

// Tile and K split by a cost model: K stages x the block rounds of the busiest
// CU, each round's start, and for K splits the reduce kernel and the partials'
// way through memory.  The constants are fitted to sweeps of every tile and
// split at 45 shapes (5..1024 rows, N and K 900..14336, all formats): its
// choice is the fastest at 40 of them and at most 8% from it at the others
// (64 x 14336 x 4096: 38.8 us as first set, now 33.3).  Tiles of 64 x 64 and
// more outputs per wave have no room for the second sum of row scales; the
// 128-row tile is for v1 weights (5% ahead of 64 rows at 512 rows and N = 28672,
// since a weight's expansion serves twice the rows; a v2 lane holds more of its
// stage and would spill).  One K split on k_qdirect needs no scratch: some plan fits.
QPlan plan(int m, int n, int k, int fmt, bool grouped, bool pair, size_t cap) {
    QPlan pl{};
    pl.slabs = (m + kSlab - 1) / kSlab;
    pl.groups = (k + kPad - 1) / kPad * (kPad / 32);
    const int stages = pl.groups / 4;
    const double f = fmt == Q_V2 ? 1.3 : fmt == Q_W8 ? 0.72 : 1.0;
    const double fa = fmt == Q_V2 ? 1.3 : fmt == Q_W8 ? 0.95 : 1.0;
    double best = 1e30;
    for (const Tile &t : kTiles) {
        if (t.mt > pl.slabs || (pair && t.nt == 1)) continue;
        if ((!grouped && t.mt * t.nt > 2) || (fmt == Q_V2 && t.mt * t.nt > 2)) continue;
        const int mz = (pl.slabs + t.mt - 1) / t.mt;
        const int nbx = pair ? (n + 127) / 128 : (n + 128 * t.nt - 1) / (128 * t.nt);
        for (int s = 1; s <= stages && s <= kMaxSplits; ++s) {
            const int len = (stages + s - 1) / s;
            if ((stages + len - 1) / len != s) continue;
            const double blocks = (double)mz * nbx * s / kCUs;
            const double rounds = std::max(1.0, ceil(blocks / t.grain) * t.grain);
            double us = len * std::max(rounds * t.busy * f, t.alone * fa) + 1.2 * ceil(blocks / 2);
            if (s > 1) us += 3.0 + (double)(pair ? 2 : 1) * s * m * n * 1.57e-6;
            for (int d = 0; d < 2; ++d) {
                if (d && (t.mt > 1 || (t.nt == 2 && !pair))) continue;
                // the record kernel, or every block's own conversion
                const double ud =
                    us + (d ? 1.0 + (len * 4 > kDirectGroups ? 0.7 : 0.25) * len * rounds : 5.0);
                const size_t bytes = scratch_of(pl, s, d != 0, m, n, pair);
                if (ud < best && bytes <= cap) {
                    best = pl.us = ud;
                    pl.bytes = bytes;
                    pl.mt = t.mt; pl.nt = t.nt; pl.mz = mz; pl.nbx = nbx;
                    pl.splits = s; pl.slen = len * 4; pl.direct = d != 0;
                }
            }
        }
    }
    return pl;
}

// SwiGLU pairs come as INT4 with group scales and as INT8.
constexpr bool takes_pair(int fmt, bool grouped) { return fmt == Q_W8 || (fmt == Q_W4 && grouped); }

template <int FMT, int SM>
int launch(const QArgs &a, const QPlan &pl, bool pair, hipStream_t st) {
    constexpr bool PAIRS = takes_pair(FMT, SM != 2);
    const long tiles = (long)pl.mz * pl.nbx * pl.splits;
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8)), block(256);
    if (pl.direct) {
        const size_t lds = (size_t)std::min(pl.slen, kDirectGroups) * kGroupBytes;
#define TB_QDIRECT(LONG_)                                                                        \
    do {                                                                                         \
        if constexpr (PAIRS) {                                                                   \
            if (pair) {                                                                          \
                hipLaunchKernelGGL((k_qdirect<FMT, 2, SM, true, LONG_>), grid, block, lds, st, a); \
                break;                                                                           \
            }                                                                                    \
        }                                                                                        \
        hipLaunchKernelGGL((k_qdirect<FMT, 1, SM, false, LONG_>), grid, block, lds, st, a);      \
    } while (0)
        if (pl.slen > kDirectGroups) TB_QDIRECT(true);
        else TB_QDIRECT(false);
#undef TB_QDIRECT
        TB_LAUNCHED();
        return TB_OK;
    }
#define TB_QGO(MT_, NT_, PAIR_)                                                                  \
    hipLaunchKernelGGL((k_qgemm<FMT, MT_, NT_, SM, PAIR_>), grid, block, 0, st, a)
    if constexpr (FMT == Q_W4 && SM != 2) {   // see plan()
        if (pl.mt * pl.nt > 2) {
            if (pl.mt == 4) {
                if (pair) TB_QGO(4, 2, true);
                else TB_QGO(4, 2, false);
            } else {
                if (pair) TB_QGO(2, 2, true);
                else TB_QGO(2, 2, false);
            }
            TB_LAUNCHED();
            return TB_OK;
        }
    }
    if constexpr (PAIRS) {
        if (pair) {
            TB_QGO(1, 2, true);
            TB_LAUNCHED();
            return TB_OK;
        }
    }
    if (pl.mt == 2) TB_QGO(2, 1, false);
    else if (pl.nt == 2) TB_QGO(1, 2, false);
    else TB_QGO(1, 1, false);
#undef TB_QGO
    TB_LAUNCHED();
    return TB_OK;
}

// Rows of a k_qsplit block: 4, or 2 where that leaves fewer than 128 blocks.
static int split_rows(const QPlan &pl) { return pl.slabs * 8 * pl.splits < 128 ? 2 : 4; }

}  // namespace

bool qgemm_shape_ok(int64_t m, int64_t n, int64_t k, int fmt) {
    if (m < 1 || n < 1 || k < 32 || k % (fmt == Q_V2 ? 64 : 32) != 0) return false;
    return k <= (int64_t)1 << 30 && m < (int64_t)1 << 24 && n < ((int64_t)1 << 31) - 512;
}

QPlan qgemm_plan(int m, int n, int k, int fmt, bool grouped, bool pair, size_t cap) {
    return plan(m, n, k, fmt, grouped, pair, cap);
}

int qgemm(const QGemmParams &p, const QPlan &pl, void *scratch, hipStream_t st) {
    const bool pair = p.w1 != nullptr;
    TB_REQUIRE(qgemm_shape_ok(p.m, p.n, p.k, p.fmt), TB_ERR_UNSUPPORTED,
               "TB_UNSUPPORTED: batched projection needs K % 32 == 0");
    TB_REQUIRE(!pair || takes_pair(p.fmt, p.grouped != 0), TB_ERR_UNSUPPORTED,
               "TB_UNSUPPORTED: batched SwiGLU pairs are INT8, or INT4 with group scales");
    uint8_t *rec = static_cast<uint8_t *>(scratch);
    float *inv = nullptr, *part = reinterpret_cast<float *>(rec);
    if (!pl.direct) {
        inv = reinterpret_cast<float *>(rec + rec_bytes(pl));
        part = reinterpret_cast<float *>(rec + rec_bytes(pl) + inv_bytes(pl, pl.splits));
    }
    if (!pl.direct) {
        const int r = split_rows(pl);
        const dim3 pg((unsigned)(pl.slabs * (kSlab / r)), (unsigned)pl.splits);
        const int want = r * pl.slen;   // 4 pieces of 8 a thread
        const unsigned threads = want <= 256 ? 256 : want <= 512 ? 512 : 1024;
#define TB_QS(W4, R)                                                                      \
    hipLaunchKernelGGL((k_qsplit<W4, R>), pg, dim3(threads), 0, st, p.x, rec, inv, p.m, p.k, \
                       pl.slabs, pl.groups, pl.slen)
        if (p.fmt == Q_W8) {
            if (r == 2) TB_QS(false, 2);
            else TB_QS(false, 4);
        } else {
            if (r == 2) TB_QS(true, 2);
            else TB_QS(true, 4);
        }
#undef TB_QS
        TB_LAUNCHED();
    }
    QArgs a{};
    a.x = p.x; a.rec = rec; a.inv = inv;
    a.w0 = static_cast<const uint8_t *>(p.w0);
    a.w1 = static_cast<const uint8_t *>(p.w1);
    a.s0 = p.s0; a.s1 = p.s1; a.b0 = p.b0; a.b1 = p.b1; a.res = p.res;
    a.y = pl.splits > 1 ? part : p.y;
    a.m = p.m; a.n = p.n; a.k = p.k;
    a.scols = p.grouped ? p.k >> p.gshift : 0;
    a.gshift = p.gshift; a.s0_len = p.s0_len; a.s1_len = p.s1_len;
    a.slabs = pl.slabs; a.groups = pl.groups;
    a.mz = pl.mz; a.nbx = pl.nbx; a.splits = pl.splits; a.slen = pl.slen;
    int rc;
    if (p.fmt == Q_W8) rc = launch<Q_W8, 2>(a, pl, pair, st);
    else if (p.fmt == Q_V2) rc = launch<Q_V2, 1>(a, pl, pair, st);
    else if (!p.grouped) rc = launch<Q_W4, 2>(a, pl, pair, st);
    else if (p.gshift == 5) rc = launch<Q_W4, 0>(a, pl, pair, st);
    else rc = launch<Q_W4, 1>(a, pl, pair, st);
    if (rc || pl.splits == 1) return rc;
    const size_t total = (size_t)p.m * p.n;
    const bool v4 = p.n % 4 == 0 && !(((uintptr_t)p.y | (uintptr_t)p.b0 | (uintptr_t)p.b1 |
                                       (uintptr_t)p.res) & 15);
    const unsigned rb = (unsigned)std::min<size_t>((total / (v4 ? 4 : 1) + 255) / 256, 4096);
#define TB_QRED(PAIR_, VEC_)                                                                     \
    hipLaunchKernelGGL((k_qreduce<PAIR_, VEC_>), dim3(rb), dim3(256), 0, st, part, pl.splits,    \
                       p.m, p.n, p.b0, p.b1, p.res, p.y)
    if (pair) {
        if (v4) TB_QRED(true, 4);
        else TB_QRED(true, 1);
    } else {
        if (v4) TB_QRED(false, 4);
        else TB_QRED(false, 1);
    }
#undef TB_QRED
    TB_LAUNCHED();
    return TB_OK;
}

}  // namespace tb
