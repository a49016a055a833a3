// Weight quantizers on gfx950: the formats the GEMVs read, produced on the
// device straight from f32 checkpoint tensors.
//
//   * grouped INT4 (python/torchburn/quantization.py:53-118): per group of
//     group_size elements s = max(max|w| / 7, 1e-8), q = clamp(
//     round_half_even(w / s), -8, 7), byte j = (q[2j] + 8) | (q[2j+1] + 8) << 4.
//     Groups of 32 or 64 divide every row, so the tensor is one run of groups: a
//     lane takes four elements per load and the group maximum is a butterfly
//     over the group's 8 or 16 lanes (weights that are not 16-byte aligned: one
//     element per lane).  Any other group size: one wavefront per group for the scales,
//     then one thread per byte (its two elements may lie in two groups).
//   * per-channel INT8 (src/quantization/fused_ops.rs:554-589): s = max|w| / 127
//     (1 when max|w| <= 1e-8), q = clamp(round_half_away(w * (1 / s)), -127, 127).
//     One block per row, four elements per load where the row allows it.
//   * per-channel INT4 (quantize_linear_weights_int4, src/quantization/fused_ops.rs:
//     592-639): s = max|w| / 7 (1 when max|w| <= 1e-8), q = clamp(round_half_away(
//     w * (1 / s)), -8, 7) + 8 packed two per byte; an odd K pads its last byte
//     with the nibble 8.  One block per row.
//   * v2 -> v1 (python/torchburn/llm/loader.py:540-561, the cache migration):
//     32 nibble bytes copied, the binary16 scale widened to f32.
#include <math.h>

#include <algorithm>

#include "gemv_common.hpp"
#include "quantize.hpp"
#include "tb_common.hpp"

namespace tb {

using namespace gemv;

namespace {

// q + 8 of an element of a group of scale s.
__device__ __forceinline__ uint32_t nibble_of(float v, float s) {
    const float q = __builtin_rintf(__fdiv_rn(v, s));
    return (uint32_t)((int)fminf(fmaxf(q, -8.0f), 7.0f) + 8);
}

// Bound: the weights' stream in.  One element per lane (k_quant_int4) issued a
// load and a byte store per 64 elements and waited for each; four elements per
// load and kQuantLoads loads in flight per lane take 14336 x 4096 (group 64) from
// 194 to 50 us (5.3 TB/s in and out; a large copy moves 5.0).
constexpr int kQuantLoads = 4;

template <int GS>
__global__ __launch_bounds__(256) void k_quant_int4_flat(const float *__restrict__ w,
                                                         uint16_t *__restrict__ packed,
                                                         float *__restrict__ scales,
                                                         int64_t quads) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int LG = GS / 4;   // lanes per group
    const int64_t q0 = (int64_t)blockIdx.x * (256 * kQuantLoads) + threadIdx.x;
    f32x4 v[kQuantLoads];
#pragma unroll
    for (int u = 0; u < kQuantLoads; ++u) {
        const int64_t i = q0 + 256 * u;   // whole groups are inside or outside
        v[u] = i < quads ? __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(w) + i)
                         : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < kQuantLoads; ++u) {
        const int64_t i = q0 + 256 * u;
        float amax = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
#pragma unroll
        for (int off = 1; off < LG; off <<= 1) amax = fmaxf(amax, shfl_xor_u(amax, off));
        const float s = fmaxf(__fdiv_rn(amax, 7.0f), 1e-8f);
        const uint32_t b = nibble_of(v[u].x, s) | (nibble_of(v[u].y, s) << 4) |
                           (nibble_of(v[u].z, s) << 8) | (nibble_of(v[u].w, s) << 12);
        if (i < quads) {
            packed[i] = (uint16_t)b;
            if (i % LG == 0) scales[i / LG] = s;
        }
    }
}

template <int GS>
__global__ __launch_bounds__(256) void k_quant_int4(const float *__restrict__ w,
                                                    uint8_t *__restrict__ packed,
                                                    float *__restrict__ scales, int64_t n, int k) {
    const int lane = threadIdx.x & 63;
    const int spans = (k + 63) / 64;
    const int64_t span = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (span >= n * spans) return;   // whole waves leave together
    const int64_t row = span / spans;
    const int c0 = (int)(span - row * spans) * 64;
    const bool valid = c0 + lane < k;
    const float v = valid ? w[row * k + c0 + lane] : 0.f;
    float amax = fabsf(v);
#pragma unroll
    for (int off = 1; off < GS; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    const float s = fmaxf(__fdiv_rn(amax, 7.0f), 1e-8f);
    const uint32_t u = nibble_of(v, s);
    const uint32_t hi = (uint32_t)__shfl_down((int)u, 1);
    if (valid && (lane & 1) == 0)
        packed[row * (k / 2) + (c0 + lane) / 2] = (uint8_t)(u | (hi << 4));
    if (valid && (lane % GS) == 0) scales[row * (k / GS) + (c0 + lane) / GS] = s;
}

// Any group size: the scale of group id (row id / (k / gs)), one wavefront each.
__global__ __launch_bounds__(256) void k_quant_int4_scales(const float *__restrict__ w,
                                                           float *__restrict__ scales, int64_t n,
                                                           int k, int gs) {
    const int lane = threadIdx.x & 63;
    const int64_t ng = k / gs;
    for (int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); id < n * ng;
         id += (int64_t)gridDim.x * 4) {   // wave-uniform trip count
        const int64_t row = id / ng;
        const float *p = w + row * k + (id - row * ng) * gs;
        float amax = 0.f;
        for (int e = lane; e < gs; e += 64) amax = fmaxf(amax, fabsf(p[e]));
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
        if (lane == 0) scales[id] = fmaxf(__fdiv_rn(amax, 7.0f), 1e-8f);
    }
}

// Any group size: byte j of a row from elements 2 j and 2 j + 1 and their
// groups' scales.
__global__ __launch_bounds__(256) void k_quant_int4_pack(const float *__restrict__ w,
                                                         const float *__restrict__ scales,
                                                         uint8_t *__restrict__ packed, int64_t n,
                                                         int k, int gs) {
    const int64_t bpr = k / 2;
    for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < n * bpr;
         id += (int64_t)gridDim.x * 256) {
        const int64_t row = id / bpr;
        const int e = 2 * (int)(id - row * bpr);
        const float *wr = w + row * k;
        const float *sr = scales + row * (k / gs);
        auto nib = [&](int c) { return nibble_of(wr[c], sr[c / gs]); };
        packed[id] = (uint8_t)(nib(e) | (nib(e + 1) << 4));
    }
}

// The same rows four elements at a time (K % 4 == 0, 16-byte aligned weights,
// 4-byte aligned codes): the first 4096 elements of a row stay in registers
// between the maximum and the rounding.
__global__ __launch_bounds__(256) void k_quant_int8_vec(const float *__restrict__ w,
                                                        int8_t *__restrict__ q,
                                                        float *__restrict__ scales, int k) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int NV = 4;
    __shared__ float red[4];
    const int t = threadIdx.x, quads = k >> 2;
    const f32x4 *wr = reinterpret_cast<const f32x4 *>(w + (size_t)blockIdx.x * k);
    f32x4 v[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = t + 256 * u;
        v[u] = i < quads ? wr[i] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float mx = 0.f;
    auto see = [&](const f32x4 &a) {
        mx = fmaxf(fmaxf(mx, fmaxf(fabsf(a.x), fabsf(a.y))), fmaxf(fabsf(a.z), fabsf(a.w)));
    };
#pragma unroll
    for (int u = 0; u < NV; ++u) see(v[u]);
    for (int i = t + 256 * NV; i < quads; i += 256) see(wr[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = mx > 1e-8f ? __fdiv_rn(mx, 127.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, s);
    if (t == 0) scales[blockIdx.x] = s;
    uint32_t *qr = reinterpret_cast<uint32_t *>(q + (size_t)blockIdx.x * k);
    auto put = [&](int i, const f32x4 &a) {
        uint32_t b = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = roundf(__fmul_rn(a[e], inv));   // roundf: ties away
            b |= ((uint32_t)(int8_t)fminf(fmaxf(x, -127.0f), 127.0f) & 0xFFu) << (8 * e);
        }
        qr[i] = b;
    };
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (t + 256 * u < quads) put(t + 256 * u, v[u]);
    for (int i = t + 256 * NV; i < quads; i += 256) put(i, wr[i]);
}

__global__ __launch_bounds__(256) void k_quant_int8(const float *__restrict__ w,
                                                    int8_t *__restrict__ q,
                                                    float *__restrict__ scales, int k) {
    __shared__ float red[4];
    const float *wr = w + (size_t)blockIdx.x * k;
    float mx = 0.f;
    for (int i = threadIdx.x; i < k; i += blockDim.x) mx = fmaxf(mx, fabsf(wr[i]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = mx > 1e-8f ? __fdiv_rn(mx, 127.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, s);
    if (threadIdx.x == 0) scales[blockIdx.x] = s;
    int8_t *qr = q + (size_t)blockIdx.x * k;
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        const float t = __fmul_rn(wr[i], inv);
        qr[i] = (int8_t)fminf(fmaxf(roundf(t), -127.0f), 127.0f);   // roundf: ties away
    }
}

__global__ __launch_bounds__(256) void k_quant_int4_rows(const float *__restrict__ w,
                                                         uint8_t *__restrict__ packed,
                                                         float *__restrict__ scales, int k) {
    __shared__ float red[4];
    const float *wr = w + (size_t)blockIdx.x * k;
    float mx = 0.f;
    for (int i = threadIdx.x; i < k; i += blockDim.x) mx = fmaxf(mx, fabsf(wr[i]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = mx > 1e-8f ? __fdiv_rn(mx, 7.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, s);
    if (threadIdx.x == 0) scales[blockIdx.x] = s;
    const int kp = (k + 1) / 2;
    uint8_t *pr = packed + (size_t)blockIdx.x * kp;
    for (int j = threadIdx.x; j < kp; j += blockDim.x) {
        uint32_t nib[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = 2 * j + h;
            // roundf: ties away from zero, as Rust's f32::round; a NaN (a NaN
            // weight, or an infinite one times inv = 0) stays NaN through
            // Rust's clamp and casts to 0, so its nibble is 8
            const float t = e < k ? roundf(__fmul_rn(wr[e], inv)) : 0.f;
            const float q = __builtin_isnan(t) ? 0.f : fminf(fmaxf(t, -8.0f), 7.0f);
            nib[h] = (uint32_t)((int)q + 8) & 15u;
        }
        pr[j] = (uint8_t)(nib[0] | (nib[1] << 4));
    }
}

// One thread per block: 32 nibble bytes, then the f16 scale as f32.
__global__ __launch_bounds__(256) void k_unpack_v2(const uint8_t *__restrict__ blocked,
                                                   uint8_t *__restrict__ w,
                                                   float *__restrict__ s, int64_t total) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const uint32_t o = (uint32_t)(t * kV2Block);
    const u32x4 a = load_v2_chunk(blocked, o), b = load_v2_chunk(blocked, o + 16u);
    uint4 *dst = reinterpret_cast<uint4 *>(w + t * 32);
    dst[0] = make_uint4(a.x, a.y, a.z, a.w);
    dst[1] = make_uint4(b.x, b.y, b.z, b.w);
    s[t] = load_v2_scale(blocked, o);
}

}  // namespace

int quantize_int4_grouped(const float *w, uint8_t *packed, float *scales, int64_t n, int64_t k,
                          int gs, hipStream_t st) {
    if (gs != 32 && gs != 64) {
        const int64_t groups = n * (k / gs), bytes = n * (k / 2);
        if (groups == 0) return TB_OK;
        // grid-stride loops: at most 65536 blocks of each
        hipLaunchKernelGGL(k_quant_int4_scales,
                           dim3((unsigned)std::min<int64_t>((groups + 3) / 4, 65536)), dim3(256),
                           0, st, w, scales, n, (int)k, gs);
        TB_LAUNCHED();
        if (bytes == 0) return TB_OK;
        hipLaunchKernelGGL(k_quant_int4_pack,
                           dim3((unsigned)std::min<int64_t>((bytes + 255) / 256, 65536)),
                           dim3(256), 0, st, w, scales, packed, n, (int)k, gs);
        TB_LAUNCHED();
        return TB_OK;
    }
    // k % gs == 0: whole groups, one after another
    const int64_t quads = n * k / 4, per = 256 * kQuantLoads;
    if (quads == 0) return TB_OK;
    if ((reinterpret_cast<uintptr_t>(w) & 15) == 0 && (reinterpret_cast<uintptr_t>(packed) & 1) == 0 &&
        (quads + per - 1) / per < ((int64_t)1 << 31)) {
        const dim3 fg((unsigned)((quads + per - 1) / per));
        uint16_t *p16 = reinterpret_cast<uint16_t *>(packed);
        if (gs == 32)
            hipLaunchKernelGGL(k_quant_int4_flat<32>, fg, dim3(256), 0, st, w, p16, scales, quads);
        else
            hipLaunchKernelGGL(k_quant_int4_flat<64>, fg, dim3(256), 0, st, w, p16, scales, quads);
        TB_LAUNCHED();
        return TB_OK;
    }
    const int64_t waves = n * ((k + 63) / 64);
    const dim3 grid((unsigned)((waves + 3) / 4));
    if (gs == 32)
        hipLaunchKernelGGL(k_quant_int4<32>, grid, dim3(256), 0, st, w, packed, scales, n, (int)k);
    else
        hipLaunchKernelGGL(k_quant_int4<64>, grid, dim3(256), 0, st, w, packed, scales, n, (int)k);
    TB_LAUNCHED();
    return TB_OK;
}

int quantize_int4_rows(const float *w, uint8_t *packed, float *scales, int64_t n, int64_t k,
                       hipStream_t st) {
    if (n == 0) return TB_OK;
    hipLaunchKernelGGL(k_quant_int4_rows, dim3((unsigned)n), dim3(256), 0, st, w, packed, scales,
                       (int)k);
    TB_LAUNCHED();
    return TB_OK;
}

int quantize_int8(const float *w, int8_t *q, float *scales, int64_t n, int64_t k,
                  hipStream_t st) {
    if (n == 0) return TB_OK;
    if (k % 4 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
        (reinterpret_cast<uintptr_t>(q) & 3) == 0)
        hipLaunchKernelGGL(k_quant_int8_vec, dim3((unsigned)n), dim3(256), 0, st, w, q, scales,
                           (int)k);
    else
        hipLaunchKernelGGL(k_quant_int8, dim3((unsigned)n), dim3(256), 0, st, w, q, scales,
                           (int)k);
    TB_LAUNCHED();
    return TB_OK;
}

int unpack_v2_to_v1(const uint8_t *blocked, uint8_t *w, float *s, int64_t n, int64_t k,
                    hipStream_t st) {
    const int64_t total = n * (k / 64);
    if (total == 0) return TB_OK;
    hipLaunchKernelGGL(k_unpack_v2, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                       blocked, w, s, total);
    TB_LAUNCHED();
    return TB_OK;
}

}  // namespace tb
