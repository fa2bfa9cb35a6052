// Shared device helpers for the gfx950 kernels: storage types, bf16 conversion,
// wave64 reductions.  Storage precision is separate from arithmetic: every
// reduction, softmax statistic and accumulator is float.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define WAVE 64

typedef uint16_t bf16_t;

// dtype codes shared with the Python wrappers
enum { DT_F32 = 0, DT_BF16 = 1 };

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
    return __uint_as_float(((uint32_t)v) << 16);
}

// round to nearest even, NaN stays NaN (the rule of the reference's kernels/precision.cuh:13-20),
// done by the hardware conversion of gfx950 (v_cvt_pk_bf16_f32)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    return __builtin_bit_cast(bf16_t, (__bf16)f);
}

// two floats to a pair of bf16 in one register (low half first)
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f32x2_t;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
    const f32x2_t v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Where a sum over `units` pieces of a row of `of` (which matrix, which group of its rows) begins; it goes round from there.
// Rows of a power of two in bytes lie on the same few memory channels at the same piece, and blocks that all begin at the
// first piece ask the same channels for everything at once: 16 matrices of 2048 x 4096 bf16 in 67 us (3.7 TB/s), 42 with
// beginnings spread over the row.
__device__ __forceinline__ int first_unit(int matrix, int group, int units) { return (int)((unsigned)(group + 9 * matrix) % (unsigned)units); }

__device__ __forceinline__ float load_f32(const float* p) { return *p; }
__device__ __forceinline__ float load_f32(const bf16_t* p) { return bf16_to_f32(*p); }
__device__ __forceinline__ void store_f32(float* p, float v) { *p = v; }
__device__ __forceinline__ void store_f32(bf16_t* p, float v) { *p = f32_to_bf16(v); }

// V neighbouring elements as floats, by one load or store where V is 4 (16 bytes of floats, 8 of bf16, which the address is a multiple of)
template <int V>
__device__ __forceinline__ void load_run(const float* p, float (&v)[V]) {
    if constexpr (V == 4) { const float4 w = *(const float4*)p; v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w; }
    else for (int i = 0; i < V; ++i) v[i] = p[i];
}
template <int V>
__device__ __forceinline__ void load_run(const bf16_t* p, float (&v)[V]) {
    if constexpr (V == 4) {
        const uint2 w = *(const uint2*)p;
        v[0] = __uint_as_float(w.x << 16); v[1] = __uint_as_float(w.x & 0xffff0000u);
        v[2] = __uint_as_float(w.y << 16); v[3] = __uint_as_float(w.y & 0xffff0000u);
    } else {
        for (int i = 0; i < V; ++i) v[i] = load_f32(p + i);
    }
}
template <int V>
__device__ __forceinline__ void store_run(float* p, const float (&v)[V]) {
    if constexpr (V == 4) *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    else for (int i = 0; i < V; ++i) p[i] = v[i];
}
template <int V>
__device__ __forceinline__ void store_run(bf16_t* p, const float (&v)[V]) {
    if constexpr (V == 4) *(uint2*)p = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    else for (int i = 0; i < V; ++i) store_f32(p + i, v[i]);
}

// 1 / sqrt(total inv_k + eps), a row's factor in an RMSNorm that a product finishes: the approximate reciprocal root and one step of
// Newton's.  The instruction knows no numbers below the normal ones, so a mean that is nearly one of them is taken 2^64 times as large.  Off
// by at most 2 units in the last place (the mean rounds twice, the step once; the library's quotient, root and quotient as much).  Those three
// are the last thing that a short kernel does: 16 steps of one row, 61 such products each, 9,456 us with them, 9,359 so; of eight rows 12,664 / 12,616.
__device__ __forceinline__ float row_factor(float total, float inv_k, float eps) {
    const float mean = fmaf(total, inv_k, eps);
    const bool tiny = mean < 0x1p-100f;
    const float m = tiny ? mean * 0x1p64f : mean, f = __builtin_amdgcn_rsqf(m);
    const float g = m > 0.f && m < INFINITY ? fmaf(f, fmaf(-0.5f * m * f, f, 0.5f), f) : f;
    return tiny ? g * 0x1p32f : g;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, WAVE));
    return v;
}

// Sum over a block of NT threads (NT a multiple of 64, at most 1024).  `red`
// is LDS scratch of at least NT/64 floats.  Every thread gets the total.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < NT / WAVE; ++w) total += red[w];
    return total;
}

// The law of a gated activation act(gate, up), the epilogue of a product over [gate; up]:
//   limit 0:     silu(g) u
//   limit > 0:   g' sigmoid(slope g') (u' + shift) with g' = min(g, limit), u' = clamp(u, -limit, limit)
//   limit < 0:   gelu(g) u, the gelu's tanh form
// A struct of zeros is the first law.
struct GateLaw { float limit, slope, shift; };

// g sigmoid(z) where it goes on to bf16.  exp(-z) = 2^t exp(rho) with t = -z / ln 2 rounded and rho what the rounding left, in two
// pieces of ln 2; then the quotient from the approximate reciprocal and one correction, both of a quarter of the divisor, as the
// reciprocal of 1 + exp(87.4) and beyond is below the smallest normal number.  Relative error at most 2.1e-7 (g / (1 + expf(-z)):
// 1.9e-7) down to z = -88.72; below, where the exponential is past the largest float, the sigmoid is 0 as there.  Over 2^24 products silu(g) u of
// normal g (0.3 to 30 wide) and u the error of the bf16 results against 64 bits is the same in all ten digits.  The maximum keeps g = inf from
// inf - inf.  As the epilogue of a product nothing runs beside it: with this, and the law asked for once a row, the gated ring product
// takes 13.2 us for 14.8 at 1,777 x 3,072, K 576 (13.0 without the quarter, whose results between z = -87.34 and -88.72 were 0),
// 74.5 for 78.2 at 1,061 x 16,384, K 2,048, 155 for 165 at 2,345 rows, 203 for 213 at 907 x 28,672, K 4,096.
__device__ __forceinline__ float times_sigmoid_to_bf16(float g, float z) {
    const float c = __builtin_amdgcn_fmed3f(z, -88.7228f, 88.f);
    const float t = c * -1.44269502f, rho = fmaf(t, 1.90465432e-9f, fmaf(t, -0.693147182f, -c));
    float e = __builtin_amdgcn_exp2f(t);
    e = fmaf(e, rho, e);
    const float d = fmaf(e, 0.25f, 0.25f), h = 0.25f * g;
    const float r = z < -88.7228f ? 0.f : __builtin_amdgcn_rcpf(d), q = h * r;
    return fmaf(fmaxf(fmaf(-d, q, h), -3.0e38f), r, q);
}

template <typename TC>
__device__ __forceinline__ float times_sigmoid(float g, float z) {
    if constexpr (sizeof(TC) == 2) return times_sigmoid_to_bf16(g, z);
    return g / (1.0f + expf(-z));
}

// the law for results of type TC
template <typename TC>
__device__ __forceinline__ float gated_activation(float g, float u, const GateLaw& law) {
    if (law.limit > 0.f) {
        g = fminf(g, law.limit);
        u = fminf(fmaxf(u, -law.limit), law.limit);
        return times_sigmoid<TC>(g, law.slope * g) * (u + law.shift);
    }
    if (law.limit < 0.f)      // (0.5 (1 + tanh z) = 1 / (1 + exp(-2 z)))
        return times_sigmoid<TC>(g, 1.5957691216057308f * (g + 0.044715f * g * g * g)) * u;
    return times_sigmoid<TC>(g, g) * u;
}

// An ungated activation, the epilogue of a product that feeds a feed-forward's second matrix:
//   1: z Phi(z), the gelu with the error function     2: its tanh form 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3)))
//   3: relu(z)^2
enum { ACT_NONE = 0, ACT_GELU = 1, ACT_GELU_TANH = 2, ACT_RELU2 = 3 };

__device__ __forceinline__ float unary_activation(float z, int act) {
    if (act == ACT_GELU) return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
    if (act == ACT_RELU2) { const float r = fmaxf(z, 0.f); return r * r; }
    return 0.5f * z * (1.0f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
}

// The gelu with the error function where the result is rounded to bf16: z / 2 erfc(-z / sqrt 2), with erfc(x) = t 2^(p(t) - x^2 / ln 2),
// t = 1 / (1 + x / 2), for x >= 0 and 2 - erfc(|x|) below, the form of W. H. Press et al., Numerical Recipes; p is a polynomial fitted here
// (Chebyshev nodes, t from 1/8 to 1) to log2(e^(x^2) erfc(x) / t).  Relative error of erfc(-z / sqrt 2) in 32 bits: 6e-7 for z > -1, 1.4e-6 to
// -5, 4.5e-6 to -8, 1.4e-5 to -13.2 (x^2 / ln 2 is rounded where it is large); 1 + erff(z / sqrt 2) has 1.4e-7 for z > -1, 7e-6 to -3,
// 4e-2 to -5 and no digit beyond.  A sixth of erff's instructions: as the epilogue of 1,999 x 8,192, K 2,048 the activation took 30 us of 86.
__device__ __forceinline__ float gelu_to_bf16(float z) {
    const float x = fabsf(z) * 0.70710678118654752f, t = __builtin_amdgcn_rcpf(fmaf(0.5f, x, 1.0f));
    float p = 0.0669854358f;
    p = fmaf(p, t, -0.578201771f); p = fmaf(p, t, 1.67653584f); p = fmaf(p, t, -2.0672853f); p = fmaf(p, t, 0.893760622f);
    p = fmaf(p, t, -0.20385237f); p = fmaf(p, t, 0.600722373f); p = fmaf(p, t, 1.43684995f); p = fmaf(p, t, -1.82551515f);
    const float tail = t * __builtin_amdgcn_exp2f(fmaf(-x * 1.4426950408889634f, x, p));
    return 0.5f * z * (z < 0.f ? tail : 2.0f - tail);
}

// the activation of a result of type TC
template <typename TC>
__device__ __forceinline__ float activation_to(float z, int act) {
    return sizeof(TC) == 2 && act == ACT_GELU ? gelu_to_bf16(z) : unary_activation(z, act);
}

// as the epilogue of a product: the sum is rounded to the output's type first, as the path of two kernels does
template <typename TC>
__device__ __forceinline__ float activated(float v, int act) {
    if (sizeof(TC) == 2) v = bf16_to_f32(f32_to_bf16(v));
    return activation_to<TC>(v, act);
}

#define CISR_LAUNCH_CHECK() ((int)hipGetLastError())
