// Device helpers shared by the surrogate-MLP kernels (mlp_kernels.hip, mlp_rows.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cfd {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// round-to-nearest-even float -> bf16 bits, one value or two in a word (the first in the low half)
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
    const bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint2 f2bf4(const float *f) { return make_uint2(f2bf2(f[0], f[1]), f2bf2(f[2], f[3])); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// 1 / (1 + e^-z). The reciprocal of x in [1, 2^126) is the hardware's estimate with one step of
// Newton's method, which equals the correctly rounded quotient for every such float (compared
// exhaustively) in 3 instructions instead of the division's 10.
__device__ __forceinline__ float sigmoidf_(float z) {
    const float x = 1.0f + __expf(-z);
    if (!(x < 0x1p126f)) return 1.0f / x;
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}

// sigmoidf_ of four values, with one branch for their rare divisions.
__device__ __forceinline__ void sigmoid4(const float (&z)[4], float (&s)[4]) {
    float x[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        x[q] = 1.0f + __expf(-z[q]);
        const float r = __builtin_amdgcn_rcpf(x[q]);
        s[q] = __builtin_fmaf(__builtin_fmaf(-x[q], r, 1.0f), r, r);
    }
    if (fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])) >= 0x1p126f)
        for (int q = 0; q < 4; q++) s[q] = 1.0f / x[q];
}

__device__ __forceinline__ bf16x8 load8(const uint16_t *p) {
    return *reinterpret_cast<const bf16x8 *>(p);
}

// Minibatch sample of a row: a counter-based hash (SplitMix64) of (seed, step, row), modulo n.
__device__ __forceinline__ int sample_index(unsigned long long seed, int step, int rows, int r, int n) {
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * ((unsigned long long)step * (unsigned long long)rows + r + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (int)(z % (unsigned long long)n);
}

// Place of W[m][k] (rows of K) in MFMA operand order: blocks of 16 x 32, a lane's eight values together,
// so that a wave's operand load is 1 KB in one run.
__device__ __forceinline__ size_t operand_at(int m, int k, int K) {
    return (size_t)((m / 16) * (K / 32) + k / 32) * 512 + 8 * (m % 16 + 16 * (k % 32 / 8)) + k % 8;
}

// One Adam update of weight w from gradient gi: moments m1, m2 and w -= lr (m1 c1) / (sqrt(m2 c2) + eps).
__device__ __forceinline__ void adam_one(float &w, float &m1, float &m2, float gi, float lr, float b1, float b2,
                                         float eps, float c1, float c2) {
    m1 = b1 * m1 + (1.0f - b1) * gi;
    m2 = b2 * m2 + (1.0f - b2) * gi * gi;
    w -= lr * (m1 * c1) / (sqrtf(m2 * c2) + eps);
}

// s + the eight bf16 values of v, in pairs.
__device__ __forceinline__ float add8(float s, uint4 v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; q++) s += bf2f((uint16_t)(w[q] & 0xffff)) + bf2f((uint16_t)(w[q] >> 16));
    return s;
}

// Part tt of 256 of the sum of a bf16 row of n values (a multiple of 512), from value j on: eight values
// per step (one 16-byte load, at(j)), four steps in flight, on top of the sums s4.
template <class At>
__device__ __forceinline__ float row_part(const At &at, int j, int n, float (&s4)[4]) {
    for (; j + 3 * 2048 < n; j += 4 * 2048)
#pragma unroll
        for (int u = 0; u < 4; u++) s4[u] = add8(s4[u], *reinterpret_cast<const uint4 *>(at(j + u * 2048)));
    for (; j < n; j += 2048) s4[0] = add8(s4[0], *reinterpret_cast<const uint4 *>(at(j)));
    return (s4[0] + s4[1]) + (s4[2] + s4[3]);
}

}  // namespace
}  // namespace cfd
