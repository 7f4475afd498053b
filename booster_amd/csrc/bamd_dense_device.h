// bamd_dense_device.h — device-side pieces shared by the kernels of the configured layer stacks: operand fragments and their matrix-core products for both
// activation types, block reductions, and the row mechanisms in the form that both the row kernels and the prologues of the few-row product use.
#pragma once
#include "bamd_dense.h"
#include <type_traits>

typedef __bf16 bamd_bf;
typedef __bf16 bamd_bf8 __attribute__((ext_vector_type(8)));
typedef float bamd_v4 __attribute__((ext_vector_type(4)));
typedef unsigned int bamd_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ float bf_f(uint16_t u) { return __uint_as_float((uint32_t) u << 16); }

// eight consecutive k of one row / column
template <typename T> struct Frag;
template <> struct Frag<bamd_bf> {
    bamd_bf8 v;
    __device__ __forceinline__ void zero() { v = __builtin_bit_cast(bamd_bf8, bamd_u4{ 0, 0, 0, 0 }); }
    __device__ __forceinline__ void load(const bamd_bf * p) { v = *(const bamd_bf8 *) p; }
    __device__ __forceinline__ void set(int i, float f) { v[i] = (bamd_bf) f; }
    __device__ __forceinline__ void store(bamd_bf * p) const { *(bamd_bf8 *) p = v; }
};
template <> struct Frag<float> {
    bamd_v4 a, b;
    __device__ __forceinline__ void zero() { a = bamd_v4{ 0, 0, 0, 0 }; b = a; }
    __device__ __forceinline__ void load(const float * p) { a = *(const bamd_v4 *) p; b = *(const bamd_v4 *) (p + 4); }
    __device__ __forceinline__ void set(int i, float f) { if (i < 4) a[i] = f; else b[i - 4] = f; }
    __device__ __forceinline__ void store(float * p) const { *(bamd_v4 *) p = a; *(bamd_v4 *) (p + 4) = b; }
};
// D[row = (lane / 16) * 4 + i][col = lane % 16] += sum over 32 k of A[row][k] B[k][col]
__device__ __forceinline__ bamd_v4 mma(const Frag<bamd_bf> & a, const Frag<bamd_bf> & b, bamd_v4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0); }
__device__ __forceinline__ bamd_v4 mma(const Frag<float> & a, const Frag<float> & b, bamd_v4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.a[i], b.a[i], c, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.b[i], b.b[i], c, 0, 0, 0);
    return c;
}
template <typename T> __device__ __forceinline__ T to_act(float f) { return (T) f; }

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.0f) + log1pf(expf(-fabsf(x))); }

// sum over the wave, the same in every lane: rows of sixteen lanes by data-parallel moves, then the four rows
__device__ __forceinline__ float wave_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));      // lane ^ 1
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true));      // lane ^ 2
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true));     // the other four of eight
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, true));     // the other eight of sixteen
    const int i = __float_as_int(v);
    return (__int_as_float(__builtin_amdgcn_readlane(i, 0)) + __int_as_float(__builtin_amdgcn_readlane(i, 16))) + (__int_as_float(__builtin_amdgcn_readlane(i, 32)) + __int_as_float(__builtin_amdgcn_readlane(i, 48)));
}
// maximum and sum over the sixteen lanes of a row
__device__ __forceinline__ float row_sum16(float v) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, true));
    return v;
}
__device__ __forceinline__ float row_max16(float v) {
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, true)));
    return v;
}
// The tile of a flash kernel's block.  Tiles come with the longest key ranges first; where every CU gets a second block and none a third one, the second ones are taken the other way round,
// so that the longest range shares its CU with the shortest.
__device__ __forceinline__ int paired_tile(int heads) {
    const int at = blockIdx.x / heads, n = gridDim.x / heads, half = 256 / heads;
    return at >= half && n <= 2 * half ? n - 1 - (at - half) : at;
}
__device__ __forceinline__ float wave_max(float v) {
    const int i = __float_as_int(row_max16(v));
    return fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(i, 0)), __int_as_float(__builtin_amdgcn_readlane(i, 16))), fmaxf(__int_as_float(__builtin_amdgcn_readlane(i, 32)), __int_as_float(__builtin_amdgcn_readlane(i, 48))));
}
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); }

// sums of NV values over the block; red: NV * 16 floats of LDS.  Every thread gets the result.  The waves' sums are read by sixteen lanes at once: a loop over them is a chain of up to
// 16 NV reads of LDS, in front of every product of one row and in every row kernel
// (131 tokens read and 24 chatted at width 2048: 11.73 -> 11.57 ms; sixteen sequences served at 4096: 34.89 -> 34.62)
template <int NV> __device__ __forceinline__ void block_sum(float (&v)[NV], float * red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
    __syncthreads();
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) red[i * 16 + wave] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = row_sum16((lane & 15) < nw ? red[i * 16 + (lane & 15)] : 0.f);
}

template <typename T> __device__ __forceinline__ void store4(T * h, bamd_v4 v);
template <> __device__ __forceinline__ void store4<float>(float * h, bamd_v4 v) { *(bamd_v4 *) h = v; }
template <> __device__ __forceinline__ void store4<bamd_bf>(bamd_bf * h, bamd_v4 v) {
    typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
    *(bf4 *) h = bf4{ (bamd_bf) v[0], (bamd_bf) v[1], (bamd_bf) v[2], (bamd_bf) v[3] };
}
// A 32-bit operand is the sum of three bfloat16 numbers in planes 32 elements apart: the largest one below it, the largest below what is left, and the rest, which has eight bits.  All three are
// exact and have the number's sign, none is zero (from 1e-28 on) unless the number is, and an infinity or NaN is what is left of itself: so a product with a number or a weight that is not
// finite is what it would be in 32 bits, without a test for it.
// The number is fixed before it is taken apart: where it is a product, the compiler would fuse that into the subtraction, and the parts were those of the product without its rounding, cut off at the third
struct Split { uint32_t p[3]; };                                   // in the upper sixteen bits
__device__ __forceinline__ Split split_f(float v) {
    asm("" : "+v"(v));
    const uint32_t some = v != 0.f, h = __float_as_uint(v) - some;
    const float m = v - __uint_as_float(h & 0xffff0000u);
    const uint32_t g = __float_as_uint(m) - some;
    return { { h, g, __float_as_uint(m - __uint_as_float(g & 0xffff0000u)) } };
}
struct bamd_s3 {
    uint16_t v;
    __device__ __forceinline__ void operator=(Split s) { (&v)[0] = (uint16_t) (s.p[0] >> 16); (&v)[32] = (uint16_t) (s.p[1] >> 16); (&v)[64] = (uint16_t) (s.p[2] >> 16); }
};
template <typename T> struct OperandOf { typedef T type; };
template <> struct OperandOf<float> { typedef bamd_s3 type; };
template <typename T> using Operand = typename OperandOf<T>::type;      // what the operand rows of products in compute type T are made of
template <typename T> constexpr int bamd_planes = sizeof(T) == 4 ? 3 : 1;
template <typename O> __device__ __forceinline__ auto to_operand(float f) { if constexpr (std::is_same<O, bamd_s3>::value) return split_f(f); else return (O) f; }
template <> __device__ __forceinline__ void store4<bamd_s3>(bamd_s3 * h, bamd_v4 v) {
    Split s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = split_f(v[i]);
#pragma unroll
    for (int n = 0; n < 3; ++n) *(uint2 *) ((uint16_t *) h + n * 32) = uint2{ (s[0].p[n] >> 16) | (s[1].p[n] & 0xffff0000u), (s[2].p[n] >> 16) | (s[3].p[n] & 0xffff0000u) };
}
// a row of operands (O) being written (null: not wanted)
template <typename O> struct RowOut {
    static constexpr int P = std::is_same<O, bamd_s3>::value ? 3 : 1;
    O * p; int cb;
    __device__ __forceinline__ explicit operator bool() const { return p != nullptr; }
    __device__ __forceinline__ O * at(int i) const { return p + (i >> 5) * cb + (i & 31); }
    __device__ __forceinline__ O * at(int base, int j, int lane) const { return p + ((base >> 5) + (j >> 1)) * cb + ((j & 1) * 16 + lane); }      // column base + 16 j + lane of a base that is a multiple of 32
};
template <typename O> __device__ __forceinline__ RowOut<O> row_out(void * h, int row, int ld, int cb) {
    constexpr int P = RowOut<O>::P;
    return { h ? (O *) h + (size_t) row * (cb ? 32 * P : ld * P) : nullptr, cb ? cb : 32 * P };
}
template <typename O> __device__ __forceinline__ void zero_tail(RowOut<O> h, int n, int ld) { for (int i = n + threadIdx.x; i < ld; i += blockDim.x) *h.at(i) = to_operand<O>(0.f); }

// A row of n floats spread over the block, kept in registers between the passes over it: four at a time, or (ONE) one at a time, a block's width apart, where n is no multiple of four and rows start
// anywhere.  `fits`: at most RC pieces of four per thread; longer rows are read again for every sum.  Odd widths on registers, before and after, us: a token of four layers of 3098 371 -> 327 (Mafurax), 1998 208 -> 188 (Tupitar), eight sequences of 587 190 -> 165
template <int RC, bool ONE> struct RowRegs {
    bamd_v4 v[RC];
    static __device__ __forceinline__ bool fits(int n) { return (ONE || (n & 3) == 0) && n <= (int) blockDim.x * 4 * RC; }
    static __device__ __forceinline__ int at(int c, int k) { return ONE ? (int) threadIdx.x + (c * 4 + k) * (int) blockDim.x : ((int) threadIdx.x + c * (int) blockDim.x) * 4 + k; }
    __device__ __forceinline__ void load(const float * p, int n) {
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            if constexpr (ONE && RC > 4) {                        // long rows (PolyNorm's): a branch for four values of the block, none for a thread's.  32 tests of a thread's were 1.5 us of a kernel's 8
                v[c] = bamd_v4{ 0, 0, 0, 0 };
                if (c * 4 * (int) blockDim.x < n)
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[c][k] = p[at(c, k) < n ? at(c, k) : n - 1];
            } else if constexpr (ONE)
#pragma unroll
                for (int k = 0; k < 4; ++k) v[c][k] = at(c, k) < n ? p[at(c, k)] : 0.f;
            else v[c] = at(c, 0) < n ? *(const bamd_v4 *) (p + at(c, 0)) : bamd_v4{ 0, 0, 0, 0 };
        }
        if constexpr (ONE && RC > 4)                              // (once all of them are asked for)
#pragma unroll
            for (int c = 0; c < RC; ++c) if (c * 4 * (int) blockDim.x < n && (c + 1) * 4 * (int) blockDim.x > n)
#pragma unroll
                for (int k = 0; k < 4; ++k) v[c][k] = at(c, k) < n ? v[c][k] : 0.f;
    }
    // the sum of one or two planes
    __device__ __forceinline__ void load(const float * p, int n, int parts, size_t plane) {
        load(p, n);
        if (parts <= 1) return;
        RowRegs b; b.load(p + plane, n);
#pragma unroll
        for (int i = 0; i < RC; ++i) v[i] = v[i] + b.v[i];
    }
    __device__ __forceinline__ void store(float * p, int n) const {
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            if constexpr (ONE) {
#pragma unroll
                for (int k = 0; k < 4; ++k) if (at(c, k) < n) p[at(c, k)] = v[c][k];
            } else if (at(c, 0) < n) *(bamd_v4 *) (p + at(c, 0)) = v[c];
        }
    }
    template <typename O> __device__ __forceinline__ void put(RowOut<O> h, int n, int from = 0) const {      // from: pieces in front of these
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            if constexpr (ONE) {
#pragma unroll
                for (int k = 0; k < 4; ++k) if (at(from + c, k) < n) *h.at(at(from + c, k)) = to_operand<O>(v[c][k]);
            } else if (at(from + c, 0) < n) store4<O>(h.at(at(from + c, 0)), v[c]);
        }
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int c = 0; c < RC; ++c) v[c] = bamd_v4{ 0, 0, 0, 0 };
    }
    __device__ __forceinline__ float squares() const {
        float t = 0.f;
#pragma unroll
        for (int c = 0; c < RC; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) { if constexpr (ONE) t = fmaf(v[c][k], v[c][k], t); else t += v[c][k] * v[c][k]; }      // (ONE: as rows that are read again are summed)
        return t;
    }
};

__device__ __forceinline__ float parts_sum(const float * p, int parts, size_t plane) { return parts > 1 ? p[0] + p[plane] : p[0]; }

// mean and variance (mean of the squared deviations) of a row in registers: per wave around its own mean, then over the waves; ONE: around the row's mean, as rows that are read again.  red: 48
// floats of LDS.  Which square of a sum is rounded by itself is written out: left to the compiler, it changes with the code around it, and a last place of a variance moves every result behind it
template <int RC, bool ONE> __device__ __forceinline__ void row_moments(const RowRegs<RC, ONE> & r, int n, float * red, float & mean, float & var) {
    if constexpr (ONE) {
        float v[1] = { 0.f };
#pragma unroll
        for (int i = 0; i < RC; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) v[0] += r.v[i][k];        // (zero behind the row)
        block_sum<1>(v, red);
        mean = v[0] / (float) n; v[0] = 0.f;
#pragma unroll
        for (int i = 0; i < RC; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) { const float d = r.v[i][k] - mean; if (r.at(i, k) < n) v[0] = fmaf(d, d, v[0]); }
        block_sum<1>(v, red);
        var = v[0] / (float) n;
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    float s = 0.f, c = 0.f, q = 0.f;
#pragma unroll
    for (int i = 0; i < RC; ++i) if (r.at(i, 0) < n) { s += (r.v[i][0] + r.v[i][1]) + (r.v[i][2] + r.v[i][3]); c += 4.f; }
    s = wave_sum(s); c = wave_sum(c);
    const float m = c > 0.f ? s / c : 0.f;
#pragma unroll
    for (int i = 0; i < RC; ++i) if (r.at(i, 0) < n) {
        const bamd_v4 d = r.v[i] - m;
        if (i == 0) q = fmaf(d[0], d[0], d[1] * d[1]);
        else { q = fmaf(d[0], d[0], q); q = fmaf(d[1], d[1], q); }
        q = fmaf(d[2], d[2], q); q = fmaf(d[3], d[3], q);
    }
    q = wave_sum(q);
    __syncthreads();
    if (lane == 0) { red[wave] = m; red[16 + wave] = q; red[32 + wave] = c; }
    __syncthreads();
    const int w = lane & 15;
    const float mw = w < nw ? red[w] : 0.f, qw = w < nw ? red[16 + w] : 0.f, cw = w < nw ? red[32 + w] : 0.f;
    mean = row_sum16(mw * cw) / (float) n;
    const float d = mw - mean;
    var = row_sum16(qw + cw * d * d) / (float) n;
}
// residual sum with the layer norm of the sublayer's output, and the layer norm (gain gi, null: none) the next sublayer reads, of one row by the whole block
template <typename T, bool ONE>
__device__ __forceinline__ void layer_row(const bamd_residual_args & a, int row, const float * gi, RowOut<T> h, bool write, float * red) {
    constexpr int RC = 2;
    const int E = a.E;
    const float * x = a.x + (size_t) row * E, * y = a.y ? a.y + (size_t) row * a.ldy : nullptr;
    float * xo = a.xo + (size_t) row * E;
    if (RowRegs<RC, ONE>::fits(E)) {
        RowRegs<RC, ONE> xr, yr, g, w;
        xr.load(x, E);
        if (y) { yr.load(y, E, a.parts, a.plane); g.load(a.g, E); }
        if (gi) w.load(gi, E);
        float mean, var;
        if (y) {
            row_moments(yr, E, red, mean, var);
            const float r = 1.0f / sqrtf(var + a.eps);
#pragma unroll
            for (int c = 0; c < RC; ++c) xr.v[c] = xr.v[c] + (yr.v[c] - mean) * r * g.v[c];
        }
        if (write) xr.store(xo, E);
        if (!h) return;
        if (gi) {
            if constexpr (ONE)                                    // (what lies behind the row is not zero any more)
#pragma unroll
                for (int c = 0; c < RC; ++c)
#pragma unroll
                    for (int k = 0; k < 4; ++k) if (xr.at(c, k) >= E) xr.v[c][k] = 0.f;
            row_moments(xr, E, red, mean, var);
            const float r = 1.0f / sqrtf(var + a.eps);
#pragma unroll
            for (int c = 0; c < RC; ++c) xr.v[c] = (xr.v[c] - mean) * r * w.v[c];
        }
        xr.put(h, E);
        zero_tail(h, E, a.ldh);
        return;
    }
    float my = 0.f, ry = 0.f, v[1];
    if (y) {
        v[0] = 0.f;
        for (int i = threadIdx.x; i < E; i += blockDim.x) v[0] += parts_sum(y + i, a.parts, a.plane);
        block_sum<1>(v, red);
        my = v[0] / (float) E; v[0] = 0.f;
        for (int i = threadIdx.x; i < E; i += blockDim.x) { const float d = parts_sum(y + i, a.parts, a.plane) - my; v[0] += d * d; }
        block_sum<1>(v, red);
        ry = 1.0f / sqrtf(v[0] / (float) E + a.eps);
    }
    auto at = [&](int i) { return y ? x[i] + (parts_sum(y + i, a.parts, a.plane) - my) * ry * a.g[i] : x[i]; };
    float mx = 0.f, rx = 1.f;
    if (gi && h) {
        v[0] = 0.f;
        for (int i = threadIdx.x; i < E; i += blockDim.x) v[0] += at(i);
        block_sum<1>(v, red);
        mx = v[0] / (float) E; v[0] = 0.f;
        for (int i = threadIdx.x; i < E; i += blockDim.x) { const float d = at(i) - mx; v[0] += d * d; }
        block_sum<1>(v, red);
        rx = 1.0f / sqrtf(v[0] / (float) E + a.eps);
    }
    for (int i = threadIdx.x; i < E; i += blockDim.x) {
        const float xn = at(i);
        if (write) xo[i] = xn;
        if (h) *h.at(i) = to_operand<T>(gi ? (xn - mx) * rx * gi[i] : xn);
    }
    if (h) zero_tail(h, E, a.ldh);
}
__device__ __forceinline__ float clamped_glu(float gate, float up, float limit) {
    const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
    return g / (1.0f + __expf(-1.702f * g)) * (u + 1.0f);
}
// columns [from, to) of a row
template <typename T>
__device__ __forceinline__ void glu_row(const bamd_glu_args & a, int row, RowOut<T> h, int from, int to) {
    const float * z = a.z + (size_t) row * a.ldz;
    for (int i = from + threadIdx.x * 4; i < to; i += blockDim.x * 4) {
        const bamd_v4 g = *(const bamd_v4 *) (z + (i >> 4) * 32 + (i & 15)), u = *(const bamd_v4 *) (z + (i >> 4) * 32 + 16 + (i & 15));
        store4<T>(h.at(i), bamd_v4{ clamped_glu(g[0], u[0], a.limit), clamped_glu(g[1], u[1], a.limit), clamped_glu(g[2], u[2], a.limit), clamped_glu(g[3], u[3], a.limit) });
    }
}

// residual sum, norm of the sublayer's output and token shift of one row by the whole block.  h: LDS or global row (null: none).  write: this block also stores x' and the
// state.  SINGLE: the step has one row
template <typename T, bool SINGLE, bool ONE>
__device__ __forceinline__ void residual_row(const bamd_batch_dev & b, const bamd_residual_args & a, int row, RowOut<T> h, bool write, float * red) {
    constexpr int RC = 2;
    const bool shifted = a.mu != nullptr;
    const int E = a.E;
    const float * x = a.x + (size_t) row * E, * y = a.y ? a.y + (size_t) row * a.ldy : nullptr;
    bamd_entry e; bool first = true, last = true;
    if (shifted) {
        e = b.ent[SINGLE ? 0 : b.row_entry[row]];
        if (!SINGLE) { first = row == e.row0; last = row == e.row0 + e.n - 1; }
    }
    const bool before = !SINGLE && shifted && !first;            // x' of the row in front is rebuilt here: another block may be the one that stores it
    const float * xp = before ? x - E : nullptr, * yp = before && y ? y - a.ldy : nullptr;
    const float * sp = shifted && first && e.pos0 > 0 ? a.prev + ((size_t) e.par * b.n_seq + e.seq) * E : nullptr;
    float * so = shifted && last && write ? a.prev + ((size_t) (e.par ^ 1) * b.n_seq + e.seq) * E : nullptr;
    if (RowRegs<RC, ONE>::fits(E)) {
        RowRegs<RC, ONE> xr, yr, pr, qr, mu;
        xr.load(x, E);
        if (y) yr.load(y, E, a.parts, a.plane);
        if (shifted) { mu.load(a.mu, E); if (before) { pr.load(xp, E); if (yp) qr.load(yp, E, a.parts, a.plane); } else if (sp) pr.load(sp, E); else pr.clear(); }
        float r = 0.f, rp = 0.f;
        if (y) {
            const float g = a.g[0];
            if constexpr (SINGLE) { float v[1] = { yr.squares() }; block_sum<1>(v, red); r = g / sqrtf(v[0] / (float) E + a.eps); }
            else { float v[2] = { yr.squares(), yp ? qr.squares() : 0.f }; block_sum<2>(v, red); r = g / sqrtf(v[0] / (float) E + a.eps); rp = g / sqrtf(v[1] / (float) E + a.eps); }
#pragma unroll
            for (int c = 0; c < RC; ++c) xr.v[c] = xr.v[c] + yr.v[c] * r;
        }
        if (write) { xr.store(a.xo + (size_t) row * E, E); if (so) xr.store(so, E); }
        if (!h) return;
        if (shifted)
#pragma unroll
            for (int c = 0; c < RC; ++c) { bamd_v4 pv = pr.v[c]; if (yp) pv = pv + qr.v[c] * rp; xr.v[c] = xr.v[c] + (pv - xr.v[c]) * mu.v[c]; }
        xr.put(h, E);
        zero_tail(h, E, a.ldh);
        return;
    }
    float r = 0.f, rp = 0.f;
    if (y) {
        float v[2] = { 0.f, 0.f };
        for (int i = threadIdx.x; i < E; i += blockDim.x) { const float t = parts_sum(y + i, a.parts, a.plane); v[0] += t * t; if (yp) { const float u = parts_sum(yp + i, a.parts, a.plane); v[1] += u * u; } }
        block_sum<2>(v, red);
        const float g = a.g[0];
        r = g / sqrtf(v[0] / (float) E + a.eps); rp = g / sqrtf(v[1] / (float) E + a.eps);
    }
    for (int i = threadIdx.x; i < E; i += blockDim.x) {
        const float xn = y ? x[i] + parts_sum(y + i, a.parts, a.plane) * r : x[i];
        float hn = xn;
        if (shifted) {
            const float pv = before ? (yp ? xp[i] + parts_sum(yp + i, a.parts, a.plane) * rp : xp[i]) : (sp ? sp[i] : 0.f);
            hn = xn + (pv - xn) * a.mu[i];
        }
        if (write) { a.xo[(size_t) row * E + i] = xn; if (so) so[i] = xn; }
        if (h) *h.at(i) = to_operand<T>(hn);
    }
    if (h) zero_tail(h, E, a.ldh);
}
template <typename T, bool ONE>
__device__ __forceinline__ void final_row(const bamd_residual_args & a, int row, const float * gf, RowOut<T> h, float * red) {
    constexpr int RC = 4;
    const int E = a.E;
    const float * x = a.x + (size_t) row * E, * y = a.y ? a.y + (size_t) row * a.ldy : nullptr;
    float v[1] = { 0.f }, w[1] = { 0.f };
    if (RowRegs<RC, ONE>::fits(E)) {
        RowRegs<RC, ONE> xr, yr;
        xr.load(x, E);
        if (y) {
            yr.load(y, E, a.parts, a.plane);
            v[0] = yr.squares();
            block_sum<1>(v, red);
            const float r = a.g[0] / sqrtf(v[0] / (float) E + a.eps);
#pragma unroll
            for (int c = 0; c < RC; ++c) xr.v[c] = xr.v[c] + yr.v[c] * r;
        }
        w[0] = xr.squares();
        block_sum<1>(w, red);
        const float rf = gf[0] / sqrtf(w[0] / (float) E + a.eps);
#pragma unroll
        for (int c = 0; c < RC; ++c) xr.v[c] = xr.v[c] * rf;
        xr.put(h, E);
        zero_tail(h, E, a.ldh);
        return;
    }
    float r = 0.f;
    if (y) {
        for (int i = threadIdx.x; i < E; i += blockDim.x) { const float t = parts_sum(y + i, a.parts, a.plane); v[0] += t * t; }
        block_sum<1>(v, red);
        r = a.g[0] / sqrtf(v[0] / (float) E + a.eps);
    }
    for (int i = threadIdx.x; i < E; i += blockDim.x) { const float xn = y ? x[i] + parts_sum(y + i, a.parts, a.plane) * r : x[i]; w[0] += xn * xn; }
    block_sum<1>(w, red);
    const float rf = gf[0] / sqrtf(w[0] / (float) E + a.eps);
    for (int i = threadIdx.x; i < E; i += blockDim.x) *h.at(i) = to_operand<T>((y ? x[i] + parts_sum(y + i, a.parts, a.plane) * r : x[i]) * rf);
    zero_tail(h, E, a.ldh);
}
template <typename T, bool ONE>
__device__ __forceinline__ void poly_row(const bamd_poly_args & a, int row, RowOut<T> h, float * red) {
    constexpr int RC = 8;
    const float * z = a.z + (size_t) row * a.ldz;
    float v[3] = { 0.f, 0.f, 0.f }, c0, c1, c2, c3;
    auto sums = [&](float t) { const float t2 = t * t, t3 = t2 * t; v[0] += t2; v[1] += t2 * t2; v[2] += t3 * t3; };
    auto coefficients = [&] {
        block_sum<3>(v, red);
        const float n = (float) a.F;
        c1 = a.coef[0] / sqrtf(v[0] / n + a.eps); c2 = a.coef[1] / sqrtf(v[1] / n + a.eps); c3 = a.coef[2] / sqrtf(v[2] / n + a.eps); c0 = a.coef[3];
    };
    auto value = [&](float t) { const float t2 = t * t; return c1 * t + c2 * t2 + c3 * (t2 * t) + c0; };
    if (RowRegs<RC, ONE>::fits(a.F)) {
        RowRegs<RC, ONE> zr;
        zr.load(z, a.F);
        // pieces that no thread has are passed over: two of eight are there for 8192 values on 1024 threads
#pragma unroll
        for (int c = 0; c < RC; ++c)
            if (c * 4 * (int) blockDim.x < a.F)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float t = zr.v[c][k], t2 = t * t, t3 = t2 * t;
                    if constexpr (ONE) { v[0] = fmaf(t, t, v[0]); v[1] = fmaf(t2, t2, v[1]); v[2] = fmaf(t3, t3, v[2]); } else sums(t);
                }
        coefficients();
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            if (c * 4 * (int) blockDim.x >= a.F) break;
            RowRegs<1, ONE> o;
#pragma unroll
            for (int k = 0; k < 4; ++k) o.v[0][k] = value(zr.v[c][k]);
            o.put(h, a.F, c);
        }
    } else {
        for (int i = threadIdx.x; i < a.F; i += blockDim.x) sums(z[i]);
        coefficients();
        for (int i = threadIdx.x; i < a.F; i += blockDim.x) *h.at(i) = to_operand<T>(value(z[i]));
    }
    zero_tail(h, a.F, a.ldh);
}
// inv: LDS, one float per part and 16 more
template <typename T>
__device__ __forceinline__ void group_norm_row(const bamd_group_norm_args & a, int row, RowOut<T> h, float * inv) {
    constexpr int RC = 4;
    const float * y = a.y + (size_t) row * a.ldy;
    const int per = a.n / a.groups, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6, wp = nw / a.groups;      // wp: waves per part
    if (wp >= 1 && nw % a.groups == 0 && (per & 3) == 0 && per <= wp * 256 * RC) {
        const int g = wave / wp, base = g * per, at0 = ((wave % wp) * 64 + lane) * 4, by = wp * 256;
        bamd_v4 v[RC]; float t = 0.f;
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            v[c] = at0 + c * by < per ? *(const bamd_v4 *) (y + base + at0 + c * by) : bamd_v4{ 0, 0, 0, 0 };
#pragma unroll
            for (int k = 0; k < 4; ++k) t += v[c][k] * v[c][k];
        }
        t = wave_sum(t);
        __syncthreads();
        if (lane == 0) inv[wave] = t;
        __syncthreads();
        const float sum = row_sum16((lane & 15) < wp ? inv[g * wp + (lane & 15)] : 0.f);
        const float r = 1.0f / sqrtf(sum / (float) per + a.eps);
#pragma unroll
        for (int c = 0; c < RC; ++c) { const int i = at0 + c * by; if (i < per) store4<T>(h.at(base + i), v[c] * r * *(const bamd_v4 *) (a.w + base + i)); }
        zero_tail(h, a.n, a.ldh);
        return;
    }
    if (a.groups >= nw) {                                        // parts are taken by waves in turn
        for (int g = wave; g < a.groups; g += nw) {
            float v = 0.f;
            for (int i = lane; i < per; i += 64) { const float t = y[g * per + i]; v += t * t; }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
            if (lane == 0) inv[g] = 1.0f / sqrtf(v / (float) per + a.eps);
        }
        __syncthreads();
    } else {
        for (int g = 0; g < a.groups; ++g) {
            float v[1] = { 0.f };
            for (int i = threadIdx.x; i < per; i += blockDim.x) { const float t = y[g * per + i]; v[0] += t * t; }
            block_sum<1>(v, inv + a.groups);
            if (threadIdx.x == 0) inv[g] = 1.0f / sqrtf(v[0] / (float) per + a.eps);
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < a.n; i += blockDim.x) *h.at(i) = to_operand<T>(y[i] * inv[i / per] * a.w[i]);
    zero_tail(h, a.n, a.ldh);
}
