// FP32 matrix products on the fp16 matrix cores: every FP32 operand, scaled by a power of two, is split into two fp16 terms
// and the product is summed from three fp16 products (the splitting of Dekker 1971, doi:10.1007/BF01397083, and Ootomo and Yokota
// 2022, doi:10.1177/10943420221090256).
//
// x·2^s = h + l + e with h = fp16(x·2^s) and l = fp16(x·2^s - h), each rounded to nearest even: 22 significant bits and a
// sign, |e| <= 2^-23 of |x·2^s| while l is a normal number (|x·2^s| >= 2^-3), and at most 2^-25 below that. x·y is then
// hl + lh + hh; the term left out, ll, is below 2^-22 of |x·y|. fp16 products are exact in FP32, and
// v_mfma_f32_32x32x16_f16 adds 16 of them per accumulator rounding, so a dot product rounds far less often than on
// v_mfma_f32_32x32x2f32, which more than makes up for the two bits.
//
// The scales put the largest magnitude of an operand's rows at 2^8 or more, so what is lost below 2^-3 is at most 2^-33 of it:
// far below FP32's own rounding of any sum that small elements share with the large ones. A result that does not share its sums
// with the rows that set the scale (a mask hides them, or their weights are 0) may lose more than FP32 does, up to all of it.
// Callers therefore test how far a result's rows lie below the scale, and compute again with FP32 MFMAs where it is too far.
//
// An element that is not finite, or that passes 65504 after scaling, has h = ±inf and l = ∓inf or NaN: every result that it
// enters is NaN (inf - inf, or 0·inf). Callers test for these too and compute them again in the same way.
//
// Cost: v_mfma_f32_32x32x16_f16 does 16 times the work of an FP32 MFMA per cycle, so three products take 3/16 of its time,
// and unlike FP32 MFMAs they co-execute with VALU work. Splitting takes 2.5 VALU instructions per element (1.5
// unscaled): v_fma_mixlo/mixhi_f16 scale, subtract and round in one. (Three bf16 terms and six products need no scale, but at twice the
// MFMAs, 5.5 instructions per element and half as much LDS traffic again: the 64 x 1024 x 64 forward took 84 µs so.)
#pragma once

#include <type_traits>

#include "attention_device.hpp"

namespace rk {

typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) float *LdsFloats;

__device__ __forceinline__ f32x16 mfma_f16(const h16x8 a, const h16x8 b, const f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// The two terms of a pair of floats times `scale` (a power of two), packed; SCALED = false takes them as they are. The high
// terms are hidden from the compiler between their conversion and their use: it otherwise converts the two again one by one
// (and, unscaled, turns each fused subtraction into a conversion and a subtraction).
template<bool SCALED>
__device__ __forceinline__ void split_pair(const float a, const float b, const float scale, uint32_t &h, uint32_t &l) {
    h = __builtin_bit_cast(uint32_t, __builtin_convertvector((SCALED ? f32x2{a * scale, b * scale} : f32x2{a, b}), h16x2));
    __asm__("" : "+v"(h));
    const h16x2 hi = __builtin_bit_cast(h16x2, h);
    const h16x2 lo{static_cast<_Float16>(fmaf(a, scale, -static_cast<float>(hi[0]))),
            static_cast<_Float16>(fmaf(b, scale, -static_cast<float>(hi[1])))};
    l = __builtin_bit_cast(uint32_t, lo);
}

// 1.0 in a scalar register, the scale of an unscaled split (as a constant it would fold the fused subtraction away).
__device__ __forceinline__ float split_unit_scale() {
    float one = 1.0f;
    __asm__("" : "+s"(one));
    return one;
}

// Exponent e of a non-zero magnitude in [2^e, 2^(e + 1)); 0 for zero (denormals count as 2^-127).
__device__ __forceinline__ int exponent_of(const float magnitude) {
    return magnitude > 0.0f ? static_cast<int>(__float_as_uint(magnitude) >> 23) - 127 : 0;
}

// 2^e for e in -126 .. 127.
__device__ __forceinline__ float power_of_two(const int e) { return __uint_as_float(static_cast<uint32_t>(e + 127) << 23); }

constexpr int kMaxExponent = 100; // largest scale exponent: 2^±100 times a sum of products stays far inside FP32's range

// 2^-e, e clamped to the exponents a scale may have (beyond them callers use FP32 MFMAs).
__device__ __forceinline__ float scale_down(const int e) { return power_of_two(-min(max(e, -kMaxExponent), kMaxExponent)); }
__device__ __forceinline__ bool scale_fits(const int e) { return e >= -kMaxExponent && e <= kMaxExponent; }

__device__ __forceinline__ float largest(const f32x4 x) { return fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))); }

template<bool VEC>
__device__ __forceinline__ f32x4 load_chunk(const Buffer r, const uint32_t voffset, const uint32_t soffset) {
    if constexpr (VEC) return buffer_load4(r, voffset, soffset);
    else return f32x4{buffer_load(r, voffset, soffset), buffer_load(r, voffset + 4u, soffset), buffer_load(r, voffset + 8u, soffset),
            buffer_load(r, voffset + 12u, soffset)};
}

// Largest |x| and |y| over the workgroup's threads (each passes its own), by way of `slots`; contains a barrier.
template<int WAVES>
__device__ __forceinline__ void workgroup_largest(float &x, float &y, float (&slots)[2][WAVES]) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
        x = fmaxf(x, __shfl_xor(x, m));
        y = fmaxf(y, __shfl_xor(y, m));
    }
    const int wave = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        slots[0][wave] = x;
        slots[1][wave] = y;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        x = fmaxf(x, slots[0][w]);
        y = fmaxf(y, slots[1][w]);
    }
}

// The same over every live row of a window of n rows, for a scale that the sampled rows don't tell: they may all be 0 where the
// others are not (the gradient of one token's loss), and terms of a fixed scale would lose values far below it. A workgroup of
// THREADS threads reads ROWS rows at a time, CPR 4-float chunks each: live(row) says whether a row counts, load(row, on, a, b)
// fetches this thread's two chunks of it (zeros unless on). Returns how many of this thread's y chunks are not 0. Costs a pass
// over the window (from L2), taken only where all sampled rows are 0 or masked.
template<int THREADS, int CPR, class Live, class Load>
__device__ __forceinline__ int window_largest(float &x, float &y, const int n, const Live &live, const Load &load) {
    constexpr int ROWS = THREADS / CPR, TRIP = 4;
    int found = 0;
#pragma unroll 1
    for (int r0 = threadIdx.x / CPR; r0 - static_cast<int>(threadIdx.x / CPR) < n; r0 += TRIP * ROWS) {
        bool on[TRIP], any = false;
#pragma unroll
        for (int u = 0; u < TRIP; ++u) on[u] = live(r0 + u * ROWS);
#pragma unroll
        for (int u = 0; u < TRIP; ++u) {
            on[u] = on[u] && r0 + u * ROWS < n;
            any = any || on[u];
        }
        if (__ballot(any) == 0) continue;
        f32x4 a[TRIP], b[TRIP];
#pragma unroll
        for (int u = 0; u < TRIP; ++u) load(r0 + u * ROWS, on[u], a[u], b[u]);
#pragma unroll
        for (int u = 0; u < TRIP; ++u) {
            x = fmaxf(x, largest(a[u]));
            const float z = largest(b[u]);
            y = fmaxf(y, z);
            found += z > 0.0f;
        }
    }
    return found;
}

// Eight floats times `scale` as an operand's two terms.
__device__ __forceinline__ void split_operand(const f32x4 x, const f32x4 y, const float scale, h16x8 &high, h16x8 &low) {
    u32x4 hi, lo;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        uint32_t h, l;
        split_pair<true>(x[2 * j], x[2 * j + 1], scale, h, l);
        hi[j] = h;
        lo[j] = l;
        split_pair<true>(y[2 * j], y[2 * j + 1], scale, h, l);
        hi[2 + j] = h;
        lo[2 + j] = l;
    }
    high = __builtin_bit_cast(h16x8, hi);
    low = __builtin_bit_cast(h16x8, lo);
}

// Calls f(0), .., f(N - 1) with compile-time indexes.
template<int N, int I = 0, class F>
__device__ __forceinline__ void unrolled(const F &f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<N, I + 1>(f);
    }
}

// Transposing LDS read: lane L of each 16-lane group points at row L / 4 of four rows, elements 4 (L mod 4) .. + 3 of their
// sixteen, and receives element L of the four rows.
__device__ __forceinline__ u32x2 read_transposed(const uint16_t *p) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(p)));
}

// Position (in 2-byte elements) of element 0 of 16-byte chunk c of row r in a staged plane of D columns that is read both by
// rows (16 lanes: 16 rows, one chunk each) and transposed (32 lanes: 4 rows of 64 bytes). Rows are unpadded; their chunks are
// permuted so that either read meets every bank once: at D = 64 (8 chunks, two rows to the 64 banks) the even and the odd
// rows of 16 take all eight permutations, and rows r and r + 2 of four lie in different halves of their row.
template<int D>
__device__ __forceinline__ int staged_chunk(const int r, const int c) {
    const int swizzle = D == 64 ? ((r & 2) << 1 | (r & 4) >> 1 | (r & 8) >> 3) : ((r >> 2) & 3);
    return r * D + 8 * (c ^ swizzle);
}

} // namespace rk
