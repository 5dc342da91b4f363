// FP32 attention backward for gfx950 (MI355X) on the fp16 matrix cores, head width 32 or 64: the two deterministic kernels of
// attention_backward.hip (the reference's Attention.hip:32-189, Attention64.hip:34-191) with each FP32 product formed from
// three fp16 products of two-term operands (attention_split.hpp). No atomics, no workspace beyond the caller's delta.
//
//   1. attention_dq_split_kernel (query-major). A workgroup owns QB query tiles of 32 of one sequence, one per wave of a key
//      stream; KS key streams take alternate 64-key tiles. The QB waves of a stream load each K and V tile together, split it
//      once and stage its terms in LDS (double-buffered), as the forward does. Each wave: δ of its rows (written), then per 32
//      keys Sᵀ = K·Qᵀ, dPᵀ = V·dOᵀ, dSᵀ = Pᵀ(dPᵀ - δ) and dQᵀ += Kᵀ·dSᵀ (K's operand by transposing LDS reads, dSᵀ in place).
//   2. attention_dkdv_split_kernel (key-major). A workgroup owns KB key tiles of 32, one per wave of a query stream, K's and V's
//      terms in registers; the waves stage the terms of Q and dO tiles and per 32 queries S = Q·Kᵀ, dP = dO·Vᵀ, P, dS, then dVᵀ
//      += dOᵀ·P and dKᵀ += Qᵀ·dS (transposing reads; P and dS in place).
// Streams are summed through LDS in a fixed order, so results are bit-identical from run to run.
//
// Scales (powers of two): the operands a wave keeps in registers by their own largest magnitude (rows in kernel 1, the
// workgroup's block in kernel 2), the streamed ones by that of rows sampled over the workgroup's window, as in the forward
// (of all its rows where the sampled ones are 0). P is kept at 2^9 times exp(s - max) in kernel 1 (the row's 1/sum is applied
// to dQ at the end) and at 2^14 times its value in kernel 2; dS in units in which |dP - δ| of that size still fits fp16.
// Whatever leaves the range becomes NaN, and a wave whose gradients are not finite computes its tile again with FP32 MFMAs. So
// does one with a row or a key whose terms lost bits: the rows that set a scale may be hidden from it or have no weight, and a
// key may have small weights only. Kernel 1 tells from O and the row maximum, kernel 2 from Σ P² and Σ dS² of each key (the
// dot products of the high terms with themselves, 16 VALU instructions a tile: 2 to 4% of its time).
//
// What bounds them: 21 fp16 MFMAs of 32 x 32 x 16 per 32 x 32 tile and 16 columns of width in the two (12 and 9) do what 7 x 8 FP32
// ones of twice the time did, beside 16 exponentials and about 100 other VALU instructions per lane and kernel; at d = 64, 32 x
// 2048 causal, MFMAs take a third of the SIMD cycles, VALU issue a third, and waits a third of the wave cycles: with the terms
// of two operands and the accumulators in registers only two waves fit a SIMD. Measured, whole backward, back-to-back launches,
// against the deterministic FP32 pair (µs): d = 64, 32 x 2048 causal 510 -> 232, 96 x 2048 full 2640 -> 1067; d = 32, 24 x 1024
// full 103 -> 69, 96 x 2048 full 1353 -> 622; against the fused FP32 kernels 16 x 8192 causal, radius 256 257 -> 172, 24 x 1024
// causal at d = 32 54.6 -> 50.7. Errors against 64 bits fell too (dQ 3e-7, dK and dV 4e-7 to 6e-7 of the norm, FP32 pair 4e-7 to
// 1.1e-6, N(0,1) values): fp16 products are exact and their terms are summed 16 at a time.
#include <algorithm>

#include "attention_launch.hpp"
#include "attention_split.hpp"

namespace rk {

namespace {

constexpr int kStep = 2 * kTile; // keys of a step of kernel 1

struct SplitBackwardParams {
    Tensor q, k, v, o, u;
    const uint8_t *mask;
    const float *lse;
    float *dq, *dk, *dv, *delta;
    Shape s;
    float scale;
};

__device__ __forceinline__ const SplitBackwardParams &uniform_params(const SplitBackwardParams *params) {
    const auto address = reinterpret_cast<uint64_t>(params);
    const uint64_t uniform = static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(address >> 32))) << 32 |
            static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(address)));
    return *reinterpret_cast<const SplitBackwardParams *>(uniform);
}

// Sums acc over the workgroup's WAVES waves into wave 0 through `slots` (16 N floats a lane for each wave but one), in order.
template<int WAVES, int N>
__device__ __forceinline__ void sum_waves(f32x16 (&acc)[N], const int wave, const LdsFloats slots) {
    constexpr int SLOT = 16 * N * kWave;
    const int lane = threadIdx.x & (kWave - 1);
    __syncthreads(); // the slots' last use
    if (wave > 0) {
#pragma unroll
        for (int t = 0; t < N; ++t) {
#pragma unroll
            for (int j = 0; j < 16; ++j) slots[(wave - 1) * SLOT + (16 * t + j) * kWave + lane] = acc[t][j];
        }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll 1
        for (int w = 0; w < WAVES - 1; ++w) {
#pragma unroll
            for (int t = 0; t < N; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[t][j] += slots[w * SLOT + (16 * t + j) * kWave + lane];
            }
        }
    }
}

// dQ of one query tile on FP32 MFMAs by the workgroup's WAVES waves, for inputs that the split products cannot carry: operands
// straight from memory, alternate key tiles a wave.
template<int D, bool VEC, int WAVES>
__device__ __attribute__((noinline)) void exact_dq_tile(const SplitBackwardParams *params, const LdsFloats slots, const int seq_, const int q0_) {
    const SplitBackwardParams &P = uniform_params(params);
    const int seq = __builtin_amdgcn_readfirstlane(seq_), q0 = __builtin_amdgcn_readfirstlane(q0_);
    constexpr int HALF = D / 2, DT = D / 32;
    const Shape s = P.s;
    const int lane = threadIdx.x & (kWave - 1), col = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int query = q0 + col;
    const bool valid = query < s.queries;
    const int b = seq / s.heads, head = seq - b * s.heads;
    const Buffer qbuf = make_buffer(sequence(P.q, b, head), sequence_bytes(s.queries, P.q.st, D));
    const Buffer ubuf = make_buffer(sequence(P.u, b, head), sequence_bytes(s.queries, P.u.st, D));
    const Buffer kbuf = make_buffer(sequence(P.k, b, head), sequence_bytes(s.keys, P.k.st, D));
    const Buffer vbuf = make_buffer(sequence(P.v, b, head), sequence_bytes(s.keys, P.v.st, D));
    const Buffer mbuf = make_buffer(P.mask + static_cast<int64_t>(b) * s.keys, static_cast<uint32_t>(s.keys));
    const uint32_t kstep = 4u * P.k.st, vstep = 4u * P.v.st;
    const float c2 = P.scale * kLog2e;
    const int wlo = window_lo(s, query), whi = window_hi(s, query);
    int first, last;
    forward_key_range(s, q0 / kTile, first, last);
    const int64_t row = static_cast<int64_t>(seq) * s.queries + query;
    float qr[HALF], ur[HALF];
    buffer_load_span<VEC>(qr, qbuf, valid ? static_cast<uint32_t>(query) * (4u * P.q.st) + 4u * h * HALF : kNoRow);
    buffer_load_span<VEC>(ur, ubuf, valid ? static_cast<uint32_t>(query) * (4u * P.u.st) + 4u * h * HALF : kNoRow);
    const float m = valid ? P.lse[2 * row] : -INFINITY, l = valid ? P.lse[2 * row + 1] : 0.0f, dlt = valid ? P.delta[row] : 0.0f;
    const float mc = m != -INFINITY ? fmaf(m, kLog2e, __log2f(l)) : INFINITY;
    f32x16 acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = f32x16{};
#pragma unroll 1
    for (int key0 = first + wave * kTile; key0 < last; key0 += WAVES * kTile) {
        const uint32_t bits = static_cast<uint32_t>(__ballot(buffer_load_byte(mbuf, static_cast<uint32_t>(key0 + col)) != 0));
        if (bits == 0) continue;
        float kr[HALF], vr[HALF];
        buffer_load_span<VEC>(kr, kbuf, static_cast<uint32_t>(key0 + col) * kstep + 4u * h * HALF);
        buffer_load_span<VEC>(vr, vbuf, static_cast<uint32_t>(key0 + col) * vstep + 4u * h * HALF);
        f32x16 sc{}, dp{};
#pragma unroll
        for (int c = 0; c < HALF; ++c) sc = mfma(kr[c], qr[c], sc);
        __builtin_amdgcn_sched_barrier(0); // what follows takes the registers of K's rows
#pragma unroll
        for (int c = 0; c < HALF; ++c) dp = mfma(vr[c], ur[c], dp);
        float kc[16 * DT];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int r = tile_row(j, h);
            const uint32_t at = (bits >> r) & 1u ? static_cast<uint32_t>(key0 + r) * kstep + 4u * col : kNoRow;
#pragma unroll
            for (int t = 0; t < DT; ++t) kc[j * DT + t] = buffer_load(kbuf, at + 128u * t, 0);
        }
        const uint32_t visible = (bits & bit_range(wlo - key0, whi - key0)) >> (4 * h);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float p = exp2_fast(fmaf(sc[j], c2, -mc));
            sc[j] = (visible >> (8 * (j >> 2) + (j & 3))) & 1u ? p * (dp[j] - dlt) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
#pragma unroll
            for (int t = 0; t < DT; ++t) acc[t] = mfma(kc[j * DT + t], sc[j], acc[t]);
        }
    }
    sum_waves<WAVES, DT>(acc, wave, slots);
    if (wave > 0 || !valid) return;
#pragma unroll
    for (int t = 0; t < DT; ++t) store_tile_row<VEC>(P.dq + row * D + 32 * t, acc[t], P.scale, h);
}

// dK and dV of one key tile on FP32 MFMAs by the workgroup's WAVES waves, alternate query tiles a wave.
template<int D, bool VEC, int WAVES>
__device__ __attribute__((noinline)) void exact_dkdv_tile(const SplitBackwardParams *params, const LdsFloats slots, const int seq_, const int kt_) {
    const SplitBackwardParams &P = uniform_params(params);
    const int seq = __builtin_amdgcn_readfirstlane(seq_), kt = __builtin_amdgcn_readfirstlane(kt_);
    constexpr int HALF = D / 2, DT = D / 32;
    const Shape s = P.s;
    const int lane = threadIdx.x & (kWave - 1), col = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int key = kt * kTile + col;
    const int b = seq / s.heads, head = seq - b * s.heads;
    const Buffer qbuf = make_buffer(sequence(P.q, b, head), sequence_bytes(s.queries, P.q.st, D));
    const Buffer ubuf = make_buffer(sequence(P.u, b, head), sequence_bytes(s.queries, P.u.st, D));
    const Buffer kbuf = make_buffer(sequence(P.k, b, head), sequence_bytes(s.keys, P.k.st, D));
    const Buffer vbuf = make_buffer(sequence(P.v, b, head), sequence_bytes(s.keys, P.v.st, D));
    const Buffer mbuf = make_buffer(P.mask + static_cast<int64_t>(b) * s.keys, static_cast<uint32_t>(s.keys));
    const Buffer lbuf = make_buffer(P.lse + static_cast<int64_t>(seq) * s.queries * 2, static_cast<uint32_t>(s.queries) * 8u);
    const Buffer dbuf = make_buffer(P.delta + static_cast<int64_t>(seq) * s.queries, static_cast<uint32_t>(s.queries) * 4u);
    const uint32_t qstep = 4u * P.q.st, ustep = 4u * P.u.st;
    const float c2 = P.scale * kLog2e;
    const bool visible = key < s.keys && buffer_load_byte(mbuf, static_cast<uint32_t>(key)) != 0;
    float kr[HALF], vr[HALF];
    buffer_load_span<VEC>(kr, kbuf, visible ? static_cast<uint32_t>(key) * (4u * P.k.st) + 4u * h * HALF : kNoRow);
    buffer_load_span<VEC>(vr, vbuf, visible ? static_cast<uint32_t>(key) * (4u * P.v.st) + 4u * h * HALF : kNoRow);
    int first, last;
    dkdv_query_range(s, kt, first, last);
    const int qlo = window_query_lo(s, key), qhi = min(window_query_hi(s, key), last - 1);
    f32x16 acc_k[DT], acc_v[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc_k[t] = acc_v[t] = f32x16{};
#pragma unroll 1
    for (int q0 = first + wave * kTile; q0 < last; q0 += WAVES * kTile) {
        float qr[HALF], ur[HALF];
        buffer_load_span<VEC>(qr, qbuf, static_cast<uint32_t>(q0 + col) * qstep + 4u * h * HALF);
        buffer_load_span<VEC>(ur, ubuf, static_cast<uint32_t>(q0 + col) * ustep + 4u * h * HALF);
        const float rm = buffer_load(lbuf, static_cast<uint32_t>(q0 + col) * 8u, 0), rl = buffer_load(lbuf, static_cast<uint32_t>(q0 + col) * 8u + 4u, 0);
        const float delta = buffer_load(dbuf, static_cast<uint32_t>(q0 + col) * 4u, 0); // of row col
        f32x16 sc{}, dp{};
#pragma unroll
        for (int c = 0; c < HALF; ++c) sc = mfma(qr[c], kr[c], sc);
        const float offset = rm != -INFINITY ? fmaf(rm, kLog2e, __log2f(rl)) : INFINITY;
#pragma unroll
        for (int c = 0; c < HALF; ++c) dp = mfma(ur[c], vr[c], dp);
        const uint32_t keep = visible ? bit_range(qlo - q0, qhi - q0) >> (4 * h) : 0u;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float to = __shfl(offset, tile_row(j, h)), d = __shfl(delta, tile_row(j, h));
            const bool ok = ((keep >> (8 * (j >> 2) + (j & 3))) & 1u) && to != INFINITY;
            const float p = ok ? exp2_fast(fmaf(sc[j], c2, -to)) : 0.0f;
            sc[j] = p;
            dp[j] = ok ? p * (dp[j] - d) : 0.0f;
        }
#pragma unroll
        for (int part = 0; part < 2; ++part) { // the columns of 8 rows a half-wave at a time: registers hold no more at D = 64
            __builtin_amdgcn_sched_barrier(0);
            float uc[8 * DT], qc[8 * DT];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t qq = static_cast<uint32_t>(q0 + tile_row(8 * part + j, h));
#pragma unroll
                for (int t = 0; t < DT; ++t) {
                    uc[j * DT + t] = buffer_load(ubuf, qq * ustep + 4u * (32 * t + col), 0);
                    qc[j * DT + t] = buffer_load(qbuf, qq * qstep + 4u * (32 * t + col), 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
#pragma unroll
                for (int t = 0; t < DT; ++t) {
                    acc_v[t] = mfma(uc[j * DT + t], sc[8 * part + j], acc_v[t]);
                    acc_k[t] = mfma(qc[j * DT + t], dp[8 * part + j], acc_k[t]);
                }
            }
        }
    }
    sum_waves<WAVES, DT>(acc_k, wave, slots);
    sum_waves<WAVES, DT>(acc_v, wave, slots);
    if (wave > 0 || key >= s.keys) return;
    const int64_t krow = (static_cast<int64_t>(seq) * s.keys + key) * D;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        store_tile_row<VEC>(P.dk + krow + 32 * t, acc_k[t], P.scale, h);
        store_tile_row<VEC>(P.dv + krow + 32 * t, acc_v[t], 1.0f, h);
    }
}

// Row and transposed operand reads of a staged 32-row tile (two planes of D columns, PLANE elements apart).
template<int D, int PLANE>
struct StagedReads {
    int row[D / 16], tr[D / 32][2];
    __device__ __forceinline__ StagedReads() {
        const int lane = threadIdx.x & (kWave - 1), col = lane & 31, h = lane >> 5;
#pragma unroll
        for (int i = 0; i < D / 16; ++i) row[i] = staged_chunk<D>(col, 2 * i + h);
        // Rows r0 .. r0 + 3 with r0 = 16u + 8p + 4h, features 32 t2 + 16 (col / 16) .. + 15.
#pragma unroll
        for (int t2 = 0; t2 < D / 32; ++t2) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
                tr[t2][p] = staged_chunk<D>(8 * p + 4 * h + ((lane & 15) >> 2), 4 * t2 + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + 4 * (lane & 1);
        }
    }
    // Features 16i + 8h .. + 7 of the lane's row, i = 0 .. D/16 - 1.
    __device__ __forceinline__ void rows(h16x8 (&x)[D / 16], const uint16_t *tile, const int term) const {
#pragma unroll
        for (int i = 0; i < D / 16; ++i) x[i] = *reinterpret_cast<const h16x8 *>(tile + term * PLANE + row[i]);
    }
    // Rows tile_row(8u + j, h), j = 0 .. 7, of features 32 t2 + col.
    __device__ __forceinline__ void columns(h16x8 (&x)[D / 32], const uint16_t *tile, const int u, const int term) const {
#pragma unroll
        for (int t2 = 0; t2 < D / 32; ++t2) {
            const uint16_t *const at = tile + term * PLANE + 16 * u * D;
            const u32x2 lo = read_transposed(at + tr[t2][0]), hi = read_transposed(at + tr[t2][1]);
            x[t2] = __builtin_bit_cast(h16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
        }
    }
};

// MFMA M of the 3·D/16 of a row product: A low with B high, A high with B low, A high with B high.
template<int M, int KC>
__device__ __forceinline__ void row_mfma(f32x16 &acc, const h16x8 (&low)[KC], const h16x8 (&high)[KC], const h16x8 (&bh)[KC], const h16x8 (&bl)[KC]) {
    acc = mfma_f16(M < KC ? low[M % KC] : high[M % KC], M < KC || M >= 2 * KC ? bh[M % KC] : bl[M % KC], acc);
}

// MFMAs M (of 6, D/32 each) of a column product: for each half of the tile's rows the same three.
template<int M, int DT>
__device__ __forceinline__ void column_mfma(f32x16 (&acc)[DT], const h16x8 (&low)[DT], const h16x8 (&high)[DT], const uint32_t (&b)[2][8]) {
    constexpr int U = M / 3, Y = M % 3 == 1;
    const h16x8 x = __builtin_bit_cast(h16x8, u32x4{b[Y][4 * U], b[Y][4 * U + 1], b[Y][4 * U + 2], b[Y][4 * U + 3]});
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = mfma_f16(M % 3 == 0 ? low[t] : high[t], x, acc[t]);
}

// Splits pair E (of 2) of a chunk's four floats; the second writes the chunk's terms to `at`.
template<int E, int PLANE>
__device__ __forceinline__ void stage_pair(const f32x4 x, const float factor, u32x2 (&terms)[2], uint16_t *at) {
    uint32_t y, z;
    split_pair<true>(x[2 * E], x[2 * E + 1], factor, y, z);
    terms[0][E] = y;
    terms[1][E] = z;
    if constexpr (E == 1) {
        *reinterpret_cast<u32x2 *>(at) = terms[0];
        *reinterpret_cast<u32x2 *>(at + PLANE) = terms[1];
    }
}

// acc += A·B over D features: A's rows from a staged tile, B's terms in registers; the small products first.
template<int D, int PLANE>
__device__ __forceinline__ void row_product(f32x16 &acc, const StagedReads<D, PLANE> &reads, const uint16_t *tile, const h16x8 (&bh)[D / 16],
        const h16x8 (&bl)[D / 16]) {
    h16x8 low[D / 16], high[D / 16];
    reads.rows(low, tile, 1);
    reads.rows(high, tile, 0);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) acc = mfma_f16(low[i], bh[i], acc);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) acc = mfma_f16(high[i], bl[i], acc);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) acc = mfma_f16(high[i], bh[i], acc);
}

// acc += Aᵀ·B over a tile's 32 rows: A by transposing reads, B's terms packed in the accumulator layout.
template<int D, int PLANE>
__device__ __forceinline__ void column_product(f32x16 (&acc)[D / 32], const StagedReads<D, PLANE> &reads, const uint16_t *tile,
        const uint32_t (&b)[2][8]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        h16x8 low[D / 32], high[D / 32];
        reads.columns(low, tile, u, 1);
        reads.columns(high, tile, u, 0);
        const h16x8 bh = __builtin_bit_cast(h16x8, u32x4{b[0][4 * u], b[0][4 * u + 1], b[0][4 * u + 2], b[0][4 * u + 3]});
        const h16x8 bl = __builtin_bit_cast(h16x8, u32x4{b[1][4 * u], b[1][4 * u + 1], b[1][4 * u + 2], b[1][4 * u + 3]});
#pragma unroll
        for (int t = 0; t < D / 32; ++t) acc[t] = mfma_f16(low[t], bh, acc[t]);
#pragma unroll
        for (int t = 0; t < D / 32; ++t) acc[t] = mfma_f16(high[t], bl, acc[t]);
#pragma unroll
        for (int t = 0; t < D / 32; ++t) acc[t] = mfma_f16(high[t], bh, acc[t]);
    }
}

// Sums acc over the streams of a workgroup into stream 0 (fixed order); `slot` is this wave's tile slot of stream 1.
template<int N, int STREAMS>
__device__ __forceinline__ void sum_streams(f32x16 (&acc)[N], const int stream, float *slot, const int stride) {
    if constexpr (STREAMS > 1) {
        __syncthreads(); // every wave is done with this memory
        if (stream > 0) {
            float *const mine = slot + (stream - 1) * stride;
#pragma unroll
            for (int t = 0; t < N; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) mine[(16 * t + j) * kWave] = acc[t][j];
            }
        }
        __syncthreads();
        if (stream == 0) {
#pragma unroll
            for (int x = 0; x < STREAMS - 1; ++x) {
#pragma unroll
                for (int t = 0; t < N; ++t) {
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc[t][j] += slot[x * stride + (16 * t + j) * kWave];
                }
            }
        }
    }
}

template<int N>
__device__ __forceinline__ float largest(const f32x16 (&acc)[N]) {
    float x = 0.0f;
#pragma unroll
    for (int t = 0; t < N; ++t) {
#pragma unroll
        for (int j = 0; j < 16; ++j) x = fmaxf(x, fabsf(acc[t][j]));
    }
    return x;
}

// sum + x² + y² of a packed pair.
__device__ __forceinline__ float add_squares(const uint32_t pair, const float sum) {
    const h16x2 x = __builtin_bit_cast(h16x2, pair);
    return __builtin_amdgcn_fdot2(x, x, sum, false);
}

template<int N>
__device__ __forceinline__ bool finite(const f32x16 (&acc)[N]) {
    float probe = 0.0f;
#pragma unroll
    for (int t = 0; t < N; ++t) {
#pragma unroll
        for (int j = 0; j < 16; ++j) probe = fmaf(acc[t][j], 0.0f, probe);
    }
    return __ballot(probe != 0.0f) == 0;
}

} // namespace

// Two waves per SIMD (256 registers): Q's and dO's terms stay in registers (D of them), a step covers two 32-key halves so that
// each group of MFMAs has another half's VALU work beside it (d = 64, 32 x 2048 causal: 90 µs; one half per step 118).
template<int D, bool VEC, int QB, int KS>
__global__ __launch_bounds__(kWave * QB * KS) __attribute__((amdgpu_waves_per_eu(2))) void attention_dq_split_kernel(const SplitBackwardParams P) {
    constexpr int KC = D / 16, DT = D / 32, CPR = D / 4;
    constexpr int CH = kStep * CPR / (kWave * QB);   // chunks per lane of a K tile, and of a V tile
    constexpr int PLANE = kStep * D;                 // elements of one term of one tile
    constexpr int STAGE = 4 * PLANE;                 // K's two terms, high and low, then V's
    constexpr int RPC = kWave * QB / CPR;
    constexpr int STAGE_BYTES = 2 * KS * STAGE * 2, MERGE_BYTES = (KS - 1) * QB * 16 * DT * kWave * 4;
    __shared__ __align__(16) unsigned char smem[STAGE_BYTES > MERGE_BYTES ? STAGE_BYTES : MERGE_BYTES];
    static_assert((QB * KS - 1) * 16 * DT * kWave * 4 <= STAGE_BYTES); // the slots of exact_dq_tile
    __shared__ float amax[2][QB * KS];
    __shared__ int redone[QB]; // query tiles to compute again
    __shared__ float norms[KS > 1 ? KS - 1 : 1][QB][kWave]; // of streams 1 ..: Σ dS'² of each lane

    const Shape &s = P.s;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int qi = wave % QB, stream = wave / QB;
    const int col = lane & 31, h = lane >> 5;
    const float one = split_unit_scale();
    const int seqs = s.batch * s.heads;
    const int seq = static_cast<int>(blockIdx.x) % seqs, rank = static_cast<int>(blockIdx.x) / seqs; // as in the forward
    const int b = seq / s.heads, head = seq - b * s.heads;
    const int nblocks = (s.queries + QB * kTile - 1) / (QB * kTile);
    const int qb = s.causal ? nblocks - 1 - rank : rank;
    const int q0 = (qb * QB + qi) * kTile, query = q0 + col;
    const bool tile_valid = q0 < s.queries, valid = query < s.queries;
    const int64_t row = static_cast<int64_t>(seq) * s.queries + query;

    const Buffer qbuf = make_buffer(sequence(P.q, b, head), sequence_bytes(s.queries, P.q.st, D));
    const Buffer obuf = make_buffer(sequence(P.o, b, head), sequence_bytes(s.queries, P.o.st, D));
    const Buffer ubuf = make_buffer(sequence(P.u, b, head), sequence_bytes(s.queries, P.u.st, D));
    const Buffer kbuf = make_buffer(sequence(P.k, b, head), sequence_bytes(s.keys, P.k.st, D));
    const Buffer vbuf = make_buffer(sequence(P.v, b, head), sequence_bytes(s.keys, P.v.st, D));
    const Buffer mbuf = make_buffer(P.mask + static_cast<int64_t>(b) * s.keys, static_cast<uint32_t>(s.keys));
    const uint32_t kstep = 4u * P.k.st, vstep = 4u * P.v.st;

    int first, last, ufirst, ulast, unused;
    forward_key_range(s, q0 / kTile, first, last);
    forward_key_range(s, qb * QB, ufirst, unused);
    forward_key_range(s, min(qb * QB + QB - 1, (s.queries - 1) / kTile), unused, ulast);
    const int ntiles = ulast > ufirst ? (ulast - ufirst + kStep - 1) / kStep : 0;
    const int nsteps = (ntiles + KS - 1) / KS; // tile of stream x at step i: i·KS + x
    const int wlo = window_lo(s, query), whi = window_hi(s, query);

    // This lane's chunks of a tile: chunk i is row crow + RPC·i, 4 floats from column 4 (lane mod CPR).
    const int crow = (qi * kWave + lane) / CPR;
    const uint32_t kofs = static_cast<uint32_t>(crow) * kstep + 16u * static_cast<uint32_t>(lane % CPR);
    const uint32_t vofs = static_cast<uint32_t>(crow) * vstep + 16u * static_cast<uint32_t>(lane % CPR);
    int write[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) write[i] = staged_chunk<D>(crow + RPC * i, (lane % CPR) >> 1) + 4 * (lane & 1);
    const StagedReads<D, PLANE> reads;
    uint16_t *const stages = reinterpret_cast<uint16_t *>(smem) + stream * (2 * STAGE);

    f32x4 kraw[CH], vraw[CH];
    auto tile_key = [&](const int i) { return ufirst + (i * KS + stream) * kStep; };
    auto load_mask = [&](const int i) __attribute__((always_inline)) {
        return buffer_load_byte_s(mbuf, static_cast<uint32_t>(lane), i * KS + stream < ntiles ? static_cast<uint32_t>(tile_key(i)) : kNoRow);
    };
    auto load_tile = [&](const int i) __attribute__((always_inline)) {
        const bool live = i * KS + stream < ntiles;
        const uint32_t k0 = live ? static_cast<uint32_t>(tile_key(i)) * kstep : kNoRow, v0 = live ? static_cast<uint32_t>(tile_key(i)) * vstep : kNoRow;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            kraw[c] = load_chunk<VEC>(kbuf, kofs, k0 + static_cast<uint32_t>(RPC * c) * kstep);
            vraw[c] = load_chunk<VEC>(vbuf, vofs, v0 + static_cast<uint32_t>(RPC * c) * vstep);
        }
    };

    // Requests, in the order they are waited for: sampled rows (for the scales), dO, O and Q rows, the first tile.
    constexpr int ROWS = kWave * QB * KS / CPR;
    const int n = min(ulast, s.keys) - ufirst;
    const int sampled = ufirst + (n > 0 ? static_cast<int>(static_cast<int64_t>(static_cast<int>(threadIdx.x) / CPR) * n / ROWS) : 0);
    const int seen = buffer_load_byte(mbuf, static_cast<uint32_t>(sampled));
    const f32x4 sk = load_chunk<VEC>(kbuf, static_cast<uint32_t>(sampled) * kstep + 16u * (threadIdx.x % CPR), 0);
    const f32x4 sv = load_chunk<VEC>(vbuf, static_cast<uint32_t>(sampled) * vstep + 16u * (threadIdx.x % CPR), 0);
    f32x4 qraw[2 * KC], uraw[2 * KC], oraw[2 * KC];
#pragma unroll
    for (int i = 0; i < 2 * KC; ++i) {
        const uint32_t f = 4u * (16 * (i / 2) + 8 * h + 4 * (i % 2)), r = static_cast<uint32_t>(query);
        uraw[i] = load_chunk<VEC>(ubuf, valid ? r * (4u * P.u.st) + f : kNoRow, 0);
        oraw[i] = load_chunk<VEC>(obuf, valid ? r * (4u * P.o.st) + f : kNoRow, 0);
        qraw[i] = load_chunk<VEC>(qbuf, valid ? r * (4u * P.q.st) + f : kNoRow, 0);
    }
    const float m = valid ? P.lse[2 * row] : -INFINITY, l = valid ? P.lse[2 * row + 1] : 0.0f;
    load_tile(0);
    const int mask0 = load_mask(0);

    float mk = seen != 0 ? largest(sk) : 0.0f, mv = seen != 0 ? largest(sv) : 0.0f;
    workgroup_largest(mk, mv, amax);
    if (n > ROWS && __builtin_amdgcn_readfirstlane(mk == 0.0f || mv == 0.0f)) {
        window_largest<kWave * QB * KS, CPR>(mk, mv, n, [&](const int r) { return buffer_load_byte(mbuf, static_cast<uint32_t>(ufirst + r)) != 0; },
                [&](const int r, const bool on, f32x4 &x, f32x4 &y) {
                    const uint32_t at = 16u * (threadIdx.x % CPR), row = static_cast<uint32_t>(ufirst + r);
                    x = load_chunk<VEC>(kbuf, on ? row * kstep + at : kNoRow, 0);
                    y = load_chunk<VEC>(vbuf, on ? row * vstep + at : kNoRow, 0);
                });
        __syncthreads(); // amax is read
        workgroup_largest(mk, mv, amax);
    }
    const int ek = __builtin_amdgcn_readfirstlane(exponent_of(mk)) - 8; // K = K'·2^ek, V = V'·2^ev, sampled largest at 2^8
    const int ev = __builtin_amdgcn_readfirstlane(exponent_of(mv)) - 8;
    const bool k_zero = __builtin_amdgcn_readfirstlane(mk == 0.0f), v_zero = __builtin_amdgcn_readfirstlane(mv == 0.0f);

    // δ in the order every backward path sums it (group_dot, pairwise tree): this lane holds groups 4i + 2h and 4i + 2h + 1.
    float dlt;
    {
        float part[KC];
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const float x[8] = {uraw[2 * i][0], uraw[2 * i][1], uraw[2 * i][2], uraw[2 * i][3], uraw[2 * i + 1][0], uraw[2 * i + 1][1], uraw[2 * i + 1][2], uraw[2 * i + 1][3]};
            const float y[8] = {oraw[2 * i][0], oraw[2 * i][1], oraw[2 * i][2], oraw[2 * i][3], oraw[2 * i + 1][0], oraw[2 * i + 1][1], oraw[2 * i + 1][2], oraw[2 * i + 1][3]};
            part[i] = halves_sum(group_dot(x, y) + group_dot(x + 4, y + 4));
        }
        dlt = group_tree(part);
        if (stream == 0 && h == 0 && valid) P.delta[row] = dlt;
    }
    float mq = 0.0f, mu = 0.0f, mo = 0.0f;
#pragma unroll
    for (int i = 0; i < 2 * KC; ++i) {
        mq = fmaxf(mq, largest(qraw[i]));
        mu = fmaxf(mu, largest(uraw[i]));
        mo = fmaxf(mo, largest(oraw[i]));
    }
    mq = halves_max(mq);
    mu = halves_max(mu);
    mo = halves_max(mo);
    const int eq = exponent_of(mq) - 14, eu = exponent_of(mu) - 14;
    // Rows that only use rows far below the ones that set the scales (hidden from them, or of no weight), whose terms are off by 2^-25
    // in V' and K'. Of V': the row's weighted mean, which O is, must reach 2^-3/√l. Of K': scores must not move, as in the
    // forward (both: see there); what K' loses in dQ' itself shows at the end. Rows of dO = 0 have no gradient to lose.
    const float c2 = __builtin_amdgcn_ldexpf(P.scale * kLog2e, eq + ek);
    const bool faint = valid && m != -INFINITY && mu > 0.0f && ((!v_zero && mo * sqrtf(l) < __builtin_amdgcn_ldexpf(1.0f, ev - 3)) ||
            (c2 > 0x1p-16f && fabsf(m) < __builtin_amdgcn_ldexpf(P.scale, eq + ek + 16)));
    // Outside the range of scales: for K and V the whole workgroup keeps from the loop; for a wave's own queries only its
    // products do, as its siblings need the rows that it stages and its barriers.
    const bool unfit = !scale_fits(ek) || !scale_fits(ev), own_unfit = __ballot(!scale_fits(eq) || !scale_fits(eu) || faint) != 0;
    const float kfactor = scale_down(ek), vfactor = scale_down(ev);
    h16x8 qh[KC], ql[KC], uh[KC], ul[KC];
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        split_operand(qraw[2 * i], qraw[2 * i + 1], scale_down(eq), qh[i], ql[i]);
        split_operand(uraw[2 * i], uraw[2 * i + 1], scale_down(eu), uh[i], ul[i]);
    }
    // P̃ = 2^9·exp(s - max) = exp2(S'·c2 + base); dP - δ in units of 2^(eu + ev + 23), twice the product of the largest |dO| of
    // the row and the largest sampled |V|: r = dP'·2^-23 - δ'. P̃·r then stays below 2^16 while |r| < 2^7.
    const float base = m != -INFINITY ? fmaf(m, -kLog2e, 9.0f) : -INFINITY;
    const float dl = __builtin_amdgcn_ldexpf(dlt, -(eu + ev + 23));
    constexpr float kUnit = 1.0f / (1 << 23);

    f32x16 acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = f32x16{};
    float ds_norm = 0.0f; // Σ dS'² of the lane's query over its half of the keys, from the high terms

    auto clear_masked = [&](const uint64_t bits) __attribute__((always_inline)) {
        if (__builtin_expect(bits != ~0ull, 0)) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int keep = -static_cast<int>((bits >> (crow + RPC * c)) & 1u);
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    __asm__("v_and_b32 %0, %1, %0" : "+v"(kraw[c][x]) : "v"(keep)); // in place
                    __asm__("v_and_b32 %0, %1, %0" : "+v"(vraw[c][x]) : "v"(keep));
                }
            }
        }
    };
    // Staging of the rows in flight into stage p, in units of a pair of floats: 2·CH of K and as many of V.
    u32x2 terms[2];
    auto stage_unit = [&](auto unit, auto of_v, const int p) __attribute__((always_inline)) {
        constexpr int C = decltype(unit)::value / 2, E = decltype(unit)::value % 2;
        constexpr bool V = decltype(of_v)::value;
        stage_pair<E, PLANE>(V ? vraw[C] : kraw[C], V ? vfactor : kfactor, terms, stages + p * STAGE + (V ? 2 * PLANE : 0) + write[C]);
    };
    constexpr std::integral_constant<bool, false> kOfK{};
    constexpr std::integral_constant<bool, true> kOfV{};
    auto stage = [&](const int p) __attribute__((always_inline)) {
        unrolled<2 * CH>([&](auto u) __attribute__((always_inline)) { stage_unit(u, kOfK, p); });
        unrolled<2 * CH>([&](auto u) __attribute__((always_inline)) { stage_unit(u, kOfV, p); });
    };
    // Scores 2u, 2u + 1 to P̃; then, with dP, to the terms of dS.
    auto exp_unit = [&](auto unit, f32x16 &sc) __attribute__((always_inline)) {
        constexpr int J = 2 * decltype(unit)::value;
        sc[J] = exp2_fast(fmaf(sc[J], c2, base));
        sc[J + 1] = exp2_fast(fmaf(sc[J + 1], c2, base));
    };
    auto ds_unit = [&](auto unit, const f32x16 &sc, const f32x16 &dp, uint32_t (&ds)[2][8]) __attribute__((always_inline)) {
        constexpr int U = decltype(unit)::value, J = 2 * U;
        split_pair<false>(sc[J] * fmaf(dp[J], kUnit, -dl), sc[J + 1] * fmaf(dp[J + 1], kUnit, -dl), one, ds[0][U], ds[1][U]);
        ds_norm = add_squares(ds[0][U], ds_norm);
        __asm__ volatile("" : "+v"(ds[1][U]), "+v"(ds_norm)); // here, not at its use behind the next group
    };
    // A whole 64-key tile without masks, halves A and B, and the staging of the next one: six groups of MFMAs, each beside
    // independent VALU work spread over it (as in the forward): Sᵀ of A with the staging of K, dPᵀ of A with A's exponentials,
    // Sᵀ of B with A's dS, dPᵀ of B with B's exponentials, dQᵀ of A with B's dS, dQᵀ of B with the staging of V.
    auto full_step = [&](const int p) __attribute__((always_inline)) {
        constexpr int NS = 3 * KC, LEAD = 2;
        const uint16_t *const ka = stages + p * STAGE, *const kb2 = ka + kTile * D, *const va = ka + 2 * PLANE, *const vb = va + kTile * D;
        h16x8 low[KC], high[KC], cl[DT], ch[DT];
        f32x16 sa{}, sb{}, da{}, db{};
        uint32_t dsa[2][8], dsb[2][8];
        reads.rows(low, ka, 1);
        reads.rows(high, ka, 0);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<NS>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M * 2 * CH / NS, U1 = (M + 1) * 2 * CH / NS;
            row_mfma<M, KC>(sa, low, high, qh, ql);
            if constexpr (M == KC) reads.rows(low, va, 1);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) { stage_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, kOfK, p ^ 1); });
            __builtin_amdgcn_sched_barrier(0);
        });
        reads.rows(high, va, 0);
        // N units over the MFMAs from LEAD on.
        unrolled<NS>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M < LEAD ? 0 : (M - LEAD) * 8 / (NS - LEAD), U1 = M < LEAD ? 0 : (M + 1 - LEAD) * 8 / (NS - LEAD);
            row_mfma<M, KC>(da, low, high, uh, ul);
            if constexpr (M == KC) reads.rows(low, kb2, 1);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) { exp_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, sa); });
            __builtin_amdgcn_sched_barrier(0);
        });
        reads.rows(high, kb2, 0);
        unrolled<NS>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M < LEAD ? 0 : (M - LEAD) * 8 / (NS - LEAD), U1 = M < LEAD ? 0 : (M + 1 - LEAD) * 8 / (NS - LEAD);
            row_mfma<M, KC>(sb, low, high, qh, ql);
            if constexpr (M == KC) reads.rows(low, vb, 1);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) { ds_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, sa, da, dsa); });
            __builtin_amdgcn_sched_barrier(0);
        });
        reads.rows(high, vb, 0);
        unrolled<NS>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M < LEAD ? 0 : (M - LEAD) * 8 / (NS - LEAD), U1 = M < LEAD ? 0 : (M + 1 - LEAD) * 8 / (NS - LEAD);
            row_mfma<M, KC>(db, low, high, uh, ul);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) { exp_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, sb); });
            if constexpr (M == NS - 2) reads.columns(cl, ka, 0, 1);
            if constexpr (M == NS - 1) reads.columns(ch, ka, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
        unrolled<6>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M * 8 / 6, U1 = (M + 1) * 8 / 6;
            column_mfma<M, DT>(acc, cl, ch, dsa);
            if constexpr (M % 3 == 0) reads.columns(cl, M == 0 ? ka : kb2, 1 - M / 3, 1); // (A, 1), then (B, 0)
            if constexpr (M % 3 == 2) reads.columns(ch, M == 2 ? ka : kb2, 1 - M / 3, 0);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) { ds_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, sb, db, dsb); });
            __builtin_amdgcn_sched_barrier(0);
        });
        unrolled<6>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M * 2 * CH / 6, U1 = (M + 1) * 2 * CH / 6;
            column_mfma<M, DT>(acc, cl, ch, dsb);
            if constexpr (M == 0) reads.columns(cl, kb2, 1, 1);
            if constexpr (M == 2) reads.columns(ch, kb2, 1, 0);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) { stage_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, kOfV, p ^ 1); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // Half x (32 keys) of the tile in stage p, masked.
    auto half_step = [&](const int p, const int x, const int key0, const uint32_t bits) __attribute__((always_inline)) {
        const uint16_t *const kt = stages + p * STAGE + x * kTile * D;
        f32x16 sc{}, dp{};
        row_product<D, PLANE>(sc, reads, kt, qh, ql);
        row_product<D, PLANE>(dp, reads, kt + 2 * PLANE, uh, ul);
        const uint32_t visible = (bits & bit_range(wlo - key0, whi - key0)) >> (4 * h);
#pragma unroll
        for (int j = 0; j < 16; ++j) sc[j] = (visible >> (8 * (j >> 2) + (j & 3))) & 1u ? sc[j] : -INFINITY;
        uint32_t ds[2][8];
        unrolled<8>([&](auto u) __attribute__((always_inline)) {
            exp_unit(u, sc);
            ds_unit(u, sc, dp, ds);
        });
        column_product<D, PLANE>(acc, reads, kt, ds);
    };

    if (nsteps > 0 && !unfit) {
        uint64_t bits0 = __ballot(mask0 != 0);
        clear_masked(bits0);
        stage(0);
        load_tile(1);
        int mbyte = load_mask(1);
        auto step = [&](const int i, const int p) __attribute__((always_inline)) {
            __syncthreads(); // tile i is staged; every wave is done with the other stage
            const int key0 = tile_key(i);
            const bool live = i * KS + stream < ntiles && tile_valid && !own_unfit;
            const bool inside = live && bits0 == ~0ull && key0 >= first && key0 + kStep <= last && tile_in_window(s, q0, key0) &&
                    tile_in_window(s, q0, key0 + kTile);
            const uint64_t bits1 = __ballot(mbyte != 0);
            clear_masked(bits1);
            if (__builtin_expect(inside, 1)) {
                full_step(p);
            } else {
#pragma unroll 1
                for (int x = 0; x < 2; ++x) {
                    const int k0 = key0 + x * kTile;
                    const uint32_t bits = static_cast<uint32_t>(bits0 >> (32 * x));
                    if (live && bits != 0 && k0 < last && k0 + kTile > first) half_step(p, x, k0, bits);
                }
                stage(p ^ 1);
            }
            load_tile(i + 2);
            mbyte = load_mask(i + 2);
            bits0 = bits1;
        };
        for (int i = 0; i < nsteps; i += 2) {
            step(i, 0);
            if (i + 1 < nsteps) step(i + 1, 1);
        }
    }
    if (KS > 1 && stream > 0) norms[stream - 1][qi][lane] = ds_norm;
    sum_streams<DT, KS>(acc, stream, reinterpret_cast<float *>(smem) + qi * (16 * DT * kWave) + lane, QB * 16 * DT * kWave);
    bool redo = false;
    if (stream == 0 && tile_valid) {
#pragma unroll
        for (int x = 0; x < KS - 1; ++x) ds_norm += norms[x][qi][lane];
        // dQ' is off by 2^-25·√(Σ dS'²) from K', below 2^-21 of the largest |dQ'| if that reaches 2^-4·√(Σ dS'²).
        const float top = halves_max(largest(acc));
        const bool faint_k = valid && !k_zero && 256.0f * top * top < halves_sum(ds_norm);
        redo = unfit || own_unfit || __ballot(faint_k) != 0 || !finite(acc);
    }
    if (stream == 0 && valid && __builtin_expect(!redo, 1)) {
        const float factor = l > 0.0f ? __builtin_amdgcn_ldexpf(P.scale / l, ek + eu + ev + 23 - 9) : 0.0f;
#pragma unroll
        for (int t = 0; t < DT; ++t) store_tile_row<VEC>(P.dq + row * D + 32 * t, acc[t], factor, h);
    }
    if (stream == 0 && lane == 0) redone[qi] = redo;
    __syncthreads();
#pragma unroll 1
    for (int x = 0; x < QB; ++x) {
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(redone[x]), 0))
            exact_dq_tile<D, VEC, QB * KS>((const SplitBackwardParams *)__builtin_amdgcn_kernarg_segment_ptr(), (LdsFloats)smem, seq, (qb * QB + x) * kTile);
    }
}

template<int D, bool VEC, int KB, int QS>
__global__ __launch_bounds__(kWave * KB * QS) __attribute__((amdgpu_waves_per_eu(2))) void attention_dkdv_split_kernel(const SplitBackwardParams P) {
    constexpr int KC = D / 16, DT = D / 32, CPR = D / 4;
    constexpr int CH = kTile * CPR / (kWave * KB);   // chunks per lane of a Q tile, and of a dO tile
    static_assert(CH >= 1);
    constexpr int PLANE = kTile * D;
    constexpr int STAGE = 4 * PLANE;                 // Q's two terms, high and low, then dO's
    constexpr int RPC = kWave * KB / CPR;
    constexpr int STAGE_BYTES = 2 * QS * STAGE * 2, MERGE_BYTES = (QS - 1) * KB * 16 * DT * kWave * 4;
    __shared__ __align__(16) unsigned char smem[STAGE_BYTES > MERGE_BYTES ? STAGE_BYTES : MERGE_BYTES];
    __shared__ __align__(16) float stats[QS][2][2][kTile]; // per stage: exponent offset of P, and δ'
    static_assert((KB * QS - 1) * 16 * DT * kWave * 4 <= STAGE_BYTES); // the slots of exact_dkdv_tile
    __shared__ float amax[2][KB * QS];
    __shared__ int redone[KB]; // key tiles to compute again
    __shared__ int gradient_chunks; // at least the rows of dO in the window that are not 0, where they were counted
    // Operands in LDS instead of registers, V's low terms and then K's: what 256 registers don't hold at D = 64, as far as the
    // workgroups of a CU have room. In scratch their reloads wait for the rows in flight (whole backward, 32 x 2048 causal 233
    // against 251 µs, 15 x 777 x 1001 68 against 78).
    constexpr int PARKED = D == 32 ? 0 : KB == 4 ? (QS == 1 ? 4 : 3) : (QS == 4 ? 8 : 6);
    __shared__ __align__(16) uint16_t parked[PARKED > 0 ? KB * PARKED * kWave * 8 : 8];
    __shared__ float norms[QS > 1 ? QS - 1 : 1][KB][2][kWave]; // of streams 1 ..: Σ P'² and Σ dS'² of each lane

    const Shape &s = P.s;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int ki = wave % KB, stream = wave / KB;
    const int col = lane & 31, h = lane >> 5;
    const float one = split_unit_scale();
    const int seqs = s.batch * s.heads;
    // Key blocks in order: under a causal mask the first ones see the most queries.
    const int seq = static_cast<int>(blockIdx.x) % seqs, kb = static_cast<int>(blockIdx.x) / seqs;
    const int b = seq / s.heads, head = seq - b * s.heads;
    const int kt = kb * KB + ki, key0 = kt * kTile, key = key0 + col;
    const bool tile_valid = key0 < s.keys;

    const Buffer qbuf = make_buffer(sequence(P.q, b, head), sequence_bytes(s.queries, P.q.st, D));
    const Buffer ubuf = make_buffer(sequence(P.u, b, head), sequence_bytes(s.queries, P.u.st, D));
    const Buffer kbuf = make_buffer(sequence(P.k, b, head), sequence_bytes(s.keys, P.k.st, D));
    const Buffer vbuf = make_buffer(sequence(P.v, b, head), sequence_bytes(s.keys, P.v.st, D));
    const Buffer mbuf = make_buffer(P.mask + static_cast<int64_t>(b) * s.keys, static_cast<uint32_t>(s.keys));
    const Buffer lbuf = make_buffer(P.lse + static_cast<int64_t>(seq) * s.queries * 2, static_cast<uint32_t>(s.queries) * 8u);
    const Buffer dbuf = make_buffer(P.delta + static_cast<int64_t>(seq) * s.queries, static_cast<uint32_t>(s.queries) * 4u);
    const uint32_t qstep = 4u * P.q.st, ustep = 4u * P.u.st;

    // This wave's queries [first, last) and the block's union of them, in whole tiles from ufirst.
    int first = 0, last = 0, ufirst = 0x7fffffff, ulast = 0;
#pragma unroll
    for (int x = 0; x < KB; ++x) {
        int f, e;
        if ((kb * KB + x) * kTile < s.keys && dkdv_query_range(s, kb * KB + x, f, e) > 0) {
            ufirst = min(ufirst, f / kTile * kTile);
            ulast = max(ulast, e);
            if (x == ki) {
                first = f;
                last = e;
            }
        }
    }
    const int ntiles = ulast > ufirst ? (ulast - ufirst + kTile - 1) / kTile : 0;
    if (ntiles == 0) ufirst = 0;
    const int nsteps = (ntiles + QS - 1) / QS;
    const int qlo = window_query_lo(s, key), qhi = min(window_query_hi(s, key), s.queries - 1);

    const int crow = (ki * kWave + lane) / CPR;
    const uint32_t qofs = static_cast<uint32_t>(crow) * qstep + 16u * static_cast<uint32_t>(lane % CPR);
    const uint32_t uofs = static_cast<uint32_t>(crow) * ustep + 16u * static_cast<uint32_t>(lane % CPR);
    int write[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) write[i] = staged_chunk<D>(crow + RPC * i, (lane % CPR) >> 1) + 4 * (lane & 1);
    const StagedReads<D, PLANE> reads;
    uint16_t *const stages = reinterpret_cast<uint16_t *>(smem) + stream * (2 * STAGE);

    f32x4 qraw[CH], uraw[CH];
    float rm, rl, rd; // statistics of query col of the tile (wave ki = 0 of the stream stages them)
    auto tile_query = [&](const int i) { return ufirst + (i * QS + stream) * kTile; };
    auto load_tile = [&](const int i) __attribute__((always_inline)) {
        const bool live = i * QS + stream < ntiles;
        const uint32_t t0 = static_cast<uint32_t>(tile_query(i));
        const uint32_t r0 = live ? t0 * qstep : kNoRow, w0 = live ? t0 * ustep : kNoRow;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            qraw[c] = load_chunk<VEC>(qbuf, qofs, r0 + static_cast<uint32_t>(RPC * c) * qstep);
            uraw[c] = load_chunk<VEC>(ubuf, uofs, w0 + static_cast<uint32_t>(RPC * c) * ustep);
        }
        rm = buffer_load(lbuf, 8u * col, live ? 8u * t0 : kNoRow);
        rl = buffer_load(lbuf, 8u * col + 4u, live ? 8u * t0 : kNoRow);
        rd = buffer_load(dbuf, 4u * col, live ? 4u * t0 : kNoRow);
    };

    constexpr int ROWS = kWave * KB * QS / CPR;
    const int n = min(ulast, s.queries) - ufirst;
    const int sampled = ufirst + (n > 0 ? static_cast<int>(static_cast<int64_t>(static_cast<int>(threadIdx.x) / CPR) * n / ROWS) : 0);
    const f32x4 sq = load_chunk<VEC>(qbuf, static_cast<uint32_t>(sampled) * qstep + 16u * (threadIdx.x % CPR), 0);
    const f32x4 su = load_chunk<VEC>(ubuf, static_cast<uint32_t>(sampled) * ustep + 16u * (threadIdx.x % CPR), 0);
    const bool visible = key < s.keys && buffer_load_byte(mbuf, key < s.keys ? static_cast<uint32_t>(key) : kNoRow) != 0;
    f32x4 kraw[2 * KC], vraw[2 * KC]; // rows of masked keys read 0
#pragma unroll
    for (int i = 0; i < 2 * KC; ++i) {
        const uint32_t f = 4u * (16 * (i / 2) + 8 * h + 4 * (i % 2)), r = static_cast<uint32_t>(key);
        kraw[i] = load_chunk<VEC>(kbuf, visible ? r * (4u * P.k.st) + f : kNoRow, 0);
        vraw[i] = load_chunk<VEC>(vbuf, visible ? r * (4u * P.v.st) + f : kNoRow, 0);
    }
    load_tile(0);
    const uint32_t bits = static_cast<uint32_t>(__ballot(visible));

    float mq = largest(sq), mu = largest(su);
    workgroup_largest(mq, mu, amax);
    if (threadIdx.x == 0) gradient_chunks = 0x40000000;
    if (n > ROWS && __builtin_amdgcn_readfirstlane(mq == 0.0f || mu == 0.0f)) {
        if (threadIdx.x == 0) gradient_chunks = 0;
        const int found = window_largest<kWave * KB * QS, CPR>(mq, mu, n, [&](const int) { return true; },
                [&](const int r, const bool on, f32x4 &x, f32x4 &y) {
                    const uint32_t at = 16u * (threadIdx.x % CPR), row = static_cast<uint32_t>(ufirst + r);
                    x = load_chunk<VEC>(qbuf, on ? row * qstep + at : kNoRow, 0);
                    y = load_chunk<VEC>(ubuf, on ? row * ustep + at : kNoRow, 0);
                });
        __syncthreads(); // amax is read
        if (found != 0) atomicAdd(&gradient_chunks, found);
        workgroup_largest(mq, mu, amax);
    }
    const int eq = __builtin_amdgcn_readfirstlane(exponent_of(mq)) - 11; // Q = Q'·2^eq, dO = dO'·2^eu, sampled largest at 2^11, 2^8
    const int eu = __builtin_amdgcn_readfirstlane(exponent_of(mu)) - 8;
    float mk = 0.0f, mv = 0.0f;
#pragma unroll
    for (int i = 0; i < 2 * KC; ++i) {
        mk = fmaxf(mk, largest(kraw[i]));
        mv = fmaxf(mv, largest(vraw[i]));
    }
    const float own_k = halves_max(mk), own_v = halves_max(mv); // of this lane's key
    __syncthreads(); // amax is read
    workgroup_largest(mk, mv, amax);
    const int ek = __builtin_amdgcn_readfirstlane(exponent_of(mk)) - 14;
    int ev = __builtin_amdgcn_readfirstlane(exponent_of(mv)) - 14;
    // A key whose own row lies below 2^-2 beside the block's largest.
    const bool faint_key = (own_k > 0.0f && own_k < __builtin_amdgcn_ldexpf(1.0f, ek - 2)) ||
            (own_v > 0.0f && own_v < __builtin_amdgcn_ldexpf(1.0f, ev - 2));
    float md = 1.0f;
    if (__builtin_amdgcn_readfirstlane(mv == 0.0f)) { // dP = 0: the unit of dP - δ below comes from the largest |δ|, put at 2^-4
        float none = 0.0f;
        md = 0.0f;
        for (int r = threadIdx.x; r < n; r += kWave * KB * QS) md = fmaxf(md, fabsf(buffer_load(dbuf, 4u * static_cast<uint32_t>(ufirst + r), 0)));
        __syncthreads(); // amax is read
        workgroup_largest(md, none, amax);
        if (md > 0.0f) ev = __builtin_amdgcn_readfirstlane(exponent_of(md)) - eu - 20;
    }
    // Exactly 0 whatever the scales: dV and dK, and dK alone.
    const bool no_dv = __builtin_amdgcn_readfirstlane(mu == 0.0f), no_dk = __builtin_amdgcn_readfirstlane(mu == 0.0f || mq == 0.0f || md == 0.0f);
    const float qfactor = scale_down(eq), ufactor = scale_down(eu);
    h16x8 kh[KC], kl[KC], vh[KC], vl[KC];
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        split_operand(kraw[2 * i], kraw[2 * i + 1], scale_down(ek), kh[i], kl[i]);
        split_operand(vraw[2 * i], vraw[2 * i + 1], scale_down(ev), vh[i], vl[i]);
    }
    h16x8 *const park = reinterpret_cast<h16x8 *>(parked) + ki * PARKED * kWave + lane;
    if (stream == 0) {
#pragma unroll
        for (int x = 0; x < PARKED; ++x) park[x * kWave] = x < KC ? vl[x % KC] : kl[x % KC];
    }
    // Low terms of K or V, from the first barrier of the loop on.
    auto low_terms = [&](auto of_k, h16x8 (&x)[KC], const h16x8 (&held)[KC]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int at = i + (decltype(of_k)::value ? KC : 0);
            if (at < PARKED) x[i] = park[at * kWave];
            else x[i] = held[i];
        }
    };
    // P' = 2^14·P = exp2(S'·c2 + offset); dP - δ in units of 2^(eu + ev + 24): r = dP'·2^-24 - δ'. P'·r stays below 2^16 while
    // P·|dP - δ| is below 4 times the product of the largest |dO| (sampled) and |V|.
    const float c2 = __builtin_amdgcn_ldexpf(P.scale * kLog2e, eq + ek);
    constexpr float kUnit = 1.0f / (1 << 24);
    // FP32 MFMAs from the start: for the whole workgroup where a scale does not fit, or where rows of Q below 2^-3, whose terms are
    // off by 2^-25, could move a score by more than 2^-22 (2^-7·c2: K' below 2^15, errors of D features adding up at random); for one
    // wave where a key of its own is faint (it goes on staging for the others).
    const bool unfit = !scale_fits(ek) || !scale_fits(ev) || !scale_fits(eq) || !scale_fits(eu) || c2 > 0x1p-15f;
    const bool own_unfit = __ballot(faint_key) != 0;

    f32x16 acc_k[DT], acc_v[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc_k[t] = acc_v[t] = f32x16{};
    float p_norm = 0.0f, ds_norm = 0.0f; // Σ P'² and Σ dS'² of the lane's key over its half of the rows, from the high terms

    auto stage = [&](const int i, const int p) __attribute__((always_inline)) {
        u32x2 terms[2];
#pragma unroll
        for (int c = 0; c < 2 * CH; ++c) {
            const f32x4 x = c < CH ? qraw[c % CH] : uraw[c % CH];
            uint16_t *const at = stages + p * STAGE + (c < CH ? 0 : 2 * PLANE) + write[c % CH];
            stage_pair<0, PLANE>(x, c < CH ? qfactor : ufactor, terms, at);
            stage_pair<1, PLANE>(x, c < CH ? qfactor : ufactor, terms, at);
        }
        if (ki == 0 && h == 0) {
            const bool ok = tile_query(i) + col < s.queries && i * QS + stream < ntiles && rm != -INFINITY;
            stats[stream][p][0][col] = ok ? 14.0f - fmaf(rm, kLog2e, __log2f(rl)) : -INFINITY;
            stats[stream][p][1][col] = __builtin_amdgcn_ldexpf(-rd, -(eu + ev + 24));
        }
    };
    // The tile in stage p. The order is left to the compiler: at D = 64, some operands in LDS, the step just fits 256 registers, and
    // with its groups pinned as in kernel 1 50 of them are spilled (32 x 2048 causal 123 -> 256 µs; with one wave per SIMD
    // instead 142).
    auto tile_step = [&](auto masked, const int p, const int q0) __attribute__((always_inline)) {
        const uint16_t *const qt = stages + p * STAGE;
        f32x16 sc{}, dp{};
        h16x8 low[KC];
        low_terms(std::integral_constant<bool, true>{}, low, kl);
        row_product<D, PLANE>(sc, reads, qt, kh, low);
        low_terms(std::integral_constant<bool, false>{}, low, vl);
        row_product<D, PLANE>(dp, reads, qt + 2 * PLANE, vh, low);
        uint32_t keep = 0;
        if constexpr (decltype(masked)::value) keep = visible ? bit_range(qlo - q0, qhi - q0) >> (4 * h) : 0u;
        uint32_t pt[2][8], ds[2][8];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const f32x4 offset = *reinterpret_cast<const f32x4 *>(&stats[stream][p][0][8 * u + 4 * h]);
            const f32x4 dl = *reinterpret_cast<const f32x4 *>(&stats[stream][p][1][8 * u + 4 * h]);
            float x[4], y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                x[j] = exp2_fast(fmaf(sc[4 * u + j], c2, offset[j]));
                if constexpr (decltype(masked)::value) x[j] = (keep >> (8 * u + j)) & 1u ? x[j] : 0.0f;
                y[j] = x[j] * fmaf(dp[4 * u + j], kUnit, dl[j]);
            }
            split_pair<false>(x[0], x[1], one, pt[0][2 * u], pt[1][2 * u]);
            split_pair<false>(x[2], x[3], one, pt[0][2 * u + 1], pt[1][2 * u + 1]);
            split_pair<false>(y[0], y[1], one, ds[0][2 * u], ds[1][2 * u]);
            split_pair<false>(y[2], y[3], one, ds[0][2 * u + 1], ds[1][2 * u + 1]);
            p_norm = add_squares(pt[0][2 * u + 1], add_squares(pt[0][2 * u], p_norm));
            ds_norm = add_squares(ds[0][2 * u + 1], add_squares(ds[0][2 * u], ds_norm));
        }
        column_product<D, PLANE>(acc_v, reads, qt + 2 * PLANE, pt);
        column_product<D, PLANE>(acc_k, reads, qt, ds);
    };

    if (nsteps > 0 && !unfit) {
        stage(0, 0);
        load_tile(1);
        auto step = [&](const int i, const int p) __attribute__((always_inline)) {
            __syncthreads(); // tile i is staged; every wave is done with the other stage
            const int q0 = tile_query(i);
            const bool work = i * QS + stream < ntiles && bits != 0 && !own_unfit && q0 < last && q0 + kTile > first;
            stage(i + 1, p ^ 1);
            load_tile(i + 2);
            if (__builtin_expect(work, 1)) {
                if (__builtin_expect(bits == 0xffffffffu && q0 + kTile <= s.queries && tile_in_window(s, q0, key0), 1))
                    tile_step(std::integral_constant<bool, false>{}, p, q0);
                else tile_step(std::integral_constant<bool, true>{}, p, q0);
            }
        };
        for (int i = 0; i < nsteps; i += 2) {
            step(i, 0);
            if (i + 1 < nsteps) step(i + 1, 1);
        }
    }
    float *const slot = reinterpret_cast<float *>(smem) + ki * (16 * DT * kWave) + lane;
    if (QS > 1 && stream > 0) {
        norms[stream - 1][ki][0][lane] = p_norm;
        norms[stream - 1][ki][1][lane] = ds_norm;
    }
    sum_streams<DT, QS>(acc_k, stream, slot, KB * 16 * DT * kWave);
    sum_streams<DT, QS>(acc_v, stream, slot, KB * 16 * DT * kWave);
    bool redo = false;
    if (stream == 0 && tile_valid) {
#pragma unroll
        for (int x = 0; x < QS - 1; ++x) {
            p_norm += norms[x][ki][0][lane];
            ds_norm += norms[x][ki][1][lane];
        }
        // Keys whose sums are made of terms that lost bits (below 2^-3 they are off by 2^-25): because the rows of dO or Q that count for
        // the key lie far below the ones that set the scales (hidden from it, or without weight), or its weights or dS are small
        // throughout. With Σ P'² of n rows, dV' is off by 2^-25·√(Σ P'²) from dO' and by 2^-26·√n·|dO'| from P': the first is below
        // 2^-21 of the largest |dV'| if that reaches 2^-4·√(Σ P'²), the second below 2^-20 if Σ P'² reaches 2^-12·n and, where the
        // rows that make Σ P'² up are not those that make dV up, |dV'| 2·√n (|dO'| of 2^7). The same for dK' with dS' and Q' (of 2^10:
        // 16·√n). A small Σ dS'² also does no harm where FP32's own rounding of dP is larger (a key of weight near 1, whose dP - δ
        // cancels): 2^-24·Σ |dO'|·|V'| in units of 2^24, |dO'| taken from dV' feature by feature.
        p_norm = halves_sum(p_norm);
        ds_norm = halves_sum(ds_norm);
        const float top_v = halves_max(largest(acc_v)), top_k = halves_max(largest(acc_k));
        const float seen = static_cast<float>(min(qhi - max(qlo, 0) + 1, gradient_chunks)); // rows that can be off (dO = 0: exact)
        const float root = sqrtf(seen);
        bool faint = visible && ((!no_dv && (256.0f * top_v * top_v < p_norm || p_norm < 0x1p-12f * seen || top_v < 2.0f * root)) ||
                (!no_dk && (256.0f * top_k * top_k < ds_norm || (ds_norm >= 0x1p-12f * seen && top_k < 16.0f * root))));
        const bool faint_ds = visible && !no_dk && ds_norm < 0x1p-12f * seen;
        if (__builtin_expect(__ballot(faint_ds) != 0, 0)) {
            float products = 0.0f;
            unrolled<DT>([&](auto t) {
                unrolled<4>([&](auto g) { // features of accumulator registers 4g .. 4g + 3
                    const uint32_t f = 4u * (32 * t.value + 8 * g.value + 4 * h);
                    const f32x4 own = load_chunk<VEC>(vbuf, visible ? static_cast<uint32_t>(key) * (4u * P.v.st) + f : kNoRow, 0);
                    unrolled<4>([&](auto x) { products += fabsf(acc_v[t.value][4 * g.value + x.value] * own[x.value]); });
                });
            });
            faint = faint || (faint_ds && halves_sum(products) * scale_down(ev) < 0x1p24f * root);
        }
        redo = unfit || own_unfit || __ballot(faint) != 0 || !finite(acc_k) || !finite(acc_v);
    }
    if (stream == 0 && key < s.keys && __builtin_expect(!redo, 1)) {
        const int64_t krow = (static_cast<int64_t>(seq) * s.keys + key) * D;
        const float kscale = __builtin_amdgcn_ldexpf(P.scale, eq + eu + ev + 24 - 14), vscale = __builtin_amdgcn_ldexpf(1.0f, eu - 14);
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            store_tile_row<VEC>(P.dk + krow + 32 * t, acc_k[t], kscale, h);
            store_tile_row<VEC>(P.dv + krow + 32 * t, acc_v[t], vscale, h);
        }
    }
    if (stream == 0 && lane == 0) redone[ki] = redo;
    __syncthreads();
#pragma unroll 1
    for (int x = 0; x < KB; ++x) {
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(redone[x]), 0))
            exact_dkdv_tile<D, VEC, KB * QS>((const SplitBackwardParams *)__builtin_amdgcn_kernarg_segment_ptr(), (LdsFloats)smem, seq, kb * KB + x);
    }
}

namespace {

SplitBackwardParams params_of(const BackwardArgs &a, const int D) {
    const auto tensor = [](const float *p, const rocmkernels_strides &st) { return Tensor{p, st.batch, st.head, st.token}; };
    return SplitBackwardParams{tensor(a.q, a.qs), tensor(a.k, a.ks), tensor(a.v, a.vs), tensor(a.output, a.os), tensor(a.upstream, a.us),
            reinterpret_cast<const uint8_t *>(a.mask), a.lse, a.gradient_q, a.gradient_k, a.gradient_v, a.delta,
            Shape{a.batch, a.heads, a.queries, a.keys, a.radius, a.causal}, 1.0f / sqrtf(static_cast<float>(D))};
}

template<int D, bool VEC, int QB, int KS>
void launch_dq(const BackwardArgs &a, hipStream_t stream) {
    const int64_t blocks = static_cast<int64_t>(a.batch) * a.heads * ((a.queries + QB * kTile - 1) / (QB * kTile));
    hipLaunchKernelGGL((attention_dq_split_kernel<D, VEC, QB, KS>), dim3(static_cast<unsigned>(blocks)), dim3(kWave * QB * KS), 0, stream, params_of(a, D));
}
template<int D, bool VEC, int KB, int QS>
void launch_dkdv(const BackwardArgs &a, hipStream_t stream) {
    const int64_t blocks = static_cast<int64_t>(a.batch) * a.heads * ((a.keys + KB * kTile - 1) / (KB * kTile));
    hipLaunchKernelGGL((attention_dkdv_split_kernel<D, VEC, KB, QS>), dim3(static_cast<unsigned>(blocks)), dim3(kWave * KB * QS), 0, stream, params_of(a, D));
}

// Work of one kernel: 32-row items (query tiles in kernel 1, key tiles in kernel 2), and the tiles streamed for the widest.
struct Work {
    int64_t items;
    int tiles;
};

Work query_work(const BackwardArgs &a) {
    const Shape s{a.batch, a.heads, a.queries, a.keys, a.radius, a.causal};
    const int qtiles = (a.queries + kTile - 1) / kTile;
    return Work{static_cast<int64_t>(qtiles) * a.batch * a.heads, std::max(forward_item_tiles(s, qtiles / 2), forward_item_tiles(s, qtiles - 1))};
}

Work key_work(const BackwardArgs &a) {
    const int ktiles = (a.keys + kTile - 1) / kTile;
    int first, last;
    return Work{static_cast<int64_t>(ktiles) * a.batch * a.heads, std::max(key_tile_queries(a.queries, a.radius, a.causal, 0, first, last),
            key_tile_queries(a.queries, a.radius, a.causal, ktiles / 2, first, last))};
}

// Whether item costs run from one tile to many over much of the sequence.
bool ramp(const BackwardArgs &a) { return a.causal != 0 && (a.radius < 0 || a.radius >= a.queries / 2); }

} // namespace

// Workgroup shapes. Every µs below: items, tiles of the widest: this choice against the next best one.
//   Kernel 1. Up to two items per CU two query tiles and two streams, so that every CU has work (d = 32: 256, 64: 28.2 against
//   37.2; d = 64: 384, 32: 18.3 against 22.3), also under a ramp up to four if its items are long, where the longest end last
//   (d = 32: 768, 32: 19.8 against 23.0; d = 64: 1024, 64: 64.3 against 69.2). Four and two while a workgroup's items are long
//   and the workgroups few (1024, 64: d = 32 48.1 against 50.2, d = 64 84.5 against 86.4; ramps of 2048, 128: 99.7 against 107.9
//   and 169 against 184). Else four and one, whose waves are in step with the fewest others (d = 32: 3072, 32: 72.9 against
//   85.0; d = 64: 123 against 143; 768, 8: 10.1 against 11.4).
SplitWorkgroup dq_split_workgroup(const int D, const BackwardArgs &a, const int cus) {
    const Work w = query_work(a);
    if (w.items <= 2ll * cus ? w.tiles > 2 : ramp(a) && w.items <= 4ll * cus && w.tiles >= D / 2) return SplitWorkgroup{2, 2};
    if (w.tiles >= 64 && w.items <= (ramp(a) ? 8ll : 4ll) * cus) return SplitWorkgroup{4, 2};
    return SplitWorkgroup{4, 1};
}

//   Kernel 2. Up to two items per CU two key tiles and four streams if the items are long (d = 32: 512, 128: 72 against 89; d =
//   64: 256, 64: 69 against 92), two and two if not (d = 32: 384, 8: 10.7 against 13.8). Up to four per CU, and under a ramp up
//   to eight, two and two at d = 32 (768, up to 32: 27.3 against 32.7; 1536, up to 64: 58.7 against 62.4), but four and two
//   without a ramp (768, 32: 33.6 against 35.4) and at d = 64, where the steps of a workgroup with more key tiles share more
//   (768, 32: 60.4 against 71.5; ramp of 2048, 128: 242 against 290). Else four and one (3072, 32: 107 against 116 and 198
//   against 203; 2048, 8: 24.0 against 28.6).
SplitWorkgroup dkdv_split_workgroup(const int D, const BackwardArgs &a, const int cus) {
    const Work w = key_work(a);
    if (w.items <= 2ll * cus) {
        if (w.tiles >= 16) return SplitWorkgroup{2, 4};
        if (w.tiles > 2) return SplitWorkgroup{2, 2};
    } else if (w.items <= 4ll * cus ? D == 32 || w.tiles > 4 : ramp(a) && w.items <= 8ll * cus && w.tiles >= D / 2) {
        return D == 64 || (!ramp(a) && w.tiles >= 16) ? SplitWorkgroup{4, 2} : SplitWorkgroup{2, 2};
    }
    return SplitWorkgroup{4, 1};
}

namespace {

template<int D, bool VEC>
void dispatch_dq(const BackwardArgs &a, const int cus, hipStream_t stream) {
    const SplitWorkgroup g = dq_split_workgroup(D, a, cus);
    if (g.tiles == 2) launch_dq<D, VEC, 2, 2>(a, stream);
    else if (g.streams == 2) launch_dq<D, VEC, 4, 2>(a, stream);
    else launch_dq<D, VEC, 4, 1>(a, stream);
}

template<int D, bool VEC>
void dispatch_dkdv(const BackwardArgs &a, const int cus, hipStream_t stream) {
    const SplitWorkgroup g = dkdv_split_workgroup(D, a, cus);
    if (g.tiles == 2) g.streams == 4 ? launch_dkdv<D, VEC, 2, 4>(a, stream) : launch_dkdv<D, VEC, 2, 2>(a, stream);
    else if (g.streams == 2) launch_dkdv<D, VEC, 4, 2>(a, stream);
    else launch_dkdv<D, VEC, 4, 1>(a, stream);
}

template<int D, bool VEC>
hipError_t dispatch(const BackwardArgs &a, const int cus, hipStream_t stream) {
    dispatch_dq<D, VEC>(a, cus, stream);
    const hipError_t error = hipGetLastError();
    if (error != hipSuccess) return error;
    dispatch_dkdv<D, VEC>(a, cus, stream);
    return hipGetLastError();
}

} // namespace

// Long items (32 tiles and more) always beat the deterministic FP32 pair, whose waves pay more per tile (d = 32, 4 x 2048: 62
// against 71 µs; d = 64, 4 x 1024: 68 against 72), if their loads are 128-bit ones (else 114 against 72). Otherwise the grid has
// to be filled: from more than one item per CU on (d = 32, 384 items of 8 tiles: 19.6 µs against the key-block kernel's 28.8
// and the pair's 25.4; 256 of 16: 25.5 against 24.1 for the pair) in both kernels (four fifths: 67 x 3 query
// tiles, 12 key tiles: 25.9 against 20.7 for the key-block kernel; 6 sequences of 777 of 2001: 47.5 against 42.9), a little further at d = 64 against the key-block kernel (280 items of
// 14: 47.0 against 44.3; 288, 48: 98.8 against 98.7; 308, 14: 52.4 against 63.1). Under a ramp half the pairs are seen but the
// longest items last as long, so that the key-block kernel's balanced pieces win for longer, the more so the longer the items: at
// d = 32 up to about two per CU (264, 88: 81 against 50; 384, 32: 38.6 against 34.5; 490, 70: 70.0 against 67.2; but 448, 8: 20.9
// against 21.8; 768, 32: 46.4 against 54.8), at d = 64 up to three (512, up to 128: 210 against 199; 594, 54: 134 against 114; 640,
// 20: 69 against 67; but 768, 32: 92 against 98; 768, 8: 43.5 against 54.9; 384 of 4: 27.5 against 31.1). Against the pair d = 64
// wins at once (384, 16: 49 against 58), and at d = 32 the pair's planned grid lasts to two per CU (384, up to 16: 26.1 against
// 25.0; 512, up to 32: 38.7 against 46.0).
// Sequences of one or two tiles leave most waves of a workgroup idle: against the pair's one item per wave that costs more than the
// products save at d = 32 (600 x 1 query tile, 32: 121 against 145; 4096 x 1, 1: 44 against 90), at d = 64 only in large launches of
// short items (4096 x 1, 1: 80 against 131). Nor do odd query tiles pay at d = 64 where they make more two-tile workgroups than
// CUs (102 x 5, 3: 35.0 against 41.6), and short items of few launches at d = 32 (260, 3: 16.4 against 18.2).
bool backward_split_pays(const int D, const BackwardArgs &a, const int cus, const bool vec, const bool deterministic) {
    const Work q = query_work(a), k = key_work(a);
    const int64_t items = (q.items + k.items) / 2, fewer = std::min(q.items, k.items);
    const int tiles = std::max(q.tiles, k.tiles), qtiles = (a.queries + kTile - 1) / kTile;
    if (deterministic && D == 32 && qtiles == 1) return false;
    if (deterministic && vec && tiles >= 32) return true;
    if (items <= cus || 5 * fewer < (vec ? 4ll : 5ll) * cus) return false;
    if (D == 32 && 4 * items <= 5ll * cus && tiles < 6) return false;
    if (D == 64 && tiles < 16 && q.tiles > 2 && q.items <= 2ll * cus && static_cast<int64_t>(a.batch) * a.heads * ((qtiles + 1) / 2) > cus) return false;
    if (deterministic && qtiles <= 2 && tiles <= 5 && items >= 8ll * cus) return false;
    if (!deterministic && a.radius < 0) { // against the key-block kernel
        if (!ramp(a)) return D == 32 || 8 * items > 9ll * cus;
        if (D == 32) return tiles * (2ll * cus - items) <= 5ll * cus;
        return items >= 3ll * cus || tiles <= 4 || (items > 2ll * cus && tiles <= 12);
    }
    if (!ramp(a)) return true;
    if (D == 32) return items >= 2ll * cus;
    return items > 2ll * cus || tiles <= 4 || (deterministic && vec && a.radius < 0);
}

hipError_t launch_backward_split(const int D, const bool vec, const BackwardArgs &a, const int cus, hipStream_t stream) {
    if (D == 32) return vec ? dispatch<32, true>(a, cus, stream) : dispatch<32, false>(a, cus, stream);
    return vec ? dispatch<64, true>(a, cus, stream) : dispatch<64, false>(a, cus, stream);
}

} // namespace rk
