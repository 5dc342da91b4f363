// FP32 attention forward for gfx950 (MI355X) on the fp16 matrix cores, head width 32 or 64: the maths of
// attention_forward.hip (Attention.hip:32-115, AttentionFlash32.h:23-170, Attention64.hip:34-129 in the reference), with
// each FP32 product formed from three fp16 products of two-term operands (attention_split.hpp).
//
// Mapping. A workgroup owns QB query tiles of 32 of one sequence, one per wave of a key stream; its KS key streams take
// alternate 64-key tiles of the workgroup's window. The QB waves of a stream load each K and V tile together (a share of
// the rows each, whole lines, a step ahead), split it into terms once, and write the terms to the stream's double-buffered
// LDS stage, from which all of them read their MFMA operands; so the loads and the splitting of K and V cost each wave
// 1 / QB of a tile. Q's terms stay in registers; P is split in registers (its accumulator layout is the PV operand's).
//   * Sᵀ = K·Qᵀ: operands K rows (128-bit LDS reads), Q rows; the small products first.
//   * Oᵀ += Vᵀ·Pᵀ: operands V through transposing LDS reads (ds_read_b64_tr_b16), P in place.
// A step is one barrier and a 64-key tile in two halves A and B of 32 keys, in four groups of MFMAs, each beside VALU work
// that does not depend on it: Sᵀ of A beside the split of the next tile's K; Sᵀ of B beside A's softmax; Oᵀ of A beside B's
// softmax; Oᵀ of B beside the split of the next tile's V. The source spreads that work evenly over a group's MFMAs and pins
// the order (the compiler's own order puts the MFMAs first, and the two no longer co-execute).
//
// Scales (powers of two): each query row its own; K and V one each for the workgroup, from the largest magnitudes of rows
// sampled over its window (of all its rows where the sampled ones are 0). They put those at 2^8 (K) and 2^9 (V), so rows up to
// 64 times larger than any sampled one are still in range; larger ones make the result NaN. A query tile is computed again with
// FP32 MFMAs, by the whole workgroup, where its wave finds a non-finite result (as it must anyway for infinities, whose
// meaning the split products lose) or a row whose keys and values all lie so far below the scales that their terms lost
// bits: the rows that set a scale may be hidden from it by the masks, or have no weight.
#include <algorithm>
#include <type_traits>

#include "attention_launch.hpp"
#include "attention_split.hpp"

namespace rk {

namespace {

constexpr int kStep = 2 * kTile;  // keys of a step

struct SplitForwardParams {
    Tensor q, k, v;
    const uint8_t *mask;
    float *out;
    int osb, osh, ost;
    float *lse;
    Shape s;
    float scale;
};

// Position (in 2-byte elements) of element 0 of 16-byte chunk c of row r in a staged plane of D columns: rows are
// unpadded and their chunks permuted. K's row-layout reads (16 lanes: 16 rows, one chunk each) then meet 16 distinct
// 16-byte bank groups; V's transposing reads (32 lanes: 4 rows of 64 bytes) cover all 64 banks once.
template<int D>
__device__ __forceinline__ int k_chunk(const int r, const int c) {
    const int swizzle = D == 64 ? ((r & 7) ^ ((r >> 3) & 1)) : ((r >> 2) & 3);
    return r * D + 8 * (c ^ swizzle);
}
template<int D>
__device__ __forceinline__ int v_chunk(const int r, const int c) {
    return r * D + 8 * (D == 64 ? c ^ (2 * (r & 3)) : c);
}

// Writes the output rows and statistics of a wave's query tile: state (m_raw, l) with l summed over both half-waves, O
// = o / l times 2^ev, the row maximum m_raw·2^e, and l relative to the true maximum `sum`.
template<int D, bool VEC>
__device__ __forceinline__ void store_rows(const SplitForwardParams &P, const int seq, const int query, const int h, const f32x16 (&o)[D / 32],
        const float l, const float row_max, const float sum, const int ev) {
    if (query >= P.s.queries) return;
    const int b = seq / P.s.heads, head = seq - b * P.s.heads;
    const bool nan_row = isnan(l);
    const bool has_keys = l > 0.0f;
    const float factor = has_keys ? __builtin_amdgcn_ldexpf(1.0f / l, ev) : (nan_row ? NAN : 0.0f);
    float *orow = P.out + static_cast<int64_t>(b) * P.osb + static_cast<int64_t>(head) * P.osh + static_cast<int64_t>(query) * P.ost;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) {
        if (has_keys) {
            store_tile_row<VEC>(orow + 32 * t, o[t], factor, h);
        } else {
            const f32x16 fill{};
            store_tile_row<VEC>(orow + 32 * t, fill + factor, 1.0f, h);
        }
    }
    if (h == 0) {
        const int64_t row = static_cast<int64_t>(seq) * P.s.queries + query;
        P.lse[2 * row] = has_keys ? row_max : (nan_row ? NAN : -INFINITY);
        P.lse[2 * row + 1] = has_keys ? sum : (nan_row ? NAN : 0.0f);
    }
}

// One query tile on FP32 MFMAs by the workgroup's WAVES waves, for inputs that the split products cannot carry: the arithmetic of
// attention_forward.hip, operands straight from memory, K a tile ahead. The waves take alternate key tiles and are merged in order
// through `slots` (3 + D/2 floats a lane for each wave but one). Kept out of line (and given the kernel's arguments by
// address), so that the main loop's registers do not depend on it, and one for each register budget of a kernel (WPE). With
// one wave a tile instead, a single tile that needed it held its launch up for 200 µs (24 x 1024 at width 32).
template<int D, bool VEC, int WAVES, int WPE>
__device__ __attribute__((noinline)) void exact_query_tile(const SplitForwardParams *params, LdsFloats slots, const int seq_, const int q0_) {
    const auto address = reinterpret_cast<uint64_t>(params);
    const uint64_t uniform = static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(address >> 32))) << 32 |
            static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(address)));
    const SplitForwardParams &P = *reinterpret_cast<const SplitForwardParams *>(uniform);
    const int seq = __builtin_amdgcn_readfirstlane(seq_), q0 = __builtin_amdgcn_readfirstlane(q0_);
    constexpr int HALF = D / 2, DT = D / 32, SLOT = (3 + 16 * DT) * kWave;
    const Shape s = P.s;
    const int lane = threadIdx.x & (kWave - 1), col = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int query = q0 + col;
    const int b = seq / s.heads, head = seq - b * s.heads;
    const Buffer qbuf = make_buffer(sequence(P.q, b, head), sequence_bytes(s.queries, P.q.st, D));
    const Buffer kbuf = make_buffer(sequence(P.k, b, head), sequence_bytes(s.keys, P.k.st, D));
    const Buffer vbuf = make_buffer(sequence(P.v, b, head), sequence_bytes(s.keys, P.v.st, D));
    const Buffer mbuf = make_buffer(P.mask + static_cast<int64_t>(b) * s.keys, static_cast<uint32_t>(s.keys));
    const uint32_t kstep = 4u * P.k.st, vstep = 4u * P.v.st;
    const float c2 = P.scale * kLog2e;
    const int wlo = window_lo(s, query), whi = window_hi(s, query);
    int first, last;
    forward_key_range(s, q0 / kTile, first, last);

    float qr[HALF], kr[HALF];
    buffer_load_span<VEC>(qr, qbuf, static_cast<uint32_t>(query) * (4u * P.q.st) + 4u * h * HALF);
    int mbyte = 0;
    auto load_keys = [&](const int key0) __attribute__((always_inline)) {
        const bool live = key0 < last;
        mbyte = buffer_load_byte(mbuf, live ? static_cast<uint32_t>(key0 + col) : kNoRow);
        buffer_load_span<VEC>(kr, kbuf, live ? static_cast<uint32_t>(key0 + col) * kstep + 4u * h * HALF : kNoRow);
    };
    float m = -INFINITY, base = -INFINITY, l = 0.0f; // m over this half-wave's keys; base of l and o, in log2 units
    f32x16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = f32x16{};
    load_keys(first + wave * kTile);
#pragma unroll 1
    for (int key0 = first + wave * kTile; key0 < last; key0 += WAVES * kTile) {
        const uint32_t bits = static_cast<uint32_t>(__ballot(mbyte != 0));
        if (bits == 0) {
            load_keys(key0 + WAVES * kTile);
            continue;
        }
        float vc[16 * DT];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int r = tile_row(j, h);
            // Masked keys contribute exactly nothing, whatever their stored values hold.
            const uint32_t at = (bits >> r) & 1u ? static_cast<uint32_t>(key0 + r) * vstep + 4u * col : kNoRow;
#pragma unroll
            for (int t = 0; t < DT; ++t) vc[j * DT + t] = buffer_load(vbuf, at + 128u * t, 0);
        }
        f32x16 sc{};
#pragma unroll
        for (int c = 0; c < HALF; ++c) sc = mfma(kr[c], qr[c], sc);
        load_keys(key0 + WAVES * kTile);
        const uint32_t visible = (bits & bit_range(wlo - key0, whi - key0)) >> (4 * h);
        float mx = m;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            sc[j] = (visible >> (8 * (j >> 2) + (j & 3))) & 1u ? sc[j] : -INFINITY;
            mx = fmaxf(mx, sc[j]);
        }
        m = mx;
        const float row = halves_max(m);
        const float base_new = row == -INFINITY ? -INFINITY : row * c2;
        const float alpha = base_new == -INFINITY ? 1.0f : exp2_fast(base - base_new);
        base = base_new;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] *= alpha;
        const float offset = base == -INFINITY ? 0.0f : base;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            sc[j] = exp2_fast(fmaf(sc[j], c2, -offset));
            l += sc[j];
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
#pragma unroll
            for (int t = 0; t < DT; ++t) o[t] = mfma(vc[j * DT + t], sc[j], o[t]);
        }
    }
    m = halves_max(m);
    if (wave > 0) {
        const LdsFloats slot = slots + (wave - 1) * SLOT + lane;
        slot[0] = m;
        slot[kWave] = l;
        slot[2 * kWave] = base;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
#pragma unroll
            for (int j = 0; j < 16; ++j) slot[(3 + 16 * t + j) * kWave] = o[t][j];
        }
    }
    __syncthreads();
    if (wave == 0) {
        float top = base;
#pragma unroll
        for (int w = 0; w < WAVES - 1; ++w) {
            m = fmaxf(m, slots[w * SLOT + lane]);
            top = fmaxf(top, slots[w * SLOT + 2 * kWave + lane]);
        }
        const float to = top == -INFINITY ? 0.0f : top;
        const float own = exp2_fast(base - to);
        l *= own;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] *= own;
#pragma unroll 1
        for (int w = 0; w < WAVES - 1; ++w) {
            const LdsFloats slot = slots + w * SLOT + lane;
            const float a = exp2_fast(slot[2 * kWave] - to);
            l = fmaf(slot[kWave], a, l);
#pragma unroll
            for (int t = 0; t < DT; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) o[t][j] = fmaf(slot[(3 + 16 * t + j) * kWave], a, o[t][j]);
            }
        }
        l = halves_sum(l);
        const float sum = m == -INFINITY ? l : l * exp2_fast(to - m * c2);
        store_rows<D, VEC>(P, seq, query, h, o, l, m * P.scale, sum, 0);
    }
    __syncthreads(); // the slots are read
}

} // namespace

template<int D, bool VEC, int QB, int KS, int WPE>
__global__ __launch_bounds__(kWave * QB * KS) __attribute__((amdgpu_waves_per_eu(WPE))) void attention_forward_split_kernel(
        const SplitForwardParams P) {
    constexpr int KC = D / 16;                       // 16-feature steps of Sᵀ
    constexpr int DT = D / 32;                       // 32-feature slices of the output
    constexpr int CPR = D / 4;                       // 4-float chunks per row
    constexpr int CH = kStep * CPR / (kWave * QB);   // chunks per lane of a K tile, and of a V tile
    static_assert(CH >= 1 && CH * kWave * QB == kStep * CPR);
    constexpr int PLANE = kStep * D;                 // elements of one term of one tile
    constexpr int STAGE = 4 * PLANE;                 // K's two terms, high and low, then V's
    constexpr int NREG = 16 * DT + 3;                // merged per lane: maximum, sum, base and the accumulators
    constexpr int STAGE_BYTES = 2 * KS * STAGE * 2;
    constexpr int MERGE_BYTES = (KS - 1) * QB * NREG * kWave * 4;
    static_assert((QB * KS - 1) * NREG * kWave * 4 <= STAGE_BYTES); // the slots of exact_query_tile
    __shared__ __align__(16) unsigned char smem[STAGE_BYTES > MERGE_BYTES ? STAGE_BYTES : MERGE_BYTES];
    __shared__ float amax[2][QB * KS];               // largest sampled |K| and |V| of each wave
    __shared__ int redone[QB];                       // query tiles to compute again

    const Shape &s = P.s;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int qi = wave % QB;     // query tile of the block
    const int stream = wave / QB; // key stream
    const int col = lane & 31;
    const int h = lane >> 5;
    const float one = split_unit_scale();

    // Workgroup g takes a query block of sequence g mod B·H, the heaviest blocks first: with B·H a multiple of 8 each XCD
    // (workgroup g runs on XCD g mod 8) streams the K/V rows of its own eighth of the sequences from its L2.
    const int seqs = s.batch * s.heads;
    const int seq = static_cast<int>(blockIdx.x) % seqs;
    const int rank = static_cast<int>(blockIdx.x) / seqs;
    const int b = seq / s.heads, head = seq - b * s.heads;
    const int nblocks = (s.queries + QB * kTile - 1) / (QB * kTile);

    const Buffer qbuf = make_buffer(sequence(P.q, b, head), sequence_bytes(s.queries, P.q.st, D));
    const Buffer kbuf = make_buffer(sequence(P.k, b, head), sequence_bytes(s.keys, P.k.st, D));
    const Buffer vbuf = make_buffer(sequence(P.v, b, head), sequence_bytes(s.keys, P.v.st, D));
    const Buffer mbuf = make_buffer(P.mask + static_cast<int64_t>(b) * s.keys, static_cast<uint32_t>(s.keys));
    const uint32_t qstep = 4u * P.q.st, kstep = 4u * P.k.st, vstep = 4u * P.v.st;

    // This lane's chunks of a tile: chunk i is row crow + RPC·i, 4 floats from column 4 (lane mod CPR).
    constexpr int RPC = kWave * QB / CPR;
    const int crow = (qi * kWave + lane) / CPR;
    const uint32_t kofs = static_cast<uint32_t>(crow) * kstep + 16u * static_cast<uint32_t>(lane % CPR);
    const uint32_t vofs = static_cast<uint32_t>(crow) * vstep + 16u * static_cast<uint32_t>(lane % CPR);
    int kwrite[CH], vwrite[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int chunk = lane % CPR;
        kwrite[i] = k_chunk<D>(crow + RPC * i, chunk >> 1) + 4 * (chunk & 1);
        vwrite[i] = v_chunk<D>(crow + RPC * i, chunk >> 1) + 4 * (chunk & 1);
    }
    int kread[KC], vread[DT];
#pragma unroll
    for (int i = 0; i < KC; ++i) kread[i] = k_chunk<D>(col, 2 * i + h);
    // Transposing reads: lane L of each 16-lane group points at row r0 + (L mod 16) / 4, features f0 + 4 (L mod 4) .. + 3,
    // and receives feature f0 + L mod 16 of rows r0 .. r0 + 3, with r0 = 16u + 8p + 4h and f0 = 32 t2 + 16 (col / 16).
#pragma unroll
    for (int t2 = 0; t2 < DT; ++t2)
        vread[t2] = v_chunk<D>(4 * h + ((lane & 15) >> 2), 4 * t2 + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + 4 * (lane & 1);
    uint16_t *const stages = reinterpret_cast<uint16_t *>(smem) + stream * (2 * STAGE);

    const int qb = s.causal ? nblocks - 1 - rank : rank;
    const int q0 = (qb * QB + qi) * kTile;
    const int query = q0 + col;
    const bool tile_valid = q0 < s.queries;

    // This wave's window of keys [first, last) and the workgroup's union of windows, in tiles from ufirst.
    int first, last, ufirst, ulast, unused;
    forward_key_range(s, q0 / kTile, first, last);
    forward_key_range(s, qb * QB, ufirst, unused);
    forward_key_range(s, min(qb * QB + QB - 1, (s.queries - 1) / kTile), unused, ulast);
    const int ntiles = ulast > ufirst ? (ulast - ufirst + kStep - 1) / kStep : 0;
    const int nsteps = (ntiles + KS - 1) / KS; // tile of stream x at step i: i·KS + x
    const int wlo = window_lo(s, query);
    const int whi = window_hi(s, query);

    // Rows in flight, and their mask (one byte per key, 64 lanes). Rows of masked keys are cleared before they are split:
    // they contribute exactly nothing, whatever they hold.
    f32x4 kraw[CH], vraw[CH];
    auto tile_key = [&](const int i) { return ufirst + (i * KS + stream) * kStep; };
    auto load_mask = [&](const int i) __attribute__((always_inline)) {
        return buffer_load_byte_s(mbuf, static_cast<uint32_t>(lane), i * KS + stream < ntiles ? static_cast<uint32_t>(tile_key(i)) : kNoRow);
    };
    auto load_chunks = [&](f32x4 (&raw)[CH], const Buffer buf, const uint32_t at, const uint32_t step, const int i) __attribute__((always_inline)) {
        const uint32_t row0 = i * KS + stream < ntiles ? static_cast<uint32_t>(tile_key(i)) * step : kNoRow;
#pragma unroll
        for (int c = 0; c < CH; ++c) raw[c] = load_chunk<VEC>(buf, at, row0 + static_cast<uint32_t>(RPC * c) * step);
    };
    // Scales. Every thread reads a chunk of K and V in one of ROWS rows spread over the workgroup's window; masked rows
    // (keys past the end too) count as 0.
    constexpr int ROWS = kWave * QB * KS / CPR;
    int ek, ev; // K = K'·2^ek, V = V'·2^ev
    f32x4 qraw[2 * KC];
    int mask0;
    // Magnitudes that FP32 powers of two cannot bring into range: FP32 MFMAs from the start. Those of K and V keep the whole
    // workgroup from the loop; those of a wave's own queries keep only its products from it, as its siblings need the rows that
    // it stages and its barriers.
    bool unfit, own_unfit, v_zero; // v_zero: every visible row of V is 0
    {
        const int n = min(ulast, s.keys) - ufirst;
        const int key = ufirst + (n > 0 ? static_cast<int>(static_cast<int64_t>(static_cast<int>(threadIdx.x) / CPR) * n / ROWS) : 0);
        const uint32_t at = 16u * (threadIdx.x % CPR);
        const int seen = buffer_load_byte(mbuf, static_cast<uint32_t>(key));
        const f32x4 x = load_chunk<VEC>(kbuf, static_cast<uint32_t>(key) * kstep + at, 0), y = load_chunk<VEC>(vbuf, static_cast<uint32_t>(key) * vstep + at, 0);
        // Q and the first tile behind them: one round trip for all.
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const uint32_t at = tile_valid ? static_cast<uint32_t>(query) * qstep + 4u * (16 * i + 8 * h) : kNoRow;
            qraw[2 * i] = load_chunk<VEC>(qbuf, at, 0);
            qraw[2 * i + 1] = load_chunk<VEC>(qbuf, at + 16u, 0);
        }
        load_chunks(kraw, kbuf, kofs, kstep, 0);
        load_chunks(vraw, vbuf, vofs, vstep, 0);
        mask0 = load_mask(0);
        __builtin_amdgcn_sched_barrier(0);
        float mk = seen != 0 ? largest(x) : 0.0f, mv = seen != 0 ? largest(y) : 0.0f;
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
        ek = __builtin_amdgcn_readfirstlane(exponent_of(mk)) - 8;
        ev = __builtin_amdgcn_readfirstlane(exponent_of(mv)) - 9;
        unfit = !scale_fits(ek) || !scale_fits(ev);
        v_zero = __builtin_amdgcn_readfirstlane(mv == 0.0f);
    }

    // Q's terms, scaled so that the row's largest magnitude is in [2^14, 2^15).
    h16x8 qh[KC], ql[KC];
    int e; // S = S'·2^e
    {
        float span[KC][8], mq = 0.0f;
#pragma unroll
        for (int i = 0; i < KC; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                span[i][j] = qraw[2 * i][j];
                span[i][4 + j] = qraw[2 * i + 1][j];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) mq = fmaxf(mq, fabsf(span[i][j]));
        }
        const int eq = exponent_of(halves_max(mq)) - 14;
        own_unfit = __ballot(!scale_fits(eq)) != 0;
        const float factor = scale_down(eq);
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            u32x4 hi, lo;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t x, y;
                split_pair<true>(span[i][2 * j], span[i][2 * j + 1], factor, x, y);
                hi[j] = x;
                lo[j] = y;
            }
            qh[i] = __builtin_bit_cast(h16x8, hi);
            ql[i] = __builtin_bit_cast(h16x8, lo);
        }
        e = eq + ek;
    }
    const float kfactor = scale_down(ek), vfactor = scale_down(ev);

    // Online-softmax state, as in attention_forward.hip (lazy re-basing: see there), in units of S' and V'. P is kept at
    // 2^kShift times its value, so that its terms lose nothing above 2^-10 and at most 2^-32.
    constexpr float kLazy = 8.0f, kShift = 7.0f;
    const float c2 = __builtin_amdgcn_ldexpf(P.scale * kLog2e, e);
    const float lazy_raw = fminf(kLazy / c2, 1e30f);
    float m_half = -INFINITY, m_lazy = -INFINITY, mc = -INFINITY, mcx = 0.0f, l_run = 0.0f, alpha = 1.0f;
    f32x16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = f32x16{};

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
    // Splitting of the next tile's rows into stage p, in units of a pair of floats (the second of a chunk also writes).
    u32x2 chunk[2];
    auto split_unit = [&](auto unit, auto is_v, const int p) __attribute__((always_inline)) {
        constexpr int C = decltype(unit)::value / 2, E = decltype(unit)::value % 2;
        constexpr bool V = decltype(is_v)::value;
        const f32x4 &raw = V ? vraw[C] : kraw[C];
        uint32_t x, y;
        split_pair<true>(raw[2 * E], raw[2 * E + 1], V ? vfactor : kfactor, x, y);
        chunk[0][E] = x;
        chunk[1][E] = y;
        if constexpr (E == 1) {
            uint16_t *const st = stages + p * STAGE + (V ? 2 * PLANE + vwrite[C] : kwrite[C]);
            *reinterpret_cast<u32x2 *>(st) = chunk[0];
            *reinterpret_cast<u32x2 *>(st + PLANE) = chunk[1];
        }
    };
    constexpr std::integral_constant<bool, false> kOfK{};
    constexpr std::integral_constant<bool, true> kOfV{};

    // Operands of half x of the tile in stage p.
    auto read_k = [&](h16x8 (&kt)[KC], const int p, const int x, const int term) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KC; ++i)
            kt[i] = *reinterpret_cast<const h16x8 *>(stages + p * STAGE + term * PLANE + x * kTile * D + kread[i]);
    };
    auto read_v = [&](h16x8 (&vt)[DT], const int p, const int x, const int u, const int term) __attribute__((always_inline)) {
#pragma unroll
        for (int t2 = 0; t2 < DT; ++t2) {
            const uint16_t *const at = stages + p * STAGE + (2 + term) * PLANE + (x * kTile + 16 * u) * D + vread[t2];
            const u32x2 lo = read_transposed(at), hi = read_transposed(at + 8 * D);
            vt[t2] = __builtin_bit_cast(h16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
        }
    };
    // MFMA M of Sᵀ: K low with Q high, K high with Q low, K high with Q high.
    auto score_mfma = [&](auto index, f32x16 &sc, const h16x8 (&kl)[KC], const h16x8 (&kh)[KC]) __attribute__((always_inline)) {
        constexpr int M = decltype(index)::value;
        sc = mfma_f16(M < KC ? kl[M % KC] : kh[M % KC], M < KC || M >= 2 * KC ? qh[M % KC] : ql[M % KC], sc);
    };
    uint32_t ps[2][8]; // P's terms: the PV operand of MFMA step u is words 4u .. 4u + 3
    // MFMAs M of Oᵀ (DT each): V low with P high, V high with P low, V high with P high, for each half u of the 32 keys.
    auto output_mfma = [&](auto index, const uint32_t (&pt)[2][8], const h16x8 (&vl)[DT], const h16x8 (&vh)[DT]) __attribute__((always_inline)) {
        constexpr int M = decltype(index)::value;
        constexpr int U = M / 3, Y = M % 3 == 1;
        const h16x8 x = __builtin_bit_cast(h16x8, u32x4{pt[Y][4 * U], pt[Y][4 * U + 1], pt[Y][4 * U + 2], pt[Y][4 * U + 3]});
#pragma unroll
        for (int t2 = 0; t2 < DT; ++t2) o[t2] = mfma_f16(M % 3 == 0 ? vl[t2] : vh[t2], x, o[t2]);
    };
    auto mask_scores = [&](f32x16 &sc, const int key0, const uint32_t bits) __attribute__((always_inline)) {
        const uint32_t visible = (bits & bit_range(wlo - key0, whi - key0)) >> (4 * h);
#pragma unroll
        for (int j = 0; j < 16; ++j) sc[j] = (visible >> (8 * (j >> 2) + (j & 3))) & 1u ? sc[j] : -INFINITY;
    };
    // Running maximum over half a tile's scores; when some row must be re-based, moves every row's base to its current
    // maximum and returns true: o is then to be rescaled by alpha once the products already due are added.
    auto maxima = [&](const f32x16 &sc) __attribute__((always_inline)) {
        float mx = m_half;
#pragma unroll
        for (int j = 0; j < 16; ++j) mx = fmaxf(mx, sc[j]);
        m_half = mx;
        const bool due = __ballot(m_half > m_lazy) != 0;
        if (__builtin_expect(due, 0)) {
            const float m_row = halves_max(m_half);
            const float mc_new = m_row == -INFINITY ? -INFINITY : m_row * c2;
            m_lazy = m_row + lazy_raw;
            alpha = mc_new == -INFINITY ? 1.0f : exp2_fast(mc - mc_new);
            l_run *= alpha;
            mc = mc_new;
            mcx = mc_new == -INFINITY ? 0.0f : mc_new - kShift;
        }
        return due;
    };
    auto rescale = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t2 = 0; t2 < DT; ++t2) o[t2] *= alpha;
    };
    // Exponentials and terms of scores 2u and 2u + 1.
    float psum = 0.0f;
    auto softmax_unit = [&](auto unit, const f32x16 &sc, uint32_t (&pt)[2][8]) __attribute__((always_inline)) {
        constexpr int U = decltype(unit)::value;
        const float x = exp2_fast(fmaf(sc[2 * U], c2, -mcx)), y = exp2_fast(fmaf(sc[2 * U + 1], c2, -mcx));
        psum = U == 0 ? x + y : psum + (x + y);
        split_pair<false>(x, y, one, pt[0][U], pt[1][U]);
        __asm__ volatile("" : "+v"(psum), "+v"(pt[1][U])); // here, not where they are next used (behind the next group's branch)
    };

    // A whole step, both halves seen by this wave; MASKED applies the boundary masks to both.
    auto full_step = [&](auto masked, const int p, const int key0, const uint64_t bits) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
        constexpr int NS = 3 * KC, UNITS = 2 * CH; // MFMAs of Sᵀ; units of K, and of V
        h16x8 kl[KC], kh[KC], vl[DT], vh[DT];
        f32x16 sa{}, sb{};
        read_k(kl, p, 0, 1);
        read_k(kh, p, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<NS>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M * UNITS / NS, U1 = (M + 1) * UNITS / NS;
            score_mfma(m, sa, kl, kh);
            if constexpr (M == KC) read_k(kl, p, 1, 1);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) {
                split_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, kOfK, p ^ 1);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        read_k(kh, p, 1, 0);
        bool due = false;
        uint32_t pa[2][8];
        unrolled<NS>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, LEAD = 2; // MFMAs before the maxima
            score_mfma(m, sb, kl, kh);
            if constexpr (M == LEAD - 1) {
                if constexpr (MASKED) mask_scores(sa, key0, static_cast<uint32_t>(bits));
                if (__builtin_expect(maxima(sa), 0)) rescale();
            } else if constexpr (M >= LEAD) {
                constexpr int U0 = (M - LEAD) * 8 / (NS - LEAD), U1 = (M - LEAD + 1) * 8 / (NS - LEAD);
                unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) {
                    softmax_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, sa, pa);
                });
            }
            if constexpr (M == NS - 2) read_v(vl, p, 0, 0, 1);
            if constexpr (M == NS - 1) read_v(vh, p, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
        l_run += psum;
        unrolled<6>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value;
            output_mfma(m, pa, vl, vh);
            if constexpr (M % 3 == 0) read_v(vl, p, M / 3, 1 - M / 3, 1); // (half A, u = 1), then (half B, u = 0)
            if constexpr (M % 3 == 2) read_v(vh, p, M / 3, 1 - M / 3, 0);
            if constexpr (M == 0) {
                if constexpr (MASKED) mask_scores(sb, key0 + kTile, static_cast<uint32_t>(bits >> 32));
                due = maxima(sb);
            } else {
                constexpr int U0 = (M - 1) * 8 / 5, U1 = M * 8 / 5;
                unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) {
                    softmax_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, sb, ps);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        l_run += psum;
        if (__builtin_expect(due, 0)) rescale();
        unrolled<6>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value, U0 = M * UNITS / 6, U1 = (M + 1) * UNITS / 6;
            output_mfma(m, ps, vl, vh);
            if constexpr (M == 0) read_v(vl, p, 1, 1, 1);
            if constexpr (M == 2) read_v(vh, p, 1, 1, 0);
            unrolled<U1 - U0>([&](auto u) __attribute__((always_inline)) {
                split_unit(std::integral_constant<int, U0 + decltype(u)::value>{}, kOfV, p ^ 1);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // Half x of a tile alone.
    auto half_step = [&](const int p, const int x, const int key0, const uint32_t bits) __attribute__((always_inline)) {
        h16x8 kl[KC], kh[KC], vl[DT], vh[DT];
        f32x16 sc{};
        read_k(kl, p, x, 1);
        read_k(kh, p, x, 0);
        unrolled<3 * KC>([&](auto m) __attribute__((always_inline)) { score_mfma(m, sc, kl, kh); });
        mask_scores(sc, key0, bits);
        if (maxima(sc)) rescale();
        unrolled<8>([&](auto u) __attribute__((always_inline)) { softmax_unit(u, sc, ps); });
        l_run += psum;
        unrolled<6>([&](auto m) __attribute__((always_inline)) {
            constexpr int M = decltype(m)::value;
            if constexpr (M % 3 == 0) {
                read_v(vl, p, x, M / 3, 1);
                read_v(vh, p, x, M / 3, 0);
            }
            output_mfma(m, ps, vl, vh);
        });
    };
    auto split_rows = [&](const int p) __attribute__((always_inline)) {
        unrolled<2 * CH>([&](auto u) __attribute__((always_inline)) { split_unit(u, kOfK, p); });
        unrolled<2 * CH>([&](auto u) __attribute__((always_inline)) { split_unit(u, kOfV, p); });
    };

    if (nsteps > 0 && !unfit) {
        uint64_t bits0 = __ballot(mask0 != 0);
        clear_masked(bits0);
        split_rows(0);
        load_chunks(kraw, kbuf, kofs, kstep, 1);
        load_chunks(vraw, vbuf, vofs, vstep, 1);
        int mbyte = load_mask(1);
        auto step = [&](const int i, const int p) __attribute__((always_inline)) {
            __syncthreads(); // tile i is staged; every wave is done with the other stage
            const int key0 = tile_key(i);
            const bool live = i * KS + stream < ntiles && tile_valid && !own_unfit;
            const bool see_a = live && static_cast<uint32_t>(bits0) != 0 && key0 < last && key0 + kTile > first;
            const bool see_b = live && static_cast<uint32_t>(bits0 >> 32) != 0 && key0 + kTile < last && key0 + kStep > first;
            const bool inside = bits0 == ~0ull && tile_in_window(s, q0, key0) && tile_in_window(s, q0, key0 + kTile);
            const uint64_t bits1 = __ballot(mbyte != 0);
            clear_masked(bits1);
            if (__builtin_expect(see_a && see_b && inside, 1)) {
                full_step(std::integral_constant<bool, false>{}, p, key0, bits0);
            } else if (see_a && see_b) {
                full_step(std::integral_constant<bool, true>{}, p, key0, bits0);
            } else {
                if (see_a || see_b) {
                    const int x = see_a ? 0 : 1;
                    half_step(p, x, key0 + x * kTile, static_cast<uint32_t>(bits0 >> (32 * x)));
                }
                split_rows(p ^ 1);
            }
            load_chunks(kraw, kbuf, kofs, kstep, i + 2);
            load_chunks(vraw, vbuf, vofs, vstep, i + 2);
            mbyte = load_mask(i + 2);
            bits0 = bits1;
        };
        for (int i = 0; i < nsteps; i += 2) {
            step(i, 0);
            if (i + 1 < nsteps) step(i + 1, 1);
        }
    }

    float m_all = halves_max(m_half), mc_all = mc, l_all = l_run;
    if constexpr (KS > 1) {
        // Streams 1 .. KS - 1 hand (row maximum, sum, base, accumulators) to stream 0 through LDS, which adds them in
        // order, each rescaled to the largest base.
        float *const slots = reinterpret_cast<float *>(smem) + qi * (NREG * kWave) + lane;
        constexpr int SLOT = QB * NREG * kWave;
        __syncthreads(); // every wave is done with the stages
        if (stream > 0) {
            float *const slot = slots + (stream - 1) * SLOT;
            slot[0] = m_all;
            slot[kWave] = l_run;
            slot[2 * kWave] = mc;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) slot[(3 + 16 * t + j) * kWave] = o[t][j];
            }
        }
        __syncthreads();
        if (stream == 0) {
#pragma unroll
            for (int x = 0; x < KS - 1; ++x) {
                m_all = fmaxf(m_all, slots[x * SLOT]);
                mc_all = fmaxf(mc_all, slots[x * SLOT + 2 * kWave]);
            }
            const float base = mc_all == -INFINITY ? 0.0f : mc_all;
            const float a0 = exp2_fast(mc - base);
            l_all = l_run * a0;
#pragma unroll
            for (int t = 0; t < DT; ++t) o[t] *= a0;
#pragma unroll
            for (int x = 0; x < KS - 1; ++x) {
                const float *const slot = slots + x * SLOT;
                const float a = exp2_fast(slot[2 * kWave] - base);
                l_all = fmaf(slot[kWave], a, l_all);
#pragma unroll
                for (int t = 0; t < DT; ++t) {
#pragma unroll
                    for (int j = 0; j < 16; ++j) o[t][j] = fmaf(slot[(3 + 16 * t + j) * kWave], a, o[t][j]);
                }
            }
        }
    }

    bool redo = false;
    if (stream == 0 && tile_valid) {
        l_all = halves_sum(l_all); // each half-wave summed the exponentials of its own keys
        // A non-finite result: some input of the tile is not finite or out of its scale's range, or the result overflows.
        float probe = l_all * 0.0f, largest_o = 0.0f;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                probe = fmaf(o[t][j], 0.0f, probe);
                largest_o = fmaxf(largest_o, fabsf(o[t][j]));
            }
        }
        largest_o = halves_max(largest_o);
        const float base = mc_all == -INFINITY ? 0.0f : mc_all;
        // O is o / l in any offset; lse's sum is Σ exp(s - max) = l · exp2(offset - max·c2).
        const float sum = m_all == -INFINITY ? l_all : l_all * exp2_fast(base - kShift - m_all * c2);
        // A row that used only rows far below the ones that set the scales (hidden from it, or of no weight). Of V': where its terms
        // are below 2^-3 they are off by 2^-25, and so are weights below 2^-10 of the largest, here times at most 2^10 sampled.
        // Over a row of weights p / l these errors add up to at most 2^-25·√(Σ p²)/l, and Σ p² is at most l²/sum; so the row's
        // largest |O'| must reach 2^-3/√sum, as that of normal values does by 2^10 and more. Of K': an error of 2^-25 moves a
        // score by up to 2^-7·c2 (Q' below 2^15, errors of D features adding up at random), which must be below 2^-23, or the
        // row's largest |S'| at least 2^16, as where its keys are at 2^-2 or more.
        const bool faint = query < s.queries && ((!v_zero && 8.0f * largest_o * sqrtf(sum) < l_all) || (c2 > 0x1p-16f && fabsf(m_all) < 0x1p16f));
        redo = unfit || own_unfit || __ballot(probe != 0.0f || faint) != 0;
        if (__builtin_expect(!redo, 1)) store_rows<D, VEC>(P, seq, query, h, o, l_all, __builtin_amdgcn_ldexpf(m_all * P.scale, e), sum, ev);
    }
    if (stream == 0 && lane == 0) redone[qi] = redo;
    __syncthreads(); // also: every wave is done with the stages and the merged state
#pragma unroll 1
    for (int x = 0; x < QB; ++x) {
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(redone[x]), 0))
            exact_query_tile<D, VEC, QB * KS, WPE>((const SplitForwardParams *)__builtin_amdgcn_kernarg_segment_ptr(), (LdsFloats)smem, seq, (qb * QB + x) * kTile);
    }
}

namespace {

template<int D, bool VEC, int QB, int KS, int WPE = 2>
void launch(const ForwardArgs &a, hipStream_t stream) {
    const int64_t blocks = static_cast<int64_t>(a.batch) * a.heads * ((a.queries + QB * kTile - 1) / (QB * kTile));
    const SplitForwardParams params{Tensor{a.q, a.qs.batch, a.qs.head, a.qs.token}, Tensor{a.k, a.ks.batch, a.ks.head, a.ks.token},
            Tensor{a.v, a.vs.batch, a.vs.head, a.vs.token}, reinterpret_cast<const uint8_t *>(a.mask), a.output, a.os.batch, a.os.head,
            a.os.token, a.lse, Shape{a.batch, a.heads, a.queries, a.keys, a.radius, a.causal}, 1.0f / sqrtf(static_cast<float>(D))};
    hipLaunchKernelGGL((attention_forward_split_kernel<D, VEC, QB, KS, WPE>), dim3(static_cast<unsigned>(blocks)), dim3(kWave * QB * KS), 0,
            stream, params);
}

// Shape of the launch's work: sequences and their 32-query items, 32-key tiles of the widest item, and whether item costs run from
// one tile to many over much of the sequence.
struct Work {
    int64_t seqs, items;
    int tiles;
    bool ramp;
};

Work work_of(const ForwardArgs &a) {
    const Shape s{a.batch, a.heads, a.queries, a.keys, a.radius, a.causal};
    const int qtiles = (a.queries + kTile - 1) / kTile;
    const int64_t seqs = static_cast<int64_t>(a.batch) * a.heads;
    return Work{seqs, qtiles * seqs, std::max(forward_item_tiles(s, qtiles / 2), forward_item_tiles(s, qtiles - 1)),
            a.causal != 0 && (a.radius < 0 || a.radius >= a.queries / 2)};
}

} // namespace

// Workgroup shape. Every µs below: items, key tiles per item: this choice against the next best one.
//   * Up to two items per CU: two query tiles per workgroup, so that every CU has work, and as many key streams as LDS
//     holds (d = 64: 384, 32: 24.2 against 28.2 with four query tiles; d = 32, 512, 64: 24.1 with four streams, 28.0 with two;
//     384, 16: 10.7 both).
//   * Up to four items per CU: four query tiles and two streams if the items are long (d = 64: 768, 32: 29.7 against 32.4;
//     d = 32: 768, 32: 20.2 against 23.0), one if not (d = 64: 768, 8: 13.1 against 14.3). Under a ramp at d = 32 two and two
//     (768, up to 32: 16.9 against 20.0): the longest item ends sooner.
//   * Above that four query tiles and one stream (d = 32 held to three waves per SIMD: 3072, 32: 51.5 against 55.8), except
//     that a ramp up to eight items per CU keeps two streams (d = 64: 2048, up to 64: 68 against 74; d = 32: 2048, up to 128:
//     74 against 86): there all workgroups are resident at once and the longest ones would end alone. At d = 64 eight query
//     tiles split K and V half as often, and are taken where their workgroups fill whole rounds of the CUs (2048, 128: 195
//     against 209; 1536, 32: 47.0 against 51.5; but 3072, 32, one and a half rounds: 97 against 88).
SplitWorkgroup forward_split_workgroup(const int D, const ForwardArgs &a, const int cus) {
    const Work w = work_of(a);
    const bool ramp = w.ramp && a.radius < 0;
    if (w.items <= 2ll * cus) return D == 32 && w.tiles >= 20 ? SplitWorkgroup{2, 4} : SplitWorkgroup{2, 2};
    if (w.items <= 4ll * cus) {
        if (D == 32 && ramp) return SplitWorkgroup{2, 2};
        if (w.tiles >= (D == 32 ? 16 : 24)) return SplitWorkgroup{4, 2};
    } else if (ramp && w.items <= 8ll * cus && w.tiles >= (D == 32 ? 32 : 48)) {
        return SplitWorkgroup{4, 2};
    }
    const int64_t wide = w.seqs * ((a.queries + 8 * kTile - 1) / (8 * kTile));
    if (D == 64 && w.items > 4ll * cus && !ramp && a.radius < 0 && w.tiles >= 24 && (wide <= cus || wide >= 3ll * cus)) return SplitWorkgroup{8, 1};
    return SplitWorkgroup{4, 1};
}

namespace {

template<int D, bool VEC>
void dispatch(const ForwardArgs &a, const int cus, hipStream_t stream) {
    const SplitWorkgroup g = forward_split_workgroup(D, a, cus);
    if (g.tiles == 2) {
        if constexpr (D == 32) {
            if (g.streams == 4) return launch<D, VEC, 2, 4>(a, stream);
        }
        return launch<D, VEC, 2, 2, D == 32 ? 2 : 1>(a, stream); // d = 64: its 128 KB of LDS admit one workgroup per CU
    }
    if constexpr (D == 64) {
        if (g.tiles == 8) return launch<D, VEC, 8, 1>(a, stream);
    }
    if (g.streams == 2) return launch<D, VEC, 4, 2>(a, stream);
    launch<D, VEC, 4, 1, D == 32 ? 3 : 2>(a, stream);
}

} // namespace

// Where the FP32 kernel wins, from 7230 launches of 130 to 4096 items and 1 to 64 tiles on both kernels (µs: FP32 against this one;
// by this rule 3761 of them run here, 1.53 times as fast in the geometric mean, and three of those are slower than on the FP32 kernel by
// more than 3%, the worst by 5%):
//   * Few items, whose work its four waves per item and shorter start finish sooner: up to one item per CU (d = 64, 128 of 32: 23.4
//     against 24.6), up to two under a ramp, and above that short items (d = 64, 384 of 5: 12.6 against 12.5, of 8: 15.1 against
//     12.9; d = 32, 384 of 8: 9.2 against 9.4, of 12: 11.8 against 10.8) and sequences of odd query tiles that make more
//     workgroups than CUs (d = 64, 102 x 5 query tiles, 12: 24.1 against 29.9).
//   * Waves without a query tile, if they are more than a third (d = 64, 2048 x 1 query tile, 24: 164 against 218; d = 32, 600 x 1, 16:
//     21.3 against 37.8; but half of them for two query tiles of some keys: d = 64, 768 x 2, 8: 44.5 against 30.5).
//   * Launches of a tile or so per item, which are all start and end (d = 64, 1024 of 1: 9.0 against 9.8; d = 32, 600 of 1: 5.9
//     against 7.0, of 3: 8.2 both).
//   * At d = 32 its planned grid, up to three items per CU, also balances what a ramp or a window leaves uneven: while the ramp is
//     short (608 of up to 16: 11.4 against 12.0; 600 of 24: 15.9 both), or some waves are idle up to four per CU (900 of up to 5: 10.8
//     against 13.6), or the window's work is small (264 of 17: 11.1 against 13.7; 768 of 33: 33.2 against 23.8; and at d = 64 up
//     to two items per CU: 264 of 9: 13.2 against 14.5).
bool forward_split_pays(const int D, const ForwardArgs &a, const int cus) {
    const Work w = work_of(a);
    if (w.items <= (w.ramp ? 2ll : 1ll) * cus) return false;
    const int width = forward_split_workgroup(D, a, cus).tiles, qtiles = static_cast<int>(w.items / w.seqs);
    const int64_t groups = w.seqs * ((qtiles + width - 1) / width), waves = groups * width;
    if (2 * waves > 3 * w.items && (waves > 2 * w.items || qtiles != 2 || w.tiles < 5 || w.items <= 3ll * cus)) return false;
    if (w.items <= 2ll * cus)
        return groups <= cus && (a.radius < 0 ? w.tiles >= (D == 32 ? 9 : 8) : w.items * w.tiles >= (D == 32 ? 32ll : 18ll) * cus);
    if (D == 64) return w.tiles >= 2;
    if (w.ramp) return w.items <= 3ll * cus ? w.tiles >= 24 : w.items <= 4ll * cus ? w.tiles >= 4 && 10 * waves <= 11 * w.items : w.tiles >= 3;
    if (a.radius >= 0) return w.items <= 3ll * cus ? w.items * w.tiles >= 32ll * cus : w.tiles >= 5 || w.items >= 16ll * cus;
    return w.tiles >= (w.items <= 3ll * cus ? 5 : 2);
}

void launch_forward_split(const int D, const bool vec, const ForwardArgs &a, const int cus, hipStream_t stream) {
    if (D == 32) vec ? dispatch<32, true>(a, cus, stream) : dispatch<32, false>(a, cus, stream);
    else vec ? dispatch<64, true>(a, cus, stream) : dispatch<64, false>(a, cus, stream);
}

} // namespace rk
