// Softmax forward and backward over rows of any length and 2-byte alignment.
//
// A lane holds K chunks of eight elements, as in softmax.hip, so a row is read once and written once; the chunks are
// read and written with 16-byte accesses at whatever address they fall on (the memory path takes them unaligned: a
// wave's kilobyte touches nine 128-byte lines instead of eight). The last chunk of a row is read as the eight elements
// that end the row and shifted into place, so nothing beyond a row is read; it is written in pieces of 8, 4 and 2 bytes.
//
// Bounded by memory, as the aligned kernels are: [8, 12, 380, 1021] fp16 with a padding mask, forward 151 -> 28 us
// (149 MB of scores and probabilities), backward 113 -> 36 us (224 MB, 6.3 TB/s). Non-temporal accesses, as there, although
// the lines at the ends of a row are shared with its neighbours: [4, 16, 1000, 2047] forward 108 -> 100 us, backward 145
// -> 134. The scalar kernels (2-byte accesses, three passes over a row), which
// took these rows before, remain for rows of fewer than 8 or more than 16384 elements.
#include "softmax_ragged.hpp"

namespace nhp {

typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32_any __attribute__((aligned(2)));
typedef uint64_t u64_byte __attribute__((aligned(1)));

constexpr int64_t kMaxRaggedRow = 16384;

template <int L, int W>
struct RaggedGeo {
    static constexpr int kRowsPerWave = kWave / L;
    static constexpr int kRowsPerBlock = W > 1 ? 1 : 4 * kRowsPerWave;
};

// Elements [col, col + 8) of a row of n >= 8, those beyond n as zeros.
__device__ __forceinline__ u32x4 load_chunk(const uint16_t* row, uint32_t col, uint32_t n)
{
    const uint32_t at = min(col, n - 8);
    const u32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(row + at));
    if (col == at) return raw;
    uint64_t lo = (uint64_t)raw[1] << 32 | raw[0], hi = (uint64_t)raw[3] << 32 | raw[2];
    uint32_t shift = (col - at) * 16;   // 16 .. 112
    if (shift >= 64) {
        lo = hi;
        hi = 0;
        shift -= 64;
    }
    lo = lo >> shift | (hi << 1) << (63 - shift);
    hi >>= shift;
    return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

__device__ __forceinline__ void store_chunk(uint16_t* row, uint32_t col, uint32_t n, u32x4 v)
{
    uint16_t* p = row + col;
    const uint32_t left = n - col;
    if (left >= 8) {
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any*>(p));
        return;
    }
    if (left & 4) {
        *reinterpret_cast<u32x2_any*>(p) = u32x2{v[0], v[1]};
        p += 4;
        v[0] = v[2];
        v[1] = v[3];
    }
    if (left & 2) {
        *reinterpret_cast<u32_any*>(p) = v[0];
        p += 2;
        v[0] = v[1];
    }
    if (left & 1) *p = (uint16_t)v[0];
}

// Bit j set: mask byte col + j is 1, or col + j lies beyond the row or at or beyond key_end.
__device__ __forceinline__ uint32_t masked_bits(const uint8_t* row, uint32_t col, uint32_t n, uint32_t key_end)
{
    const uint32_t at = min(col, n - 8);
    const uint64_t raw = *reinterpret_cast<const u64_byte*>(row + at) >> ((col - at) * 8);
    uint32_t bits = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) bits |= ((uint32_t)(raw >> (8 * j)) & 0xffu) == 1u ? 1u << j : 0u;
    const uint32_t end = min(n, key_end);
    if (col + 8 > end) bits |= col >= end ? 0xffu : 0xffu << (end - col) & 0xffu;
    return bits;
}

// Bit j set: element e0 + j of the flat tensor is kept by the dropout (counted in aligned groups of eight).
__device__ __forceinline__ uint32_t kept_bits(const DropoutKey& dk, uint64_t e0)
{
    uint32_t bits = 0;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const Philox rnd = dropout_bits(dk, (e0 & ~(uint64_t)7) + 8 * g);
#pragma unroll
        for (int j = 0; j < 8; ++j) bits |= random16(rnd, j) < dk.threshold ? 1u << (8 * g + j) : 0u;
    }
    return bits >> (e0 & 7u) & 0xffu;
}

// MODE 0: causal (sliding window, key lengths), 1: padding mask; EXTRA: AliBi slopes, a bias tensor, dropout (any of them).
// In MODE 1 a row is taken for two heads in turn, so that its mask bytes are decoded once for both.
template <int DT, int MODE, bool EXTRA, int L, int K, int W>
__global__ void __launch_bounds__(256) ragged_fwd_kernel(RaggedArgs a)
{
    using G = RaggedGeo<L, W>;
    __shared__ float part_max[W], part_sum[W];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l = lane & (L - 1);
    const uint32_t n = a.n, np = a.np, sq = a.sq;
    constexpr uint32_t kHeads = MODE == 1 ? 2 : 1;
    const uint32_t hgs = (np + kHeads - 1) / kHeads;
    // unit (batch entry, head group, query); in MODE 0 that is the row itself
    const uint32_t units = MODE == 1 ? a.rows / np * hgs : a.rows;
    const uint32_t unit = W > 1 ? blockIdx.x : (blockIdx.x * 4 + wave) * G::kRowsPerWave + lane / L;
    const bool valid = unit < units;
    const uint32_t u = valid ? unit : units - 1;
    const uint32_t q = u % sq, hg = u / sq % hgs, bi = u / sq / hgs;
    const int w = W > 1 ? wave : 0;

    uint32_t lo = 0, hi = n;
    uint32_t skip[K];   // bit j: element j of the chunk is not read
    bool no_key = false;
    if constexpr (MODE == 0) {
        hi = min(q + 1, key_limit(a.key_lengths, bi, 1));
        lo = q > a.window ? q - a.window : 0;
        no_key = hi <= lo;   // only key lengths can empty a causal band: a uniform row
    }
    const uint32_t key_end = MODE == 1 ? key_limit(a.key_lengths, bi, 1) : 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
        skip[k] = 0xffu;
        if (col >= n) continue;
        if constexpr (MODE == 0) {
            if (col < hi && col + 8 > lo) {
                const uint32_t from = lo > col ? 0xffu << (lo - col) : 0xffu;
                const uint32_t to = hi - col < 8 ? (1u << (hi - col)) - 1u : 0xffu;
                skip[k] = ~(from & to) & 0xffu;
            }
        } else {
            skip[k] = masked_bits(a.mask + (uint64_t)(a.mask_per_batch ? bi * sq + q : q) * n, col, n, key_end);
        }
    }

    // rows of up to 1024 elements: the scores of both heads are asked for before those of the first are used (37.3 -> 35.2 us
    // at [4, 12, 1023, 1023], 34.8 -> 31.9 at [8, 12, 512, 701]; no gain with more chunks under way anyway)
    constexpr bool kBoth = MODE == 1 && K <= 2;
    u32x4 ahead[kBoth ? K : 1];
    auto fetch = [&](u32x4* to, uint32_t head) {
        const uint16_t* xr = a.in + ((uint64_t)(bi * np + head) * sq + q) * n;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            to[k] = u32x4{0, 0, 0, 0};
            if (skip[k] != 0xffu) to[k] = load_chunk(xr, (uint32_t)((k * W + w) * L + l) * 8u, n);
        }
    };
    const uint32_t head_end = min(np, hg * kHeads + kHeads);
    for (uint32_t head = hg * kHeads; head < head_end; ++head) {
        const uint64_t row = (uint64_t)(bi * np + head) * sq + q;
        uint16_t* yr = a.out + row * n;
        const uint16_t* br = EXTRA && a.bias ? a.bias + ((uint64_t)head * sq + q) * n : nullptr;
        float z[K][8];
        u32x4 raw[K];
        if (kBoth && head != hg * kHeads) {
#pragma unroll
            for (int k = 0; k < K; ++k) raw[k] = ahead[kBoth ? k : 0];
        } else {
            fetch(raw, head);
            if constexpr (kBoth) {
                if (head + 1 < head_end) fetch(ahead, head + 1);
            }
        }
        float m = kNegInf;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
            unpack8<DT>(raw[k], z[k]);
            if constexpr (EXTRA) {
                if (br && skip[k] != 0xffu) {
                    float f[8];
                    unpack8<DT>(load_chunk(br, col, n), f);
#pragma unroll
                    for (int j = 0; j < 8; ++j) z[k][j] = Half2<DT>::round(z[k][j] + f[j]);
                }
                if (a.slopes) {
                    const float slope = Half2<DT>::round(a.slopes[head]);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float dist = Half2<DT>::round(-(float)((int)q - (int)(col + j)));
                        const float z1 = Half2<DT>::round(z[k][j] + Half2<DT>::round(dist * slope));
                        z[k][j] = MODE == 0 || col + j <= q ? z1 : z[k][j];
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                // a masked element counts as -10000, one outside the band or the row not at all
                const float none = MODE == 1 && col + j < n ? kMaskFill : kNegInf;
                z[k][j] = skip[k] >> j & 1u ? none : z[k][j] * a.scale;
                m = fmaxf(m, z[k][j]);
            }
        }
        m = group_reduce<OpMax, L>(m);
        m = block_combine<OpMax, W>(m, part_max, wave, lane);
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
                const float e = exp2_raw(fmaf(z[k][j] - m, kLog2e, kExpBias));
                // (-inf scores in the band make -inf - -inf where the band holds nothing else, as they should)
                z[k][j] = (MODE == 0 ? skip[k] >> j & 1u : col + j >= n) ? 0.0f : e;
                sum += z[k][j];
            }
        sum = group_reduce<OpSum, L>(sum);
        sum = block_combine<OpSum, W>(sum, part_sum, wave, lane);
        const float inv = 1.0f / sum;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
            if (col >= n || !valid) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (MODE == 0) z[k][j] = no_key ? 1.0f / (float)n : skip[k] >> j & 1u ? 0.0f : z[k][j] * inv;
                else z[k][j] *= inv;
            }
            store_chunk(yr, col, n, pack8<DT>(z[k]));
            if (EXTRA && a.dropped) {
                const uint32_t keep = kept_bits(a.drop, row * n + col);
#pragma unroll
                for (int j = 0; j < 8; ++j) z[k][j] = keep >> j & 1u ? Half2<DT>::round(z[k][j]) * a.drop.scale : 0.0f;
                store_chunk(a.dropped + row * n, col, n, pack8<DT>(z[k]));
            }
        }
    }
}

// dx = scale * (dy * y - y * sum(dy * y)) within the band, zeros elsewhere. DROP: dy is the gradient of dropout(y); the
// kernel first forms keep * dy / (1 - p), rounded to the storage type as a separate dropout backward would store it.
template <int DT, bool CAUSAL, bool DROP, int L, int K, int W>
__global__ void __launch_bounds__(256) ragged_bwd_kernel(RaggedArgs a)
{
    using G = RaggedGeo<L, W>;
    __shared__ float part_sum[W];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l = lane & (L - 1);
    const uint32_t n = a.n;
    const uint32_t unit = W > 1 ? blockIdx.x : (blockIdx.x * 4 + wave) * G::kRowsPerWave + lane / L;
    const bool valid = unit < a.rows;
    const uint32_t row = valid ? unit : a.rows - 1;
    const int w = W > 1 ? wave : 0;
    uint32_t lo = 0, hi = n;
    if constexpr (CAUSAL) {
        const uint32_t q = row % a.sq;
        hi = min(q + 1, key_limit(a.key_lengths, row / a.sq, a.np));
        lo = q > a.window ? q - a.window : 0;
    }
    const uint64_t at = (uint64_t)row * n;
    u32x4 g[K], y[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
        g[k] = y[k] = u32x4{0, 0, 0, 0};
        if (col < hi && col + 8 > lo) {
            g[k] = load_chunk(a.in + at, col, n);
            y[k] = load_chunk(a.probs + at, col, n);
            if constexpr (DROP) {
                const uint32_t keep = kept_bits(a.drop, at + col);
                float f[8];
                unpack8<DT>(g[k], f);
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] = keep >> j & 1u ? f[j] * a.drop.scale : 0.0f;
                g[k] = pack8<DT>(f);
            }
        }
    }
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (CAUSAL) {   // elements outside the band count as zeros, whatever is stored there
                uint32_t keep = 0;
                if (col + 2 * i >= lo && col + 2 * i < hi) keep |= 0xffffu;
                if (col + 2 * i + 1 >= lo && col + 2 * i + 1 < hi) keep |= 0xffff0000u;
                g[k][i] &= keep;
                y[k][i] &= keep;
            }
            s = fmaf(Half2<DT>::lo(g[k][i]), Half2<DT>::lo(y[k][i]), s);
            s = fmaf(Half2<DT>::hi(g[k][i]), Half2<DT>::hi(y[k][i]), s);
        }
    }
    s = group_reduce<OpSum, L>(s);
    s = block_combine<OpSum, W>(s, part_sum, wave, lane);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t col = (uint32_t)((k * W + w) * L + l) * 8u;
        if (col >= n || !valid) continue;
        float f[8], p[8];
        unpack8<DT>(g[k], f);
        unpack8<DT>(y[k], p);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            f[j] = a.scale * fmaf(-p[j], s, f[j] * p[j]);
            if (CAUSAL && (col + j < lo || col + j >= hi)) f[j] = 0.0f;
        }
        store_chunk(a.out + at, col, n, pack8<DT>(f));
    }
}

bool ragged_rows(int64_t n) { return n >= 8 && n <= kMaxRaggedRow; }

// One wave per row up to 2048 elements (no barrier), four beyond; short rows share a wave. Three chunks per lane for 4099
// elements instead of four half empty: forward 54 -> 45 us at [2, 8, 700, 4099], backward 63 -> 55.
#define NHP_RAGGED_PLAN(CALL)                          \
    do {                                               \
        const uint32_t chunks = (a.n + 7) / 8;         \
        if (chunks <= 8) { CALL(8, 1, 1); }            \
        else if (chunks <= 16) { CALL(16, 1, 1); }     \
        else if (chunks <= 32) { CALL(32, 1, 1); }     \
        else if (chunks <= 64) { CALL(64, 1, 1); }     \
        else if (chunks <= 128) { CALL(64, 2, 1); }    \
        else if (chunks <= 192) { CALL(64, 3, 1); }    \
        else if (chunks <= 256) { CALL(64, 4, 1); }    \
        else if (chunks <= 512) { CALL(64, 2, 4); }    \
        else if (chunks <= 768) { CALL(64, 3, 4); }    \
        else if (chunks <= 1024) { CALL(64, 4, 4); }   \
        else if (chunks <= 1536) { CALL(64, 6, 4); }   \
        else { CALL(64, 8, 4); }                       \
    } while (0)

template <int L, int W>
static uint32_t ragged_blocks(uint32_t units)
{
    return (uint32_t)(((uint64_t)units + RaggedGeo<L, W>::kRowsPerBlock - 1) / RaggedGeo<L, W>::kRowsPerBlock);
}

template <int DT, int MODE>
static int ragged_fwd(const RaggedArgs& a, uint32_t units, hipStream_t st)
{
    const bool extra = a.slopes != nullptr || a.bias != nullptr || a.dropped != nullptr;
#define CALL(L_, K_, W_)                                                                                     \
    const uint32_t blocks = ragged_blocks<L_, W_>(units);                                                    \
    if (!grid_fits(blocks, 256)) return NHP_ERR_SHAPE;                                                       \
    if (extra) ragged_fwd_kernel<DT, MODE, true, L_, K_, W_><<<blocks, 256, 0, st>>>(a);                     \
    else ragged_fwd_kernel<DT, MODE, false, L_, K_, W_><<<blocks, 256, 0, st>>>(a)
    NHP_RAGGED_PLAN(CALL);
#undef CALL
    return launch_result();
}

template <int DT>
int ragged_causal_fwd(const RaggedArgs& a, hipStream_t st)
{
    return ragged_fwd<DT, 0>(a, a.rows, st);
}
template <int DT>
int ragged_masked_fwd(const RaggedArgs& a, hipStream_t st)
{
    return ragged_fwd<DT, 1>(a, a.rows / a.np * ((a.np + 1) / 2), st);
}

template <int DT, bool CAUSAL>
int ragged_bwd(const RaggedArgs& a, bool dropout, hipStream_t st)
{
#define CALL(L_, K_, W_)                                                 \
    const uint32_t blocks = ragged_blocks<L_, W_>(a.rows);               \
    if (!grid_fits(blocks, 256)) return NHP_ERR_SHAPE;                   \
    if (dropout) ragged_bwd_kernel<DT, CAUSAL, true, L_, K_, W_><<<blocks, 256, 0, st>>>(a);     \
    else ragged_bwd_kernel<DT, CAUSAL, false, L_, K_, W_><<<blocks, 256, 0, st>>>(a)
    NHP_RAGGED_PLAN(CALL);
#undef CALL
    return launch_result();
}

#define NHP_RAGGED_INSTANCES(DT)                                             \
    template int ragged_causal_fwd<DT>(const RaggedArgs&, hipStream_t);      \
    template int ragged_masked_fwd<DT>(const RaggedArgs&, hipStream_t);      \
    template int ragged_bwd<DT, true>(const RaggedArgs&, bool, hipStream_t);      \
    template int ragged_bwd<DT, false>(const RaggedArgs&, bool, hipStream_t);
NHP_RAGGED_INSTANCES(NHP_BF16)
NHP_RAGGED_INSTANCES(NHP_F16)

}  // namespace nhp
