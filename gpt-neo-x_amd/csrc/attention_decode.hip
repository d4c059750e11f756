// Attention of a few new positions over cached ones, and the cache's next state, in one pass over the cache.
//
// A decoding step has to read the cached keys and values and write them, with the new ones, into the tensor that the
// caller keeps (its next `layer_past`). Concatenating keys, values and the pair of them in torch and then attending moved
// every key and value seven times; here a wave loads 32 keys and values, stores them to the new cache and multiplies
// them while it has them, so they are read once and written once. That traffic is the bound; the matrix instructions and
// the softmax take a tenth of its time.
//
// Rows of the matrix instruction (16 x 16 x 32) are keys, its columns the queries that share a key/value head (new positions
// x heads of the group, at most 32). A workgroup is four waves, each with 32 keys at a time, which share nothing until the
// end, where their sums are merged. Keys go from memory into the registers in the order in which the instruction wants them
// (16 rows x 64 bytes per load); values are transposed through LDS, whose rows are padded so that the 8 rows of a transposing
// read fall on different banks. The next 32 keys and values are on their way while the wave stores and multiplies these.
//
// Split. What the memory rewards is one workgroup on every CU and long runs of addresses. So where there are many (batch entry,
// key/value head) pairs the waves of a workgroup take two or four neighbouring heads, whose rows of a position lie side by
// side, and with fewer of them the keys of a pair are cut into parts, which a second kernel merges (decode_plan).
//
// Measured (us, bf16, without the prefetch and with one head per workgroup before; copy: read and written bytes at 5.1 TB/s):
//   16 sequences of 2047, 32 heads of 128      221 -> 204 (copy 210)     32 of 1000, 32 heads of 128   221 -> 192 (206)
//   32 of 2000, 8 heads of keys of 128          90 -> 85 (103)           20 of 2000, 32 heads of 80    328 -> 231 (161)
//   9 of 2000, 32 heads of 128                 163 -> 119 (116)          5 of 3000, 32 heads of 128    119 -> 91 (96)
//   1 of 8000, 32 heads of 128                  58 -> 57 (51)            4 of 300, 8 heads of keys      14 -> 11 (2)
// (Concatenations 949 us and attention 118 us for the first of them, before there was such a kernel.)
#include "attention.hpp"

namespace nhp {

typedef uint32_t u32_byte __attribute__((aligned(1)));

struct AttnDecodeArgs {
    const uint16_t *q, *k_new, *v_new, *k_past, *v_past;
    uint16_t *k_out, *v_out, *o;
    const uint8_t* mask;
    float *part_o, *part_ml;   // with splits > 1: [split][pair][row][hd] and [split][pair][row][2]
    int64_t q_s, q_b, q_h, kn_s, kn_b, kn_h, vn_s, vn_b, vn_h, kp_s, kp_b, kp_h, vp_s, vp_b, vp_h;
    int64_t out_s, out_b, out_h, o_s, o_b, o_h, mask_b, mask_q;
    float scale_log2, fill_log2;
    int batch, kv_heads, group, sq, past, splits, keys_per_split, heads_per_block;
};

struct Yes {
    static constexpr bool value = true;
};
struct No {
    static constexpr bool value = false;
};

// Combines the lanes l, l ^ 16, l ^ 32, l ^ 48.
template <typename Op>
__device__ __forceinline__ float reduce_columns(float v)
{
    const auto r = __builtin_amdgcn_permlane16_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    v = Op::apply(bitcast<float>((uint32_t)r[0]), bitcast<float>((uint32_t)r[1]));
    const auto s = __builtin_amdgcn_permlane32_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    return Op::apply(bitcast<float>((uint32_t)s[0]), bitcast<float>((uint32_t)s[1]));
}

template <int HD>
struct DecodeGeo {
    static constexpr int kChunks = HD / 8;
    static constexpr int kSteps = (HD + 31) / 32;          // matrix instructions along the features of q k^T
    static constexpr int kLoads = 32 * kChunks / 64;       // 16-byte loads per lane for 32 values
    static constexpr int kTiles = HD / 16;                 // 16-feature tiles of the result
    static constexpr int kRowBytes = HD == 80 ? 160 : HD * 2 + 32;   // 40, 40, 56, 72 words: 8 rows on different banks
    static constexpr int kSumRow = HD + 4;                 // floats of a row of sums in LDS
    static constexpr int kValueBytes = 32 * kRowBytes, kSumBytes = 16 * kSumRow * 4;
    static constexpr int kWaveBytes = kValueBytes > kSumBytes ? kValueBytes : kSumBytes;
};

// NQ: tiles of 16 queries; NH: key/value heads of a workgroup, one or several waves each. (With two tiles of queries the
// registers for what is on its way are there for one workgroup per CU only.)
template <int DT, int HD, int NQ, int NH>
__global__ void __launch_bounds__(256, NQ == 1 ? 2 : 1) attn_decode_kernel(AttnDecodeArgs a)
{
    using G = DecodeGeo<HD>;
    constexpr int kKeyWaves = 4 / NH, kKeys = 32 * kKeyWaves;   // waves that share a head's keys, and what they take in a round
    __shared__ __attribute__((aligned(1024))) char lds[4 * G::kWaveBytes];
    __shared__ float wave_m[4][NQ * 16], wave_l[4][NQ * 16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int pairs = a.batch * a.kv_heads;
    const int groups = pairs / NH, pair0 = blockIdx.x % groups * NH;
    const int pair = pair0 + wave % NH, split = blockIdx.x / groups;
    const int b = pair / a.kv_heads, hk = pair % a.kv_heads;
    const int rows = a.sq * a.group, sk = a.past + a.sq;
    const int key_lo = split * a.keys_per_split, key_hi = min(sk, key_lo + a.keys_per_split);

    u32x4 qf[NQ][G::kSteps];
    const uint8_t* mrow[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int row = min(n * 16 + r16, rows - 1), s = row / a.group, h = hk * a.group + row % a.group;
        const uint16_t* qp = a.q + s * a.q_s + b * a.q_b + h * a.q_h;
        mrow[n] = a.mask + b * a.mask_b + s * a.mask_q;
#pragma unroll
        for (int t = 0; t < G::kSteps; ++t) qf[n][t] = 4 * t + g < G::kChunks ? load16(qp + (4 * t + g) * 8) : u32x4{0, 0, 0, 0};
    }

    const uint16_t* kp = a.k_past + b * a.kp_b + hk * a.kp_h;
    const uint16_t* vp = a.v_past + b * a.vp_b + hk * a.vp_h;
    const uint16_t* kn = a.k_new + b * a.kn_b + hk * a.kn_h;
    const uint16_t* vn = a.v_new + b * a.vn_b + hk * a.vn_h;
    uint16_t* ko = a.k_out + b * a.out_b + hk * a.out_h;
    uint16_t* vo = a.v_out + b * a.out_b + hk * a.out_h;
    char* const mine = lds + wave * G::kWaveBytes;
    const int tr = (4 * g + (r16 >> 2)) * G::kRowBytes + (r16 & 3) * 8;
    // element offsets within 32 keys: 32-bit, so that a load takes them beside a base that the whole wave shares
    const uint32_t kps = (uint32_t)a.kp_s, vps = (uint32_t)a.vp_s, outs = (uint32_t)a.out_s;
    auto value_row = [&](int i) { return (uint32_t)(i * 64 + lane) / G::kChunks; };
    auto value_col = [&](int i) { return (uint32_t)(i * 64 + lane) % G::kChunks * 8; };
    // the i-th 64 chunks of 32 values of row stride `st`: where whole rows make up 64 chunks the base moves, not the lane
    auto value_at = [&](auto* base, uint32_t st, int i) {
        if constexpr (64 % G::kChunks == 0) return base + (uint64_t)(i * (64 / G::kChunks)) * st + (value_row(0) * st + value_col(0));
        else return base + (value_row(i) * st + value_col(i));
    };

    f32x4 o[NQ][G::kTiles];
    float m[NQ], l[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        m[n] = kFarBelow;
        l[n] = 0.0f;
#pragma unroll
        for (int d = 0; d < G::kTiles; ++d) o[n][d] = f32x4{};
    }

    // bytes 4 g .. 4 g + 3 of each 16 keys of this lane's query; the last ones of a row are read as the four bytes that end it
    auto read_mask = [&](int key0, uint32_t (&hidden)[NQ][2]) {
#pragma unroll
        for (int n = 0; n < NQ; ++n)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) {
                const int key = key0 + t2 * 16 + 4 * g, at = min(key, sk - 4);
                const uint32_t w = *reinterpret_cast<const u32_byte*>(mrow[n] + at);
                hidden[n][t2] = key - at < 4 ? w >> (8 * (key - at)) : 0u;
            }
    };
    using Keys = u32x4[2][G::kSteps];
    using Values = u32x4[G::kLoads];
    using Hidden = uint32_t[NQ][2];
    // 32 cached keys and values
    auto load = [&](int key0, Keys& kf, Values& vf, Hidden& hidden) {
        // opaque, so that the addresses are formed here as base + lane offset; kept as running pointers, one for each
        // access, they would not fit into the registers
        asm volatile("" : "+s"(key0));
        const uint16_t *kt = kp + (int64_t)key0 * a.kp_s, *vt = vp + (int64_t)key0 * a.vp_s;
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
            for (int t = 0; t < G::kSteps; ++t)
                kf[t2][t] = 4 * t + g < G::kChunks ? load16(kt + (uint64_t)(t2 * 16) * kps + t * 32 + (r16 * kps + g * 8)) : u32x4{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < G::kLoads; ++i) vf[i] = load16_stream(value_at(vt, vps, i));
        read_mask(key0, hidden);
        asm volatile("" ::: "memory");   // not put off until they are needed
    };
    // the last ones: cached, new, or beyond the end (the last one again)
    auto load_last = [&](int key0, Keys& kf, Values& vf, Hidden& hidden) {
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            const int key = min(key0 + t2 * 16 + r16, sk - 1);
            const uint16_t* p = key < a.past ? kp + key * a.kp_s : kn + (key - a.past) * a.kn_s;
#pragma unroll
            for (int t = 0; t < G::kSteps; ++t) kf[t2][t] = 4 * t + g < G::kChunks ? load16(p + (4 * t + g) * 8) : u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < G::kLoads; ++i) {
            const int key = min(key0 + (int)value_row(i), sk - 1);
            vf[i] = load16((key < a.past ? vp + key * a.vp_s : vn + (key - a.past) * a.vn_s) + value_col(i));
        }
        read_mask(key0, hidden);
    };
    // Stores and multiplies them; `whole`: all 32 exist.
    auto use = [&](auto whole, int key0, Keys& kf, Values& vf, Hidden& hidden) {
        constexpr bool kWhole = decltype(whole)::value;
        asm volatile("" : "+s"(key0));
        uint16_t *kd = ko + (int64_t)key0 * a.out_s, *vd = vo + (int64_t)key0 * a.out_s;
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            if (!kWhole && key0 + t2 * 16 + r16 >= key_hi) continue;
#pragma unroll
            for (int t = 0; t < G::kSteps; ++t)
                if (4 * t + g < G::kChunks) *reinterpret_cast<u32x4*>(kd + (uint64_t)(t2 * 16) * outs + t * 32 + (r16 * outs + g * 8)) = kf[t2][t];
        }
        // the values of the previous round have been read by all lanes (their results were waited for)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < G::kLoads; ++i) {
            *reinterpret_cast<u32x4*>(mine + value_row(i) * G::kRowBytes + value_col(i) * 2) = vf[i];
            if (kWhole || key0 + (int)value_row(i) < key_hi) store16_stream(value_at(vd, outs, i), vf[i]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        u32x4 pf[NQ];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            f32x4 s[2] = {f32x4{}, f32x4{}};
#pragma unroll
            for (int t = 0; t < G::kSteps; ++t)
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2) s[t2] = mma16<DT>(kf[t2][t], qf[n][t], s[t2]);
            float mx = kNegInf;
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = key0 + t2 * 16 + 4 * g + i;
                    float x = hidden[n][t2] >> (8 * i) & 0xffu ? a.fill_log2 : s[t2][i] * a.scale_log2;
                    if (!kWhole) x = key < key_hi ? x : kNegInf;
                    s[t2][i] = x;
                    mx = fmaxf(mx, x);
                }
            mx = reduce_columns<OpMax>(mx);
            if (__any(mx > m[n] + kLazy)) {
                const float mn = fmaxf(m[n], mx), alpha = exp2_raw(m[n] - mn);
                m[n] = mn;
                l[n] *= alpha;
#pragma unroll
                for (int d = 0; d < G::kTiles; ++d)
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[n][d][i] *= alpha;
            }
            float sum = 0.0f;
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[t2][i] = exp2_raw(s[t2][i] - m[n]);
                    sum += s[t2][i];
                }
            l[n] += sum;
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                for (int i = 0; i < 2; ++i) pf[n][2 * t2 + i] = Half2<DT>::pack(s[t2][2 * i], s[t2][2 * i + 1]);
        }
#pragma unroll
        for (int d = 0; d < G::kTiles; ++d) {
            const u32x4 vt = lds_read_tr(mine + tr + d * 32, mine + tr + d * 32 + 16 * G::kRowBytes);
#pragma unroll
            for (int n = 0; n < NQ; ++n) o[n][d] = mma16<DT>(vt, pf[n], o[n][d]);
        }
    };
    int key0 = key_lo + wave / NH * 32;
    const int last_whole = min(a.past, key_hi) - 32;
    Keys kf[2];
    Values vf[2];
    Hidden hidden[2];
    if (key0 <= last_whole) {
        load(key0, kf[0], vf[0], hidden[0]);
        for (;;) {
            if (key0 + kKeys <= last_whole) load(key0 + kKeys, kf[1], vf[1], hidden[1]);
            use(Yes{}, key0, kf[0], vf[0], hidden[0]);
            key0 += kKeys;
            if (key0 > last_whole) break;
            if (key0 + kKeys <= last_whole) load(key0 + kKeys, kf[0], vf[0], hidden[0]);
            use(Yes{}, key0, kf[1], vf[1], hidden[1]);
            key0 += kKeys;
            if (key0 > last_whole) break;
        }
    }
    for (; key0 < key_hi; key0 += kKeys) {
        load_last(key0, kf[0], vf[0], hidden[0]);
        use(No{}, key0, kf[0], vf[0], hidden[0]);
    }

    // the four waves' sums, 16 queries at a time
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        l[n] = reduce_columns<OpSum>(l[n]);
        if (g == 0) {
            wave_m[wave][n * 16 + r16] = m[n];
            wave_l[wave][n * 16 + r16] = l[n];
        }
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        __syncthreads();
        float* sums = reinterpret_cast<float*>(mine);
#pragma unroll
        for (int d = 0; d < G::kTiles; ++d) *reinterpret_cast<f32x4*>(sums + r16 * G::kSumRow + d * 16 + 4 * g) = o[n][d];
        __syncthreads();
        for (int item = tid; item < NH * 256; item += 256) {
            const int hh = item >> 8, r = (item >> 4) & 15, c = item & 15, row = n * 16 + r;
            if (c >= G::kChunks || row >= rows) continue;
            const int pr = pair0 + hh, b2 = pr / a.kv_heads, hk2 = pr % a.kv_heads;
            float big = kFarBelow, total = 0.0f, acc[8] = {};
#pragma unroll
            for (int w = 0; w < kKeyWaves; ++w) big = fmaxf(big, wave_m[w * NH + hh][row]);
#pragma unroll
            for (int w = 0; w < kKeyWaves; ++w) {
                const float f = exp2_raw(wave_m[w * NH + hh][row] - big);
                total = fmaf(wave_l[w * NH + hh][row], f, total);
                const float* p = reinterpret_cast<const float*>(lds + (w * NH + hh) * G::kWaveBytes) + r * G::kSumRow + c * 8;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[j] = fmaf(p[j], f, acc[j]);
            }
            if (a.splits == 1) {
                const float inv = 1.0f / total;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[j] *= inv;
                uint16_t* op = a.o + row / a.group * a.o_s + b2 * a.o_b + (hk2 * a.group + row % a.group) * a.o_h;
                *reinterpret_cast<u32x4*>(op + c * 8) = pack8<DT>(acc);
            } else {
                const int64_t at = ((int64_t)split * pairs + pr) * rows + row;
                *reinterpret_cast<f32x4*>(a.part_o + at * HD + c * 8) = f32x4{acc[0], acc[1], acc[2], acc[3]};
                *reinterpret_cast<f32x4*>(a.part_o + at * HD + c * 8 + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
                if (c == 0) *reinterpret_cast<f32x2*>(a.part_ml + at * 2) = f32x2{big, total};
            }
        }
    }
}

// Merges the workgroups of each pair: 16 lanes per query.
template <int DT, int HD>
__global__ void __launch_bounds__(256) attn_decode_merge_kernel(AttnDecodeArgs a)
{
    const int rows = a.sq * a.group, pairs = a.batch * a.kv_heads;
    const int64_t at0 = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4), count = (int64_t)pairs * rows;
    const int c = threadIdx.x & 15;
    if (at0 >= count || c >= HD / 8) return;
    float big = kFarBelow, total = 0.0f, acc[8] = {};
    for (int s = 0; s < a.splits; ++s) big = fmaxf(big, a.part_ml[(s * count + at0) * 2]);
    for (int s = 0; s < a.splits; ++s) {
        const int64_t at = s * count + at0;
        const float f = exp2_raw(a.part_ml[at * 2] - big);
        total = fmaf(a.part_ml[at * 2 + 1], f, total);
        const f32x4 x = *reinterpret_cast<const f32x4*>(a.part_o + at * HD + c * 8);
        const f32x4 y = *reinterpret_cast<const f32x4*>(a.part_o + at * HD + c * 8 + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[j] = fmaf(x[j], f, acc[j]);
            acc[4 + j] = fmaf(y[j], f, acc[4 + j]);
        }
    }
    const float inv = 1.0f / total;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] *= inv;
    const int row = (int)(at0 % rows), pair = (int)(at0 / rows), b = pair / a.kv_heads, hk = pair % a.kv_heads;
    uint16_t* op = a.o + row / a.group * a.o_s + b * a.o_b + (hk * a.group + row % a.group) * a.o_h;
    *reinterpret_cast<u32x4*>(op + c * 8) = pack8<DT>(acc);
}

// keys (k_out[key, b, h] = past or new) and values (blockIdx.y 1), 16 bytes per thread
struct CacheArgs {
    const uint16_t *k_new, *v_new, *k_past, *v_past;
    uint16_t* out;   // [2, past + sq, batch, kv_heads, hd]
    int64_t kn_s, kn_b, kn_h, vn_s, vn_b, vn_h, kp_s, kp_b, kp_h, vp_s, vp_b, vp_h;
    int batch, kv_heads, past, chunks;
    int64_t items;   // 16-byte chunks of the keys
};

__global__ void __launch_bounds__(256) cache_append_kernel(CacheArgs a)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.items) return;
    const bool value = blockIdx.y != 0;
    const int c = (int)(i % a.chunks);
    const uint32_t head = (uint32_t)(i / a.chunks);   // (position, batch entry, head)
    const uint32_t h = head % a.kv_heads, b = head / a.kv_heads % a.batch;
    const int64_t s = head / a.kv_heads / a.batch;
    const uint16_t* p;
    if (s < a.past) p = value ? a.v_past + s * a.vp_s + b * a.vp_b + h * a.vp_h : a.k_past + s * a.kp_s + b * a.kp_b + h * a.kp_h;
    else p = value ? a.v_new + (s - a.past) * a.vn_s + b * a.vn_b + h * a.vn_h : a.k_new + (s - a.past) * a.kn_s + b * a.kn_b + h * a.kn_h;
    *reinterpret_cast<u32x4*>(a.out + (value ? a.items * 8 : 0) + i * 8) = load16(p + c * 8);
}

// Heads of a workgroup and workgroups of a pair of batch entry and key/value head.
//
// Heads: four or two where that leaves about one workgroup for each CU (1024 pairs of 128 features, 4 / 2 / 1 heads: 192 / 212
// / 217 us, 768: 161 / 164 / 172, 512: 199 / 204 / 221, of which the first needs a second kernel, 384: 165 / 162 / 171, 288: 147
// / 125 / 121), earlier where rows of 160 or 192 bytes end within a cache line (640 pairs of 80 features: 231 / 251 / 304).
//
// Workgroups: few, but so many that they go evenly on 256 CUs, with 256 keys at least (128 where there are less workgroups than
// CUs). More of them cost the cache's bandwidth and the second kernel (256 pairs of 2000 keys: 85 us with one each, 89 with two;
// 12 pairs of 200 keys: 6.2, 7.4), uneven ones leave CUs idle (288 pairs: 154 us with one each, 130 with two, 121 with four;
// 160: 115 with two, 96 with four; 32 of 300: 14 with two, 11 with three).
struct DecodePlan {
    int heads_per_block, splits, keys_per_split;
};
static DecodePlan decode_plan(int64_t batch, int64_t kv_heads, int64_t rows, int64_t sk, int64_t hd)
{
    const int64_t pairs = batch * kv_heads;
    const bool whole_lines = hd % 64 == 0;
    int heads = 1;
    if (rows <= 16 && kv_heads % 4 == 0 && pairs >= (whole_lines ? 640 : 512)) heads = 4;
    else if (rows <= 16 && kv_heads % 2 == 0 && pairs >= 384) heads = 2;
    const int64_t groups = pairs / heads, most = sk <= 256 ? 1 : (sk + 127) / 128;
    int64_t splits = 1, best = 0;
    for (int64_t s = 1; s <= most && s <= 256; ++s) {
        const int64_t blocks = groups * s, rounds = (blocks + 255) / 256;
        if (s > 1 && rounds > 1 && sk < s * 256) break;
        // rounds of workgroups against their number (192 of them, or 160 with four heads, need no second kernel), and in
        // hundredths 3 for the second kernel and 1 for each split
        const bool full = s == 1 && rounds == 1 && blocks >= (heads == 4 ? 160 : 192);
        const int64_t cost = (full ? 1000 : rounds * 256 * 1000 / blocks) * (100 + (s > 1 ? 3 + s : 0));
        if (s == 1 || cost < best) {
            best = cost;
            splits = s;
        }
    }
    const int64_t keys = ((sk + splits - 1) / splits + 127) / 128 * 128;
    return {heads, (int)((sk + keys - 1) / keys), (int)keys};   // no empty split
}

template <int DT, int HD>
static int launch_decode(const AttnDecodeArgs& a, hipStream_t st)
{
    const int64_t pairs = (int64_t)a.batch * a.kv_heads, grid = pairs / a.heads_per_block * a.splits, rows = (int64_t)a.sq * a.group;
    if (!grid_fits(grid, 256) || !grid_fits((pairs * rows + 15) / 16, 256)) return NHP_ERR_SHAPE;
    launch_prepare();
    if (rows > 16) attn_decode_kernel<DT, HD, 2, 1><<<dim3((unsigned)grid), dim3(256), 0, st>>>(a);
    else if (a.heads_per_block == 1) attn_decode_kernel<DT, HD, 1, 1><<<dim3((unsigned)grid), dim3(256), 0, st>>>(a);
    else if (a.heads_per_block == 2) attn_decode_kernel<DT, HD, 1, 2><<<dim3((unsigned)grid), dim3(256), 0, st>>>(a);
    else attn_decode_kernel<DT, HD, 1, 4><<<dim3((unsigned)grid), dim3(256), 0, st>>>(a);
    if (a.splits > 1) attn_decode_merge_kernel<DT, HD><<<dim3((unsigned)((pairs * rows + 15) / 16)), dim3(256), 0, st>>>(a);
    return launch_result();
}

template <int DT>
static int launch_decode_hd(const AttnDecodeArgs& a, int64_t hd, hipStream_t st)
{
    switch (hd) {
    case 64: return launch_decode<DT, 64>(a, st);
    case 80: return launch_decode<DT, 80>(a, st);
    case 96: return launch_decode<DT, 96>(a, st);
    case 128: return launch_decode<DT, 128>(a, st);
    }
    return NHP_ERR_SHAPE;
}

static bool decode_sizes_ok(int64_t batch, int64_t heads, int64_t kv_heads, int64_t sq, int64_t past, int64_t hd)
{
    if (batch <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || sq <= 0 || past < 0 || hd <= 0 || hd % 8) return false;
    if (sq > (1 << 24) || past > (1 << 24) || batch > (1 << 24) || heads > (1 << 24)) return false;
    return batch * heads <= (1 << 24) && (past + sq) * batch * kv_heads < ((int64_t)1 << 31) && batch * kv_heads * hd < (1 << 24);
}

}  // namespace nhp

extern "C" {

int64_t nhp_attention_decode_workspace_bytes(int64_t batch, int64_t heads, int64_t kv_heads, int64_t sq, int64_t past, int64_t head_dim)
{
    using namespace nhp;
    if (!decode_sizes_ok(batch, heads, kv_heads, sq, past, head_dim)) return 0;
    const int64_t splits = decode_plan(batch, kv_heads, sq * (heads / kv_heads), past + sq, head_dim).splits;
    return splits == 1 ? 0 : splits * batch * heads * sq * (head_dim + 2) * 4;
}

int nhp_attention_decode(void* out, void* cache_out, const void* q, const void* k_new, const void* v_new, const void* k_past,
                         const void* v_past, const void* mask, int64_t mask_batch_stride, int64_t mask_row_stride, float mask_fill,
                         void* workspace, float scale, int64_t batch, int64_t heads, int64_t kv_heads, int64_t sq, int64_t past,
                         int64_t head_dim, const int64_t* out_strides, const int64_t* q_strides, const int64_t* k_new_strides,
                         const int64_t* v_new_strides, const int64_t* k_past_strides, const int64_t* v_past_strides, int dtype,
                         void* stream)
{
    using namespace nhp;
    if (!out || !cache_out || !q || !k_new || !v_new || !k_past || !v_past || !mask) return NHP_ERR_NULL;
    for (const int64_t* s : {out_strides, q_strides, k_new_strides, v_new_strides, k_past_strides, v_past_strides})
        if (!s) return NHP_ERR_NULL;
    if (!decode_sizes_ok(batch, heads, kv_heads, sq, past, head_dim) || past < 1 || past + sq < 4) return NHP_ERR_SHAPE;
    if (sq * (heads / kv_heads) > 32 || !(scale > 0.0f) || mask_batch_stride < 0 || mask_row_stride < 0) return NHP_ERR_SHAPE;
    if (!ptr_aligned16(cache_out)) return NHP_ERR_SHAPE;
    AttnDecodeArgs a{};
    const uint16_t* o;
    int rc = fill_operand(o, a.o_s, a.o_b, a.o_h, out, out_strides);
    if (rc == NHP_OK) rc = fill_operand(a.q, a.q_s, a.q_b, a.q_h, q, q_strides);
    if (rc == NHP_OK) rc = fill_operand(a.k_new, a.kn_s, a.kn_b, a.kn_h, k_new, k_new_strides);
    if (rc == NHP_OK) rc = fill_operand(a.v_new, a.vn_s, a.vn_b, a.vn_h, v_new, v_new_strides);
    if (rc == NHP_OK) rc = fill_operand(a.k_past, a.kp_s, a.kp_b, a.kp_h, k_past, k_past_strides);
    if (rc == NHP_OK) rc = fill_operand(a.v_past, a.vp_s, a.vp_b, a.vp_h, v_past, v_past_strides);
    if (rc != NHP_OK) return rc;
    a.o = static_cast<uint16_t*>(out);
    const int64_t sk = past + sq;
    a.out_s = batch * kv_heads * head_dim;
    a.out_b = kv_heads * head_dim;
    a.out_h = head_dim;
    a.k_out = static_cast<uint16_t*>(cache_out);
    a.v_out = a.k_out + sk * a.out_s;
    a.mask = static_cast<const uint8_t*>(mask);
    a.mask_b = mask_batch_stride;
    a.mask_q = mask_row_stride;
    a.scale_log2 = scale * kLog2e;
    a.fill_log2 = fmaxf(mask_fill * kLog2e, -1e30f);
    a.batch = (int)batch;
    a.kv_heads = (int)kv_heads;
    a.group = (int)(heads / kv_heads);
    a.sq = (int)sq;
    a.past = (int)past;
    const DecodePlan plan = decode_plan(batch, kv_heads, sq * a.group, sk, head_dim);
    a.splits = plan.splits;
    a.keys_per_split = plan.keys_per_split;
    a.heads_per_block = plan.heads_per_block;
    if (a.splits > 1) {
        if (!workspace || !ptr_aligned16(workspace)) return NHP_ERR_NULL;
        a.part_o = static_cast<float*>(workspace);
        a.part_ml = a.part_o + a.splits * batch * heads * sq * head_dim;
    }
    if (dtype == NHP_BF16) return launch_decode_hd<NHP_BF16>(a, head_dim, static_cast<hipStream_t>(stream));
    if (dtype == NHP_F16) return launch_decode_hd<NHP_F16>(a, head_dim, static_cast<hipStream_t>(stream));
    return NHP_ERR_DTYPE;
}

int nhp_kv_cache_append(void* cache_out, const void* k_new, const void* v_new, const void* k_past, const void* v_past, int64_t batch,
                        int64_t kv_heads, int64_t sq, int64_t past, int64_t head_dim, const int64_t* k_new_strides,
                        const int64_t* v_new_strides, const int64_t* k_past_strides, const int64_t* v_past_strides, int dtype,
                        void* stream)
{
    using namespace nhp;
    if (!cache_out || !k_new || !v_new || !k_new_strides || !v_new_strides) return NHP_ERR_NULL;
    if (past > 0 && (!k_past || !v_past || !k_past_strides || !v_past_strides)) return NHP_ERR_NULL;
    if (dtype != NHP_BF16 && dtype != NHP_F16) return NHP_ERR_DTYPE;
    if (!decode_sizes_ok(batch, kv_heads, kv_heads, sq, past, head_dim) || !ptr_aligned16(cache_out)) return NHP_ERR_SHAPE;
    CacheArgs a{};
    int rc = fill_operand(a.k_new, a.kn_s, a.kn_b, a.kn_h, k_new, k_new_strides);
    if (rc == NHP_OK) rc = fill_operand(a.v_new, a.vn_s, a.vn_b, a.vn_h, v_new, v_new_strides);
    if (rc == NHP_OK && past > 0) rc = fill_operand(a.k_past, a.kp_s, a.kp_b, a.kp_h, k_past, k_past_strides);
    if (rc == NHP_OK && past > 0) rc = fill_operand(a.v_past, a.vp_s, a.vp_b, a.vp_h, v_past, v_past_strides);
    if (rc != NHP_OK) return rc;
    a.out = static_cast<uint16_t*>(cache_out);
    a.batch = (int)batch;
    a.kv_heads = (int)kv_heads;
    a.past = (int)past;
    a.chunks = (int)(head_dim / 8);
    a.items = (past + sq) * batch * kv_heads * a.chunks;
    const int64_t blocks = (a.items + 255) / 256;
    if (!grid_fits(blocks, 256)) return NHP_ERR_SHAPE;
    launch_prepare();
    cache_append_kernel<<<dim3((unsigned)blocks, 2), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(a);
    return launch_result();
}

}  // extern "C"
