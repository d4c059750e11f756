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
// Measured (us, bf16, without the prefetch and with one head per workgroup before; copy: read and written bytes at 5.1 TB/s;
// cards, and runs on one card, differ by up to 8 %):
//   16 sequences of 2047, 32 heads of 128      223 -> 196 (copy 210)     32 of 1000, 32 heads of 128   225 -> 186 (206)
//   32 of 2000, 8 heads of keys of 128          94 -> 89 (103)           20 of 2000, 32 heads of 80    328 -> 212 (161)
//   9 of 2000, 32 heads of 128                 161 -> 114 (116)          5 of 3000, 32 heads of 128    126 -> 94 (96)
//   1 of 8000, 32 heads of 128                  59 -> 58 (51)            4 of 300, 8 heads of keys      14 -> 11 (2)
// The registers of the prefetch leave room for two workgroups on a CU instead of three: 24 of 200 to 400, 32 heads of 128, which are
// three for each CU, take longer (34 -> 39, 59 -> 66); a variant without it is as fast there and slower in between.
// (Concatenations 949 us and attention 118 us for the first of them, before there was such a kernel.)
#include "attention.hpp"

#include <cmath>

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
template <int N>
struct Index {
    static constexpr int value = N;
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

// Workgroups of a CU that the registers leave room for: with four sums of 128 features, or two with twice the heads, there is one.
// (Two with six registers spilled: [16 sequences of 2047, 32 heads of 128] 206 -> 208 us, [24 of 1000] 156 -> 170.)
constexpr int decode_blocks_per_cu(int head_dim, int heads) { return heads == 4 || (heads == 2 && head_dim == 128) ? 1 : 2; }

// NQ: tiles of 16 queries; NH: key/value heads of a workgroup, one or several waves each.
//
// The keys of a head (of its split) always go into four sums, the 32 of chunk c into sum c % 4, whichever waves take them: a wave
// keeps NH of the four. So the result does not depend on NH. With one sum for each wave two heads per workgroup had two sums and
// four heads one, and the fewer there are the further off is the result: the probability of a sum's first maximum is 1, which has no
// error in 16 bits. Relative error against 64 bits, bf16, 128 features: [16 sequences of 2047, 32 heads] 2.312e-3 with four sums
// and 2.324e-3 with two, [64 of 400, 32 heads] 2.251e-3 and with one 2.324e-3. It costs 0 to 3 % of the time.
template <int DT, int HD, int NQ, int NH>
__global__ void __launch_bounds__(256, decode_blocks_per_cu(HD, NH)) attn_decode_kernel(AttnDecodeArgs a)
{
    using G = DecodeGeo<HD>;
    // With two tiles of queries the registers for what is on its way are there up to 64 features; beyond, two workgroups on a CU
    // without it are faster than one with it (512 pairs of 1000 keys, 20 queries, 128 features: 98 us, 107).
    constexpr bool kAhead = NQ == 1 || HD == 64;
    constexpr int kKeyWaves = 4 / NH, kKeys = 32 * kKeyWaves;   // waves that share a head's keys, and what they take in a round
    __shared__ __attribute__((aligned(1024))) char lds[4 * G::kWaveBytes];
    __shared__ float part_m[4][NH][NQ * 16], part_l[4][NH][NQ * 16];
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

    f32x4 sums_o[NH][NQ][G::kTiles];
    float sums_m[NH][NQ], sums_l[NH][NQ];
#pragma unroll
    for (int i = 0; i < NH; ++i)
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            sums_m[i][n] = kFarBelow;
            sums_l[i][n] = 0.0f;
#pragma unroll
            for (int d = 0; d < G::kTiles; ++d) sums_o[i][n][d] = f32x4{};
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
    // Stores and multiplies them; `whole`: all 32 exist, `sum_index`: the wave's sum that takes them.
    auto use = [&](auto whole, auto sum_index, int key0, Keys& kf, Values& vf, Hidden& hidden) {
        constexpr bool kWhole = decltype(whole)::value;
        auto& o = sums_o[decltype(sum_index)::value];
        auto& m = sums_m[decltype(sum_index)::value];
        auto& l = sums_l[decltype(sum_index)::value];
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
    Keys kf[kAhead ? 2 : 1];
    Values vf[kAhead ? 2 : 1];
    Hidden hidden[kAhead ? 2 : 1];
    // one chunk, the next of this wave being asked for first; the i-th of a turn of the loop
    auto step = [&](auto index) {
        constexpr int i = decltype(index)::value, now = i & 1, next = now ^ 1;
        if (key0 + kKeys <= last_whole) load(key0 + kKeys, kf[next], vf[next], hidden[next]);
        use(Yes{}, Index<i % NH>{}, key0, kf[now], vf[now], hidden[now]);
        key0 += kKeys;
        return key0 <= last_whole;
    };
    if constexpr (!kAhead) {
        for (; key0 <= last_whole; key0 += kKeys) {
            load(key0, kf[0], vf[0], hidden[0]);
            use(Yes{}, Index<0>{}, key0, kf[0], vf[0], hidden[0]);
        }
    } else if (key0 <= last_whole) {
        load(key0, kf[0], vf[0], hidden[0]);
        if constexpr (NH < 4) {
            while (step(Index<0>{}) && step(Index<1>{})) {}
        } else {
            while (step(Index<0>{}) && step(Index<1>{}) && step(Index<2>{}) && step(Index<3>{})) {}
        }
    }
    for (; key0 < key_hi; key0 += kKeys) {
        load_last(key0, kf[0], vf[0], hidden[0]);
        const int sum = (key0 - key_lo) / kKeys % NH;
        if (sum == 0) use(No{}, Index<0>{}, key0, kf[0], vf[0], hidden[0]);
        if constexpr (NH > 1)
            if (sum == 1) use(No{}, Index<1>{}, key0, kf[0], vf[0], hidden[0]);
        if constexpr (NH > 2) {
            if (sum == 2) use(No{}, Index<2>{}, key0, kf[0], vf[0], hidden[0]);
            if (sum == 3) use(No{}, Index<3>{}, key0, kf[0], vf[0], hidden[0]);
        }
    }

    // the four sums of each head, 16 queries at a time: in LDS as many as there are waves for a head
#pragma unroll
    for (int i = 0; i < NH; ++i)
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            const float l = reduce_columns<OpSum>(sums_l[i][n]);
            if (g == 0) {
                part_m[i * kKeyWaves + wave / NH][wave % NH][n * 16 + r16] = sums_m[i][n];
                part_l[i * kKeyWaves + wave / NH][wave % NH][n * 16 + r16] = l;
            }
        }
    const int r = tid >> 4, c = tid & 15;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int row = n * 16 + r;
        const bool mine_too = c < G::kChunks && row < rows;
        float big[NH], total[NH], acc[NH][8];
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) {
            big[hh] = kFarBelow;
            total[hh] = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[hh][j] = 0.0f;
        }
#pragma unroll
        for (int i = 0; i < NH; ++i) {
            if (i > 0 && key_lo + i * kKeys >= key_hi) break;   // no keys in these sums
            __syncthreads();
            float* sums = reinterpret_cast<float*>(mine);
#pragma unroll
            for (int d = 0; d < G::kTiles; ++d) *reinterpret_cast<f32x4*>(sums + r16 * G::kSumRow + d * 16 + 4 * g) = sums_o[i][n][d];
            __syncthreads();
            if (!mine_too) continue;
#pragma unroll
            for (int hh = 0; hh < NH; ++hh) {
                if (i == 0)
#pragma unroll
                    for (int s = 0; s < 4; ++s) big[hh] = fmaxf(big[hh], part_m[s][hh][row]);
#pragma unroll
                for (int w = 0; w < kKeyWaves; ++w) {
                    const int s = i * kKeyWaves + w;
                    const float f = exp2_raw(part_m[s][hh][row] - big[hh]);
                    total[hh] = fmaf(part_l[s][hh][row], f, total[hh]);
                    const float* p = reinterpret_cast<const float*>(lds + (w * NH + hh) * G::kWaveBytes) + r * G::kSumRow + c * 8;
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[hh][j] = fmaf(p[j], f, acc[hh][j]);
                }
            }
        }
        if (!mine_too) continue;
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) {
            const int pr = pair0 + hh, b2 = pr / a.kv_heads, hk2 = pr % a.kv_heads;
            if (a.splits == 1) {
                const float inv = 1.0f / total[hh];
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[hh][j] *= inv;
                uint16_t* op = a.o + row / a.group * a.o_s + b2 * a.o_b + (hk2 * a.group + row % a.group) * a.o_h;
                *reinterpret_cast<u32x4*>(op + c * 8) = pack8<DT>(acc[hh]);
            } else {
                const int64_t at = ((int64_t)split * pairs + pr) * rows + row;
                *reinterpret_cast<f32x4*>(a.part_o + at * HD + c * 8) = f32x4{acc[hh][0], acc[hh][1], acc[hh][2], acc[hh][3]};
                *reinterpret_cast<f32x4*>(a.part_o + at * HD + c * 8 + 4) = f32x4{acc[hh][4], acc[hh][5], acc[hh][6], acc[hh][7]};
                if (c == 0) *reinterpret_cast<f32x2*>(a.part_ml + at * 2) = f32x2{big[hh], total[hh]};
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

// Heads of a workgroup and workgroups of a pair of batch entry and key/value head: the cheapest of those that are open.
//
// Splits: at least as many as give each CU a workgroup with 256 keys (each has four sums, and with less the result is further off:
// 192 pairs of 500 keys 2.17e-3 with two splits, 2.24e-3 with one), at most as many as have 128 keys. With more than 16 queries a
// pair, beyond eight splits, 256 keys, since the second kernel has 16 KB of each to read (32 queries, 8 pairs of 4000 keys: 16
// splits 25.4 us, 32 splits 30.4; 16 pairs of 2000: 8 splits 20.6, 16 splits 22.3).
//
// Heads: two from 320 pairs and four from 640, for caches that are long enough: 768 keys, 256 where a row has less than the 256
// bytes of 128 features (24 sequences of 600, 32 heads of 128: 85 us with one, 94 with four; 20 of 500, 32 heads of 80: 68 with one,
// 55 with two and four splits), and unsplit four heads of 128 from 256 keys on (1024 pairs of 500: 97 -> 92). From 1024 pairs on also
// for caches so short that waves would be idle: 32 keys are one wave's, 64 two waves'.
//
// Time, us: what a copy of the bytes takes at 5 TB/s, 7 or 14 % less with two or four heads and another 7 % less where rows end
// within a cache line; times the unevenness (rounds of 256 workgroups over those there are) to the power of 0.6, because the
// bandwidth of an idle CU goes to the others in part (288 pairs of 2000 keys, 1 / 2 / 4 / 8 splits: 153 / 129 / 121 / 120 us); and
// 0.2 for each round and head, twice that where one workgroup fills a CU, 1 for the second kernel, 0.2 for each split. Against
// the best plan that was measured, 84 sizes of 32 to 2048 pairs, 30 to 3000 keys and 64 to 128 features: 2 % behind on average,
// 14 % at most.
struct DecodePlan {
    int heads_per_block, splits, keys_per_split;
};
static bool decode_heads_open(int heads, int64_t pairs, int64_t sk, int64_t hd, int64_t splits)
{
    if (heads == 2) return (pairs >= 320 && sk >= (hd < 128 ? 256 : 768)) || (pairs >= 1024 && sk <= 64 && hd < 128);
    if (heads == 4) return (pairs >= 640 && (sk >= 768 || (sk >= 256 && hd == 128 && splits == 1))) || (pairs >= 1024 && sk <= 32);
    return true;
}
static DecodePlan decode_plan(int64_t batch, int64_t kv_heads, int64_t rows, int64_t sk, int64_t hd)
{
    const int64_t pairs = batch * kv_heads, by_256 = (sk + 255) / 256, for_all = (256 + pairs - 1) / pairs;
    const int64_t least = for_all < by_256 ? for_all : by_256;
    int64_t most = sk <= 256 ? 1 : (sk + 127) / 128;
    if (rows > 16 && most > 8) most = by_256 > 8 ? by_256 : 8;
    if (most > least + 7) most = least + 7;   // more have never been the best, and the host waits for this
    const double copy = (double)(pairs * sk * hd * 8) / 5e6;
    DecodePlan plan{1, 1, 0};
    double best = 0.0;
    for (int heads = 1; heads <= (rows <= 16 ? 4 : 1); heads *= 2) {
        if (kv_heads % heads) break;
        const double gain = (heads == 1 ? 1.0 : heads == 2 ? 0.93 : 0.86) * (heads > 1 && hd % 64 ? 0.93 : 1.0);
        for (int64_t s = least; s <= most; ++s) {
            const int64_t keys = ((sk + s - 1) / s + 127) / 128 * 128, splits = (sk + keys - 1) / keys;   // none of them empty
            if (!decode_heads_open(heads, pairs, sk, hd, splits)) continue;
            const int64_t blocks = pairs / heads * splits, rounds = (blocks + 255) / 256;
            const double us = copy * gain * std::pow((double)(rounds * 256) / (double)blocks, 0.6) +
                              (decode_blocks_per_cu((int)hd, heads) == 1 ? 0.4 : 0.2) * (double)(rounds * heads) +
                              (splits > 1 ? 1.0 + 0.2 * (double)splits : 0.0);
            if (plan.keys_per_split == 0 || us < best) {
                best = us;
                plan = {heads, (int)splits, (int)keys};
            }
        }
    }
    return plan;
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
