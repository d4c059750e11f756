// Attention on the matrix cores: softmax(scale * q k^T + mask) v and its gradients without the scores ever leaving the
// chip (causal by index with an optional sliding window; forward also by a bit mask).
//
// Against the separate products and softmax, the [b, np, sq, sk] tensors are not written and read back (at 128 features
// their traffic costs more than the products themselves). A workgroup is four waves of 32 queries (keys in the kernel of
// the key and value gradients); every wave multiplies the same 64-row tiles, which arrive in LDS by direct loads one tile
// ahead, with one barrier per tile. What bounds them: per 32 x 32 x 16 matrix instruction (32 cycles on one of the four
// SIMDs) a wave reads one 1 KiB A operand from LDS, which at 128 bytes per cycle is just what LDS delivers to four SIMDs,
// and the exponentials and roundings of the softmax take the vector ALU about as long as the products take the matrix
// cores at 128 features (twice as long at 64); two workgroups per CU let these overlap.
//
// The gradients take two kernels, one over blocks of queries (gradient of q) and one over blocks of keys (of k and v),
// each recomputing the scores: seven products instead of five, but no atomic sums, so results are the same on every run.
//
// Measured (us, causal, forward / backward; products and softmax separately before, both per pass of the module; cards differ
// by up to 8 %):
//   [8192, 1, 32 heads, 8 of keys, 128] bf16   490 / 1738 (1122 / 1107 TFLOP/s)  whole pass 5786 -> 2230
//   [2048, 8, 16, 128] bf16                    148 / 512  (930 / 940)            about 1930 -> 690
//   [1024, 4, 12, 64] fp16                     19 / 52    (340 / 435)            whole pass 428 -> 84, with the host
//   [1531, 1, 32, 128] bf16, by mask           48 + 5 for the bits               650 -> 53
// Of that the reads ahead of the products and the probabilities between them (forward, us): [8192, 1, 32 on 8, 128] 527 -> 486,
// [4096, 2, 16, 96] 126 -> 110, [4096, 2, 32, 80] 219 -> 208, [2048, 8, 16, 128] 157 -> 148, [8192, 1, 12, 64] 148 -> 145; by mask
// (its bits ahead too) [1531, 1, 32, 128] 54 -> 48. Gradient
// of q the same way: both kernels 1754 -> 1738, [1024, 4, 12, 64] 53.3 -> 51.9. In the kernel of k and v there are no registers
// for it (one pair of operands ahead: no change, two: 13 registers spilled and 2 % slower).
#include "attention.hpp"

namespace nhp {

struct First {
    static constexpr int value = 0;
};
struct Second {
    static constexpr int value = 1;
};
constexpr int kReadsAhead = 4;   // reads of keys that are under way in the forward kernel (6: no faster)

// MODE of the forward kernel
constexpr int kCausal = 0;   // key k is visible to query q when q + shift - window <= k <= q + shift, by index
constexpr int kBits = 1;     // one bit per (query, key), set = masked: the score is replaced by `fill`

template <int DT, int HD, int MODE>
__global__ void __launch_bounds__(256, 2) attn_fwd_kernel(AttnFwdArgs a)
{
    using G = AttnGeo<HD>;
    using F = Frag<DT>;
    __shared__ __attribute__((aligned(1024))) char lds[4 * G::kTileBytes];
    __shared__ uint32_t tile_visible[MODE == kBits ? kMaxMaskTiles / 32 : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ql = lane & 31, half = lane >> 5;

    const int nqb = (a.sq + kFwdRows - 1) / kFwdRows;
    const Place at_block = place(a.batch * a.heads);
    const int bh = at_block.unit, qb = nqb - 1 - at_block.block;
    const int b = bh / a.heads, h = bh % a.heads, hk = h / a.group;
    const int q0 = qb * kFwdRows, qw = q0 + wave * 32;
    const int qi = min(qw + ql, a.sq - 1);

    const uint16_t* qp = a.q + b * a.q_b + h * a.q_h + (int64_t)qi * a.q_s + half * 8;
    u32x4 qf[G::kSteps];
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) qf[t] = load16(qp + t * 16);

#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) arrive(qf[t]);

    int kt_lo = 0, kt_hi = (a.sk + 63) >> 6;
    if constexpr (MODE == kCausal) {
        kt_hi = min(kt_hi, ((min(q0 + kFwdRows, a.sq) - 1 + a.shift) >> 6) + 1);
        kt_lo = max(0, q0 + a.shift - a.window) >> 6;
    }
    const int wave_hi = min(qw + 31, a.sq - 1) + a.shift;      // last key this wave can see
    const int wave_lo = qw + a.shift - a.window;               // first one its first query sees
    const uint64_t* bits = nullptr;
    if constexpr (MODE == kBits) {
        bits = a.bits + (a.bits_batches == 1 ? 0 : b) * (int64_t)a.sq * kt_hi;
        // tiles in which all of the workgroup's queries are masked are skipped (see the loop over `pass`)
        for (int i = tid; i < (kt_hi + 31) / 32; i += 256) tile_visible[i] = 0;
        __syncthreads();
        for (int kt = wave; kt < kt_hi; kt += 4) {
            const uint64_t w0 = bits[(int64_t)min(q0 + lane, a.sq - 1) * kt_hi + kt];
            const uint64_t w1 = bits[(int64_t)min(q0 + 64 + lane, a.sq - 1) * kt_hi + kt];
            if (__any((w0 & w1) != ~0ull) && lane == 0) atomicOr(&tile_visible[kt >> 5], 1u << (kt & 31));
        }
        __syncthreads();
    }

    const uint16_t* kbase = a.k + b * a.k_b + hk * a.k_h;
    const uint16_t* vbase = a.v + b * a.v_b + hk * a.v_h;
    TileLoader<HD> kload(a.k_s, lane, wave), vload(a.v_s, lane, wave);
    const int krow = G::row_addr(ql, half), vrow = G::tr_addr(lane);

    f32x16 o[G::kDTiles];
    float m, l;
    bool skip = MODE == kBits;
    for (;;) {
#pragma unroll
        for (int d = 0; d < G::kDTiles; ++d) o[d] = f32x16{};
        m = kFarBelow;
        l = 0.0f;
        auto next_tile = [&](int kt) {
            if constexpr (MODE == kBits) {
                while (skip && kt < kt_hi && !((tile_visible[kt >> 5] >> (kt & 31)) & 1)) ++kt;
            }
            return kt;
        };
        auto fetch = [&](int kt, int buf) {
            const int left = a.sk - kt * 64;
            kload.load(kbase + (int64_t)kt * 64 * a.k_s, lds + buf * G::kTileBytes, left);
            vload.load(vbase + (int64_t)kt * 64 * a.v_s, lds + (2 + buf) * G::kTileBytes, left);
        };
        // Mask bits are asked for a tile ahead, before that tile, and waited for together with it: asked for where they are
        // needed, they would be waited for behind the tile that is under way.
        uint64_t word = 0;
        auto fetch_word = [&](int kt) {
            if constexpr (MODE == kBits) word = bits[(int64_t)qi * kt_hi + kt];
        };
        int kt = next_tile(kt_lo);
        if (kt < kt_hi) {
            fetch_word(kt);
            fetch(kt, 0);
        }
        // (two tiles a turn of the loop: the addresses in LDS are then those of the first plus a constant)
        auto turn = [&](auto which) {
            constexpr int buf = decltype(which)::value;
            wait_lds_loads();
            if constexpr (MODE == kBits) asm volatile("" : "+v"(word));
            const uint64_t w = word;
            __syncthreads();
            const int following = next_tile(kt + 1);
            if (following < kt_hi) {
                fetch_word(following);
                fetch(following, buf ^ 1);
            }
            const int key0 = kt * 64;
            const char* kt_lds = lds + buf * G::kTileBytes;
            const char* vt_lds = lds + (2 + buf) * G::kTileBytes;
            const bool active = MODE == kBits || (key0 <= wave_hi && key0 + 63 >= wave_lo);
            if (active) {
                f32x16 s[2] = {f32x16{}, f32x16{}};
                // The compiler would read two operands, wait for them and multiply them, sixteen times over: the reads are
                // dealt out here, four of them ahead of the products (sched_group_barrier: 0x100 reads, 0x008 products).
                // The wave that multiplies goes first, so that the other one of the SIMD is left with its softmax (4 to 5 %
                // of the kernel, no gain in the kernels of the gradients).
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int t = 0; t < G::kSteps; ++t) {
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const u32x4 kf = lds_read16(kt_lds + (krow ^ (t << 5)) + n * 32 * G::kRowBytes);
                        s[n] = F::mma(kf, qf[t], s[n]);
                    }
                }
                __builtin_amdgcn_sched_group_barrier(0x100, kReadsAhead, 0);
#pragma unroll
                for (int i = 0; i < 2 * G::kSteps - kReadsAhead; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x008, kReadsAhead, 0);
                __builtin_amdgcn_s_setprio(0);
                if constexpr (MODE == kBits) {
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const uint32_t wn = (uint32_t)(w >> (32 * n)) >> (4 * half);
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            float x = s[n][i] * a.scale_log2;
                            x = (wn >> ((i >> 2) * 8 + (i & 3))) & 1 ? a.fill_log2 : x;
                            s[n][i] = x;
                        }
                    }
                }
                if (key0 + 63 >= a.sk || (MODE == kCausal && (key0 + 63 > qw + a.shift || key0 < wave_lo + 31))) {
                    // keys from `last` on do not exist or are not visible to this lane's query
                    const int q = qw + ql + a.shift;
                    const int last = (MODE == kCausal ? min(a.sk - 1, q) : a.sk - 1) - key0 - 4 * half;
                    const int first = (MODE == kCausal ? q - a.window : 0) - key0 - 4 * half;
#pragma unroll
                    for (int n = 0; n < 2; ++n)
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const int key = n * 32 + (i >> 2) * 8 + (i & 3);
                            if (key > last || (MODE == kCausal && key < first)) s[n][i] = kNegInf;
                        }
                }
                // Values by 16 keys: those of the first are read ahead of the softmax, those of the next while one lot is
                // multiplied, and between those products the next eight probabilities are formed (sched_barrier keeps the
                // order as it is written).
                u32x4 vf[2][G::kDTiles];
                auto read_v = [&](int ks) {
#pragma unroll
                    for (int d = 0; d < G::kDTiles; ++d)
                        vf[ks & 1][d] = lds_read_tr(vt_lds + (vrow ^ (d << 6)) + ks * 16 * G::kRowBytes,
                                                    vt_lds + (vrow ^ (d << 6 | 32)) + (ks * 16 + 8) * G::kRowBytes);
                };
                read_v(0);
                __builtin_amdgcn_sched_barrier(0);
                const float c = MODE == kBits ? 1.0f : a.scale_log2;
                float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
                for (int i = 1; i < 16; ++i) mx = fmaxf(fmaxf(mx, s[0][i]), s[1][i]);
                mx = max_halves(mx) * c;
                // the running maximum only moves when a score exceeds it by more than 2^kLazy: the factor stays exact,
                // probabilities of up to 2^kLazy are no less precise, and most tiles leave the accumulators alone
                if (__any(mx > m + kLazy)) {
                    const float mn = fmaxf(m, mx), alpha = exp2_raw(m - mn);
                    m = mn;
                    l *= alpha;
#pragma unroll
                    for (int d = 0; d < G::kDTiles; ++d)
#pragma unroll
                        for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
                }
                float sum = 0.0f;
                u32x4 pf;
                auto element = [&](int i) {
                    const float x = exp2_raw(fmaf(s[i >> 4][i & 15], c, -m));
                    s[i >> 4][i & 15] = x;
                    sum += x;
                };
#pragma unroll
                for (int i = 0; i < 8; ++i) element(i);
                pf = F::pack8(s[0], 0);
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    if (ks < 3) read_v(ks + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int d = 0; d < G::kDTiles; ++d) {
                        o[d] = F::mma(vf[ks & 1][d], pf, o[d]);
                        if (ks < 3) {
#pragma unroll
                            for (int i = 8 * d / G::kDTiles; i < 8 * (d + 1) / G::kDTiles; ++i) element((ks + 1) * 8 + i);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (ks < 3) pf = F::pack8(s[(ks + 1) >> 1], ((ks + 1) & 1) * 8);
                }
                l += sum;
                __builtin_amdgcn_s_setprio(0);
            }
            kt = following;
        };
        while (kt < kt_hi) {
            turn(First{});
            if (kt >= kt_hi) break;
            turn(Second{});
        }
        if constexpr (MODE == kBits) {
            // A row without a visible key (or with nothing but scores as low as the fill value) is an average over the
            // masked keys as well: go over all tiles then.
            const int redo = __syncthreads_or(skip && m <= a.fill_log2 + 200.0f);
            if (redo) {
                skip = false;
                continue;
            }
        }
        break;
    }
    l = sum_halves(l);
    if (qw + ql < a.sq) {
        const float inv = 1.0f / l;
        if (a.lse && half == 0) a.lse[(int64_t)bh * a.sq + qw + ql] = m + __log2f(l);
        const int64_t at = b * a.o_b + h * a.o_h + (int64_t)(qw + ql) * a.o_s;
        store_transposed<DT, HD>(a.o + at, a.kept ? a.kept + at : nullptr, o, inv, half);
    }
}

// One bit per (query, key) of a byte mask [batches, 1, sq, sk], set where the byte is not zero; the bits of keys
// beyond sk are set. Output [batches, sq, ceil(sk / 64)] words.
__global__ void __launch_bounds__(256) pack_mask_kernel(uint64_t* out, const uint8_t* mask, int64_t rows, int sk, int words)
{
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    const uint8_t* p = mask + row * sk;
    // eight words at a time: one after the other, a row of 1531 keys waited for memory 24 times (12.8 -> 7.5 us for 1531 rows)
    for (int w0 = 0; w0 < words; w0 += 8) {
        uint8_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[min((w0 + j) * 64 + lane, sk - 1)];
        uint64_t mine = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint64_t word = __ballot((w0 + j) * 64 + lane >= sk || v[j] != 0);
            mine = lane == j ? word : mine;
        }
        if (lane < min(8, words - w0)) out[row * words + w0 + lane] = mine;
    }
}

template <int DT, int HD>
static int launch_fwd(const AttnFwdArgs& a, int mode, hipStream_t st)
{
    const int64_t nqb = (a.sq + kFwdRows - 1) / kFwdRows;
    const int64_t grid = (int64_t)a.batch * a.heads * nqb;
    if (!grid_fits(grid, 256)) return NHP_ERR_SHAPE;
    launch_prepare();
    if (mode == kCausal)
        attn_fwd_kernel<DT, HD, kCausal><<<dim3((unsigned)grid), dim3(256), 0, st>>>(a);
    else
        attn_fwd_kernel<DT, HD, kBits><<<dim3((unsigned)grid), dim3(256), 0, st>>>(a);
    return launch_result();
}

template <int DT>
static int launch_fwd_hd(const AttnFwdArgs& a, int hd, int mode, hipStream_t st)
{
    switch (hd) {
    case 64: return launch_fwd<DT, 64>(a, mode, st);
    case 80: return launch_fwd<DT, 80>(a, mode, st);
    case 96: return launch_fwd<DT, 96>(a, mode, st);
    case 128: return launch_fwd<DT, 128>(a, mode, st);
    }
    return NHP_ERR_SHAPE;
}

// Gradient of q. As the forward kernel: 32 queries per wave as columns, K and V tiles of 64 keys in LDS. Per 32 keys:
// S^T = K q^T and dP^T = V dO^T, dS^T = P^T (dP^T - delta), dq^T += K^T dS^T. Also forms delta (the dot product of
// each row of out and dO), which the kernel of the key and value gradients reads.
template <int DT, int HD>
__global__ void __launch_bounds__(256, 2) attn_dq_kernel(AttnBwdArgs a)
{
    using G = AttnGeo<HD>;
    using F = Frag<DT>;
    __shared__ __attribute__((aligned(1024))) char lds[4 * G::kTileBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ql = lane & 31, half = lane >> 5;
    const int nqb = (a.sq + kFwdRows - 1) / kFwdRows;
    const Place at_block = place(a.batch * a.heads);
    const int bh = at_block.unit, qb = nqb - 1 - at_block.block;
    const int b = bh / a.heads, h = bh % a.heads, hk = h / a.group;
    const int q0 = qb * kFwdRows, qw = q0 + wave * 32;
    const int qi = min(qw + ql, a.sq - 1);

    const uint16_t* qp = a.q + b * a.q_b + h * a.q_h + (int64_t)qi * a.q_s + half * 8;
    const uint16_t* gp = a.d_o + b * a.do_b + h * a.do_h + (int64_t)qi * a.do_s + half * 8;
    const uint16_t* op = a.o + b * a.o_b + h * a.o_h + (int64_t)qi * a.o_s + half * 8;
    u32x4 qf[G::kSteps], gf[G::kSteps];
    float delta = 0.0f;
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) {
        qf[t] = load16(qp + t * 16);
        gf[t] = load16(gp + t * 16);
    }
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) {
        const u32x4 of = load16(op + t * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            delta = fmaf(Half2<DT>::lo(of[i]), Half2<DT>::lo(gf[t][i]), delta);
            delta = fmaf(Half2<DT>::hi(of[i]), Half2<DT>::hi(gf[t][i]), delta);
        }
    }
    delta = sum_halves(delta);
    float lse = a.lse[(int64_t)bh * a.sq + qi];
    if (half == 0 && qw + ql < a.sq) a.delta[(int64_t)bh * a.sq + qi] = delta;
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) {
        arrive(qf[t]);
        arrive(gf[t]);
    }
    asm volatile("" : "+v"(lse));

    const int kt_hi = min((a.sk + 63) >> 6, ((min(q0 + kFwdRows, a.sq) - 1 + a.shift) >> 6) + 1);
    const int kt_lo = max(0, q0 + a.shift - a.window) >> 6;
    const int wave_hi = min(qw + 31, a.sq - 1) + a.shift, wave_lo = qw + a.shift - a.window;
    const uint16_t* kbase = a.k + b * a.k_b + hk * a.k_h;
    const uint16_t* vbase = a.v + b * a.v_b + hk * a.v_h;
    TileLoader<HD> kload(a.k_s, lane, wave), vload(a.v_s, lane, wave);
    const int krow = G::row_addr(ql, half), ktr = G::tr_addr(lane);
    auto fetch = [&](int kt, int buf) {
        const int left = a.sk - kt * 64;
        kload.load(kbase + (int64_t)kt * 64 * a.k_s, lds + buf * G::kTileBytes, left);
        vload.load(vbase + (int64_t)kt * 64 * a.v_s, lds + (2 + buf) * G::kTileBytes, left);
    };

    f32x16 dq[G::kDTiles];
#pragma unroll
    for (int d = 0; d < G::kDTiles; ++d) dq[d] = f32x16{};
    fetch(kt_lo, 0);
    auto turn = [&](auto which, int kt) {
        constexpr int buf = decltype(which)::value;
        wait_lds_loads();
        __syncthreads();
        if (kt + 1 < kt_hi) fetch(kt + 1, buf ^ 1);
        const int key0 = kt * 64;
        if (key0 > wave_hi || key0 + 63 < wave_lo) return;
        const char* kt_lds = lds + buf * G::kTileBytes;
        const char* vt_lds = lds + (2 + buf) * G::kTileBytes;
        const bool edge = key0 + 63 >= a.sk || key0 + 63 > qw + a.shift || key0 < wave_lo + 31;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            // reads ahead of the products and probabilities between them, as in the forward kernel
            f32x16 s{}, dp{};
            constexpr int kAhead = 3;
            u32x4 kf[kAhead], vf[kAhead];
            auto read = [&](int t) {
                kf[t % kAhead] = lds_read16(kt_lds + (krow ^ (t << 5)) + n * 32 * G::kRowBytes);
                vf[t % kAhead] = lds_read16(vt_lds + (krow ^ (t << 5)) + n * 32 * G::kRowBytes);
            };
            u32x4 tf[2][G::kDTiles];
            auto read_t = [&](int ks) {
                const char* base = kt_lds + (n * 32 + ks * 16) * G::kRowBytes;
#pragma unroll
                for (int d = 0; d < G::kDTiles; ++d)
                    tf[ks][d] = lds_read_tr(base + (ktr ^ (d << 6)), base + (ktr ^ (d << 6 | 32)) + 8 * G::kRowBytes);
            };
#pragma unroll
            for (int t = 0; t < kAhead && t < G::kSteps; ++t) read(t);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < G::kSteps; ++t) {
                s = F::mma(kf[t % kAhead], qf[t], s);
                dp = F::mma(vf[t % kAhead], gf[t], dp);
                if (t + kAhead < G::kSteps) read(t + kAhead);
                __builtin_amdgcn_sched_barrier(0);
            }
            read_t(0);
            if (edge) {
                const int q = qw + ql + a.shift;
                const int last = min(a.sk - 1, q) - key0 - 4 * half, first = q - a.window - key0 - 4 * half;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key = n * 32 + (i >> 2) * 8 + (i & 3);
                    if (key > last || key < first) s[i] = kNegInf;
                }
            }
            auto element = [&](int i) {
                const float p = exp2_raw(fmaf(s[i], a.scale_log2, -lse));
                s[i] = p * (dp[i] - delta);
            };
#pragma unroll
            for (int i = 0; i < 8; ++i) element(i);
            u32x4 f = F::pack8(s, 0);
            read_t(1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = 0; d < G::kDTiles; ++d) {
                dq[d] = F::mma(tf[0][d], f, dq[d]);
#pragma unroll
                for (int i = 8 * d / G::kDTiles; i < 8 * (d + 1) / G::kDTiles; ++i) element(8 + i);
                __builtin_amdgcn_sched_barrier(0);
            }
            f = F::pack8(s, 8);
#pragma unroll
            for (int d = 0; d < G::kDTiles; ++d) dq[d] = F::mma(tf[1][d], f, dq[d]);
        }
    };
    for (int kt = kt_lo; kt < kt_hi; kt += 2) {
        turn(First{}, kt);
        if (kt + 1 < kt_hi) turn(Second{}, kt + 1);
    }
    if (qw + ql < a.sq)
        store_transposed<DT, HD>(a.dq + b * a.dq_b + h * a.dq_h + (int64_t)(qw + ql) * a.dq_s, nullptr, dq, a.scale, half);
}

// Gradients of k and v: 32 keys per wave as columns, their k and v rows in registers; Q and dO tiles of 64 queries (and
// their row statistics) in LDS. Per 32 queries: S = Q k^T, dP = dO v^T, dS = P (dP - delta), dv^T += dO^T P,
// dk^T += Q^T dS. A workgroup goes over the queries of `fold` heads that share its keys, one after the other into the same
// accumulators; what remains to be added up (fold < group) it leaves in fp32.
template <int DT, int HD>
__global__ void __launch_bounds__(256, 2) attn_dkv_kernel(AttnBwdArgs a)
{
    using G = AttnGeo<HD>;
    using F = Frag<DT>;
    // from 96 features on, k, v and the two accumulators leave no registers for addresses (22 to 48 spilled ones cost a
    // factor of 1.9 at 128: 1926 against 1028 us at 8192 positions)
    constexpr bool kLean = HD >= 96;
    __shared__ __attribute__((aligned(1024))) char lds[4 * G::kTileBytes + 1024];
    char* const stats = lds + 4 * G::kTileBytes;   // [2 buffers][lse, delta][64]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kl = lane & 31, half = lane >> 5;
    const int units = a.heads / a.fold;
    const Place at_block = place(a.batch * units);   // (batch entry, `fold` heads); the first keys are seen by most queries
    const int unit = at_block.unit;
    const int b = unit / units, h0 = unit % units * a.fold, hk = h0 / a.group;
    const int k0 = at_block.block * kFwdRows, kw = k0 + wave * 32;
    const int ki = min(kw + kl, a.sk - 1);

    const uint16_t* kp = a.k + b * a.k_b + hk * a.k_h + (int64_t)ki * a.k_s + half * 8;
    const uint16_t* vp = a.v + b * a.v_b + hk * a.v_h + (int64_t)ki * a.v_s + half * 8;
    u32x4 kf[G::kSteps], vf[G::kSteps];
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) {
        kf[t] = load16(kp + t * 16);
        vf[t] = load16(vp + t * 16);
    }
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) {
        arrive(kf[t]);
        arrive(vf[t]);
    }

    // queries that see one of the workgroup's keys, and one of the wave's
    const int q_lo = max(0, k0 - a.shift), q_hi = min(a.sq, k0 + kFwdRows - a.shift + a.window);
    const int qt_lo = q_lo >> 6, qt_hi = (q_hi + 63) >> 6;
    const int wave_lo = kw - a.shift, wave_hi = min(kw + 31, a.sk - 1) - a.shift + a.window;
    const uint16_t* qbase = a.q + b * a.q_b;
    const uint16_t* gbase = a.d_o + b * a.do_b;
    TileLoader<HD, kLean> qload(a.q_s, lane, wave), gload(a.do_s, lane, wave);
    const int row = G::row_addr(kl, half), tr = G::tr_addr(lane);
    auto fetch = [&](int h, int qt, int buf) {
        const int left = a.sq - qt * 64;
        const int64_t row0 = ((int64_t)b * a.heads + h) * a.sq + qt * 64;
        qload.load(qbase + h * a.q_h + (int64_t)qt * 64 * a.q_s, lds + buf * G::kTileBytes, left);
        gload.load(gbase + h * a.do_h + (int64_t)qt * 64 * a.do_s, lds + (2 + buf) * G::kTileBytes, left);
        if (wave == 0) load_floats(a.lse + row0, stats + buf * 512, lane, left);
        if (wave == 1) load_floats(a.delta + row0, stats + buf * 512 + 256, lane, left);
    };

    f32x16 dk[G::kDTiles], dv[G::kDTiles];
#pragma unroll
    for (int d = 0; d < G::kDTiles; ++d) dk[d] = dv[d] = f32x16{};
    // the tiles of all heads in one sequence: the first one of a head is on its way during the last one of the head before
    int buf = 1, h = h0, qt = qt_lo;
    if (qt_lo < qt_hi) fetch(h, qt, 0);
    for (int left = (qt_hi - qt_lo) * a.fold; left > 0; --left) {
        const int r0 = qt * 64;
        buf ^= 1;
        wait_lds_loads();
        __syncthreads();
        if (++qt == qt_hi) {
            qt = qt_lo;
            ++h;
        }
        if (left > 1) fetch(h, qt, buf ^ 1);
        if (r0 + 63 < wave_lo || r0 > wave_hi) continue;
        const char* qt_lds = lds + buf * G::kTileBytes;
        const char* gt_lds = lds + (2 + buf) * G::kTileBytes;
        const char* st = stats + buf * 512 + half * 16;
        const bool edge = r0 + 63 >= a.sq || r0 < wave_lo + 31 || r0 + 63 > kw - a.shift + a.window;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            int row_n = row, tr_n = tr;
            if constexpr (kLean) asm volatile("" : "+v"(row_n), "+v"(tr_n));   // formed here every time, not kept
            f32x16 s{}, dp{};
#pragma unroll
            for (int t = 0; t < G::kSteps; ++t) {
                s = F::mma(lds_read16(qt_lds + (row_n ^ (t << 5)) + n * 32 * G::kRowBytes), kf[t], s);
                dp = F::mma(lds_read16(gt_lds + (row_n ^ (t << 5)) + n * 32 * G::kRowBytes), vf[t], dp);
            }
            if (edge) {
                const int key = kw + kl - a.shift;
                const int first = key - r0 - 4 * half, last = min(a.sq - 1, key + a.window) - r0 - 4 * half;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int q = n * 32 + (i >> 2) * 8 + (i & 3);
                    if (q > last || q < first) s[i] = kNegInf;
                }
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 l4 = *reinterpret_cast<const f32x4*>(st + (n * 32 + g * 8) * 4);
                const f32x4 d4 = *reinterpret_cast<const f32x4*>(st + 256 + (n * 32 + g * 8) * 4);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = exp2_raw(fmaf(s[4 * g + i], a.scale_log2, -l4[i]));
                    s[4 * g + i] = p;
                    dp[4 * g + i] = p * (dp[4 * g + i] - d4[i]);
                }
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const u32x4 pf = F::pack8(s, ks * 8), df = F::pack8(dp, ks * 8);
                const int at = (n * 32 + ks * 16) * G::kRowBytes;
#pragma unroll
                for (int d = 0; d < G::kDTiles; ++d) {
                    dv[d] = F::mma(lds_read_tr(gt_lds + at + (tr_n ^ (d << 6)), gt_lds + at + (tr_n ^ (d << 6 | 32)) + 8 * G::kRowBytes), pf, dv[d]);
                    dk[d] = F::mma(lds_read_tr(qt_lds + at + (tr_n ^ (d << 6)), qt_lds + at + (tr_n ^ (d << 6 | 32)) + 8 * G::kRowBytes), df, dk[d]);
                }
            }
        }
    }
    if (kw + kl < a.sk && a.dk_parts) {
        const int64_t at = ((int64_t)unit * a.sk + kw + kl) * HD;
        store_transposed<HD>(a.dk_parts + at, dk, a.scale, half);
        store_transposed<HD>(a.dv_parts + at, dv, 1.0f, half);
    } else if (kw + kl < a.sk) {
        store_transposed<DT, HD>(a.dk + b * a.dk_b + hk * a.dk_h + (int64_t)(kw + kl) * a.dk_s, nullptr, dk, a.scale, half);
        store_transposed<DT, HD>(a.dv + b * a.dv_b + hk * a.dv_h + (int64_t)(kw + kl) * a.dv_s, nullptr, dv, 1.0f, half);
    }
}

// Adds up what the workgroups of a key/value head have left and rounds the sums. blockIdx.z picks dk or dv.
template <int DT>
__global__ void __launch_bounds__(256) attn_group_sum_kernel(AttnBwdArgs a, int hd)
{
    const int kv_heads = a.heads / a.group, parts = a.group / a.fold, chunks = hd / 8;
    const int64_t items = (int64_t)a.sk * a.batch * kv_heads * chunks;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= items) return;
    const int c = (int)(i % chunks);
    int64_t r = i / chunks;
    const int hk = (int)(r % kv_heads);
    r /= kv_heads;
    const int b = (int)(r % a.batch);
    const int64_t s = r / a.batch;
    const bool second = blockIdx.z != 0;
    const float* p = (second ? a.dv_parts : a.dk_parts) + (((int64_t)b * kv_heads + hk) * parts * a.sk + s) * hd + c * 8;
    float sum[8] = {};
    for (int g = 0; g < parts; ++g) {
        const f32x4* x = reinterpret_cast<const f32x4*>(p + (int64_t)g * a.sk * hd);
        const f32x4 lo = __builtin_nontemporal_load(x), hi = __builtin_nontemporal_load(x + 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            sum[j] += lo[j];
            sum[4 + j] += hi[j];
        }
    }
    uint16_t* o = second ? a.dv + s * a.dv_s + b * a.dv_b + hk * a.dv_h : a.dk + s * a.dk_s + b * a.dk_b + hk * a.dk_h;
    *reinterpret_cast<u32x4*>(o + c * 8) = pack8<DT>(sum);
}

// Query heads that a workgroup of the second gradient kernel goes over: as many as leave enough workgroups. Every head that is
// not added up in registers costs 8 bytes written and read again per element of k and v, but causal key blocks differ in
// length by up to a factor of 2 * blocks, and with few workgroups the longest one is what the launch takes. Two workgroups
// fit on a CU: 512 at once, which is enough where a row is at most eight blocks long; beyond, twice that. All kernels of the
// backward, us, fold 1 / 2 / 4 of a group of 4, 128 features:
//   [1024, 4, 32 heads] 198 / 183 / 239 (1024 / 512 / 256 workgroups), [1024, 16, 16] 405 / 327 / 318,
//   [2048, 1, 32] 181 / 249 / 401 (512 / 256 / 128), [2048, 8, 16] 569 / 515 / 570 (2048 / 1024 / 512),
//   [4096, 1, 32] 497 / 577 / 862, [4096, 2, 32 of 80] 678 / 677 / 748, [8192, 1, 32] 1743 / 1727 / 2144,
//   [8192, 4, 16] 3545 / 3478 / 3513, [300, 1, 32] 44 / 55 / 77.
static int bwd_fold(int64_t batch, int64_t heads, int64_t kv_heads, int64_t sk)
{
    const int64_t group = heads / kv_heads, blocks = batch * heads * ((sk + kFwdRows - 1) / kFwdRows);
    const int64_t least = sk <= 1024 ? 512 : 1024;
    for (int64_t fold = group < blocks / least ? group : blocks / least; fold > 1; --fold)
        if (group % fold == 0) return (int)fold;
    return 1;
}

template <int DT, int HD>
static int launch_bwd(AttnBwdArgs a, hipStream_t st)
{
    const int64_t nqb = (a.sq + kFwdRows - 1) / kFwdRows, nkb = (a.sk + kFwdRows - 1) / kFwdRows;
    const int64_t sum_blocks = ((int64_t)a.sk * a.batch * (a.heads / a.group) * (HD / 8) + 255) / 256;
    const int64_t dq_blocks = (int64_t)a.batch * a.heads * nqb, dkv_blocks = (int64_t)a.batch * (a.heads / a.fold) * nkb;
    if (!grid_fits(dq_blocks, 256) || !grid_fits(dkv_blocks, 256) || !grid_fits(sum_blocks, 256)) return NHP_ERR_SHAPE;
    launch_prepare();
    attn_dq_kernel<DT, HD><<<dim3((unsigned)dq_blocks), dim3(256), 0, st>>>(a);
    attn_dkv_kernel<DT, HD><<<dim3((unsigned)dkv_blocks), dim3(256), 0, st>>>(a);
    if (a.fold < a.group) attn_group_sum_kernel<DT><<<dim3((unsigned)sum_blocks, 1, 2), dim3(256), 0, st>>>(a, HD);
    return launch_result();
}

template <int DT>
static int launch_bwd_hd(const AttnBwdArgs& a, int hd, hipStream_t st)
{
    switch (hd) {
    case 64: return launch_bwd<DT, 64>(a, st);
    case 80: return launch_bwd<DT, 80>(a, st);
    case 96: return launch_bwd<DT, 96>(a, st);
    case 128: return launch_bwd<DT, 128>(a, st);
    }
    return NHP_ERR_SHAPE;
}

}  // namespace nhp

extern "C" {

int nhp_attention_mask_bits(void* bits, const void* mask, int64_t batches, int64_t sq, int64_t sk, void* stream)
{
    using namespace nhp;
    if (!bits || !mask) return NHP_ERR_NULL;
    if (batches <= 0 || sq <= 0 || sk <= 0 || sk > 64 * (int64_t)kMaxMaskTiles) return NHP_ERR_SHAPE;
    const int64_t rows = batches * sq;
    if (!grid_fits((rows + 3) / 4, 256)) return NHP_ERR_SHAPE;
    launch_prepare();
    pack_mask_kernel<<<dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<uint64_t*>(bits), static_cast<const uint8_t*>(mask), rows, (int)sk, (int)((sk + 63) / 64));
    return launch_result();
}

int nhp_attention_fwd_keep(void* out, void* kept, float* lse, const void* q, const void* k, const void* v, const void* mask_bits,
                           int64_t mask_batches, float mask_fill, float scale, int64_t window, int64_t batch, int64_t heads,
                           int64_t kv_heads, int64_t sq, int64_t sk, int64_t head_dim, const int64_t* q_strides,
                           const int64_t* k_strides, const int64_t* v_strides, const int64_t* out_strides, int dtype, void* stream)
{
    using namespace nhp;
    if (!out || !q || !k || !v || !q_strides || !k_strides || !v_strides || !out_strides) return NHP_ERR_NULL;
    if (batch <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || sq <= 0 || sk <= 0 || sq > (1 << 24) || sk > (1 << 24) ||
        batch * heads > (1 << 24))
        return NHP_ERR_SHAPE;
    if (!(scale > 0.0f)) return NHP_ERR_SHAPE;
    if (!mask_bits && sk < sq) return NHP_ERR_SHAPE;   // a query before the first key would see none
    if (mask_bits && (sk > 64 * (int64_t)kMaxMaskTiles || (mask_batches != 1 && mask_batches != batch))) return NHP_ERR_SHAPE;
    AttnFwdArgs a{};
    int rc = fill_operand(a.q, a.q_s, a.q_b, a.q_h, q, q_strides);
    if (rc == NHP_OK) rc = fill_operand(a.k, a.k_s, a.k_b, a.k_h, k, k_strides);
    if (rc == NHP_OK) rc = fill_operand(a.v, a.v_s, a.v_b, a.v_h, v, v_strides);
    const uint16_t* o = nullptr;
    if (rc == NHP_OK) rc = fill_operand(o, a.o_s, a.o_b, a.o_h, out, out_strides);
    if (rc != NHP_OK) return rc;
    if (!ptr_aligned16(kept)) return NHP_ERR_SHAPE;
    a.o = static_cast<uint16_t*>(out);
    a.kept = static_cast<uint16_t*>(kept);
    a.lse = lse;
    a.bits = static_cast<const uint64_t*>(mask_bits);
    a.bits_batches = (int)mask_batches;
    a.fill_log2 = fmaxf(mask_fill * kLog2e, -1e30f);
    a.scale_log2 = scale * kLog2e;
    a.batch = (int)batch;
    a.heads = (int)heads;
    a.group = (int)(heads / kv_heads);
    a.sq = (int)sq;
    a.sk = (int)sk;
    a.shift = (int)(sk - sq);
    a.window = window < 0 || window > sk ? (int)sk : (int)window;
    const int mode = mask_bits ? kBits : kCausal;
    if (dtype == NHP_BF16) return launch_fwd_hd<NHP_BF16>(a, (int)head_dim, mode, static_cast<hipStream_t>(stream));
    if (dtype == NHP_F16) return launch_fwd_hd<NHP_F16>(a, (int)head_dim, mode, static_cast<hipStream_t>(stream));
    return NHP_ERR_DTYPE;
}

int nhp_attention_fwd(void* out, float* lse, const void* q, const void* k, const void* v, const void* mask_bits,
                      int64_t mask_batches, float mask_fill, float scale, int64_t window, int64_t batch, int64_t heads,
                      int64_t kv_heads, int64_t sq, int64_t sk, int64_t head_dim, const int64_t* q_strides,
                      const int64_t* k_strides, const int64_t* v_strides, const int64_t* out_strides, int dtype, void* stream)
{
    return nhp_attention_fwd_keep(out, nullptr, lse, q, k, v, mask_bits, mask_batches, mask_fill, scale, window, batch, heads,
                                  kv_heads, sq, sk, head_dim, q_strides, k_strides, v_strides, out_strides, dtype, stream);
}

int64_t nhp_attention_bwd_workspace_bytes(int64_t batch, int64_t heads, int64_t kv_heads, int64_t sq, int64_t sk, int64_t head_dim)
{
    if (batch <= 0 || heads <= 0 || kv_heads <= 0 || sq <= 0 || sk <= 0 || head_dim <= 0) return 0;
    if (heads % kv_heads) return 0;
    const int64_t delta = (batch * heads * sq * 4 + 255) / 256 * 256;
    const int64_t fold = nhp::bwd_fold(batch, heads, kv_heads, sk);
    return delta + (fold * kv_heads < heads ? 2 * sk * batch * (heads / fold) * head_dim * 4 : 0);
}

int nhp_attention_bwd(void* dq, void* dk, void* dv, const void* d_out, const void* q, const void* k, const void* v,
                      const void* out, const float* lse, void* workspace, float scale, int64_t window, int64_t batch,
                      int64_t heads, int64_t kv_heads, int64_t sq, int64_t sk, int64_t head_dim, const int64_t* dq_strides,
                      const int64_t* dk_strides, const int64_t* dv_strides, const int64_t* d_out_strides,
                      const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                      const int64_t* out_strides, int dtype, void* stream)
{
    using namespace nhp;
    if (!dq || !dk || !dv || !d_out || !q || !k || !v || !out || !lse || !workspace) return NHP_ERR_NULL;
    for (const int64_t* s : {dq_strides, dk_strides, dv_strides, d_out_strides, q_strides, k_strides, v_strides, out_strides})
        if (!s) return NHP_ERR_NULL;
    if (batch <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || sq <= 0 || sk < sq || sk > (1 << 24) ||
        batch * heads > (1 << 24) || !(scale > 0.0f))
        return NHP_ERR_SHAPE;
    AttnBwdArgs a{};
    const uint16_t *pdq, *pdk, *pdv;
    int rc = fill_operand(a.q, a.q_s, a.q_b, a.q_h, q, q_strides);
    if (rc == NHP_OK) rc = fill_operand(a.k, a.k_s, a.k_b, a.k_h, k, k_strides);
    if (rc == NHP_OK) rc = fill_operand(a.v, a.v_s, a.v_b, a.v_h, v, v_strides);
    if (rc == NHP_OK) rc = fill_operand(a.o, a.o_s, a.o_b, a.o_h, out, out_strides);
    if (rc == NHP_OK) rc = fill_operand(a.d_o, a.do_s, a.do_b, a.do_h, d_out, d_out_strides);
    if (rc == NHP_OK) rc = fill_operand(pdq, a.dq_s, a.dq_b, a.dq_h, dq, dq_strides);
    if (rc == NHP_OK) rc = fill_operand(pdk, a.dk_s, a.dk_b, a.dk_h, dk, dk_strides);
    if (rc == NHP_OK) rc = fill_operand(pdv, a.dv_s, a.dv_b, a.dv_h, dv, dv_strides);
    if (rc != NHP_OK) return rc;
    if (!ptr_aligned16(workspace)) return NHP_ERR_SHAPE;
    a.dq = static_cast<uint16_t*>(dq);
    a.dk = static_cast<uint16_t*>(dk);
    a.dv = static_cast<uint16_t*>(dv);
    a.lse = lse;
    a.delta = static_cast<float*>(workspace);
    a.fold = bwd_fold(batch, heads, kv_heads, sk);
    if (a.fold * kv_heads < heads) {
        a.dk_parts = reinterpret_cast<float*>(static_cast<char*>(workspace) + (batch * heads * sq * 4 + 255) / 256 * 256);
        a.dv_parts = a.dk_parts + sk * batch * (heads / a.fold) * head_dim;
    }
    a.scale = scale;
    a.scale_log2 = scale * kLog2e;
    a.batch = (int)batch;
    a.heads = (int)heads;
    a.group = (int)(heads / kv_heads);
    a.sq = (int)sq;
    a.sk = (int)sk;
    a.shift = (int)(sk - sq);
    a.window = window < 0 || window > sk ? (int)sk : (int)window;
    if (dtype == NHP_BF16) return launch_bwd_hd<NHP_BF16>(a, (int)head_dim, static_cast<hipStream_t>(stream));
    if (dtype == NHP_F16) return launch_bwd_hd<NHP_F16>(a, (int)head_dim, static_cast<hipStream_t>(stream));
    return NHP_ERR_DTYPE;
}

}  // extern "C"
