// y = x W^T (+ bias) for the few rows of a decoding step (at most 32), 16-bit storage, fp32 sums; also with the activation or the
// residual addition that follows it (LinearEnd).
//
// Such a product reads every weight once for a handful of rows: the weights' bytes are its time, and the matrix cores idle.
// What a CU can have on the way is the limit, so x must not take much of it: read again for every 16 weight rows it costs
// as much as the weights. One workgroup of 8 waves per CU walks over tiles of 16 weight rows; the waves share the
// contraction, and each keeps its part of x in registers for all tiles. Beyond 4096 features (16 steps of 32 for each
// wave) four workgroups share the contraction of a tile and a second kernel adds their sums up.
//
// Weights go from memory to LDS directly, in pieces of 16 rows x 64 features that belong to one wave alone: three of them are
// always under way, also across tiles, and a wave waits for its own pieces, never for those of others (the one barrier of a
// tile is that of the sums). Loaded straight into the registers in the instruction's order, a load touched 64 bytes of 16
// rows, half a cache line of each; here it takes whole lines of 8 rows. us, 16 rows, weights that are not in any cache,
// half lines -> here (a kernel that only reads as many bytes):
//   [22016, 4096] 44.3 -> 38.1 (27.5)   [12288, 4096] 26.3 -> 23.1 (16.1)   [4096, 11008] 28.2 -> 23.1 (14.5)
//   [7680, 2560] 16.6 -> 12.3           [768, 3072] 8.8 -> 7.4              [4096, 4096] 12.6 -> 12.0 (6.4)
// A ring of 6 or 7 pieces, or two workgroups per CU, are no faster; reading x costs 2 to 3 us of it (one row: 34.6, 21.1).
//
// The contraction of a workgroup goes into sixteen sums of consecutive features, two to a wave, which are added up one after the
// other: the order of sixteen waves with a sum each, as which this kernel began, so the results stay what they were. Against one sum
// a wave it costs 0.1 us, 0.5 to 0.9 with more than 16 rows ([22016, 4096] 37.7 and 38.1, 32 rows 42.2 and 43.3).
//
// Rows of the matrix instruction (16 x 16 x 32) are weight rows, its columns the rows of x. A lane takes 16 consecutive
// bytes of its row per instruction and x in the same order, which the contraction does not mind.
#include "activation.hpp"
#include "attention.hpp"

namespace nhp {

struct LinearArgs {
    uint16_t* y;
    const uint16_t *x, *w, *bias;
    float* parts;   // with splits > 1: [splits][m][n]
    int m, n, k, splits;
    int bias_words;   // the bias starts at a multiple of four bytes
    int act;          // the gate's function (kGatedRows)
    const uint16_t *x1, *bias1, *residual;   // kAddRows: [m, n], [n], [m, n], the first two may be null
};

// What is done with a sum: nothing but the bias; gelu(bias + sum); act(gate) * value, the gate being the sum n / 2 features on;
// residual + (sum + bias), or residual + ((x1 + bias1) + (sum + bias)). In all of them the sum is rounded to the storage
// type first and the rest rounded where the kernels for it round (pointwise.hip, gated.hip): the same bits with a launch less,
// but for the GeLU of an fp16 bias that is not 16-byte aligned, whose kernel rounds its last product to fp16 at once
// (a layer of 768 features, one sequence: a step 100 -> 91 us; 4096 features, gated, 16 sequences: 312 -> 307).
enum LinearEnd { kPlainRows, kGeluRows, kGatedRows, kAddRows };

constexpr int kLinearWaveBits = 3, kLinearWaves = 1 << kLinearWaveBits, kLinearBlocks = 256;
constexpr int kLinearSteps = 16;   // steps of 32 features that a wave has at most
constexpr int kLinearSplitBits = 2, kLinearSplits = 1 << kLinearSplitBits;   // of a product with more features than the next
constexpr int kLinearWhole = kLinearSteps * kLinearWaves * 32;
constexpr int kRing = 4, kPieceBytes = 2048;   // pieces of 16 rows x 64 features in LDS for each wave

template <int N>
__device__ __forceinline__ void wait_pieces()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

template <int DT>
__device__ __forceinline__ float bias_of(const LinearArgs& a, int tile, int col)
{
    if (!a.bias) return 0.0f;
    if (!a.bias_words) return Half2<DT>::from_bits(a.bias[tile * 16 + col]);
    // by scalar loads (constant memory at a uniform address): a vector load would be waited for behind the pieces that are
    // under way
    typedef const __attribute__((address_space(4))) uint32_t* Words;
    const Words words = (Words)(uintptr_t)(a.bias + __builtin_amdgcn_readfirstlane(tile) * 16);
    uint32_t w = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        uint32_t word = words[q];
        asm volatile("" : "+s"(word));   // the value, not its address, is what is picked
        w = col >> 1 == q ? word : w;
    }
    return col & 1 ? Half2<DT>::hi(w) : Half2<DT>::lo(w);
}

__device__ __forceinline__ float gate_of(int act, float g)
{
    float value, slope;
    switch (act) {
    case kActSwish: gate_eval<kActSwish>(g, value, slope); break;
    case kActGelu: gate_eval<kActGelu>(g, value, slope); break;
    case kActRelu: gate_eval<kActRelu>(g, value, slope); break;
    case kActSigmoid: gate_eval<kActSigmoid>(g, value, slope); break;
    default: gate_eval<kActIdentity>(g, value, slope); break;
    }
    return value;
}

// The result of a row and feature; `at`: its place in y, `bias`: that of the feature, `gate`: the second sum of kGatedRows.
template <int DT, int END>
__device__ __forceinline__ float finish(const LinearArgs& a, float sum, float bias, float gate, int64_t at, int feature)
{
    using H = Half2<DT>;
    if constexpr (END == kPlainRows) {
        return a.bias ? sum + bias : sum;
    } else if constexpr (END == kGeluRows) {
        return gelu_fwd(bias + H::round(sum));
    } else if constexpr (END == kGatedRows) {
        return gate_of(a.act, H::round(gate)) * H::round(sum);
    } else {
        const float v = H::round(sum) + bias, residual = H::from_bits(a.residual[at]);
        if (!a.x1) return residual + v;
        float t = H::from_bits(a.x1[at]);
        if (a.bias1) t = H::round(t + H::from_bits(a.bias1[feature]));
        return residual + H::round(t + v);
    }
}

// MT: tiles of 16 rows of x
template <int DT, int MT, int END>
__global__ void __launch_bounds__(64 * kLinearWaves) linear_decode_kernel(LinearArgs a)
{
    __shared__ __attribute__((aligned(1024))) char ring[kLinearWaves * kRing * kPieceBytes];
    __shared__ float sums[2][2 * kLinearWaves][16 * MT][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int split_bits = a.splits == 1 ? 0 : kLinearSplitBits;
    const int split = blockIdx.x & (a.splits - 1), first_tile = blockIdx.x >> split_bits, stride = gridDim.x >> split_bits;
    // groups of 32 features are dealt out evenly to the waves of all splits, a wave's being consecutive
    const int groups = a.k / 32, share = split * kLinearWaves + wave, share_bits = kLinearWaveBits + split_bits;
    const int lo = groups * share >> share_bits, count = (groups * (share + 1) >> share_bits) - lo;
    const int mid = (groups * (2 * share + 1) >> (share_bits + 1)) - lo;   // steps of the wave's first sum
    constexpr int kParts = END == kGatedRows ? 2 : 1;   // tiles of a result: its values, its gates
    const int tiles = a.n / 16 / kParts, pieces = (count + 1) / 2;

    u32x4 x[MT][kLinearSteps];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const uint16_t* xp = a.x + (int64_t)min(i * 16 + r16, a.m - 1) * a.k + lo * 32 + g * 8;
#pragma unroll
        for (int s = 0; s < kLinearSteps; ++s) x[i][s] = s < count ? load16(xp + s * 32) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int s = 0; s < kLinearSteps; ++s) arrive(x[i][s]);

    char* const mine = ring + wave * kRing * kPieceBytes;
    const uint32_t mine_at = __builtin_amdgcn_readfirstlane(lds_address(mine));
    // chunk c of row r sits in slot c ^ (r & 7); a load takes 8 rows. The last piece of an odd count has 4 chunks a row.
    const int slot = lane & 7, row8 = lane >> 3;
    const uint32_t whole = (uint32_t)row8 * a.k * 2 + ((slot ^ row8) * 16), half = (uint32_t)row8 * a.k * 2 + (((slot ^ row8) & 3) * 16);
    const uint16_t* w0 = a.w + lo * 32;
    auto fetch = [&](int tile, int piece, int at) {
        const uint16_t* w = w0 + (int64_t)tile * 16 * a.k + piece * 64;
        const uint32_t offset = 2 * piece + 1 < count ? whole : half;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            TileLoader<128>::issue(reinterpret_cast<const char*>(w + (int64_t)i * 8 * a.k), offset, mine_at + at * kPieceBytes + i * 1024);
    };
    // all pieces of all tiles, one after the other
    int left = first_tile < tiles ? ((tiles - 1 - first_tile) / stride + 1) * pieces * kParts : 0;
    int next_tile = first_tile, next_part = 0, next_piece = 0, next_at = 0;
    auto fetch_next = [&]() {
        fetch(next_tile + next_part * tiles, next_piece, next_at);
        if (++next_piece == pieces) {
            next_piece = 0;
            if (++next_part == kParts) {
                next_part = 0;
                next_tile += stride;
            }
        }
        next_at = next_at + 1 == kRing ? 0 : next_at + 1;
    };
    for (int ahead = 0; ahead < kRing - 1 && ahead < left; ++ahead) fetch_next();
    const char* frag = mine + r16 * 128;
    const int sw = r16 & 7;

    int buf = 0, at = 0;
    for (int tile = first_tile; tile < tiles; tile += stride) {
        float value = 0.0f;   // kGatedRows: the first of the two sums
        for (int part = 0; part < kParts; ++part) {
            f32x4 acc[2][MT];
#pragma unroll
            for (int r = 0; r < MT; ++r) acc[0][r] = acc[1][r] = f32x4{};
            auto multiply = [&](const u32x4& w, int step) {   // (a constant after unrolling)
                if (step < mid)
#pragma unroll
                    for (int r = 0; r < MT; ++r) acc[0][r] = mma16<DT>(w, x[r][step], acc[0][r]);
                else
#pragma unroll
                    for (int r = 0; r < MT; ++r) acc[1][r] = mma16<DT>(w, x[r][step], acc[1][r]);
            };
#pragma unroll
            for (int p = 0; p < kLinearSteps / 2; ++p) {
                if (p >= pieces) continue;
                if (left >= kRing - 1) wait_pieces<2 * (kRing - 2)>();
                else wait_pieces<0>();
                if (left >= kRing) fetch_next();
                --left;
                const char* f = frag + at * kPieceBytes;
                at = at + 1 == kRing ? 0 : at + 1;
                const u32x4 w_lo = lds_read16(f + ((g ^ sw) << 4)), w_hi = lds_read16(f + (((4 + g) ^ sw) << 4));
                multiply(w_lo, 2 * p);
                if (2 * p + 1 < count) multiply(w_hi, 2 * p + 1);
            }
#pragma unroll
            for (int r = 0; r < MT; ++r)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    sums[buf][2 * wave][r * 16 + r16][4 * g + j] = acc[0][r][j];
                    sums[buf][2 * wave + 1][r * 16 + r16][4 * g + j] = acc[1][r][j];
                }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            // (a wave is at most one tile ahead of those that add up here: the other half of the sums is free)
            const int row = tid >> 4, col = tid & 15;
            if (row < a.m && row < 16 * MT) {
                float v = 0.0f;
#pragma unroll
                for (int s = 0; s < 2 * kLinearWaves; ++s) v += sums[buf][s][row][col];
                if (a.splits > 1) {
                    a.parts[((int64_t)split * a.m + row) * a.n + (tile + part * tiles) * 16 + col] = v;
                } else if (part + 1 < kParts) {
                    value = v;
                } else {
                    const int64_t to = (int64_t)row * (a.n / kParts) + tile * 16 + col;
                    const float bias = END == kGatedRows ? 0.0f : bias_of<DT>(a, tile, col);
                    float result = finish<DT, END>(a, kParts == 2 ? value : v, bias, v, to, tile * 16 + col);
                    asm volatile("" : "+v"(result));   // in fp32, not a product that is rounded to fp16 at once
                    a.y[to] = Half2<DT>::to_bits(result);
                }
            }
            buf ^= 1;
        }
    }
}

// Adds the splits up, four columns per thread.
template <int DT, int END>
__global__ void __launch_bounds__(256) linear_merge_kernel(LinearArgs a)
{
    constexpr int kParts = END == kGatedRows ? 2 : 1;
    const int width = a.n / kParts;
    const int64_t size = (int64_t)a.m * a.n, at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (at >= size / kParts) return;
    const int row = (int)(at / width), feature = (int)(at % width);
    f32x4 v[kParts];
#pragma unroll
    for (int p = 0; p < kParts; ++p) {
        v[p] = f32x4{};
#pragma unroll
        for (int s = 0; s < kLinearSplits; ++s)
            v[p] += *reinterpret_cast<const f32x4*>(a.parts + s * size + (int64_t)row * a.n + p * width + feature);
    }
    float out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float bias = END != kGatedRows && a.bias ? Half2<DT>::from_bits(a.bias[feature + j]) : 0.0f;
        out[j] = finish<DT, END>(a, v[0][j], bias, v[kParts - 1][j], at + j, feature + j);
    }
    *reinterpret_cast<u32x2*>(a.y + at) = u32x2{Half2<DT>::pack(out[0], out[1]), Half2<DT>::pack(out[2], out[3])};
}

template <int DT, int END>
static int launch_linear(const LinearArgs& a, hipStream_t st)
{
    launch_prepare();
    const int width = END == kGatedRows ? a.n / 2 : a.n, tiles = width / 16, most = kLinearBlocks / a.splits;
    const dim3 blocks((unsigned)((tiles < most ? tiles : most) * a.splits)), threads(64 * kLinearWaves);
    if (a.m <= 16) linear_decode_kernel<DT, 1, END><<<blocks, threads, 0, st>>>(a);
    else linear_decode_kernel<DT, 2, END><<<blocks, threads, 0, st>>>(a);
    if (a.splits > 1) linear_merge_kernel<DT, END><<<dim3((unsigned)(((int64_t)a.m * width / 4 + 255) / 256)), dim3(256), 0, st>>>(a);
    return launch_result();
}

template <int END>
static int linear_rows(LinearArgs a, int dtype, void* stream)
{
    if (!a.y || !a.x || !a.w) return NHP_ERR_NULL;
    if (!ptr_aligned16(a.x) || !ptr_aligned16(a.w) || !ptr_aligned16(a.y) || !ptr_aligned16(a.parts)) return NHP_ERR_SHAPE;
    a.splits = a.k > kLinearWhole ? kLinearSplits : 1;
    if (a.splits > 1 && !a.parts) return NHP_ERR_NULL;
    a.bias_words = (reinterpret_cast<uintptr_t>(a.bias) & 3) == 0;
    if (dtype == NHP_BF16) return launch_linear<NHP_BF16, END>(a, static_cast<hipStream_t>(stream));
    if (dtype == NHP_F16) return launch_linear<NHP_F16, END>(a, static_cast<hipStream_t>(stream));
    return NHP_ERR_DTYPE;
}

static bool linear_sizes_ok(int64_t rows, int64_t out_features, int64_t in_features, int64_t multiple)
{
    return rows >= 1 && rows <= 32 && out_features >= multiple && out_features % multiple == 0 && out_features <= (1 << 24) &&
           in_features >= 32 && in_features % 32 == 0 && in_features <= kLinearWhole * kLinearSplits;
}

static LinearArgs linear_args(void* y, const void* x, const void* weight, const void* bias, void* workspace, int64_t rows,
                              int64_t out_features, int64_t in_features)
{
    LinearArgs a{};
    a.y = static_cast<uint16_t*>(y);
    a.x = static_cast<const uint16_t*>(x);
    a.w = static_cast<const uint16_t*>(weight);
    a.bias = static_cast<const uint16_t*>(bias);
    a.parts = static_cast<float*>(workspace);
    a.m = (int)rows;
    a.n = (int)out_features;
    a.k = (int)in_features;
    return a;
}

}  // namespace nhp

extern "C" {

int64_t nhp_linear_decode_workspace_bytes(int64_t rows, int64_t out_features, int64_t in_features)
{
    using namespace nhp;
    return in_features > kLinearWhole ? kLinearSplits * rows * out_features * 4 : 0;
}

int nhp_linear_decode(void* y, const void* x, const void* weight, const void* bias, void* workspace, int64_t rows,
                      int64_t out_features, int64_t in_features, int dtype, void* stream)
{
    using namespace nhp;
    if (!linear_sizes_ok(rows, out_features, in_features, 16)) return !y || !x || !weight ? NHP_ERR_NULL : NHP_ERR_SHAPE;
    return linear_rows<kPlainRows>(linear_args(y, x, weight, bias, workspace, rows, out_features, in_features), dtype, stream);
}

int nhp_linear_decode_act(void* y, const void* x, const void* weight, const void* bias, void* workspace, int64_t rows,
                          int64_t out_features, int64_t in_features, int act, int dtype, void* stream)
{
    using namespace nhp;
    const bool gelu = act == NHP_LINEAR_BIAS_GELU;
    if (!y || !x || !weight) return NHP_ERR_NULL;
    if (!gelu && (act < NHP_GATE_SWISH || act > NHP_GATE_IDENTITY || bias)) return NHP_ERR_SHAPE;
    if (!linear_sizes_ok(rows, out_features, in_features, gelu ? 16 : 32)) return NHP_ERR_SHAPE;
    LinearArgs a = linear_args(y, x, weight, bias, workspace, rows, out_features, in_features);
    a.act = act;
    return gelu ? linear_rows<kGeluRows>(a, dtype, stream) : linear_rows<kGatedRows>(a, dtype, stream);
}

int nhp_linear_decode_add(void* y, const void* x, const void* weight, const void* bias, const void* x1, const void* bias1,
                          const void* residual, void* workspace, int64_t rows, int64_t out_features, int64_t in_features, int dtype,
                          void* stream)
{
    using namespace nhp;
    if (!y || !x || !weight || !residual || (bias1 && !x1)) return NHP_ERR_NULL;
    if (!linear_sizes_ok(rows, out_features, in_features, 16)) return NHP_ERR_SHAPE;
    LinearArgs a = linear_args(y, x, weight, bias, workspace, rows, out_features, in_features);
    a.x1 = static_cast<const uint16_t*>(x1);
    a.bias1 = static_cast<const uint16_t*>(bias1);
    a.residual = static_cast<const uint16_t*>(residual);
    return linear_rows<kAddRows>(a, dtype, stream);
}

}  // extern "C"
