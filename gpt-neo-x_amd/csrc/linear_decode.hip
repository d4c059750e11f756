// y = x W^T (+ bias) for the few rows of a decoding step (at most 32), 16-bit storage, fp32 sums.
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
//   [22016, 4096] 43.9 -> 37.5 (27.5)   [12288, 4096] 26.2 -> 22.5 (16.1)   [4096, 11008] 27.9 -> 22.0 (14.5)
//   [7680, 2560] 16.0 -> 11.5           [768, 3072] 8.6 -> 6.5              [4096, 4096] 12.2 -> 11.4 (6.4)
// A ring of 6 or 7 pieces, or two workgroups per CU, are no faster; reading x costs 2 to 3 us of it (one row: 33.7, 20.2).
//
// Rows of the matrix instruction (16 x 16 x 32) are weight rows, its columns the rows of x. A lane takes 16 consecutive
// bytes of its row per instruction and x in the same order, which the contraction does not mind.
#include "attention.hpp"

namespace nhp {

struct LinearArgs {
    uint16_t* y;
    const uint16_t *x, *w, *bias;
    float* parts;   // with splits > 1: [splits][m][n]
    int m, n, k, splits;
    int bias_words;   // the bias starts at a multiple of four bytes
};

constexpr int kLinearWaves = 8, kLinearBlocks = 256, kLinearSteps = 16;   // steps of 32 features that a wave has at most
constexpr int kLinearWhole = kLinearSteps * kLinearWaves * 32, kLinearSplits = 4;   // features of an unsplit product; splits beyond
constexpr int kRing = 4, kPieceBytes = 2048;   // pieces of 16 rows x 64 features in LDS for each wave

template <int N>
__device__ __forceinline__ void wait_pieces()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// MT: tiles of 16 rows of x
template <int DT, int MT>
__global__ void __launch_bounds__(64 * kLinearWaves) linear_decode_kernel(LinearArgs a)
{
    __shared__ __attribute__((aligned(1024))) char ring[kLinearWaves * kRing * kPieceBytes];
    __shared__ float sums[2][kLinearWaves][16 * MT][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int split = blockIdx.x % a.splits, first_tile = blockIdx.x / a.splits, stride = gridDim.x / a.splits;
    // groups of 32 features are dealt out evenly to the waves of all splits, a wave's being consecutive
    const int groups = a.k / 32, shares = kLinearWaves * a.splits, share = split * kLinearWaves + wave;
    const int lo = __builtin_amdgcn_readfirstlane(groups * share / shares), count = __builtin_amdgcn_readfirstlane(groups * (share + 1) / shares - lo);
    const int tiles = a.n / 16, pieces = (count + 1) / 2;

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
    int left = first_tile < tiles ? ((tiles - 1 - first_tile) / stride + 1) * pieces : 0;
    int next_tile = first_tile, next_piece = 0, next_at = 0;
    auto fetch_next = [&]() {
        fetch(next_tile, next_piece, next_at);
        if (++next_piece == pieces) {
            next_piece = 0;
            next_tile += stride;
        }
        next_at = next_at + 1 == kRing ? 0 : next_at + 1;
    };
    for (int ahead = 0; ahead < kRing - 1 && ahead < left; ++ahead) fetch_next();
    const char* frag = mine + r16 * 128;
    const int sw = r16 & 7;

    int buf = 0, at = 0;
    for (int tile = first_tile; tile < tiles; tile += stride) {
        f32x4 acc[MT];
#pragma unroll
        for (int r = 0; r < MT; ++r) acc[r] = f32x4{};
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
#pragma unroll
            for (int r = 0; r < MT; ++r) acc[r] = mma16<DT>(w_lo, x[r][2 * p], acc[r]);
            if (2 * p + 1 < count)
#pragma unroll
                for (int r = 0; r < MT; ++r) acc[r] = mma16<DT>(w_hi, x[r][2 * p + 1], acc[r]);
        }
#pragma unroll
        for (int r = 0; r < MT; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) sums[buf][wave][r * 16 + r16][4 * g + j] = acc[r][j];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // (a wave is at most one tile ahead of those that add up here: the other half of the sums is free)
        const int row = tid >> 4, col = tid & 15;
        if (row < a.m && row < 16 * MT) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < kLinearWaves; ++s) v += sums[buf][s][row][col];
            const int64_t to = (int64_t)row * a.n + tile * 16 + col;
            if (a.splits > 1) {
                a.parts[(int64_t)split * a.m * a.n + to] = v;
            } else {
                if (a.bias && a.bias_words) {
                    // by scalar loads: a vector load would be waited for behind the pieces that are under way
                    const uint32_t* words = reinterpret_cast<const uint32_t*>(a.bias + tile * 16);
                    uint32_t w = words[0];
#pragma unroll
                    for (int q = 1; q < 8; ++q) w = col >> 1 == q ? words[q] : w;
                    v += col & 1 ? Half2<DT>::hi(w) : Half2<DT>::lo(w);
                } else if (a.bias) {
                    v += Half2<DT>::from_bits(a.bias[tile * 16 + col]);
                }
                a.y[to] = Half2<DT>::to_bits(v);
            }
        }
        buf ^= 1;
    }
}

// Adds the splits up, four columns per thread.
template <int DT>
__global__ void __launch_bounds__(256) linear_merge_kernel(LinearArgs a)
{
    const int64_t size = (int64_t)a.m * a.n, at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (at >= size) return;
    f32x4 v{};
#pragma unroll
    for (int s = 0; s < kLinearSplits; ++s) v += *reinterpret_cast<const f32x4*>(a.parts + s * size + at);
    if (a.bias)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += Half2<DT>::from_bits(a.bias[(int)(at % a.n) + j]);
    *reinterpret_cast<u32x2*>(a.y + at) = u32x2{Half2<DT>::pack(v[0], v[1]), Half2<DT>::pack(v[2], v[3])};
}

template <int DT>
static int launch_linear(const LinearArgs& a, hipStream_t st)
{
    launch_prepare();
    const int tiles = a.n / 16, most = kLinearBlocks / a.splits;
    const dim3 blocks((unsigned)((tiles < most ? tiles : most) * a.splits)), threads(64 * kLinearWaves);
    if (a.m <= 16) linear_decode_kernel<DT, 1><<<blocks, threads, 0, st>>>(a);
    else linear_decode_kernel<DT, 2><<<blocks, threads, 0, st>>>(a);
    if (a.splits > 1) linear_merge_kernel<DT><<<dim3((unsigned)(((int64_t)a.m * a.n / 4 + 255) / 256)), dim3(256), 0, st>>>(a);
    return launch_result();
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
    if (!y || !x || !weight) return NHP_ERR_NULL;
    if (rows < 1 || rows > 32 || out_features < 16 || out_features % 16 || in_features < 32 || in_features % 32) return NHP_ERR_SHAPE;
    if (in_features > kLinearWhole * kLinearSplits || out_features > (1 << 24)) return NHP_ERR_SHAPE;
    if (!ptr_aligned16(x) || !ptr_aligned16(weight) || !ptr_aligned16(y)) return NHP_ERR_SHAPE;
    const int splits = in_features > kLinearWhole ? kLinearSplits : 1;
    if (splits > 1 && !workspace) return NHP_ERR_NULL;
    if (!ptr_aligned16(workspace)) return NHP_ERR_SHAPE;
    const LinearArgs a{static_cast<uint16_t*>(y), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(weight),
                       static_cast<const uint16_t*>(bias), static_cast<float*>(workspace), (int)rows, (int)out_features,
                       (int)in_features, splits, (reinterpret_cast<uintptr_t>(bias) & 3) == 0};
    if (dtype == NHP_BF16) return launch_linear<NHP_BF16>(a, static_cast<hipStream_t>(stream));
    if (dtype == NHP_F16) return launch_linear<NHP_F16>(a, static_cast<hipStream_t>(stream));
    return NHP_ERR_DTYPE;
}

}  // extern "C"
