// y = x W^T (+ bias) for the few rows of a decoding step (at most 32), 16-bit storage, fp32 sums.
//
// Such a product reads every weight once for a handful of rows: the weights' bytes are its time, and the matrix cores idle.
// What a CU can have on the way is the limit, so x must not take much of it: read again for every 16 weight rows it costs
// as much as the weights. One workgroup of 16 waves per CU walks over tiles of 16 weight rows; the waves share the
// contraction, and each keeps its part of x in registers for all tiles. Beyond 4096 features (8 steps of 32 for each
// wave) four workgroups share the contraction of a tile and a second kernel adds their sums up.
// Weights go from memory into registers, the next ones always under way, also across tiles.
// Measured with weights that are not in any cache (16 rows, library -> here; time of the weights' bytes at 5.1 TB/s):
// [22016, 4096] 51.7 -> 43.5 us (35.4), [12288, 4096] 26.7 -> 23.8 (19.7), [4096, 11008] 38.2 -> 27.6 (17.7).
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
};

constexpr int kLinearWaves = 16, kLinearBlocks = 256, kLinearSteps = 8, kLinearPart = 4;
constexpr int kLinearWhole = kLinearSteps * kLinearWaves * 32, kLinearSplits = 4;   // features of an unsplit product; splits beyond

// MT: tiles of 16 rows of x
template <int DT, int MT>
__global__ void __launch_bounds__(64 * kLinearWaves) linear_decode_kernel(LinearArgs a)
{
    constexpr int kParts = kLinearSteps / kLinearPart;
    static_assert(kParts * kLinearPart == kLinearSteps && kParts % 2 == 0, "an even number of parts");
    __shared__ float sums[2][kLinearWaves][16 * MT][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int split = blockIdx.x % a.splits, first_tile = blockIdx.x / a.splits, stride = gridDim.x / a.splits;
    // groups of 32 features are dealt out evenly to the waves of all splits, a wave's being consecutive
    const int groups = a.k / 32, shares = kLinearWaves * a.splits, share = split * kLinearWaves + wave;
    const int lo = groups * share / shares, count = groups * (share + 1) / shares - lo;
    const int tiles = a.n / 16;
    const uint16_t* w0 = a.w + lo * 32;
    const uint32_t at = (uint32_t)r16 * a.k + g * 8;
    u32x4 part[2][kLinearPart];
    auto load = [&](u32x4 (&p)[kLinearPart], int tile, int first) {
        const uint16_t* w = w0 + (int64_t)tile * 16 * a.k + first * 32;
#pragma unroll
        for (int s = 0; s < kLinearPart; ++s)
            if (first + s < count) p[s] = load16_stream(w + s * 32 + at);
        asm volatile("" ::: "memory");   // not put off until they are needed
    };
    load(part[0], first_tile, 0);
    u32x4 x[MT][kLinearSteps];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const uint16_t* xp = a.x + (int64_t)min(i * 16 + r16, a.m - 1) * a.k + lo * 32 + g * 8;
#pragma unroll
        for (int s = 0; s < kLinearSteps; ++s) x[i][s] = s < count ? load16(xp + s * 32) : u32x4{0, 0, 0, 0};
    }

    int buf = 0;
    for (int tile = first_tile; tile < tiles; tile += stride) {
        f32x4 acc[MT];
#pragma unroll
        for (int r = 0; r < MT; ++r) acc[r] = f32x4{};
#pragma unroll
        for (int i = 0; i < kParts; ++i) {
            if (i + 1 < kParts) load(part[(i + 1) & 1], tile, (i + 1) * kLinearPart);
            else if (tile + stride < tiles) load(part[0], tile + stride, 0);
#pragma unroll
            for (int s = 0; s < kLinearPart; ++s)
                if (i * kLinearPart + s < count) {
#pragma unroll
                    for (int r = 0; r < MT; ++r) acc[r] = mma16<DT>(part[i & 1][s], x[r][i * kLinearPart + s], acc[r]);
                }
        }
#pragma unroll
        for (int r = 0; r < MT; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) sums[buf][wave][r * 16 + r16][4 * g + j] = acc[r][j];
        __syncthreads();
        // (a wave is at most one tile ahead of those that add up here: the other half of the sums is free)
        const int row = tid >> 4, col = tid & 15;
        if (row < a.m) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < kLinearWaves; ++s) v += sums[buf][s][row][col];
            const int64_t to = (int64_t)row * a.n + tile * 16 + col;
            if (a.splits > 1) {
                a.parts[(int64_t)split * a.m * a.n + to] = v;
            } else {
                if (a.bias) v += Half2<DT>::from_bits(a.bias[tile * 16 + col]);
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
                       (int)in_features, splits};
    if (dtype == NHP_BF16) return launch_linear<NHP_BF16>(a, static_cast<hipStream_t>(stream));
    if (dtype == NHP_F16) return launch_linear<NHP_F16>(a, static_cast<hipStream_t>(stream));
    return NHP_ERR_DTYPE;
}

}  // extern "C"
