// y = x W^T (+ bias) for the rows of a short prompt or of many sequences: 16-bit storage, fp32 sums on the matrix cores.
//
// A workgroup has a 64 x 64 tile of y, each of its four waves 32 x 32 of that; 64 features of both operands a step arrive in LDS by
// direct loads, three steps ahead. What bounds it is the chain of steps of a tile: 0.3 to 0.5 us each, the time of a memory access
// over the depth of the ring. Small tiles fill the CUs here; tiles of 128 x 128 or 64 x 128, or a contraction split among workgroups
// (a second launch that adds up: 3 to 6 us), took longer at all sizes that nhp_linear_tiles_pay takes. Two groups of waves that take
// the steps in turn are up to 15 % faster with 2048 features, but add up in another order than a pass with gradients does: here the
// features come one after the other, and the results were the library's bit for bit at all 86 sizes compared (bf16, 33 to 512 rows).
//
// Measured, weights not in any cache (340 MB of them in turn), us here/library, whose call costs the host 25 us besides, this one 5;
// sizes in brackets are not taken, those with a dash were not looked at:
//   rows            33          64          96          128         192         256         320         512         1024        2048        4096
//   [16, 768]       4.5/5.1     4.6/6.6     4.6/6.9     4.6/7.3     4.5/8.6     4.7/8.0     4.7/4.9     4.7/4.9     4.8/4.9     4.8/4.9     4.9/5.0
//   [256, 768]      4.9/9.9     5.0/9.8     5.0/12.5    5.0/12.2    5.1/15.6    5.1/17.5    5.1/6.7     5.1/6.7     5.1/6.9     5.2/7.1     5.4/7.5
//   [768, 768]      5.7/8.9     6.1/9.4     5.7/8.9     6.0/8.9     6.1/9.0     5.9/8.6     6.1/8.6     5.9/9.0     6.0/9.3     8.2/10.5    [13.4/12.3]
//   [2304, 768]     5.8/9.2     6.3/9.5     5.9/9.1     6.2/10.2    6.4/9.5     6.2/9.7     6.5/9.7     8.1/10.4    [11.7/12.3] [18.4/15.9] -
//   [128, 1024]     5.7/7.8     5.8/8.2     5.8/7.9     5.9/7.8     5.9/7.8     6.0/7.8     6.0/7.9     6.0/7.9     6.0/8.0     6.0/8.0     6.2/8.5
//   [1024, 1024]    6.7/10.9    7.2/11.3    6.8/10.7    7.1/10.7    7.0/10.6    7.0/10.3    7.0/11.0    7.0/10.7    7.1/11.2    11.1/12.2   [21.5/14.4]
//   [4096, 1024]    6.9/11.2    7.5/11.7    7.0/12.0    7.4/12.3    7.4/13.2    7.4/12.0    10.5/12.7   11.2/13.1   [20.1/14.5] -           -
//   [512, 512]      4.1/6.4     4.1/6.8     4.1/7.6     4.1/7.7     4.2/6.3     4.2/6.4     4.2/6.4     4.2/6.5     4.3/7.0     4.5/7.2     6.3/8.4
//   [2048, 64]      2.5/3.5     2.6/3.7     2.6/4.1     2.6/4.2     2.6/3.6     2.6/3.7     2.7/3.9     2.8/4.0     3.3/4.8     [5.2/5.9]   -
//   [2048, 2048]    -           -           -           -           -           11.4/11.9   11.4/12.8   11.5/12.7   -           -           -
//   [3072, 2048]    -           -           -           -           11.8/21.5   11.8/13.2   11.8/13.2   -           -           -           -
//   [6144, 2048]    -           -           12.4/14.2   13.0/15.5   [19.3/22.2] -           -           -           -           -           -
//   [8192, 2048]    14.2/15.2   14.8/14.8   14.6/15.6   15.3/16.7   -           -           -           -           -           -           -
//   [2560, 2560]    -           -           -           -           [15.1/14.4] 15.1/16.1   15.1/16.0   -           -           -           -
//   [7680, 2560]    [16.9/17.5] [18.4/17.6] 16.8/18.4   18.0/20.2   -           -           -           -           -           -           -
//   [2048, 4096]    -           -           -           -           -           20.2/16.1   20.3/21.6   20.5/21.2   -           -           -
//   [4096, 4096]    -           -           20.0/22.4   21.5/24.8   21.5/33.3   21.4/22.8   -           -           -           -           -
//   [6144, 4096]    -           -           21.5/23.5   22.8/25.9   [35.0/33.8] -           -           -           -           -           -
// Behind the library on the GPU, and taken for the host's time all the same:
//  - up to 160 tiles with more than 3584 features, where the library splits the contraction at some numbers of rows:
//    [4096, 4096] at 80 rows 19.6/17.1, at 112 20.6/17.1, [3072, 4096] at 160 19.6/16.8, [2048, 4096] at 256 20.2/16.1,
//  - 128 tiles with 2048 rows of weights or 112 of x beyond 2048 features, by up to 7 %: [2048, 2560] at 256 14.8/13.8,
//  - with weights that stay in the caches (16 sets of them in turn) [768, 768] up to 192 rows, 5.5/5.0, [256, 768] at
//    320 and 768 rows, 5.6/5.0, and 128 to 144 tiles of 2048 features, [2048, 2048] at 256 10.5/9.9, [3072, 2048] at 160 10.5/9.5.
// The host is what a program waits for that does not capture its layers: a layer of 4096 features (gated) without gradient at 70 / 120
// rows takes 221 / 208 us here and 273 / 228 with [4096, 4096] left to the library; in a captured graph 176 / 179 and 173 / 176. With
// all products the library's and the former host path, 349 / 301 and 172 / 175.
// Other whole layers, step by step / captured, before this kernel and the native calls -> here: 768 features, 40 rows, 298 / 56 ->
// 150 / 51; 1024, 100 rows, 269 / 71 -> 144 / 60; 2048 (16 heads), 100 rows, 273 / 87 -> 167 / 84, 200 rows 270 / 107 -> 198 / 105;
// 4096 (gated), 200 rows, 312 / 213 -> 207 / 207.
#include "attention.hpp"

namespace nhp {

struct TilesArgs {
    uint16_t* y;
    const uint16_t *x, *w, *bias;
    int m, n, k, n_tiles;
};

constexpr int kTileRows = 64;                       // of x and of W
constexpr int kTileStep = 64;                       // features per step: rows of 128 bytes in LDS
constexpr int kTileStages = 4;
constexpr int kTileLoads = 2 * kTileRows / 8 / 4;   // 1 KiB loads of a wave per step, the first half of x
constexpr int kTileStageBytes = 2 * kTileRows * 128;

template <int N>
__device__ __forceinline__ void wait_for_loads()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 16 bytes per lane from memory to LDS (see TileLoader::issue)
__device__ __forceinline__ void load_to_lds(const uint16_t* base, uint32_t offset, uint32_t dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(offset), "s"(base) : "memory", "m0");
}

template <int DT>
__global__ void __launch_bounds__(256, 2) linear_tiles_kernel(TilesArgs a)
{
    using F = Frag<DT>;
    __shared__ __attribute__((aligned(1024))) char lds[kTileStages * kTileStageBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, half = lane >> 5;
    // workgroups of one XCD take neighbouring tiles, the tiles of the same weights first
    const int tiles = gridDim.x, m_tiles = tiles / a.n_tiles;
    const int id = tiles % 8 ? blockIdx.x : (blockIdx.x & 7) * (tiles / 8) + (blockIdx.x >> 3);
    const int m0 = id % m_tiles * kTileRows, n0 = id / m_tiles * kTileRows;
    const int steps = a.k / kTileStep;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
    // chunk c of row r lies at slot c ^ (r >> 1 & 7): the 32 rows of a read fall on all banks evenly
    const int swizzle = (half ^ (l32 >> 1 & 7)) << 4;
    const int x_frag = (wm * 32 + l32) * 128 + swizzle, w_frag = (kTileRows + wn * 32 + l32) * 128 + swizzle;

    uint32_t offset[kTileLoads];
#pragma unroll
    for (int i = 0; i < kTileLoads; ++i) {
        const int row = (wave * (kTileLoads / 2) + i % (kTileLoads / 2)) * 8 + (lane >> 3);
        const int last = i < kTileLoads / 2 ? a.m - 1 - m0 : a.n - 1 - n0;   // rows past the end repeat the last one
        offset[i] = (uint32_t)min(row, last) * (uint32_t)(a.k * 2) + (((lane & 7) ^ (row >> 1 & 7)) << 4);
    }
    const uint16_t* xb = a.x + (int64_t)m0 * a.k;
    const uint16_t* wb = a.w + (int64_t)n0 * a.k;
    auto fetch = [&](int step, int buf) {
        const uint32_t dst = lds0 + buf * kTileStageBytes + wave * (kTileLoads / 2) * 1024;
#pragma unroll
        for (int i = 0; i < kTileLoads / 2; ++i) load_to_lds(xb + step * kTileStep, offset[i], dst + i * 1024);
#pragma unroll
        for (int i = 0; i < kTileLoads / 2; ++i)
            load_to_lds(wb + step * kTileStep, offset[kTileLoads / 2 + i], dst + kTileRows * 128 + i * 1024);
    };

    f32x16 acc = {};
#pragma unroll
    for (int s = 0; s < kTileStages - 1; ++s)
        if (s < steps) fetch(s, s);
    for (int step = 0; step < steps; ++step) {
        const int buf = step % kTileStages;
        if (step + kTileStages - 1 <= steps) wait_for_loads<(kTileStages - 2) * kTileLoads>();
        else wait_for_loads<0>();
        __syncthreads();   // this step has arrived, and everybody has read the one before
        if (step + kTileStages - 1 < steps) fetch(step + kTileStages - 1, (step + kTileStages - 1) % kTileStages);
        const char* base = lds + buf * kTileStageBytes;
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = F::mma(lds_read16(base + (w_frag ^ (t << 5))), lds_read16(base + (x_frag ^ (t << 5))), acc);
    }

    // lane & 31 is the row of x, the registers are features: 16 of them at a time, two lanes put together 32 bytes
    const int row = m0 + wm * 32 + l32, nb = n0 + wn * 32;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (nb + j * 16 >= a.n) continue;   // n is a multiple of 16
        float add[8] = {};
        if (a.bias) {
            const u32x2 lo = load8(a.bias + nb + j * 16 + half * 4), hi = load8(a.bias + nb + j * 16 + 8 + half * 4);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                add[2 * i] = Half2<DT>::lo(lo[i]);
                add[2 * i + 1] = Half2<DT>::hi(lo[i]);
                add[4 + 2 * i] = Half2<DT>::lo(hi[i]);
                add[4 + 2 * i + 1] = Half2<DT>::hi(hi[i]);
            }
        }
        const uint32_t x0 = Half2<DT>::pack(acc[8 * j] + add[0], acc[8 * j + 1] + add[1]);
        const uint32_t x1 = Half2<DT>::pack(acc[8 * j + 2] + add[2], acc[8 * j + 3] + add[3]);
        const uint32_t y0 = Half2<DT>::pack(acc[8 * j + 4] + add[4], acc[8 * j + 5] + add[5]);
        const uint32_t y1 = Half2<DT>::pack(acc[8 * j + 6] + add[6], acc[8 * j + 7] + add[7]);
        const auto r0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
        const auto r1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
        const u32x4 chunk = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
        if (row < a.m) *reinterpret_cast<u32x4*>(a.y + (int64_t)row * a.n + nb + j * 16 + half * 8) = chunk;
    }
}

static int64_t linear_tiles(int64_t rows, int64_t out_features)
{
    return ((rows + kTileRows - 1) / kTileRows) * ((out_features + kTileRows - 1) / kTileRows);
}

}  // namespace nhp

extern "C" {

// Contractions of up to 1024 features as long as all tiles run at once, two a CU (beyond one a CU up to 4096 rows: [128, 1024] at
// 16384 is 11.9 us, 10.3 in the library); longer ones where a tile has a CU to itself and at least half of the CUs have one, and
// beyond 2048 features where the weights are read for more than one row of tiles. Outside of that the library is ahead or the two
// take turns: with fewer tiles it splits the contraction, with more its larger ones read less. Where the rule takes sizes for the
// host's time only, the table above says so.
int nhp_linear_tiles_pay(int64_t rows, int64_t out_features, int64_t in_features)
{
    using namespace nhp;
    if (rows < 1 || rows > (1 << 24) || out_features < 16 || out_features > (1 << 24) || out_features % 16 || in_features < kTileStep ||
        in_features % kTileStep)
        return 0;
    const int64_t tiles = linear_tiles(rows, out_features);
    if (in_features <= 1024) return tiles <= 256 || (tiles <= 512 && rows <= 4096);
    return in_features <= 4096 && tiles >= 128 && tiles <= 256 && (in_features <= 2048 || rows > kTileRows);
}

int nhp_linear_tiles(void* y, const void* x, const void* weight, const void* bias, int64_t rows, int64_t out_features,
                     int64_t in_features, int dtype, void* stream)
{
    using namespace nhp;
    if (!y || !x || !weight) return NHP_ERR_NULL;
    if (rows < 1 || rows > (1 << 24) || out_features < 16 || out_features > (1 << 24) || out_features % 16 || in_features < kTileStep ||
        in_features > 65536 || in_features % kTileStep || linear_tiles(rows, out_features) > (1 << 24))
        return NHP_ERR_SHAPE;
    if (!ptr_aligned16(x) || !ptr_aligned16(weight) || !ptr_aligned16(y) || !ptr_aligned16(bias)) return NHP_ERR_SHAPE;
    TilesArgs a{};
    a.y = static_cast<uint16_t*>(y);
    a.x = static_cast<const uint16_t*>(x);
    a.w = static_cast<const uint16_t*>(weight);
    a.bias = static_cast<const uint16_t*>(bias);
    a.m = (int)rows;
    a.n = (int)out_features;
    a.k = (int)in_features;
    a.n_tiles = (int)((out_features + kTileRows - 1) / kTileRows);
    const dim3 grid((unsigned)linear_tiles(rows, out_features));
    hipStream_t st = static_cast<hipStream_t>(stream);
    launch_prepare();
    if (dtype == NHP_BF16) linear_tiles_kernel<NHP_BF16><<<grid, dim3(256), 0, st>>>(a);
    else if (dtype == NHP_F16) linear_tiles_kernel<NHP_F16><<<grid, dim3(256), 0, st>>>(a);
    else return NHP_ERR_DTYPE;
    return launch_result();
}

}  // extern "C"
