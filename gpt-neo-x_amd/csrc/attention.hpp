// Building blocks of the attention kernels (gfx950 matrix cores, LDS tiles of 64 rows).
//
// Orientation. All products are formed transposed, with the keys (or, in the kernel of the key and value
// gradients, the queries) as the rows of the 32 x 32 x 16 matrix instruction and the other sequence as its
// columns: a lane then holds 16 rows of ONE column, so a softmax row lives in two lanes (l and l + 32) and row
// statistics are per-lane scalars. The result of the first product is the B operand of the second without any
// exchange between lanes, provided the contraction runs over the rows in the order in which the lanes hold them:
// step ks takes rows 16 ks + 4 half + {0..3} and 16 ks + 8 + 4 half + {0..3}; the A operand (V^T, K^T, Q^T or
// dO^T) is read from LDS in that same order with the transposing 8-byte read.
//
// LDS tiles. 64 rows of 256 bytes (128 for a head size of 64), filled by loads that go from memory to LDS
// directly. Such a load writes 16 bytes per lane to consecutive addresses, so rows cannot be padded; the 16-byte
// chunks of a row are permuted instead (chunk c of row r sits in slot c ^ swizzle(r)) by letting each lane fetch
// the chunk that belongs in its slot. 16 rows read at one chunk (A operand) and 4 rows read at 4 chunks
// (transposing read) then both spread over all banks.
#pragma once

#include "common.hpp"

namespace nhp {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kFwdRows = 128;        // queries per workgroup of the forward kernel: 4 waves of 32
constexpr int kMaxMaskTiles = 1024;  // 64-key tiles of a bit mask: 65536 keys
constexpr float kFarBelow = -3e38f;
constexpr float kLazy = 8.0f;

struct AttnFwdArgs {
    const uint16_t *q, *k, *v;
    uint16_t *o, *kept;   // the result, and a second copy with the same strides or null
    float* lse;   // [batch * heads, sq], base-2 logarithm of the row's sum of exponentials; may be null
    const uint64_t* bits;
    int64_t q_s, q_b, q_h, k_s, k_b, k_h, v_s, v_b, v_h, o_s, o_b, o_h;   // element strides
    float scale_log2, fill_log2;
    int bits_batches, batch, heads, group, sq, sk, shift, window;
};

struct AttnBwdArgs {
    const uint16_t *q, *k, *v, *o, *d_o;
    uint16_t *dq, *dk, *dv;
    float *dk_parts, *dv_parts;   // [batch * heads / fold][sk][head size], summed up by a second kernel; null without one
    const float* lse;
    float* delta;   // [batch * heads, sq]: sum over features of out * d_out, written by the first kernel for the second
    int64_t q_s, q_b, q_h, k_s, k_b, k_h, v_s, v_b, v_h, o_s, o_b, o_h, do_s, do_b, do_h;
    int64_t dq_s, dq_b, dq_h, dk_s, dk_b, dk_h, dv_s, dv_b, dv_h;
    float scale, scale_log2;
    int batch, heads, group, sq, sk, shift, window;
    int fold;   // query heads that a workgroup of the second kernel goes over; they share a key/value head
};

// Which block of which matrix ((batch entry, head), or several heads of one batch entry) a workgroup takes; one workgroup
// for each. Under a causal mask blocks differ in length by up to their number, and they are handed out longest first (the
// caller counts them that way), the longest of all matrices ahead of the next shorter ones: matrix by matrix the last ones
// started with their longest blocks while the rest of the chip had run dry, and two long ones could meet on a CU. A matrix
// stays on one XCD, whose L2 then holds its keys and values, where the matrices divide among the XCDs; dealt out to all of
// them otherwise (12 matrices left two XCDs idle). One pass each, us, matrix by matrix -> here, forward / backward:
//   [1024, 4, 12 heads, 64] 26.4 -> 21.5 / 67.1 -> 54.5, [2048, 8, 16, 128] 188 -> 159 / 599 -> 525,
//   [3000, 1, 32 on 8, 128] 111 -> 84 / 371 -> 293, [4096, 4, 16, 128] 324 -> 292 / 1016 -> 920,
//   [8192, 1, 12, 64] 211 -> 152 / 544 -> 404 (on one XCD each 170 / 500), [8192, 1, 32 on 8, 128] 547 -> 528 / 1799 -> 1739.
struct Place {
    int unit, block;
};
__device__ __forceinline__ Place place(int units)
{
    if (units % 8 == 0) {
        const int per_xcd = units / 8, idx = blockIdx.x >> 3;
        return {(int)(blockIdx.x & 7) * per_xcd + idx % per_xcd, idx / per_xcd};
    }
    return {(int)(blockIdx.x % units), (int)(blockIdx.x / units)};
}

template <int DT>
struct Frag;
template <>
struct Frag<NHP_BF16> {
    static __device__ __forceinline__ f32x16 mma(u32x4 x, u32x4 y, f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bitcast<bf16x8>(x), bitcast<bf16x8>(y), c, 0, 0, 0);
    }
    static __device__ __forceinline__ u32x4 pack8(const f32x16& f, int at)
    {
        u32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = Half2<NHP_BF16>::pack(f[at + 2 * i], f[at + 2 * i + 1]);
        return r;
    }
};
template <>
struct Frag<NHP_F16> {
    static __device__ __forceinline__ f32x16 mma(u32x4 x, u32x4 y, f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(bitcast<f16x8>(x), bitcast<f16x8>(y), c, 0, 0, 0);
    }
    static __device__ __forceinline__ u32x4 pack8(const f32x16& f, int at)
    {
        u32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = Half2<NHP_F16>::pack(f[at + 2 * i], f[at + 2 * i + 1]);
        return r;
    }
};

// The 16 x 16 x 32 instruction, for few rows.
template <int DT>
__device__ __forceinline__ f32x4 mma16(u32x4 x, u32x4 y, f32x4 c)
{
    if constexpr (DT == NHP_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<bf16x8>(x), bitcast<bf16x8>(y), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<f16x8>(x), bitcast<f16x8>(y), c, 0, 0, 0);
}

// Geometry of a tile of 64 rows of HD elements in LDS.
template <int HD>
struct AttnGeo {
    static constexpr int kChunks = HD / 8;                   // 16-byte chunks of a row in memory
    static constexpr int kSlots = HD == 64 ? 8 : 16;         // and in LDS
    static constexpr int kRowBytes = kSlots * 16;
    static constexpr int kTileBytes = 64 * kRowBytes;
    static constexpr int kSteps = HD / 16;                   // matrix instructions along the head size
    static constexpr int kDTiles = (HD + 31) / 32;           // 32-feature tiles of a result

    static __device__ __forceinline__ int swizzle(int row)
    {
        if constexpr (kSlots == 8) return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
        return ((row & 3) << 2) | ((row >> 2) & 3);
    }
    // A operand (rows ql and ql + 32, features 16 t + 8 half ..): byte address ^ (t << 5), + 32 rows
    static __device__ __forceinline__ int row_addr(int ql, int half) { return ql * kRowBytes + ((half ^ swizzle(ql)) << 4); }
    // transposing read of 4 rows x 16 features per 16 lanes: byte address ^ (32-feature tile << 6), for the second
    // group of four rows ^ 32 and 8 rows on
    static __device__ __forceinline__ int tr_addr(int lane)
    {
        const int half = lane >> 5, g = (lane >> 4) & 1, i = lane & 15;
        const int row = 4 * half + (i >> 2), chunk = 2 * g + ((i & 3) >> 1);
        return row * kRowBytes + ((chunk ^ swizzle(row)) << 4) + (i & 1) * 8;
    }
};

#define NHP_LDS(T) __attribute__((address_space(3))) T

__device__ __forceinline__ u32x4 lds_read16(const char* p) { return *reinterpret_cast<const u32x4*>(p); }

__device__ __forceinline__ u32x4 lds_read_tr(const char* p0, const char* p1)
{
    const u32x2 a = bitcast<u32x2>(__builtin_amdgcn_ds_read_tr16_b64_v4i16((NHP_LDS(s16x4)*)p0));
    const u32x2 b = bitcast<u32x2>(__builtin_amdgcn_ds_read_tr16_b64_v4i16((NHP_LDS(s16x4)*)p1));
    return u32x4{a[0], a[1], b[0], b[1]};
}

// Makes the compiler wait here for the load that produces `v`, instead of at its first use inside a loop, where the
// wait would also cover the direct loads to LDS that are under way.
__device__ __forceinline__ void arrive(u32x4& v) { asm volatile("" : "+v"(v)); }

// Waits for this wave's direct loads to LDS.
__device__ __forceinline__ void wait_lds_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_address(const char* p) { return (uint32_t)(uintptr_t)(NHP_LDS(const char)*)p; }

// Moves a tile of 64 rows from memory to LDS; 4 waves, 16 rows each. The per-lane offsets are kept in registers, or,
// with LEAN, formed for every tile (10 % slower where the registers are there: forward at 8192 positions and 128
// features 571 against 532 us).
template <int HD, bool LEAN = false>
struct TileLoader {
    using G = AttnGeo<HD>;
    static constexpr int kRowsPerLoad = 1024 / G::kRowBytes, kLoads = 16 / kRowsPerLoad;
    uint32_t stride;  // bytes
    int row, chunk;   // of this lane in the wave's first load
    uint32_t offset[LEAN ? 1 : kLoads];

    __device__ __forceinline__ TileLoader(int64_t row_stride, int lane, int wave)
    {
        stride = (uint32_t)row_stride * 2;
        row = wave * 16 + lane / G::kSlots;
        chunk = (lane & (G::kSlots - 1)) ^ G::swizzle(row);
        if constexpr (!LEAN) {
#pragma unroll
            for (int i = 0; i < kLoads; ++i) offset[i] = (uint32_t)(row + i * kRowsPerLoad) * stride + column(chunk, i);
        }
    }
    // byte offset in a row for load i: kRowsPerLoad rows on, the swizzle changes in its bits (row >> 2) & 3 only
    static __device__ __forceinline__ uint32_t column(int c, int i) { return min(c ^ (i * kRowsPerLoad / 4), G::kChunks - 1) * 16; }
    // `rows` of the tile exist (at least one); rows beyond repeat the last one
    __device__ __forceinline__ void load(const uint16_t* tile, char* dst, int rows) const
    {
        const char* p = reinterpret_cast<const char*>(tile);
        const uint32_t d = __builtin_amdgcn_readfirstlane(lds_address(dst) + (row & ~15) * G::kRowBytes);
        int r = row, c = chunk;
        if constexpr (LEAN) asm volatile("" : "+v"(r), "+v"(c));
        if (rows >= 64) {
            const uint32_t at = (uint32_t)r * stride;
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                if constexpr (LEAN) issue(p + (uint64_t)(i * kRowsPerLoad) * stride, at + column(c, i), d + i * 1024);
                else issue(p, offset[i], d + i * 1024);
            }
        } else {
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
                issue(p, (uint32_t)min(r + i * kRowsPerLoad, rows - 1) * stride + column(c, i), d + i * 1024);
        }
    }
    // Written out because the compiler, which cannot tell which tile of the LDS buffer such a load fills, would wait
    // for it before the next LDS read of any tile. Waited for with wait_lds_loads() ahead of the barrier that hands the
    // tile over. (A scalar write of m0 needs one wait state before its use here.)
    static __device__ __forceinline__ void issue(const char* tile, uint32_t offset, uint32_t dst)
    {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(offset), "s"(tile) : "memory", "m0");
    }
};

// 64 floats from memory to LDS, one per lane of a wave; entries beyond `count` repeat the last one.
__device__ __forceinline__ void load_floats(const float* src, const char* dst, int lane, int count)
{
    const uint32_t offset = min(lane, count - 1) * 4;
    const uint32_t d = __builtin_amdgcn_readfirstlane(lds_address(dst));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(d), "v"(offset), "s"(src) : "memory", "m0");
}

__device__ __forceinline__ float max_halves(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    return fmaxf(bitcast<float>((uint32_t)r[0]), bitcast<float>((uint32_t)r[1]));
}
__device__ __forceinline__ float sum_halves(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    return bitcast<float>((uint32_t)r[0]) + bitcast<float>((uint32_t)r[1]);
}

// Stores the feature-major accumulators of one row (lane pair l, l + 32), times `f`: lane half 0 of a pair ends up
// with features 16 j .. 16 j + 7, half 1 with the next eight. `second`: another row that gets the same, or null.
template <int DT, int HD>
__device__ __forceinline__ void store_transposed(uint16_t* row, uint16_t* second, const f32x16 (&o)[AttnGeo<HD>::kDTiles], float f, int half)
{
#pragma unroll
    for (int d = 0; d < AttnGeo<HD>::kDTiles; ++d)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (d * 32 + j * 16 >= HD) continue;
            const uint32_t x0 = Half2<DT>::pack(o[d][8 * j] * f, o[d][8 * j + 1] * f);
            const uint32_t x1 = Half2<DT>::pack(o[d][8 * j + 2] * f, o[d][8 * j + 3] * f);
            const uint32_t y0 = Half2<DT>::pack(o[d][8 * j + 4] * f, o[d][8 * j + 5] * f);
            const uint32_t y1 = Half2<DT>::pack(o[d][8 * j + 6] * f, o[d][8 * j + 7] * f);
            const auto r0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
            const auto r1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
            const u32x4 chunk = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
            *reinterpret_cast<u32x4*>(row + d * 32 + j * 16 + half * 8) = chunk;
            if (second) *reinterpret_cast<u32x4*>(second + d * 32 + j * 16 + half * 8) = chunk;
        }
}

// The same as floats.
template <int HD>
__device__ __forceinline__ void store_transposed(float* row, const f32x16 (&o)[AttnGeo<HD>::kDTiles], float f, int half)
{
#pragma unroll
    for (int d = 0; d < AttnGeo<HD>::kDTiles; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (d * 32 + g * 8 >= HD) continue;
            *reinterpret_cast<f32x4*>(row + d * 32 + g * 8 + half * 4) =
                f32x4{o[d][4 * g] * f, o[d][4 * g + 1] * f, o[d][4 * g + 2] * f, o[d][4 * g + 3] * f};
        }
}

// Pointer and element strides (sequence, batch, head) of an operand whose features are contiguous; 16-byte accesses
// and 32-bit byte offsets within a tile must be possible.
static inline int fill_operand(const uint16_t*& p, int64_t& s, int64_t& b, int64_t& h, const void* ptr, const int64_t* strides)
{
    if (!ptr_aligned16(ptr)) return NHP_ERR_SHAPE;
    for (int i = 0; i < 3; ++i)
        if (strides[i] < 0 || strides[i] % 8) return NHP_ERR_SHAPE;
    if (strides[0] >= (int64_t)1 << 24) return NHP_ERR_SHAPE;
    p = static_cast<const uint16_t*>(ptr);
    s = strides[0];
    b = strides[1];
    h = strides[2];
    return NHP_OK;
}

}  // namespace nhp
