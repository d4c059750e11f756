// Softmax over rows that the chunked kernels of softmax.hip cannot take as they are: lengths that are not a multiple of
// eight elements, and pointers that are not 16-byte aligned.
#pragma once

#include "common.hpp"

namespace nhp {

constexpr float kExpBias = 64.0f;
constexpr float kMaskFill = -10000.0f;  // scaled_masked_softmax.h:180-184 of the reference

// Number of real keys of matrix `mat` ([batch * heads] matrices, one length per batch entry).
__device__ __forceinline__ uint32_t key_limit(const int32_t* key_lengths, uint32_t mat, uint32_t heads)
{
    if (key_lengths == nullptr) return 0xffffffffu;
    const int32_t len = key_lengths[mat / heads];
    return len < 0 ? 0u : (uint32_t)len;
}

struct RaggedArgs {
    uint16_t* out;             // probabilities, or the gradient of the scores
    const uint16_t* in;        // scores, or the incoming gradient (`out` may be the same memory)
    const uint16_t* probs;     // backward only
    const uint8_t* mask;       // padding-mask forward only: [1 or b, sq, n]
    const float* slopes;       // [np] AliBi slopes or null
    const uint16_t* bias;      // [np, sq, n] or null
    const int32_t* key_lengths;  // [b] or null
    float scale;
    uint32_t n, sq, np, rows;  // rows = b * np * sq
    uint32_t window;           // causal: 0xffffffff = no lower bound
    int mask_per_batch;
    uint16_t* dropped;         // forward: second output dropout(out), or null
    DropoutKey drop;
};

// Whether the kernels below take rows of n elements (the others stay with the scalar kernels).
bool ragged_rows(int64_t n);

template <int DT>
int ragged_causal_fwd(const RaggedArgs& a, hipStream_t st);
template <int DT>
int ragged_masked_fwd(const RaggedArgs& a, hipStream_t st);
template <int DT, bool CAUSAL>
int ragged_bwd(const RaggedArgs& a, bool dropout, hipStream_t st);

}  // namespace nhp
