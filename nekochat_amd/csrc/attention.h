// Shared by the attention translation units: the launch arguments, the partial results of a key split,
// and the wave reductions.
#pragma once

#include "internal.h"

namespace neko_hip {

constexpr int64_t kAttnMaxSplits = 1024;  // the merge kernel's LDS weights

struct AttnArgs {
    const void* q;
    int64_t qs;  // q row stride (elements)
    const uint16_t* kc;
    const uint16_t* vc;
    int64_t kvw;  // cache row width (halves) = n_kv * hd
    void* out;
    int64_t os;  // out row stride (elements)
    int64_t T;
    int64_t pos0;
    int n_head;
    int n_kv;
    int group;    // n_head / n_kv
    int hblocks;  // ceil(group / HB): the head blocks per kv head
    int hd;
    float scale;
    int splits;          // key splits per work item
    int64_t split_keys;  // keys per split, a multiple of the kernel's step
    float* part;         // splits > 1: [T][n_head][splits][hd + 2] = (max, sum, accumulators)
};

constexpr float kLog2e = 1.44269504088896341f;
// Base-2 exponents past which f32 no longer places a row's maximum well: within 2^20 its steps are 1/8.
constexpr float kAttnFar = 1 << 20;

// Partial results of a key split (splits > 1): the accumulators [T][n_head][splits][hd] at part, then
// (max, sum) pairs [T][n_head][splits][2] after them. The matrix-core path's maxima are base-2 exponents,
// halved; those past kAttnFar are kept as the scores themselves, which are then exact against each other.
// kAttnScore tells them apart: exponents within 2^20 (and the weights' 2^15) halve to 2^19 + 8 at most,
// scores past it are larger than 2^20 / log2(e) = 726817.
constexpr float kAttnScore = 600000.0f;
__device__ __forceinline__ float* part_acc(const AttnArgs& a, int64_t th, int split) {
    return a.part + (th * a.splits + split) * a.hd;
}
__device__ __forceinline__ float* part_ml(const AttnArgs& a, int64_t th, int split) {
    return a.part + a.T * a.n_head * a.splits * a.hd + (th * a.splits + split) * 2;
}

__device__ __forceinline__ float readlane_f32(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Maximum / sum over the wave, returned wave-uniform (16-lane DPP all-reduce, then the four row results
// combined in a fixed order). All 64 lanes active.
__device__ __forceinline__ float wave_max_f32(float v) {
    v = fmaxf(v, dpp_f32<kDppQuadXor1>(v));
    v = fmaxf(v, dpp_f32<kDppQuadXor2>(v));
    v = fmaxf(v, dpp_f32<kDppRowHalfMirror>(v));
    v = fmaxf(v, dpp_f32<kDppRowMirror>(v));
    return fmaxf(fmaxf(readlane_f32(v, 0), readlane_f32(v, 16)), fmaxf(readlane_f32(v, 32), readlane_f32(v, 48)));
}

__device__ __forceinline__ float wave_sum_f32(float v) {
    v = v + dpp_f32<kDppQuadXor1>(v);
    v = v + dpp_f32<kDppQuadXor2>(v);
    v = v + dpp_f32<kDppRowHalfMirror>(v);
    v = v + dpp_f32<kDppRowMirror>(v);
    return (readlane_f32(v, 0) + readlane_f32(v, 16)) + (readlane_f32(v, 32) + readlane_f32(v, 48));
}

// Combines the splits of a.part into a.out (log2: the maxima are base-2 exponents).
int attn_merge(neko_hip_ctx* ctx, const char* what, const AttnArgs& a, int dtype, bool log2);
// The matrix-core path (attention_mfma.hip): whether it can take a call, how it would, and its launches.
struct AttnMfmaPlan {
    int row_groups;     // of 32 rows, per workgroup
    int64_t row_tiles;  // of as many rows, per kv head
    int64_t splits;     // of the keys
    double us;          // estimated time, kv_us being that of reading K and V once (attention.hip: how measured)
};
bool attn_mfma_can(const AttnArgs& a);
AttnMfmaPlan attn_mfma_plan(const neko_hip_ctx* ctx, const AttnArgs& a, int dtype, double kv_us);
int attn_mfma(neko_hip_ctx* ctx, const char* what, AttnArgs& a, int dtype, const AttnMfmaPlan& plan);

}  // namespace neko_hip
