// Causal grouped-query attention over f16 KV caches for gfx950 (cpu::attention, cpu_ops.cpp:544-575;
// the GPU kernel Attention, attention.comp, dispatched by qwen3_model.cpp:317 and gpt2_model.cpp:255):
// for token t at position pos0 + t and query head h, out = sum_j softmax_j(scale * q_h . k_j) v_j over
// cache rows j <= pos0 + t, k_j / v_j being kv head h / (n_head / n_kv) of those rows.
//
// Calls with heads of 64 or 128 take the matrix cores (attention_mfma.hip) where that is estimated to be faster;
// what follows is the vector path for the rest, whose work items attention_item.h computes.
//
// A workgroup of four waves per work item (token, kv head, block of up to four of the query heads that
// share it, split of the keys), the item's steps of keys dealt round robin to its waves. Lane = (key
// residue, 16-byte chunk of the head): each load instruction reads whole K or V head rows (16 lanes per
// 256-byte row of a 128-dimension head), and each lane keeps its chunk of the item's q rows in
// registers. A step issues all of its K and V loads first; the scores are the lanes' 8-dimension
// partial dots summed over a row's lanes by DPP; the softmax is the streaming form (running maximum;
// the sum and the accumulators rescaled when it grows), lane = key, its weights passed through LDS;
// then each lane adds its keys' weighted v chunks. The heads of a block share every K and V load. At
// the end each wave sums its accumulators over the key residues and the waves merge through LDS.
// When tokens x kv heads x head blocks give too few waves to fill the chip (decode: one token), each
// token's keys split over several items that write (maximum, sum, accumulators) to the context's
// workspace, and attn_merge_kernel combines them. The reference's CPU loop and its shader already sum
// in different orders; any order here is one more within the same bound.
#include <algorithm>
#include <cmath>

#include "attention_item.h"

namespace neko_hip {
namespace {

constexpr int kAttnHeads = 4;              // query heads per work item, at most (HB = 4 or 1)
constexpr int kAttnWaves = 4;              // waves per work item (its steps interleaved)
constexpr int kAttnWideWaves = 8;                // the same where one workgroup then takes a head's whole row
constexpr int64_t kAttnTargetWaves = 4096;  // keys split until a launch holds about this many waves
constexpr int64_t kAttnOneHeadBytes = int64_t{32} << 20;  // K + V bytes up to which items take one head

template <typename TQ, int HDP, bool AL, int NW, int HB, bool PF>
__global__ __launch_bounds__(64 * NW) void attn_kernel(AttnArgs a) {
    __shared__ AttnItemLds<HDP, NW, HB> lds;
    // Item index -> (token, kv head, head block, split), in 32 bits (the host keeps items below 2^31;
    // 64-bit division is a loop on this target). The latest tokens (the most keys) first.
    const uint32_t per_t = static_cast<uint32_t>(a.n_kv) * static_cast<uint32_t>(a.hblocks) * static_cast<uint32_t>(a.splits);
    const uint32_t item = blockIdx.x;
    const uint32_t tr = item / per_t;
    const int64_t t = a.T - 1 - tr;
    uint32_t rest = item - tr * per_t;
    const int split = static_cast<int>(rest % static_cast<uint32_t>(a.splits));
    rest /= static_cast<uint32_t>(a.splits);
    const int hb = static_cast<int>(rest % static_cast<uint32_t>(a.hblocks));
    const int g = static_cast<int>(rest / static_cast<uint32_t>(a.hblocks));
    const int h0 = g * a.group + hb * HB;
    const int nh = min(HB, a.group - hb * HB);
    const int64_t L = a.pos0 + t + 1;
    const int64_t k0 = static_cast<int64_t>(split) * a.split_keys;
    const int64_t k1 = min(L, k0 + a.split_keys);
    attend_item<TQ, HDP, AL, NW, HB, PF, false>(a, lds, t, g, h0, nh, split, k0, k1);
}

// Merges the key splits of one (token, head) per workgroup of 256 threads: M = the largest split
// maximum, each split weighted by exp(max - M); the sums and the accumulators added over the splits
// (threads over splits and dimensions, then the waves and groups in a fixed order); out = acc / sum.
template <typename TQ, bool LOG2>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnArgs a) {
    constexpr int kPer = kAttnMaxSplits / 256;  // splits per thread, at most
    __shared__ float wsh[kAttnMaxSplits];
    __shared__ float red[2][4];
    __shared__ float osh[8][256];
    const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6;
    const int64_t th = blockIdx.x;
    const uint32_t tq = blockIdx.x / static_cast<uint32_t>(a.n_head);  // 32-bit: T * n_head < 2^31
    const int64_t t = tq;
    const int h = static_cast<int>(blockIdx.x - tq * static_cast<uint32_t>(a.n_head));
    const int hd = a.hd, S = a.splits;
    float ms[kPer], ls[kPer];
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int s = tid + 256 * k;
        const float* pm = part_ml(a, th, min(s, S - 1));
        ms[k] = s < S ? pm[0] : -INFINITY;
        ls[k] = s < S ? pm[1] : 0.0f;
        mx = fmaxf(mx, ms[k]);
    }
    mx = wave_max_f32(mx);
    if ((tid & 63) == 0) red[0][wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));  // above -inf: split 0 holds key 0
    if (LOG2 && fabsf(mx) > kAttnScore) {
        // The largest is a score, and scores are taken from it as such. (Where an exponent is the largest, any
        // scores lie so far below that their weights are 0, in whichever unit.)
#pragma unroll
        for (int k = 0; k < kPer; k++)
            ms[k] = fabsf(ms[k]) > kAttnScore ? 0.5f * kLog2e * (ms[k] - mx) : ms[k] - 0.5f * kLog2e * mx;
        mx = 0.0f;
    }
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int s = tid + 256 * k;
        // An empty split or none: exp(-inf) = 0. (A NaN row ends here: -inf - -inf.)
        const float ws = LOG2 ? __builtin_amdgcn_exp2f(__builtin_fmaf(2.0f, ms[k], -2.0f * mx)) : expf(ms[k] - mx);
        if (s < S) wsh[s] = ws;
        sum = __builtin_fmaf(ws, ls[k], sum);
    }
    sum = wave_sum_f32(sum);
    if ((tid & 63) == 0) red[1][wave] = sum;
    __syncthreads();
    const float inv = 1.0f / ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
    // Accumulators: thread (group q, dimension d); group q takes splits q, q + G, ... (G = 256 / the
    // head size rounded up to a power of two), the groups added in order at the end.
    const int G = hd <= 32 ? 8 : hd <= 64 ? 4 : hd <= 128 ? 2 : 1;
    const int per = 256 / G;
    const int q = tid / per, d = tid - q * per;
    float o = 0.0f;
    if (d < hd) {
        int s = q;
        for (; s + 7 * G < S; s += 8 * G) {  // eight splits' loads in flight
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; k++) x[k] = part_acc(a, th, s + k * G)[d];
#pragma unroll
            for (int k = 0; k < 8; k++) o = __builtin_fmaf(wsh[s + k * G], x[k], o);
        }
        for (; s < S; s += G) o = __builtin_fmaf(wsh[s], part_acc(a, th, s)[d], o);
    }
    osh[q][d] = o;
    __syncthreads();
    if (q == 0 && d < hd) {
        for (int k = 1; k < G; k++) o += osh[k][d];
        TQ* orow = static_cast<TQ*>(a.out) + t * a.os + static_cast<int64_t>(h) * hd;
        orow[d] = from_f32<TQ>(o * inv);
    }
}

template <typename TQ, int HDP, int HB>
void launch_hb(neko_hip_ctx* ctx, const AttnArgs& a, dim3 grid, bool vec, bool pf) {
    const dim3 block(64 * kAttnWaves);
    if (!vec) hipLaunchKernelGGL((attn_kernel<TQ, HDP, false, kAttnWaves, HB, false>), grid, block, 0, ctx->stream, a);
    else if (pf) hipLaunchKernelGGL((attn_kernel<TQ, HDP, true, kAttnWaves, HB, true>), grid, block, 0, ctx->stream, a);
    else hipLaunchKernelGGL((attn_kernel<TQ, HDP, true, kAttnWaves, HB, false>), grid, block, 0, ctx->stream, a);
}

template <typename TQ, int HDP>
int launch_hdp(neko_hip_ctx* ctx, const char* what, const AttnArgs& a, bool vec, int64_t items, bool one_head, bool wide) {
    const dim3 grid(static_cast<uint32_t>(items));
    if constexpr (HDP <= 128) {  // (wider heads spill in the 128 registers of such a workgroup's lanes)
        if (wide) {
            hipLaunchKernelGGL((attn_kernel<TQ, HDP, true, kAttnWideWaves, 1, false>), grid, dim3(64 * kAttnWideWaves), 0,
                               ctx->stream, a);
            return after_launch(ctx, what);
        }
    }
    // The prefetching form where a wave has more than one step (measured: 4096-position decode, one
    // step per wave, 12.7 us without and 15.5 with it; 32768 positions 56.3 -> 49.6 us, the 2048- and
    // 8192-token prefills 6% faster).
    const int step = 8 * (512 / HDP);
    const bool pf = a.split_keys > static_cast<int64_t>(kAttnWaves) * step;
    if (one_head) launch_hb<TQ, HDP, 1>(ctx, a, grid, vec, pf);
    else launch_hb<TQ, HDP, kAttnHeads>(ctx, a, grid, vec, pf);
    if (int rc = after_launch(ctx, what)) return rc;
    return a.splits == 1 ? NEKO_OK : attn_merge(ctx, what, a, sizeof(TQ) == 2 ? NEKO_DT_F16 : NEKO_DT_F32, false);
}

template <typename TQ>
int launch_typed(neko_hip_ctx* ctx, const char* what, const AttnArgs& a, bool vec, int64_t items, bool one_head, bool wide) {
    if (a.hd <= 64) return launch_hdp<TQ, 64>(ctx, what, a, vec, items, one_head, wide);
    if (a.hd <= 128) return launch_hdp<TQ, 128>(ctx, what, a, vec, items, one_head, wide);
    return launch_hdp<TQ, 256>(ctx, what, a, vec, items, one_head, wide);
}

// Estimated time of a call on the vector path: rounds of the workgroups that fit, each with a start and its
// waves' steps (of the average row; an item of one query head hides its first in the start), or the reads of
// K and V by every token and head block, and the merge.
double vector_us(const neko_hip_ctx* ctx, const AttnArgs& a, bool one_head, bool wide, int64_t items, int64_t steps,
                 double kv_us) {
    const int64_t waves = wide ? kAttnWideWaves : kAttnWaves;
    const int64_t per = ((steps + a.splits - 1) / a.splits + waves - 1) / waves;
    const int fit = wide ? 2 : one_head ? 4 : per > 1 ? 2 : 3;  // workgroups per CU, by registers
    const double rounds = std::max(1.0, static_cast<double>(items) / (static_cast<double>(ctx->cu_count) * fit));
    const double rows = static_cast<double>(a.pos0) + 0.5 * static_cast<double>(a.T);
    const double seen = rows / static_cast<double>(a.pos0 + a.T);
    const double step = one_head ? 6.0 * static_cast<double>(per - 1)
                                 : 1.6 * static_cast<double>(per) * std::min(a.group, kAttnHeads);
    return 1.0 + std::max(rounds * (5.0 + seen * step), static_cast<double>(a.T * a.hblocks) * seen * kv_us) +
           (a.splits > 1 ? 2.5 + 0.004 * static_cast<double>(a.T * a.n_head) * a.splits : 0.0);
}

}  // namespace

int attn_merge(neko_hip_ctx* ctx, const char* what, const AttnArgs& a, int dtype, bool log2) {
    const dim3 grid(static_cast<uint32_t>(a.T * a.n_head)), block(256);
    if (dtype == NEKO_DT_F16) {
        if (log2) hipLaunchKernelGGL((attn_merge_kernel<half_t, true>), grid, block, 0, ctx->stream, a);
        else hipLaunchKernelGGL((attn_merge_kernel<half_t, false>), grid, block, 0, ctx->stream, a);
    } else {
        if (log2) hipLaunchKernelGGL((attn_merge_kernel<float, true>), grid, block, 0, ctx->stream, a);
        else hipLaunchKernelGGL((attn_merge_kernel<float, false>), grid, block, 0, ctx->stream, a);
    }
    return after_launch(ctx, what);
}

}  // namespace neko_hip

using namespace neko_hip;

extern "C" int neko_hip_attention(neko_hip_ctx* ctx, const void* q, int64_t q_stride, const uint16_t* k_cache,
                                  const uint16_t* v_cache, void* out, int64_t out_stride, int64_t T, int n_head, int n_kv,
                                  int hd, int64_t pos0, float scale, int dtype) {
    const char* what = "neko_hip_attention";
    NEKO_ENTER(ctx);
    NEKO_REQUIRE(ctx, valid_dtype(dtype), "%s: bad dtype %d", what, dtype);
    NEKO_REQUIRE(ctx, T >= 0 && pos0 >= 0 && n_head > 0 && n_kv > 0 && n_head % n_kv == 0,
                 "%s: bad shape T=%lld pos0=%lld n_head=%d n_kv=%d (n_head a multiple of n_kv)", what, (long long)T,
                 (long long)pos0, n_head, n_kv);
    NEKO_REQUIRE(ctx, hd >= 2 && hd <= 256 && hd % 2 == 0, "%s: head size %d (even, 2..256)", what, hd);
    if (T == 0) return NEKO_OK;
    NEKO_REQUIRE(ctx, q && k_cache && v_cache && out, "%s: null pointer", what);
    const int64_t width = static_cast<int64_t>(n_head) * hd;
    NEKO_REQUIRE(ctx, q_stride >= width && out_stride >= width, "%s: q / out row strides (%lld, %lld) below n_head*hd = %lld",
                 what, (long long)q_stride, (long long)out_stride, (long long)width);
    NEKO_REQUIRE(ctx, pos0 <= (int64_t(1) << 40) && T <= (int64_t(1) << 31), "%s: T=%lld / pos0=%lld too large", what,
                 (long long)T, (long long)pos0);
    const size_t esz = dtype_size(dtype);
    const int64_t kvw = static_cast<int64_t>(n_kv) * hd;
    NEKO_REQUIRE(ctx, pos0 + T <= (int64_t(1) << 62) / (kvw * 2), "%s: caches of %lld rows x %lld halves span more "
                 "than 2^62 bytes", what, (long long)(pos0 + T), (long long)kvw);
    const size_t sq = rows_span(T, width, q_stride, esz), so = rows_span(T, width, out_stride, esz);
    const size_t sc = static_cast<size_t>((pos0 + T) * kvw) * 2;
    NEKO_REQUIRE(ctx, sq != 0 && so != 0, "%s: q / out rows span more than 2^62 bytes", what);
    NEKO_REQUIRE(ctx, !overlaps(out, so, q, sq) && !overlaps(out, so, k_cache, sc) && !overlaps(out, so, v_cache, sc),
                 "%s: out may not overlap q or the caches", what);
    AttnArgs a{};
    a.q = q;
    a.qs = q_stride;
    a.kc = k_cache;
    a.vc = v_cache;
    a.kvw = kvw;
    a.out = out;
    a.os = out_stride;
    a.T = T;
    a.pos0 = pos0;
    a.n_head = n_head;
    a.n_kv = n_kv;
    a.group = n_head / n_kv;
    a.hd = hd;
    a.scale = scale;
    NEKO_REQUIRE(ctx, T * n_head <= 0x7fffffff, "%s: grid too large", what);
    // One query head per item where the K and V rows are few (their re-reads by the group's heads stay
    // in L2) and the launch would otherwise be short of waves; else up to four heads share each load.
    const int64_t kv_bytes = (pos0 + T) * static_cast<int64_t>(n_kv) * hd * 4;
    const bool one_head = T * n_kv * ((a.group + kAttnHeads - 1) / kAttnHeads) * kAttnWaves < kAttnTargetWaves &&
                          kv_bytes <= kAttnOneHeadBytes;
    const int hb_size = one_head ? 1 : kAttnHeads;
    a.hblocks = (a.group + hb_size - 1) / hb_size;
    // Split the keys when tokens x kv heads x head blocks leave the chip short of waves (each split at
    // least one 64-key step per wave).
    const int64_t base = T * n_kv * a.hblocks;
    const int64_t keys = pos0 + T;  // the longest row
    const int64_t step = 8 * (512 / (hd <= 64 ? 64 : hd <= 128 ? 128 : 256));  // the kernel's keys per step
    const int64_t steps = (keys + step - 1) / step;
    int64_t splits = 1;
    if (base * kAttnWaves < kAttnTargetWaves) {
        const int64_t want = (kAttnTargetWaves + base * kAttnWaves - 1) / (base * kAttnWaves);
        splits = std::min<int64_t>({want, (steps + kAttnWaves - 1) / kAttnWaves, kAttnMaxSplits});
    }
    const bool vec = hd % 8 == 0 && aligned(k_cache, 16) && aligned(v_cache, 16);
    // Eight waves on a head's whole row instead of splits and their merge, while each wave has one step and
    // the launch's workgroups fit at once (two per CU): one token over 201 keys, 32 / 8 heads of 128, f16,
    // 8.3 us split and 6.2 whole, over 501 keys, 12 heads of 64, 8.5 and 5.8. At two steps there is
    // nothing left of that (16 waves of one step or 8 of two over 501 keys of 128: 8.6 and 8.5).
    const bool wide = vec && hd <= 128 && one_head && splits > 1 && steps <= kAttnWideWaves && base <= 2 * ctx->cu_count;
    if (wide) splits = 1;
    a.split_keys = (steps + splits - 1) / splits * step;
    a.splits = static_cast<int>((keys + a.split_keys - 1) / a.split_keys);
    const int64_t items = base * a.splits;
    // The matrix cores where their estimated time is the shorter. Both estimates were fitted to the same calls,
    // each timed on both paths (1624 calls: 1 to 600 tokens, 16 shapes of heads, 4 thousand to 3 million pairs
    // of a query head and a key, f16 and f32; rms 9% there and 15% here; K and V past the caches are read at 5.2
    // TB/s). Over 400 calls of other sizes the choice costs 0.5% over the better path on average and is never more
    // than 15% behind the vector path. A line drawn at a number of pairs cost 3.1%, and was behind by up to
    // 2.1 times: 35 tokens over 155 keys, 6 / 2 heads of 128, f32, 6.3 us here and 13.3 there, while 57 tokens from
    // 0, 32 / 32 heads, f16, take 16.3 here and 7.0 there. Asked before either path wants a workspace.
    if (attn_mfma_can(a)) {
        const double kv_us = kv_bytes > kAttnOneHeadBytes ? static_cast<double>(kv_bytes) / 5.2e6 : 0.0;
        const AttnMfmaPlan plan = attn_mfma_plan(ctx, a, dtype, kv_us);
        if (plan.us < vector_us(ctx, a, one_head, wide, items, steps, kv_us)) return attn_mfma(ctx, what, a, dtype, plan);
    }
    NEKO_REQUIRE(ctx, items <= 0x7fffffff, "%s: grid too large", what);
    if (a.splits > 1) {
        void* ws = nullptr;
        const size_t bytes = static_cast<size_t>(T) * n_head * a.splits * (hd + 2) * sizeof(float);
        if (int rc = workspace(ctx, bytes, &ws)) return rc;
        a.part = static_cast<float*>(ws);
    }
    return dtype == NEKO_DT_F16 ? launch_typed<half_t>(ctx, what, a, vec, items, one_head, wide)
                                : launch_typed<float>(ctx, what, a, vec, items, one_head, wide);
}
