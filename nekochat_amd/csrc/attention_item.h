// The vector attention of one work item -- a token, up to HB query heads of one kv head, a run of keys -- by
// a workgroup: attn_kernel's, and attn_mfma_kernel's for the rows that it does again.
#pragma once

#include <cfloat>

#include "attention.h"

namespace neko_hip {

__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Eight halves of a cache row at p -- dimensions d .. d + 7 of a head, those at or past hd read as 0 --
// packed two to a register. AL: hd % 8 == 0 and the cache 16-byte aligned, so one 16-byte load.
template <bool AL>
__device__ __forceinline__ void load8(const uint16_t* p, int d, int hd, uint32_t (&r)[4]) {
    if constexpr (AL) {
        const uint4v v = d < hd ? *reinterpret_cast<const uint4v*>(p + d) : uint4v{0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = v[e];
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t lo = d + 2 * e < hd ? p[d + 2 * e] : 0u;
            const uint32_t hi = d + 2 * e + 1 < hd ? p[d + 2 * e + 1] : 0u;
            r[e] = lo | (hi << 16);
        }
    }
}

__device__ __forceinline__ float half_at(const uint32_t (&r)[4], int e) {
    const half2v h = __builtin_bit_cast(half2v, r[e >> 1]);
    return static_cast<float>(h[e & 1]);
}

// Sum over aligned groups of DC lanes (DC = 8, 16 or 32), every lane of a group receiving the sum.
template <int DC>
__device__ __forceinline__ float group_sum_f32(float v) {
    v = v + dpp_f32<kDppQuadXor1>(v);
    v = v + dpp_f32<kDppQuadXor2>(v);
    v = v + dpp_f32<kDppRowHalfMirror>(v);
    if constexpr (DC >= 16) v = v + dpp_f32<kDppRowMirror>(v);
    if constexpr (DC >= 32) v = v + __shfl_xor(v, 16);
    return v;
}

// Lane layout: lane = (key residue r, chunk c) -- 16-byte chunk c (dimensions 8c .. 8c + 7) of key
// rows j0 + KR u + r, u = 0 .. KU - 1 -- so each load instruction reads KR whole head rows of K or V
// (16 lanes per 256-byte row of a 128-dimension head) and each lane keeps its chunk of the q rows in
// registers. HDP: the head size rounded up to 64, 128 or 256 (DC = HDP / 8 chunks); a step is KR x 8
// keys (64 / 32 / 16): eight K and eight V loads per lane, issued before the previous step's
// arithmetic. NW waves share one work item, its steps dealt round robin; their states merge through LDS at
// the end.
template <int HDP, int NW, int HB>
struct AttnItemLds {
    static constexpr int STEP = 8 * (512 / HDP);
    float ssh[NW][HB][STEP];  // the step's scores by key, then its weights by (r, u)
    float msh[NW][HB], lsh[NW][HB];
    __align__(16) float ash[NW][HB][HDP];
};

// Query heads h0 .. h0 + nh - 1 (nh <= HB, all of kv head g) of token t over keys [k0, k1): into out, or as the
// partial results of `split` where a.splits > 1 (LOG2: the matrix-core path's). Called by the
// whole workgroup; lds is free for other use after the next barrier.
template <typename TQ, int HDP, bool AL, int NW, int HB, bool PF, bool LOG2>
__device__ __forceinline__ void attend_item(const AttnArgs& a, AttnItemLds<HDP, NW, HB>& lds, int64_t t, int g, int h0, int nh,
                                            int split, int64_t k0, int64_t k1) {
    constexpr int DC = HDP / 8;
    constexpr int KR = 64 / DC;
    constexpr int KU = 8;
    constexpr int STEP = KR * KU;
    static_assert(STEP == AttnItemLds<HDP, NW, HB>::STEP, "one step");
    auto& ssh = lds.ssh;
    auto& msh = lds.msh;
    auto& lsh = lds.lsh;
    auto& ash = lds.ash;
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int c = lane % DC, r = lane / DC;
    const int hd = a.hd;

    // This lane's chunk of each q row, f32.
    const TQ* qrow = static_cast<const TQ*>(a.q) + t * a.qs + static_cast<int64_t>(h0) * hd;
    float qv[HB][8];
#pragma unroll
    for (int i = 0; i < HB; i++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int d = 8 * c + e;
            qv[i][e] = i < nh && d < hd ? to_f32(qrow[static_cast<int64_t>(i) * hd + d]) : 0.0f;
        }
    float m[HB], l[HB], acc[HB][8];
#pragma unroll
    for (int i = 0; i < HB; i++) {
        m[i] = -INFINITY;
        l[i] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) acc[i][e] = 0.0f;
    }
    const uint16_t* kbase = a.kc + static_cast<int64_t>(g) * hd;
    const uint16_t* vbase = a.vc + static_cast<int64_t>(g) * hd;
    float(*sw)[STEP] = ssh[wave];

    // The K and V rows of the step at j0 (rows j0 + KR u + r; past k1: row k1 - 1, not counted). Nothing
    // here uses the loaded registers, so the loads stay in flight.
    auto load_step = [&](int64_t j0, uint32_t(&kr)[KU][4], uint32_t(&vr)[KU][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < KU; u++) load8<AL>(kbase + min(j0 + KR * u + r, k1 - 1) * a.kvw, 8 * c, hd, kr[u]);
#pragma unroll
        for (int u = 0; u < KU; u++) load8<AL>(vbase + min(j0 + KR * u + r, k1 - 1) * a.kvw, 8 * c, hd, vr[u]);
    };
    auto step = [&](int64_t j0, const uint32_t(&kr)[KU][4], const uint32_t(&vr)[KU][4]) __attribute__((always_inline)) {
        // Scores: each lane's 8-dimension partial dot, summed over the DC lanes of its key row.
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const int key = KR * u + r;
            const bool valid = j0 + key < k1;
#pragma unroll
            for (int i = 0; i < HB; i++) {
                if (i >= nh) break;
                float p = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) p = __builtin_fmaf(qv[i][e], half_at(kr[u], e), p);
                p = group_sum_f32<DC>(p);
                sw[i][key] = valid ? p * a.scale : -INFINITY;  // the DC lanes of the key store the same bits
            }
        }
        wave_sync_lds();
        // Streaming softmax per head, lane = key; the weights go back to LDS by (r, u).
#pragma unroll
        for (int i = 0; i < HB; i++) {
            if (i >= nh) break;
            const float s = lane < STEP ? sw[i][lane] : -INFINITY;
            // Above -inf also where every score so far is -inf (or NaN): their weights are 0, not exp(-inf + inf).
            const float mn = fmaxf(fmaxf(m[i], wave_max_f32(s)), -FLT_MAX);
            const float corr = expf(m[i] - mn);             // 0 on the wave's first step (m = -inf)
            const float p = expf(s - mn);                   // 0 for keys past k1
            l[i] = l[i] * corr + wave_sum_f32(p);
#pragma unroll
            for (int e = 0; e < 8; e++) acc[i][e] *= corr;
            m[i] = mn;
            wave_sync_lds();  // every lane has read its score before the weights overwrite them
            if (lane < STEP) sw[i][(lane % KR) * KU + lane / KR] = p;
        }
        wave_sync_lds();
        // Weighted v rows: this lane's keys KR u + r, chunk c (a key past k1 adds nothing: its row is
        // another key's, and 0 x inf would be NaN).
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const bool valid = j0 + KR * u + r < k1;
            float vf[8];
#pragma unroll
            for (int e = 0; e < 8; e++) vf[e] = valid ? half_at(vr[u], e) : 0.0f;
#pragma unroll
            for (int i = 0; i < HB; i++) {
                if (i >= nh) break;
                const float w = sw[i][r * KU + u];
#pragma unroll
                for (int e = 0; e < 8; e++) acc[i][e] = __builtin_fmaf(w, vf[e], acc[i][e]);
            }
        }
        wave_sync_lds();  // the next step rewrites sw
    };
    // Steps j0, j0 + NW STEP, ...; with PF (waves of several steps) the next step's loads are issued
    // before each step's arithmetic, in two register sets that alternate (no copy of registers a load
    // is still filling; the last prefetch re-reads row k1 - 1). Without PF each step loads, then
    // computes, in half the registers.
    const int64_t stride = static_cast<int64_t>(NW) * STEP;
    int64_t j0 = k0 + static_cast<int64_t>(wave) * STEP;
    if constexpr (!PF) {
        for (; j0 < k1; j0 += stride) {
            uint32_t ka[KU][4], va[KU][4];
            load_step(j0, ka, va);
            step(j0, ka, va);
        }
    } else if (j0 < k1) {
        uint32_t ka[KU][4], va[KU][4], kb[KU][4], vb[KU][4];
        load_step(j0, ka, va);
        for (;;) {
            load_step(j0 + stride, kb, vb);
            step(j0, ka, va);
            j0 += stride;
            if (j0 >= k1) break;
            load_step(j0 + stride, ka, va);
            step(j0, kb, vb);
            j0 += stride;
            if (j0 >= k1) break;
        }
    }

    // The wave's accumulators: summed over its KR key residues (lanes DC apart), then through LDS the
    // waves merge -- wave i merging head i, in wave order.
#pragma unroll
    for (int i = 0; i < HB; i++) {
        if (i >= nh) break;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float v = acc[i][e];
#pragma unroll
            for (int x = DC; x < 64; x *= 2) v += __shfl_xor(v, x);
            acc[i][e] = v;
        }
        if (r == 0) {
#pragma unroll
            for (int e = 0; e < 8; e++) ash[wave][i][8 * c + e] = acc[i][e];
        }
        if (lane == 0) {
            msh[wave][i] = m[i];
            lsh[wave][i] = l[i];
        }
    }
    __syncthreads();
    constexpr int DPL = HDP / 64;
    const int d0 = lane * DPL;
    for (int i = wave; i < nh; i += NW) {
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; w++) mx = fmaxf(mx, msh[w][i]);
        float sum = 0.0f, o[DPL];
#pragma unroll
        for (int e = 0; e < DPL; e++) o[e] = 0.0f;
        if (mx != -INFINITY) {  // an empty split (k0 >= L) keeps max -inf, sum 0
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const float ww = expf(msh[w][i] - mx);  // a wave without steps: 0
                sum = __builtin_fmaf(ww, lsh[w][i], sum);
#pragma unroll
                for (int e = 0; e < DPL; e++) o[e] = __builtin_fmaf(ww, ash[w][i][d0 + e], o[e]);
            }
        }
        const int64_t th = t * a.n_head + h0 + i;
        if (a.splits == 1) {
            TQ* orow = static_cast<TQ*>(a.out) + t * a.os + static_cast<int64_t>(h0 + i) * hd;
            const float inv = 1.0f / sum;
#pragma unroll
            for (int e = 0; e < DPL; e++)
                if (d0 + e < hd) orow[d0 + e] = from_f32<TQ>(o[e] * inv);
        } else {
            float* pa = part_acc(a, th, split);
#pragma unroll
            for (int e = 0; e < DPL; e++)
                if (d0 + e < hd) pa[d0 + e] = o[e];
            if (lane == 0) {
                float* pm = part_ml(a, th, split);
                const float e2 = mx * kLog2e;
                pm[0] = !LOG2 || fabsf(e2) > kAttnFar ? mx : 0.5f * e2;
                pm[1] = sum;
            }
        }
    }
}

}  // namespace neko_hip
