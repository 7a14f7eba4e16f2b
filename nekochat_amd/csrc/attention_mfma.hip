// Causal grouped-query attention on the matrix cores (heads of 64 or 128): the calls of attention.hip
// whose (token, query head) pairs per kv head fill MFMA columns.
//
// The query heads of a kv head share its K and V rows, so its (token, head) pairs are flattened into
// rows r = token * group + head, 32 to a wave: the columns of v_mfma_f32_32x32x16_f16. Per tile of
// keys a wave computes S^T = K Q^T (A = 32 keys from LDS, B = its q rows, held in registers for the
// whole call), so a lane's accumulators are the scores of ONE row and 16 of 32 keys: the softmax needs
// a single exchange between lanes l and l + 32. O^T = V^T P^T then takes the probabilities straight
// from those registers as its B operand -- a contraction index may be permuted freely, so the keys
// stand in the order in which the scores lie in the lanes -- and V^T from LDS by ds_read_b64_tr_b16,
// which gives lane i of 16 column i of four rows. K and V reach LDS by global_load_lds, double
// buffered, in chunk orders (k_slot, v_slot) that keep both kinds of read on distinct banks.
//
// Precision: f32 q rows are scaled by a power of two and split into two f16 (24 bits of every element within
// 2^-16 of the row's largest, 2^-39 of that below), K and V are f16 as stored, and products are exact and
// summed in f32. Probabilities are split likewise, times 2^15: 24 bits above 2^-16 of the row's largest and
// 2^-39 of it below, where f32 would keep 24 bits. The running maximum, an integer exponent in which rescaling
// and merging are exact, is raised whenever a tile passes it, so that the scale is the largest f16 holds, and
// the scale joins after the exponential, whose argument's rounding is thus that of a number near 0. Measured
// as the sum of 8192 weights 22 nats below one dominant key, f32: off by 17% with a scale of 2^6 and a maximum
// left alone by less than 8, by 1.4e-5 now; 8192 random keys 2.8e-7 (3.0e-7 then, 3.4e-7 with the scale in the
// argument, 3.6e-7 on the vector path).
// Rows whose result is not finite (an infinity or NaN among the inputs may have met a zero weight or
// the other plane of a split), or whose scores pass 2^20 in log2 (from 2^24 the rounded maximum and the fma's
// exact product part, by any power of two), are done again by the workgroup as the vector path's items
// (attend_item). Where that takes every row a call costs more than the vector path alone would (one infinite v,
// f16; 32 / 8 heads of 128: 8192 tokens 24.1 ms and 22.3, 2048 tokens 2.65 and 1.59, 1 over 32768 keys 70 us and
// 53; 12 heads of 64, 1024 tokens, 570 and 215): a workgroup does its 128 rows one after the other and waits for
// each step's loads. Loading ahead would take the registers of a second workgroup per CU from every call.
//
// What bounds it: the MFMAs -- the work counted twice in both products with f32 q, in one with f16 q -- with
// the softmax's ~12 VALU operations per score beside them from the second wave of each SIMD. Measured
// (32 / 8 heads of 128): 8192 tokens from 0, f32, 22.3 ms on the vector path and 1.03 ms here (530 of
// the products' own TFLOP/s, twice that of MFMAs); 509 tokens after 3001, 16 / 8 heads, f16, 768 us and
// 46.6; one token over 32768 keys, f32, 55 us and 38.2, over 4096, f16, 12.8 us and 11.2.
#include <algorithm>
#include <atomic>

#include "attention_item.h"

namespace neko_hip {
namespace {

constexpr int kOffset = 15;  // probabilities are split times 2^kOffset, the largest power that f16 holds
constexpr float kScale = 1 << kOffset;
constexpr int kRedoHeads = 4;     // query heads per item of the rows done again, at most
constexpr float kNoKey = -1e30f;  // the running maximum before the first key

typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));

// The slot of 16-byte chunk c of tile row `row` in LDS. K: the 16 rows that a ds_read_b128 pass reads
// at one chunk fall on distinct banks. V: the 4 rows x 4 chunks that half a transposing read covers do.
template <int HD>
__device__ __forceinline__ int k_slot(int row, int c) {
    return HD == 128 ? c ^ (row & 15) : c ^ ((row >> 1) & 7);
}
template <int HD>
__device__ __forceinline__ int v_slot(int row, int c) {
    return HD == 128 ? c ^ ((row & 3) << 2) : c ^ ((row & 2) << 1);
}

// (The device min of 64-bit integers compares them as doubles.)
__device__ __forceinline__ int64_t smaller(int64_t a, int64_t b) { return a < b ? a : b; }

__device__ __forceinline__ float half_swap_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    return fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(r[0])), __builtin_bit_cast(float, static_cast<uint32_t>(r[1])));
}
__device__ __forceinline__ float half_swap_sum(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    return __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) + __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

// Four row groups at most: RW row groups of 32 rows x KW waves that share a group, each taking 32 KB_ of
// the tile's keys.
template <int HD, int RW, int KW, int KB_>
struct MfmaTile {
    static constexpr int waves = RW * KW, rows = 32 * RW, keys = 32 * KB_ * KW;
    static constexpr int half_bytes = keys * HD * 2;  // a tile's K (or V) rows
    static constexpr int lds = 2 * 2 * half_bytes;    // two buffers of K and V
    static constexpr int chunks = HD / 8;             // 16-byte chunks per row
    static constexpr int rpi = 64 / chunks;           // rows one wave's load instruction fills
    static constexpr int loads = keys / rpi / waves;  // load instructions per wave, tile and operand
    // Workgroups per CU, by LDS (160 KB) and registers: f32 q of 128 dimensions with a row group's keys over
    // several waves takes more than half a SIMD's. The kernel is compiled for as many, and the plan counts them.
    template <typename TQ>
    static constexpr int resident = 2 * (lds + 2048) <= 160 * 1024 && !(sizeof(TQ) == 4 && HD == 128 && KW > 1) ? 2 : 1;
    static_assert(KW == 1 || waves * 64 * (HD / 2) * 4 <= lds, "merge scratch");
    static_assert(keys % (rpi * waves) == 0, "whole load instructions");
};

template <typename TQ, int HD, int RW, int KW, int KB_>
__global__ __launch_bounds__(64 * RW * KW, (MfmaTile<HD, RW, KW, KB_>::template resident<TQ>)) void attn_mfma_kernel(AttnArgs a, int row_tiles, int vec_io) {
    typedef MfmaTile<HD, RW, KW, KB_> C;
    constexpr bool kTwo = sizeof(TQ) == 4;  // q in two f16 planes
    constexpr int NS = HD / 16, ND = HD / 32;
    // Chains per score: two where registers (and the VALU operation per score and chain) are short.
    constexpr int NC = !kTwo ? 1 : KW > 1 ? 4 : 2;
    extern __shared__ __align__(16) uint8_t attn_lds[];
    __shared__ float msh[C::waves][32], lsh[C::waves][32];
    __shared__ uint32_t bad_sh[C::waves];
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int rw = wave / KW, kw = wave % KW;
    const int l32 = lane & 31, h = lane >> 5;

    // Workgroup -> (row tile, split, kv head): the kv head fastest, so that with eight of them each XCD
    // keeps one head's K and V in its L2; the last row tiles (the most keys) first.
    uint32_t item = blockIdx.x;
    const int g = static_cast<int>(item % static_cast<uint32_t>(a.n_kv));
    item /= static_cast<uint32_t>(a.n_kv);
    const int split = static_cast<int>(item % static_cast<uint32_t>(a.splits));
    const int tile = row_tiles - 1 - static_cast<int>(item / static_cast<uint32_t>(a.splits));
    const uint32_t group = static_cast<uint32_t>(a.group);
    const uint32_t n_rows = static_cast<uint32_t>(a.T) * group;  // below 2^31 (attn_mfma_can)
    const uint32_t row0 = static_cast<uint32_t>(tile) * C::rows;

    // The keys this workgroup sees, cut into a.splits runs of whole tiles.
    const int64_t wg_last_t = min(row0 + C::rows - 1, n_rows - 1) / group;
    const int64_t wg_keys = a.pos0 + wg_last_t + 1;
    const int64_t n_tiles = (wg_keys + C::keys - 1) / C::keys;
    const int64_t per = (n_tiles + a.splits - 1) / a.splits;
    const int64_t k0 = split * per * C::keys;
    const int64_t k1 = smaller(wg_keys, k0 + per * C::keys);

    // This lane's row, and this wave's earliest causal limit (rows past the end repeat the last).
    const uint32_t row = min(row0 + 32u * rw + l32, n_rows - 1);
    const int64_t t = row / group;
    const int head = g * a.group + static_cast<int>(row - static_cast<uint32_t>(t) * group);
    const int64_t limit = smaller(a.pos0 + t + 1, k1);
    const int64_t wave_limit = smaller(a.pos0 + min(row0 + 32u * rw, n_rows - 1) / group + 1, k1);

    // q: dimensions 16 s + 8 h .. + 7 of this row as the B operand of step s. The sign of the scale goes
    // into q (the running maximum wants a positive factor); f32 rows are brought to [2^14, 2^15) by a
    // power of two first, so that both planes keep their bits.
    half8 qh[NS], ql[kTwo ? NS : 1];
    float c;
    {
        const TQ* qr = static_cast<const TQ*>(a.q) + t * a.qs + static_cast<int64_t>(head) * HD;
        // Position 0 has one key, of weight 1 whatever its score: a zero score makes that exact.
        const float sign = a.scale == 0.0f || a.pos0 + t == 0 ? 0.0f : a.scale < 0.0f ? -1.0f : 1.0f;
        c = (a.scale == 0.0f ? 1.0f : fabsf(a.scale)) * kLog2e;
        float x[NS][8];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const TQ* p = qr + 16 * s + 8 * h;
            if (vec_io) {
                typedef typename Chunk16<TQ>::V V;
                constexpr int N = Chunk16<TQ>::N;
#pragma unroll
                for (int i = 0; i < 8; i += N) {
                    const V v = *reinterpret_cast<const V*>(p + i);
#pragma unroll
                    for (int e = 0; e < N; e++) x[s][i + e] = to_f32(v[e]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) x[s][e] = to_f32(p[e]);
            }
        }
        if constexpr (kTwo) {
            float mx = 0.0f;
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(x[s][e]));
            mx = half_swap_max(mx);
            // 2^(14 - exponent), as two factors of which each is a normal float.
            const int ex = mx > 0.0f && mx < INFINITY ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
            const int e1 = ex / 2, e2 = ex - e1;
            c = ldexpf(c, -ex);
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int e = 0; e < 8; e++) x[s][e] = ldexpf(ldexpf(x[s][e], e1), e2);
        }
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v = x[s][e] * sign;
                qh[s][e] = static_cast<half_t>(v);
                if constexpr (kTwo) ql[s][e] = static_cast<half_t>(v - to_f32(qh[s][e]));
            }
    }

    // Tile loads: instruction i of this wave fills rows (wave * loads + i) * rpi ..+ rpi, lane = (row,
    // slot); the lane reads the chunk that belongs in its slot. Row offsets in 32 bits past a uniform
    // base; rows past the caches' end repeat the last.
    const int64_t cache_rows = a.pos0 + a.T;
    const uint32_t row_bytes = static_cast<uint32_t>(a.kvw) * 2;  // below 2^21 (attn_mfma_can)
    const int lr = lane / C::chunks, ls = lane % C::chunks;
    const char* kbase = reinterpret_cast<const char*>(a.kc + static_cast<int64_t>(g) * HD);
    const char* vbase = reinterpret_cast<const char*>(a.vc + static_cast<int64_t>(g) * HD);
    auto issue = [&](int64_t j0, int buf) __attribute__((always_inline)) {
        uint8_t* kd = attn_lds + buf * 2 * C::half_bytes;
        uint8_t* vd = kd + C::half_bytes;
        const uint32_t last = cache_rows - j0 <= C::keys ? static_cast<uint32_t>(cache_rows - 1 - j0) : C::keys;
        const char* kt = kbase + j0 * row_bytes;
        const char* vt = vbase + j0 * row_bytes;
#pragma unroll
        for (int i = 0; i < C::loads; i++) {
            const int first = (wave * C::loads + i) * C::rpi;
            // Opaque in the f32, 128-wide prompt kernel, so that the lane's offsets are computed per tile: kept, their
            // registers spilled (seven reloads per tile; 8192 tokens 1077 us, 1022 without).
            int row = lr;
            if constexpr (kTwo && HD == 128 && KW == 1) asm volatile("" : "+v"(row));
            const uint32_t r = static_cast<uint32_t>(first + row);
            const uint32_t off = min(r, last) * row_bytes;
            // (address-space conversions: C casts, which reinterpret_cast does not allow)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(kt + (off + 16u * k_slot<HD>(r, ls))),
                (__attribute__((address_space(3))) void*)(kd + first * HD * 2), 16, 0, 0);
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(vt + (off + 16u * v_slot<HD>(r, ls))),
                (__attribute__((address_space(3))) void*)(vd + first * HD * 2), 16, 0, 0);
        }
    };

    float16v o[ND] = {};
    float m = kNoKey, l = 0.0f;
    const int nt = static_cast<int>(k1 > k0 ? (k1 - k0 + C::keys - 1) / C::keys : 0);
    if (nt > 0) issue(k0, 0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int tq = lane & 15, tk = tq >> 2;  // transposing reads: this lane's row of four, dims 4 (tq & 3)
    for (int it = 0; it < nt; it++) {
        const int buf = it & 1;
        const int64_t j0 = k0 + static_cast<int64_t>(it) * C::keys;
        if (it + 1 < nt) issue(j0 + C::keys, buf ^ 1);  // that buffer's last readers passed the barrier
        const uint8_t* kd = attn_lds + buf * 2 * C::half_bytes;
        const uint8_t* vd = kd + C::half_bytes;
        const int kr0 = 32 * KB_ * kw;  // this wave's first key of the tile

        // Scores: with f32 q, NC chains of MFMAs over as many parts of the dimensions (the last starts with
        // the small plane), so that a step rounds at the size of its part of the score only.
        float16v s[KB_][NC] = {};
#pragma unroll
        for (int b = 0; b < KB_; b++) {
            const int r = kr0 + 32 * b + l32;
            half8 A[NS];
#pragma unroll
            for (int d = 0; d < NS; d++) A[d] = *reinterpret_cast<const half8*>(kd + r * HD * 2 + 16 * k_slot<HD>(r, 2 * d + h));
            if constexpr (kTwo) {
#pragma unroll
                for (int d = 0; d < NS; d++) s[b][NC - 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[d], ql[d], s[b][NC - 1], 0, 0, 0);
            }
            constexpr int per = NS / NC;
#pragma unroll
            for (int i = 0; i < per; i++)
#pragma unroll
                for (int n = 0; n < NC; n++)
                    s[b][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[n * per + i], qh[n * per + i], s[b][n], 0, 0, 0);
        }
        if (j0 + kr0 + 32 * KB_ > wave_limit) {  // keys past some row's limit
            const int64_t ahead = limit - (j0 + kr0);
            const int left = ahead < 0 ? 0 : ahead > 1024 ? 1024 : static_cast<int>(ahead);
#pragma unroll
            for (int b = 0; b < KB_; b++)
                unrolled<16>([&](auto ec) {
                    constexpr int e = decltype(ec)::value;
                    if (32 * b + 8 * (e >> 2) + 4 * h + (e & 3) >= left) s[b][0][e] = -INFINITY;
                });
        }
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < KB_; b++)
            unrolled<16>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                float v = s[b][0][e];
#pragma unroll
                for (int n = 1; n < NC; n++) v += s[b][n][e];
                mx = fmaxf(mx, v);
            });
        const float top = half_swap_max(mx) * c;
        float corr = 1.0f;
        if (__any(top > m)) {
            const float mn = fmaxf(m, ceilf(top));
            corr = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
        }
        // p, its sum, and its two planes.
        half8 ph[KB_][2], pl[KB_][2];
        float sum = 0.0f;  // of the tile, from zero: the row sum takes one rounding per tile
#pragma unroll
        for (int b = 0; b < KB_; b++)
            unrolled<2>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                float p[8];
                unrolled<8>([&](auto ec) {
                    constexpr int e = decltype(ec)::value;
                    // The exponent, its parts joined by fmas towards the small value that it is for the
                    // keys that matter.
                    float y = -m;
#pragma unroll
                    for (int n = NC - 1; n >= 0; n--) y = __builtin_fmaf(s[b][n][8 * i + e], c, y);
                    p[e] = __builtin_amdgcn_exp2f(y);
                    float q = p[e] * kScale;
                    asm("" : "+v"(q));  // opaque: folded into the conversion it is slower (8192 tokens, f16, 2%)
                    const half_t hi = static_cast<half_t>(q);
                    ph[b][i][e] = hi;
                    pl[b][i][e] = static_cast<half_t>(__builtin_fmaf(p[e], kScale, -to_f32(hi)));
                });
                sum += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            });
        l = __builtin_fmaf(l, corr, sum);
        // Each 32 dimensions of the tile's product from zero, then one rounding into the accumulators
        // (error against 64 bits, 8192 tokens with f32 q: 3.0e-7; with the MFMAs chained through them and
        // through one sum per score 7.5e-7; the vector path 3.6e-7).
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const int ch = 4 * d + 2 * ((lane >> 4) & 1) + ((tq & 3) >> 1);
            half8 A[KB_][2];
#pragma unroll
            for (int b = 0; b < KB_; b++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int r = kr0 + 32 * b + 16 * i + 4 * h + tk;
                    const uint8_t* p0 = vd + r * HD * 2 + 16 * v_slot<HD>(r, ch) + 8 * (tq & 1);
                    const short4v a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v*)p0);
                    const short4v a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) short4v*)(p0 + 8 * HD * 2));
                    A[b][i] = __builtin_bit_cast(half8, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7));
                }
            float16v x = {};
#pragma unroll
            for (int b = 0; b < KB_; b++)
#pragma unroll
                for (int i = 0; i < 2; i++) x = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[b][i], pl[b][i], x, 0, 0, 0);
#pragma unroll
            for (int b = 0; b < KB_; b++)
#pragma unroll
                for (int i = 0; i < 2; i++) x = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[b][i], ph[b][i], x, 0, 0, 0);
            unrolled<16>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                o[d][e] = __builtin_fmaf(o[d][e], corr, x[e]);
            });
        }
        __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of the next tile have landed
        __syncthreads();                // and every wave's; this tile's reads are done
    }

    l = half_swap_sum(l) * kScale;  // in the accumulators' unit
    float chk = l * 0.0f;
#pragma unroll
    for (int d = 0; d < ND; d++)
        unrolled<16>([&](auto ec) { chk = __builtin_fmaf(o[d][decltype(ec)::value], 0.0f, chk); });
    // Done again: rows with a value that is not finite (chk is NaN), and rows whose scores here lie too far out
    // for the exponents (below kNoKey they leave every weight 0).
    const bool far = fabsf(m) > kAttnFar && limit > k0 + 32 * KB_ * kw;
    const uint64_t again = __ballot(chk != 0.0f || far);
    if (lane == 0) bad_sh[wave] = static_cast<uint32_t>(again | (again >> 32));
    // The KW waves of a row group: their states through LDS, merged in wave order; wave kw then finishes
    // the 32-dimension blocks kw, kw + KW, ...
    if constexpr (KW > 1) {
        float* os = reinterpret_cast<float*>(attn_lds);
#pragma unroll
        for (int d = 0; d < ND; d++)
            unrolled<16>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                os[((wave * ND + d) * 16 + e) * 64 + lane] = o[d][e];
            });
        if (h == 0) {
            msh[wave][l32] = m;
            lsh[wave][l32] = l;
        }
    }
    // This row group's rows to do again.
    uint32_t bad = static_cast<uint32_t>(again | (again >> 32));
    if constexpr (KW > 1) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < KW; k++) bad |= bad_sh[rw * KW + k];
        float* os = reinterpret_cast<float*>(attn_lds);
        float w[KW];
        m = kNoKey;
#pragma unroll
        for (int k = 0; k < KW; k++) m = fmaxf(m, msh[rw * KW + k][l32]);
        l = 0.0f;
#pragma unroll
        for (int k = 0; k < KW; k++) {
            w[k] = __builtin_amdgcn_exp2f(msh[rw * KW + k][l32] - m);
            l = __builtin_fmaf(w[k], lsh[rw * KW + k][l32], l);
        }
#pragma unroll
        for (int d = 0; d < ND; d++) {
            if (d % KW != kw) continue;
            unrolled<16>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                float v = 0.0f;
#pragma unroll
                for (int k = 0; k < KW; k++) v = __builtin_fmaf(w[k], os[(((rw * KW + k) * ND + d) * 16 + e) * 64 + lane], v);
                o[d][e] = v;
            });
        }
    }
    const bool live = row0 + 32u * rw + l32 < n_rows && !((bad >> l32) & 1);
    const float inv = a.splits == 1 ? 1.0f / l : 1.0f;
    const int64_t th = t * a.n_head + head;
#pragma unroll
    for (int d = 0; d < ND; d++) {
        if (KW > 1 && d % KW != kw) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {  // dimensions 32 d + 8 q + 4 h .. + 3
            const int dim = 32 * d + 8 * q + 4 * h;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = o[d][4 * q + e];
            if (!live) continue;
            if (a.splits > 1) {
                *reinterpret_cast<float4v*>(part_acc(a, th, split) + dim) = float4v{v[0], v[1], v[2], v[3]};
                continue;
            }
            TQ* op = static_cast<TQ*>(a.out) + t * a.os + static_cast<int64_t>(head) * HD + dim;
            typedef typename VecOf<TQ, 4>::V V4;
            V4 r;
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = from_f32<TQ>(v[e] * inv);
            if (vec_io) *reinterpret_cast<V4*>(op) = r;
            else
#pragma unroll
                for (int e = 0; e < 4; e++) op[e] = r[e];
        }
    }
    if (a.splits > 1 && live && h == 0 && kw == 0) {
        float* pm = part_ml(a, th, split);
        pm[0] = l == 0.0f ? -INFINITY : 0.5f * (m - kOffset);
        pm[1] = l;
    }
    if constexpr (KW == 1) __syncthreads();
    uint32_t any_bad = 0;  // the same for the whole workgroup
#pragma unroll
    for (int k = 0; k < C::waves; k++) any_bad |= bad_sh[k];
    if (any_bad) {
        typedef AttnItemLds<HD, C::waves, kRedoHeads> Lds;
        static_assert(sizeof(Lds) <= C::lds, "LDS for the rows done again");
        Lds& lds = *reinterpret_cast<Lds*>(attn_lds);
#pragma unroll 1
        for (int w = 0; w < RW; w++) {
            uint32_t rows = 0;
#pragma unroll
            for (int k = 0; k < KW; k++) rows |= bad_sh[w * KW + k];
#pragma unroll 1
            while (rows) {
                const int i = __builtin_ctz(rows);
                const uint32_t rr = row0 + 32u * w + i;
                if (rr >= n_rows) break;
                const int64_t rt = rr / group;
                const int rh = static_cast<int>(rr - static_cast<uint32_t>(rt) * group);
                // The heads of this token that follow in the group of rows, too.
                const uint32_t rest = ~(rows >> i);
                const int run = min(rest ? __builtin_ctz(rest) : 32, min(kRedoHeads, a.group - rh));
                rows &= ~(((1u << run) - 1) << i);
                __syncthreads();  // the LDS before it
                attend_item<TQ, HD, true, C::waves, kRedoHeads, false, true>(a, lds, rt, g, g * a.group + rh, run, split, k0,
                                                                           smaller(a.pos0 + rt + 1, k1));
            }
        }
    }
}

template <typename TQ, int HD, int RW, int KW, int KB_>
int launch(neko_hip_ctx* ctx, const AttnArgs& a, MfmaTile<HD, RW, KW, KB_>, int row_tiles, bool vec_io) {
    typedef MfmaTile<HD, RW, KW, KB_> C;
    auto* kernel = &attn_mfma_kernel<TQ, HD, RW, KW, KB_>;
    static std::atomic<uint64_t> allowed{0};
    if (int rc = allow_lds(ctx, reinterpret_cast<const void*>(kernel), C::lds, allowed)) return rc;
    const dim3 grid(static_cast<uint32_t>(row_tiles) * static_cast<uint32_t>(a.splits) * static_cast<uint32_t>(a.n_kv));
    hipLaunchKernelGGL((attn_mfma_kernel<TQ, HD, RW, KW, KB_>), grid, dim3(64 * C::waves), C::lds, ctx->stream, a, row_tiles,
                       vec_io ? 1 : 0);
    return NEKO_OK;
}

// The tiles of a call with rw row groups per workgroup: f(MfmaTile{}).
template <int HD, typename F>
auto with_tile(int rw, F f) {
    switch (rw) {
        case 1: return f(MfmaTile<HD, 1, 4, 1>{});
        case 2: return f(MfmaTile<HD, 2, 2, 1>{});
        default: return f(MfmaTile<HD, 4, 1, 2>{});
    }
}

template <typename TQ, int HD>
int launch_rows(neko_hip_ctx* ctx, const AttnArgs& a, int rw, int row_tiles, bool vec_io) {
    return with_tile<HD>(rw, [&](auto tile) { return launch<TQ>(ctx, a, tile, row_tiles, vec_io); });
}

int resident(int dtype, int hd, int rw) {
    auto of = [&](auto tile) {
        typedef decltype(tile) C;
        return dtype == NEKO_DT_F16 ? C::template resident<half_t> : C::template resident<float>;
    };
    return hd == 64 ? with_tile<64>(rw, of) : with_tile<128>(rw, of);
}

}  // namespace

bool attn_mfma_can(const AttnArgs& a) {
    // 32-bit row numbers and offsets within a tile; whole 16-byte chunks.
    return (a.hd == 64 || a.hd == 128) && aligned(a.kc, 16) && aligned(a.vc, 16) && a.kvw <= (1 << 20) &&
           a.T * a.group < (int64_t{1} << 31) - 256;
}

AttnMfmaPlan attn_mfma_plan(const neko_hip_ctx* ctx, const AttnArgs& a, int dtype, double kv_us) {
    AttnMfmaPlan p;
    const int64_t rows = a.T * a.group;
    p.row_groups = rows <= 32 ? 1 : rows <= 64 ? 2 : 4;
    p.row_tiles = (rows + 32 * p.row_groups - 1) / (32 * p.row_groups);
    const int64_t tile_keys = p.row_groups == 1 ? 128 : 64;
    const int64_t tiles = (a.pos0 + a.T + tile_keys - 1) / tile_keys;
    // Keys split until the launch holds the workgroups that fit at once (a second round would double the time:
    // 12 tokens over 4000 keys, 32 / 8 heads of 128, f32, 16.4 us at one per CU and 25.6 split for two), each
    // with at least two tiles (one where there is a single row group) -- but not for four or fewer 64-key tiles
    // (two of 128), which take no longer than the merge's launch, about 3.5 us.
    const int64_t fit = static_cast<int64_t>(ctx->cu_count) * resident(dtype, a.hd, p.row_groups);
    const int64_t wgs = p.row_tiles * a.n_kv;
    const int64_t most = tiles * tile_keys <= 256 ? 1 : p.row_groups == 4 ? tiles / 2 : tiles;
    p.splits = std::max<int64_t>(1, std::min<int64_t>({fit / wgs, most, kAttnMaxSplits}));
    // The start of a launch, a tile of 1, 2 or 4 row groups, by head size and type; rounds of workgroups; the merge.
    static constexpr double kStart[2][2] = {{3.3, 3.8}, {5.1, 6.4}};
    static constexpr double kTile[2][2][3] = {{{1.7, 1.0, 1.5}, {2.2, 1.5, 1.8}}, {{1.6, 1.4, 2.2}, {1.9, 2.0, 2.5}}};
    const int wide = a.hd == 128, two = dtype == NEKO_DT_F32;
    const double rounds = std::max(1.0, static_cast<double>(wgs * p.splits) / static_cast<double>(fit));
    const double tile_us = rounds * static_cast<double>((tiles + p.splits - 1) / p.splits) * kTile[wide][two][p.row_groups / 2];
    p.us = kStart[wide][two] + std::max(tile_us, kv_us) +
           (p.splits > 1 ? 3.3 + 0.0003 * static_cast<double>(a.T * a.n_head * p.splits) : 0.0);
    return p;
}

int attn_mfma(neko_hip_ctx* ctx, const char* what, AttnArgs& a, int dtype, const AttnMfmaPlan& plan) {
    int64_t splits = plan.splits;
    const int64_t split_bytes = a.T * a.n_head * (a.hd + 2) * static_cast<int64_t>(sizeof(float));
    // Under capture the workspace cannot grow: as many splits as it holds.
    if (splits > 1 && static_cast<size_t>(splits * split_bytes) > ctx->workspace_bytes[0]) {
        bool cap = false;
        if (int rc = capturing(ctx, ctx->stream, &cap)) return rc;
        if (cap) splits = std::max<int64_t>(1, std::min<int64_t>(splits, static_cast<int64_t>(ctx->workspace_bytes[0]) / split_bytes));
    }
    a.splits = static_cast<int>(splits);
    a.part = nullptr;
    if (splits > 1) {
        void* ws = nullptr;
        if (int rc = workspace(ctx, static_cast<size_t>(splits * split_bytes), &ws)) return rc;
        a.part = static_cast<float*>(ws);
    }
    NEKO_REQUIRE(ctx, plan.row_tiles * a.n_kv * splits <= 0x7fffffff, "%s: grid too large", what);
    const size_t esz = dtype_size(dtype);
    const bool vec_io = aligned(a.q, 16) && aligned(a.out, 16) && a.qs * esz % 16 == 0 && a.os * esz % 16 == 0;
    const int rw = plan.row_groups, rt = static_cast<int>(plan.row_tiles);
    int rc;
    if (dtype == NEKO_DT_F16) rc = a.hd == 64 ? launch_rows<half_t, 64>(ctx, a, rw, rt, vec_io) : launch_rows<half_t, 128>(ctx, a, rw, rt, vec_io);
    else rc = a.hd == 64 ? launch_rows<float, 64>(ctx, a, rw, rt, vec_io) : launch_rows<float, 128>(ctx, a, rw, rt, vec_io);
    if (rc) return rc;
    if ((rc = after_launch(ctx, what))) return rc;
    return a.splits == 1 ? NEKO_OK : attn_merge(ctx, what, a, dtype, true);
}

}  // namespace neko_hip
