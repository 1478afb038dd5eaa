// Decode over narrow block tables (pools of 16 or 32 bits, or fp8 under 16-bit queries with heads of more than 32): a workgroup per (kv head, sequence), or several with a merge behind
// them (plan_short_splits of decode_plan.h: where, how many, and what they measured).
//
// Short sequences are bound by waits and by the instructions that a workgroup fetches once, not by bytes: the split pass, whose loop is unrolled
// for streams, spent 1.3 us on the table of units, 1.6 on finding its sequence, 2.6 to 3.2 on the keys and 2.5 to 4 on the merge for 17
// to 47 keys.  Here the length, the block table and the query rows are on their way at once, then all keys and values; the group's query heads (up
// to 16) are the columns of one matrix product, so that a lane holds four logits of one head and every step stays short:
//     S = K Q^T     keys as rows, 16 at a time; a lane's 16 bytes of a row are an operand as they come from memory
//     O^T += V^T P^T   S's layout is P's as an operand; V goes through the wave's own part of LDS, read transposed
// P is a sum of two 16-bit terms: with one, short sequences came out less exact than the split pass, whose every row of lanes has a weight of
// one (error against 64 bits, 14 / 2 heads of 64, 8 sequences of 94 .. 683 keys: split pass 1.78e-3, one term 2.06e-3, two 1.67e-3).
// Over fp8 pools a weight meets its block's scale, and the terms are of bf16 whatever the queries are: fp16 has no room for small scales (fp16
// queries, those sequences, terms of fp16 -> bf16: 2.071e-4 -> 2.069e-4, with values of 0.001 instead of one 1.0e-2 -> 2.4e-4).
// Over 32-bit pools both products are of 32-bit operands (16x16x4), a load's four elements one after the other, and nothing goes through LDS: with
// the rows 4 g + i of V as the i-th operand, S's layout is again P's, and a lane's 16 bytes of a row of V are operands of four tiles of columns.
// Each sum is a tree over sums of eight (logits) and of four terms (values): in one chain, as the accumulators offer it, errors against 64
// bits were 1.9 times the split pass's (14 / 2 heads of 64), in trees they are 0.95 of them (0.81 .. 1.04 over 16 kinds of batches).  What bounds it is the
// matrix unit's rate for these operands, 1024 cycles for 16 keys of 64 (0.9 us with 128), and the chain of waits: the queries of 256 wait in LDS, as registers
// for two waves a SIMD let a second workgroup's loads fly meanwhile; at 128 three waves spill.  us, the split pass -> this: 14 / 2 heads of 64, 5
// sequences of 38 keys 11.8 -> 5.8; 8 / 2 of 128, 19 of 61 11.2 -> 5.9; 14 / 2 of 256, 28 of 195 26.5 -> 13.
// Waves take tiles of 16 keys in turn, two at a time up to 64 elements a row; their sums meet in LDS with two barriers.  One tile at a time at
// 128 leaves registers for four workgroups a compute unit: 256 sequences of 16 keys, 32 / 8 heads, 16.1 -> 9.0 us.
#pragma once
#include "decode_impl.h"

namespace pa_decode_detail {

template <typename T> struct ShortMfma;
template <> struct ShortMfma<pa_bf16> {
    typedef __bf16 x8 __attribute__((ext_vector_type(8)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ f4 mul(pa_u4 a, pa_u4 b, f4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(x8, a), __builtin_bit_cast(x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float x, float y) {
        typedef __bf16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, v2{(__bf16)x, (__bf16)y});
    }
    static __device__ __forceinline__ float2 unpack(uint32_t w) {
        return make_float2(__builtin_bit_cast(float, w << 16), __builtin_bit_cast(float, w & 0xffff0000u));
    }
};
template <> struct ShortMfma<pa_f16> {
    typedef _Float16 x8 __attribute__((ext_vector_type(8)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ f4 mul(pa_u4 a, pa_u4 b, f4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(x8, a), __builtin_bit_cast(x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float x, float y) {
        typedef _Float16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, v2{(_Float16)x, (_Float16)y});
    }
    static __device__ __forceinline__ float2 unpack(uint32_t w) {
        typedef _Float16 v2 __attribute__((ext_vector_type(2)));
        const v2 h = __builtin_bit_cast(v2, w);
        return make_float2((float)h[0], (float)h[1]);
    }
};

template <> struct ShortMfma<float> {
    typedef float f4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ f4 mul(uint32_t a, uint32_t b, f4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b), c, 0, 0, 0);
    }
};

constexpr int kShortHeads = kPlanShortHeads, kShortKeys = kPlanShortTile;  // query heads of a workgroup, keys of a tile

// Four consecutive outputs (rows are multiples of 16 bytes long; the first need not lie on one of 8).
template <typename QT, typename Num> __device__ __forceinline__ void short_store(QT *to, const Num &num, float best, float den, int ez) {
    using M = ShortMfma<QT>;
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = finish_row(num[i], best, den, ez);
    if constexpr (sizeof(QT) == 2) {
        if (((uintptr_t)to & 7u) == 0) {
            *reinterpret_cast<uint2 *>(to) = make_uint2(M::pack(y[0], y[1]), M::pack(y[2], y[3]));
            return;
        }
    } else if (((uintptr_t)to & 15u) == 0) {
        *reinterpret_cast<float4 *>(to) = make_float4(y[0], y[1], y[2], y[3]);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) pa_scalar<QT>::store(to + i, y[i]);
}

// Blocks are whole tiles (block_size % 16 == 0).
// A workgroup has one of a.splits equal runs of its sequence's tiles and, with a.leave, leaves the maximum, sum and unnormalised outputs of its
// keys for the merge.
// Neighbouring workgroups have the heads and runs of one sequence, the sequences come one after the other (z): with the runs further apart, as many
// as there are sequences and heads, all runs of a long one came to few compute units, often after every other one had run.  us, one sequence of n keys among
// others of n / 20, runs furthest apart -> next to each other: 32-bit 14 / 2 heads of 64, 64 of 11200 74 -> 38; 40 / 8 of 128, 16 of 2800 34 -> 26; 16-bit
// 40 / 8 of 128, 16 of 5600 50 -> 24; fp8 14 / 2 of 256, 64 of 5600 0.65 of the time.  (Over 486 batches each of equal steps of length, drawn ones and such: 0.97, 0.95 and 0.93.)
template <typename KV, typename QT, int D> __global__ __launch_bounds__(kThreads, D == 256 || (sizeof(KV) == 4 && D == 128) ? 2 : sizeof(KV) == 4 ? 3 : 4) void decode_short_kernel(const DecodeArgs a) {
    using M = ShortMfma<QT>;
    constexpr bool kFp8 = sizeof(KV) == 1, k32 = sizeof(KV) == 4;
    using VT = std::conditional_t<kFp8, pa_bf16, QT>;  // the second product's type (fp8 values are exact in either)
    using W = ShortMfma<VT>;
    using f4 = typename M::f4;
    constexpr int EL = 16 / sizeof(KV), KL = D / (4 * EL), QL = EL == 16 ? 2 : 1;  // elements of a 16-byte load; loads of a tile of K, and of V; of a query for each
    constexpr int NT = D >= 128 ? 1 : 2;                    // tiles at a time (registers for four waves a SIMD, at 256 two; 32 bits: for three and two)
    constexpr int kPitch = D + 16;                          // (four rows of a transposing read lie 32 bytes apart modulo 64)
    constexpr int HR = D == 256 ? 8 : kShortHeads, kPitchO = D + 4;  // heads merged at a time
    constexpr int kBytesV = k32 ? 0 : kWaves * NT * kShortKeys * kPitch * 2, kBytesO = kWaves * HR * kPitchO * 4;
    __shared__ __align__(16) char room[kBytesV > kBytesO ? kBytesV : kBytesO];
    constexpr bool kLdsQ = k32 && D == 256;  // the queries are read from LDS: registers for two waves a SIMD
    __shared__ pa_u4 s_q[kLdsQ ? KL : 1][64];
    __shared__ float s_m[kWaves][kShortHeads], s_l[kWaves][kShortHeads];
    const PoolArgs &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int kvh = blockIdx.x, b = blockIdx.z, rep0 = (blockIdx.y / a.splits) * kShortHeads, nr = min(kShortHeads, p.n_rep - rep0);
    const int split = blockIdx.y % a.splits;
    const int32_t *bt_row = p.bt + (int64_t)b * p.bt_stride;
    const int tiles_per_block = p.bs / kShortKeys;
    auto table = [&](int first) {  // the block of tile first + lane (-1: there is none)
        const int blk = (first + lane) / tiles_per_block;
        const int bid = blk < p.bt_stride ? bt_row[blk] : -1;
        return bid < p.num_blocks ? bid : -1;
    };
    const bool known = p.window == 0 && a.splits == 1;  // the first tile, ahead of the length
    int bids = known ? table(0) : -1;
    const int L = a.seq_lens[b];
    QT *orow = reinterpret_cast<QT *>(a.out) + ((int64_t)b * p.hq + kvh * p.n_rep + rep0) * p.d;
    // queries: lane l16 has head rep0 + l16, the elements of its loads of K
    pa_u4 qr[kLdsQ ? KL / kWaves : KL][QL];
    {
        const QT *qp = reinterpret_cast<const QT *>(a.q) + ((int64_t)b * p.hq + kvh * p.n_rep + rep0 + (l16 < nr ? l16 : 0)) * p.d;
#pragma unroll
        for (int j = 0; j < (kLdsQ ? KL / kWaves : KL); ++j)
#pragma unroll
            for (int e = 0; e < QL; ++e) {
                const int d = EL * (4 * (kLdsQ ? wave * (KL / kWaves) + j : j) + g) + 8 * e;
                qr[j][e] = l16 < nr && d < p.d ? *reinterpret_cast<const pa_u4 *>(qp + d) : pa_u4{0, 0, 0, 0};
            }
    }
    if (L <= 0 && !a.leave) {  // uniform
        for (int i = tid; i < nr * p.d; i += kThreads) pa_scalar<QT>::store(orow + i, 0.f);
        return;
    }
    if constexpr (kLdsQ) {
#pragma unroll
        for (int j = 0; j < KL / kWaves; ++j) s_q[wave * (KL / kWaves) + j][lane] = qr[j][0];
        __syncthreads();
    } else if constexpr (k32) {
#pragma unroll
        for (int j = 0; j < KL; ++j) asm volatile("" : "+v"(qr[j][0]));  // (waits for them here: in the loop for K alone)
    }
    const int ez = a.extra_zero ? max(0, a.extra_zero[b]) : 0;
    const int k_lo = plan_first_key(L, p.window);
    int t0 = k_lo / kShortKeys, n_tiles = L > 0 ? (L - 1) / kShortKeys + 1 - t0 : 0;
    if (a.splits > 1) {
        const int from = (int)((int64_t)n_tiles * split / a.splits);
        n_tiles = (int)((int64_t)n_tiles * (split + 1) / a.splits) - from;
        t0 += from;
    }
    const int tok = p.hkv * p.d * (int)sizeof(KV), head = kvh * p.d * (int)sizeof(KV);  // bytes between tokens, before the head
    uint16_t *vs = reinterpret_cast<uint16_t *>(room) + wave * NT * kShortKeys * kPitch;

    float m, l;
    f4 acc[D / 16];  // O^T: d = 16 dt + 4 g + i (32 bits: 64 (dt / 4) + 16 g + 4 i + dt % 4), head l16
    pa_u4 kr[NT][KL], vr[NT][KL];
    float kscale = 1.f, vscale = 1.f;  // of tile `lane` of the 64 at hand
    // An infinite value times a weight's second term, which is zero or negative as often as not, makes a sum NaN that is infinite.  So a wave whose
    // sums are not all finite goes over its keys once more with the first terms alone, as the split pass has them: twice, and halved behind the loop.
    // (us: 8 sequences of 94 .. 683 keys, 32 / 8 heads of 128, 9.6 -> 9.9, 14 / 2 of 64 7.4 -> 7.4, of 256 11.6 -> 12.0)
    bool again = false;
#pragma unroll 1
    for (;; again = true) {
        m = kNegBig;
        l = 0.f;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) acc[dt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int first = 0; first < n_tiles; first += 64) {
            const int n = min(64, n_tiles - first), tile0 = t0 + first;
            if (first > 0 || !known || again) bids = table(tile0);
            if constexpr (kFp8) {
                const int64_t at = bids >= 0 ? (int64_t)bids * p.hkv + kvh : 0;
                kscale = bids >= 0 ? p.k_scale[at] : 1.f;
                vscale = bids >= 0 ? p.v_scale[at] : 1.f;
            }
            auto fetch = [&](int at, bool keys, bool values) {  // (constants)
                int at16 = l16, at4 = g;
                if constexpr (k32) asm volatile("" : "+v"(at16), "+v"(at4));  // (the offsets of 32 loads are not kept over the loop)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int tile = tile0 + at + t, bid = at + t < n ? __builtin_amdgcn_readlane(bids, at + t) : -1;
                    const int rows = bid >= 0 ? min(kShortKeys, L - tile * kShortKeys) : 0;  // (rows past them read as zeros)
                    const int skip = k_lo - tile * kShortKeys;                               // rows before the window: zeros of V
                    const int64_t slot = ((int64_t)max(bid, 0) * p.bs + tile % tiles_per_block * kShortKeys) * tok;
                    const int bytes = rows > 0 ? (rows - 1) * tok + head + p.d * (int)sizeof(KV) : 0;
                    const __amdgpu_buffer_rsrc_t k = __builtin_amdgcn_make_buffer_rsrc((void *)(reinterpret_cast<const char *>(p.k) + slot), 0, bytes, 0x00020000);
                    const __amdgpu_buffer_rsrc_t v = __builtin_amdgcn_make_buffer_rsrc((void *)(reinterpret_cast<const char *>(p.v) + slot), 0, bytes, 0x00020000);
#pragma unroll
                    for (int j = 0; j < (keys ? KL : 0); ++j) {
                        const int d = EL * (4 * j + at4);
                        kr[t][j] = __builtin_amdgcn_raw_buffer_load_b128(k, d < p.d ? at16 * tok + head + d * (int)sizeof(KV) : kDeadLaneOffset, 0, kStreamPolicy);
                    }
#pragma unroll
                    for (int j = 0; j < (values ? KL : 0); ++j) {
                        const int c = lane + 64 * j, row = k32 ? 4 * at4 + j / (D / 64) : c / (D / EL), d = k32 ? 64 * (j % (D / 64)) + 4 * at16 : c % (D / EL) * EL;
                        vr[t][j] = __builtin_amdgcn_raw_buffer_load_b128(v, d < p.d && row >= skip ? row * tok + head + d * (int)sizeof(KV) : kDeadLaneOffset, 0, kStreamPolicy);
                    }
                }
            };
            if (wave * NT < n) fetch(wave * NT, true, true);
#pragma unroll 1
            for (int at = wave * NT; at < n; at += kWaves * NT) {
                if constexpr (kLdsQ) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (else they are kept over the loop)
                float x[NT][4], mx = m;
                f4 raw[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    f4 s = f4{0.f, 0.f, 0.f, 0.f}, odd[6], last[2];
                    // Adds the j-th of the terms of a logit to the sums of two, of four ... of them: the whole sum behind the last one.
                    auto tree = [&](int j, f4 y) {
#pragma unroll
                        for (int level = 0; level < 6; ++level) {
                            asm volatile("" : "+v"(y));  // (now)
                            if (!(j >> level & 1)) {
                                odd[level] = y;
                                break;
                            }
                            y = odd[level] + y;
                        }
                        return y;
                    };
#pragma unroll
                    for (int j = 0; j < KL; ++j) {
                        if constexpr (kFp8) {
                            uint32_t w[8];
                            PoolWords<KV, QT>::unpack(kr[t][j], w);
                            s = M::mul(pa_u4{w[0], w[1], w[2], w[3]}, qr[j][0], s);
                            s = M::mul(pa_u4{w[4], w[5], w[6], w[7]}, qr[j][1], s);
                        } else if constexpr (k32) {
                            pa_u4 qj;
                            if constexpr (kLdsQ) qj = s_q[j][lane];
                            else qj = qr[j][0];
                            const f4 none = f4{0.f, 0.f, 0.f, 0.f};
                            const f4 u = M::mul(kr[t][j][1], qj[1], M::mul(kr[t][j][0], qj[0], none));
                            const f4 w = M::mul(kr[t][j][3], qj[3], M::mul(kr[t][j][2], qj[2], none));
                            if (j > 0) tree(j - 1, last[0] + last[1]);
                            last[0] = u;
                            last[1] = w;
                            if (j == KL - 1) s = tree(j, u + w);
                            __builtin_amdgcn_sched_barrier(0);  // (products in order need few registers)
                        } else {
                            s = M::mul(kr[t][j], qr[j][0], s);
                        }
                    }
                    const int lim = at + t < n ? L - (tile0 + at + t) * kShortKeys : 0, lo = k_lo - (tile0 + at + t) * kShortKeys;
                    raw[t] = s;
                    float f = p.scale_log2;
                    if constexpr (kFp8) f *= __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, kscale), (at + t) & 63));
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        x[t][i] = 4 * g + i < lim && 4 * g + i >= lo ? s[i] * f : -INFINITY;
                        mx = fmaxf(mx, x[t][i]);
                    }
                    // V, for the transposing reads
#pragma unroll
                    for (int j = 0; j < (k32 ? 0 : KL); ++j) {
                        const int c = lane + 64 * j, row = t * kShortKeys + c / (D / EL), d = c % (D / EL) * EL;
                        pa_u4 *to = reinterpret_cast<pa_u4 *>(vs + row * kPitch + d);
                        if constexpr (kFp8) {
                            uint32_t w[8];
                            PoolWords<KV, VT>::unpack(vr[t][j], w);
                            to[0] = pa_u4{w[0], w[1], w[2], w[3]};
                            to[1] = pa_u4{w[4], w[5], w[6], w[7]};
                        } else {
                            to[0] = vr[t][j];
                        }
                    }
                }
                // (32 bits: behind the last tiles too, of no bytes: where both are without a condition, K's products wait for K alone)
                if (k32 || at + kWaves * NT < n) fetch(at + kWaves * NT, true, !k32);
                {
                    const float2 y = lane_pair<16>(mx, 16);
                    mx = fmaxf(y.x, y.y);
                    const float2 z = lane_pair<32>(mx, 32);
                    mx = fmaxf(z.x, z.y);
                }
                const float alpha = __builtin_amdgcn_exp2f(m - mx);
                m = mx;
                l *= alpha;
                if constexpr (k32) {
                    // (a logit's own rounding is in m, but not in the product here: up to a quarter below 2^23, 128 from 2^31 on, where no weight is finite
                    // or none is left.  Rows that have such logits take the rounded ones.  us without -> with it: 14 / 2 heads of 64, 4 of 64 keys 6.02 -> 6.06, 200 of
                    // 1000 47.1 -> 47.4; of 256, 100 of 500 51.4 -> 52.3; 40 / 8 of 128, 100 of 1000 152.8 -> 153.7)
                    float factor = p.scale_log2;
                    const bool far = !(fabsf(m) < 0x1p23f);
                    if (__builtin_amdgcn_ballot_w64(far) != 0) {  // uniform
                        factor = far ? 1.f : factor;
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int i = 0; i < 4; ++i) raw[t][i] = far ? x[t][i] : raw[t][i];
                    }
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            x[t][i] = x[t][i] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(fmaf(raw[t][i], factor, -m));
#pragma unroll
                    for (int t = 0; t < NT; ++t) l += (x[t][0] + x[t][1]) + (x[t][2] + x[t][3]);
                    f4 sum[2][4];  // (of the 16 keys and columns at hand, and of those before)
#pragma unroll
                    for (int c = 0; c <= D / 16 * NT; ++c) {
                        if (c < D / 16 * NT) {
                            const int t = c % NT, dt = c / NT;
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                sum[c & 1][i] = M::mul(vr[t][i * (D / 64) + dt / 4][dt % 4], __builtin_bit_cast(uint32_t, x[t][i]), f4{0.f, 0.f, 0.f, 0.f});
                        }
                        if (c > 0) {
                            const int dt = (c - 1) / NT;
                            const f4(&u)[4] = sum[~c & 1], y = (u[0] + u[1]) + (u[2] + u[3]);
#pragma unroll
                            for (int i = 0; i < 4; ++i) acc[dt][i] = (c - 1) % NT == 0 ? fmaf(acc[dt][i], alpha, y[i]) : acc[dt][i] + y[i];
                            asm volatile("" : "+v"(acc[dt]));
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    fetch(at + kWaves * NT, false, true);
                    continue;
                } else {
                    uint32_t pw[4] = {0, 0, 0, 0}, pl[4] = {0, 0, 0, 0};  // the weights as a sum of two terms
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        float e[4], f = 1.f;
                        if constexpr (kFp8) f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, vscale), (at + t) & 63));
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            e[i] = __builtin_amdgcn_exp2f(x[t][i] - m);  // 0 for masked keys
                            l += e[i];
                            if constexpr (kFp8) e[i] *= f;
                        }
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            pw[2 * t + i] = W::pack(e[2 * i], e[2 * i + 1]);
                            const float2 high = W::unpack(pw[2 * t + i]);
                            pl[2 * t + i] = W::pack(e[2 * i] - high.x, e[2 * i + 1] - high.y);
                        }
                    }
                    const pa_u4 pb{pw[0], pw[1], pw[2], pw[3]}, pc = again ? pb : pa_u4{pl[0], pl[1], pl[2], pl[3]};
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int dt = 0; dt < D / 16; ++dt) {
                        typedef short s4 __attribute__((ext_vector_type(4)));
                        auto column = [&](int t) {
                            uint16_t *from = vs + (t * kShortKeys + 4 * g + l16 / 4) * kPitch + 16 * dt + 4 * (l16 % 4);
                            return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s4 __attribute__((address_space(3))) *)from));
                        };
                        const uint2 v0 = column(0), v1 = NT == 2 ? column(1) : make_uint2(0, 0);
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[dt][i] *= alpha;
                        const pa_u4 v{v0.x, v0.y, v1.x, v1.y};
                        acc[dt] = W::mul(v, pb, acc[dt]);
                        acc[dt] = W::mul(v, pc, acc[dt]);
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
            }
        }
        if constexpr (kFp8 || k32) break;  // (that type has no infinities; one weight of 32 bits)
        f4 odd = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) odd += acc[dt] * 0.f;
        if (again || __builtin_amdgcn_ballot_w64(!(odd[0] + odd[1] + odd[2] + odd[3] == 0.f)) == 0) break;
    }
    {
        const float2 y = lane_pair<16>(l, 16);
        l = y.x + y.y;
        const float2 z = lane_pair<32>(l, 32);
        l = z.x + z.y;
    }
    if (g == 0) {
        s_m[wave][l16] = m;
        s_l[wave][l16] = l;
    }
    __syncthreads();
    float top = kNegBig;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) top = fmaxf(top, s_m[w][l16]);
    const float mine = __builtin_amdgcn_exp2f(m - top) * (again ? 0.5f : 1.f);
    float *part = reinterpret_cast<float *>(room);  // (every wave is through with V)
#pragma unroll
    for (int h0 = 0; h0 < kShortHeads; h0 += HR) {
        if (h0 >= nr) break;  // uniform
        if (h0 > 0) __syncthreads();
        if (l16 >= h0 && l16 < min(h0 + HR, nr)) {
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) {
                f4 y = acc[dt];
                if constexpr (k32) y = f4{acc[dt / 4 * 4][dt % 4], acc[dt / 4 * 4 + 1][dt % 4], acc[dt / 4 * 4 + 2][dt % 4], acc[dt / 4 * 4 + 3][dt % 4]};
                const int d = k32 ? 64 * (dt / 4) + 16 * g + 4 * (dt % 4) : 16 * dt + 4 * g;
                *reinterpret_cast<f4 *>(part + (wave * HR + l16 - h0) * kPitchO + d) = f4{y[0] * mine, y[1] * mine, y[2] * mine, y[3] * mine};
            }
        }
        __syncthreads();
        const int heads = min(HR, nr - h0);
#pragma unroll 1
        for (int item = tid; item < heads * (D / 4); item += kThreads) {
            const int h = item / (D / 4), d = item % (D / 4) * 4;
            float best = kNegBig, den = 0.f;
            f4 num = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kWaves; ++w) best = fmaxf(best, s_m[w][h0 + h]);
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                den = fmaf(__builtin_amdgcn_exp2f(s_m[w][h0 + h] - best), s_l[w][h0 + h], den);
                num += *reinterpret_cast<const f4 *>(part + (w * HR + h) * kPitchO + d);
            }
            if (d >= p.d) continue;
            if (a.leave) {  // uniform
                const int64_t at = ((int64_t)b * p.hq + kvh * p.n_rep + rep0 + h0 + h) * a.splits + split;
                *reinterpret_cast<f4 *>(a.part_acc + at * p.d + d) = num;
                if (d == 0) *reinterpret_cast<float2 *>(a.part_ml + 2 * at) = make_float2(best, den);
                continue;
            }
            short_store<QT>(orow + (int64_t)(h0 + h) * p.d + d, num, best, den, ez);
        }
    }
}

// One thread per row, four of its elements and eight runs, a wave for 64 of these; P waves of a workgroup take P eights of runs, so that all loads of a row
// are on their way at once.  What it takes is waits: one thread for all runs of its elements, whose loads the compiler moved to where each is used,
// waited for one run after the other.  us a call, that -> this, all dense: 14 / 2 heads of 64, one sequence of 4096 keys (32 runs) 11.3 -> 7.8, of 8192 (64)
// 15.2 -> 8.4; 32 / 8 of 128, one of 1024 (8) 9.0 -> 8.8, of 4096 (32) 12.5 -> 9.4; fp8 14 / 2 of 256, one of 8192 17.7 -> 10.8.
template <typename QT, int P> __global__ __launch_bounds__(64 * P) void decode_short_merge_kernel(const DecodeArgs a) {
    using f4 = typename ShortMfma<QT>::f4;
    constexpr int kPipe = 8, kItems = 64;
    __shared__ float part[P > 1 ? P - 1 : 1][6][kItems];
    const PoolArgs &p = a.p;
    const int per = p.d / 4, at_item = threadIdx.x % kItems, eight = P > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kItems) : 0, item = blockIdx.x * kItems + at_item;
    const bool live = item < a.batch * p.hq * per;
    const int row = live ? item / per : 0, d = (live ? item - row * per : 0) * 4;
    const float *ml = a.part_ml + (int64_t)row * a.splits * 2, *acc = a.part_acc + (int64_t)row * a.splits * p.d + d;
    const int ez = a.extra_zero && a.seq_lens[row / p.hq] > 0 ? max(0, a.extra_zero[row / p.hq]) : 0;
    float best = kNegBig, den = 0.f, num[4] = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](float f, float l, f4 x) {
        den = fmaf(f, l, den);
#pragma unroll
        for (int i = 0; i < 4; ++i) num[i] = fmaf(f, x[i], num[i]);
    };
    auto rise = [&](float top) {
        const float old = __builtin_amdgcn_exp2f(best - top);
        best = top;
        den *= old;
#pragma unroll
        for (int i = 0; i < 4; ++i) num[i] *= old;
    };
#pragma unroll 1
    for (int s = kPipe * eight; s < a.splits; s += kPipe * P) {
        float m[kPipe], l[kPipe], top = best;
        f4 x[kPipe];
#pragma unroll
        for (int j = 0; j < kPipe; ++j) {
            const int at = min(s + j, a.splits - 1);
            const float2 y = *reinterpret_cast<const float2 *>(ml + 2 * at);
            x[j] = *reinterpret_cast<const f4 *>(acc + (int64_t)at * p.d);
            m[j] = y.x;
            l[j] = y.y;
        }
        static_assert(kPipe == 8);
        // (all of them are on their way before the first one is waited for)
        asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]));
#pragma unroll
        for (int j = 0; j < kPipe; ++j) {  // (past the last run: nothing)
            const bool is = s + j < a.splits;
            m[j] = is ? m[j] : kNegBig;
            l[j] = is ? l[j] : 0.f;
            x[j] = is ? x[j] : f4{0.f, 0.f, 0.f, 0.f};
            top = fmaxf(top, m[j]);
        }
        rise(top);
#pragma unroll
        for (int j = 0; j < kPipe; ++j) add(__builtin_amdgcn_exp2f(m[j] - top), l[j], x[j]);
    }
    if constexpr (P > 1) {
        if (eight > 0) {
            float *to = &part[eight - 1][0][at_item];
            to[0] = best;
            to[kItems] = den;
#pragma unroll
            for (int i = 0; i < 4; ++i) to[(2 + i) * kItems] = num[i];
        }
        __syncthreads();
        if (eight > 0) return;
        float top = best;
#pragma unroll
        for (int j = 0; j < P - 1; ++j) top = fmaxf(top, part[j][0][at_item]);
        rise(top);
#pragma unroll
        for (int j = 0; j < P - 1; ++j) {
            const float *from = &part[j][0][at_item];
            add(__builtin_amdgcn_exp2f(from[0] - top), from[kItems], f4{from[2 * kItems], from[3 * kItems], from[4 * kItems], from[5 * kItems]});
        }
    }
    if (!live) return;
    short_store<QT>(reinterpret_cast<QT *>(a.out) + (int64_t)row * p.d + d, num, best, den, ez);
}

template <typename KV, typename QT> KernelSet with_short(KernelSet k, int d) {
    if (!k.split) return k;
    k.few_merge[0] = decode_short_merge_kernel<QT, 1>;
    k.few_merge[1] = decode_short_merge_kernel<QT, 2>;
    k.few_merge[2] = decode_short_merge_kernel<QT, 4>;
    k.few_merge[3] = decode_short_merge_kernel<QT, 8>;
    if (d == 64 || (d == 32 && sizeof(KV) == 4)) k.few = decode_short_kernel<KV, QT, 64>;
    if (d == 128) k.few = decode_short_kernel<KV, QT, 128>;
    if (d == 256) k.few = decode_short_kernel<KV, QT, 256>;
    return k;
}

}  // namespace pa_decode_detail
