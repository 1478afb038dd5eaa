// Portions of prompts of attention with score terms on the matrix cores (16-bit pools, keys and values of up to 256).
//
// A wave owns 32 rows of one query head, a workgroup four (row block, head) pairs of one kv head in turn, which share tiles of
// 64 keys and values in LDS; the next tile is on its way in registers.  As in prefill_mfma.h everything is transposed:
// S^T = K Q^T leaves a lane 16 keys of one row, which in register order are the operand of O^T += V^T P^T.  The distance
// biases of a wave's head lie in LDS, newest key last, with margins on both sides, so that a lane reads the biases of
// consecutive keys side by side; keys past the last distance read its margin.
//
// Bound by a wave's own chain: staging a tile (8 KB of a wave's loads and writes, 1500 of 6000 cycles), scores and weights (four
// transcendentals for two elements with a cap), and no more than two waves of 220 registers on a SIMD to cover it; products of one
// block beside the scores of the other changed nothing.  What did: reads of a product issued together, one wait for the biases, no
// division in the walk over blocks, and the order of the workgroups.  8 prompts of 700 .. 4000 rows, 16 heads of 128 over 4, us:
// window 1024 and cap 176 -> 147, no window 277 -> 192, one prompt of 4000 rows 188 -> 145.
#include "prefill_mfma.h"
#include "scored_attn.h"
#include "sequence_turns.h"

namespace {

using namespace pa_decode_detail;

constexpr int kSpKeys = 64, kSpLow = 32, kSpHigh = 64, kSpMaxBias = 4096;  // (margins of a bias table: its oldest side, its newest)
constexpr float kSpSlack = 8.f;  // log2 of the factor by which a row's reference maximum may lag

// (values: a transposing read takes 64 bytes of four rows, which spread over the banks at a pitch of 64 modulo 256 bytes; at 16 two prompts of
// 754 .. 2313 rows, 16 heads of 128 over 4, took 62.4 us, now 59.9; keys and values of 64 gain nothing: 8 heads over 2, 6 prompts of
// 420 .. 671 rows, 22.3 us at 16, 22.6 at 64)
template <int DK, int DV> struct SpTile {
    static constexpr int k_pitch = DK + 8, v_pitch = DK == 64 && DV == 64 ? DV + 8 : DV + 32;
    static constexpr size_t tiles = (size_t)kSpKeys * (k_pitch + v_pitch) * 2;
};

template <int DK, int DV, bool CAP> __global__ __launch_bounds__(256, DV == 256 ? 1 : 2) void scored_prefill_kernel(const ScoredArgs a, int bias_n, int cus) {
    using M = Mfma16<pa_bf16>;
    using X8 = M::x8;
    using X4 = M::x4;
    using L = SpTile<DK, DV>;
    constexpr bool kAhead = DK <= 128;  // all reads of a product before its first instruction (more would not fit the registers)
    constexpr int KS = DK / 16, DT = DV / 32, NK = kSpKeys * DK / 8 / 256, NV = kSpKeys * DV / 8 / 256;
    extern __shared__ __align__(16) char sp_lds[];
    uint16_t *ks = reinterpret_cast<uint16_t *>(sp_lds), *vs = ks + kSpKeys * L::k_pitch;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, col = lane & 31;
    const int table_n = bias_n + kSpLow + kSpHigh;
    float *bias = reinterpret_cast<float *>(sp_lds + L::tiles) + wave * table_n;
    // The rows with the most keys of all sequences come first, and sequences take turns on the dies and inside them (an odd number of
    // them does by itself: 9 of 700 .. 4000 rows in turn 435 us, else 320); the second workgroup of each compute unit comes the other
    // way round, so that the longest shares its unit with a short one.  8 sequences of 400 .. 4000 rows, 16 heads of 128, in turn, on the
    // dies alone, with fixed places: over one head of keys 171 / 406 / 659 us, two 172 / 239 / 627; on the dies alone, with fixed places:
    // over four 185 / 625, eight 185 / 366, sixteen 176 / 228 (unordered about 240); 4 of them over four 197 / 329 / 277; 8 equal ones
    // 93 / 95 / 91.
    int kvh = blockIdx.x, turn = blockIdx.z, y = blockIdx.y;
    const uint64_t per = (uint64_t)gridDim.x * gridDim.y, place = per * turn + gridDim.x * (uint64_t)y + kvh;
    const uint32_t both = (uint32_t)min(2 * (uint64_t)cus, per * gridDim.z);
    if (place >= (uint32_t)cus && place < both) {
        const uint32_t back = both - 1 - ((uint32_t)place - cus), one = (uint32_t)min(per, (uint64_t)both);
        turn = back / one;
        kvh = back % one % gridDim.x;
        y = back % one / gridDim.x;
    }
    const int b = gridDim.y % 2 == 0 ? sequence_in_turn(y, turn, (int)gridDim.y, turns_miss_groups(gridDim.x, gridDim.y)) : y;
    ScoredPortion p;
    if (!scored_portion(a, b, p)) return;
    const int n_tasks = (p.n + 31) / 32 * a.n_rep;
    const int group = gridDim.z - 1 - turn;
    if (group * 4 >= n_tasks) return;
    const int task = group * 4 + wave, last_task = min(n_tasks, group * 4 + 4) - 1;
    const bool live = task < n_tasks;
    const int row0 = (live ? task / a.n_rep : 0) * 32, h = kvh * a.n_rep + (live ? task % a.n_rep : 0);
    const int row = row0 + col, pos = p.pos0 + min(row, p.n - 1);
    const int my_first = scored_first_key(a, pos);                       // this lane's row: first key, last key is pos
    const int wave_lo = scored_first_key(a, p.pos0 + row0), wave_hi = p.pos0 + min(row0 + 32, p.n);  // keys [lo, hi) of the wave
    const int wg_lo = scored_first_key(a, p.pos0 + group * 4 / a.n_rep * 32);
    const int wg_hi = p.pos0 + min(last_task / a.n_rep * 32 + 32, p.n);
    const float to2 = kScoredLog2e, plain = a.scale * kScoredLog2e;
    const float cap_in = CAP ? 2.f * plain / a.cap : 0.f, cap_out = a.cap * kScoredLog2e;  // tanh(z) = 1 - 2 / (1 + e^(2z))
    // bias[kSpLow - 1 + bias_n - dist]: one entry per distance from bias_n - 1 + kSpLow down to -kSpHigh
    const float shift = CAP ? cap_out : 0.f;
    for (int i = lane; i < table_n; i += 64) {
        const int dist = min(max(kSpLow - 1 + bias_n - i, 0), bias_n - 1);
        bias[i] = (a.bias ? a.bias[(int64_t)h * a.bias_n + dist] * to2 : 0.f) + shift;
    }
    X8 q[KS];
    {
        const uint16_t *src = reinterpret_cast<const uint16_t *>(a.q1) + (p.row0 + min(row, p.n - 1)) * a.q1_row + h * a.q1_head;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int d = 16 * k + 8 * half;
            q[k] = __builtin_bit_cast(X8, d < a.n1 ? *reinterpret_cast<const uint4 *>(src + d) : make_uint4(0, 0, 0, 0));
        }
    }
    f32x16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = 0.f;
    float m = a.sink ? a.sink[h] * to2 : kScoredNone, l = a.sink && half == 0 ? 1.f : 0.f;

    const int32_t *table = a.bt + b * a.bt_stride;
    const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)kvh * a.k_dim, *vp = reinterpret_cast<const uint16_t *>(a.v) + (int64_t)kvh * a.v_dim;
    const int64_t k_tok = (int64_t)a.hkv * a.k_dim, v_tok = (int64_t)a.hkv * a.v_dim;
    const int kreal = (a.n1 + 7) / 8 * 8, vreal = (a.vdim + 7) / 8 * 8;
    // This lane's key of the tile that is fetched next: its block and its place there, carried along (a division for each tile would
    // cost as much as the tile's loads), and the block's id, loaded a tile ahead.
    const int k_start = wg_lo / kSpKeys * kSpKeys, step_blk = kSpKeys / a.bs, step_rem = kSpKeys % a.bs, last_blk = (int)min(a.bt_stride, (int64_t)0x7fffffff) - 1;
    int blk = (k_start + lane) / a.bs, rem = (k_start + lane) % a.bs, id = table[min(blk, last_blk)];
    const bool small = scored_small(a, a.k_dim) && scored_small(a, a.v_dim);
    const ScoredRows k_rows = scored_rows(a, a.k, a.k_dim, kvh), v_rows = scored_rows(a, a.v, a.v_dim, kvh);
    scored_u4 kr[NK], vr[NV];
    auto fetch = [&](int k0) {
        const int slots = k0 + lane < wg_hi && blk <= last_blk && (uint32_t)id < (uint32_t)a.num_blocks ? id * a.bs + rem : -1;
        if (small) {
#pragma unroll
            for (int n = 0; n < NK; ++n) {
                const int c = tid + 256 * n, e = c % (DK / 8) * 8;
                kr[n] = k_rows.load16(__shfl(slots, c / (DK / 8), 64), e < kreal ? 2u * e : kScoredAway);
            }
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                const int c = tid + 256 * n, e = c % (DV / 8) * 8;
                vr[n] = v_rows.load16(__shfl(slots, c / (DV / 8), 64), e < vreal ? 2u * e : kScoredAway);
            }
        } else {
#pragma unroll
            for (int n = 0; n < NK; ++n) {
                const int c = tid + 256 * n, s = __shfl(slots, c / (DK / 8), 64), e = c % (DK / 8) * 8;
                kr[n] = scored_load16(kp + s * k_tok + e, s >= 0 && e < kreal);
            }
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                const int c = tid + 256 * n, s = __shfl(slots, c / (DV / 8), 64), e = c % (DV / 8) * 8;
                vr[n] = scored_load16(vp + s * v_tok + e, s >= 0 && e < vreal);
            }
        }
        blk += step_blk;
        rem += step_rem;
        if (rem >= a.bs) {
            rem -= a.bs;
            ++blk;
        }
        id = table[min(blk, last_blk)];
    };
    const int g16 = lane >> 4, s16 = lane & 15;
    const uint16_t *v_at = vs + (4 * (g16 >> 1) + (s16 >> 2)) * L::v_pitch + 16 * (g16 & 1) + 4 * (s16 & 3);
    const int last_first = scored_first_key(a, wave_hi - 1);
    // The steps of a block of 32 keys from kb, at row `at` of the tile.  Element i: key kb + 8 (i / 4) + 4 half + i % 4.
    auto key = [&](int at, int k) {
        return __builtin_bit_cast(X8, *reinterpret_cast<const uint4 *>(ks + (at + col) * L::k_pitch + 16 * k + 8 * half));
    };
    auto read_bias = [&](float (&add)[16], int kb) {  // (below the table every distance shares the last bias, as in its margin)
        const float *bp = bias + max(kSpLow - 1 + bias_n - (p.pos0 + row) + kb + 4 * half, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) add[i] = bp[8 * (i >> 2) + (i & 3)];
    };
    auto read_values = [&](X8 (&va)[DT], int at) {
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const X4 x = M::tr_read(v_at + at * L::v_pitch + 32 * t), y = M::tr_read(v_at + (at + 8) * L::v_pitch + 32 * t);
#pragma unroll
            for (int e = 0; e < 4; ++e) { va[t][e] = x[e]; va[t][4 + e] = y[e]; }
        }
    };
    auto score = [&](float x, float add) {
        if constexpr (CAP) return fmaf(-2.f * cap_out, __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * cap_in)), add);
        else return fmaf(x, plain, add);
    };
    auto settle = [&](f32x16 &s, int kb) {  // masks, and the row's reference maximum
        if (kb + 31 > p.pos0 + row0 || kb < last_first) {
            const int hi = pos - kb - 4 * half, lo = my_first - kb - 4 * half;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int idx = 8 * (i >> 2) + (i & 3);
                s[i] = idx <= hi && idx >= lo ? s[i] : kScoredNone;
            }
        }
        float top = fmaxf(s[0], s[1]);
#pragma unroll
        for (int i = 2; i < 16; ++i) top = fmaxf(top, s[i]);
        const auto other = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, top), __builtin_bit_cast(uint32_t, top), false, false);
        top = fmaxf(__builtin_bit_cast(float, (uint32_t)other[0]), __builtin_bit_cast(float, (uint32_t)other[1]));
        if (__ballot(top > m + kSpSlack) != 0) {
            const float next = fmaxf(m, top), keep = __builtin_amdgcn_exp2f(m - next);
            m = next;
            l *= keep;
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[t][i] *= keep;
        }
    };
    auto weigh = [&](const f32x16 &s, uint32_t (&w)[8], int i) {
        const float x = __builtin_amdgcn_exp2f(s[2 * i] - m), y = __builtin_amdgcn_exp2f(s[2 * i + 1] - m);
        l += x + y;
        w[i] = row_pack_bf16(x, y);
    };
    auto weights = [&](const uint32_t (&w)[8], int k2) {
        return __builtin_bit_cast(X8, make_uint4(w[4 * k2], w[4 * k2 + 1], w[4 * k2 + 2], w[4 * k2 + 3]));
    };
    fetch(k_start);
    for (int k0 = k_start; k0 < wg_hi; k0 += kSpKeys) {
#pragma unroll
        for (int n = 0; n < NK; ++n) {
            const int c = tid + 256 * n;
            *reinterpret_cast<scored_u4 *>(ks + c / (DK / 8) * L::k_pitch + c % (DK / 8) * 8) = kr[n];
        }
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int c = tid + 256 * n;
            *reinterpret_cast<scored_u4 *>(vs + c / (DV / 8) * L::v_pitch + c % (DV / 8) * 8) = vr[n];
        }
        __syncthreads();
        if (k0 + kSpKeys < wg_hi) fetch(k0 + kSpKeys);
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int kb = k0 + 32 * sub;  // (uniform per wave)
            if (!live || kb >= wave_hi || kb + 32 <= wave_lo) continue;
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.f;
            X8 va[2][DT];
            float add[16];
            uint32_t w[8];
            if constexpr (kAhead) {
                X8 kf[KS];
#pragma unroll
                for (int k = 0; k < KS; ++k) kf[k] = key(32 * sub, k);
                read_bias(add, kb);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < KS; ++k) s = M::mma(kf[k], q[k], s);
            } else {
#pragma unroll
                for (int k = 0; k < KS; ++k) s = M::mma(key(32 * sub, k), q[k], s);
                read_bias(add, kb);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = score(s[i], add[i]);
            settle(s, kb);
            if constexpr (kAhead) {
                read_values(va[0], 32 * sub);
                read_values(va[1], 32 * sub + 16);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int k2 = 0; k2 < 2; ++k2) {
#pragma unroll
                for (int i = 4 * k2; i < 4 * k2 + 4; ++i) weigh(s, w, i);
                if constexpr (!kAhead) read_values(va[k2], 32 * sub + 16 * k2);
#pragma unroll
                for (int t = 0; t < DT; ++t) o[t] = M::mma(va[k2][t], weights(w, k2), o[t]);
            }
        }
        __syncthreads();
    }
    const float f = 1.f / (l + __shfl_xor(l, 32, 64));
    if (!live || row >= p.n) return;
    pa_bf16 *out = reinterpret_cast<pa_bf16 *>(a.out) + ((p.row0 + row) * a.heads + h) * a.vdim;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d = 32 * t + 8 * g + 4 * half;
            if (d >= a.vdim) continue;
            if (a.vdim % 4 == 0) {
                *reinterpret_cast<uint2 *>(out + d) = make_uint2(row_pack_bf16(o[t][4 * g] * f, o[t][4 * g + 1] * f),
                                                                 row_pack_bf16(o[t][4 * g + 2] * f, o[t][4 * g + 3] * f));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (d + i < a.vdim) pa_scalar<pa_bf16>::store(out + d + i, o[t][4 * g + i] * f);
            }
        }
}

template <int DK, int DV, bool CAP> int launch_prefill(const ScoredArgs &a, int bias_n, int cus, hipStream_t s) {
    const size_t lds = SpTile<DK, DV>::tiles + (size_t)4 * (bias_n + kSpLow + kSpHigh) * sizeof(float);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(scored_prefill_kernel<DK, DV, CAP>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return pa_fail(PA_ERR_HIP, "pa_scored_attention: %s", hipGetErrorString(e));
    }
    const int groups = ((a.max_q_len + 31) / 32 * a.n_rep + 3) / 4;
    PA_REQUIRE(groups <= 65535, "pa_scored_attention: max_q_len=%d is too long for one launch", a.max_q_len);
    scored_prefill_kernel<DK, DV, CAP><<<dim3((unsigned)a.hkv, (unsigned)a.batch, (unsigned)groups), dim3(256), lds, s>>>(a, bias_n, cus);
    PA_CHECK_LAUNCH("pa_scored_attention (portions)");
    return PA_OK;
}

template <int DK, int DV> int launch_prefill_cap(const ScoredArgs &a, int bias_n, int cus, hipStream_t s) {
    return a.cap > 0.f ? launch_prefill<DK, DV, true>(a, bias_n, cus, s) : launch_prefill<DK, DV, false>(a, bias_n, cus, s);
}

}  // namespace

bool pa_scored_prefill_launch(const ScoredArgs &a, int dtype, int cus, hipStream_t s, int &rc) {
    const int most = a.n1 > a.vdim ? a.n1 : a.vdim;
    const uintptr_t at = (uintptr_t)a.q1 | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.out;
    int bias_n = a.bias ? a.bias_n : 1;
    if (a.window > 0 && bias_n > a.window) bias_n = a.window;  // (no distance reaches the window)
    if (dtype != PA_BF16 || !a.q_lens || a.n2 != 0 || most > 256 || bias_n > kSpMaxBias || (at & 15u) != 0 || a.n1 % 8 != 0 ||
        a.k_dim % 8 != 0 || a.v_dim % 8 != 0 || a.q1_row % 8 != 0 || a.q1_head % 8 != 0 || a.num_blocks * a.bs >= 0x7fffffff ||
        a.bt_stride == 0 || !(a.scale > 0.f))
        return false;
    rc = most <= 64                        ? launch_prefill_cap<64, 64>(a, bias_n, cus, s)
         : most <= 128                     ? launch_prefill_cap<128, 128>(a, bias_n, cus, s)
         : a.n1 <= 192 && a.vdim <= 128    ? launch_prefill_cap<192, 128>(a, bias_n, cus, s)
                                           : launch_prefill_cap<256, 256>(a, bias_n, cus, s);
    return true;
}
