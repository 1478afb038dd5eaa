// Portions of prompts of attention with mixed heads on the matrix cores (16-bit pools, keys and values of up to 128, up to 32
// heads).
//
// The first kernel leaves every row's and head's sum: a wave owns 32 rows of one head, a workgroup four (row block, head) pairs
// of one kv head, which share tiles of 64 keys in LDS (as in scored_prefill.hip, without values).  The second one makes the
// scores again, for all heads at once: a workgroup owns 16 rows and 16 out heads, its eight waves have their own heads' queries
// and two out heads' accumulators in registers.  Per tile of 32 keys
//   1. S^T = K Q^T leaves a lane four keys of one row per head; the weights go to LDS, all heads of a (key, row) pair side by
//      side, as two bf16 terms;
//   2. T times these, the pairs of four keys per wave, and back to LDS as weights of (out head, row), keys side by side;
//   3. O^T += V^T W^T per out head, V by transposing reads from the wave's own part of LDS.
// The next tile's keys and values are on their way in registers.  Distance biases of a head are one logarithm per lane and
// tile, spread by LDS.  Up to 16 heads whose fours share a kv head have a kernel whose waves are of two kinds (talk_pipe_kernel).
#include "linear_tiles.h"
#include "prefill_mfma.h"
#include "talking.h"
#include "talking_plan.h"

namespace {

using namespace pa_decode_detail;

// A key whose block is missing: zeros for a row of up to 128 elements.  (Read as global memory, like kScoredZeros.)
__device__ const uint32_t kTalkNoKey[64] __attribute__((aligned(16))) = {0};
typedef const __attribute__((address_space(1))) scored_u4 *talk_global;

constexpr float kTpSlack = 8.f;  // log2 of the factor by which a row's reference maximum may lag

__device__ __forceinline__ void tp_own_lds() {  // a wave's own part of LDS: its writes before its reads
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ------------------------------------------------------------------ sums
constexpr int kTsKeys = 64;
template <int DK> __global__ __launch_bounds__(256, 2) void talk_sums_kernel(const TalkArgs a) {
    using M = Mfma16<pa_bf16>;
    using X8 = M::x8;
    constexpr int KS = DK / 16, NK = kTsKeys * DK / 8 / 256, kPitch = DK + 8;
    __shared__ __align__(16) uint16_t ks[kTsKeys * kPitch];
    __shared__ float biases[4][2][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, col = lane & 31;
    const int kvh = blockIdx.y, b = talk_sequence(a, blockIdx.x, blockIdx.z);
    ScoredPortion p;
    if (!scored_portion(a, b, p)) return;
    const int n_tasks = (p.n + 31) / 32 * a.n_rep;
    const int group = gridDim.z - 1 - blockIdx.z;  // (the rows with the most keys first)
    if (group * 4 >= n_tasks) return;
    const int task = group * 4 + wave, last_task = min(n_tasks, group * 4 + 4) - 1;
    const bool live = task < n_tasks;
    const int row0 = (live ? task / a.n_rep : 0) * 32, h = kvh * a.n_rep + (live ? task % a.n_rep : 0);
    const int row = row0 + col, wave_hi = p.pos0 + min(row0 + 32, p.n);
    const int wg_hi = p.pos0 + min(last_task / a.n_rep * 32 + 32, p.n);
    const float plain = a.scale * kScoredLog2e, size = a.size ? a.size[h] : 0.f, rate = a.rate ? a.rate[h] : 0.f;
    X8 q[KS];
    {
        const uint16_t *src = reinterpret_cast<const uint16_t *>(a.q1) + (p.row0 + min(row, p.n - 1)) * a.q1_row + h * a.q1_head;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int d = 16 * k + 8 * half;
            q[k] = __builtin_bit_cast(X8, d < a.n1 ? *reinterpret_cast<const uint4 *>(src + d) : make_uint4(0, 0, 0, 0));
        }
    }
    // the row's reference m, which the products start from (as -m / plain), and the sum of 2^(score - m)
    float m = 0.f, l = 0.f;
    const float unplain = 1.f / plain;
    f32x16 start;
#pragma unroll
    for (int i = 0; i < 16; ++i) start[i] = 0.f;
    const int32_t *table = a.bt + b * a.bt_stride;
    const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + (int64_t)kvh * a.k_dim;
    const int64_t k_tok = (int64_t)a.hkv * a.k_dim;
    auto id_of = [&](int k0) { return talk_block_id(a, table, min(k0 + lane, wg_hi - 1)); };
    scored_u4 kr[NK];
    auto fetch = [&](int id, int k0) {
        const int slots = talk_slot_of(a, id, k0 + lane, wg_hi);
#pragma unroll
        for (int n = 0; n < NK; ++n) {
            const int c = tid + 256 * n, s = __shfl(slots, c / (DK / 8), 64), e = c % (DK / 8) * 8;
            kr[n] = scored_load16(kp + s * k_tok + e, s >= 0 && e < a.n1);
        }
    };
    fetch(id_of(0), 0);
    int id = id_of(kTsKeys);
    for (int k0 = 0; k0 < wg_hi; k0 += kTsKeys) {
#pragma unroll
        for (int n = 0; n < NK; ++n) {
            const int c = tid + 256 * n;
            *reinterpret_cast<scored_u4 *>(ks + c / (DK / 8) * kPitch + c % (DK / 8) * 8) = kr[n];
        }
        __syncthreads();
        if (k0 + kTsKeys < wg_hi) {
            fetch(id, k0 + kTsKeys);
            id = id_of(k0 + 2 * kTsKeys);
        }
        if (live && k0 < wave_hi) {  // distances p.pos0 + row0 + i - k of i < 32 and each half's 32 keys, from their smallest
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
                biases[wave][sub][lane] = talk_masked_bias(size, rate, p.pos0 + row0 - (k0 + 32 * sub + 31) + lane);
            tp_own_lds();
        }
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int kb = k0 + 32 * sub;  // (uniform per wave)
            if (!live || kb >= wave_hi) continue;
            f32x16 s = start;
#pragma unroll
            for (int k = 0; k < KS; ++k)
                s = M::mma(__builtin_bit_cast(X8, *reinterpret_cast<const uint4 *>(ks + (32 * sub + col) * kPitch + 16 * k + 8 * half)), q[k], s);
            // element i: key kb + 8 (i / 4) + 4 half + i % 4
            const float *bp = biases[wave][sub] + col + 31 - 4 * half;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = fmaf(s[i], plain, bp[-(8 * (i >> 2) + (i & 3))]);
            float top = fmaxf(s[0], s[1]);
#pragma unroll
            for (int i = 2; i < 16; ++i) top = fmaxf(top, s[i]);
            // (every lane has a reference of its own; it follows when a score is far above it, or the first ones all far below)
            if (__ballot(top > kTpSlack || (l == 0.f && top > 0.5f * kScoredNone && top < -kTpSlack)) != 0) {
                const float by = top > kTpSlack || (l == 0.f && top > 0.5f * kScoredNone) ? top : 0.f;
                l *= __builtin_amdgcn_exp2f(-by);
                m += by;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[i] -= by;
                    start[i] = -m * unplain;
                }
            }
#pragma unroll
            for (int i = 0; i < 16; i += 2) l += __builtin_amdgcn_exp2f(s[i]) + __builtin_amdgcn_exp2f(s[i + 1]);
        }
        __syncthreads();
    }
    // (a lane that saw no key has nothing to say)
    if (l == 0.f) m = kScoredNone;
    const float other = __shfl_xor(m, 32, 64), top = fmaxf(m, other);
    l *= __builtin_amdgcn_exp2f(m - top);
    l += __shfl_xor(l, 32, 64);
    if (live && row < p.n && half == 0) a.lse[(p.row0 + row) * a.heads + h] = top + __builtin_amdgcn_logf(l);
}

// ------------------------------------------------------------------ mixed weights times values
constexpr int kTmRows = 16, kTmKeys = 32, kTmWaves = 8, kTmThreads = 64 * kTmWaves;
constexpr int kTmOut = 2 * kTmWaves;  // out heads of a workgroup, two per wave

// Up to 16 heads there is room for the weights of two tiles, and the next tile's are made beside the mixing of this one's: a tile takes 4600 cycles,
// else 4850, of which the mixing's few reads and products were 500 (8 prompts of 700 .. 4000 rows, 16 heads of 128: 419 -> 407 us).  It begins with two more
// barriers and a wait for the second tile's keys, so up to eight tiles stay as they were (25 .. 111 rows, 8 heads: 19.8 us, else 20.5).
constexpr int kTmAhead = 8;

// HW: heads per wave, 2 or 4.  NG: kv heads of the out heads, whose values are staged by the whole workgroup (0: each wave
// stages its own).  With two heads per wave the keys of up to NG kv heads are staged as well, and there is room for the weights of two tiles.
template <int D, int HW, int NG> struct TmTile {
    static constexpr int heads = kTmWaves * HW, kPitch = D + 16, vPitch = NG ? D + 16 : D + 8;
    static constexpr bool ahead = NG > 0 && HW == 2;
    static constexpr int pair = 4 * heads;  // bytes of a (key, row) pair: both terms of all heads
    static constexpr int pTile = kTmKeys * kTmRows * pair, pBytes = (ahead ? 2 : 1) * pTile, wBytes = kTmOut * kTmRows * kTmKeys * 2, kTile = kTmKeys * kPitch, vTile = kTmKeys * vPitch + (NG ? 3 * 64 : 0);
    // (a transposing read takes four rows of four sets eight apart)
    static constexpr __device__ int vRow(int row) { return row * vPitch + (NG ? row / 8 * 64 : 0); }
    static constexpr int vBytes = (NG ? NG : kTmWaves) * vTile * 2, kBytes = ahead ? NG * kTile * 2 : 0;
    static constexpr int biasFloats = HW * 48;
    static constexpr size_t bytes = (size_t)pBytes + wBytes + vBytes + kBytes + kTmWaves * biasFloats * 4;
};

// D: keys and values padded to 64 or 128; FULL: they fill it.  NG > 0: a wave's heads share a kv head, and so do its out heads.
template <int D, int HW, bool FULL, int NG> __global__ __launch_bounds__(kTmThreads) void talk_mix_kernel(const TalkArgs a) {
    using L = TmTile<D, HW, NG>;
    constexpr bool SAME = NG > 0;
    constexpr int HP = L::heads, KS = D / 32, ET = D / 16;
    constexpr int kPer = D / 8, kTile = kTmKeys * kPer;                     // 16-byte pieces of a row, of a kv head's tile
    constexpr int NV = SAME ? NG * kTile / kTmThreads : kTile / 64, NK = L::ahead ? NV : 2 * KS;
    extern __shared__ __align__(16) char tm_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    char *w_s = tm_lds + L::pBytes;
    __bf16 *v_all = reinterpret_cast<__bf16 *>(w_s + L::wBytes), *k_s = v_all + L::vBytes / 2;
    float *biases = reinterpret_cast<float *>(w_s + L::wBytes + L::vBytes + L::kBytes) + wave * L::biasFloats;
    const int b = talk_sequence(a, blockIdx.x, blockIdx.y);
    ScoredPortion p;
    if (!scored_portion(a, b, p)) return;
    const int row0 = (int)(gridDim.y - 1 - blockIdx.y) * kTmRows;  // (the rows with the most keys first)
    if (row0 >= p.n) return;
    const int row = row0 + l16, first_pos = p.pos0 + row0, end = p.pos0 + min(row0 + kTmRows, p.n);
    const float plain = a.scale * kScoredLog2e;
    const int head0 = wave * HW, out0 = blockIdx.z * kTmOut, own0 = out0 + 2 * wave;  // the wave's heads and out heads
    auto kv_of = [&](int h) { return min(h, a.heads - 1) / a.n_rep; };
    // T in the pairs' k order (terms of 32 heads, or both of 16): out head out0 + l16; the second term of T meets the first of
    // the weights only
    bf8 t_hi, t_lo;
    bool t_rest;  // (a matrix stored in 16 bits has no second term)
    {
        LaSplit sp;
        bool exact = true;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int turned = HW == 4 ? j ^ (2 * (wave & 1)) : j ^ (wave & 3);  // (as the weights of this wave's keys lie)
                const int out = out0 + l16, in = (8 * g + 2 * turned + e) % HP;
                x[e] = out < a.heads && in < a.heads ? a.talk[(int64_t)out * a.heads + in] : 0.f;
            }
            la_split2(x[0], x[1], sp.hi[j], sp.lo[j]);
            exact = exact && sp.lo[j] == 0;
            if (HP == 16 && g >= 2) sp.lo[j] = 0;
        }
        t_hi = sp.high();
        t_lo = sp.low();
        t_rest = __ballot(!exact) != 0;
    }
    bf8 q[HW][KS];
    float lse[HW], size[HW], rate[HW];
    f4 start[HW];  // two heads per wave: the products start from -lse
    {
        const int64_t mem_row = p.row0 + min(row, p.n - 1);
#pragma unroll
        for (int i = 0; i < HW; ++i) {
            const int h = min(head0 + i, a.heads - 1);
            const uint16_t *src = reinterpret_cast<const uint16_t *>(a.q1) + mem_row * a.q1_row + h * a.q1_head;
#pragma unroll
            for (int k = 0; k < KS; ++k) q[i][k] = __builtin_bit_cast(bf8, scored_load16(src + 32 * k + 8 * g, 32 * k + 8 * g < a.n1));
            lse[i] = row < p.n && head0 + i < a.heads ? a.lse[mem_row * a.heads + h] : -kScoredNone;  // (no head, no row: no weight)
            size[i] = a.size ? a.size[h] : 0.f;
            rate[i] = a.rate ? a.rate[h] : 0.f;
            const float from = HW == 2 ? -lse[i] / plain : 0.f;
            start[i] = f4{from, from, from, from};
        }
    }
    f4 o[2][ET];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < ET; ++t) o[i][t] = f4{0.f, 0.f, 0.f, 0.f};

    const int32_t *table = a.bt + b * a.bt_stride;
    const uint32_t k_tok = (uint32_t)(a.hkv * a.k_dim), v_tok = (uint32_t)(a.hkv * a.v_dim);
    const int vreal = (a.vdim + 7) / 8 * 8;
    // the kv heads that are staged: from the first of the out heads, from the first of all
    const int v_kv0 = kv_of(out0);
    __bf16 *v_s = v_all + (SAME ? kv_of(own0) - v_kv0 : wave) * L::vTile;
    // Block and pool row of the key that this thread stages (values staged by all: the piece of a tile; else key lane % 32); past
    // the last key: the last one's, which nothing weighs.  -1: its block is missing, a key and a value of zeros.  LATE: the pool's first row is loaded then, and
    // zeros take its place where the loads are waited for, in a branch that no other tile takes; else by a choice of addresses for each load, where the
    // branch costs registers that are spilled or saves nothing.  (us, no zeros -> by choice -> LATE: 8 prompts of 818 .. 3868 rows, 6 / 3 heads of 128
    // 451 -> 462 -> 458; 18 of 300, 16 / 4 of 128 46.9 -> 48.3 -> 47.2; kernel alone, heads of a wave of two kv heads, 6 / 2 of 40 x 56 351 -> 370 -> 369, 24 / 8
    // of 64 1040 -> 1083 -> 1104.)
    constexpr bool LATE = SAME && (HW == 2 || D == 64);
    uint64_t k_gone = 0, v_gone = 0;  // LATE: the lanes whose keys are missing of the tiles in kr and vr
    const int my_row = SAME ? tid % kTile / kPer : lane & 31;
    auto key_of = [&](int k0) { return min(k0 + my_row, end - 1); };
    auto id_of = [&](int k0) { return talk_block_id(a, table, key_of(k0)); };
    auto slot_of = [&](int id, int k0) { return talk_slot_of(a, id, key_of(k0), end); };
    scored_u4 kr[NK], vr[NV];
    // staged by the workgroup: piece tid + 512 n is of kv head (tid + 512 n) / kTile, the thread's own row
    auto stage_from = [&](const void *pool, int slot, uint32_t tok, int head_dim, int kv_first, int real, scored_u4 *to) {
        const uint16_t *src = reinterpret_cast<const uint16_t *>(pool) + (uint64_t)(uint32_t)(LATE ? max(slot, 0) : slot) * tok + tid % kPer * 8;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const uint16_t *at = src + min(kv_first + (tid + kTmThreads * n) / kTile, a.hkv - 1) * head_dim;
            to[n] = scored_load16(at, (LATE || slot >= 0) && (FULL || tid % kPer * 8 < real));
        }
    };
    auto stage_to = [&](__bf16 *tiles, int tile, int row_at, const scored_u4 *from) {
#pragma unroll
        for (int n = 0; n < NV; ++n) *reinterpret_cast<scored_u4 *>(tiles + (tid + kTmThreads * n) / kTile * tile + row_at + tid % kPer * 8) = from[n];
    };
    // straight to operands: keys 16 kb + l16 of one kv head (slots: of key lane % 32)
    auto direct_k = [&](int kv, int slots) {
        if constexpr (!L::ahead) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const int slot = __shfl(slots, 16 * kb + l16, 64);
                const uint16_t *pool = reinterpret_cast<const uint16_t *>(a.k) + (uint64_t)(uint32_t)(LATE ? max(slot, 0) : slot) * k_tok + kv * a.k_dim;
                const uintptr_t src = (LATE || slot >= 0 ? reinterpret_cast<uintptr_t>(pool) : reinterpret_cast<uintptr_t>(kTalkNoKey)) + 16 * g;
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    kr[kb * KS + k] = FULL ? *reinterpret_cast<talk_global>(src + 64 * k) : scored_load16(reinterpret_cast<const uint16_t *>(src) + 32 * k, 32 * k + 8 * g < a.n1);
            }
        }
    };
    auto fetch_k = [&](int slots, int near) {  // (near: the slots of keys lane % 32)
        if constexpr (LATE) k_gone = __ballot((L::ahead ? slots : near) < 0);
        if constexpr (L::ahead) stage_from(a.k, slots, k_tok, a.k_dim, 0, a.n1, kr);
        else direct_k(kv_of(head0), near);
    };
    auto own_v = [&](int kv, int slots) {
        if constexpr (!SAME) {
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                const int slot = __shfl(slots, (64 * n + lane) / kPer, 64);
                const uint16_t *src = reinterpret_cast<const uint16_t *>(a.v) + (uint64_t)(uint32_t)slot * v_tok + kv * a.v_dim + lane % kPer * 8;
                vr[n] = scored_load16(src, slot >= 0 && lane % kPer * 8 < vreal);
            }
        }
    };
    auto fetch_v = [&](int slots) {
        if constexpr (LATE) v_gone = __ballot(slots < 0);
        if constexpr (SAME) stage_from(a.v, slots, v_tok, a.v_dim, v_kv0, vreal, vr);
        else own_v(kv_of(own0), slots);
    };
    auto put_v = [&]() {
        if (LATE && (v_gone >> lane & 1)) {
#pragma unroll
            for (int n = 0; n < NV; ++n) vr[n] = scored_u4{0, 0, 0, 0};
        }
        if constexpr (SAME) {
            stage_to(v_all, L::vTile, L::vRow(my_row), vr);
        } else {
#pragma unroll
            for (int n = 0; n < NV; ++n) *reinterpret_cast<scored_u4 *>(v_s + L::vRow((64 * n + lane) / kPer) + lane % kPer * 8) = vr[n];
        }
    };
    // keys by key lane % 32, where they go straight to operands beside values staged by all
    auto near_id = [&](int k0) { return SAME && !L::ahead ? talk_block_id(a, table, min(k0 + (lane & 31), end - 1)) : 0; };
    auto near_slot = [&](int id, int k0, int slots) {
        return SAME && !L::ahead ? talk_slot_of(a, id, min(k0 + (lane & 31), end - 1), end) : slots;
    };
    // 16-byte pieces of a pair's row and of a (head, row)'s keys at places that spread over the banks (by the groups of lanes that a
    // read serves together, linear_tiles.h; with the keys' pitch 8 prompts of 818 .. 3868 tokens 508 -> 494 us); inside a piece the place of a
    // wave's weights also turns with key / 4, and that of its keys with head / 4
    const int turn16 = -(l16 >> 2) & 3;
    char *pairs = tm_lds;  // of the tile whose weights are made
    auto pair_at = [&](int key, int piece) {
        const int at = HP == 32 ? piece ^ ((l16 >> 1) & 7) : piece ^ turn16;
        return pairs + (key * kTmRows + l16) * L::pair + 16 * at;
    };
    auto weights_at = [&](int head, int piece) { return w_s + (head * kTmRows + l16) * (kTmKeys * 2) + 16 * (piece ^ turn16); };

    // ---- scores and weights of keys 16 kb + 4 g + j of row l16 ----
    // (distances first_pos + r - k of 16 rows and 32 keys, from their smallest; a key behind its row gets no weight)
    auto score_tile = [&](int k0, int slots) {
#pragma unroll
        for (int i = 0; i < HW; ++i) {
            const float x = talk_masked_bias(size[i], rate[i], first_pos - (k0 + 31) + lane);
            if (lane < 48) biases[i * 48 + lane] = x;
        }
        tp_own_lds();
        if constexpr (LATE && !L::ahead) {
            if (k_gone != 0) {
#pragma unroll
                for (int i = 0; i < 2 * KS; ++i)
                    if (k_gone >> (16 * (i / KS) + l16) & 1) kr[i] = scored_u4{0, 0, 0, 0};
            }
        }
        auto weights = [&](int i, int kb, f4 s, float *w) {
            const float *bp = biases + i * 48 + l16 + 31 - 16 * kb - 4 * g;
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = __builtin_amdgcn_exp2f(fmaf(s[j], plain, bp[-j]) - (HW == 2 ? 0.f : lse[i]));
        };
        auto put = [&](int kb, float (*w)[4]) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int key = 16 * kb + 4 * g + j;
                if constexpr (HW == 4) {
                    uint2 hi, lo;
                    la_split2(w[0][j], w[1][j], hi.x, lo.x);
                    la_split2(w[2][j], w[3][j], hi.y, lo.y);
                    *reinterpret_cast<uint2 *>(pair_at(key, wave >> 1) + 8 * ((wave ^ g) & 1)) = hi;
                    *reinterpret_cast<uint2 *>(pair_at(key, 4 + (wave >> 1)) + 8 * ((wave ^ g) & 1)) = lo;
                } else {
                    uint32_t hi, lo;
                    la_split2(w[0][j], w[1][j], hi, lo);
                    *reinterpret_cast<uint32_t *>(pair_at(key, wave >> 2) + 4 * ((wave & 3) ^ g)) = hi;
                    *reinterpret_cast<uint32_t *>(pair_at(key, 2 + (wave >> 2)) + 4 * ((wave & 3) ^ g)) = lo;
                }
            }
        };
        if constexpr (SAME) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                float w[HW][4];
                f4 s[HW];
#pragma unroll
                for (int i = 0; i < HW; ++i) s[i] = start[i];
#pragma unroll
                for (int k = 0; k < KS; ++k) {
                    bf8 key;
                    if constexpr (L::ahead) key = la_read8(k_s + kv_of(head0) * L::kTile + (16 * kb + l16) * L::kPitch + 32 * k + 8 * g);
                    else key = __builtin_bit_cast(bf8, kr[kb * KS + k]);
#pragma unroll
                    for (int i = 0; i < HW; ++i) s[i] = la_mfma(key, q[i][k], s[i]);
                }
#pragma unroll
                for (int i = 0; i < HW; ++i) weights(i, kb, s[i], w[i]);
                put(kb, w);
                if (HW == 4) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            float w[2][HW][4];
            int kv = kv_of(head0);
#pragma unroll
            for (int i = 0; i < HW; ++i) {
                if (kv_of(head0 + i) != kv) direct_k(kv = kv_of(head0 + i), slots);
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    f4 s = start[i];
#pragma unroll
                    for (int k = 0; k < KS; ++k) s = la_mfma(__builtin_bit_cast(bf8, kr[kb * KS + k]), q[i][k], s);
                    weights(i, kb, s, w[kb][i]);
                }
            }
            put(0, w[0]);
            put(1, w[1]);
        }
    };
    // ---- mixed: keys 4 wave .. 4 wave + 3 of row l16, out heads 4 g + i ----
    auto mix_tile = [&]() {
        {
            f4 x[4];
            bf8 one[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) one[k] = la_read8(reinterpret_cast<const __bf16 *>(pair_at(4 * wave + k, g)));
#pragma unroll
            for (int k = 0; k < 4; ++k) x[k] = la_mfma(t_hi, one[k], f4{0.f, 0.f, 0.f, 0.f});
            if (t_rest) {
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = la_mfma(t_lo, one[k], x[k]);
            }
            if constexpr (HP == 32) {
#pragma unroll
                for (int k = 0; k < 4; ++k) one[k] = la_read8(reinterpret_cast<const __bf16 *>(pair_at(4 * wave + k, 4 + g)));
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = la_mfma(t_hi, one[k], x[k]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<uint2 *>(weights_at(4 * g + i, wave >> 1) + 8 * ((wave ^ g) & 1)) =
                    make_uint2(row_pack_bf16(x[0][i], x[1][i]), row_pack_bf16(x[2][i], x[3][i]));
        }
    };
    // ---- values ----
    auto value_tile = [&](int now, int slots) {
        bf8 x[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) x[i] = la_read8(reinterpret_cast<const __bf16 *>(weights_at(2 * wave + i, g)));
        const int turn = (wave >> 1 & 1) * 4 * L::vPitch;  // (which four keys come first)
        auto values = [&](int t) {
            const __bf16 *va = v_s + L::vRow(8 * g + (l16 >> 2)) + 16 * t + 4 * (l16 & 3);
            return la_join(la_read_tr(va + turn), la_read_tr(va + 4 * L::vPitch - turn));
        };
        if (SAME || kv_of(own0 + 1) == kv_of(own0)) {
#pragma unroll
            for (int t = 0; t < ET; ++t) {
                const bf8 v = values(t);
#pragma unroll
                for (int i = 0; i < 2; ++i) o[i][t] = la_mfma(v, x[i], o[i][t]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < ET; ++t) o[0][t] = la_mfma(values(t), x[0], o[0][t]);
            own_v(kv_of(own0 + 1), now);
            tp_own_lds();
            put_v();
            tp_own_lds();
#pragma unroll
            for (int t = 0; t < ET; ++t) o[1][t] = la_mfma(values(t), x[1], o[1][t]);
            own_v(kv_of(own0), slots);
        }
    };

    int slots = slot_of(id_of(0), 0), id = id_of(kTmKeys), id_near = near_id(kTmKeys);
    fetch_k(slots, near_slot(near_id(0), 0, slots));
    fetch_v(slots);
    auto put_k = [&] {
        if constexpr (L::ahead) {
            if (LATE && (k_gone >> lane & 1)) {
#pragma unroll
                for (int n = 0; n < NK; ++n) kr[n] = scored_u4{0, 0, 0, 0};
            }
            stage_to(k_s, L::kTile, my_row * L::kPitch, kr);
        }
    };
    if constexpr (L::ahead) {
        put_k();
        __syncthreads();
    }
    if (L::ahead && end > kTmAhead * kTmKeys) {
        // The next tile's weights are made beside the mixing, whose few reads and products alone would only be waited for
        char *mine = tm_lds;
        int k_slots = slot_of(id, kTmKeys);
        id = id_of(2 * kTmKeys);
        fetch_k(k_slots, 0);
        score_tile(0, slots);
        __syncthreads();
        put_k();
        slots = k_slots;
        k_slots = slot_of(id, 2 * kTmKeys);
        id = id_of(3 * kTmKeys);
        fetch_k(k_slots, 0);
        __syncthreads();
        for (int k0 = 0; k0 < end; k0 += kTmKeys) {
            pairs = mine;
            mix_tile();
            put_v();
            fetch_v(slots);  // (past the last key these are the last key's again)
            mine = mine == tm_lds ? tm_lds + L::pTile : tm_lds;
            pairs = mine;
            if (k0 + kTmKeys < end) score_tile(k0 + kTmKeys, 0);
            __syncthreads();
            put_k();
            slots = k_slots;
            k_slots = slot_of(id, k0 + 3 * kTmKeys);
            id = id_of(k0 + 4 * kTmKeys);
            fetch_k(k_slots, 0);
            value_tile(0, 0);
            __syncthreads();  // the next tile's values and mixed weights may be written now
        }
    } else {
        for (int k0 = 0; k0 < end; k0 += kTmKeys) {
            score_tile(k0, slots);
            const int now = slots;
            // (always, so that waits can be counted: past the last key these are the last key's again)
            slots = slot_of(id, k0 + kTmKeys);
            id = id_of(k0 + 2 * kTmKeys);
            const int near = near_slot(id_near, k0 + kTmKeys, slots);
            id_near = near_id(k0 + 2 * kTmKeys);
            fetch_k(slots, near);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            mix_tile();
            put_v();
            put_k();
            fetch_v(slots);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            value_tile(now, slots);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (row >= p.n) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (own0 + i >= a.heads) continue;
        pa_bf16 *out = reinterpret_cast<pa_bf16 *>(a.out) + ((p.row0 + row) * a.heads + own0 + i) * a.vdim;
#pragma unroll
        for (int t = 0; t < ET; ++t) {
            const f4 x = o[i][t];
            const int d = 16 * t + 4 * g;
            if (d >= a.vdim) continue;
            if (FULL || a.vdim % 4 == 0) {
                *reinterpret_cast<uint2 *>(out + d) = make_uint2(row_pack_bf16(x[0], x[1]), row_pack_bf16(x[2], x[3]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (d + e < a.vdim) pa_scalar<pa_bf16>::store(out + d + e, x[e]);
            }
        }
    }
}

// ------------------------------------------------------------------ mixed weights times values, waves of two kinds
// Up to 16 heads whose fours share a kv head: half of the waves make the weights of a tile of 32 keys while the others mix those of the tile before it
// and multiply the mixed ones of the tile before that by the values, so that the vector unit (exponentials, terms) and the matrix cores and LDS
// (mixing, values) are busy side by side, and a tile has one barrier.  A wave has the heads of one kv head, and half of the keys or of the value
// columns: keys go straight to its operands, values to its own part of LDS.  Up to 8 heads two workgroups share a compute unit.
// A tile of 16 heads takes 3500 .. 4400 cycles, of which the vector unit is busy 1750, LDS 1950, the matrix cores 1280 and the first cache 3200 (a
// load of keys that lie 16 bytes a row takes 64 cycles, of whole 128-byte rows 19): what bounds it is the chain of a wave through LDS, at the 128
// registers that 16 waves leave it.  Eight waves of twice the registers took as long (444 us), keys by way of LDS longer (452).
// us a call, the kernel above -> this one: 16 / 4 heads of 128, 8 prompts of 818 .. 3868 rows 480 -> 428, one of 1100 106 -> 91; 8 / 2 of 128, one of 1100
// 87 -> 59; 8 / 2 of 64, 11 of 534 .. 695 55 -> 47, 10 of 28 .. 145 17.1 -> 15.0.  Of more than 8 heads, calls whose blocks meet few keys stay with the kernel
// above (talk_pipe_takes).
constexpr int kTpRows = kTalkPipeRows, kTpKeys = 32;
template <int DV, int G> struct TpTile {  // G: fours of heads, 2 or 4
    static constexpr int heads = 4 * G, part = 2 * G, threads = 64 * 2 * part;       // waves of a kind
    static constexpr int pair = 16 * G, pTile = kTpKeys * kTpRows * pair;            // bytes of a (key, row) pair: both terms of all heads
    static constexpr int wTile = heads * kTpRows * kTpKeys * 2;
    static constexpr int cols = DV / 2, vTile = kTpKeys * cols * 2;                  // a wave's value columns
    static constexpr int biasFloats = 4 * 32;                                        // distances of a wave's heads, twice
    static constexpr int tBytes = G / 2 * 2 * 1024;                                  // both terms of T as operands, in one or two orders
    static constexpr int ring = 4 * kTpKeys;                                         // pool rows of the tiles to come
    static constexpr size_t bytes = 2 * (size_t)pTile + 2 * (size_t)wTile + part * ((size_t)vTile + 2 * biasFloats * 4 + 256) + tBytes + ring * 4;
    // Value rows of 64 or 128 bytes without padding: the 64-byte halves of 128 change places in every second two rows, so that a transposing read (64
    // bytes of four rows) spreads over the banks.
    static constexpr __device__ int vTurn(int row) { return cols == 32 ? 0 : (row >> 1 & 1) * 64; }
};

// A value that is the same in all lanes, as a scalar
__device__ __forceinline__ float tp_scalar(float x) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x))); }

// Which block of 16 rows of which of up to 64 portions has `rank` in their order from the rows furthest behind to the first ones, and that portion (each
// wave by itself).
__device__ __forceinline__ bool tp_block(const TalkArgs &a, int rank, int &b, int &block, ScoredPortion &p) {
    const int lane = threadIdx.x & 63, most = (a.max_q_len + kTpRows - 1) / kTpRows;
    ScoredPortion mine;
    const int blocks = lane < a.batch && scored_portion(a, lane, mine) ? min((mine.n + kTpRows - 1) / kTpRows, most) : 0;
    auto behind = [&](int i) { return __builtin_amdgcn_readlane(la_scan(max(blocks - i, 0), lane), 63); };  // blocks whose number in their portion is at least i
    if (rank >= behind(0)) return false;
    int low = 0, high = most;  // behind(low) > rank >= behind(high)
    while (high - low > 1) {
        const int mid = (low + high) / 2;
        if (behind(mid) > rank) low = mid;
        else high = mid;
    }
    block = low;
    rank -= behind(high);
    const uint64_t there = __ballot(blocks > low);
    b = __builtin_ctzll(__ballot((there >> lane & 1) != 0 && __builtin_popcountll(there & ((1ull << lane) - 1)) == rank));
    p.n = __builtin_amdgcn_readlane(mine.n, b);
    p.pos0 = __builtin_amdgcn_readlane(mine.pos0, b);
    p.row0 = __builtin_amdgcn_readlane((int)mine.row0, b);  // (q_starts has 32 bits)
    return true;
}

template <int DK, int DV, int G, bool FULL> __global__ __launch_bounds__(256 * G, 4) void talk_pipe_kernel(const TalkArgs a) {
    using L = TpTile<DV, G>;
    constexpr int KS = DK / 32, NC = L::cols / 32;
    typedef float f16 __attribute__((ext_vector_type(16)));
    extern __shared__ __align__(16) char tm_lds[];
    // Blocks with the most keys first: in order over all portions where those can be looked over by a wave at once and not all workgroups begin together
    // anyway, else in every portion.  (Beyond 64 portions a look takes as many loads in a row as there are 64s of them, and a search ten looks: 16 / 4 heads
    // of 128, 511 of 16 .. 64 rows and one of 300 287 us, without the search 155; 8 / 2 of 64, 200 of 1 .. 1000 514, 384.)
    int b = talk_sequence(a, blockIdx.x, blockIdx.y), block = (int)(gridDim.y - 1 - blockIdx.y);
    ScoredPortion p;
    if (a.in_order ? !tp_block(a, (int)(blockIdx.y * gridDim.x + blockIdx.x), b, block, p) : !scored_portion(a, b, p)) return;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = all % L::part;
    char *w_all = tm_lds + 2 * L::pTile, *v_all = w_all + 2 * L::wTile;
    float *bias_all = reinterpret_cast<float *>(v_all + L::part * L::vTile);
    f4 *from_all = reinterpret_cast<f4 *>(bias_all + L::part * 2 * L::biasFloats);
    bf8 *t_all = reinterpret_cast<bf8 *>(from_all + L::part * 16);
    int *ring = reinterpret_cast<int *>(reinterpret_cast<char *>(t_all) + L::tBytes);
    const int four = wave % G, head0 = 4 * four, half = wave / G;  // the wave's heads, and which half of keys or columns
    const int kv = min(head0, a.heads - 4) / a.n_rep;
    // Places in LDS that spread over the banks: 16-byte pieces of a pair of 16 heads and of a (head, row)'s keys turn with the row, those of a pair
    // of 8 heads with key / 8; the 8-byte halves of a pair's pieces change places with key / 4, those of a (head, row)'s with head / 4.
    const int turn16 = -(l16 >> 2) & 3;
    const int row0 = block * kTpRows;
    if (row0 >= p.n) return;
    const int row = row0 + l16, first_pos = p.pos0 + row0, end = p.pos0 + min(row0 + kTpRows, p.n), tiles = (end + kTpKeys - 1) / kTpKeys;
    // Pool row of a key, from its block; past the last key: the last one's, which nothing weighs; -1: its block is missing, a key and a value of zeros.
    const int32_t *table = a.bt + b * a.bt_stride;
    const int last_block = (int)min(a.bt_stride, (int64_t)0x7fffffff) - 1, known = (int)a.num_blocks;
    auto block_of = [&](int key) { return (int)(__umulhi(2u * (uint32_t)min(key, end - 1), a.bs_magic) >> a.bs_magic_shift); };
    auto id_of = [&](int key) { return table[min(block_of(key), last_block)]; };
    auto slot_of = [&](int id, int key) {
        const int blk = block_of(key);
        const bool there = (blk <= last_block) & ((uint32_t)id < (uint32_t)known);
        return there ? min(key, end - 1) + (id - blk) * a.bs : -1;
    };
    const int first_id = id_of(tid % (4 * kTpKeys));

    if (all < L::part) {
        // ---- weights of keys 16 half + 4 g + j of row l16 ----
        float *biases = bias_all + wave * 2 * L::biasFloats;
        const float plain = tp_scalar(a.scale * kScoredLog2e);
        bf8 q[4][KS];
        float from[4];
        const int64_t mem_row = p.row0 + min(row, p.n - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int h = min(head0 + i, a.heads - 1);
            const uint16_t *src = reinterpret_cast<const uint16_t *>(a.q1) + mem_row * a.q1_row + h * a.q1_head;
#pragma unroll
            for (int k = 0; k < KS; ++k) q[i][k] = __builtin_bit_cast(bf8, scored_load16(src + 32 * k + 8 * g, FULL || 32 * k + 8 * g < a.n1));
            from[i] = a.lse[mem_row * a.heads + h];
        }
        // keys straight to operands: a lane's pieces of key 16 half + l16 (columns past the last: zeros)
        const uint32_t k_tok = (uint32_t)(a.hkv * a.k_dim) * 2u;
        const char *kp = reinterpret_cast<const char *>(a.k) + ((int64_t)kv * a.k_dim + 8 * g) * 2;
        const int my_key = 16 * half + l16;
        bf8 kr[KS];
        auto fetch = [&](int slot) {
            const char *src = kp + (uint64_t)(uint32_t)slot * k_tok;
            auto load = [&](bool there) {
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    kr[k] = __builtin_bit_cast(bf8, scored_load16(reinterpret_cast<const uint16_t *>(src) + 32 * k, there && (FULL || 32 * k + 8 * g < a.n1)));
            };
            if (__ballot(slot < 0) == 0) load(true);  // (a choice of addresses for each load in place of a branch: 1 to 2 % of a call)
            else load(slot >= 0);
        };
        // (distances first_pos + r - k of 16 rows and 16 keys, from their smallest, of two heads a lane; a key behind its row gets no weight)
        float size[2], rate[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int h = min(head0 + lane / 32 * 2 + i, a.heads - 1);
            const float x = (a.size ? a.size : a.talk)[h], y = (a.rate ? a.rate : a.talk)[h];
            size[i] = a.size ? x : 0.f;
            rate[i] = a.rate ? y : 0.f;
        }
        auto put_biases = [&](int k0, float *to) {
#pragma unroll
            for (int i = 0; i < 2; ++i) to[lane / 32 * 64 + i * 32 + lane % 32] = talk_masked_bias(size[i], rate[i], first_pos - (k0 + 16 * half + 15) + lane % 32);
        };
        if (tid < 3 * kTpKeys) ring[tid] = slot_of(first_id, tid);
        __syncthreads();
        fetch(ring[my_key]);
#pragma unroll
        for (int i = 0; i < 4; ++i) from[i] = -(row < p.n && head0 + i < a.heads ? from[i] : -kScoredNone) / plain;  // (no head, no row: no weight)
        f4 *const start = from_all + wave * 16 + l16;  // the products start from -lse (in LDS: in registers, operands were spilled)
        if (g == 0) *start = f4{from[0], from[1], from[2], from[3]};
        put_biases(0, biases);
        const int my_pairs = ((16 * half + 4 * g) * kTpRows + l16) * L::pair + 8 * ((four ^ g) & 1) + 16 * ((four >> 1) ^ (G == 4 ? turn16 : g >> 1));
        for (int t = 0; t < tiles; ++t) {
            const int pairs = my_pairs + (t & 1) * L::pTile;
            tp_own_lds();
            const int slot = ring[((t + 1) * kTpKeys + my_key) & (L::ring - 1)];
            const float *bp = biases + (t & 1) * L::biasFloats + l16 + 15 - 4 * g;
            f4 s[4];
            const f4 first = *start;
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] = f4{first[i], first[i], first[i], first[i]};
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[i] = la_mfma(kr[k], q[i][k], s[i]);
            fetch(slot);  // (past the last key any)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) s[i][j] = __builtin_amdgcn_exp2f(fmaf(s[i][j], plain, bp[i * 32 - j]));
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint2 hi, lo;
                la_split2(s[0][j], s[1][j], hi.x, lo.x);
                la_split2(s[2][j], s[3][j], hi.y, lo.y);
                *reinterpret_cast<uint2 *>(tm_lds + pairs + j * kTpRows * L::pair) = hi;
                *reinterpret_cast<uint2 *>(tm_lds + (pairs ^ 8 * G) + j * kTpRows * L::pair) = lo;
            }
            put_biases((t + 1) * kTpKeys, biases + (~t & 1) * L::biasFloats);
            __syncthreads();  // the pairs are there, those of the tile before have been read
        }
        __syncthreads();
        return;
    }

    // ---- mixing and values ----
    // T in the pairs' k order.  16 heads: row l16 of T, k = 8 g + e: both terms of 16 heads; 8 heads: two keys at once, rows 8 (key) + head,
    // k = 16 (key) + 8 (term) + head.  The second term of T meets the first of the weights only.  (In LDS: eight registers less.)
    const bf8 *t_s = t_all + (G == 4 ? wave & 1 : 0) * 128 + lane;
    bool t_rest = false;  // (a matrix stored in 16 bits has no second term)
    {
        LaSplit sp;
        bool exact = true;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int turned = j ^ 2 * (G == 4 ? wave & 1 : g >> 1);
                const int out = G == 4 ? l16 : l16 & 7, in = (8 * g + 2 * turned + e) % L::heads;
                const bool there = (out < a.heads) & (in < a.heads) & (G == 4 || l16 >> 3 == g >> 1);
                const float y = a.talk[min(out, a.heads - 1) * a.heads + min(in, a.heads - 1)];  // (loaded without a branch: one trip to memory for all)
                x[e] = there ? y : 0.f;
            }
            la_split2(x[0], x[1], sp.hi[j], sp.lo[j]);
            exact = exact && sp.lo[j] == 0;
            if (G == 4 ? g >= 2 : g & 1) sp.lo[j] = 0;
        }
        if (wave < G / 2) {
            const_cast<bf8 *>(t_s)[0] = sp.high();
            const_cast<bf8 *>(t_s)[64] = sp.low();
        }
        t_rest = __ballot(!exact) != 0;
    }

    f16 o[2][NC];  // out heads head0 + 2 i + (l16's half of 32 lanes), columns col0 + 32 c + ..
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[i][c][e] = 0.f;
    // the wave's values: a whole row of its columns at a time by four or eight lanes, in the order of the lanes (columns past the last: the first ones
    // again, for nobody)
    constexpr int kPer = L::cols / 8, kEach = 64 / kPer, NV = kTpKeys / kEach;
    char *const v_s = v_all + wave * L::vTile;
    const int col0 = half * L::cols, vreal = (a.vdim + 7) / 8 * 8;
    const uint32_t v_tok = (uint32_t)(a.hkv * a.v_dim) * 2u;
    const int my_col = col0 + (lane % kPer * 8 ^ L::vTurn(lane / kPer) / 2), my_key = lane / kPer;
    const char *vp = reinterpret_cast<const char *>(a.v) + ((int64_t)kv * a.v_dim + (FULL || my_col < vreal ? my_col : 0)) * 2;
    scored_u4 vr[NV];
    auto fetch = [&](int k0) {
        const int *slots = ring + ((k0 + my_key) & (L::ring - 1));
        int slot[NV], least = 0;
#pragma unroll
        for (int n = 0; n < NV; ++n) least |= slot[n] = slots[n * kEach];
        auto load = [&](auto there) {
#pragma unroll
            for (int n = 0; n < NV; ++n) vr[n] = scored_load16(reinterpret_cast<const uint16_t *>(vp + (uint64_t)(uint32_t)slot[n] * v_tok), there(slot[n]));
        };
        if (__ballot(least < 0) == 0) load([](int) { return true; });
        else load([](int x) { return x >= 0; });
    };
    auto put_v = [&]() {
#pragma unroll
        for (int n = 0; n < NV; ++n) *reinterpret_cast<scored_u4 *>(v_s + lane * 16 + n * 1024) = vr[n];
    };
    // mixed: keys 4 wave + m of row l16, out heads 4 g + i (8 heads: keys 8 wave + 4 (g / 2) + m, out heads 4 (g % 2) + i)
    const int mix_key = G == 4 ? 4 * wave : 8 * wave + 4 * (g >> 1), mix_head = 4 * (G == 4 ? g : g & 1);
    const int pair_at = (mix_key * kTpRows + l16) * L::pair + 16 * (G == 4 ? g ^ turn16 : (g & 1) ^ (wave & 1));
    const int mixed_at = (mix_head * kTpRows + l16) * (kTpKeys * 2) + 16 * ((mix_key >> 3) ^ turn16) + 8 * ((mix_key >> 2 ^ mix_head >> 2) & 1);
    auto mix = [&](const char *pairs, char *w_s) {
        // (two keys at a time: of four, the loop's registers were spilled)
        uint32_t mixed[2][4];
#pragma unroll
        for (int m = 0; m < 4; m += 2) {
            const bf8 one = la_read8(reinterpret_cast<const __bf16 *>(pairs + pair_at + m * kTpRows * L::pair));
            const bf8 two = la_read8(reinterpret_cast<const __bf16 *>(pairs + pair_at + (m + 1) * kTpRows * L::pair));
            const bf8 t_hi = t_s[0];
            f4 x = la_mfma(t_hi, one, f4{0.f, 0.f, 0.f, 0.f}), y = la_mfma(t_hi, two, f4{0.f, 0.f, 0.f, 0.f});
            if (t_rest) {
                const bf8 t_lo = t_s[64];
                x = la_mfma(t_lo, one, x);
                y = la_mfma(t_lo, two, y);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) mixed[m / 2][i] = row_pack_bf16(x[i], y[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2 *>(w_s + mixed_at + i * kTpRows * kTpKeys * 2) = make_uint2(mixed[0][i], mixed[1][i]);
    };
    const int side = lane >> 5, mine = lane >> 4 & 1;  // (of a product's 32 columns the second 16 are another head's)
    const int x_at = ((head0 + mine) * kTpRows + l16) * (kTpKeys * 2) + 16 * (side ^ turn16);
    const int v_row = 8 * side + (l16 >> 2), v_first = (v_row * L::cols * 2 + mine * 32 + (l16 & 3) * 8) ^ L::vTurn(v_row);  // (rows 4 on: the same turn)
    const int va0 = v_first + (four & 1 ? 4 * L::cols * 2 : 0), va1 = v_first + (four & 1 ? 0 : 4 * L::cols * 2);  // (which four keys come first)
    auto values = [&](const char *w_s) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {  // 16 keys
            bf8 x[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) x[i] = la_read8(reinterpret_cast<const __bf16 *>(w_s + (x_at ^ 32 * k) + 2 * i * kTpRows * kTpKeys * 2));
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const bf8 v = la_join(la_read_tr(reinterpret_cast<const __bf16 *>(v_s + (va0 ^ 64 * c) + k * 16 * L::cols * 2)),
                                      la_read_tr(reinterpret_cast<const __bf16 *>(v_s + (va1 ^ 64 * c) + k * 16 * L::cols * 2)));
#pragma unroll
                for (int i = 0; i < 2; ++i) o[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, x[i], o[i][c], 0, 0, 0);
            }
        }
    };
    int id = id_of(3 * kTpKeys + (lane & 31));
    __syncthreads();
    fetch(0);
    for (int t = 0; t < tiles; ++t) {
        __syncthreads();  // this tile's pairs are there, the mixed weights of the one before too
        if (t > 0) {
            values(w_all + (~t & 1) * L::wTile);
            tp_own_lds();
        }
        __builtin_amdgcn_sched_barrier(0);
        mix(tm_lds + (t & 1) * L::pTile, w_all + (t & 1) * L::wTile);
        put_v();
        fetch((t + 1) * kTpKeys);  // (past the last key any)
        if (wave == 0) {  // pool rows of three tiles ahead: read behind the next barriers, written over four tiles later
            const int key = (t + 3) * kTpKeys + (lane & 31);
            ring[key & (L::ring - 1)] = slot_of(id, key);
            id = id_of(key + kTpKeys);
        }
        tp_own_lds();
    }
    __syncthreads();
    values(w_all + (~tiles & 1) * L::wTile);
    if (row >= p.n) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int h = head0 + 2 * i + mine;
        if (h >= a.heads) continue;
        pa_bf16 *out = reinterpret_cast<pa_bf16 *>(a.out) + ((p.row0 + row) * a.heads + h) * a.vdim;
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
                const f16 x = o[i][c];
                const int d = col0 + 32 * c + 2 * e + 4 * side;
                if (d >= a.vdim) continue;
                if (FULL || a.vdim % 4 == 0) {
                    *reinterpret_cast<uint2 *>(out + d) = make_uint2(row_pack_bf16(x[e], x[e + 1]), row_pack_bf16(x[e + 2], x[e + 3]));
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (d + j < a.vdim) pa_scalar<pa_bf16>::store(out + d + j, x[e + j]);
                }
            }
    }
}

template <int DK, int DV, int G, bool FULL> int launch_pipe(const TalkArgs &a, hipStream_t s) {
    constexpr size_t lds = TpTile<DV, G>::bytes;
    static_assert(lds <= 160 * 1024 / (4 / G), "LDS of one compute unit");
    if (int rc = la_big_lds(talk_pipe_kernel<DK, DV, G, FULL>, lds, "pa_talking_attention")) return rc;
    // (two dimensions: in one, the threads of 1024 portions of up to 65535 rows are more than a launch can have)
    const dim3 grid((unsigned)a.batch, (unsigned)((a.max_q_len + kTpRows - 1) / kTpRows));
    TalkArgs args = a;
    args.in_order = talk_pipe_in_order(a.heads, a.batch, a.max_q_len, la_cus());
    talk_pipe_kernel<DK, DV, G, FULL><<<grid, dim3(TpTile<DV, G>::threads), lds, s>>>(args);
    PA_CHECK_LAUNCH("pa_talking_attention (portions)");
    return PA_OK;
}
template <int DK, int DV> int launch_pipe_size(const TalkArgs &a, hipStream_t s) {
    const bool full = a.n1 == DK && a.vdim == DV;
    if (a.heads <= 8) return full ? launch_pipe<DK, DV, 2, true>(a, s) : launch_pipe<DK, DV, 2, false>(a, s);
    return full ? launch_pipe<DK, DV, 4, true>(a, s) : launch_pipe<DK, DV, 4, false>(a, s);
}

template <int D, int HW, bool FULL, int NG> int launch_mix(const TalkArgs &a, hipStream_t s) {
    constexpr size_t lds = TmTile<D, HW, NG>::bytes;
    static_assert(lds <= 160 * 1024, "LDS of one compute unit");
    if (int rc = la_big_lds(talk_mix_kernel<D, HW, FULL, NG>, lds, "pa_talking_attention")) return rc;
    const dim3 grid((unsigned)a.batch, (unsigned)((a.max_q_len + kTmRows - 1) / kTmRows), (unsigned)((a.heads + kTmOut - 1) / kTmOut));
    talk_mix_kernel<D, HW, FULL, NG><<<grid, dim3(kTmThreads), lds, s>>>(a);
    PA_CHECK_LAUNCH("pa_talking_attention (portions)");
    return PA_OK;
}
template <int D, int HW> int launch_mix_size(const TalkArgs &a, hipStream_t s) {
    // kv heads beside each other that 16 out heads use at most (all of them, with two heads per wave)
    const int use = HW == 2 ? a.hkv : a.n_rep % kTmOut == 0 ? 1 : kTmOut % a.n_rep == 0 ? kTmOut / a.n_rep : (kTmOut - 2) / a.n_rep + 2;
    if (a.n_rep % HW != 0 || use > 4) return launch_mix<D, HW, false, 0>(a, s);
    return a.n1 == D && a.vdim == D ? launch_mix<D, HW, true, 4>(a, s) : launch_mix<D, HW, false, 4>(a, s);
}

}  // namespace

bool pa_talking_prefill_launch(const TalkArgs &a, int dtype, hipStream_t s, int &rc) {
    const int most = a.n1 > a.vdim ? a.n1 : a.vdim;
    const uintptr_t at = (uintptr_t)a.q1 | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.out;
    if (dtype != PA_BF16 || !a.q_lens || most > 128 || a.heads > 32 || (at & 15u) != 0 || a.n1 % 8 != 0 || a.k_dim % 8 != 0 ||
        a.v_dim % 8 != 0 || a.q1_row % 8 != 0 || a.q1_head % 8 != 0 || a.num_blocks * a.bs >= 0x7fffffff || a.num_blocks == 0 || a.bt_stride == 0 || !(a.scale > 0.f))
        return false;
    rc = [&]() -> int {
        const int groups = ((a.max_q_len + 31) / 32 * a.n_rep + 3) / 4;
        PA_REQUIRE(groups <= 65535, "pa_talking_attention: max_q_len=%d is too long for one launch", a.max_q_len);
        const dim3 grid((unsigned)a.batch, (unsigned)a.hkv, (unsigned)groups);
        if (a.n1 <= 64) talk_sums_kernel<64><<<grid, dim3(256), 0, s>>>(a);
        else talk_sums_kernel<128><<<grid, dim3(256), 0, s>>>(a);
        PA_CHECK_LAUNCH("pa_talking_attention (sums)");
        if (talk_pipe_takes(a.heads, a.n_rep, a.batch, a.max_q_len, a.n_rows, a.bt_stride * a.bs, la_cus()) && (int64_t)a.hkv * (a.k_dim > a.v_dim ? a.k_dim : a.v_dim) < (1 << 30)) {
            if (a.n1 <= 64) return a.vdim <= 64 ? launch_pipe_size<64, 64>(a, s) : launch_pipe_size<64, 128>(a, s);
            return a.vdim <= 64 ? launch_pipe_size<128, 64>(a, s) : launch_pipe_size<128, 128>(a, s);
        }
        if (a.heads <= 16) return most <= 64 ? launch_mix_size<64, 2>(a, s) : launch_mix_size<128, 2>(a, s);
        return most <= 64 ? launch_mix_size<64, 4>(a, s) : launch_mix_size<128, 4>(a, s);
    }();
    return true;
}
