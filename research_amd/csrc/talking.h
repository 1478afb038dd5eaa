// Attention whose heads' weights are mixed before they meet the values, over a paged context:
//     s_g(i, j) = scale q_i . k_j - size[g] ln(1 + rate[g] (i - j)),   p_g(i, j) = e^s_g(i, j) / sum over visible j' of e^s_g(i, j')
//     out_h(i) = sum over visible j of (sum_g talk[h][g] p_g(i, j)) v_j        (v of h's own kv head)
// A weight enters the mixture normalised, so every head's sum comes first: a pass over the keys alone leaves
// lse = log2 of the sum of 2^(s log2 e) per row and head.
#pragma once
#include "scored_attn.h"
#include "sequence_turns.h"

struct TalkArgs : ScoredArgs {  // (q1, n1: the queries; cap, bias, sink, window unused)
    const float *size, *rate;   // [heads], or NULL: no distance bias
    const float *talk;          // [heads][heads]
    float *lse;                 // [rows][heads], base 2
    float *scores;              // decode: [batch][heads][keys_cap], base 2
    int64_t keys_cap;
    int bs_shift;               // log2 of the block size, -1: it is no power of two
    uint32_t bs_magic;          // key / block size = (2 key * bs_magic >> 32) >> bs_magic_shift (key < 2^31)
    int bs_magic_shift;
    bool in_order;              // portions: workgroups take the blocks of rows in the order of their keys
};

// scored_block_id and scored_slot_of without a division where the block size allows it (key < 2^31, bt_stride > 0)
__device__ __forceinline__ int talk_block(const TalkArgs &a, int key) { return a.bs_shift >= 0 ? key >> a.bs_shift : key / a.bs; }
__device__ __forceinline__ int talk_block_id(const TalkArgs &a, const int32_t *table, int key) {
    return table[min((int64_t)talk_block(a, key), a.bt_stride - 1)];
}
__device__ __forceinline__ int talk_slot_of(const TalkArgs &a, int id, int key, int end) {
    const int blk = talk_block(a, key);
    return key < end && blk < a.bt_stride && (uint32_t)id < (uint64_t)a.num_blocks ? id * a.bs + (key - blk * a.bs) : -1;
}

// The distance bias in units of the base-2 exponential.
__device__ __forceinline__ float talk_bias(float size, float rate, int dist) {
    return -size * __builtin_amdgcn_logf(fmaf(rate, (float)dist, 1.f));
}

// The same, and nothing where the key lies behind the row.
__device__ __forceinline__ float talk_masked_bias(float size, float rate, int dist) {
    return dist >= 0 ? talk_bias(size, rate, dist) : kScoredNone;
}

// Which sequence a workgroup takes whose index in them is x, in the row block (from the longest rows) y.  Workgroups go to the
// eight XCDs in turn, so that b = x would keep a sequence on one of them where their number is a multiple of 8, on some where it is
// even, and a batch of ragged lengths would wait for the one with the longest: 8 sequences of 818 to 3868 tokens with 16 heads
// 1260 us, in turn 508.  An odd number turns by itself, and equal lengths are better off with a sequence's keys on one XCD (7 ragged
// ones with 32 heads of 96 x 64: 91 us, in turn 100; 16 of 500 tokens 77, in turn 80).
__device__ __forceinline__ int talk_sequence(const TalkArgs &a, int x, int y) {
    const bool turn = a.batch % 2 == 0 && a.n_rows != (int64_t)a.batch * a.max_q_len;
    return turn ? sequence_in_turn(x, y, a.batch, true) : x;
}

constexpr int kTalkMaxHeads = 128;

// false: no matrix-core kernels for these sizes
bool pa_talking_decode_launch(const TalkArgs &a, int dtype, void *workspace, size_t workspace_bytes, hipStream_t s, int &rc);
bool pa_talking_prefill_launch(const TalkArgs &a, int dtype, hipStream_t s, int &rc);
size_t pa_talking_decode_bytes(int batch, int heads, int kv_heads, int vdim, int64_t max_keys);
