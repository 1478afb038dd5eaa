// Host-testable arithmetic of attention with mixed heads: which kernel takes a call's prompts, and a division that kernels make without one.  Plain C++.
#pragma once
#include <algorithm>
#include <stdint.h>

// key / block size = (2 key * mul >> 32) >> shift for keys of 0 .. 2^31 - 1 (2^shift is the next power of two, at most 2^31)
struct TalkDivision {
    uint32_t mul;
    int shift;
};
static inline TalkDivision talk_division(int block_size) {
    TalkDivision d{0, 0};
    while (d.shift < 31 && (1ll << d.shift) < block_size) ++d.shift;
    d.mul = (uint32_t)(((1ull << (31 + d.shift)) + block_size - 1) / block_size);
    return d;
}

constexpr int kTalkPipeRows = 16;  // rows of a block

// Whether prompts go to the kernel with waves of two kinds: up to 16 heads, whose fours share a kv head.
// More than 8 heads: a workgroup of it has a compute unit to itself, and nothing covers its set-up; two of the kernel with waves of one kind share
// one, which begin sooner.  So the keys that a block meets on average have to make up for each round of workgroups (as measured, for
// no more than three); where blocks go in order over portions of unequal length, which ends the last round sooner, for one alone.  From shapes alone: the tables' width stands for the longest context.
// us, waves of one kind -> of two, prompts of n rows, 16 / 4 heads of 128: one round, 18 of 224 37.7 -> 38.3, 14 of 288 43.0 -> 42.5, 8 of 512 59 -> 56;
// two, 18 of 300 50.8 -> 56.1, 12 of 416 54 -> 57, 9 of 512 61 -> 58; three, 22 of 512 111 -> 113, 12 of 896 148 -> 144; eight, 333 of 96 161 -> 176, 62 of 512
// 292 -> 312, 50 of 640 323 -> 332, 36 of 896 390 -> 381; in order, 40 of 1 .. 400 76 -> 69, 40 of 300 .. 600 171 -> 163; 128 of 64 behind 300 97 -> 95.  Over 202 such
// batches with 16 and 12 heads of 64 to 128 the choice takes 0.955 of the one kind's time, 1.02 at worst (16 of 175 .. 355).
static inline bool talk_pipe_takes(int heads, int n_rep, int batch, int max_q_len, int64_t n_rows, int64_t room, int cus) {  // room: keys that a row of the tables has places for
    if (heads > 16 || n_rep % 4 != 0) return false;
    if (heads <= 8) return true;
    const int64_t most = (max_q_len + kTalkPipeRows - 1) / kTalkPipeRows, whole = (int64_t)batch * max_q_len;
    const int64_t blocks = std::min(batch * most, n_rows / kTalkPipeRows + batch / 2), rounds = std::min<int64_t>((blocks + cus - 1) / cus, 3);
    const bool uneven = batch <= 64 && 5 * n_rows <= 4 * whole;
    const int64_t behind = std::max<int64_t>(room - max_q_len, 0), mean = uneven ? max_q_len / 2 : std::min<int64_t>(max_q_len / 2, n_rows / batch);
    return behind + mean >= 128 * (uneven ? 1 : rounds);
}

// Whether its workgroups take the blocks in the order of their keys: where a wave can look over all portions at once and not all workgroups begin
// together anyway (one of more than 8 heads has a compute unit, two of up to 8).
static inline bool talk_pipe_in_order(int heads, int batch, int max_q_len, int cus) {
    const int64_t blocks = (int64_t)batch * ((max_q_len + kTalkPipeRows - 1) / kTalkPipeRows);
    return batch <= 64 && blocks > (int64_t)cus * (heads <= 8 ? 2 : 1);
}
