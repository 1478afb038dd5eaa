// Bookkeeping of the matrix-core prefill launches: how many pieces a workgroup's tiles are cut into, which tiles a
// piece runs, how many groups of tasks a workgroup runs in turn and which ones, and the size of the workspace.
// Integer arithmetic only; shared by the host entry points (prefill.hip), the kernels (prefill_asm.h,
// prefill_d256.h) and a plain C++ replay that the CPU tests compile with g++ (no HIP needed).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "decode_plan.h"  // PA_PLAN_FN

namespace pa_decode_detail {

constexpr int kPlanMaxPrefillSplits = 8;
constexpr int kPlanMinTilesPerSplit = 8;   // of a piece, whose set-up and write-out cost about six
constexpr int kPlanPieceFixedTiles = 6;    // set-up and write-out of a workgroup, in tiles of its loop
constexpr int kPlanMergeTiles = 9;         // the merge launch, in the same unit (a tile takes about a microsecond)
constexpr int64_t kPlanMergeBytesPerTile = 4500000;  // and what it and the pieces move meanwhile
constexpr int kPlanMaxGroupsPerWorkgroup = 8;

// What a launch costs with its workgroups' tiles cut into s pieces, in tile times: the launch takes rounds of
// `cus` workgroups, each lasting a piece's tiles plus its fixed cost.
PA_PLAN_FN int64_t plan_prefill_cost(int64_t workgroups, int cus, int64_t tiles, int s) {
    const int64_t rounds = (workgroups * s + cus - 1) / cus;
    return rounds * (tiles / s + kPlanPieceFixedTiles);
}

// Pieces to cut every workgroup's tiles into, from shapes alone.  The matrix-core kernels run one workgroup per
// compute unit, each owning 256 (head_dim 256: 128) row-head pairs and all their keys, so a launch of few rows
// leaves compute units idle however long the context is.  The split with the lowest cost wins (the smaller on
// ties), as long as a piece keeps kPlanMinTilesPerSplit tiles of the longest context the block tables can describe.  The cost has the merge in
// it, part_bytes of partial results for each piece.
PA_PLAN_FN int plan_prefill_splits(int64_t workgroups, int cus, int64_t max_keys, int tile_keys, int64_t part_bytes) {
    const int64_t tiles = max_keys / tile_keys;
    int best = 1;
    int64_t best_cost = 0;
    for (int s = 1; s <= kPlanMaxPrefillSplits; ++s) {
        if (s > 1 && tiles / s < kPlanMinTilesPerSplit) break;
        const int64_t merge = s > 1 ? kPlanMergeTiles + 2 * s * part_bytes / kPlanMergeBytesPerTile : 0;
        const int64_t cost = plan_prefill_cost(workgroups, cus, tiles, s) + merge;
        if (s == 1 || cost < best_cost) {
            best_cost = cost;
            best = s;
        }
    }
    return best;
}

// Workgroups with rows that a launch of one group (of `tasks` tasks) each has, about: the longest prompt's length would give all `batch`
// sequences `groups`; `rows` rows fill fewer, and a sequence's last task and last group are half full on average.  A few more than that,
// as one too many for the device costs a round and one too few only a small part of one.
PA_PLAN_FN int64_t plan_prefill_units(int num_kv_heads, int64_t groups, int batch, int64_t rows, int n_rep, int rows_per_task, int tasks) {
    int step = tasks;  // tasks that a sequence's may leave over in its last group: multiples of step
    while (n_rep % step) step /= 2;
    int64_t filled = (2 * rows * n_rep / rows_per_task + (int64_t)batch * (n_rep + tasks - step)) / (2 * tasks) + (batch + 15) / 16;
    filled = filled < batch ? batch : filled;
    return num_kv_heads * (filled < groups * batch ? filled : groups * batch);
}

// Whether a launch's workgroups are numbered by the chunks that have rows (about `units`), not by the places of a grid in which the longest prompt's
// length gives all sequences as many (`places`).  The grid's places go to compute units in turn, with rows or without, so that some get one workgroup
// more than others: by number where that is a round less and the last round is well filled (an emptier one finds room among the places
// without rows).  us, by places -> by number, rounds of 256 places and of chunks: 8 / 2 heads of 128, 29 prompts of 133 .. 319 rows behind
// 4080 keys (1.1, 0.8) 191 -> 115; 32 / 8 of 128, 13 of 75 .. 158 behind 1504 (1.2, 1.0) 88 -> 57, 48 of 99 .. 145 behind 1008 (4.5, 3.7) 172 -> 150;
// 14 / 2 of 128, 13 of 385 .. 962 behind 1104 (2.5, 1.8) 118 -> 96, but 47 of 36 .. 218 behind 720 (2.6, 1.4) 58 -> 60; 32 / 8 of 128, 32 of 97 .. 249
// behind 2048 (4.0, 3.2) 225 -> 234.  Over 311 batches (1 to 64 prompts of up to 8192 rows behind nothing or up to 8192 keys, and one of 200 000; head sizes
// 64 to 256) the rule takes 0.99 of the time of numbering by places, 0.56 at best, and is never slower by more than 3.5 %.
PA_PLAN_FN bool plan_prefill_dense(int64_t units, int64_t places, int cus) {
    const int64_t rounds = (units + cus - 1) / cus;
    return rounds < (places + cus - 1) / cus && 8 * (units - (rounds - 1) * cus) >= 5 * cus;
}

// workspace = [part_o float[row][head][piece][D]] [part_ml float[row][head][piece][2]]
PA_PLAN_FN size_t plan_prefill_ws_bytes(int64_t total_q, int num_q_heads, int head_dim, int splits) {
    return splits <= 1 ? 0 : (size_t)total_q * num_q_heads * splits * ((size_t)head_dim + 2) * sizeof(float);
}

// Piece `piece` of `n_splits` of the n_all tiles from tile t0 on runs the tiles [tb, te) (empty when there are
// fewer tiles than pieces): consecutive, disjoint, sizes that differ by one at most.
PA_PLAN_FN void plan_piece_tiles(int t0, int n_all, int piece, int n_splits, int &tb, int &te) {
    tb = t0 + (int)((int64_t)piece * n_all / n_splits);
    te = t0 + (int)((int64_t)(piece + 1) * n_all / n_splits);
}

// Groups (of 8 tasks) of one (sequence, kv head) that a workgroup of the plain assembly-loop instance runs in turn:
// they share the set-up of lengths and slot tables.  As many (up to 8) as leave a workgroup for every compute unit.
PA_PLAN_FN int plan_groups_per_workgroup(int num_kv_heads, int64_t groups, int batch, int cus) {
    int gpw = 1;
    for (int g = 2; g <= kPlanMaxGroupsPerWorkgroup && g <= groups; ++g)
        if ((int64_t)num_kv_heads * ((groups + g - 1) / g) * batch >= cus) gpw = g;
    return gpw;
}

// The same for prompts of unequal length, given the `rows` of q of all of them: of the groups that equal prompts would share a set-up
// for, the longest prompt's keep one compute unit at work while others have none left.  A launch of U groups, each c tiles of time, takes
// about (U / cus) (c + s / g) + g c e, of which s is a workgroup's set-up and the last term the wait for the workgroups that end
// last, with e the part of the longest prompt's rows that the others lack on average: least at g^2 = s U / (c cus e).  s measures 1.1 tiles (equal
// prompts, 1 against 4 groups: 32 of 256 rows behind 2048 keys 268 and 261 us; 1 against 8: 64 of 512 rows 316 and 284 us).
// us, as for equal prompts -> this: 32 / 8 heads of 128, 16 prompts of 64 .. 1024 rows behind 512 keys 196 -> 144 and 200 -> 127 (two batches), 32 of 97
// .. 512 rows 98 -> 81 and 96 -> 71, 57 of 26 .. 239 behind 1696 278 -> 229, 64 of 30 .. 250 rows 60 -> 59 and 67 -> 68; 14 / 2 heads of 128, 82 of 12 ..
// 122 rows behind 3824 keys 242 -> 177; 8 / 2, 65 of 64 .. 227 behind 1616 90 -> 88 and 124 -> 88.  Of 8200 batches (1 to 100 prompts of up to 2048 rows, behind
// nothing or up to 4096 keys), which took 0.95 of the time on average, 80 were slower by more than 2 %, one by more than a sixth (where the
// former groups happen to fill the device: 16 / 8 heads of 128, 30 of 49 .. 392 rows behind 32 keys 32.6 -> 39.4).
// Prompts whose rows are 7 / 8 of the longest's or more on average, and calls that do not know (rows <= 0), keep `most`; so do pairs, which
// leave little to spread (16 / 8 heads of 64, 64 prompts of 30 .. 250 rows behind 512 keys: 69 us, one by one 70).
// Never so few that the longest prompt's `groups` need more than the 65535 workgroups a launch has along y.
PA_PLAN_FN int plan_ragged_groups(int most, int64_t groups, int num_kv_heads, int batch, int64_t rows, int64_t max_q_len, int64_t rows_per_group,
                                  int64_t max_keys, int tile_keys, int cus) {
    if (most <= 2 || rows <= 0 || 8 * rows >= 7 * max_q_len * batch) return most;
    const int64_t units = num_kv_heads * (rows / (rows_per_group > 0 ? rows_per_group : 1) + (batch + 1) / 2);  // (a last group is half full)
    const int64_t behind = max_keys > max_q_len ? max_keys - max_q_len : 0;          // keys before a prompt's own rows
    const int64_t c = (behind + max_q_len / 2) / tile_keys + 3;                      // tiles, and what a group costs beside its loop
    int g = 1;
    const double even = 1.1 * (double)units / ((double)c * cus * (1.0 - (double)rows / ((double)max_q_len * batch)));
    while (g < most && ((g + 1) * (g + 1) <= even || (groups + g - 1) / g > 65535)) ++g;
    return g;
}

// Which chunk of sequence `b` workgroup `y` of its n_chunks takes.  Workgroups go to the eight dies, and inside one to its shader engines, in turn, so
// with the same chunk for the same y and an even number of them the first chunks, which every sequence has, would meet on a few of those while
// the last ones, which only long sequences have, leave the rest idle.  The sum of b's digits to the base four moves them on.
// (us, one group a workgroup, 4 chunks: 32 / 8 heads of 64, 49 prompts of 24 .. 213 rows behind 624 keys 109 -> 69; 14 / 2 of 128, 82 of 12 .. 122 behind
// 3824 272 -> 177; 8 / 2 of 128, 65 of 64 .. 227 behind 1616 133 -> 88)
PA_PLAN_FN int plan_turned_chunk(int y, int b, int n_chunks) {
    return n_chunks & 1 ? y : (y + b + (b >> 2) + (b >> 4) + (b >> 6)) % n_chunks;
}

// The i-th group of the workgroup that is chunk `wg_chunk` of `n_chunks`: one of every n_chunks consecutive groups,
// counted from the front in even rounds and from the back in odd ones, so that under the causal mask (later groups
// see more keys) the workgroups' totals come out equal.  Strictly increasing in i; a workgroup stops at its first
// group past the sequence's last.
PA_PLAN_FN int plan_group_of(int i, int n_chunks, int wg_chunk) {
    return i * n_chunks + ((i & 1) ? n_chunks - 1 - wg_chunk : wg_chunk);
}

}  // namespace pa_decode_detail
