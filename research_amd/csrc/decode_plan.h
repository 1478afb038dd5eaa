// Bookkeeping of the split pass of paged decode attention: how the (plane, sequence, block) space is cut into
// workgroup ranges, which workgroup owns a block, where a range's partial result goes in the workspace and how
// the workspace is laid out.  Integer arithmetic only; shared by the kernels (decode_impl.h), the host entry
// point (decode.hip) and a plain C++ replay of both passes that the CPU tests compile with g++ (no HIP needed).
#pragma once
#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define PA_PLAN_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define PA_PLAN_FN inline
#endif

namespace pa_decode_detail {

constexpr int kPlanMaxBatch = 8192;      // sequences per call (their block prefix sum lives in LDS)
constexpr int kPlanMaxSplitGrid = 4096;  // upper bound of the split pass's grid, fixes the caller's workspace size
// Arrival tickets of the merge inside the split pass: 64-bit counters in a region of fixed size at the start of
// every workspace, so that calls of any shape use the same bytes for the same purpose and nothing else is ever
// written there: kPlanTicketSlots counters per (plane, sequence), then 2 per workgroup of the largest grid for the
// groups that the pieces of a many-piece sequence are merged in.  The caller zero-fills the region once; every call
// leaves it at zero.
constexpr int kPlanTicketSlots = 65536;
constexpr size_t kPlanGroupTicketOff = (size_t)kPlanTicketSlots * 8;
constexpr size_t kPlanTicketBytes = kPlanGroupTicketOff + 2 * (size_t)kPlanMaxSplitGrid * 8 + 64 * 1024;  // 640 KiB

// How the heads are spread over wave loads and planes (a plane = one group of hpw kv heads x one group of <= nrep_t
// query heads per kv head).  lpr lanes of 16 bytes hold one K/V row; a wave load covers rpw = 64/lpr rows, mapped
// to hpw neighbouring kv heads of tpw consecutive tokens.
struct HeadPlan {
    int hq, hkv, n_rep;
    int hpw, tpw, n_hgroups, n_rgroups;
    int nrep_t;  // padded group size (kernel template parameter); 0 = no kernel for this head_dim / element size
    int d_pad;   // head_dim rounded up to the next of 32, 64, 128, 256: the head size the kernel is compiled for
    PA_PLAN_FN int planes() const { return n_hgroups * n_rgroups; }
    PA_PLAN_FN int heads_per_slot() const { return hpw * nrep_t; }
};

// The kernels are compiled for head sizes 32, 64, 128 and 256; any other head_dim up to 256 whose rows are whole
// 16-byte vectors runs the next larger one with the lanes past the row's end idle.
PA_PLAN_FN int plan_pad_dim(int head_dim) { return head_dim <= 32 ? 32 : head_dim <= 64 ? 64 : head_dim <= 128 ? 128 : 256; }

PA_PLAN_FN HeadPlan plan_heads(int num_q_heads, int num_kv_heads, int head_dim_real, int kv_elem_bytes) {
    HeadPlan h = {};
    if (kv_elem_bytes <= 0 || head_dim_real <= 0 || head_dim_real > 256 || head_dim_real * kv_elem_bytes % 16 != 0 ||
        head_dim_real % 8 != 0)
        return h;
    if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads != 0) return h;
    const int head_dim = plan_pad_dim(head_dim_real);
    h.d_pad = head_dim;
    const int lpr = head_dim * kv_elem_bytes / 16;  // lanes per K/V row
    const int rpw = 64 / lpr;                        // rows per wave load
    int hpw = 1;                                     // kv heads per wave load: power of two dividing num_kv_heads
    while (hpw * 2 <= rpw && num_kv_heads % (hpw * 2) == 0) hpw *= 2;
    const int n_rep = num_q_heads / num_kv_heads;
    int nrep_t = 1;
    while (nrep_t < n_rep && nrep_t < 8) nrep_t *= 2;
    h.hq = num_q_heads;
    h.hkv = num_kv_heads;
    h.n_rep = n_rep;
    h.hpw = hpw;
    h.tpw = rpw / hpw;
    h.n_hgroups = num_kv_heads / hpw;
    h.n_rgroups = (n_rep + nrep_t - 1) / nrep_t;
    h.nrep_t = nrep_t;
    return h;
}

// First key that the query at position len-1 sees.  window > 0: a sliding window, keys j >= len - window; window < 0:
// chunks of -window positions counted from the sequence's start, keys of the query's own chunk; 0: all keys.
PA_PLAN_FN int plan_first_key(int len, int window) {
    if (window > 0) return len > window ? len - window : 0;
    return window < 0 && len > 0 ? (len - 1) - (len - 1) % -window : 0;
}
// Keys that a window or chunk lets a query see at most (0: no bound).
PA_PLAN_FN int64_t plan_window_span(int window) { return window < 0 ? -(int64_t)window : window; }
// Blocks of a sequence of `len` keys that hold visible keys: [first_key / bs, ceil(len / bs)).
PA_PLAN_FN int plan_blocks_of(int len, int block_size, int window) {
    if (len <= 0) return 0;
    return (len + block_size - 1) / block_size - plan_first_key(len, window) / block_size;
}

// Workgroup w of a grid of G owns the flattened units [floor(w*T/G), floor((w+1)*T/G)) of T.
PA_PLAN_FN int64_t plan_unit_begin(int64_t w, int64_t total, int64_t grid) { return w * total / grid; }
PA_PLAN_FN int plan_owner_of(int64_t u, int64_t total, int64_t grid) { return (int)(((u + 1) * grid - 1) / total); }

// Short launches are flattened in runs of u blocks of one (plane, sequence) instead of single blocks, with a workgroup per
// run: what a workgroup spends is a chain of waits per sequence that it touches (5 to 10 us), hardly more for one block of
// it than for eight, so a range that crosses from one sequence into the next takes twice as long.  Returns u: the smallest of
// 1, 2, 4 with which the runs fit the grid, 4 where (plane, sequence) pairs have many blocks (hundreds of one-block partials
// of a pair would take longer to merge than they save); else 1, and the ranges of plan_unit_begin.  units(u): the runs of u
// blocks of the launch.  Ranges of at least four blocks took 20.7 us for 4 sequences of 100 keys at 32 / 8 heads of 128, runs
// take 13.9; 31 -> 14 us for 256 sequences of 16 keys; at 14 / 2 heads of 64, 4 sequences of 16 keys 52.6 -> 13.7, 16 of 1000
// keys 31 -> 17, 4 of 6000 keys 33 -> 20.  (Single blocks for one sequence of 6000 keys: 20 us at 8 / 2 heads of 128, runs of
// four 15; hence the line at 48 blocks per pair.)  Above kPlanWaveScanBatch sequences, where the table of units comes from one scan,
// single blocks and the whole grid: 600 sequences of up to 16 keys 39 -> 31 us at 32 / 8 heads of 128, 54 -> 24 at 14 / 2 of 64; 900 of up to
// 24 keys 55 -> 54 at 32 / 8.
constexpr int kPlanWaveScanBatch = 512;
constexpr int kPlanRunMost = 4, kPlanShortBlocks = 48;
template <typename F> PA_PLAN_FN int plan_run_blocks(int64_t total, int64_t keys, int grid, F units) {
    if (total > (int64_t)kPlanRunMost * grid) return 1;
    for (int u = total > keys * kPlanShortBlocks ? kPlanRunMost : 1; u <= kPlanRunMost; u *= 2)
        if ((u == 1 ? total : units(u)) <= grid) return u;
    return 1;
}
PA_PLAN_FN int plan_runs_of(int blocks, int u) { return (blocks + u - 1) / u; }
// The same where every wave fills the prefix table by itself, without a barrier: scan(u, keep) returns the runs of u blocks of all
// sequences and, with `keep`, stores the table.  Only the final table is ever stored: waves that lag behind store what the others read.
template <typename F> PA_PLAN_FN int plan_wave_prefix(int planes, int batch, int grid, int &run, F scan) {
    run = plan_run_blocks((int64_t)scan(1, false) * planes, (int64_t)planes * batch, grid,
                          [&](int u) { return (int64_t)scan(u, false) * planes; });
    return scan(run, true);
}
// Workgroups that take part in a launch of `total` runs.
PA_PLAN_FN int plan_run_grid(int64_t total, int grid) { return total < grid ? (int)total : grid; }

// Partial slot of the piece of (plane, sequence) that workgroup w computed: unique, because along the flattened
// order both w and plane*batch + sequence only grow.
PA_PLAN_FN int64_t plan_slot(int w, int plane, int batch, int b) { return (int64_t)w + (int64_t)plane * batch + b; }

// How the pieces of one (plane, sequence) are merged inside the split pass.  Up to kPlanInlinePieces pieces: the
// workgroup that delivers the last of them merges them all.  More (one sequence that dominates its batch is cut
// into hundreds): the pieces form groups of `group` consecutive workgroups, the last arrival of a group merges the
// group into the slot of the group's first piece, and the last group to finish merges the groups - two levels of
// at most 32 partials each instead of one workgroup reading hundreds.
constexpr int kPlanInlinePieces = 8;
struct PieceTree {
    int pieces, group, n_groups;
};
PA_PLAN_FN PieceTree plan_piece_tree(int pieces) {
    PieceTree t;
    t.pieces = pieces;
    t.group = pieces <= kPlanInlinePieces ? pieces : pieces <= 64 ? 8 : pieces <= 256 ? 16 : 32;
    t.n_groups = (pieces + t.group - 1) / t.group;
    return t;
}
// A group's ticket is found by the workgroup of its first piece; a workgroup can be that for the sequence that runs on into
// it (a later group of it) and for the sequence that starts in it (group 0 of it).
PA_PLAN_FN int64_t plan_group_ticket(int first, int group) { return 2 * (int64_t)first + (group == 0 ? 1 : 0); }

// workspace = [tickets uint64[kPlanTicketSlots]] [block_prefix int32[batch+1]] [part_ml float[slots][heads][2]]
//             [part_acc float[slots][heads][D]], heads = hpw*nrep_t query heads of one plane,
// slots = grid_cap + planes*batch (slot indices stay below grid + planes*batch - 1).
struct WsPlan {
    size_t prefix_off, ticket_off, ml_off, acc_off, total;
    int64_t slots;
};
PA_PLAN_FN size_t plan_align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }
PA_PLAN_FN WsPlan plan_workspace(int batch, const HeadPlan &h, int head_dim, int grid_cap) {
    WsPlan w;
    const size_t heads = (size_t)h.heads_per_slot();
    const size_t keys = (size_t)h.planes() * (size_t)batch;
    w.slots = (int64_t)grid_cap + (int64_t)keys;
    w.ticket_off = 0;
    w.prefix_off = kPlanTicketBytes;
    w.ml_off = w.prefix_off + plan_align_up((size_t)(batch + 1) * 4, 256);
    w.acc_off = w.ml_off + plan_align_up((size_t)w.slots * heads * 2 * 4, 256);
    w.total = w.acc_off + plan_align_up((size_t)w.slots * heads * (size_t)head_dim * 4, 256);
    return w;
}

// LDS of the merge of a workgroup's row-group partials (decode_impl.h: merge_rows): rows = 4 waves x rows per wave
// load, each D + 2 floats plus 3 floats of weights; as many query heads per round (8, 4, 2 or 1 of the nrep_t) as
// 28 KB hold.
constexpr int kPlanThreads = 256;
constexpr int kPlanMergeBudget = 28 * 1024;
PA_PLAN_FN constexpr int plan_merge_rows(int head_dim, int kv_elem_bytes) { return 4 * (64 / (head_dim * kv_elem_bytes / 16)); }
PA_PLAN_FN constexpr int plan_merge_heads_per_round(int head_dim, int kv_elem_bytes, int nrep_t) {
    const int per_head = plan_merge_rows(head_dim, kv_elem_bytes) * (head_dim + 2 + 3) * 4;
    return nrep_t >= 8 && 8 * per_head <= kPlanMergeBudget   ? 8
           : nrep_t >= 4 && 4 * per_head <= kPlanMergeBudget ? 4
           : nrep_t >= 2 && 2 * per_head <= kPlanMergeBudget ? 2
                                                             : 1;
}
PA_PLAN_FN constexpr int plan_merge_floats(int head_dim, int kv_elem_bytes, int nrep_t) {
    return plan_merge_heads_per_round(head_dim, kv_elem_bytes, nrep_t) * plan_merge_rows(head_dim, kv_elem_bytes) *
           (head_dim + 2 + 3);
}
// LDS of one workgroup of the split pass: the block prefix sums (dynamic), the scan scratch, the merge area, a flag.
PA_PLAN_FN constexpr size_t plan_split_lds_bytes(int batch, int head_dim, int kv_elem_bytes, int nrep_t) {
    return (size_t)(batch + 1) * 4 + kPlanThreads * 4 + (size_t)plan_merge_floats(head_dim, kv_elem_bytes, nrep_t) * 4 + 4;
}

// Whether the split pass merges the pieces of a sequence itself (the workgroup that delivers the last outstanding
// piece of a sequence, or of a group of its pieces, merges) instead of leaving them to a second launch: when the
// batch is so large that a (plane, sequence) has two pieces on average at most.  Measured on MI355X: 256 sequences
// (two pieces each) gain 1 % over the two launches; 64 sequences (four pieces each) lose 2 % - delivering a piece
// costs round trips to the memory side, about 9 us at the end of a 100 us launch where the second launch costs 7 -
// and a few long sequences spread over the whole grid are merged much faster by the second launch, whose
// workgroups take one output row each.
PA_PLAN_FN bool plan_merge_in_split(int batch, const HeadPlan &h, int grid) {
    const int64_t keys = (int64_t)h.planes() * batch;  // one ticket each
    return (int64_t)grid <= 2 * keys && keys <= kPlanTicketSlots;
}

// How decode_short.h's kernel takes the launch: 0: not at all; else the runs a sequence's tiles are cut into, a workgroup per (kv head, sequence,
// run).  From shapes alone; the tables' width stands for the longest sequence.
// Head sizes up to 32 over 16 bits and fp8 stay with the generic loop of the split pass, whose weights have 32 bits: 11.8 us for 16 sequences of 16 .. 250 keys, 4 / 4
// heads of 32, where weights of two bf16 terms took 5.0, but erred by up to 1.1e-6 of the sum of |weight value| where 32 bits err by 0.2e-6.
// Runs: one for each compute unit, of at least 128 keys, where the longest sequence takes longer than a merging launch: from 600 keys of 128 on over 16 bits and fp8 (measured with a merge
// of 3.5 us), from 256 on over 32 bits (with the present one, 2.5 us).
// us, the split pass (one launch or two) -> this, sequences of n keys each: 32 / 8 heads of 128, 1 of 256 keys 14.1 -> 7.4, 1024 15.5 -> 9.0, 4096
// 16.2 -> 12.0; 32 of 256 19.6 -> 8.3; 96 of 256 33.9 -> 19.7; 14 / 2 of 64, 1 of 256 15.2 -> 5.8, 4096 16.4 -> 11.0; 32 of 1024 22.1 -> 11.0, 16384
// 64 -> 51; 192 of 1024 45 -> 21; fp8 32 / 8 of 128, 32 of 256 24.5 -> 6.8; fp8 14 / 2 of 256, 16 of 2048 47 -> 14.5, 256 of 2048 185 -> 91.
// Where the split pass stays: its ranges are equal whatever the lengths, so that unequal sequences in long runs are faster there once memory
// counts.  More than four query heads a kv head hold up its vector unit, so the line lies further out, for fp8 furthest (unequal, keys n / 8 .. n,
// the split pass -> runs of that length: 32 / 4 heads of 128, 32 of 8192 65 -> 76, 96 of 2048 57 -> 61, equal ones 70 -> 66); the less so the more kv
// heads of 64 a wave of that pass takes at once (unequal: 14 / 2 of 64, 49 of 10359, runs of 432 KB, 45 -> 49, 141 of 3004, of 376 KB, 45 -> 41; 28 /
// 4, 25 of 11157, of 465 KB, 45 -> 50; 64 / 8, 34 of 3981, of 498 KB, 54 -> 72).  32 / 8 of 128, unequal: 16 of 2048 22.4 -> 24.2, 48 of 2048
// 44.8 -> 47.4, 1024 33 -> 27; equal, 256 of 512 90 -> 94.  One or two query heads a kv head: 16 / 8 of 256, 16 of 1024 19.5 -> 24; 8 / 8 of 64, 3 of
// 8192 18 -> 24; over fp8, where the kernel's conversions count, 8 / 8 of 64, 3 of 8064 in runs of 806 keys 12.7 -> 15.0, 32 / 16, 66 of 917 38 -> 51.
// 8 / 2 of 128, 1 of 8192 14.6 -> 15.2, 4096 14 -> 12.
// The lines that depend on the merge, whose loads are all on their way at once, were measured with it: above 64 elements a row, from five query heads a kv head on, runs of
// 16-bit pools up to 416 KB (16 / 2 of 128, 5 of 6169 keys 50 -> 41, 106 of 1351 38 -> 25; beyond, unequal, 4 of 113400 61 -> 70) and of more than 512
// keys of 128 cut in two where the units have room for it (fp8 16 / 2 of 128, 17 of 12251 29 -> 20, 5 of 57391 36 -> 26; of 256 not: 38 of 4315 35 -> 38); over
// fp8 up to four heads more in all, of 256 longer ones too (32 / 8 of 128, 93 of 763 41 -> 25, of 256, 68 of 565 43 -> 21; 16 / 8 of 256, 1 of 8756 25 ->
// 15; but 32 / 8 of 128, 66 of 2214 65 -> 70).  From three heads of 64 on, runs begin at 800 keys while they are few (32 / 8, 3 of 1040 10.8 -> 7.9).
// (Over 321 batches over 16 bits and 216 over fp8, such lengths, 0.90 and 0.85 of the time before these lines, the slowest 1.04.)
// 32-bit pools, the split pass -> this: from five query heads a kv head on wherever a run of the longest sequence, which all others may have to wait for, is short enough; the split pass spends a vector
// instruction on every head, key and element, but divides any batch equally (14 / 2 of 72, 105 of 34 .. 127 keys 26.7 -> 8.1, 16 / 2 of 128, 102 of 236 51 -> 24).  Runs of 192 KB at up to 64
// elements a row (14 / 2 of 64, 64 of 30000 and 1500 48 -> 179 in runs of 940 KB, 8 of 22400 and 1120 23 -> 34 of 350, equal steps 32 -> 29; 16 of 8000 23 -> 19 of 125), of 384 where sequences
// are so few that each has 32 runs (1 of 40000 26 -> 20, 81920 35 -> 33, 130000 42 -> 47) or there are two workgroups for every four units without runs (200 of 4000 122 -> 51); above 64 416
// (5 / 1 of 128, 1 of 60000, runs of 470 KB, 34 -> 37; 40 / 8 of 128, 4 of 5600, 350, 44 -> 30) and 832 (40 / 8 of 128, 100 of 1000 155 -> 80, 14 / 2 of 256, 250 of 1000 274 -> 126).
// Three or four: up to 48 MB of keys, in runs of 176 KB (32 / 8 of 64, 4 of 155 14.5 -> 8.2, 8 / 2 of 128, 29 of 819 20 -> 17; beyond, runs of 200 KB, 32 / 8 of 256,
// 3 of 2000 23 -> 27, of 64, 3 of 8000 24 -> 24, one of 8000 among 400 20 -> 23; unequal, of 128, 7 of 33764 160 -> 340), unless more than four rounds of workgroups have few keys each (32 / 8 of 64, 206 of 53 13.4 -> 15.0; at 256 more than one, 8 / 2, 163 of 138 21 -> 26) or the few there are
// have long runs (8 / 2 of 128, 2 of 4000 15.6 -> 18.1, of 64, 8 of 6831 16.5 -> 18.2; of 256, 2 of 1964 17.6 -> 18.6).  One or two: a run each, up to 32 MB
// and two rounds (16 / 8 of 128, 1 of 176 12.5 -> 8.6, 28 of 94 15.0 -> 8.9; 187 of 21 13.4 -> 18.1, 8 / 8 of 64, 16 of 600 14.5 -> 15.2).  A run is cut where four
// turns of the waves, at 256 two, take longer than a merging launch: 16 keys of 128 each in 1 us (14 / 2 of 256, 6 of 228 in one run 20.7, of 64 keys 16.4, of
// 32 11.9; 14 / 2 of 128, 16 of 101 8.2, in three 9.4); where most units have a workgroup anyway into two runs a unit, from five heads on four (unequal:
// 14 / 2 of 72, 140 of 1600 71 -> 78, with four 50; equal 116 -> 100, 77).
// (Over 3053 batches over 32-bit pools, from five heads on, lengths in equal steps, drawn ones, one long one among others of a twentieth: 0.68, 0.73 and 0.77 of the split pass's time;
// 76 were slower by more than 2 %, by up to 1.4: 5 / 1 of 128, one of 8000 among 199 of 400 46 -> 64.)
// (Over 1200 shapes of 1 .. 128 sequences that this takes, from 600 keys of 128 on, equal and unequal, 16 of 3600 batches were slower by more than 2 %, of which 4 / 4 heads of 96
// over fp8 by up to 19, 30 of 1482 keys 15.6 -> 18.6, the others by up to 6; on average they took 0.55 of the split pass's time.)
constexpr int kPlanShortHeads = 16, kPlanShortTile = 16, kPlanShortRuns = 64;
PA_PLAN_FN int plan_short_splits(int batch, const HeadPlan &h, const WsPlan &w, int kv_elem_bytes, int64_t table_blocks, int block_size, int window, int cus) {
    if (block_size % kPlanShortTile != 0 || batch > kPlanWaveScanBatch || h.hkv > 65535 || (h.d_pad < 64 && kv_elem_bytes < 4)) return 0;
    const int64_t span = plan_window_span(window);
    if (span > 0 && span / block_size + 2 < table_blocks) table_blocks = span / block_size + 2;
    const int64_t keys = table_blocks * block_size, reps = (h.n_rep + kPlanShortHeads - 1) / kPlanShortHeads, wgs = (int64_t)h.hkv * batch * reps;
    int64_t runs = 1;
    const bool f32 = kv_elem_bytes == 4;
    const int64_t d = h.d_pad < 64 ? 64 : h.d_pad, least = f32 ? 64 * 128 / d : 128;  // (least: keys of a run)
    const bool brief = keys * d <= (f32 ? 256 : h.n_rep > 2 && d == 64 && 4 * wgs <= cus ? 400 : 600) * 128;
    if (!brief) {
        runs = 4 * wgs <= cus ? cus / wgs : (!f32 ? 3 : h.n_rep > 4 ? 8 : 4) * (int64_t)cus / 2 / wgs;  // (few more workgroups than units are as slow as twice as many)
        const int64_t each = keys / (runs < 1 ? 1 : runs) * d;
        if (!f32 && h.n_rep > 4 && !(kv_elem_bytes == 1 && d == 256) && wgs <= cus && each > (runs > 1 ? 512 : 1024) * 128) runs = 2 * (runs < 1 ? 1 : runs);
        if (runs > keys / least) runs = keys / least;
        if (runs > kPlanShortRuns) runs = kPlanShortRuns;
        const int64_t room = w.slots * h.heads_per_slot() / ((int64_t)batch * h.hq);  // (their results are as long as a slot's)
        if (runs > room) runs = room;
        if (runs < 1) runs = 1;
    }
    const int64_t row = d * kv_elem_bytes, kb = 1024;
    const int64_t wide_most = row > 128 && kv_elem_bytes == 2 ? 416 * kb : row > 128 || h.hpw == 4 ? 256 * kb : h.hpw == 1 ? 512 * kb : h.hpw == 2 ? 384 * kb : 208 * kb;
    const bool wide8 = kv_elem_bytes == 1 && d > 64;
    const int64_t run_most = h.n_rep > 4 ? (kv_elem_bytes == 1 ? 4096 * row : wide_most) : (h.n_rep > 2 ? (wide8 && d > 128 ? 384 : 128) : wide8 ? 128 : 64) * kb;
    const int64_t all_most = h.n_rep > 4 ? (int64_t)1 << 62 : (h.n_rep > 2 ? (wide8 ? (d > 128 ? 200 : 100) : 64 * kv_elem_bytes) : wide8 ? 48 : 32 * kv_elem_bytes) * kb * kb;
    const bool few = h.n_rep <= 4 && wgs < 6 && keys > 4096 && !wide8;
    if (f32) {
        const bool lone = keys > 3072 ? wgs < (d == 64 ? 24 : 6) : d == 256 && !brief && wgs < 8;
        const bool full = 2 * wgs >= cus, spread = 32 * wgs <= cus && h.d_pad >= 64;
        const int64_t most = (d > 64 ? (full ? 832 : 416) : full || spread ? 384 : 192) * kb;
        const bool fits = h.n_rep > 4   ? keys / runs * row <= most
                          : h.n_rep > 2 ? !lone && wgs <= (d == 256 ? 1 : 4) * (int64_t)cus && wgs * keys * row <= 48 * kb * kb && keys / runs * row <= 176 * kb
                                        : d < 256 && brief && wgs <= 2 * (int64_t)cus && wgs * keys * row <= 32 * kb * kb;
        return fits && runs * reps <= 65535 ? (int)runs : 0;
    }
    const bool thin = kv_elem_bytes == 1 && h.d_pad == 64 && h.n_rep <= 2 && keys / runs > 768;
    const bool fits = (brief || keys / runs * row <= run_most) && wgs * keys * row <= all_most && !few && !thin;
    return fits && runs * reps <= 65535 ? (int)runs : 0;
}

// Of what the split pass still has (the larger calls over 32-bit pools, heads of up to 32, blocks that are no whole tiles, large batches of 16-bit ones): whether the
// block tables are so narrow that a workgroup takes a whole (plane, sequence): nothing is left to merge then, and the second launch (4 us, and its
// gap) goes.  A workgroup is a chain of waits, 1 to 2 us for each block that a wave takes (for a tile of 16 keys of longer ones), 2 to 4 us where
// eight query heads a kv head meet fp8 values or the generic loop, so the line lies where the chain takes as long as the second launch and what
// the ranges, which grow with the batch, take longer: 16 blocks, 32 from 16 workgroups on, half of it for those loops, 12 for the generic loop over 16
// bits, and 192 KB of keys and values (32-bit pools, whose loop has fewer loads in flight, 128 KB).  Large batches, whose ranges would cross from one
// sequence into the next, gain up to 64 blocks (the generic loop over 16 bits 32) and 384 KB, beyond 1024 workgroups 192 KB.
// us, ranges -> whole sequences.  bf16, blocks of 8: 14 / 2 heads of 64, 4 sequences of 64 keys 15.8 -> 12.0, of 384 keys 16.2 -> 19.7, 16 of 256
// keys 18.6 -> 16.7, 200 of 256 34 -> 19; 32 / 8 of 128, 4 of 96 keys 13.9 -> 12.2, 64 of 96 18.8 -> 12.5, 200 of 192 47 -> 34; blocks of 4, 14 / 2 of 64,
// 4 of 256 keys 16.1 -> 34, 200 of 64 32 -> 18; blocks of 1, 4 of 64 keys 16.2 -> 32, 200 of 64 40 -> 35, of 256 79 -> 109.  fp8, blocks of 8: 16 / 8 of 128,
// 4 of 96 keys 13.4 -> 12.5, 200 of 96 29 -> 17; 14 / 2 of 256, 4 of 128 keys 22 -> 24, 64 of 128 45 -> 25.  32-bit: 8 / 2 of 128, 16 of 64 keys
// 15.6 -> 11.5, 512 of 192 45 -> 42; 14 / 2 of 64, 4 of 128 keys 16.2 -> 14.9, in blocks of 8 16.3 -> 20.3.  bf16, heads of 32: 8 / 2, 4 of 128 keys
// 16.0 -> 13.7, of 512 16.4 -> 27, 200 of 512 40 -> 32; 4 / 4, 64 of 384 keys 14.9 -> 16.4.  bf16, 500 sequences: 32 / 8 of 128, of 192 keys 89 -> 77;
// 16 / 8 of 256, of 96 keys 85 -> 94.  (Batches whose equal sequences fit the ranges without a rest lose up to a tenth: 512 of 192 keys, 32 / 8 of 128, 74
// -> 78; unequal ones, of n / 8 .. n keys, gain more than equal ones throughout: 74 -> 61.)
constexpr int kPlanWholeBytes = 192 * 1024;
PA_PLAN_FN bool plan_whole_sequences(int batch, const HeadPlan &h, int head_dim, int kv_elem_bytes, int64_t table_blocks, int block_size, int window) {
    if (batch > kPlanWaveScanBatch) return false;
    const int64_t span = plan_window_span(window), units = (int64_t)h.planes() * batch;
    if (span > 0 && span / block_size + 2 < table_blocks) table_blocks = span / block_size + 2;
    const bool f32 = kv_elem_bytes == 4, many = batch >= 96 && units >= (f32 ? 512 : 192);
    const bool slow = h.d_pad == 32 && !f32, heavy = h.nrep_t == 8 && (kv_elem_bytes != 2 || slow);
    int steps = many ? 64 : (units < 16 ? 16 : 32) / (heavy ? 2 : 1);
    if (slow && steps > (many ? 32 : 12)) steps = many ? 32 : 12;
    const int64_t most = (f32 ? kPlanWholeBytes * 2 / 3 : kPlanWholeBytes) * (many && units <= 1024 ? f32 ? 3 : 2 : 1);
    return units <= 65535 && table_blocks <= steps / ((block_size + 15) / 16) &&
           table_blocks <= most / ((int64_t)block_size * h.hpw * head_dim * kv_elem_bytes * 2);
}

}  // namespace pa_decode_detail
