// Host-testable arithmetic of the linear-recurrence kernels: padded state sizes, value slices and the segments a long
// portion is cut into.  Plain C++.
#pragma once
#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define PA_LA_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define PA_LA_FN static inline
#endif

constexpr int kLaChunk = 64;      // rows multiplied at once
constexpr int kLaMinSegChunks = 8;    // a segment is at least this many chunks long ...
constexpr int kLaMaxSegments = 64;
constexpr int kLaLeastSegChunks = 2;  // ... or, of few sequences, this many
// Segments whose states the scan between the passes loads at once (8 prompts in three segments, 16 heads of 128 x 128, all passes: 2 137.4 us, 4
// 137.9, 8 139.0; one of 12000 rows in 32, 8 heads: 70.5, 69.5, 69.0).
constexpr int kLaScanAhead = 4;

static inline int la_pad16(int n) { return (n + 15) / 16 * 16; }

// Columns of the value dimension that one workgroup of the chunked kernel owns: 16 for each of its four or eight waves.
static inline int la_value_cols(int vdim) { return vdim <= 64 ? 64 : 128; }
// Workgroups of a sequence (of each of its segments): one per head and slice of the value columns.
static inline int64_t la_per_sequence(int heads, int vdim) { return heads * (int64_t)((vdim + la_value_cols(vdim) - 1) / la_value_cols(vdim)); }

// Segments of a portion of up to max_len rows: as many as (sequences x heads x value slices) leave compute units for,
// one workgroup each, but no shorter than kLaMinSegChunks chunks (a segment's start state costs a second reading of
// its keys and values and two passes over a state's bytes).
static inline int la_segments(int64_t workgroups, int cus, int max_len, int least = kLaMinSegChunks) {
    if (workgroups <= 0 || max_len <= 0) return 1;
    const int64_t chunks = (max_len + kLaChunk - 1) / kLaChunk;
    int64_t want = cus / workgroups;
    const int64_t most = chunks / least;
    if (want > most) want = most;
    if (want > kLaMaxSegments) want = kLaMaxSegments;
    return want < 1 ? 1 : (int)want;
}

// The same for a batch whose rows are known: `per_seq` workgroups for each sequence, n_rows rows in all; together: by how much
// a workgroup is slower when two share a compute unit (0: they cannot).  In units of a chunk of the second pass: without
// segments the launch lasts as long as its longest sequence or, with more workgroups than compute units, its share of the
// rows; with segments of c chunks it lasts c where a compute unit has one of them at most (of unequal portions' last segments, which
// are short and start last, half may follow another, up to an eighth of the units), c `together` where some have two, else its share
// and a third of a segment (which of one sequence, in equal segments, has to promise 5 % more), and 45 % more for the first pass, a fifth of a unit per segment for the scan between
// the two, and three units for the launches.  Segments shorter than kLaMinSegChunks only where a compute unit has one at most: what each begins
// and ends with counts (16 heads of 128 x 128, SSD, 5 prompts of 1611 .. 2178 rows, 96 us in three, 108 in eight).
// Before, no segment was shorter than eight chunks, and a segment of the scan half a unit: us, that -> this, one sequence: lightning, 8 heads of
// 128 x 128, 4000 rows 74 -> 42, 12000 84 -> 70; HGRN2, 8 heads of 128 x 128, 2500 rows 114 -> 50; mLSTM, 4 heads of 256 x 512, 700 rows 101 -> 56;
// of 64 x 128, 12000 81 -> 61; SSD, 64 heads of 128 x 64, 1500 rows 65 -> 55.  Over 250 batches (1 to 40 prompts of 200 .. 16000 rows, 1 to 64 heads,
// four recurrences)
// 1.06 to 1.27 times as fast on average, none slower by more than 2 %.
static inline int la_balanced_segments(int64_t batch, int64_t per_seq, int cus, double together, int max_len, int64_t n_rows, int most) {
    if (batch <= 0 || per_seq <= 0 || max_len <= 0) return 1;
    if (n_rows > batch * max_len) n_rows = batch * max_len;
    const int chunks = (max_len + kLaChunk - 1) / kLaChunk;
    const double rows = (double)n_rows / kLaChunk, share = rows * per_seq / cus * (together > 0 ? together / 2 : 1.0);
    const double most_spare = 0.12 * cus, spare = 0.25 * batch * per_seq < most_spare ? 0.25 * batch * per_seq : most_spare;
    double best = share > chunks ? share : chunks;
    int segments = 1;
    for (int s = 2; s <= most; ++s) {
        const double c = (chunks + s - 1) / s;
        const double spread = rows / c + 0.5 * batch, all = (double)batch * s, live = per_seq * (spread < all ? spread : all);
        double part = c;
        const bool more = live > cus + (spread < all ? spare : 0.0);
        if (more && s > chunks / kLaMinSegChunks) continue;  // (short ones, several a unit: what each begins and ends with counts)
        if (more) part = live <= 2.0 * cus && together > 0 ? c * together : share + 0.35 * c;
        if (part < c) part = c;
        const double t = (1.45 * part + 0.2 * s + 3.0) * (more && batch == 1 ? 1.05 : 1.0);
        if (t < best) {
            best = t;
            segments = s;
        }
    }
    return segments;
}
// Chunks of a segment at least: fewer where the sequences in one piece leave compute units without a workgroup.
static inline int la_least_chunks(int64_t batch, int64_t per_seq, int cus) { return batch * per_seq < cus ? kLaLeastSegChunks : kLaMinSegChunks; }
// Most segments: none shorter than `least` chunks, and states of seg_bytes for each (of all sequences) that fit `room`.
constexpr size_t kLaMostSegBytes = (size_t)256 << 20;
static inline int la_most_segments(size_t seg_bytes, int max_len, size_t room = kLaMostSegBytes, int least = kLaMinSegChunks) {
    const int most = la_segments(1, kLaMaxSegments, max_len, least);
    if (room > kLaMostSegBytes) room = kLaMostSegBytes;
    const int64_t fit = seg_bytes ? (int64_t)(room / seg_bytes) : most;
    return fit < 1 ? 1 : fit < most ? (int)fit : most;
}
// Segments whose states a launch of n_rows rows has a use for (< 0: the rows are not known yet; the most of any): 1 where the batch stays
// in one piece, such as equal portions that fill the device.
static inline int la_asked_segments(int64_t batch, int64_t per_seq, int cus, double together, int max_len, int64_t n_rows, size_t seg_bytes) {
    const int most = la_most_segments(seg_bytes, max_len, kLaMostSegBytes, la_least_chunks(batch, per_seq, cus));
    if (n_rows >= 0) return la_balanced_segments(batch, per_seq, cus, together, max_len, n_rows, most);
    int asked = 1;
    for (int i = 0; i <= 32; ++i) {  // from one long portion to equal ones
        const int s = la_balanced_segments(batch, per_seq, cus, together, max_len, max_len + (batch - 1) * max_len * i / 32, most);
        if (s > asked) asked = s;
    }
    return asked;
}
// Segments of a launch with a workspace of `room` bytes (0: none).  0: they would need the workspace, which is not aligned; a
// batch that fills the device without segments takes such a workspace for none.  shared: workgroups that a compute unit has at once.
static inline int la_launch_segments(int64_t batch, int64_t per_seq, int cus, double together, int max_len, int64_t n_rows,
                                     size_t seg_bytes, size_t room, bool aligned, int shared = 1) {
    const int most = la_most_segments(seg_bytes, max_len, room, la_least_chunks(batch, per_seq, cus));
    if (!aligned) return la_most_segments(seg_bytes, max_len, room) > 1 && la_segments(batch * per_seq, shared * cus, max_len) > 1 ? 0 : 1;
    return la_balanced_segments(batch, per_seq, cus, together, max_len, n_rows, most);
}

// Whether the delta rule's walk over `workgroups` workgroups goes to pairs of waves, of whose workgroups a compute unit has one at dim 128, or to single
// waves, of which it has `walks` for each of the others (four: of four waves, which then share their SIMDs).  A pair is faster through a chunk.  So it
// decides where no compute unit gets a second workgroup, where two of either fit or one, and where a long chain is waited for: behind unequal prompts,
// whose chunks in all keep the device busy for less than the longest one's, and above 16 chunks.  Else two walks at once need less than two pairs one
// after the other; an odd number of pairs' rounds is half a round more for walks of two waves, which pays up to two chunks.  us, walks / pairs: 4
// heads of 128 x 32, 100 prompts of 40 .. 64 rows (1.6 rounds) 20.7 / 23.4; 8 of 128 x 64, 18 of 100 .. 128 (1.1) 22.2 / 25.3; 16 of 128 x 64, 9 of
// 1000 .. 1024 (1.1) 89 / 100; 32 of 64 x 64, 20 of 120 .. 192 (2.5) 48.6 / 53.4; but 8 of 128 x 128, 9 of 30 .. 400 (1.1) 28.4 / 23.8; 16 of 128 x 128, 5
// of 64 .. 1500 (1.2) 78 / 63; 4 of 128 x 32, 160 of 500 .. 512 (2.5) 168 / 152.  Over 325 batches of one to 63 chunks the rule's choice takes 1.004 of the
// better one's time, no batch more than with pairs alone, which take 1.024 and 1.17 at most.
static inline bool la_delta_pairs(int64_t workgroups, int walks, bool four, int64_t batch, int chunks, int64_t n_rows, int cus) {
    if (walks < 2) return true;
    if (four && chunks == 1) return false;
    if (workgroups <= cus || chunks > 16) return true;
    if (chunks <= 2) return false;
    int64_t all = n_rows / kLaChunk + batch / 2;  // chunks, about
    if (all > batch * chunks) all = batch * chunks;
    return workgroups * all <= batch * cus * chunks || (!four && (workgroups + cus - 1) / cus % 2 != 0);
}

// Segments of seg_rows rows before a portion's last one.  (Rows past the longest length that a launch was told have no segment.)
PA_LA_FN int la_full_segments(int rows, int segments, int seg_rows) {
    const int full = rows > 0 ? (rows - 1) / seg_rows : 0;
    return full < segments ? full : segments - 1;
}

// Rows per segment: whole chunks.
static inline int la_segment_rows(int max_len, int segments) {
    const int chunks = (max_len + kLaChunk - 1) / kLaChunk;
    return (chunks + segments - 1) / segments * kLaChunk;
}

static inline size_t la_state_floats(int dim, int vdim) { return (size_t)la_pad16(dim) * la_pad16(vdim); }
static inline size_t la_workspace_bytes(int64_t batch, int heads, int dim, int vdim, int segments) {
    return segments <= 1 ? 0 : (size_t)batch * heads * segments * la_state_floats(dim, vdim) * sizeof(float);
}

// Gated recurrences: a head's floats in the pool (with a normaliser: S, and n and the running maximum once per 64 value
// columns) and the segments' states (S, n, and three scalars).
static inline size_t gl_state_floats(bool normaliser, int dim, int vdim) {
    return la_state_floats(dim, vdim) + (normaliser ? (size_t)((vdim + 63) / 64) * (la_pad16(dim) + 16) : 0);
}
static inline size_t gl_workspace_bytes(int64_t batch, int heads, int dim, int vdim, int segments) {
    return segments <= 1 ? 0 : (size_t)batch * heads * segments * (la_state_floats(dim, vdim) + la_pad16(dim) + 16) * sizeof(float);
}
