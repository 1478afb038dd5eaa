// Linear recurrences whose decay and input weight come with every token: per head S_t = a_t S_(t-1) + b_t k_t v_t^T and a
// read-out S_t^T q_t, with S in 32-bit floats, kept per sequence in a pool of state slots.  Two kinds:
//
//   kSsd    Mamba-2's state-space duality: a = exp(-A dt), b = dt = softplus(raw + bias); o = S^T q + D v.  Heads of a
//           group share q and k.
//   kMlstm  xLSTM's matrix memory: log gates i and f under a soft cap, a running maximum m (starting at 0) that both are
//           taken relative to, a normaliser n that follows k with the same factors; o = S^T q / (max(|n.q|, exp(-m)) + 1e-6).
//
// Two kernels, as for the constant decays of lightning.hip.  The recurrent one (a decode step, and 32-bit prompts) reads
// the state once, walks its rows token by token in registers and writes the state once.  The chunked one (16-bit
// prompts) multiplies 64 rows at a time on the matrix cores.  With F the running sum of log decays inside the chunk and
// M the running maximum of i - F (kSsd: i = 0 and M = 0; b stays a factor), both from one wave's prefix scans,
//     O = diag(e^(F_t or m0 - M_t)) Q S + ((Q K^T) * e^(F_t - F_s or i_s - F_s - M_t) b_s, s <= t) V
// and the state moves on by the same weights at the chunk's last row.  All logarithms are to base 2.
// n follows by the same products, with the weights as three bf16 terms (all 24 bits); its product with q, by the vector units,
// and the sums of the weighted scores give the denominators.
#include "linear_tiles.h"

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kGlNone = -1.0e30f;  // finite stand-in for minus infinity

enum { kSsd = PA_GL_SSD, kMlstm = PA_GL_MLSTM };

struct GlArgs {
    const void *q, *k, *v;  // row strides ldq, ldk, ldv; head h: q, k at h / per_group * dim, v at h * vdim
    int64_t ldq, ldk, ldv;
    const void *ga, *gb;    // gate logits [row][head] at stride ldg: kSsd ga = raw dt; kMlstm ga = i, gb = f
    int64_t ldg;
    const float *pa, *pb, *pc;  // [heads]: kSsd dt bias, A, D; kMlstm biases of i and f
    float cap, q_scale, den_eps;
    int64_t n_rows;
    float *state;  // [state_rows][heads][head_floats]: S [dp][vp], then per 64 value columns n [dp] and m (kMlstm)
    int64_t state_rows, head_floats;
    const int32_t *ctx_lens, *q_lens, *q_starts, *state_slots;
    void *out;  // [rows][heads * vdim]
    float *ws;  // segment states: S [dp][vp], n [dp], m, log decay, starting m
    int heads, per_group, dim, vdim, dp, vp;
    int batch, segments, seg_rows;
};

struct GlPortion {
    int n, pos0;
    int64_t row0, slot;
};
__device__ __forceinline__ bool gl_portion(const GlArgs &a, int b, GlPortion &p) {
    p.n = a.q_lens ? a.q_lens[b] : 1;
    p.row0 = a.q_starts ? a.q_starts[b] : b;
    p.pos0 = a.ctx_lens[b] - p.n;
    p.slot = a.state_slots[b];
    if (p.slot >= a.state_rows) p.slot = -1;
    return p.n > 0 && p.pos0 >= 0 && p.row0 >= 0 && p.row0 + p.n <= a.n_rows;
}

// ------------------------------------------------------------------ gates
__device__ __forceinline__ float gl_softplus(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

struct GlHead {  // a head's constants
    float a, b, c;
};
__device__ __forceinline__ GlHead gl_head(const GlArgs &a, int h) {
    return GlHead{a.pa[h], a.pb[h], a.pc ? a.pc[h] : 0.f};
}
// Log decay (base 2) and, kSsd, the input weight or, kMlstm, its logarithm (base 2).
template <int KIND> __device__ __forceinline__ void gl_gate(const GlArgs &a, const GlHead &hd, float ra, float rb, float &decay, float &in) {
    if constexpr (KIND == kSsd) {
        in = gl_softplus(ra + hd.a);
        decay = -hd.b * in * kLog2e;
    } else {
        in = a.cap * tanhf((ra + hd.a) / a.cap) * kLog2e;
        decay = -gl_softplus(-a.cap * tanhf((rb + hd.b) / a.cap)) * kLog2e;
    }
}

// ------------------------------------------------------------------ token by token
constexpr int kRecCols = 64;  // value columns per workgroup: 16 lanes x float4, 16 groups of lanes over the rows of S

// R: rows of S per thread (16 R >= dim).  kMlstm: thread d follows n[d].
template <typename T, int R, int KIND> __global__ __launch_bounds__(256, 4) void gated_recurrent_kernel(const GlArgs a) {
    __shared__ float qs[16 * R], ks[16 * R], vs[kRecCols];
    __shared__ float4 red[16][kRecCols / 4];
    __shared__ float redn[4];
    const int h = blockIdx.y, b = blockIdx.z, v0 = blockIdx.x * kRecCols;
    GlPortion p;
    if (!gl_portion(a, b, p)) return;
    const int tid = threadIdx.x, col = tid % 16 * 4, grp = tid / 16;
    const bool live = v0 + col < a.vp;  // (vp is a multiple of 16)
    float *head = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * a.head_floats : nullptr;
    float *sp = head ? head + v0 + col : nullptr;
    float *np = head ? head + (int64_t)a.dp * a.vp + blockIdx.x * (int64_t)(a.dp + 16) : nullptr;  // this workgroup's copy
    const bool resume = head && p.pos0 > 0;
    float4 s[R];
    float n = 0.f, m = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = grp + 16 * r;
        s[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (resume && live && d < a.dp) s[r] = *reinterpret_cast<const float4 *>(sp + (int64_t)d * a.vp);
    }
    if (KIND == kMlstm && resume) {
        if (tid < a.dp && tid < 16 * R) n = np[tid];
        m = np[a.dp];
    }
    const GlHead hd = gl_head(a, h);
    const int g = h / a.per_group;
    const T *q = reinterpret_cast<const T *>(a.q) + g * a.dim, *k = reinterpret_cast<const T *>(a.k) + g * a.dim;
    const T *v = reinterpret_cast<const T *>(a.v) + h * a.vdim + v0;
    for (int t = 0; t < p.n; ++t) {
        const int64_t row = p.row0 + t;
        for (int i = tid; i < 2 * 16 * R + kRecCols; i += 256) {
            if (i < 16 * R) {
                qs[i] = i < a.dim ? pa_scalar<T>::load(q + row * a.ldq + i) : 0.f;
            } else if (i < 32 * R) {
                const int d = i - 16 * R;
                ks[d] = d < a.dim ? pa_scalar<T>::load(k + row * a.ldk + d) : 0.f;
            } else {
                const int c = i - 32 * R;
                vs[c] = v0 + c < a.vdim ? pa_scalar<T>::load(v + row * a.ldv + c) : 0.f;
            }
        }
        const float ra = pa_scalar<T>::load(reinterpret_cast<const T *>(a.ga) + row * a.ldg + h);
        const float rb = KIND == kMlstm ? pa_scalar<T>::load(reinterpret_cast<const T *>(a.gb) + row * a.ldg + h) : 0.f;
        float keep, in;
        gl_gate<KIND>(a, hd, ra, rb, keep, in);
        if (KIND == kMlstm) {
            const float next = fmaxf(keep + m, in);
            keep = exp2f(keep + m - next);
            in = exp2f(in - next);
            m = next;
        } else {
            keep = exp2f(keep);
        }
        __syncthreads();
        float4 x = *reinterpret_cast<const float4 *>(vs + col);
        x = make_float4(in * x.x, in * x.y, in * x.z, in * x.w);
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float kd = ks[grp + 16 * r], qd = qs[grp + 16 * r];
            s[r].x = fmaf(keep, s[r].x, kd * x.x); s[r].y = fmaf(keep, s[r].y, kd * x.y);
            s[r].z = fmaf(keep, s[r].z, kd * x.z); s[r].w = fmaf(keep, s[r].w, kd * x.w);
            o.x = fmaf(qd, s[r].x, o.x); o.y = fmaf(qd, s[r].y, o.y);
            o.z = fmaf(qd, s[r].z, o.z); o.w = fmaf(qd, s[r].w, o.w);
        }
        red[grp][tid % 16] = o;
        if (KIND == kMlstm) {
            float nq = 0.f;
            if (tid < 16 * R) {
                n = fmaf(keep, n, in * ks[tid]);
                nq = qs[tid] * n;
            }
            nq = pa_group_sum<64>(nq);
            if (tid % 64 == 0) redn[tid / 64] = nq;
        }
        __syncthreads();
        if (tid < kRecCols && v0 + tid < a.vdim) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) sum += reinterpret_cast<const float *>(red[i])[tid];
            if (KIND == kMlstm) {
                const float den = (redn[0] + redn[1]) + (redn[2] + redn[3]);
                sum = a.q_scale * sum / (fmaxf(fabsf(a.q_scale * den), exp2f(-m)) + a.den_eps);
            } else {
                sum = fmaf(hd.c, vs[tid], sum);
            }
            pa_scalar<T>::store(reinterpret_cast<T *>(a.out) + row * ((int64_t)a.heads * a.vdim) + h * a.vdim + v0 + tid, sum);
        }
        if (KIND == kSsd) __syncthreads();  // (vs is read above)
        // (otherwise: the next token's writes to qs, ks, vs follow every thread's reads of them, before the barrier above;
        // its writes to red and redn come after its own barrier, which the threads that sum here reach afterwards)
    }
    if (!head) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = grp + 16 * r;
        if (live && d < a.dp) *reinterpret_cast<float4 *>(sp + (int64_t)d * a.vp) = s[r];
    }
    if (KIND == kMlstm) {
        if (tid < a.dp && tid < 16 * R) np[tid] = n;
        if (tid == 0) np[a.dp] = m;
    }
}

// ------------------------------------------------------------------ chunks on the matrix cores
// Per-chunk vectors in LDS (64 rows each)
struct GlRows {
    float row[64], col[64], mul[64];  // a score (t, s) is weighted by 2^(row[t] + col[s]) mul[s]
    float inter[64], add[64];         // rows' factor on Q S; weights of the chunk's rows in the new state
    float low[64];                    // exp(-m)
    float whole, pad[15];             // factor on the old state
    uint16_t one[3][64];              // kMlstm: `add` as three bf16 terms (all 24 bits)
};

// Parts that n . q of a row is summed in: the waves that hold rows of n
template <int KD, int NW> constexpr int gl_parts() { return KD / 32 < NW ? KD / 32 : NW; }
// Elements of the tiles: K and Q (hashed), V (row-major), the two terms of the weighted scores.
template <int KD, int NW> constexpr int gl_kv_elems() { return 64 * KD + 64 * (16 * NW + kLaPadV); }
template <int KD, int NW, int KIND, bool STATES> constexpr size_t gl_lds_bytes() {
    const size_t elems = STATES ? 2 * gl_kv_elems<KD, NW>()  // (double-buffered: one barrier per chunk)
                                : gl_kv_elems<KD, NW>() + 64 * KD + 2 * 64 * kLaPitchA;
    return elems * 2 + 2 * sizeof(GlRows) + (KIND == kMlstm && !STATES ? (gl_parts<KD, NW>() + 2) * 64 * 4 : 0);
}

// Inclusive scans over the wave: rows of 16 lanes by shifts inside the row, then the rows before.
template <int CTRL> __device__ __forceinline__ float gl_shift(float x, float outside) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, outside), __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float gl_lane(float x, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}
__device__ __forceinline__ float gl_scan_add(float x, int lane) {
    x += gl_shift<0x111>(x, 0.f);
    x += gl_shift<0x112>(x, 0.f);
    x += gl_shift<0x114>(x, 0.f);
    x += gl_shift<0x118>(x, 0.f);
    const float r0 = gl_lane(x, 15), r1 = r0 + gl_lane(x, 31), r2 = r1 + gl_lane(x, 47);
    return x + (lane < 16 ? 0.f : lane < 32 ? r0 : lane < 48 ? r1 : r2);
}
__device__ __forceinline__ float gl_scan_max(float x, int lane) {
    x = fmaxf(x, gl_shift<0x111>(x, kGlNone));
    x = fmaxf(x, gl_shift<0x112>(x, kGlNone));
    x = fmaxf(x, gl_shift<0x114>(x, kGlNone));
    x = fmaxf(x, gl_shift<0x118>(x, kGlNone));
    const float r0 = gl_lane(x, 15), r1 = fmaxf(r0, gl_lane(x, 31)), r2 = fmaxf(r1, gl_lane(x, 47));
    return fmaxf(x, lane < 16 ? kGlNone : lane < 32 ? r0 : lane < 48 ? r1 : r2);
}

// KD: dim padded to 64, 128 or 256.  NW: waves; each owns 16 value columns.  All products are taken transposed (value
// columns, or keys, as the rows of the result), so that a lane holds four consecutive elements of one row t.
// STATES: only the segment's own contribution to the state, to the workspace (first pass over a portion in segments).
// Rows come in 16-byte pieces and lie in LDS as they are (hashed): the rows of S that an operand's lanes hold are then 8 g .. 8 g + 7 of 32.
// A SIMD's two waves run in step (a compute unit has room for one workgroup at dim 256), so a chunk takes what its waves wait, and these waits went:
// operands are read ahead of the products before them, with no branch in between; places that follow from one by an exclusive or are not kept (kept,
// they were spilled, and each reload waited for the tile's loads); the next tile's loads are spread over the chunk; its gates are made by a wave
// without score tiles; n . q is a product, and rows' factors are divided once per row and wave.  Cycles of a chunk at 256 x 128 columns, mLSTM: 21400 ->
// 15000, of which products keep a SIMD busy for 5800 and the vector unit for 5100.
// One prompt of 15999 rows, 4 heads of 256 x 512 (mLSTM): second pass 171 -> 125 us, first 72 -> 54; 8 prompts of 1226 .. 1840 rows, 16 heads of 128 x 64 (SSD)
// 87 -> 71; 17 of 480 .. 628, 4 heads of 256 x 512 162 -> 110; single chunks, 23 of 2 .. 25 rows, 8 heads of 128 x 256, 20.1 -> 15.9.
// WIDE: rows of whole, aligned 16-byte pieces, else of 8-byte ones.  (In one kernel, with a branch, each load of the one kind waited for those of the other,
// which had never been asked for: q, k and v of a workgroup's first chunk came one after the other.)  The first chunk's gates are asked for
// ahead of its tiles and made while those are on their way.  At 64 x 64 three workgroups share a compute unit.  Single chunks, 32 heads of 64 x 64, us: branch and
// two workgroups, WIDE, gates first, three workgroups: mLSTM, 500 of 10 .. 30 rows 235, 200, 191, 152; 130 of 65 .. 128 96, 92, 86, 80.  SSD, which has three
// anyway, 500 of 10 .. 30 163, 133, 126.
template <int KD, int NW, int KIND, bool STATES, bool WIDE>
__global__ __launch_bounds__(64 * NW, NW == 4 && KD == 256 ? 1 : NW == 4 && KD == 64 ? 3 : 2) void gated_chunk_kernel(const GlArgs a) {
    constexpr int kCols = 16 * NW, kLdV = kCols + kLaPadV, kThr = 64 * NW;
    constexpr int kKP = 64 * (KD / 8) / kThr, kKRows = kThr / (KD / 8);  // 16-byte pieces of K per thread, rows between them; of V: two
    constexpr int kVRows = kThr / (kCols / 8);
    static_assert(kKP * kThr == 64 * (KD / 8) && 2 * kVRows == 64, "whole passes");
    constexpr int kST = NW == 8 ? 2 : 4;  // score tiles per wave
    constexpr int kNd = (KD / 32 + NW - 1) / NW;  // kMlstm: 32-row pieces of n per wave
    constexpr int kParts = gl_parts<KD, NW>();
    constexpr int kGates = NW == 8 ? 1 : 0;  // the wave with the fewest score tiles (of eight: none) makes the next chunk's gates meanwhile
    extern __shared__ __align__(16) char lds[];
    GlRows *rows = reinterpret_cast<GlRows *>(lds);
    float *nq_s = reinterpret_cast<float *>(rows + 2);  // kMlstm: n . q per row, kParts parts; two parts of the score sums
    float *sum_s = nq_s + 64 * kParts;
    __bf16 *tiles = reinterpret_cast<__bf16 *>(KIND == kMlstm && !STATES ? sum_s + 128 : nq_s);
    __bf16 *k_s = tiles, *v_s = k_s + 64 * KD;
    __bf16 *q_s = tiles + gl_kv_elems<KD, NW>(), *a_hi = q_s + 64 * KD, *a_lo = a_hi + 64 * kLaPitchA;

    LaPlace place;
    GlPortion p;
    if (!la_place(a, (a.vdim + 16 * NW - 1) / (16 * NW), place, p)) return;
    const int h = place.h, seg = place.seg, vsl = place.vsl, b = place.b;
    const int r_beg = seg * a.seg_rows, r_end = r_beg + a.seg_rows < p.n ? r_beg + a.seg_rows : p.n;
    // (what a portion's last segment adds is for nobody else: the second pass leaves the state behind it)
    const bool last = r_end == p.n;
    if (r_beg >= p.n || (STATES && last)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int v0 = vsl * kCols, vw = wave * 16;  // first column of the workgroup, of the wave inside it
    const int l16 = tid & 15, g = lane >> 4;
    const GlHead hd = gl_head(a, h);

    // The state slice of this wave: tile dt holds d = 32 (dt / 2) + 8 g + 4 (dt % 2) + i, v = v0 + vw + l16
    f4 s[KD / 16];
    auto s_row = [](int dt, int i) { return 32 * (dt / 2) + 4 * (dt % 2) + i; };
    const int64_t state_elems = (int64_t)a.dp * a.vp;
    float *pool = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * a.head_floats : nullptr;
    float *seg_state = a.segments > 1 ? a.ws + (((int64_t)b * a.heads + h) * a.segments + seg) * (state_elems + a.dp + 16) : nullptr;
    const float *from = STATES ? nullptr : (a.segments > 1 ? seg_state : (p.pos0 > 0 ? pool : nullptr));
    // (a state as a buffer: rows past dp lie past its end, columns past vp get an offset outside)
    const int state_bytes = (int)state_elems * 4;
    const int v = v0 + vw + l16;
    const uint32_t soff = v < a.vp ? (uint32_t)(8 * g * a.vp + v) * 4u : kLaOutside;
    {
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(from ? from : a.state), 0, from ? state_bytes : 0, 0x00020000);  // (no state: every load is past the end)
#pragma unroll
        for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s[dt][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src, soff + s_row(dt, i) * a.vp * 4, 0, 0));
    }
    // n and m of the workgroup: a wave follows its 32-row pieces of n (n[j][e][i]: row 32 (kNd wave + j) + 8 g + 4 e + i, the
    // same in all columns), one wave m
    const int rep0 = v0 / kRecCols;
    f4 n[KIND == kMlstm ? kNd : 1][2];
    float m_prev = STATES ? kGlNone : 0.f, decayed = 0.f;
    auto n_row = [&](int j, int e) { return 32 * (kNd * wave + j) + 8 * g + 4 * e; };
    if constexpr (KIND == kMlstm) {
        const float *np = from ? from + state_elems + (a.segments > 1 ? 0 : rep0 * (a.dp + 16)) : nullptr;
#pragma unroll
        for (int j = 0; j < kNd; ++j)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                n[j][e] = f4{0.f, 0.f, 0.f, 0.f};
                if (np && n_row(j, e) < a.dp) n[j][e] = *reinterpret_cast<const f4 *>(np + n_row(j, e));
            }
        if (np) m_prev = a.segments > 1 ? np[a.dp + 2] : np[a.dp];
    }

    const int grp = h / a.per_group;
    const uint16_t *uq = reinterpret_cast<const uint16_t *>(a.q) + p.row0 * a.ldq + grp * a.dim;
    const uint16_t *uk = reinterpret_cast<const uint16_t *>(a.k) + p.row0 * a.ldk + grp * a.dim;
    const uint16_t *uv = reinterpret_cast<const uint16_t *>(a.v) + p.row0 * a.ldv + h * a.vdim + v0;
    const uint16_t *ga = reinterpret_cast<const uint16_t *>(a.ga) + p.row0 * a.ldg + h;
    const uint16_t *gb = reinterpret_cast<const uint16_t *>(a.gb) + p.row0 * a.ldg + h;
    const int vcols = a.vdim - v0 < kCols ? a.vdim - v0 : kCols;
    la_u4 kb[kKP], qb[STATES ? 1 : kKP], vb[2];
    const int kr = tid / (KD / 8), kc = tid % (KD / 8), vr = tid / (kCols / 8), vc = tid % (kCols / 8);  // a thread's first row and piece
    auto fetch_rows = [&](auto &x, const uint16_t *base, int64_t ld, int r0, int row, int piece, int rows_apart, int cols) {
        const int nr = r_end - r0 < kLaChunk ? r_end - r0 : kLaChunk;
        const __amdgpu_buffer_rsrc_t t = la_tile(base + r0 * ld, ld, nr, cols);
        la_load_pieces(x, t, ld, row, piece * 8, rows_apart, cols, WIDE);
    };
    auto fetch_q = [&](int r0) { fetch_rows(qb, uq, a.ldq, r0, kr, kc, kKRows, a.dim); };
    auto fetch_k = [&](int r0) { fetch_rows(kb, uk, a.ldk, r0, kr, kc, kKRows, a.dim); };
    auto fetch_v = [&](int r0) { fetch_rows(vb, uv, a.ldv, r0, vr, vc, kVRows, vcols); };
    const int row_place = la_place_of<KD>(l16, g), tr_place = la_place_of<KD>(4 * g + l16 / 4, l16 % 4);
    auto put = [&] {
        const int at = kr * KD + (kc ^ la_hash<KD>(kr)) * 8;  // (rows 16 apart have the same hash)
        static_assert(kKRows % 16 == 0 || kKP == 1 || KD == 256, "places of a thread's pieces");
#pragma unroll
        for (int i = 0; i < kKP; ++i) {
            const int to = kKRows % 16 == 0 || kKP == 1 ? at + i * kKRows * KD : (kr + i * kKRows) * KD + (kc ^ la_hash<KD>(kr + i * kKRows)) * 8;
            *reinterpret_cast<la_u4 *>(k_s + to) = kb[i];
            if (!STATES) *reinterpret_cast<la_u4 *>(q_s + to) = qb[i];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<la_u4 *>(v_s + (vr + i * kVRows) * kLdV + vc * 8) = vb[i];
    };
    uint32_t raw_a = 0, raw_b = 0;  // (as they come: a conversion here would wait for all loads before it)
    auto fetch_gates = [&](int r0) {
        if (wave == kGates && lane < r_end - r0) {
            raw_a = ga[(r0 + lane) * a.ldg];
            if (KIND == kMlstm) raw_b = gb[(r0 + lane) * a.ldg];
        }
    };
    auto gates = [&](int r0, GlRows *to) {  // a chunk's gates, one row per lane
        const int nv = r_end - r0 < kLaChunk ? r_end - r0 : kLaChunk;
        float decay, in;
        gl_gate<KIND>(a, hd, __builtin_bit_cast(float, raw_a << 16), __builtin_bit_cast(float, raw_b << 16), decay, in);
        if (lane >= nv) decay = 0.f;
        const float f = gl_scan_add(decay, lane), f_last = gl_lane(f, 63);
        if constexpr (KIND == kSsd) {
            const float mul = lane < nv ? in : 0.f;
            to->row[lane] = f;
            to->col[lane] = -f;
            to->mul[lane] = mul;
            to->inter[lane] = exp2f(f);
            to->add[lane] = exp2f(f_last - f) * mul;
            if (lane == 0) to->whole = exp2f(f_last);
        } else {
            const float col = lane < nv ? in - f : kGlNone;
            const float top = fmaxf(m_prev, gl_scan_max(col, lane)), top_last = gl_lane(top, 63);
            to->row[lane] = -top;
            to->col[lane] = col;
            to->inter[lane] = exp2f(m_prev - top);
            float add = exp2f(col - top_last);
            to->add[lane] = add;
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const __bf16 x = (__bf16)add;
                to->one[e][lane] = __builtin_bit_cast(uint16_t, x);
                add -= (float)x;
            }
            to->low[lane] = exp2f(-(f + top));
            if (lane == 0) to->whole = exp2f(m_prev - top_last);
            m_prev = f_last + top_last;
        }
        decayed += f_last;
    };
    fetch_gates(r_beg);  // (first, and its gates are made while the tiles are on their way)
    if (!STATES) fetch_q(r_beg);
    fetch_k(r_beg);
    fetch_v(r_beg);
    if (wave == kGates) gates(r_beg, rows);
    fetch_gates(r_beg + kLaChunk);
    for (int r0 = r_beg; r0 < r_end; r0 += kLaChunk) {
        const int nv = r_end - r0 < kLaChunk ? r_end - r0 : kLaChunk;
        GlRows *next = rows == reinterpret_cast<GlRows *>(lds) ? rows + 1 : reinterpret_cast<GlRows *>(lds);
        put();
        __syncthreads();
        // (the next tile's loads are spread over the chunk: all at once would hold up a wave for 2500 cycles)
        const bool more = r0 + kLaChunk < r_end;

        bf8 av[2];  // V: the wave's columns as rows
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) av[kk] = la_read_rows_tr(v_s, kLdV, 32 * kk, vw, l16, g);
        f4 o[4];  // O^T: v = 4 g + i of the wave's columns, t = 16 tt + l16
        if constexpr (STATES) {
            if (wave == kGates && more) {
                gates(r0 + kLaChunk, next);
                fetch_gates(r0 + 2 * kLaChunk);
            }
            if (more) {
                fetch_k(r0 + kLaChunk);
                fetch_v(r0 + kLaChunk);
            }
        } else {
            // score tiles (st, rt): keys 16 st + 4 g + i, rows 16 rt + l16.  (No branch inside: each product would wait for its own read.)
            const int rt = NW == 8 ? wave >> 1 : wave;
            f4 sc[kST];
#pragma unroll
            for (int m = 0; m < kST; ++m) sc[m] = f4{0.f, 0.f, 0.f, 0.f};
            auto scores = [&](auto count) {
                constexpr int kN = decltype(count)::value;
                bf8 bq[2], ak[2][kN];
                const int at = la_again(row_place), at_q = at + rt * (32 * KD), at_k = at + (NW == 8 ? wave & 1 : 0) * (32 * KD);
                auto read = [&](int kk) {
                    bq[kk & 1] = la_read_place<KD>(q_s, at_q, 0, kk);
#pragma unroll
                    for (int m = 0; m < kN; ++m) ak[kk & 1][m] = la_read_place<KD>(k_s, at_k, 16 * (NW == 8 ? 2 * m : m), kk);
                };
                read(0);
#pragma unroll
                for (int kk = 0; kk < KD / 32; ++kk) {
                    if (kk + 1 < KD / 32) read(kk + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int m = 0; m < kN; ++m) sc[m] = la_mfma(ak[kk & 1][m], bq[kk & 1], sc[m]);
                }
            };
            if (wave == kGates && more) {
                gates(r0 + kLaChunk, next);
                fetch_gates(r0 + 2 * kLaChunk);
            }
            if (NW == 4 || wave != kGates) {
                if (rt >= 2) scores(std::integral_constant<int, kST>());
                else scores(std::integral_constant<int, kST / 2>());
            }
            // the rows' part from before the chunk: Q S, then its factors (a sequence's first chunk has none)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) o[tt] = f4{0.f, 0.f, 0.f, 0.f};
            const bool carried = from || r0 > r_beg;
            if (!carried && more) {
                fetch_q(r0 + kLaChunk);
                fetch_k(r0 + kLaChunk);
            }
            if (carried) {
                bf8 bq[2][4];
                const int at = la_again(row_place);
                auto read = [&](int dd) {
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) bq[dd & 1][tt] = la_read_place<KD>(q_s, at, 16 * tt, dd);
                };
                read(0);
                if (more) fetch_q(r0 + kLaChunk);
#pragma unroll
                for (int dd = 0; dd < KD / 32; ++dd) {
                    if (dd + 1 < KD / 32) read(dd + 1);
                    const LaSplit sp = la_split_pair(s[2 * dd], s[2 * dd + 1]);
                    const bf8 hi = sp.high(), lo = sp.low();
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) o[tt] = la_mfma(hi, bq[dd & 1][tt], o[tt]);
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) o[tt] = la_mfma(lo, bq[dd & 1][tt], o[tt]);
                    if (dd == KD / 64 && more) fetch_k(r0 + kLaChunk);
                }
            }
            if constexpr (KIND == kMlstm) {  // n . q over the wave's rows of n, all 24 bits of them; the same in all rows of the result
                if (wave < kParts) {
                    const int at = la_again(row_place);
                    f4 nq[4];
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) nq[tt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < kNd; ++j) {
                        if (!carried) break;  // (uniform)
                        const LaSplit3 x = la_split3(n[j][0], n[j][1]);
                        bf8 bq[4];
#pragma unroll
                        for (int tt = 0; tt < 4; ++tt) bq[tt] = la_read_place<KD>(q_s, at, 16 * tt, kNd * wave + j);
#pragma unroll
                        for (int e = 0; e < 3; ++e)
#pragma unroll
                            for (int tt = 0; tt < 4; ++tt) nq[tt] = la_mfma(x.term[e], bq[tt], nq[tt]);
                    }
                    nq_s[lane * kParts + wave] = g == 0 ? nq[0][0] : g == 1 ? nq[1][0] : g == 2 ? nq[2][0] : nq[3][0];
                }
            }
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                const float f = rows->inter[16 * tt + l16];
#pragma unroll
                for (int i = 0; i < 4; ++i) o[tt][i] *= f;
            }
            if (more) fetch_v(r0 + kLaChunk);
            // the scores' weights
            const int t = 16 * rt + l16;
            const float row_w = rows->row[t];
            float sum = 0.f;
#pragma unroll
            for (int m = 0; m < kST; ++m) {
                const int st = NW == 8 ? 2 * m + (wave & 1) : m;
                if (st > rt + 1) continue;  // (tile rt + 1 is read as zeros when the last k-step covers it)
                const int c = 16 * st + 4 * g;
                const f4 cw = *reinterpret_cast<const f4 *>(rows->col + c);
                f4 x;
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = c + i <= t ? sc[m][i] * __builtin_amdgcn_exp2f(row_w + cw[i]) : 0.f;
                if constexpr (KIND == kSsd) {
                    const f4 mul = *reinterpret_cast<const f4 *>(rows->mul + c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = fmaf(x[i], mul[i], c + i == t ? hd.c : 0.f);
                } else {
                    sum += (x[0] + x[1]) + (x[2] + x[3]);
                }
                uint2 hi, lo;
                la_split2(x[0], x[1], hi.x, lo.x);
                la_split2(x[2], x[3], hi.y, lo.y);
                *reinterpret_cast<uint2 *>(a_hi + t * kLaPitchA + la_paired(c)) = hi;
                *reinterpret_cast<uint2 *>(a_lo + t * kLaPitchA + la_paired(c)) = lo;
            }
            if constexpr (KIND == kMlstm) {
                sum += __shfl_xor(sum, 16, 64);
                sum += __shfl_xor(sum, 32, 64);
                if (g == 0) sum_s[(NW == 8 ? wave & 1 : 0) * 64 + t] = sum;
                if (NW == 4 && g == 1) sum_s[64 + t] = 0.f;
            }
            __syncthreads();
            bf8 ah[2][4], al[2][4];  // (all reads ahead of the products)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) {
                    ah[kk][tt] = la_read8(a_hi + (16 * tt + l16) * kLaPitchA + 32 * kk + 8 * g);
                    al[kk][tt] = la_read8(a_lo + (16 * tt + l16) * kLaPitchA + 32 * kk + 8 * g);
                }
            }
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) o[tt] = la_mfma(av[kk], ah[kk][tt], o[tt]);
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) o[tt] = la_mfma(av[kk], al[kk][tt], o[tt]);
            }
            const int ldo = a.heads * a.vdim;
            const uint16_t *first = reinterpret_cast<const uint16_t *>(a.out) + (p.row0 + r0) * (int64_t)ldo + h * a.vdim + v0;
            const __amdgpu_buffer_rsrc_t dst = la_tile(first, ldo, nv, vcols);
            const int c = vw + 4 * g;
            float row_f = a.q_scale;  // of row `lane`
            if constexpr (KIND == kMlstm) {
                float nq = 0.f;
#pragma unroll
                for (int x = 0; x < kParts; ++x) nq += nq_s[lane * kParts + x];
                const float den = fmaf(rows->inter[lane], nq, sum_s[lane] + sum_s[64 + lane]);
                row_f /= fmaxf(fabsf(row_f * den), rows->low[lane]) + a.den_eps;
            }
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                const int row = 16 * tt + l16;
                const float f = KIND == kMlstm ? __shfl(row_f, row, 64) : row_f;
                const la_u2 x = {row_pack_bf16(o[tt][0] * f, o[tt][1] * f), row_pack_bf16(o[tt][2] * f, o[tt][3] * f)};
                __builtin_amdgcn_raw_buffer_store_b64(x, dst, c < vcols ? (uint32_t)(row * ldo + c) * 2u : kLaOutside, 0, 0);
            }
        }
        // S <- whole S + K^T (weights V), operands a group of tiles ahead of their products
        constexpr int kGroup = 4, kGroups = KD / 16 / kGroup;
        bf8 ak[2][kGroup];
        const int at = la_again(tr_place);
        auto read = [&](int step) {  // (kk, group)
#pragma unroll
            for (int j = 0; j < kGroup; ++j) ak[step & 1][j] = la_read_place_tr<KD>(k_s, at, 32 * (step / kGroups), step % kGroups * kGroup + j);
        };
        read(0);
        const float whole = rows->whole;
        auto keep = [&](int first) {
#pragma unroll
            for (int dt = first; dt < first + kGroup; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[dt][i] *= whole;
        };
        keep(0);
        if constexpr (KIND == kMlstm) {
#pragma unroll
            for (int j = 0; j < kNd; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    n[j][0][i] *= whole;
                    n[j][1][i] *= whole;
                }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const f4 w0 = *reinterpret_cast<const f4 *>(rows->add + 32 * kk + 4 * g), w1 = *reinterpret_cast<const f4 *>(rows->add + 32 * kk + 16 + 4 * g);
            const LaSplit sp = la_split_weighted(av[kk], w0, w1);
            const bf8 hi = sp.high(), lo = sp.low();
#pragma unroll
            for (int x = 0; x < kGroups; ++x) {
                const int step = kk * kGroups + x;
                if (step + 1 < 2 * kGroups) read(step + 1);
                if (step + 1 < kGroups) keep((step + 1) * kGroup);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < kGroup; ++j) s[x * kGroup + j] = la_mfma(ak[step & 1][j], hi, s[x * kGroup + j]);
#pragma unroll
                for (int j = 0; j < kGroup; ++j) s[x * kGroup + j] = la_mfma(ak[step & 1][j], lo, s[x * kGroup + j]);
            }
            if constexpr (KIND == kMlstm) {  // n likewise, with k alone: the weights in every column
                bf8 ones[3];
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    const __bf16 *x = reinterpret_cast<const __bf16 *>(rows->one[e]) + 32 * kk + 4 * g;
                    ones[e] = la_read44(x, x + 16);
                }
#pragma unroll
                for (int j = 0; j < kNd; ++j) {
                    const int piece = kNd * wave + j;
                    if (piece >= KD / 32) break;  // (uniform)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const bf8 x = la_read_place_tr<KD>(k_s, at, 32 * kk, 2 * piece + e);
#pragma unroll
                        for (int y = 0; y < 3; ++y) n[j][e] = la_mfma(x, ones[y], n[j][e]);
                    }
                }
            }
        }
        rows = next;
        if constexpr (!STATES) {
            __syncthreads();  // the next chunk's tiles may be written now
        } else {              // the other half of the tiles
            k_s = k_s == tiles ? tiles + gl_kv_elems<KD, NW>() : tiles;
            v_s = k_s + 64 * KD;
        }
    }
    float *to = STATES ? seg_state : last ? pool : nullptr;
    if (!to) return;
    const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc((void *)to, 0, state_bytes, 0x00020000);
    uint32_t base = soff;
    asm volatile("" : "+v"(base));  // (offsets made again here instead of kept in registers over the loop)
#pragma unroll
    for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float f = s[dt][i];
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, f), dst, base + s_row(dt, i) * a.vp * 4, 0, 0);
        }
    auto put_n = [&](float *np) {
        if constexpr (KIND == kMlstm) {
#pragma unroll
            for (int j = 0; j < kNd; ++j)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    if (l16 == 0 && n_row(j, e) < a.dp) *reinterpret_cast<f4 *>(np + n_row(j, e)) = n[j][e];
        }
    };
    const bool one = tid == 64 * kGates;  // (of the wave that knows m)
    if constexpr (STATES) {  // (every value slice has the same n, m and decay)
        if (vsl != 0) return;
        put_n(to + state_elems);
        if (one) {
            to[state_elems + a.dp] = m_prev;
            to[state_elems + a.dp + 1] = decayed;
        }
    } else if constexpr (KIND == kMlstm) {  // the copies of this workgroup's columns
        const int reps = (a.vdim + kRecCols - 1) / kRecCols;
        for (int r = rep0; r < reps && r < rep0 + (kCols + kRecCols - 1) / kRecCols; ++r) {
            float *np = to + state_elems + r * (a.dp + 16);
            put_n(np);
            if (one) np[a.dp] = m_prev;
        }
    }
}

// Segment contributions -> start states, in place.  One thread per four elements of S, then of n; the first of n's threads
// also writes m.
template <int KIND> __global__ __launch_bounds__(256) void gated_scan_kernel(const GlArgs a) {
    const int h = blockIdx.y, b = blockIdx.z;
    GlPortion p;
    if (!gl_portion(a, b, p)) return;
    const int64_t n4 = (int64_t)a.dp * a.vp / 4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4 + (KIND == kMlstm ? a.dp / 4 : 0)) return;
    const float *pool = p.slot >= 0 && p.pos0 > 0 ? a.state + (p.slot * a.heads + h) * a.head_floats : nullptr;
    const int64_t stride = 4 * n4 + a.dp + 16;
    float *seg = a.ws + ((int64_t)b * a.heads + h) * a.segments * stride;
    const int segments = (p.n + a.seg_rows - 1) / a.seg_rows;
    float4 cur = pool ? reinterpret_cast<const float4 *>(pool)[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    float m = KIND == kMlstm && pool ? pool[4 * n4 + a.dp] : 0.f;
#pragma unroll 1
    for (int first = 0; first < segments; first += kLaScanAhead, seg += kLaScanAhead * stride) {
        float4 add[kLaScanAhead];  // (the last one leaves nothing)
        float decay[kLaScanAhead], top[kLaScanAhead];
#pragma unroll
        for (int j = 0; j < kLaScanAhead; ++j)
            if (first + j + 1 < segments) {
                add[j] = reinterpret_cast<const float4 *>(seg + j * stride)[i];
                decay[j] = seg[j * stride + 4 * n4 + a.dp + 1];
                if (KIND == kMlstm) top[j] = seg[j * stride + 4 * n4 + a.dp];
            }
#pragma unroll
        for (int j = 0; j < kLaScanAhead; ++j) {
            if (first + j >= segments) break;
            reinterpret_cast<float4 *>(seg + j * stride)[i] = cur;
            if (KIND == kMlstm && i == n4) seg[j * stride + 4 * n4 + a.dp + 2] = m;
            if (first + j + 1 >= segments) break;
            float keep, take = 1.f;
            if (KIND == kMlstm) {
                const float m_next = fmaxf(decay[j] + m, top[j]);
                keep = exp2f(decay[j] + m - m_next);
                take = exp2f(top[j] - m_next);
                m = m_next;
            } else {
                keep = exp2f(decay[j]);
            }
            cur = make_float4(fmaf(keep, cur.x, take * add[j].x), fmaf(keep, cur.y, take * add[j].y), fmaf(keep, cur.z, take * add[j].z),
                              fmaf(keep, cur.w, take * add[j].w));
        }
    }
}

template <int KD, int NW, int KIND, bool WIDE> int launch_chunks(const GlArgs &a, int batch, hipStream_t s) {
    constexpr size_t lds = gl_lds_bytes<KD, NW, KIND, false>(), lds_states = gl_lds_bytes<KD, NW, KIND, true>();
    static_assert(lds <= 160 * 1024 && lds_states <= 160 * 1024, "LDS of one compute unit");
    const int slices = (a.vdim + 16 * NW - 1) / (16 * NW);
    const dim3 grid = la_grid(a.heads, slices, batch, a.segments), block(64 * NW);
    if (a.segments > 1) {
        if (int rc = la_big_lds(gated_chunk_kernel<KD, NW, KIND, true, WIDE>, lds_states, "pa_gated_linear")) return rc;
        gated_chunk_kernel<KD, NW, KIND, true, WIDE><<<grid, block, lds_states, s>>>(a);
        const unsigned gx = (unsigned)(((int64_t)a.dp * a.vp / 4 + a.dp / 4 + 255) / 256);
        gated_scan_kernel<KIND><<<dim3(gx, (unsigned)a.heads, (unsigned)batch), dim3(256), 0, s>>>(a);
    }
    if (int rc = la_big_lds(gated_chunk_kernel<KD, NW, KIND, false, WIDE>, lds, "pa_gated_linear")) return rc;
    gated_chunk_kernel<KD, NW, KIND, false, WIDE><<<grid, block, lds, s>>>(a);
    PA_CHECK_LAUNCH("pa_gated_linear (chunks)");
    return PA_OK;
}

template <int KIND, bool WIDE> int launch_chunks_of(const GlArgs &a, int batch, hipStream_t s) {
    const bool many = la_value_cols(a.vdim) == 128;
    if (a.dim <= 64) return many ? launch_chunks<64, 8, KIND, WIDE>(a, batch, s) : launch_chunks<64, 4, KIND, WIDE>(a, batch, s);
    if (a.dim <= 128) return many ? launch_chunks<128, 8, KIND, WIDE>(a, batch, s) : launch_chunks<128, 4, KIND, WIDE>(a, batch, s);
    return many ? launch_chunks<256, 8, KIND, WIDE>(a, batch, s) : launch_chunks<256, 4, KIND, WIDE>(a, batch, s);
}

template <int KIND> int launch_chunks_kind(const GlArgs &a, int batch, hipStream_t s) {
    // rows of whole, aligned 16-byte pieces
    const bool wide = a.dim % 8 == 0 && a.vdim % 8 == 0 && a.ldq % 8 == 0 && a.ldk % 8 == 0 && a.ldv % 8 == 0 &&
                      (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v) & 15u) == 0;
    return wide ? launch_chunks_of<KIND, true>(a, batch, s) : launch_chunks_of<KIND, false>(a, batch, s);
}

template <typename T, int KIND> void launch_recurrent(const GlArgs &a, int batch, hipStream_t s) {
    // (a head's slices, whose rows lie side by side in memory, run at the same time)
    const dim3 grid((unsigned)((a.vdim + kRecCols - 1) / kRecCols), (unsigned)a.heads, (unsigned)batch), block(256);
    if (a.dim <= 64) gated_recurrent_kernel<T, 4, KIND><<<grid, block, 0, s>>>(a);
    else if (a.dim <= 128) gated_recurrent_kernel<T, 8, KIND><<<grid, block, 0, s>>>(a);
    else gated_recurrent_kernel<T, 16, KIND><<<grid, block, 0, s>>>(a);
}

// (two workgroups of four waves share a compute unit)
double gl_together(int dim, int vdim) { return la_value_cols(vdim) == 64 && dim <= 128 ? 1.25 : 0.0; }
size_t gl_segment_bytes(int64_t batch, int heads, int dim, int vdim) { return gl_workspace_bytes(batch, heads, dim, vdim, 2) / 2; }

}  // namespace

extern "C" size_t pa_gated_linear_state_floats(int kind, int dim, int vdim) {
    return (kind == kSsd || kind == kMlstm) && dim > 0 && vdim > 0 ? gl_state_floats(kind == kMlstm, dim, vdim) : 0;
}

extern "C" size_t pa_gated_linear_workspace_bytes_of(int batch, int num_heads, int dim, int vdim, int max_q_len, int64_t n_rows) {
    pa_clear_error();
    if (batch < 0 || num_heads <= 0 || dim <= 0 || vdim <= 0 || max_q_len < 0) {
        pa_fail(PA_ERR_INVALID_ARG, "pa_gated_linear_workspace_bytes: sizes out of range");
        return 0;
    }
    return gl_workspace_bytes(batch, num_heads, dim, vdim,
                              la_asked_segments(batch, la_per_sequence(num_heads, vdim), la_cus(), gl_together(dim, vdim), max_q_len, n_rows,
                                                gl_segment_bytes(batch, num_heads, dim, vdim)));
}

extern "C" size_t pa_gated_linear_workspace_bytes(int batch, int num_heads, int dim, int vdim, int max_q_len) {
    return pa_gated_linear_workspace_bytes_of(batch, num_heads, dim, vdim, max_q_len, -1);
}

extern "C" int pa_gated_linear(int kind, const void *q, int64_t q_stride, const void *k, int64_t k_stride, const void *v,
                               int64_t v_stride, int heads_per_group, const void *gate_a, const void *gate_b,
                               int64_t gate_stride, const float *head_a, const float *head_b, const float *head_c, float cap,
                               float q_scale, float den_eps, int64_t n_rows, float *state, int64_t state_rows,
                               const int32_t *ctx_lens, const int32_t *q_lens, const int32_t *q_starts,
                               const int32_t *state_slots, int batch, int max_q_len, void *out, int num_heads, int dim,
                               int vdim, int dtype, void *workspace, size_t workspace_bytes, void *stream) {
    pa_clear_error();
    PA_REQUIRE(kind == kSsd || kind == kMlstm, "pa_gated_linear: kind=%d is unknown", kind);
    PA_REQUIRE(n_rows >= 0 && batch >= 0 && state_rows >= 0 && max_q_len >= 0, "pa_gated_linear: a count is negative");
    PA_REQUIRE(num_heads > 0 && dim > 0 && vdim > 0, "pa_gated_linear: heads / dim / vdim must be positive");
    PA_REQUIRE(heads_per_group > 0 && num_heads % heads_per_group == 0, "heads_per_group=%d does not divide num_heads=%d",
               heads_per_group, num_heads);
    PA_REQUIRE(num_heads <= 65535 && batch <= 65535, "pa_gated_linear: heads=%d / batch=%d above 65535", num_heads, batch);
    if (dtype != PA_F32 && dtype != PA_BF16) return pa_fail(PA_ERR_UNSUPPORTED, "pa_gated_linear: dtype=%d is not F32 or BF16", dtype);
    if (dim > 256) return pa_fail(PA_ERR_UNSUPPORTED, "pa_gated_linear: dim=%d above 256", dim);
    const int groups = num_heads / heads_per_group;
    PA_REQUIRE(q_stride >= (int64_t)groups * dim && k_stride >= (int64_t)groups * dim && v_stride >= (int64_t)num_heads * vdim &&
                   gate_stride >= num_heads, "pa_gated_linear: a stride is shorter than its row");
    PA_REQUIRE((int64_t)num_heads * (dim + vdim) <= 0x7fffffff, "pa_gated_linear: rows are too long");
    PA_REQUIRE((q_lens == nullptr) == (q_starts == nullptr), "pa_gated_linear: q_lens and q_starts come together");
    PA_REQUIRE(kind == kSsd || cap > 0.f, "pa_gated_linear: cap must be positive");
    if (n_rows == 0 || batch == 0 || (q_lens && max_q_len == 0)) return PA_OK;
    PA_REQUIRE(q && k && v && gate_a && (gate_b || kind == kSsd) && head_a && head_b && (head_c || kind == kMlstm) && state &&
                   ctx_lens && state_slots && out, "pa_gated_linear: NULL argument");
    PA_REQUIRE(q_lens || n_rows >= batch, "n_rows=%lld below batch=%d", (long long)n_rows, batch);
    PA_REQUIRE(pa_aligned16(state), "pa_gated_linear: the state must be 16-byte aligned");
    GlArgs a{};
    a.q = q; a.k = k; a.v = v; a.ldq = q_stride; a.ldk = k_stride; a.ldv = v_stride; a.per_group = heads_per_group;
    a.ga = gate_a; a.gb = kind == kSsd ? gate_a : gate_b; a.ldg = gate_stride; a.pa = head_a; a.pb = head_b; a.pc = head_c;
    a.cap = cap; a.q_scale = kind == kSsd ? 1.f : q_scale; a.den_eps = den_eps; a.n_rows = n_rows; a.state = state; a.state_rows = state_rows;
    a.ctx_lens = ctx_lens; a.q_lens = q_lens; a.q_starts = q_starts; a.state_slots = state_slots; a.out = out;
    a.heads = num_heads; a.dim = dim; a.vdim = vdim; a.dp = la_pad16(dim); a.vp = la_pad16(vdim);
    a.head_floats = (int64_t)gl_state_floats(kind == kMlstm, dim, vdim);
    a.segments = 1;
    hipStream_t s = (hipStream_t)stream;
    // single rows, 32-bit rows, rows that are not whole 8-byte vectors, rows too far apart for 32-bit offsets
    const uintptr_t at = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out;
    const int64_t most = 1 << 22;
    if (!q_lens || dtype == PA_F32 || dim % 4 != 0 || vdim % 4 != 0 || q_stride % 4 != 0 || k_stride % 4 != 0 ||
        v_stride % 4 != 0 || (at & 7u) != 0 || q_stride > most || k_stride > most || v_stride > most ||
        (int64_t)num_heads * vdim > most) {
        if (dtype == PA_F32) {
            if (kind == kSsd) launch_recurrent<float, kSsd>(a, batch, s);
            else launch_recurrent<float, kMlstm>(a, batch, s);
        } else {
            if (kind == kSsd) launch_recurrent<pa_bf16, kSsd>(a, batch, s);
            else launch_recurrent<pa_bf16, kMlstm>(a, batch, s);
        }
        PA_CHECK_LAUNCH("pa_gated_linear");
        return PA_OK;
    }
    a.segments = la_launch_segments(batch, la_per_sequence(num_heads, vdim), la_cus(), gl_together(dim, vdim), max_q_len, n_rows,
                                    gl_segment_bytes(batch, num_heads, dim, vdim), workspace ? workspace_bytes : 0,
                                    pa_aligned16(workspace), gl_together(dim, vdim) > 0 ? 2 : 1);
    PA_REQUIRE(a.segments, "the workspace must be 16-byte aligned");
    a.batch = batch;
    a.seg_rows = la_segment_rows(max_q_len, a.segments);
    a.ws = (float *)workspace;
    return kind == kSsd ? launch_chunks_kind<kSsd>(a, batch, s) : launch_chunks_kind<kMlstm>(a, batch, s);
}
