// Lightning attention: per head S_t = decay S_(t-1) + k_t v_t^T, o_t = S_t^T q_t, with q, k, v = silu(projections) and
// S in 32-bit floats, kept per sequence in a pool of state slots.
//
// Two kernels.  The recurrent one (a decode step, and 32-bit prompts) reads the state once, walks its rows token by
// token in registers and writes the state once: HBM-bound on the state for one token.  The chunked one (16-bit
// prompts) multiplies 64 rows at a time on the matrix cores:
//     O = diag(decay^(t+1)) Q S + ((Q K^T) * decay^(t-s), s <= t) V
//     S = decay^64 S + K^T diag(decay^(63-s)) V
// The 32-bit factors of these products (S, the decayed scores, the decayed values) enter the bf16 matrix cores as a
// sum of two bf16 terms, which keeps 16 bits of their mantissa; q, k and v are bf16 to begin with.
//
// The state never leaves the registers of its wave between chunks: a wave owns a slice of the value columns, its
// accumulator tile [16 d][16 v] of S is, in register order, the B operand of Q S when the operand Q is read with the
// same order of d.
#include "linear_tiles.h"

namespace {

struct LaArgs {
    const void *u;  // [rows][ldu]: heads * dim of q, heads * dim of k, heads * vdim of v, anything
    int64_t ldu, n_rows;
    float *state;  // [state_rows][heads][pad16(dim)][pad16(vdim)]
    int64_t state_rows;
    const float *decay;  // [heads][kLaChunk + 1]: powers 0 .. 64 of a head's decay
    const int32_t *ctx_lens, *q_lens, *q_starts, *state_slots;
    void *out;  // [rows][heads * vdim]
    float *ws;  // segment states
    int heads, dim, vdim, dp, vp;
    int batch, segments, seg_rows;
};

// The portion of sequence b: rows [row0, row0 + n), the first at position pos0.  False: nothing to do.
struct Portion {
    int n, pos0;
    int64_t row0, slot;
};
__device__ __forceinline__ bool la_portion(const LaArgs &a, int b, Portion &p) {
    p.n = a.q_lens ? a.q_lens[b] : 1;
    p.row0 = a.q_starts ? a.q_starts[b] : b;
    p.pos0 = a.ctx_lens[b] - p.n;
    p.slot = a.state_slots[b];
    if (p.slot >= a.state_rows) p.slot = -1;
    return p.n > 0 && p.pos0 >= 0 && p.row0 >= 0 && p.row0 + p.n <= a.n_rows;
}

// ------------------------------------------------------------------ token by token
constexpr int kRecCols = 64;  // value columns per workgroup: 16 lanes x float4, 16 groups of lanes over the rows of S

// silu as the products of a layer see it: in the type of the activations
template <typename T> __device__ __forceinline__ float la_act(float x) {
    x = row_silu<T>(x);
    if constexpr (sizeof(T) == 2) return (float)(__bf16)x;
    return x;
}

// R: rows of S per thread (16 R >= dim)
template <typename T, int R> __global__ __launch_bounds__(256) void lightning_recurrent_kernel(const LaArgs a) {
    __shared__ float qs[16 * R], ks[16 * R], vs[kRecCols];
    __shared__ float4 red[16][kRecCols / 4];
    const int b = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * kRecCols;
    Portion p;
    if (!la_portion(a, b, p)) return;
    const int tid = threadIdx.x, col = tid % 16 * 4, grp = tid / 16;
    const bool live = v0 + col < a.vp;  // (vp is a multiple of 16)
    float *sp = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * (int64_t)a.dp * a.vp + v0 + col : nullptr;
    float4 s[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = grp + 16 * r;
        s[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (sp && p.pos0 > 0 && live && d < a.dp) s[r] = *reinterpret_cast<const float4 *>(sp + (int64_t)d * a.vp);
    }
    const float lam = a.decay[h * (kLaChunk + 1) + 1];
    const T *u = reinterpret_cast<const T *>(a.u);
    for (int t = 0; t < p.n; ++t) {
        const T *row = u + (p.row0 + t) * a.ldu;
        for (int i = tid; i < 2 * 16 * R + kRecCols; i += 256) {
            if (i < 16 * R) {
                qs[i] = i < a.dim ? la_act<T>(pa_scalar<T>::load(row + h * a.dim + i)) : 0.f;
            } else if (i < 32 * R) {
                const int d = i - 16 * R;
                ks[d] = d < a.dim ? la_act<T>(pa_scalar<T>::load(row + (a.heads + h) * a.dim + d)) : 0.f;
            } else {
                const int v = i - 32 * R;
                vs[v] = v0 + v < a.vdim
                            ? la_act<T>(pa_scalar<T>::load(row + 2 * a.heads * a.dim + h * a.vdim + v0 + v)) : 0.f;
            }
        }
        __syncthreads();
        const float4 v = *reinterpret_cast<const float4 *>(vs + col);
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float k = ks[grp + 16 * r], q = qs[grp + 16 * r];
            s[r].x = fmaf(lam, s[r].x, k * v.x); s[r].y = fmaf(lam, s[r].y, k * v.y);
            s[r].z = fmaf(lam, s[r].z, k * v.z); s[r].w = fmaf(lam, s[r].w, k * v.w);
            o.x = fmaf(q, s[r].x, o.x); o.y = fmaf(q, s[r].y, o.y);
            o.z = fmaf(q, s[r].z, o.z); o.w = fmaf(q, s[r].w, o.w);
        }
        red[grp][tid % 16] = o;
        __syncthreads();
        if (tid < kRecCols && v0 + tid < a.vdim) {
            float sum = 0.f;
#pragma unroll
            for (int g = 0; g < 16; ++g) sum += reinterpret_cast<const float *>(red[g])[tid];
            pa_scalar<T>::store(reinterpret_cast<T *>(a.out) + (p.row0 + t) * ((int64_t)a.heads * a.vdim) + h * a.vdim + v0 + tid,
                                sum);
        }
        // (the next token's writes to qs, ks, vs follow every thread's reads of them, before the barrier above; its
        // writes to red come after its own barrier, which the threads that sum here reach afterwards)
    }
    if (!sp || !live) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = grp + 16 * r;
        if (d < a.dp) *reinterpret_cast<float4 *>(sp + (int64_t)d * a.vp) = s[r];
    }
}

// ------------------------------------------------------------------ chunks on the matrix cores
// Elements of the tiles: K and Q (hashed), V (row-major), the two terms of the decayed scores.
template <int KD, int NW> constexpr int la_kv_elems() { return 64 * KD + 64 * (16 * NW + kLaPadV); }
template <int KD, int NW, bool STATES> constexpr size_t la_lds_bytes() {
    const size_t elems = STATES ? 2 * la_kv_elems<KD, NW>()  // (double-buffered: one barrier per chunk)
                                : la_kv_elems<KD, NW>() + 64 * KD + 2 * 64 * kLaPitchA;
    return elems * 2 + (64 + 64 + 64 + 80) * 4;
}

// KD: dim padded to 64, 128 or 256.  NW: waves; each owns 16 value columns.  All products are taken transposed (value
// columns, or keys, as the rows of the result), so that a lane holds four consecutive elements of one row t.
// STATES: only the segment's own contribution to the state, to the workspace (first pass over a portion in segments).
// Bound by the vector instructions: the silu of Q, K and V (two quarter-rate instructions an element) takes a SIMD 4800 of a chunk's 11600 cycles at
// 128 x 128, the terms of 32-bit factors and the factors themselves 3500; the matrix cores work for 2700.  So rows come in 16-byte pieces and lie
// in LDS as they are, in the one layout that both of a tile's products read, with operands ahead of their products and no branch in between; results
// leave the registers straight for the output, and the first pass leaves out each portion's last segment, whose state the second pass itself
// writes to the pool.  8 prompts of 700 .. 4000 rows, 16 x 128 x 128, in three segments: first pass 41.5 -> 41.0 us, second 90.9 -> 86.7 (one read, one
// product at a time, blocks of 4 x 4 -> this); 16 of 900 .. 1000 rows, 16 heads of 256 x 64, 138 -> 121; 10 of 28 .. 81, 32 heads of 128 x 64, 23.0 -> 20.9.
// PAIR: at dim 128 a workgroup of eight waves has a compute unit to itself.  128 registers, with places in LDS worked out in every
// chunk, let two share one.  Where segments outnumber the units: 6 prompts of 400 .. 2600 rows, 32 heads of 128 x 128, all passes,
// 155 -> 144 us; 4 of 1271 .. 5972, 40 heads of 96 x 80, 259 -> 232.  Elsewhere up to 4 % slower.
template <int KD, int NW, bool STATES, bool PAIR>
__global__ __launch_bounds__(64 * NW, PAIR || (KD == 64 && NW == 8) ? 4 : KD == 256 && NW == 4 ? 1 : 2) void lightning_chunk_kernel(const LaArgs a) {
    constexpr int kCols = 16 * NW, kLdV = kCols + kLaPadV, kThr = 64 * NW;
    constexpr int kKP = 64 * (KD / 8) / kThr, kKRows = kThr / (KD / 8);  // 16-byte pieces of K per thread, rows between them; of V: two
    constexpr int kVRows = kThr / (kCols / 8);
    static_assert(kKP * kThr == 64 * (KD / 8) && 2 * kVRows == 64, "whole passes");
    constexpr bool kTight = !STATES && (PAIR || (KD == 64 && NW == 8));  // 128 registers
    constexpr int kGroup = kTight ? 2 : 4, kGroups = KD / 16 / kGroup;  // state tiles whose products go together
    constexpr int kST = NW == 8 ? 2 : 4;  // score tiles per wave
    extern __shared__ __align__(16) char lds[];
    float *rev = reinterpret_cast<float *>(lds);  // decay from row s to the last row of a whole chunk ...
    float *rev_tail = rev + 64;                   // ... and of a portion's last chunk
    float *pw = rev + 192;                        // powers 0 .. 64, behind 64 zeros for the keys after a row
    __bf16 *tiles = reinterpret_cast<__bf16 *>(rev + 272);
    __bf16 *k_s = tiles, *v_s = k_s + 64 * KD;
    __bf16 *q_s = tiles + la_kv_elems<KD, NW>(), *a_hi = q_s + 64 * KD, *a_lo = a_hi + 64 * kLaPitchA;

    LaPlace place;
    Portion p;
    if (!la_place(a, (a.vdim + 16 * NW - 1) / (16 * NW), place, p)) return;
    const int h = place.h, seg = place.seg, vsl = place.vsl, b = place.b;
    const int r_beg = seg * a.seg_rows, r_end = r_beg + a.seg_rows < p.n ? r_beg + a.seg_rows : p.n;
    // (what a portion's last segment adds is for nobody else: the second pass leaves the state behind it)
    const bool last = r_end == p.n;
    if (r_beg >= p.n || (STATES && last)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int v0 = vsl * kCols, vw = wave * 16;  // first column of the workgroup, of the wave inside it
    const float *powers = a.decay + h * (kLaChunk + 1);
    if (tid <= kLaChunk) pw[tid] = powers[tid];
    if (tid < 64) {
        rev[tid] = powers[63 - tid];
        pw[tid - 64] = 0.f;
    }
    const int l16 = tid & 15, g = lane >> 4;

    // The state slice of this wave: tile dt holds d = 32 (dt / 2) + 8 g + 4 (dt % 2) + i, v = v0 + vw + l16
    f4 s[KD / 16];
    auto s_row = [](int dt, int i) { return 32 * (dt / 2) + 4 * (dt % 2) + i; };
    const int64_t state_elems = (int64_t)a.dp * a.vp;
    float *pool = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * state_elems : nullptr;
    float *seg_state = a.segments > 1 ? a.ws + (((int64_t)b * a.heads + h) * a.segments + seg) * state_elems : nullptr;
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

    const uint16_t *u = reinterpret_cast<const uint16_t *>(a.u) + p.row0 * a.ldu;
    const uint16_t *uq = u + h * a.dim, *uk = u + (a.heads + h) * a.dim;
    const uint16_t *uv = u + 2 * a.heads * a.dim + h * a.vdim + v0;
    const int vcols = a.vdim - v0 < kCols ? a.vdim - v0 : kCols;
    la_u4 kb[kKP], qb[STATES ? 1 : kKP], vb[2];
    // PAIR: what follows from a thread's number is made again wherever it is asked for
    auto thread = [&] { return PAIR ? la_again(tid) : tid; };
    auto fetch_rows = [&](auto &x, const uint16_t *base, int r0, int per_row, int apart, int cols) {
        const int rows = r_end - r0 < kLaChunk ? r_end - r0 : kLaChunk, t = thread();
        la_load_pieces(x, la_tile(base + (int64_t)r0 * a.ldu, a.ldu, rows, cols), a.ldu, t / per_row, t % per_row * 8, apart, cols, true);
    };
    auto fetch_q = [&](int r0) { fetch_rows(qb, uq, r0, KD / 8, kKRows, a.dim); };
    auto fetch_k = [&](int r0) { fetch_rows(kb, uk, r0, KD / 8, kKRows, a.dim); };
    auto fetch_v = [&](int r0) { fetch_rows(vb, uv, r0, kCols / 8, kVRows, vcols); };
    auto put = [&] {
        const int t = thread(), kr = t / (KD / 8), kc = t % (KD / 8), vr = t / (kCols / 8), vc = t % (kCols / 8);
#pragma unroll
        for (int i = 0; i < kKP; ++i) {  // (rows 16 apart have the same hash)
            const int row = kr + (kKRows % 16 == 0 ? 0 : i * kKRows), to = row * KD + (kc ^ la_hash<KD>(row)) * 8 + (kKRows % 16 == 0 ? i * kKRows * KD : 0);
            *reinterpret_cast<la_u4 *>(k_s + to) = kb[i];
            if (!STATES) *reinterpret_cast<la_u4 *>(q_s + to) = qb[i];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<la_u4 *>(v_s + (vr + i * kVRows) * kLdV + vc * 8) = vb[i];
    };
    const int row_place = PAIR ? 0 : la_place_of<KD>(l16, g), tr_place = PAIR ? 0 : la_place_of<KD>(4 * g + l16 / 4, l16 % 4);
    auto rows_at = [&] { const int t = thread(); return PAIR ? la_place_of<KD>(t & 15, (t & 63) >> 4) : la_again(row_place); };
    auto tr_at = [&] { const int t = thread(); return PAIR ? la_place_of<KD>((t & 63) >> 2, t & 3) : la_again(tr_place); };
    if (!STATES) fetch_q(r_beg);
    fetch_k(r_beg);
    fetch_v(r_beg);
    auto silu = [](auto &x) {
#pragma unroll
        for (auto &piece : x)
#pragma unroll
            for (int e = 0; e < 4; ++e) piece[e] = la_silu2(piece[e]);
    };
    for (int r0 = r_beg; r0 < r_end; r0 += kLaChunk) {
        const int nv = r_end - r0 < kLaChunk ? r_end - r0 : kLaChunk;
        const bool more = r0 + kLaChunk < r_end;
        // (beside the products of the chunk before, this was no faster: 8 prompts of 700 .. 4000 rows, 16 heads of 128 x 128, us: first pass 43.9, second
        // 89.1, here 41.0 and 86.7)
        silu(vb);
        silu(kb);
        if (!STATES) silu(qb);
        put();
        if (nv < kLaChunk && tid < 64) rev_tail[tid] = tid < nv ? powers[nv - 1 - tid] : 0.f;
        __syncthreads();

        const int lt = thread(), l16 = lt & 15, g = (lt & 63) >> 4;
        bf8 av[2];  // V: the wave's columns as rows
        auto read_v = [&] {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) av[kk] = la_read_rows_tr(v_s, kLdV, 32 * kk, vw, l16, g);
        };
        if (!kTight) read_v();
        f4 o[4];  // O^T: v = 4 g + i of the wave's columns, t = 16 tt + l16
        if constexpr (STATES) {
            if (more) {
                fetch_k(r0 + kLaChunk);
                fetch_v(r0 + kLaChunk);
            }
        } else {
            // score tiles (st, rt): keys 16 st + 4 g + i, rows 16 rt + l16
            const int rt = NW == 8 ? wave >> 1 : wave;
            f4 sc[kST];
#pragma unroll
            for (int m = 0; m < kST; ++m) sc[m] = f4{0.f, 0.f, 0.f, 0.f};
            // (no branch inside: each product would wait for its own read)
            auto scores = [&](auto count) {
                constexpr int kN = decltype(count)::value;
                bf8 bq[2], ak[2][kN];
                const int at = rows_at(), at_q = at + rt * (32 * KD), at_k = at + (NW == 8 ? wave & 1 : 0) * (32 * KD);
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
            if (rt >= 2) scores(std::integral_constant<int, kST>());
            else scores(std::integral_constant<int, kST / 2>());
            // the rows' part from before the chunk: Q S, then the decay of the way from the chunk's start (a sequence's first chunk has none)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) o[tt] = f4{0.f, 0.f, 0.f, 0.f};
            if (!from && r0 == r_beg) {
                if (more) {
                    fetch_q(r0 + kLaChunk);
                    fetch_k(r0 + kLaChunk);
                }
            } else {
                bf8 bq[2][4];
                const int at = rows_at();
                auto read = [&](int dd) {
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) bq[dd & 1][tt] = la_read_place<KD>(q_s, at, 16 * tt, dd);
                };
                read(0);
                if (more) fetch_q(r0 + kLaChunk);
#pragma unroll
                for (int dd = 0; dd < KD / 32; ++dd) {
                    if (!kTight && dd + 1 < KD / 32) read(dd + 1);
                    if (kTight && dd) read(dd);
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
            if (more) fetch_v(r0 + kLaChunk);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                const float f = pw[16 * tt + l16 + 1];  // decay from the chunk's start to the row
#pragma unroll
                for (int i = 0; i < 4; ++i) o[tt][i] *= f;
            }
#pragma unroll
            for (int m = 0; m < kST; ++m) {
                const int st = NW == 8 ? 2 * m + (wave & 1) : m;
                if (st > rt + 1) continue;  // (tile rt + 1 is read as zeros when the last k-step covers it)
                const int t = 16 * rt + l16, c = 16 * st + 4 * g;
                const float *f = pw + t - c;
                f4 x;  // (a later row's key may be no number: its score is put away ahead of the zero that it meets)
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = (c + i <= t ? sc[m][i] : 0.f) * f[-i];
                uint2 hi, lo;
                la_split2(x[0], x[1], hi.x, lo.x);
                la_split2(x[2], x[3], hi.y, lo.y);
                *reinterpret_cast<uint2 *>(a_hi + t * kLaPitchA + la_paired(c)) = hi;
                *reinterpret_cast<uint2 *>(a_lo + t * kLaPitchA + la_paired(c)) = lo;
            }
            __syncthreads();
            if (kTight) read_v();
            bf8 ah[2][4], al[2][4];  // (all reads ahead of the products)
            auto read = [&](int kk) {
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) {
                    ah[kk][tt] = la_read8(a_hi + (16 * tt + l16) * kLaPitchA + 32 * kk + 8 * g);
                    al[kk][tt] = la_read8(a_lo + (16 * tt + l16) * kLaPitchA + 32 * kk + 8 * g);
                }
            };
            read(0);
            if (!kTight) read(1);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                if (kTight && kk) read(1);
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) o[tt] = la_mfma(av[kk], ah[kk][tt], o[tt]);
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) o[tt] = la_mfma(av[kk], al[kk][tt], o[tt]);
            }
            const int ldo = a.heads * a.vdim, c = vw + 4 * g;
            const uint16_t *first = reinterpret_cast<const uint16_t *>(a.out) + (p.row0 + r0) * (int64_t)ldo + h * a.vdim + v0;
            const __amdgpu_buffer_rsrc_t dst = la_tile(first, ldo, nv, vcols);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                const la_u2 x = {row_pack_bf16(o[tt][0], o[tt][1]), row_pack_bf16(o[tt][2], o[tt][3])};
                __builtin_amdgcn_raw_buffer_store_b64(x, dst, c < vcols ? (uint32_t)((16 * tt + l16) * ldo + c) * 2u : kLaOutside, 0, 0);
            }
        }
        // S <- decay^nv S + K^T (decay^(nv-1-s) V)
        // (operands a group of tiles ahead of their products)
        bf8 ak[2][kGroup];
        const int at = tr_at();
        auto read = [&](int step) {  // (kk, group)
#pragma unroll
            for (int j = 0; j < kGroup; ++j) ak[step & 1][j] = la_read_place_tr<KD>(k_s, at, 32 * (step / kGroups), step % kGroups * kGroup + j);
        };
        read(0);
        const float whole = pw[nv];
        const float *wt = nv < kLaChunk ? rev_tail : rev;
        auto keep = [&](int group) {
#pragma unroll
            for (int dt = group * kGroup; dt < (group + 1) * kGroup; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[dt][i] *= whole;
        };
        keep(0);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const LaSplit sp = la_split_weighted(av[kk], *reinterpret_cast<const f4 *>(wt + 32 * kk + 4 * g), *reinterpret_cast<const f4 *>(wt + 32 * kk + 16 + 4 * g));
            const bf8 hi = sp.high(), lo = sp.low();
#pragma unroll
            for (int x = 0; x < kGroups; ++x) {
                const int step = kk * kGroups + x;
                if (step + 1 < 2 * kGroups) read(step + 1);
                if (step + 1 < kGroups) keep(step + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < kGroup; ++j) s[x * kGroup + j] = la_mfma(ak[step & 1][j], hi, s[x * kGroup + j]);
#pragma unroll
                for (int j = 0; j < kGroup; ++j) s[x * kGroup + j] = la_mfma(ak[step & 1][j], lo, s[x * kGroup + j]);
            }
        }
        if constexpr (!STATES) {
            __syncthreads();  // the next chunk's tiles may be written now
        } else {              // the other half of the tiles
            k_s = k_s == tiles ? tiles + la_kv_elems<KD, NW>() : tiles;
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
}

// Segment contributions -> start states, in place.  The loads of kLaScanAhead segments are in flight at once.
__global__ __launch_bounds__(256) void lightning_scan_kernel(const LaArgs a) {
    const int h = blockIdx.y, b = blockIdx.z;
    Portion p;
    if (!la_portion(a, b, p)) return;
    const int64_t n4 = (int64_t)a.dp * a.vp / 4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const float4 *pool = p.slot >= 0 && p.pos0 > 0 ? reinterpret_cast<const float4 *>(a.state) + (p.slot * a.heads + h) * n4 + i : nullptr;
    float4 *seg = reinterpret_cast<float4 *>(a.ws) + ((int64_t)b * a.heads + h) * a.segments * n4 + i;
    const int segments = (p.n + a.seg_rows - 1) / a.seg_rows;
    float4 cur = pool ? *pool : make_float4(0.f, 0.f, 0.f, 0.f);
    float f = 1.f;  // decay^seg_rows, seg_rows a multiple of the chunk
    for (int c = 0; c < a.seg_rows / kLaChunk; ++c) f *= a.decay[h * (kLaChunk + 1) + kLaChunk];
#pragma unroll 1
    for (int first = 0; first < segments; first += kLaScanAhead) {
        float4 add[kLaScanAhead];  // (the last one leaves nothing)
#pragma unroll
        for (int j = 0; j < kLaScanAhead; ++j)
            if (first + j + 1 < segments) add[j] = seg[(first + j) * n4];
#pragma unroll
        for (int j = 0; j < kLaScanAhead; ++j) {
            if (first + j >= segments) break;
            seg[(first + j) * n4] = cur;
            if (first + j + 1 < segments)
                cur = make_float4(fmaf(f, cur.x, add[j].x), fmaf(f, cur.y, add[j].y), fmaf(f, cur.z, add[j].z), fmaf(f, cur.w, add[j].w));
        }
    }
}

template <int KD, int NW, bool PAIR> int launch_passes(const LaArgs &a, const dim3 &grid, int batch, hipStream_t s) {
    constexpr size_t lds = la_lds_bytes<KD, NW, false>(), lds_states = la_lds_bytes<KD, NW, true>();
    static_assert(lds <= 160 * 1024 && lds_states <= 160 * 1024, "LDS of one compute unit");
    const dim3 block(64 * NW);
    if (a.segments > 1) {
        if (int rc = la_big_lds(lightning_chunk_kernel<KD, NW, true, false>, lds_states, "pa_lightning_chunked")) return rc;
        lightning_chunk_kernel<KD, NW, true, false><<<grid, block, lds_states, s>>>(a);
        const unsigned gx = (unsigned)(((int64_t)a.dp * a.vp / 4 + 255) / 256);
        lightning_scan_kernel<<<dim3(gx, (unsigned)a.heads, (unsigned)batch), dim3(256), 0, s>>>(a);
    }
    if (int rc = la_big_lds(lightning_chunk_kernel<KD, NW, false, PAIR>, lds, "pa_lightning_chunked")) return rc;
    lightning_chunk_kernel<KD, NW, false, PAIR><<<grid, block, lds, s>>>(a);
    PA_CHECK_LAUNCH("pa_lightning_chunked");
    return PA_OK;
}

template <int KD, int NW> int launch_chunks(const LaArgs &a, int batch, hipStream_t s) {
    const int slices = (a.vdim + 16 * NW - 1) / (16 * NW);
    const dim3 grid = la_grid(a.heads, slices, batch, a.segments);
    // unequal portions in more segments than compute units (a segment for each of its lengths, and half a one per portion)
    const double parts = (double)a.n_rows / a.seg_rows + 0.5 * batch;
    const bool pair = KD == 128 && NW == 8 && a.segments > 1 && parts < (double)batch * a.segments && parts * a.heads * slices > 1.1 * la_cus();
    if constexpr (KD == 128 && NW == 8) {
        if (pair) return launch_passes<KD, NW, true>(a, grid, batch, s);
    }
    return launch_passes<KD, NW, false>(a, grid, batch, s);
}

template <typename T> void launch_recurrent(const LaArgs &a, int batch, hipStream_t s) {
    const dim3 grid((unsigned)batch, (unsigned)a.heads, (unsigned)((a.vdim + kRecCols - 1) / kRecCols)), block(256);
    if (a.dim <= 64) lightning_recurrent_kernel<T, 4><<<grid, block, 0, s>>>(a);
    else if (a.dim <= 128) lightning_recurrent_kernel<T, 8><<<grid, block, 0, s>>>(a);
    else lightning_recurrent_kernel<T, 16><<<grid, block, 0, s>>>(a);
}

int la_fill(const char *what, LaArgs &a, const void *u, int64_t u_stride, int64_t n_rows, float *state, int64_t state_rows,
            const float *decay_powers, const int32_t *ctx_lens, const int32_t *q_lens, const int32_t *q_starts,
            const int32_t *state_slots, int batch, void *out, int num_heads, int dim, int vdim, int dtype) {
    PA_REQUIRE(n_rows >= 0 && batch >= 0 && state_rows >= 0, "%s: a count is negative", what);
    PA_REQUIRE(num_heads > 0 && dim > 0 && vdim > 0, "%s: heads / dim / vdim must be positive", what);
    PA_REQUIRE(num_heads <= 65535 && batch <= 65535, "%s: heads=%d / batch=%d above 65535", what, num_heads, batch);
    if (dtype != PA_F32 && dtype != PA_BF16) return pa_fail(PA_ERR_UNSUPPORTED, "%s: dtype=%d is not F32 or BF16", what, dtype);
    if (dim > 256) return pa_fail(PA_ERR_UNSUPPORTED, "%s: dim=%d above 256", what, dim);
    PA_REQUIRE(u_stride >= (int64_t)num_heads * (2 * dim + vdim), "%s: u_stride=%lld is shorter than q, k and v", what,
               (long long)u_stride);
    PA_REQUIRE((int64_t)num_heads * (2 * dim + vdim) <= 0x7fffffff, "%s: rows are too long", what);
    PA_REQUIRE((q_lens == nullptr) == (q_starts == nullptr), "%s: q_lens and q_starts come together", what);
    if (n_rows == 0 || batch == 0) return PA_OK;
    PA_REQUIRE(u && state && decay_powers && ctx_lens && state_slots && out, "%s: NULL argument", what);
    PA_REQUIRE(pa_aligned16(state), "%s: the state must be 16-byte aligned", what);
    a = LaArgs{};
    a.u = u; a.ldu = u_stride; a.n_rows = n_rows; a.state = state; a.state_rows = state_rows; a.decay = decay_powers;
    a.ctx_lens = ctx_lens; a.q_lens = q_lens; a.q_starts = q_starts; a.state_slots = state_slots; a.out = out;
    a.heads = num_heads; a.dim = dim; a.vdim = vdim; a.dp = la_pad16(dim); a.vp = la_pad16(vdim);
    a.segments = 1;
    return PA_OK;
}

// (two workgroups of four waves share a compute unit, or two of eight at dim 64)
double la_together(int dim, int vdim) { return la_value_cols(vdim) == 64 && dim <= 128 ? 1.25 : dim <= 64 ? 1.6 : 0.0; }
size_t la_segment_bytes(int64_t batch, int heads, int dim, int vdim) { return la_workspace_bytes(batch, heads, dim, vdim, 2) / 2; }

}  // namespace

extern "C" size_t pa_lightning_state_floats(int dim, int vdim) {
    return dim > 0 && vdim > 0 ? la_state_floats(dim, vdim) : 0;
}

extern "C" int pa_lightning_recurrent(const void *u, int64_t u_stride, int64_t n_rows, float *state, int64_t state_rows,
                                      const float *decay_powers, const int32_t *ctx_lens, const int32_t *q_lens,
                                      const int32_t *q_starts, const int32_t *state_slots, int batch, void *out,
                                      int num_heads, int dim, int vdim, int dtype, void *stream) {
    pa_clear_error();
    LaArgs a;
    if (int rc = la_fill("pa_lightning_recurrent", a, u, u_stride, n_rows, state, state_rows, decay_powers, ctx_lens, q_lens,
                         q_starts, state_slots, batch, out, num_heads, dim, vdim, dtype))
        return rc;
    if (n_rows == 0 || batch == 0) return PA_OK;
    PA_REQUIRE(q_lens || n_rows >= batch, "n_rows=%lld below batch=%d", (long long)n_rows, batch);
    if (dtype == PA_F32) launch_recurrent<float>(a, batch, (hipStream_t)stream);
    else launch_recurrent<pa_bf16>(a, batch, (hipStream_t)stream);
    PA_CHECK_LAUNCH("pa_lightning_recurrent");
    return PA_OK;
}

extern "C" size_t pa_lightning_workspace_bytes_of(int batch, int num_heads, int dim, int vdim, int max_q_len, int64_t n_rows) {
    pa_clear_error();
    if (batch < 0 || num_heads <= 0 || dim <= 0 || vdim <= 0 || max_q_len < 0) {
        pa_fail(PA_ERR_INVALID_ARG, "pa_lightning_workspace_bytes: sizes out of range");
        return 0;
    }
    return la_workspace_bytes(batch, num_heads, dim, vdim,
                              la_asked_segments(batch, la_per_sequence(num_heads, vdim), la_cus(), la_together(dim, vdim), max_q_len, n_rows,
                                                la_segment_bytes(batch, num_heads, dim, vdim)));
}

extern "C" size_t pa_lightning_workspace_bytes(int batch, int num_heads, int dim, int vdim, int max_q_len) {
    return pa_lightning_workspace_bytes_of(batch, num_heads, dim, vdim, max_q_len, -1);
}

extern "C" int pa_lightning_chunked(const void *u, int64_t u_stride, int64_t n_rows, float *state, int64_t state_rows,
                                    const float *decay_powers, const int32_t *ctx_lens, const int32_t *q_lens,
                                    const int32_t *q_starts, const int32_t *state_slots, int batch, int max_q_len,
                                    void *out, int num_heads, int dim, int vdim, int dtype, void *workspace,
                                    size_t workspace_bytes, void *stream) {
    pa_clear_error();
    LaArgs a;
    PA_REQUIRE(max_q_len >= 0, "max_q_len=%d is negative", max_q_len);
    if (dtype != PA_BF16)
        return pa_fail(PA_ERR_UNSUPPORTED, "pa_lightning_chunked: dtype=%d is not BF16 (32-bit rows take pa_lightning_recurrent)",
                       dtype);
    if (int rc = la_fill("pa_lightning_chunked", a, u, u_stride, n_rows, state, state_rows, decay_powers, ctx_lens, q_lens,
                         q_starts, state_slots, batch, out, num_heads, dim, vdim, dtype))
        return rc;
    if (n_rows == 0 || batch == 0 || max_q_len == 0) return PA_OK;
    PA_REQUIRE(q_lens, "NULL q_lens / q_starts");
    a.segments = la_launch_segments(batch, la_per_sequence(num_heads, vdim), la_cus(), la_together(dim, vdim), max_q_len, n_rows,
                                    la_segment_bytes(batch, num_heads, dim, vdim), workspace ? workspace_bytes : 0,
                                    pa_aligned16(workspace));
    PA_REQUIRE(a.segments, "the workspace must be 16-byte aligned");
    a.batch = batch;
    a.seg_rows = la_segment_rows(max_q_len, a.segments);
    a.ws = (float *)workspace;
    hipStream_t s = (hipStream_t)stream;
    // rows that are not whole 16-byte vectors, or too far apart for a tile's 32-bit offsets: token by token
    if (dim % 8 != 0 || vdim % 8 != 0 || u_stride % 8 != 0 || !pa_aligned16(u) || !pa_aligned16(out) ||
        u_stride > (1 << 22) || (int64_t)num_heads * vdim > (1 << 22)) {
        launch_recurrent<pa_bf16>(a, batch, s);
        PA_CHECK_LAUNCH("pa_lightning_chunked");
        return PA_OK;
    }
    const bool wide = la_value_cols(vdim) == 128;
    if (dim <= 64) return wide ? launch_chunks<64, 8>(a, batch, s) : launch_chunks<64, 4>(a, batch, s);
    if (dim <= 128) return wide ? launch_chunks<128, 8>(a, batch, s) : launch_chunks<128, 4>(a, batch, s);
    return wide ? launch_chunks<256, 8>(a, batch, s) : launch_chunks<256, 4>(a, batch, s);
}
