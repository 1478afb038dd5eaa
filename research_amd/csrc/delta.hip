// The gated delta rule: per head S <- g S, u = beta (v - S^T k), S <- S + k u^T, o = S^T q, with S in 32-bit floats, kept
// per sequence in a pool of state slots.  q and k are made unit vectors here (q also times its scale), g and beta come from
// gate logits: g = exp(-rate softplus(raw + bias)), beta = sigmoid(raw).
//
// Two kernels, as for the other recurrences.  The recurrent one (a decode step, and 32-bit prompts) reads the state once,
// walks its rows token by token in registers and writes the state once.
//
// Portions of 16-bit rows go in chunks of 64 on the matrix cores, in two passes.  With F the running sum of log decays in a
// chunk, all u of a chunk satisfy one triangular system: with A_ts = beta_t (k_t . k_s) e^(F_t - F_s) below the diagonal,
//     U = T (V - e^F K S),   T = (I + A)^-1 diag(beta),
//     O = e^F Q S + C U,     C_ts = (q_t . k_s) e^(F_t - F_s) for s <= t,
//     S <- e^(F_last) S + (e^(F_last - F) K)^T U.
// T and C do not depend on S: the first pass makes them for all chunks at once (T by inverting 16 x 16 blocks on the
// diagonal row by row and joining them with 32-bit matrix products).  The second pass walks a portion's chunks with S in
// accumulator registers; a wave owns value columns, which do not depend on each other.  Unit norms are factors of rows,
// so q and k enter the products as they are stored; T, C, S, U and V - e^F K S are split into two bf16 terms each.
#include "linear_tiles.h"

namespace {

constexpr float kUnitEps = 1e-6f;

struct DeltaArgs {
    const void *q, *k, *v;  // row strides ldq, ldk, ldv; head h: q, k at h / per_group * dim, v at h * vdim
    int64_t ldq, ldk, ldv;
    const void *ga, *gb;    // [row][head] at stride ldg: raw decay and beta logits
    int64_t ldg;
    const float *bias, *rate;  // [heads]
    float q_scale;
    int64_t n_rows;
    float *state;  // [state_rows][heads][dp][vp]
    int64_t state_rows;
    const int32_t *ctx_lens, *q_lens, *q_starts, *state_slots;
    void *out;  // [rows][heads * vdim]
    char *ws;   // per chunk and head: DeltaChunk
    int heads, per_group, dim, vdim, dp, vp, chunks;  // chunks: most chunks of a portion
};

struct DeltaPortion {
    int n, pos0;
    int64_t row0, slot;
};
__device__ __forceinline__ bool delta_portion(const DeltaArgs &a, int b, DeltaPortion &p) {
    p.n = a.q_lens ? a.q_lens[b] : 1;
    p.row0 = a.q_starts ? a.q_starts[b] : b;
    p.pos0 = a.ctx_lens[b] - p.n;
    p.slot = a.state_slots[b];
    if (p.slot >= a.state_rows) p.slot = -1;
    return p.n > 0 && p.pos0 >= 0 && p.row0 >= 0 && p.row0 + p.n <= a.n_rows;
}

__device__ __forceinline__ float delta_softplus(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }
// Log decay to base 2
__device__ __forceinline__ float delta_log_decay(const DeltaArgs &a, int h, float raw) {
    return -a.rate[h] * delta_softplus(raw + a.bias[h]) * 1.4426950408889634f;
}
__device__ __forceinline__ float delta_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

// ------------------------------------------------------------------ token by token
constexpr int kDeltaCols = 64;  // value columns per workgroup: 16 lanes x float4, 16 groups of lanes over the rows of S

// R: rows of S per thread (16 R >= dim)
template <typename T, int R> __global__ __launch_bounds__(256, 4) void delta_recurrent_kernel(const DeltaArgs a) {
    __shared__ float qs[16 * R], ks[16 * R], vs[kDeltaCols];
    __shared__ float4 red[16][kDeltaCols / 4];
    __shared__ float redn[2][4];
    const int h = blockIdx.y, b = blockIdx.z, v0 = blockIdx.x * kDeltaCols;
    DeltaPortion p;
    if (!delta_portion(a, b, p)) return;
    const int tid = threadIdx.x, c4 = tid % 16, col = c4 * 4, grp = tid / 16;
    const bool live = v0 + col < a.vp;  // (vp is a multiple of 16)
    float *sp = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * (int64_t)a.dp * a.vp + v0 + col : nullptr;
    float4 s[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = grp + 16 * r;
        s[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (sp && p.pos0 > 0 && live && d < a.dp) s[r] = *reinterpret_cast<const float4 *>(sp + (int64_t)d * a.vp);
    }
    const int g = h / a.per_group;
    const T *q = reinterpret_cast<const T *>(a.q) + g * a.dim, *k = reinterpret_cast<const T *>(a.k) + g * a.dim;
    const T *v = reinterpret_cast<const T *>(a.v) + h * a.vdim + v0;
    for (int t = 0; t < p.n; ++t) {
        const int64_t row = p.row0 + t;
        float qd = 0.f, kd = 0.f;
        if (tid < 16 * R) {  // (16 R <= 256)
            if (tid < a.dim) {
                qd = pa_scalar<T>::load(q + row * a.ldq + tid);
                kd = pa_scalar<T>::load(k + row * a.ldk + tid);
            }
            qs[tid] = qd;
            ks[tid] = kd;
        }
        if (tid < kDeltaCols) vs[tid] = v0 + tid < a.vdim ? pa_scalar<T>::load(v + row * a.ldv + tid) : 0.f;
        const float q2 = pa_group_sum<64>(qd * qd), k2 = pa_group_sum<64>(kd * kd);
        if (tid % 64 == 0) {
            redn[0][tid / 64] = q2;
            redn[1][tid / 64] = k2;
        }
        const float keep = exp2f(delta_log_decay(a, h, pa_scalar<T>::load(reinterpret_cast<const T *>(a.ga) + row * a.ldg + h)));
        const float beta = delta_sigmoid(pa_scalar<T>::load(reinterpret_cast<const T *>(a.gb) + row * a.ldg + h));
        __syncthreads();
        const float qn = a.q_scale / sqrtf(redn[0][0] + redn[0][1] + redn[0][2] + redn[0][3] + kUnitEps);
        const float kn = 1.f / sqrtf(redn[1][0] + redn[1][1] + redn[1][2] + redn[1][3] + kUnitEps);
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float f = ks[grp + 16 * r] * kn;
            s[r].x *= keep; s[r].y *= keep; s[r].z *= keep; s[r].w *= keep;
            x.x = fmaf(f, s[r].x, x.x); x.y = fmaf(f, s[r].y, x.y);
            x.z = fmaf(f, s[r].z, x.z); x.w = fmaf(f, s[r].w, x.w);
        }
        red[grp][c4] = x;
        __syncthreads();
        const float4 vv = *reinterpret_cast<const float4 *>(vs + col);
        float4 u = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float4 y = red[i][c4];
            u.x += y.x; u.y += y.y; u.z += y.z; u.w += y.w;
        }
        u = make_float4(beta * (vv.x - u.x), beta * (vv.y - u.y), beta * (vv.z - u.z), beta * (vv.w - u.w));
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float f = ks[grp + 16 * r] * kn, e = qs[grp + 16 * r] * qn;
            s[r].x = fmaf(f, u.x, s[r].x); s[r].y = fmaf(f, u.y, s[r].y);
            s[r].z = fmaf(f, u.z, s[r].z); s[r].w = fmaf(f, u.w, s[r].w);
            o.x = fmaf(e, s[r].x, o.x); o.y = fmaf(e, s[r].y, o.y);
            o.z = fmaf(e, s[r].z, o.z); o.w = fmaf(e, s[r].w, o.w);
        }
        __syncthreads();  // red has been read
        red[grp][c4] = o;
        __syncthreads();
        if (tid < kDeltaCols && v0 + tid < a.vdim) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) sum += reinterpret_cast<const float *>(red[i])[tid];
            pa_scalar<T>::store(reinterpret_cast<T *>(a.out) + row * ((int64_t)a.heads * a.vdim) + h * a.vdim + v0 + tid, sum);
        }
        // (the next token's writes to qs, ks, vs and redn follow every thread's reads of them, before the barrier above; its
        // writes to red come after its own first barrier, which the threads that sum here reach afterwards)
    }
    if (!sp) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int d = grp + 16 * r;
        if (live && d < a.dp) *reinterpret_cast<float4 *>(sp + (int64_t)d * a.vp) = s[r];
    }
}

// ------------------------------------------------------------------ chunks: T and C
// What the first pass leaves per chunk and head.  T and C lie as the walk's operands: piece f (rows 16 tt .., columns 32 kk ..) holds for
// lane 16 g + l16 the eight elements of row l16 in the paired order, so that a wave reads and writes whole lines; the quarter above the
// diagonal blocks of 32, all zeros, is left out.
constexpr int kDeltaPieces = 6;
__host__ __device__ constexpr int delta_piece(int tt, int kk) { return kk ? 2 + tt : tt; }
struct DeltaChunk {
    uint16_t t[2][kDeltaPieces][64][8], c[2][kDeltaPieces][64][8];  // both terms of each
    float k_in[64];   // e^F times k's unit factor (on K S)
    float q_in[64];   // e^F times q's unit factor and scale (on Q S)
    float k_out[64];  // e^(F_last - F) times k's unit factor (on U in the new state)
    float keep;       // e^(F_last)
    float pad[63];
};
constexpr int kDeltaMat = 2 * kDeltaPieces * 64 * 8;  // elements of T, of C
// Operand of a matrix in LDS
__device__ __forceinline__ bf8 delta_operand(const __bf16 *m, int term, int tt, int kk, int lane) {
    return la_read8(m + ((term * kDeltaPieces + delta_piece(tt, kk)) * 64 + lane) * 8);
}

__device__ __forceinline__ f4 delta_mfma32(float x, float y, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }

// Inclusive sum over the wave
__device__ __forceinline__ float delta_scan(float x, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const float y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    return x;
}

// Workgroup: one chunk of one head.  Wave w: rows 16 w .. of the products.
template <int KD> __global__ __launch_bounds__(256, KD == 256 ? 2 : 4) void delta_prepare_kernel(const DeltaArgs a) {
    constexpr int kMat = 68, kRowBytes = 2 * 64 * KD * 2, kMatBytes = 2 * 64 * kMat * 4;
    __shared__ __align__(16) char room[kRowBytes > kMatBytes ? kRowBytes : kMatBytes];
    __bf16 *q_s = reinterpret_cast<__bf16 *>(room), *k_s = q_s + 64 * KD;
    // in their place once the products are made: A below the diagonal, (I + A)^-1
    float(*mat)[kMat] = reinterpret_cast<float(*)[kMat]>(room), (*inv)[kMat] = mat + 64;
    __shared__ float part[4][16][17];
    __shared__ float f_s[64], beta_s[64], kn_s[64], qn_s[64];
    const int h = blockIdx.x, chunk = blockIdx.y, b = blockIdx.z;
    DeltaPortion p;
    if (!delta_portion(a, b, p)) return;
    const int r0 = chunk * 64, nv = p.n - r0 < 64 ? p.n - r0 : 64;
    if (nv <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int grp = h / a.per_group;
    const uint16_t *uq = reinterpret_cast<const uint16_t *>(a.q) + (p.row0 + r0) * a.ldq + grp * a.dim;
    const uint16_t *uk = reinterpret_cast<const uint16_t *>(a.k) + (p.row0 + r0) * a.ldk + grp * a.dim;
    {
        const __amdgpu_buffer_rsrc_t tq = la_tile(uq, a.ldq, nv, a.dim), tk = la_tile(uk, a.ldk, nv, a.dim);
        constexpr int kBlocks = 16 * (KD / 4), kPass = kBlocks / 256;
        static_assert(kBlocks % 256 == 0, "whole passes");
#pragma unroll
        for (int i = 0; i < kPass; ++i) {
            const int blk = tid + 256 * i, r = blk / (KD / 4) * 4, c = blk % (KD / 4) * 4;
            const LaBlock x = la_load_block(tq, la_block_off(a.ldq, r, c, a.dim), (uint32_t)a.ldq * 2u);
            const LaBlock y = la_load_block(tk, la_block_off(a.ldk, r, c, a.dim), (uint32_t)a.ldk * 2u);
            la_put_hashed<KD>(x, r, c, q_s);
            la_put_hashed<KD>(y, r, c, k_s);
        }
    }
    if (wave == 0) {
        float decay = 0.f, beta = 0.f;
        if (lane < nv) {
            const int64_t row = p.row0 + r0 + lane;
            decay = delta_log_decay(a, h, pa_scalar<pa_bf16>::load(reinterpret_cast<const pa_bf16 *>(a.ga) + row * a.ldg + h));
            beta = delta_sigmoid(pa_scalar<pa_bf16>::load(reinterpret_cast<const pa_bf16 *>(a.gb) + row * a.ldg + h));
        }
        f_s[lane] = delta_scan(decay, lane);
        beta_s[lane] = beta;
    }
    __syncthreads();
    {   // unit factors: four lanes per row
        const int r = tid / 4;
        float q2 = 0.f, k2 = 0.f;
#pragma unroll 4
        for (int d = tid % 4 * 8; d < KD; d += 32) {
            const bf8 x = la_read_hashed<KD>(q_s, r, d / 8), y = la_read_hashed<KD>(k_s, r, d / 8);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                q2 = fmaf((float)x[j], (float)x[j], q2);
                k2 = fmaf((float)y[j], (float)y[j], k2);
            }
        }
        q2 = pa_group_sum<4>(q2);
        k2 = pa_group_sum<4>(k2);
        if (tid % 4 == 0) {
            qn_s[r] = a.q_scale / sqrtf(q2 + kUnitEps);
            kn_s[r] = 1.f / sqrtf(k2 + kUnitEps);
        }
    }
    __syncthreads();
    DeltaChunk *out = reinterpret_cast<DeltaChunk *>(a.ws) + ((int64_t)b * a.chunks + chunk) * a.heads + h;
    if (tid < 64) {
        const float f = f_s[tid], last = f_s[63];
        out->k_in[tid] = exp2f(f) * kn_s[tid];
        out->q_in[tid] = exp2f(f) * qn_s[tid];
        out->k_out[tid] = exp2f(last - f) * kn_s[tid];
        if (tid == 0) out->keep = exp2f(last);
    }
    // rows t = 16 wave + l16 (as columns of the results), keys s = 16 st + 4 g + i
    f4 kk[4], qk[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) kk[st] = qk[st] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < KD / 32; ++d) {
        const bf8 bk = la_read_hashed<KD>(k_s, 16 * wave + l16, 4 * d + g), bq = la_read_hashed<KD>(q_s, 16 * wave + l16, 4 * d + g);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (st > wave) continue;
            const bf8 x = la_read_hashed<KD>(k_s, 16 * st + l16, 4 * d + g);
            kk[st] = la_mfma(x, bk, kk[st]);
            qk[st] = la_mfma(x, bq, qk[st]);
        }
    }
    __syncthreads();
    const int t = 16 * wave + l16;
    const float ft = f_s[t], bt = beta_s[t] * kn_s[t], qt = qn_s[t];
    f4 c[4];
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int s = 16 * st + 4 * g + i;
            const float w = s <= t ? __builtin_amdgcn_exp2f(ft - f_s[s]) * kn_s[s] : 0.f;
            mat[t][s] = s < t ? kk[st][i] * w * bt : 0.f;
            c[st][i] = qk[st][i] * w * qt;
        }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half && wave < 2) continue;
        const LaSplit x = la_split_pair(c[2 * half], c[2 * half + 1]);
        *reinterpret_cast<bf8 *>(out->c[0][delta_piece(wave, half)][lane]) = x.high();
        *reinterpret_cast<bf8 *>(out->c[1][delta_piece(wave, half)][lane]) = x.low();
    }
    // (the wave's own 16 rows of mat: its accesses are in order, the compiler must keep them so)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // diagonal block: column l16 of the inverse, row after row
    const int d0 = 16 * wave;
    if (lane < 16) {
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float y = i == l16 ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < i; ++j) y = fmaf(-mat[d0 + i][d0 + j], x[j], y);
            x[i] = y;
            inv[d0 + i][d0 + l16] = y;
        }
    }
    __syncthreads();
    // block (i, j), i - j = level: -inv_ii (sum over j <= k < i of mat_ik inv_kj)
    for (int level = 1; level < 4; ++level) {
        const int j = wave, i = wave + level;
        if (i < 4) {
            f4 x = f4{0.f, 0.f, 0.f, 0.f};
            for (int k = j; k < i; ++k)
#pragma unroll
                for (int q = 0; q < 4; ++q) x = delta_mfma32(mat[16 * i + l16][16 * k + 4 * q + g], inv[16 * k + 4 * q + g][16 * j + l16], x);
#pragma unroll
            for (int e = 0; e < 4; ++e) part[wave][4 * g + e][l16] = x[e];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            f4 y = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 4; ++q) y = delta_mfma32(inv[16 * i + l16][16 * i + 4 * q + g], part[wave][4 * q + g][l16], y);
#pragma unroll
            for (int e = 0; e < 4; ++e) inv[16 * i + 4 * g + e][16 * j + l16] = -y[e];
        }
        __syncthreads();
    }
    for (int i = tid; i < kDeltaPieces * 64; i += 256) {
        const int f = i / 64, tt = f < 4 ? f : f - 2, half = f / 4, r = 16 * tt + l16, col = 32 * half + 4 * g;
        f4 x, y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = 2 * half <= tt ? inv[r][col + e] * beta_s[col + e] : 0.f;
            y[e] = 2 * half < tt ? inv[r][col + 16 + e] * beta_s[col + 16 + e] : 0.f;
        }
        const LaSplit z = la_split_pair(x, y);
        *reinterpret_cast<bf8 *>(out->t[0][f][lane]) = z.high();
        *reinterpret_cast<bf8 *>(out->t[1][f][lane]) = z.low();
    }
}

// ------------------------------------------------------------------ chunks: the walk
// Bound by the chain of one wave per SIMD: the products of a chunk take a quarter of it, 64 KB through the compute unit's 64 bytes
// a cycle another seventh.  So operands are read a step ahead of their products, and the next tile's loads are spread over the
// chunk, in the order in which they are written to LDS.  A second set of tiles, written while the first is read, gave nothing (the
// walk then lacks registers).  8 prompts of 700 .. 4000 rows, 16 heads of 128 x 128: 273 -> 187 us; eight waves a workgroup, whose
// SIMDs have two each: 32 prompts of about 900 rows, with the first pass, 324 -> 311.
template <int KD, int COLS> constexpr size_t delta_walk_lds() {
    return (size_t)(2 * 64 * KD + 64 * (COLS + kLaPadV) + 2 * kDeltaMat) * 2 + 3 * 64 * 4 + 64;
}

// KD: dim padded to 64, 128 or 256.  A workgroup of NW waves owns 16 NW value columns of a head and all chunks of a portion.
template <int KD, int NW> __global__ __launch_bounds__(64 * NW, KD == 64 && NW == 4 ? 2 : 1) void delta_walk_kernel(const DeltaArgs a) {
    constexpr int kCols = 16 * NW, kThr = 64 * NW, kLv = kCols + kLaPadV;
    constexpr int kBlocks = 16 * (KD / 4), kKB = (kBlocks + kThr - 1) / kThr;  // 4 x 4 blocks of K, of V; 16-byte pieces of T and C
    constexpr bool kFew = NW < 8;  // a SIMD has one wave: all its registers
    constexpr int kVB = 16 * (kCols / 4) / kThr, kMB = 2 * kDeltaMat / 8 / kThr;
    constexpr int kSteps = kFew && KD > 64 ? 1 : 2;  // parts of the next chunk's loads beside a product of 32 columns
    static_assert(16 * (kCols / 4) % kThr == 0 && (kBlocks % kThr == 0 || kKB == 1) && 2 * kDeltaMat / 8 % kThr == 0, "whole passes");
    const bool k_live = kBlocks >= kThr || (int)threadIdx.x < kBlocks;
    extern __shared__ __align__(16) char lds[];
    __bf16 *q_s = reinterpret_cast<__bf16 *>(lds), *k_s = q_s + 64 * KD, *v_s = k_s + 64 * KD;
    __bf16 *m_s = v_s + 64 * kLv;  // T, C
    float *rows = reinterpret_cast<float *>(m_s + 2 * kDeltaMat);  // k_in, q_in, k_out
    const __bf16 *t_s = m_s, *c_s = m_s + kDeltaMat;
    const int h = blockIdx.x, v0 = blockIdx.y * kCols, b = blockIdx.z;
    DeltaPortion p;
    if (!delta_portion(a, b, p)) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), vw = wave * 16, l16 = tid & 15, g = (tid & 63) >> 4;
    // S: tile dt holds d = 16 dt + 4 g + i, v = v0 + vw + l16
    f4 s[KD / 16];
    const int64_t state_elems = (int64_t)a.dp * a.vp;
    float *pool = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * state_elems : nullptr;
    const int v = v0 + vw + l16;
    const uint32_t soff = v < a.vp ? (uint32_t)(4 * g * a.vp + v) * 4u : kLaOutside;
    {
        const float *from = p.pos0 > 0 ? pool : nullptr;
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void *)(from ? from : a.state), 0, from ? (int)state_elems * 4 : 0, 0x00020000);
#pragma unroll
        for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s[dt][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src, soff + (16 * dt + i) * a.vp * 4, 0, 0));
    }
    const int grp = h / a.per_group;
    const uint16_t *uq = reinterpret_cast<const uint16_t *>(a.q) + p.row0 * a.ldq + grp * a.dim;
    const uint16_t *uk = reinterpret_cast<const uint16_t *>(a.k) + p.row0 * a.ldk + grp * a.dim;
    const uint16_t *uv = reinterpret_cast<const uint16_t *>(a.v) + p.row0 * a.ldv + h * a.vdim + v0;
    const int vcols = a.vdim - v0 < kCols ? a.vdim - v0 : kCols;
    const DeltaChunk *mats = reinterpret_cast<const DeltaChunk *>(a.ws) + (int64_t)b * a.chunks * a.heads + h;
    LaBlock qb[kKB], kb[kKB], vb[kVB];
    la_u4 mb[kMB];
    float keep_next = 0.f, row_g0 = 0.f, row_g1 = 0.f, row_g2 = 0.f;
    // (with too few registers places in memory are worked out again: 48 heads of 128 x 128, 8 prompts of 900 .. 1000 rows, 257 us, else
    // 328; of 64 x 128, which has them, 216, else 225)
    auto again = [](int x) { return kFew || KD == 64 ? x : la_again(x); };
    // Tiles in eight parts: loads all at once would hold up a wave for longer than it computes.
    auto fetch = [&](int part, int r0) {
        if (r0 >= p.n) return;
        const int ft = again(tid);
        const int nr = p.n - r0 < 64 ? p.n - r0 : 64;
        const DeltaChunk *m = mats + (int64_t)(r0 / 64) * a.heads;
        if (part < 2) {
#pragma unroll
            for (int i = 0; i < kMB; ++i) {
                if (i * 2 / kMB != part) continue;
                mb[i] = reinterpret_cast<const la_u4 *>(m)[ft + kThr * i];
            }
        } else if (part < 6) {
            const bool keys = part < 4;
            const int64_t ld = keys ? a.ldk : a.ldq;
            const __amdgpu_buffer_rsrc_t tile = keys ? la_tile(uk + r0 * ld, ld, nr, a.dim) : la_tile(uq + r0 * ld, ld, nr, a.dim);
#pragma unroll
            for (int i = 0; i < kKB; ++i) {
                if (i * 2 / kKB != part % 2) continue;
                const int blk = ft + kThr * i, r = blk / (KD / 4) * 4, c = blk % (KD / 4) * 4;
                (keys ? kb : qb)[i] = la_load_block(tile, k_live ? la_block_off(ld, r, c, a.dim) : kLaOutside, (uint32_t)ld * 2u);
            }
        } else if (part == 6) {
            const __amdgpu_buffer_rsrc_t tv = la_tile(uv + r0 * a.ldv, a.ldv, nr, vcols);
#pragma unroll
            for (int i = 0; i < kVB; ++i) {
                const int blk = ft + kThr * i, r = blk / (kCols / 4) * 4, c = blk % (kCols / 4) * 4;
                vb[i] = la_load_block(tv, la_block_off(a.ldv, r, c, vcols), (uint32_t)a.ldv * 2u);
            }
        } else {
            row_g0 = m->k_in[ft & 63];
            row_g1 = m->q_in[ft & 63];
            row_g2 = m->k_out[ft & 63];
            keep_next = m->keep;
        }
    };
#pragma unroll
    for (int part = 0; part < 8; ++part) fetch(part, 0);
    for (int r0 = 0; r0 < p.n; r0 += 64) {
        const int lt = again(tid);  // (written in the order of loading)
        const int nv = p.n - r0 < 64 ? p.n - r0 : 64;
#pragma unroll
        for (int i = 0; i < kMB; ++i) reinterpret_cast<la_u4 *>(m_s)[lt + kThr * i] = mb[i];
#pragma unroll
        for (int i = 0; i < kKB; ++i) {
            const int blk = lt + kThr * i, r = blk / (KD / 4) * 4, c = blk % (KD / 4) * 4;
            if (!k_live) continue;
            la_put_paired<KD>(kb[i], r, c, k_s);
            la_put_paired<KD>(qb[i], r, c, q_s);
        }
#pragma unroll
        for (int i = 0; i < kVB; ++i) {
            const int blk = lt + kThr * i, r = blk / (kCols / 4) * 4, c = blk % (kCols / 4) * 4;
            la_put_block(vb[i], r, c, v_s, kLv);
        }
        if (lt < 64) {
            rows[lt] = row_g0;
            rows[64 + lt] = row_g1;
            rows[128 + lt] = row_g2;
        }
        const float keep = keep_next;
        __syncthreads();
        const int lr = again(tid) & 63, l16 = lr & 15, g = lr >> 4;
        // K S (rows t = 16 tt + 4 g + i, columns v) and, transposed, Q S (v = 4 g + i of the wave's columns, t = 16 tt + l16).
        // Operands are read a step ahead of their products: nothing else covers the wait, a SIMD has this one wave.
        f4 u[4], o[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) u[tt] = o[tt] = f4{0.f, 0.f, 0.f, 0.f};
        bf8 xk[2][4], xq[2][4], th[4], tl[4], th2[2], tl2[2];
        f4 ki[4];
        la_bf4 vv[4];
        float qi[4];
        auto ahead = [] {
            if constexpr (kFew) __builtin_amdgcn_sched_barrier(0);
        };
        auto read_rows = [&](int dd) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                xk[dd & 1][tt] = la_read_paired<KD>(k_s, 16 * tt + l16, l16, dd, g);
                xq[dd & 1][tt] = la_read_paired<KD>(q_s, 16 * tt + l16, l16, dd, g);
            }
        };
        auto mat = [&](const __bf16 *m, int term, int tt, int kk) { return delta_operand(m, term, tt, kk, lr); };
        read_rows(0);
#pragma unroll
        for (int dd = 0; dd < KD / 32; ++dd) {
            if (dd + 1 < KD / 32) {
                read_rows(dd + 1);
            } else {
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    ki[tt] = *reinterpret_cast<const f4 *>(rows + 16 * tt + 4 * g);
                    vv[tt] = la_read_tr(v_s + (16 * tt + 4 * g + l16 / 4) * kLv + vw + l16 % 4 * 4);
                    qi[tt] = rows[64 + 16 * tt + l16];
                }
            }
#pragma unroll
            for (int part = kSteps * dd; part < kSteps * (dd + 1) && part < 4; ++part) fetch(part, r0 + 64);
            ahead();
            const LaSplit sp = la_split_pair(s[2 * dd], s[2 * dd + 1]);
            const bf8 hi = sp.high(), lo = sp.low();
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                u[tt] = la_mfma(xk[dd & 1][tt], hi, u[tt]);
                o[tt] = la_mfma(hi, xq[dd & 1][tt], o[tt]);
            }
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) {
                u[tt] = la_mfma(xk[dd & 1][tt], lo, u[tt]);
                o[tt] = la_mfma(lo, xq[dd & 1][tt], o[tt]);
            }
        }
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            th[tt] = mat(t_s, 0, tt, 0);
            tl[tt] = mat(t_s, 1, tt, 0);
        }
        fetch(4, r0 + 64);
        if constexpr (!kFew) fetch(5, r0 + 64);
        ahead();
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                u[tt][i] = (float)vv[tt][i] - ki[tt][i] * u[tt][i];
                o[tt][i] *= qi[tt];
            }
        // U = T R
        f4 w[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) w[tt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            th2[tt] = mat(t_s, 0, 2 + tt, 1);
            tl2[tt] = mat(t_s, 1, 2 + tt, 1);
        }
        f4 ko[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) ko[tt] = *reinterpret_cast<const f4 *>(rows + 128 + 16 * tt + 4 * g);
        if constexpr (!kFew) fetch(6, r0 + 64);
        fetch(kFew ? 5 : 7, r0 + 64);
        ahead();
        auto times_t = [&](bf8 x, bf8 y, bf8 hi, bf8 lo, f4 &to) {
            to = la_mfma(x, hi, to);
            to = la_mfma(x, lo, to);
            to = la_mfma(y, hi, to);
        };
        const LaSplit r_lo = la_split_pair(u[0], u[1]), r_hi = la_split_pair(u[2], u[3]);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) times_t(th[tt], tl[tt], r_lo.high(), r_lo.low(), w[tt]);
        bf8 ch[4], cl[4], kt[KD / 16];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            ch[tt] = mat(c_s, 0, tt, 0);
            cl[tt] = mat(c_s, 1, tt, 0);
        }
        ahead();
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) times_t(th2[tt], tl2[tt], r_hi.high(), r_hi.low(), w[2 + tt]);
        // O += C U (transposed), S <- keep S + K^T (k_out U)
#pragma unroll
        for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[dt][i] *= keep;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
            for (int dt = 0; dt < KD / 16; ++dt) kt[dt] = la_read_paired_tr<KD>(k_s, 32 * kk, dt, l16, g);
            if constexpr (kFew) fetch(6 + kk, r0 + 64);
            ahead();
            {
                const LaSplit sp = la_split_pair(w[2 * kk], w[2 * kk + 1]);
                const bf8 hi = sp.high(), lo = sp.low();
#pragma unroll
                for (int tt = 2 * kk; tt < 4; ++tt) {
                    o[tt] = la_mfma(hi, ch[tt], o[tt]);
                    o[tt] = la_mfma(lo, ch[tt], o[tt]);
                    o[tt] = la_mfma(hi, cl[tt], o[tt]);
                }
            }
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int i = 0; i < 4; ++i) w[2 * kk + half][i] *= ko[2 * kk + half][i];
            const LaSplit sp = la_split_pair(w[2 * kk], w[2 * kk + 1]);
            const bf8 hi = sp.high(), lo = sp.low();
            if (kk == 0) {
#pragma unroll
                for (int tt = 2; tt < 4; ++tt) {
                    ch[tt] = mat(c_s, 0, tt, 1);
                    cl[tt] = mat(c_s, 1, tt, 1);
                }
            }
#pragma unroll
            for (int dt = 0; dt < KD / 16; ++dt) s[dt] = la_mfma(kt[dt], hi, s[dt]);
#pragma unroll
            for (int dt = 0; dt < KD / 16; ++dt) s[dt] = la_mfma(kt[dt], lo, s[dt]);
        }
        const int ldo = a.heads * a.vdim, c = vw + 4 * g;
        const uint16_t *first = reinterpret_cast<const uint16_t *>(a.out) + (p.row0 + r0) * (int64_t)ldo + h * a.vdim + v0;
        const __amdgpu_buffer_rsrc_t dst = la_tile(first, ldo, nv, vcols);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            const la_u2 x = {row_pack_bf16(o[tt][0], o[tt][1]), row_pack_bf16(o[tt][2], o[tt][3])};
            __builtin_amdgcn_raw_buffer_store_b64(x, dst, c < vcols ? (uint32_t)((16 * tt + l16) * ldo + c) * 2u : kLaOutside, 0, 0);
        }
        __syncthreads();  // the next chunk's tiles may be written now
    }
    if (!pool) return;
    const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc((void *)pool, 0, (int)state_elems * 4, 0x00020000);
#pragma unroll
    for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float f = s[dt][i];
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, f), dst, soff + (16 * dt + i) * a.vp * 4, 0, 0);
        }
}

// The same walk with its chain and its outputs in different waves.  What a chunk hands to the next one, K S, the system and the new state, is
// half of its products; as one wave's instructions the other half, Q S, C U, the loads and the stores, lengthen the chain by as much again.
// So waves 0 .. NW - 1 follow the state, and wave NW + w makes wave w's outputs beside it on the same SIMD: it gets the state's terms and
// U's through LDS, each lane what the same lane wrote, and the waves of that half bring the tiles.  Two barriers a chunk: until the first
// one the state's terms, T, V and Q are read (and C written), from there on U's terms and C; K, read in both parts, is there twice.
// A chunk takes 5600 cycles, about half of them before the first barrier: the waits for LDS and for the other half's products (a SIMD has 2100
// cycles of them) there, the new state and its split behind.  The loads must be out before the products of their part (behind them: 0.3 us a
// chunk); operands of T and C straight from memory, or a word of every line touched four chunks ahead, make the requests the limit (239 and
// 257 us, else 215).
// 8 prompts of 700 .. 4000 rows, 16 heads of 128 x 128, both passes and two tokens: 245 -> 215 us (one wave a SIMD -> this); 3 prompts of 326 .. 492 rows, 8
// heads of 96 x 80, 39.7 -> 32.0; 63 of 200 .. 250, 32 heads of 128 x 64, 273 -> 241.
template <int KD, int NW> constexpr size_t delta_pair_lds() {
    return (size_t)(3 * 64 * KD + 64 * (16 * NW + kLaPadV) + 2 * kDeltaMat) * 2 + (size_t)NW * (KD / 32 + 2) * 2048;
}

// KD: dim padded to 64 or 128.  A workgroup of 2 NW waves owns 16 NW value columns of a head and all chunks of a portion.  Rows come in
// 16-byte pieces (dim, vdim and strides multiples of 8, 16-byte aligned rows).
template <int KD, int NW> __global__ __launch_bounds__(128 * NW, 1) void delta_pair_kernel(const DeltaArgs a) {
    constexpr int kCols = 16 * NW, kThr = 64 * NW, kLv = kCols + kLaPadV, kD = KD / 32;
    constexpr int kKB = 64 * (KD / 8) / kThr, kVB = 64 * (kCols / 8) / kThr, kMB = kDeltaMat / 8 / kThr;  // 16-byte pieces per thread of half the workgroup
    static_assert(64 * (KD / 8) % kThr == 0 && 64 * (kCols / 8) % kThr == 0 && kDeltaMat / 8 % kThr == 0, "whole passes");
    constexpr int kTerms = 64 * 8;  // elements of an operand of a wave
    extern __shared__ __align__(16) char lds[];
    __bf16 *k2_s = reinterpret_cast<__bf16 *>(lds), *q_s = k2_s + 2 * 64 * KD, *v_s = q_s + 64 * KD;
    __bf16 *t_s = v_s + 64 * kLv, *c_s = t_s + kDeltaMat, *s_s = c_s + kDeltaMat, *u_s = s_s + NW * kD * 2 * kTerms;
    const int h = blockIdx.x, v0 = blockIdx.y * kCols, b = blockIdx.z;
    DeltaPortion p;
    if (!delta_portion(a, b, p)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = tid & 15, g = lane >> 4;
    const int pair = wave % NW, vw = pair * 16, chunks = (p.n + 63) / 64;
    // terms [pair][operand][hi, lo][lane]
    s_s += pair * kD * 2 * kTerms + lane * 8;
    u_s += pair * 2 * 2 * kTerms + lane * 8;
    auto mat = [&](const __bf16 *m, int term, int tt, int kk) { return delta_operand(m, term, tt, kk, lane); };
    const int vcols = a.vdim - v0 < kCols ? a.vdim - v0 : kCols, grp = h / a.per_group;
    const DeltaChunk *first = reinterpret_cast<const DeltaChunk *>(a.ws) + (int64_t)b * a.chunks * a.heads + h;
    auto chunk = [&](int c) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(first + (int64_t)(c < chunks ? c : chunks - 1) * a.heads), 0, sizeof(DeltaChunk), 0x00020000);
    };
    if (wave < NW) {
        __builtin_amdgcn_s_setprio(1);
        // S: tile dt holds d = 32 (dt / 2) + 8 g + 4 (dt % 2) + i (the rows of K lie in LDS as they are), v = v0 + vw + l16
        auto s_row = [](int dt, int i) { return 32 * (dt / 2) + 4 * (dt % 2) + i; };
        f4 s[KD / 16];
        const int64_t state_elems = (int64_t)a.dp * a.vp;
        float *pool = p.slot >= 0 ? a.state + (p.slot * a.heads + h) * state_elems : nullptr;
        const int v = v0 + vw + l16;
        const uint32_t soff = v < a.vp ? (uint32_t)(8 * g * a.vp + v) * 4u : kLaOutside;
        {
            const float *from = p.pos0 > 0 ? pool : nullptr;
            const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void *)(from ? from : a.state), 0, from ? (int)state_elems * 4 : 0, 0x00020000);
#pragma unroll
            for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s[dt][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src, soff + s_row(dt, i) * a.vp * 4, 0, 0));
        }
        f4 ki[4], ko[4];  // rows' factors, a chunk ahead
        float keep;
        auto four = [&](__amdgpu_buffer_rsrc_t x, size_t at, int tt) {
            return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(x, g * 16, (int)at + 64 * tt, 0));
        };
        auto fetch_in = [&](__amdgpu_buffer_rsrc_t x) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) ki[tt] = four(x, offsetof(DeltaChunk, k_in), tt);
            keep = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x, 0, (int)offsetof(DeltaChunk, keep), 0));
        };
        auto fetch_out = [&](__amdgpu_buffer_rsrc_t x) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) ko[tt] = four(x, offsetof(DeltaChunk, k_out), tt);
        };
        fetch_in(chunk(0));
        fetch_out(chunk(0));
        LaSplit sp[kD];
        auto terms = [&](int dd) {
            sp[dd] = la_split_pair(s[2 * dd], s[2 * dd + 1]);
            *reinterpret_cast<bf8 *>(s_s + dd * 2 * kTerms) = sp[dd].high();
            *reinterpret_cast<bf8 *>(s_s + dd * 2 * kTerms + kTerms) = sp[dd].low();
        };
        bf8 xk[2][4];
        auto read_k = [&](const __bf16 *k_s, int dd) {
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) xk[dd & 1][tt] = la_read_hashed<KD>(k_s, 16 * tt + l16, 4 * dd + g);
        };
#pragma unroll
        for (int dd = 0; dd < kD; ++dd) terms(dd);
        __syncthreads();
        read_k(k2_s, 0);
        for (int c = 0; c < chunks; ++c) {  // (no branches inside: loads would be moved behind them, to their use)
            const __bf16 *k_s = k2_s + (c & 1) * 64 * KD;
            // K S (rows t = 16 tt + 4 g + i, columns v)
            bf8 th[4], tl[4], th2[2], tl2[2];
            la_bf4 vv[4];
            f4 u[4];
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) u[tt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int dd = 0; dd < kD; ++dd) {
                if (dd + 1 < kD) {
                    read_k(k_s, dd + 1);
                } else {
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) vv[tt] = la_read_tr(v_s + (16 * tt + 4 * g + l16 / 4) * kLv + vw + l16 % 4 * 4);
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) {
                        th[tt] = mat(t_s, 0, tt, 0);
                        tl[tt] = mat(t_s, 1, tt, 0);
                    }
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) {
                        th2[tt] = mat(t_s, 0, 2 + tt, 1);
                        tl2[tt] = mat(t_s, 1, 2 + tt, 1);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) u[tt] = la_mfma(xk[dd & 1][tt], sp[dd].high(), u[tt]);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) u[tt] = la_mfma(xk[dd & 1][tt], sp[dd].low(), u[tt]);
            }
#pragma unroll
            for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[dt][i] *= keep;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) u[tt][i] = (float)vv[tt][i] - ki[tt][i] * u[tt][i];
            // U = T R
            f4 w[4];
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) w[tt] = f4{0.f, 0.f, 0.f, 0.f};
            auto times_t = [&](bf8 x, bf8 y, const LaSplit &r, f4 &to) {
                to = la_mfma(x, r.high(), to);
                to = la_mfma(x, r.low(), to);
                to = la_mfma(y, r.high(), to);
            };
            const LaSplit r_lo = la_split_pair(u[0], u[1]), r_hi = la_split_pair(u[2], u[3]);
            __builtin_amdgcn_sched_barrier(0);
            fetch_in(chunk(c + 1));
            bf8 kt[KD / 16];
#pragma unroll
            for (int dt = 0; dt < KD / 16; ++dt) kt[dt] = la_read_paired_tr<KD>(k_s, 0, dt, l16, g);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) times_t(th[tt], tl[tt], r_lo, w[tt]);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) times_t(th2[tt], tl2[tt], r_hi, w[2 + tt]);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) *reinterpret_cast<f4 *>(u_s + tt * kTerms) = w[tt];
            __syncthreads();
            // S <- keep S + K^T (k_out U)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                for (int half = 0; half < 2; ++half)
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[2 * kk + half][i] *= ko[2 * kk + half][i];
                const LaSplit x = la_split_pair(w[2 * kk], w[2 * kk + 1]);
                // (a group of tiles ends before the next one starts: its terms are made beside the others' products)
                constexpr int kGroup = 4;
#pragma unroll
                for (int d0 = 0; d0 < KD / 16; d0 += kGroup) {
#pragma unroll
                    for (int dt = d0; dt < d0 + kGroup; ++dt) s[dt] = la_mfma(kt[dt], x.high(), s[dt]);
#pragma unroll
                    for (int dt = d0; dt < d0 + kGroup; ++dt) s[dt] = la_mfma(kt[dt], x.low(), s[dt]);
#pragma unroll
                    for (int dt = d0; dt < d0 + kGroup; ++dt)
                        if (kk == 0) kt[dt] = la_read_paired_tr<KD>(k_s, 32, dt, l16, g);
                    if (kk == 1 && d0 == 0) {
                        read_k(k2_s + ((c + 1) & 1) * 64 * KD, 0);
                        fetch_out(chunk(c + 1));
                    }
                    if (kk == 1)
#pragma unroll
                        for (int dd = d0 / 2; dd < (d0 + kGroup) / 2; ++dd) terms(dd);
                }
            }
            __syncthreads();
        }
        if (!pool) return;
        const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc((void *)pool, 0, (int)state_elems * 4, 0x00020000);
#pragma unroll
        for (int dt = 0; dt < KD / 16; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float f = s[dt][i];
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, f), dst, soff + s_row(dt, i) * a.vp * 4, 0, 0);
            }
        return;
    }
    const int ht = tid - kThr;  // thread of this half
    const int ldo = a.heads * a.vdim;
    const uint16_t *uq = reinterpret_cast<const uint16_t *>(a.q) + p.row0 * a.ldq + grp * a.dim;
    const uint16_t *uk = reinterpret_cast<const uint16_t *>(a.k) + p.row0 * a.ldk + grp * a.dim;
    const uint16_t *uv = reinterpret_cast<const uint16_t *>(a.v) + p.row0 * a.ldv + h * a.vdim + v0;
    const uint16_t *uo = reinterpret_cast<const uint16_t *>(a.out) + p.row0 * ldo + h * a.vdim + v0;
    auto tile = [&](const uint16_t *base, int64_t ld, int c, int cols) {  // a chunk's rows; none past the last
        const int left = p.n - 64 * c, nr = left < 64 ? left : 64, bytes = ((nr - 1) * (int)ld + cols) * 2;
        return __builtin_amdgcn_make_buffer_rsrc((void *)(base + 64 * c * ld), 0, left > 0 ? bytes : 0, 0x00020000);
    };
    la_u4 kb[kKB], qb[kKB], vb[kVB], tb[kMB], cb[kMB];
    // 16-byte pieces of rows of N elements
    auto load_rows = [&](auto n, auto &x, const uint16_t *base, int64_t ld, int c, int cols) {
        constexpr int N = decltype(n)::value, COUNT = sizeof(x) / sizeof(la_u4);
        const __amdgpu_buffer_rsrc_t t = tile(base, ld, c, cols);
        const int row = ht / (N / 8), col = ht % (N / 8) * 8;
        const uint32_t off = la_block_off(ld, row, col, cols);
#pragma unroll
        for (int i = 0; i < COUNT; ++i) x[i] = __builtin_bit_cast(la_u4, __builtin_amdgcn_raw_buffer_load_b128(t, off + i * (kThr / (N / 8)) * (int)ld * 2, 0, 0));
    };
    auto put_rows = [&](const la_u4 (&x)[kKB], __bf16 *to) {
#pragma unroll
        for (int i = 0; i < kKB; ++i) {
            const int row = ht / (KD / 8) + i * (kThr / (KD / 8));
            *reinterpret_cast<la_u4 *>(to + row * KD + ((ht % (KD / 8)) ^ la_hash<KD>(row)) * 8) = x[i];
        }
    };
    auto load_k = [&](int c) { load_rows(std::integral_constant<int, KD>(), kb, uk, a.ldk, c, a.dim); };
    auto load_q = [&](int c) { load_rows(std::integral_constant<int, KD>(), qb, uq, a.ldq, c, a.dim); };
    auto load_v = [&](int c) { load_rows(std::integral_constant<int, kCols>(), vb, uv, a.ldv, c, vcols); };
    auto put_v = [&] {
#pragma unroll
        for (int i = 0; i < kVB; ++i)
            *reinterpret_cast<la_u4 *>(v_s + (ht / (kCols / 8) + i * (kThr / (kCols / 8))) * kLv + ht % (kCols / 8) * 8) = vb[i];
    };
    auto load_mat = [&](la_u4 (&x)[kMB], size_t at, int c) {
        const __amdgpu_buffer_rsrc_t t = chunk(c);
#pragma unroll
        for (int i = 0; i < kMB; ++i) x[i] = __builtin_bit_cast(la_u4, __builtin_amdgcn_raw_buffer_load_b128(t, ht * 16, (int)at + i * kThr * 16, 0));
    };
    auto put_mat = [&](const la_u4 (&x)[kMB], __bf16 *to) {
#pragma unroll
        for (int i = 0; i < kMB; ++i) reinterpret_cast<la_u4 *>(to)[ht + i * kThr] = x[i];
    };
    float qi[4], qn[4];
    auto load_q_in = [&](int c) {
        const __amdgpu_buffer_rsrc_t x = chunk(c);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
            qn[tt] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x, l16 * 4, (int)offsetof(DeltaChunk, q_in) + 64 * tt, 0));
    };
    constexpr size_t kT = offsetof(DeltaChunk, t), kC = offsetof(DeltaChunk, c);
    load_k(0);
    load_mat(tb, kT, 0);
    load_v(0);
    load_q(0);
    load_q_in(0);
    load_mat(cb, kC, 0);
    put_rows(kb, k2_s);
    put_mat(tb, t_s);
    put_v();
    put_rows(qb, q_s);
    load_k(1);
    load_mat(tb, kT, 1);
    load_v(1);
    load_q(1);
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {  // (past the last chunk: rows that are not there, the last one's matrices)
        // Q S (transposed: v = 4 g + i of the wave's columns, t = 16 tt + l16)
        f4 o[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            o[tt] = f4{0.f, 0.f, 0.f, 0.f};
            qi[tt] = qn[tt];
        }
        load_q_in(c + 1);
#pragma unroll
        for (int dd = 0; dd < kD; ++dd) {
            const bf8 hi = la_read8(s_s + dd * 2 * kTerms), lo = la_read8(s_s + dd * 2 * kTerms + kTerms);
            bf8 x[4];
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) x[tt] = la_read_hashed<KD>(q_s, 16 * tt + l16, 4 * dd + g);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) o[tt] = la_mfma(hi, x[tt], o[tt]);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) o[tt] = la_mfma(lo, x[tt], o[tt]);
        }
        put_mat(cb, c_s);
        put_rows(kb, k2_s + ((c + 1) & 1) * 64 * KD);
        load_mat(cb, kC, c + 1);
        load_k(c + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[tt][i] *= qi[tt];
        __syncthreads();
        put_mat(tb, t_s);
        put_v();
        put_rows(qb, q_s);
        load_mat(tb, kT, c + 2);
        load_v(c + 2);
        load_q(c + 2);
        __builtin_amdgcn_sched_barrier(0);
        // O += C U, and out
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const LaSplit u = la_split_pair(*reinterpret_cast<const f4 *>(u_s + 2 * kk * kTerms), *reinterpret_cast<const f4 *>(u_s + (2 * kk + 1) * kTerms));
            const bf8 hi = u.high(), lo = u.low();
#pragma unroll
            for (int tt = 2 * kk; tt < 4; ++tt) {
                const bf8 x = mat(c_s, 0, tt, kk), y = mat(c_s, 1, tt, kk);
                o[tt] = la_mfma(hi, x, o[tt]);
                o[tt] = la_mfma(lo, x, o[tt]);
                o[tt] = la_mfma(hi, y, o[tt]);
            }
        }
        const __amdgpu_buffer_rsrc_t dst = tile(uo, ldo, c, vcols);
        const int col = vw + 4 * g;
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            const la_u2 x = {row_pack_bf16(o[tt][0], o[tt][1]), row_pack_bf16(o[tt][2], o[tt][3])};
            __builtin_amdgcn_raw_buffer_store_b64(x, dst, col < vcols ? (uint32_t)((16 * tt + l16) * ldo + col) * 2u : kLaOutside, 0, 0);
        }
        __syncthreads();
    }
}

template <int KD, int NW> int launch_walk(const DeltaArgs &a, int batch, hipStream_t s) {
    constexpr size_t lds = delta_walk_lds<KD, 16 * NW>();
    static_assert(lds <= 160 * 1024, "LDS of one compute unit");
    if (int rc = la_big_lds(delta_walk_kernel<KD, NW>, lds, "pa_delta")) return rc;
    delta_walk_kernel<KD, NW><<<dim3((unsigned)a.heads, (unsigned)((a.vdim + 16 * NW - 1) / (16 * NW)), (unsigned)batch), dim3(64 * NW), lds, s>>>(a);
    PA_CHECK_LAUNCH("pa_delta (chunks)");
    return PA_OK;
}

template <int KD, int NW> int launch_pair(const DeltaArgs &a, int batch, hipStream_t s) {
    constexpr size_t lds = delta_pair_lds<KD, NW>();
    static_assert(lds <= 160 * 1024, "LDS of one compute unit");
    if (int rc = la_big_lds(delta_pair_kernel<KD, NW>, lds, "pa_delta")) return rc;
    delta_pair_kernel<KD, NW><<<dim3((unsigned)a.heads, (unsigned)((a.vdim + 16 * NW - 1) / (16 * NW)), (unsigned)batch), dim3(128 * NW), lds, s>>>(a);
    PA_CHECK_LAUNCH("pa_delta (chunks)");
    return PA_OK;
}

bool delta_pieces_of_16(const DeltaArgs &a) {
    return a.dim % 8 == 0 && a.vdim % 8 == 0 && a.ldq % 8 == 0 && a.ldk % 8 == 0 && a.ldv % 8 == 0 &&
           (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v) & 15u) == 0;
}

template <int KD> int launch_delta_chunks(const DeltaArgs &a, int batch, hipStream_t s) {
    delta_prepare_kernel<KD><<<dim3((unsigned)a.heads, (unsigned)a.chunks, (unsigned)batch), dim3(256), 0, s>>>(a);
    PA_CHECK_LAUNCH("pa_delta (triangular systems)");
    // the widest slices of the value columns that leave no compute unit without one
    const int64_t heads = (int64_t)batch * a.heads;
    // (at dim 256 four waves' registers hold the state and the next chunk)
    if constexpr (KD == 256) {
        return launch_walk<KD, 4>(a, batch, s);
    } else {
        if (a.vdim > 64 && heads * ((a.vdim + 127) / 128) >= la_cus()) return launch_walk<KD, 8>(a, batch, s);
        const bool four = a.vdim > 32 && heads * ((a.vdim + 63) / 64) >= la_cus();
        const int cols = four ? 64 : 32;
        if (delta_pieces_of_16(a) && la_delta_pairs(heads * ((a.vdim + cols - 1) / cols), (KD == 64) == four ? 2 : 1, four, batch, a.chunks, a.n_rows, la_cus()))
            return four ? launch_pair<KD, 4>(a, batch, s) : launch_pair<KD, 2>(a, batch, s);
        return four ? launch_walk<KD, 4>(a, batch, s) : launch_walk<KD, 2>(a, batch, s);
    }
}

// (what a chunk takes in the interface: two whole matrices of two terms and 1 KB, of which the walk's order leaves a quarter unused)
constexpr size_t kDeltaChunkBytes = 4 * 64 * 64 * 2 + 1024;
static_assert(sizeof(DeltaChunk) <= kDeltaChunkBytes && sizeof(DeltaChunk) % 16 == 0, "a chunk's room");
size_t delta_ws_bytes(int batch, int heads, int max_q_len) { return (size_t)batch * heads * ((max_q_len + 63) / 64) * kDeltaChunkBytes; }

template <typename T> void launch_delta_recurrent(const DeltaArgs &a, int batch, hipStream_t s) {
    const dim3 grid((unsigned)((a.vdim + kDeltaCols - 1) / kDeltaCols), (unsigned)a.heads, (unsigned)batch), block(256);
    if (a.dim <= 64) delta_recurrent_kernel<T, 4><<<grid, block, 0, s>>>(a);
    else if (a.dim <= 128) delta_recurrent_kernel<T, 8><<<grid, block, 0, s>>>(a);
    else delta_recurrent_kernel<T, 16><<<grid, block, 0, s>>>(a);
}

}  // namespace

extern "C" size_t pa_delta_workspace_bytes(int batch, int num_heads, int dim, int vdim, int max_q_len) {
    pa_clear_error();
    if (batch < 0 || num_heads <= 0 || dim <= 0 || vdim <= 0 || max_q_len < 0) {
        pa_fail(PA_ERR_INVALID_ARG, "pa_delta_workspace_bytes: sizes out of range");
        return 0;
    }
    return dim > 256 ? 0 : delta_ws_bytes(batch, num_heads, max_q_len);
}

extern "C" int pa_delta(const void *q, int64_t q_stride, const void *k, int64_t k_stride, const void *v, int64_t v_stride,
                        int heads_per_group, const void *decay_logits, const void *beta_logits, int64_t gate_stride,
                        const float *decay_bias, const float *decay_rate, float q_scale, int64_t n_rows, float *state,
                        int64_t state_rows, const int32_t *ctx_lens, const int32_t *q_lens, const int32_t *q_starts,
                        const int32_t *state_slots, int batch, int max_q_len, void *out, int num_heads, int dim, int vdim,
                        int dtype, void *workspace, size_t workspace_bytes, void *stream) {
    pa_clear_error();
    PA_REQUIRE(n_rows >= 0 && batch >= 0 && state_rows >= 0 && max_q_len >= 0, "pa_delta: a count is negative");
    PA_REQUIRE(num_heads > 0 && dim > 0 && vdim > 0, "pa_delta: heads / dim / vdim must be positive");
    PA_REQUIRE(heads_per_group > 0 && num_heads % heads_per_group == 0, "heads_per_group=%d does not divide num_heads=%d",
               heads_per_group, num_heads);
    PA_REQUIRE(num_heads <= 65535 && batch <= 65535, "pa_delta: heads=%d / batch=%d above 65535", num_heads, batch);
    if (dtype != PA_F32 && dtype != PA_BF16) return pa_fail(PA_ERR_UNSUPPORTED, "pa_delta: dtype=%d is not F32 or BF16", dtype);
    if (dim > 256) return pa_fail(PA_ERR_UNSUPPORTED, "pa_delta: dim=%d above 256", dim);
    const int groups = num_heads / heads_per_group;
    PA_REQUIRE(q_stride >= (int64_t)groups * dim && k_stride >= (int64_t)groups * dim && v_stride >= (int64_t)num_heads * vdim &&
                   gate_stride >= num_heads, "pa_delta: a stride is shorter than its row");
    PA_REQUIRE((int64_t)num_heads * (dim + vdim) <= 0x7fffffff, "pa_delta: rows are too long");
    PA_REQUIRE((q_lens == nullptr) == (q_starts == nullptr), "pa_delta: q_lens and q_starts come together");
    if (n_rows == 0 || batch == 0 || (q_lens && max_q_len == 0)) return PA_OK;
    PA_REQUIRE(q && k && v && decay_logits && beta_logits && decay_bias && decay_rate && state && ctx_lens && state_slots && out,
               "pa_delta: NULL argument");
    PA_REQUIRE(q_lens || n_rows >= batch, "n_rows=%lld below batch=%d", (long long)n_rows, batch);
    PA_REQUIRE(pa_aligned16(state), "pa_delta: the state must be 16-byte aligned");
    DeltaArgs a{};
    a.q = q; a.k = k; a.v = v; a.ldq = q_stride; a.ldk = k_stride; a.ldv = v_stride; a.per_group = heads_per_group;
    a.ga = decay_logits; a.gb = beta_logits; a.ldg = gate_stride; a.bias = decay_bias; a.rate = decay_rate; a.q_scale = q_scale;
    a.n_rows = n_rows; a.state = state; a.state_rows = state_rows; a.ctx_lens = ctx_lens; a.q_lens = q_lens;
    a.q_starts = q_starts; a.state_slots = state_slots; a.out = out; a.heads = num_heads; a.dim = dim; a.vdim = vdim;
    a.dp = la_pad16(dim); a.vp = la_pad16(vdim);
    hipStream_t s = (hipStream_t)stream;
    // (single rows, 32-bit rows, rows that are not whole 8-byte vectors, rows too far apart for 32-bit offsets go one by one)
    const uintptr_t at = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out;
    const int64_t most = 1 << 22;
    if (q_lens && dtype == PA_BF16 && workspace && workspace_bytes >= delta_ws_bytes(batch, num_heads, max_q_len) && pa_aligned16(workspace) &&
        dim % 4 == 0 && vdim % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 && (at & 7u) == 0 && q_stride <= most &&
        k_stride <= most && v_stride <= most && (int64_t)num_heads * vdim <= most && (max_q_len + 63) / 64 <= 65535) {
        a.ws = (char *)workspace;
        a.chunks = (max_q_len + 63) / 64;
        return dim <= 64 ? launch_delta_chunks<64>(a, batch, s) : dim <= 128 ? launch_delta_chunks<128>(a, batch, s) : launch_delta_chunks<256>(a, batch, s);
    }
    if (dtype == PA_F32) launch_delta_recurrent<float>(a, batch, s);
    else launch_delta_recurrent<pa_bf16>(a, batch, s);
    PA_CHECK_LAUNCH("pa_delta");
    return PA_OK;
}
