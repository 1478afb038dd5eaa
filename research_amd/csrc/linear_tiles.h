// What the chunked linear-recurrence kernels share: 64-row tiles of bf16 rows loaded in 4 x 4 blocks and laid out in LDS
// so that operands are whole reads in either direction, 32-bit factors as a sum of two bf16 terms, states as buffers.
#pragma once
#include <type_traits>
#include "lightning_plan.h"
#include "row_common.h"

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 la_bf4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t la_u2 __attribute__((ext_vector_type(2)));
typedef uint32_t la_u4 __attribute__((ext_vector_type(4)));

// x, as a value that the compiler knows nothing of: places in LDS that follow from it are worked out again in every chunk
// instead of kept in registers over the loop.
__device__ __forceinline__ int la_again(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// LDS tiles of Q and K: [64][KD], columns paired, 16-byte chunk c of row r at position c ^ la_hash(r).  Operands that meet a
// result as their partner have the inner order 4 g + 0 .. 3, 16 + 4 g + 0 .. 3 within 32: stored in that order, a lane's
// eight elements are one chunk, and four rows of a result's columns are one transposing read, so that no tile is stored
// transposed as well (which took the conflicting 8-byte writes of a 64-row tile and its space in LDS).
// A 16-byte read is served in four groups of lanes, 0 .. 3, 12 .. 15, 20 .. 27 and the rest of 0 .. 31, and the same of 32 .. 63: it takes 4
// cycles where a group's places spread over 256 bytes, else 8.  For an operand (lane: row lane % 16, chunk lane / 16) that is rows 0 .. 3
// and 12 .. 15 of a chunk beside rows 4 .. 11 of the next, hence the minus in la_hash; rows at a pitch of 32 modulo 64 bytes spread too.
// An 8-byte read is served to lanes 0 .. 31 and 32 .. 63: four-row reads of rows 32 modulo 64 bytes apart take 2 cycles, else 4.
// (8 prompts of 700 .. 4000 rows, us, with both in their way -> without: lightning 142.4 -> 139.9, delta rule 255.4 -> 250.1, HGRN2 466.0 -> 460.5;
// mLSTM, 15999 rows, 255.8 -> 253.4.)
__host__ __device__ constexpr int la_paired(int c) { return (c & ~31) | (c & 12) << 1 | (c & 16) >> 2 | (c & 3); }
template <int KD> __device__ __forceinline__ int la_hash(int r) { return (KD == 64 ? (r & 2) << 1 : (r & 3) << 2) | (-(r >> 2) & 3); }

__device__ __forceinline__ f4 la_mfma(bf8 x, bf8 y, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0); }

__device__ __forceinline__ bf8 la_read8(const __bf16 *p) { return *reinterpret_cast<const bf8 *>(p); }
__device__ __forceinline__ bf8 la_join(la_bf4 x, la_bf4 y) { return bf8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}; }
__device__ __forceinline__ bf8 la_read44(const __bf16 *p, const __bf16 *q) {
    return la_join(*reinterpret_cast<const la_bf4 *>(p), *reinterpret_cast<const la_bf4 *>(q));
}
// Lane i of 16 gets column i of four rows from a 4 x 16 block in LDS whose lane s points at row s / 4, columns 4 (s % 4) ..
__device__ __forceinline__ la_bf4 la_read_tr(const __bf16 *p) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(la_bf4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s4 __attribute__((address_space(3))) *)p));
}
// Pairs x = hi + lo, packed bf16
__device__ __forceinline__ void la_split2(float x0, float x1, uint32_t &hi, uint32_t &lo) {
    hi = row_pack_bf16(x0, x1);
    asm("" : "+v"(hi));  // (else the compiler converts x0 once more by itself for `hi << 16`: seven instructions a pair instead of six)
    lo = row_pack_bf16(x0 - __builtin_bit_cast(float, hi << 16), x1 - __builtin_bit_cast(float, hi & 0xffff0000u));
}
struct LaSplit {  // eight values as two operands
    uint32_t hi[4], lo[4];
    __device__ __forceinline__ bf8 high() const { return __builtin_bit_cast(bf8, la_u4{hi[0], hi[1], hi[2], hi[3]}); }
    __device__ __forceinline__ bf8 low() const { return __builtin_bit_cast(bf8, la_u4{lo[0], lo[1], lo[2], lo[3]}); }
};

struct LaBlock {  // four rows of four consecutive columns, raw bf16
    uint2 r[4];
};

// A tile of `rows` rows (none: 0 or less) of `cols` columns at row stride `ld` as a buffer: loads past its end give zeros,
// stores past it are dropped.  (Columns past `cols` inside a row are the caller's: it gives such lanes the offset kLaOutside.)
constexpr uint32_t kLaOutside = 0x40000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t la_tile(const uint16_t *base, int64_t ld, int rows, int cols) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, rows > 0 ? (int)(((rows - 1) * ld + cols) * 2) : 0, 0x00020000);
}
// Byte offset of the 4 x 4 block at (row s, column c)
__device__ __forceinline__ uint32_t la_block_off(int64_t ld, int s, int c, int cols) {
    return c < cols ? (uint32_t)(s * ld + c) * 2u : kLaOutside;
}
__device__ __forceinline__ LaBlock la_load_block(__amdgpu_buffer_rsrc_t tile, uint32_t off, uint32_t row_bytes) {
    LaBlock b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const la_u2 x = __builtin_amdgcn_raw_buffer_load_b64(tile, off + i * row_bytes, 0, 0);
        b.r[i] = make_uint2(x[0], x[1]);
    }
    return b;
}

// 16-byte pieces of rows `apart` rows apart from (row, column c) on.  wide: cols a multiple of 8 and rows 16-byte aligned; else in halves
// (cols a multiple of 4, 8-byte aligned).
template <int N> __device__ __forceinline__ void la_load_pieces(la_u4 (&x)[N], __amdgpu_buffer_rsrc_t tile, int64_t ld, int row, int c, int apart, int cols, bool wide) {
    const uint32_t off = la_block_off(ld, row, c, cols), step = (uint32_t)apart * (uint32_t)ld * 2u;
    if (wide) {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = __builtin_bit_cast(la_u4, __builtin_amdgcn_raw_buffer_load_b128(tile, off + i * step, 0, 0));
    } else {
        const uint32_t off2 = la_block_off(ld, row, c + 4, cols);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const la_u2 lo = __builtin_amdgcn_raw_buffer_load_b64(tile, off + i * step, 0, 0), hi = __builtin_amdgcn_raw_buffer_load_b64(tile, off2 + i * step, 0, 0);
            x[i] = la_u4{lo[0], lo[1], hi[0], hi[1]};
        }
    }
}

// silu of a raw pair, packed again
__device__ __forceinline__ uint32_t la_silu2(uint32_t w) {
    return row_pack_bf16(row_silu<pa_bf16>(__builtin_bit_cast(float, w << 16)),
                         row_silu<pa_bf16>(__builtin_bit_cast(float, w & 0xffff0000u)));
}

// The block to a row-major tile, and to a paired one
__device__ __forceinline__ void la_put_block(const LaBlock &b, int s, int c, __bf16 *rm, int ld_rm) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2 *>(rm + (s + i) * ld_rm + c) = b.r[i];
}
template <int KD> __device__ __forceinline__ void la_put_paired(const LaBlock &b, int r, int c, __bf16 *tile) {
    const int e = la_paired(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2 *>(tile + (r + i) * KD + (((e >> 3) ^ la_hash<KD>(r + i)) << 3) + (e & 4)) = b.r[i];
}
// The same without pairs: chunk c of row r at c ^ la_hash(r)
template <int KD> __device__ __forceinline__ void la_put_hashed(const LaBlock &b, int r, int c, __bf16 *tile) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2 *>(tile + (r + i) * KD + (((c >> 3) ^ la_hash<KD>(r + i)) << 3) + (c & 4)) = b.r[i];
}
template <int KD> __device__ __forceinline__ bf8 la_read_hashed(const __bf16 *tile, int row, int chunk) {
    return la_read8(tile + row * KD + (chunk ^ la_hash<KD>(row)) * 8);
}
// The same places as bytes: a lane's place for the first 32 columns (of row `row`, of which a multiple of 16 may be added later; `low`: which
// of their four chunks), and for the 32 columns number dd.  What follows from one place is one exclusive or, not an address kept for each.
template <int KD> __device__ __forceinline__ int la_place_of(int row, int low) { return row * (KD * 2) + ((low ^ la_hash<KD>(row)) << 4); }
template <int KD> __device__ __forceinline__ int la_place_at(int place, int dd) { return (place ^ (dd & 3) << 6) + (dd >> 2 << 8); }
template <int KD> __device__ __forceinline__ bf8 la_read_place(const __bf16 *tile, int place, int row, int dd) {
    return *reinterpret_cast<const bf8 *>(reinterpret_cast<const char *>(tile) + la_place_at<KD>(place, dd) + row * (KD * 2));
}
// Four rows, then four 16 further on, of column 8 (lane / 4 % 4) + 4 (dt % 2) + lane % 4 of the 32 number dt / 2: an operand whose partner's rows
// are a lane's two result tiles in a row.  place: la_place_of(4 g + l16 / 4, l16 % 4)
template <int KD> __device__ __forceinline__ bf8 la_read_place_tr(const __bf16 *tile, int place, int row, int dt) {
    const __bf16 *at = reinterpret_cast<const __bf16 *>(reinterpret_cast<const char *>(tile) + la_place_at<KD>(place, dt / 2) + row * (KD * 2)) + dt % 2 * 4;
    return la_join(la_read_tr(at), la_read_tr(at + 16 * KD));
}
// Row `row` (row % 16 = l16) of a paired tile, elements of the 32 columns from 32 dd on
template <int KD> __device__ __forceinline__ bf8 la_read_paired(const __bf16 *tile, int row, int l16, int dd, int g) {
    return la_read8(tile + row * KD + ((4 * dd + g) ^ la_hash<KD>(l16)) * 8);
}
// Column 16 dt + l16 of rows first + 4 g + 0 .. 3 and first + 16 + 4 g + 0 .. 3: of a paired tile, and of a row-major one
template <int KD> __device__ __forceinline__ bf8 la_read_paired_tr(const __bf16 *tile, int first, int dt, int l16, int g) {
    const int row = 4 * g + l16 / 4;
    const __bf16 *at = tile + (first + row) * KD + ((dt / 2 * 4 + l16 % 4) ^ la_hash<KD>(row)) * 8 + dt % 2 * 4;
    return la_join(la_read_tr(at), la_read_tr(at + 16 * KD));
}
__device__ __forceinline__ bf8 la_read_rows_tr(const __bf16 *tile, int ld, int first, int col, int l16, int g) {
    const __bf16 *at = tile + (first + 4 * g + l16 / 4) * ld + col + l16 % 4 * 4;
    return la_join(la_read_tr(at), la_read_tr(at + 16 * ld));
}
// Two bf16 terms of eight values of a result tile pair, as an operand in the paired order
__device__ __forceinline__ LaSplit la_split_pair(const f4 &x, const f4 &y) {
    LaSplit s;
    la_split2(x[0], x[1], s.hi[0], s.lo[0]);
    la_split2(x[2], x[3], s.hi[1], s.lo[1]);
    la_split2(y[0], y[1], s.hi[2], s.lo[2]);
    la_split2(y[2], y[3], s.hi[3], s.lo[3]);
    return s;
}
// All 24 bits of eight values, as three terms
struct LaSplit3 {
    bf8 term[3];
};
__device__ __forceinline__ LaSplit3 la_split3(const f4 &x, const f4 &y) {
    la_u4 t[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float a = (j < 2 ? x : y)[2 * j % 4], b = (j < 2 ? x : y)[2 * j % 4 + 1];
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            t[n][j] = row_pack_bf16(a, b);
            a -= __builtin_bit_cast(float, t[n][j] << 16);
            b -= __builtin_bit_cast(float, t[n][j] & 0xffff0000u);
        }
    }
    return LaSplit3{{__builtin_bit_cast(bf8, t[0]), __builtin_bit_cast(bf8, t[1]), __builtin_bit_cast(bf8, t[2])}};
}
// Two terms of eight raw values times weights (x: rows 4 g + 0 .. 3, y: 16 further on)
__device__ __forceinline__ LaSplit la_split_weighted(bf8 raw, const f4 &x, const f4 &y) {
    const la_u4 v = __builtin_bit_cast(la_u4, raw);
    LaSplit s;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        la_split2(__builtin_bit_cast(float, v[j] << 16) * (j < 2 ? x : y)[2 * j % 4],
                  __builtin_bit_cast(float, v[j] & 0xffff0000u) * (j < 2 ? x : y)[2 * j % 4 + 1], s.hi[j], s.lo[j]);
    return s;
}

// Which piece a workgroup of a chunked kernel takes.  Workgroups go to the dies, and there to groups of compute units, in the order of
// their ids, and wait for the one whose turn it is: pieces that short portions do not have would leave some units idle and others with
// two.  So the pieces that there are get the first ids, found from the lengths (by each wave, a scan, under 1 us): first the segments
// before the portions' last ones, which have as many rows each, then the last ones, the longest first.  Heads and value slices, which
// read the same rows, lie side by side; a single portion's slices have their segments in a row instead, so that those of one segment share
// a die (15999 rows: 236 us, else 245).  us, with ids for all possible pieces by portion / by segment / this, as many segments: 8 prompts
// of 400 .. 4000 rows, mLSTM, 4 heads of 256 x 512, 230 / 175 / 144, 8 heads 432 / 283 / 271; lightning, 16 heads of 128 x 128, 115 / 115 / 83,
// of 64 x 64, 63 / 73 / 51; 12 prompts, 8 heads, 106 / 177 / 97, 16 heads 157 / 178 / 157.
struct LaPlace {
    int h, vsl, b, seg;
};
__device__ __forceinline__ int la_scan(int x, int lane) {  // inclusive sums over the wave
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    const int r0 = __builtin_amdgcn_readlane(x, 15), r1 = r0 + __builtin_amdgcn_readlane(x, 31), r2 = r1 + __builtin_amdgcn_readlane(x, 47);
    return x + (lane < 16 ? 0 : lane < 32 ? r0 : lane < 48 ? r1 : r2);
}
// Also the portion `p` (of the caller's type; all that is known of up to 64 sequences is loaded at once, as a second round of loads would
// keep every workgroup waiting).  False: nothing to do.
template <typename Args, typename Portion> __device__ __forceinline__ bool la_place(const Args &a, int slices, LaPlace &at, Portion &p) {
    int n, start, ctx, slot;
    if (a.segments == 1 || a.batch == 1) {
        const int y = a.segments == 1 ? 0 : blockIdx.x / a.heads;
        at = a.segments == 1 ? LaPlace{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, 0} : LaPlace{(int)blockIdx.x % a.heads, y / a.segments, 0, y % a.segments};
        n = a.q_lens[at.b], start = a.q_starts[at.b], ctx = a.ctx_lens[at.b], slot = a.state_slots[at.b];
    } else {
        const int lane = threadIdx.x & 63, y = blockIdx.x / a.heads;
        at.h = blockIdx.x % a.heads, at.vsl = y % slices;
        int u = y / slices, first = 0, from = -1;
        auto load = [&] {
            const int b = first + lane;
            n = start = ctx = slot = 0;
            if (b < a.batch) n = a.q_lens[b], start = a.q_starts[b], ctx = a.ctx_lens[b], slot = a.state_slots[b];
            return la_full_segments(n, a.segments, a.seg_rows);
        };
        for (; from < 0 && first < a.batch; first += 64) {
            const int full = load(), upto = la_scan(full, lane), all = __builtin_amdgcn_readlane(upto, 63);
            if (u < all) {  // (uniform)
                from = __builtin_ctzll(__ballot(upto > u));
                at.b = first + from, at.seg = u - __builtin_amdgcn_readlane(upto - full, from);
                break;
            }
            u -= all;
        }
        if (from < 0) {  // a last one: of up to 64 sequences the longest first
            if (u >= a.batch) return false;
            first = a.batch <= 64 ? 0 : u & ~63, from = u & 63;
            const int full = load(), rest = n - full * a.seg_rows;
            if (a.batch <= 64) {
                int longer = 0;
                for (int i = 0; i < a.batch; ++i) {
                    const int x = __builtin_amdgcn_readlane(rest, i);
                    longer += x > rest || (x == rest && i < lane);
                }
                from = __builtin_ctzll(__ballot(lane < a.batch && longer == u));
            }
            at.b = first + from, at.seg = __builtin_amdgcn_readlane(full, from);
        }
        n = __builtin_amdgcn_readlane(n, from), start = __builtin_amdgcn_readlane(start, from);
        ctx = __builtin_amdgcn_readlane(ctx, from), slot = __builtin_amdgcn_readlane(slot, from);
    }
    p.n = n, p.row0 = start, p.pos0 = ctx - n, p.slot = slot < a.state_rows ? slot : -1;
    return p.n > 0 && p.pos0 >= 0 && p.row0 >= 0 && p.row0 + p.n <= a.n_rows;
}
// (segments > 1: the number of workgroups is bounded by the workspace of 256 MB)
inline dim3 la_grid(int heads, int slices, int batch, int segments) {
    return segments == 1 ? dim3((unsigned)heads, (unsigned)slices, (unsigned)batch) : dim3((unsigned)heads * slices * batch * segments);
}

constexpr int kLaPitchA = 80;  // bf16 per row of the decayed scores
constexpr int kLaPadV = 16;    // bf16 behind a row of values

int la_cus() {
    static int cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        __atomic_store_n(&cached[dev], n, __ATOMIC_RELAXED);
    }
    return n;
}

template <typename K> int la_big_lds(K kernel, size_t bytes, const char *what) {
    if (bytes > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return pa_fail(PA_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
    }
    return PA_OK;
}

}  // namespace
