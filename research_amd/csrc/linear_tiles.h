// What the chunked linear-recurrence kernels share: 64-row tiles of bf16 rows loaded in 4 x 4 blocks and laid out in LDS
// so that operands are whole reads in either direction, 32-bit factors as a sum of two bf16 terms, states as buffers.
#pragma once
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
// transposed as well (which took the conflicting 8-byte writes of a 64-row tile and its space in LDS).  Operand reads (16 rows,
// one chunk) and transposing reads (four rows, four chunks) both spread over the banks.
__host__ __device__ constexpr int la_paired(int c) { return (c & ~31) | (c & 12) << 1 | (c & 16) >> 2 | (c & 3); }
template <int KD> __device__ __forceinline__ int la_hash(int r) { return (KD == 64 ? (r & 2) << 1 : (r & 3) << 2) | (r >> 2 & 3); }

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

// silu of a raw pair, packed again
__device__ __forceinline__ uint32_t la_silu2(uint32_t w) {
    return row_pack_bf16(row_silu<pa_bf16>(__builtin_bit_cast(float, w << 16)),
                         row_silu<pa_bf16>(__builtin_bit_cast(float, w & 0xffff0000u)));
}

template <bool ACT> __device__ __forceinline__ void la_act_block(LaBlock &b) {
    if constexpr (ACT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) b.r[i] = make_uint2(la_silu2(b.r[i].x), la_silu2(b.r[i].y));
    }
}
// The block, or with ACT its silu, to a row-major tile, and to a paired one
template <bool ACT> __device__ __forceinline__ void la_put_block(LaBlock b, int s, int c, __bf16 *rm, int ld_rm) {
    la_act_block<ACT>(b);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2 *>(rm + (s + i) * ld_rm + c) = b.r[i];
}
template <bool ACT, int KD> __device__ __forceinline__ void la_put_paired(LaBlock b, int r, int c, __bf16 *tile) {
    la_act_block<ACT>(b);
    const int e = la_paired(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2 *>(tile + (r + i) * KD + (((e >> 3) ^ la_hash<KD>(r + i)) << 3) + (e & 4)) = b.r[i];
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

// Which piece a workgroup of a chunked kernel takes.  Workgroups go to the dies, and there to groups of compute units, in the order
// of their ids, and wait for the one whose turn it is.  With 16 heads or 32 a segment fills its turn by itself, and a portion's
// segments follow each other (8 portions of 400 .. 4000 rows, lightning, 16 heads of 128 x 128: 151 us, with sequences side by side
// 211).  With fewer the places of the last segments, which only long portions have, would come to the same units each time (5
// portions of 1100 .. 2400 rows in 4 segments, 4 heads of 256 x 512, mLSTM 274 us, with sequences side by side 153): so heads and
// value slices lie side by side, then sequences, and the last segments behind all others.  A single sequence's slices of one
// segment, which read the same keys, share a die (15999 rows: 236 us, else 245).
struct LaPlace {
    int h, vsl, b, seg;
};
__host__ __device__ __forceinline__ bool la_by_portion(int heads, int batch, int segments) { return segments == 1 || batch == 1 || heads % 16 == 0; }
__device__ __forceinline__ LaPlace la_place(int segments, int slices, int batch) {
    const int h = blockIdx.x, y = blockIdx.y, z = blockIdx.z;
    return la_by_portion(gridDim.x, batch, segments) ? LaPlace{h, y / segments, z, y % segments} : LaPlace{h, y % slices, y / slices, z};
}
inline dim3 la_grid(int heads, int slices, int batch, int segments) {  // (segments > 1: batch and vdim are bounded by their workspace)
    return la_by_portion(heads, batch, segments) ? dim3((unsigned)heads, (unsigned)(slices * segments), (unsigned)batch)
                                                 : dim3((unsigned)heads, (unsigned)(slices * batch), (unsigned)segments);
}

constexpr int kLaPitchA = 72;  // bf16 per row of the decayed scores

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
