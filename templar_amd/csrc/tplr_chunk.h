// Chunks of (R, C) tensors and of batches of them: row loads and stores, the 2-D transform of a chunk in registers, where a
// chunk of a batch lies.  Shared by the translation units that work on 64x64 chunks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tplr_hip.h"
#include "tplr_device.h"

namespace tplr {

// =========================================================================================
// chunk loaders / storers for the (R, C) row-major side: lane = column
// =========================================================================================
// Chunk rows through buffer instructions: one resource descriptor per chunk (scalar base,
// byte range for bounds checking), the row offset r*ld in a scalar register and lane*4 as the
// only vector operand, so addressing costs no vector ALU work.  ld*4*63 must fit in 31 bits.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t chunk_rsrc(const void* chunk0, int64_t ld) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(chunk0), 0, static_cast<int>((63 * ld + 64) * 4),
                                             0x00020000);
}

template <int kRow0 = 0, int kRow1 = 64>
__device__ __forceinline__ void load_chunk_rows(float (&v)[64], const void* chunk0, int64_t ld, int lane) {
    const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(chunk0, ld);
    const int ld4 = static_cast<int>(ld) * 4;
#pragma unroll
    for (int r = kRow0; r < kRow1; ++r)
        v[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 4, r * ld4, 2));
}

// drop (wave-uniform): the stores are issued against a range of zero bytes, whose bounds check
// discards them - the instruction stream stays the same for a chunk that must not be written
__device__ __forceinline__ void store_chunk_rows(const float (&v)[64], void* chunk0, int64_t ld, int lane,
                                                 bool drop = false) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        chunk0, 0, drop ? 0 : static_cast<int>((63 * ld + 64) * 4), 0x00020000);
    const int ld4 = static_cast<int>(ld) * 4;
#pragma unroll
    for (int r = 0; r < 64; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v[r]), rs, lane * 4, r * ld4, 2);
}

__device__ __forceinline__ void load_chunk_cols(float (&v)[64], const float* __restrict__ x, int64_t ld,
                                                int64_t y, int64_t xc, int lane) {
    load_chunk_rows(v, x + (y * 64) * ld + xc * 64, ld, lane);
}

__device__ __forceinline__ void store_chunk_cols(const float (&v)[64], float* __restrict__ x, int64_t ld,
                                                 int64_t y, int64_t xc, int lane) {
    store_chunk_rows(v, x + (y * 64) * ld + xc * 64, ld, lane);
}

// forward 2-D transform of the chunk held column-per-lane; result row-per-lane:
// v[d] = coef[lane][d], and the tile is left free
// registers column-per-lane (v[r] = M[r][lane]) -> registers row-per-lane (w[c] = M[lane][c])
// through a 32-row staging buffer: rows 0..31 go first and lanes 0..31 pick theirs up, then rows
// 32..63 for lanes 32..63.  Half the LDS of a whole-chunk tile, which is what lets twice as many
// waves stay resident.
__device__ __forceinline__ void transpose_via_half(const float (&v)[64], float (&w)[64], float* buf, int lane) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int r = 0; r < kHalfRows; ++r) buf[r * kLd + lane] = v[half * kHalfRows + r];
        wave_lds_fence();
        if ((lane >> 5) == half) tile_rows_to_regs(w, buf, lane & 31);
        wave_lds_fence();
    }
}

// Forward 2-D transform of a chunk held column-per-lane (v[r] = X[r][lane]); the result is
// row-per-lane: w[d] = 32 * coef[lane][d] with the transform, X[lane][d] without.
template <bool kUseDct>
__device__ __forceinline__ void chunk_forward(float (&v)[64], float (&w)[64], float* buf, int lane) {
    if (kUseDct) dct64_fwd(v);  // along rows k: v[b] = sum_k X[k][lane] F[k][b]
    transpose_via_half(v, w, buf, lane);
    if (kUseDct) dct64_fwd(w);  // along columns l: w[d] = sum_l T[lane][l] F[l][d]
}

// inverse: tile holds coef rows; result column-per-lane v[k] = x[k][lane]
// (the tile must hold the coefficients times 2^-5: the two passes multiply by 32; kScaleInput
// applies that factor here for callers whose tile holds plain coefficients)
template <bool kUseDct, bool kScaleInput = false>
__device__ __forceinline__ void chunk_inverse(float (&v)[64], float* tile, int lane) {
    if (kUseDct) {
        tile_rows_to_regs(v, tile, lane);
        if (kScaleInput) {
#pragma unroll
            for (int d = 0; d < 64; ++d) v[d] *= kDctPow2Scale;
        }
        dct64_inv(v);  // along d: v[l] = sum_d Y[lane][d] F[l][d]
        wave_lds_fence();
        regs_to_tile_rows(v, tile, lane);
        wave_lds_fence();
    }
    tile_cols_to_regs(v, tile, lane);
    if (kUseDct) dct64_inv(v);  // along b: v[k] = sum_b Z[b][lane] F[k][b]
}

// -----------------------------------------------------------------------------------------
// Persistent kernels walk a contiguous range of the batch's chunk list.  A cursor keeps the
// current tensor's descriptor and the chunk's (y, x) position in wave-uniform registers.
// -----------------------------------------------------------------------------------------
struct Cursor {
    const tplr_tensor_desc* table;
    int n_tensors;
    int t;
    gfloat* base;
    int64_t ld;
    int64_t begin, end;  // chunk ids covered by tensor t
    int X;
    int64_t y;
    int xc;
};

// descriptor fields are the same for every lane: move them to scalar registers so that chunk
// rows are addressed as scalar base + 32-bit lane offset
__device__ __forceinline__ int64_t uniform64(int64_t x) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(x));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(static_cast<uint64_t>(x) >> 32));
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

__device__ __forceinline__ void cursor_take(Cursor& c, const tplr_tensor_desc& d) {
    c.base = (gfloat*)uniform64(reinterpret_cast<int64_t>(d.dense));
    c.ld = uniform64(d.ld);
    c.begin = uniform64(d.chunk_begin);
    c.X = __builtin_amdgcn_readfirstlane(d.x_chunks);
    c.end = c.begin + static_cast<int64_t>(c.X) * __builtin_amdgcn_readfirstlane(d.y_chunks);
}

__device__ __forceinline__ void cursor_seek(Cursor& c, const tplr_tensor_desc* table, const tplr_tensor_desc& single,
                                            int n_tensors, int64_t g) {
    c.table = table;
    c.n_tensors = n_tensors;
    c.t = 0;
    if (table) {
        int lo = 0, hi = n_tensors;  // last tensor whose chunk_begin <= g and that is not empty
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (table[mid].chunk_begin <= g)
                lo = mid;
            else
                hi = mid;
        }
        c.t = lo;
        cursor_take(c, table[lo]);
    } else {
        cursor_take(c, single);
    }
    const int64_t local = g - c.begin;
    c.y = local / c.X;
    c.xc = static_cast<int>(local - c.y * c.X);
}

// advance to chunk g (= previous chunk + 1)
__device__ __forceinline__ void cursor_next(Cursor& c, int64_t g) {
    if (++c.xc == c.X) {
        c.xc = 0;
        ++c.y;
    }
    while (g >= c.end && c.t + 1 < c.n_tensors) {  // batch mode only: single tensors never get here
        ++c.t;
        cursor_take(c, c.table[c.t]);
        c.y = 0;
        c.xc = 0;
    }
}

// the contiguous slice of [0, total) that workgroup `bid` of a grid of G (multiple of 8) owns;
// workgroups b, b+8, b+16, ... run on the same XCD and take neighbouring slices
// `align` > 1 (a power of two): where slices are long (64 items and more), the boundaries between the
// slices of one XCD fall on multiples of `align` counted from -`first`, i.e. on absolute multiples when
// [0, total) stands for the items first .. first + total - 1 of a longer list
__device__ __forceinline__ void my_range(int64_t total, int64_t& g0, int64_t& g1, int align = 1, int64_t first = 0) {
    const int64_t bid = blockIdx.x, S = gridDim.x >> 3;
    const int64_t xcd = bid & 7, slot = bid >> 3;
    const int64_t per = (total + 7) >> 3;
    const int64_t xb = xcd * per;
    int64_t xe = xb + per;
    xe = xe > total ? total : xe;
    const int64_t len = xe > xb ? xe - xb : 0;
    g0 = xb + len * slot / S;
    g1 = xb + len * (slot + 1) / S;
    if (align > 1 && len >= 64 * S) {
        if (slot > 0) g0 = ((g0 + first) & ~static_cast<int64_t>(align - 1)) - first;
        if (slot + 1 < S) g1 = ((g1 + first) & ~static_cast<int64_t>(align - 1)) - first;
        g0 = g0 < xb ? xb : g0;
        g1 = g1 < xb ? xb : g1;
    }
}

template <int kRow0 = 0, int kRow1 = 64>
__device__ __forceinline__ void load_chunk_cols(float (&v)[64], const Cursor& c, int lane) {
    load_chunk_rows<kRow0, kRow1>(v, (const void*)(c.base + (c.y * 64) * c.ld + static_cast<int64_t>(c.xc) * 64),
                                  c.ld, lane);
}

// the wave's issue priority (0 .. 3; the instruction takes an immediate, hence the ladder); `level` is wave-uniform
__device__ __forceinline__ void set_wave_priority(int level) {
    if (level == 0) __builtin_amdgcn_s_setprio(0);
    else if (level == 1) __builtin_amdgcn_s_setprio(1);
    else if (level == 2) __builtin_amdgcn_s_setprio(2);
    else __builtin_amdgcn_s_setprio(3);
}

// Where chunk g of a batch lies, for a wave that takes one chunk.  The tensor is looked up through the scalar cache, eight
// ways at a time: a set of a few hundred tensors is three trips of loads that do not wait for one another.  (Vector loads
// queue behind the compute unit's streaming ones; a binary search is a chain of eight.)
struct Place {
    gfloat* chunk0;  // the chunk's first element
    int64_t ld;
    int t;  // its tensor
};
__device__ __forceinline__ int find_tensor(const tplr_tensor_desc* __restrict__ table, int n_tensors, uint32_t g) {
    // the last tensor whose chunk_begin <= g (empty tensors share theirs with the one behind them); 2^32 chunks are 64 TB
    int lo = 0, len = n_tensors;
    while (len > 1) {  // wave-uniform
        const int step = (len + 7) >> 3;
        uint32_t begin[8];
#pragma unroll
        for (int i = 1; i < 8; ++i)  // (past the end the last one: a load behind a branch would be waited for there)
            begin[i] = static_cast<uint32_t>(table[lo + (i * step < len ? i * step : len - 1)].chunk_begin);
        int k = 0;
#pragma unroll
        for (int i = 1; i < 8; ++i) k += i * step < len && begin[i] <= g ? step : 0;
        lo += k;
        len = len - k < step ? len - k : step;
    }
    return lo;
}

__device__ __forceinline__ Place place_of(const tplr_tensor_desc* __restrict__ table, const tplr_tensor_desc& single, int n_tensors,
                                          int64_t g) {
    tplr_tensor_desc d = single;
    int t = 0;
    if (table) {  // wave-uniform
        t = find_tensor(table, n_tensors, static_cast<uint32_t>(g));
        d = table[t];
    }
    const int64_t ld = uniform64(d.ld), begin = uniform64(d.chunk_begin);
    const uint32_t X = __builtin_amdgcn_readfirstlane(d.x_chunks);
    const uint32_t local = static_cast<uint32_t>(g - begin), y = local / X, xc = local - y * X;
    gfloat* const base = (gfloat*)uniform64(reinterpret_cast<int64_t>(d.dense));
    return Place{base + static_cast<int64_t>(y) * 64 * ld + static_cast<int64_t>(xc) * 64, ld, t};
}

// ---- half a chunk in LDS: 32 rows of 64 floats, without padding.  Row r's sixteen quads of columns are permuted by r mod 16,
// so that a row per lane (16 bytes at a time) and a column per lane (4 bytes) both reach all banks.
constexpr int kHalfWords = 32 * 64;
// where coefficient e = 64 row + column of the chunk lies, counted over both halves
__device__ __forceinline__ uint32_t half_pos(uint32_t e) { return e ^ ((e >> 4) & 0x3cu); }

__device__ __forceinline__ void half_rows_to_regs(float (&w)[64], const float* tile, int row) {  // row: 0 .. 31
    const float4* r4 = reinterpret_cast<const float4*>(tile + row * 64);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        const float4 t = r4[c ^ (row & 15)];
        w[4 * c] = t.x, w[4 * c + 1] = t.y, w[4 * c + 2] = t.z, w[4 * c + 3] = t.w;
    }
}
__device__ __forceinline__ void regs_to_half_rows(const float (&w)[64], float* tile, int row) {
    float4* r4 = reinterpret_cast<float4*>(tile + row * 64);
#pragma unroll
    for (int c = 0; c < 16; ++c) r4[c ^ (row & 15)] = make_float4(w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]);
}
// v[32 half + r] = row r, column `lane`
template <int kHalf>
__device__ __forceinline__ void half_cols_to_regs(float (&v)[64], const float* tile, int lane) {
#pragma unroll
    for (int r = 0; r < 32; ++r) v[32 * kHalf + r] = tile[r * 64 + (lane ^ ((r & 15) << 2))];
}

// Where several peers sent a coefficient, its sum over its count: a lane scans the counters of half a row - four bits each,
// or eight - and divides, one coefficient per trip of a lane-divergent loop.
__device__ __forceinline__ void half_means4(float* tile, const uint32_t* cnt, int lane) {
    // bit 4 j + q of m: the counter of the lane's coefficient 8 q + j is at least two
    const uint4 w = reinterpret_cast<const uint4*>(cnt)[lane];
    auto multi = [](uint32_t c) { return ((c >> 1) | (c >> 2) | (c >> 3)) & 0x11111111u; };
    uint32_t m = multi(w.x) | multi(w.y) << 1 | multi(w.z) << 2 | multi(w.w) << 3;
    while (m) {
        const int b = __builtin_ctz(m);
        m &= m - 1;
        const uint32_t w01 = (b & 1) ? w.y : w.x, w23 = (b & 1) ? w.w : w.z;
        const uint32_t n = (((b & 2) ? w23 : w01) >> (b & 28)) & 15u;
        float* const t = &tile[lane * 32 + (b & 3) * 8 + (b >> 2)];
        *t = *t / static_cast<float>(n);
    }
}
__device__ __forceinline__ void half_means8(float* tile, const uint32_t* cnt, int lane) {  // counts up to 31
    // bit 8 j + q of m: that of coefficient 4 q + j
    uint32_t m = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint4 w = reinterpret_cast<const uint4*>(cnt)[lane * 2 + h];
        auto multi = [](uint32_t c) { return ((c >> 1) | (c >> 2) | (c >> 3) | (c >> 4)) & 0x01010101u; };
        m |= (multi(w.x) | multi(w.y) << 1 | multi(w.z) << 2 | multi(w.w) << 3) << (4 * h);
    }
    while (m) {
        const int b = __builtin_ctz(m);
        m &= m - 1;
        const int at = lane * 32 + (b & 7) * 4 + (b >> 3);
        const uint32_t n = reinterpret_cast<const uint8_t*>(cnt)[at];
        tile[at] = tile[at] / static_cast<float>(n);
    }
}

}  // namespace tplr
