// Rows of values outside the 64x64 chunk path: top-k of given rows, the 1-D parameters, scatters into rows.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tplr_hip.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

// =========================================================================================
// top-k select + pack
// =========================================================================================
// Rows of 4096: a chunk in the (Y, X, 64, 64) layout.
template <bool kTwo>
__global__ __launch_bounds__(64) void k_topk_rows(const float* __restrict__ coef, int64_t n_rows, int k,
                                                  uint8_t* __restrict__ idx12, float* __restrict__ val) {
    __shared__ __align__(16) float tile[kTileFloats];
    __shared__ uint64_t cand[kCandCap];
    const int lane = threadIdx.x;
    const int64_t row = xcd_contiguous(blockIdx.x, gridDim.x);
    if (row >= n_rows) return;
    flat_to_tile(coef + row * 4096, tile, lane);
    wave_lds_fence();
    float w[64];
    tile_rows_to_regs(w, tile, lane);
    wave_lds_fence();
    const Selected s = select_topk<kTwo>(w, tile, cand, lane, k, 1.0f);
    emit_selected<kTwo>(s, lane, k, row, idx12, val);
}

// Rows of 129 .. 4095 elements (chunks with other edges): one wave per row.  A row of n is dealt out so that every lane
// has its share of it, ceil(n / 64) neighbouring elements in the leading registers of its 64: with 64 elements per lane
// and the row in the first lanes, as it lies in memory, the lanes' maxima bound the k-th largest magnitude badly (a
// row of 400 reaches seven lanes) and the select falls back to its bitwise search.  The registers past the share hold
// zeros, one of which could be selected in place of a later zero of the row's own: a row with fewer than k values other
// than zero (and denormals, for good measure) is therefore taken as it lies.  All of a row's loads are requested before the
// first is used.  In us, k = 32: 1000 rows of 3000 7.3 (as rows of 4096, four loads at a time: 10.0), 1000 of 400 6.7 (15.9),
// 10 000 of 400 all zeros 71 (66; selecting twice 123).
template <bool kTwo>
__global__ __launch_bounds__(64) void k_topk_rows_any(const float* __restrict__ coef, int64_t n_rows, int row_len,
                                                      int k, uint8_t* __restrict__ idx12, float* __restrict__ val) {
    __shared__ __align__(16) float tile[kTileFloats];
    __shared__ uint64_t cand[kCandCap];
    const int lane = threadIdx.x;
    const int64_t row = xcd_contiguous(blockIdx.x, gridDim.x);
    if (row >= n_rows) return;
    // (elements past the row read as zero: the buffer's range check)
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(coef + row * row_len), 0, row_len * 4, 0x00020000);
    float w[64];
#pragma unroll
    for (int i = 0; i < 64; ++i)
        w[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 4, i * 256, 0));
    // a word of padding every 32: lanes `per` elements apart meet in few banks whatever `per` is
    auto pos = [](int e) { return e + (e >> 5); };
#pragma unroll
    for (int i = 0; i < 64; ++i) tile[pos(i * 64 + lane)] = w[i];
    int normal = 0;
#pragma unroll
    for (int i = 0; i < 64; i += 8)
        if (normal < k) {  // wave-uniform: most rows have them in their first 512 elements
#pragma unroll
            for (int j = i; j < i + 8; ++j) normal += __popcll(__ballot(!(__builtin_fabsf(w[j]) < 1.17549435e-38f)));
        }
    const int per = normal < k ? 64 : (row_len + 63) >> 6;  // elements per lane
    wave_lds_fence();
    // (a lane's elements past its share are its neighbour's, read and dropped; the last lanes' lie past the tile)
    const int first = lane * per;
#pragma unroll
    for (int d = 0; d < 64; ++d) {
        const int e = first + d < 4095 ? first + d : 4095;
        w[d] = d < per ? tile[pos(e)] : 0.0f;
    }
    wave_lds_fence();
    Selected s = select_topk<kTwo>(w, tile, cand, lane, k, 1.0f);
    s.idx0 = (s.idx0 >> 6) * static_cast<uint32_t>(per) + (s.idx0 & 63u);
    if (kTwo) s.idx1 = (s.idx1 >> 6) * static_cast<uint32_t>(per) + (s.idx1 & 63u);
    emit_selected<kTwo>(s, lane, k, row, idx12, val);
}

// Rows of at most 64 (kTwo: 128) elements, a 1-D parameter's: one (two) per lane, sorted as 64-bit keys (magnitude,
// 127 - index, sign) - the canonical order, as select_topk unpacks it.  Lanes past the row hold the key zero, which no
// element has while any lane is past the row.  Four rows per workgroup.  The 32 rows of a 2048-element vector take
// 3 us; as rows of 4096 mostly zeros they took 12 us.
template <bool kTwo>
__device__ __forceinline__ Selected sort_row(float x0, float x1, bool in0, bool in1) {
    const int lane = threadIdx.x & 63;
    auto key = [](float x, int ix, bool in) -> uint64_t {
        const uint32_t bits = __float_as_uint(x);
        return in ? (static_cast<uint64_t>(mag_key(bits)) << 32) | ((127u - ix) << 1) | (bits >> 31) : 0ull;
    };
    uint64_t e0 = key(x0, lane, in0), e1 = 0;
    if constexpr (kTwo) {
        e1 = key(x1, lane + 64, in1);
        sort128_desc(e0, e1, lane);
    } else {
        sort64_desc(e0, lane);
    }
    auto unpack = [](uint64_t e, uint32_t& ix, float& v) {
        const uint32_t lo = static_cast<uint32_t>(e), m = static_cast<uint32_t>(e >> 32);
        ix = 127u - ((lo >> 1) & 127u);
        v = __uint_as_float((m == 0x7fffffffu ? 0x7fc00000u : m) | (lo << 31));
    };
    Selected s;
    unpack(e0, s.idx0, s.val0);
    unpack(e1, s.idx1, s.val1);
    return s;
}

template <bool kTwo>
__global__ __launch_bounds__(256) void k_topk_short(const float* __restrict__ coef, int64_t n_rows, int row_len, int k,
                                                    uint8_t* __restrict__ idx12, float* __restrict__ val) {
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    if (row >= n_rows) return;  // wave-uniform
    const float* src = coef + row * row_len;
    const bool in0 = lane < row_len, in1 = kTwo && lane + 64 < row_len;
    const Selected s = sort_row<kTwo>(in0 ? src[lane] : 0.f, in1 ? src[lane + 64] : 0.f, in0, in1);
    emit_selected<kTwo>(s, lane, k, row, idx12, val);
}

// Any k up to the row length: the whole row sorted.  One workgroup of 256 threads per row, the row as
// 4096 keys (magnitude, 4095 - index, sign: the canonical order of select_topk, elements past the row
// as zeros at their own indices, which no real element ranks below) in LDS, a bitonic network of 78
// steps in descending order, then the k leading keys unpacked as select_topk unpacks its candidates.
// Not a fast path: it serves selections larger than the register-resident select holds (k > 128).
__global__ __launch_bounds__(256) void k_topk_rows_sorted(const float* __restrict__ coef, int64_t n_rows, int row_len,
                                                          int k, uint8_t* __restrict__ idx12, float* __restrict__ val) {
    __shared__ uint64_t keys[4096];
    const int tid = threadIdx.x;
    const int64_t row = xcd_contiguous(blockIdx.x, gridDim.x);
    if (row >= n_rows) return;  // (the whole workgroup)
    const float* src = coef + row * row_len;
    for (int e = tid; e < 4096; e += 256) {
        const uint32_t bits = e < row_len ? __float_as_uint(src[e]) : 0u;
        keys[e] = (static_cast<uint64_t>(mag_key(bits)) << 32) | ((4095u - static_cast<uint32_t>(e)) << 1) | (bits >> 31);
    }
    __syncthreads();
    for (int size = 2; size <= 4096; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = tid; i < 2048; i += 256) {
                const int pos = 2 * i - (i & (stride - 1));
                const uint64_t a = keys[pos], b = keys[pos + stride];
                const bool down = (pos & size) == 0;  // this run is sorted in descending order
                if ((a < b) == down) {
                    keys[pos] = b;
                    keys[pos + stride] = a;
                }
            }
            __syncthreads();
        }
    }
    float* vrow = val + row * k;
    uint8_t* irow = idx12 + row * (k + (k >> 1));
    for (int j = tid; j < (k >> 1); j += 256) {
        uint32_t ix[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint64_t e = keys[2 * j + h];
            const uint32_t lo = static_cast<uint32_t>(e), key = static_cast<uint32_t>(e >> 32);
            ix[h] = 4095u - ((lo >> 1) & 4095u);
            const uint32_t mag = key == 0x7fffffffu ? 0x7fc00000u : key;
            vrow[2 * j + h] = __uint_as_float(mag | (lo << 31));
        }
        const uint32_t w = ix[0] | (ix[1] << 12);
        irow[3 * j] = static_cast<uint8_t>(w);
        irow[3 * j + 1] = static_cast<uint8_t>(w >> 8);
        irow[3 * j + 2] = static_cast<uint8_t>(w >> 16);
    }
}

// The 64-point transform of kRowsPerWave rows of 64 elements per wave: the wave's rows staged through its part of the
// tile, a row per lane in registers, `keep` receives the tile row by row (stride kLd).  One pass is sqrt(32) times
// the orthonormal transform.
// 1-D parameters are few and short (a model's norm vectors are a thousand rows), so what counts is the chain of one
// wave: four rows per wave (one 16-byte load per lane) where that leaves no SIMD with more than a few waves, 64 rows
// (every lane a transform of its own) for long ones.
template <int kRowsPerWave>
__device__ __forceinline__ void load_rows(const gfloat* src, int64_t left, float* tile, int lane) {
    constexpr int kQ = kRowsPerWave * 16;  // 16-byte pieces
#pragma unroll
    for (int c = 0; c < (kQ + 63) / 64; ++c) {
        const int q = c * 64 + lane, r = q >> 4;
        v4f x = {0.f, 0.f, 0.f, 0.f};
        if (q < kQ && r < left) x = *reinterpret_cast<const __attribute__((address_space(1))) v4f*>(src + q * 4);
        if (q < kQ) *reinterpret_cast<v4f*>(tile + r * kLd + ((q & 15) << 2)) = x;
    }
    wave_lds_fence();
}

template <int kRowsPerWave>
__device__ __forceinline__ void transform_rows(float* tile, int lane, int inverse) {
    if (lane < kRowsPerWave) {
        float v[64];
        tile_rows_to_regs(v, tile, lane);
        if (inverse)
            dct64_inv(v);
        else
            dct64_fwd(v);
#pragma unroll
        for (int d = 0; d < 64; ++d) v[d] *= 0.17677669529663687f;
        regs_to_tile_rows(v, tile, lane);
    }
    wave_lds_fence();
}

template <int kRowsPerWave>
__global__ __launch_bounds__(64) void k_dct1d(const float* __restrict__ in, int64_t n_vec, int inverse,
                                              float* __restrict__ out) {
    __shared__ __align__(16) float tile[kRowsPerWave * kLd];
    const int lane = threadIdx.x;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kRowsPerWave;
    const int64_t left = n_vec - base;
    load_rows<kRowsPerWave>((const gfloat*)in + base * 64, left, tile, lane);
    transform_rows<kRowsPerWave>(tile, lane, inverse);
#pragma unroll
    for (int c = 0; c < (kRowsPerWave * 16 + 63) / 64; ++c) {
        const int q = c * 64 + lane, r = q >> 4;
        if (r < kRowsPerWave && r < left)
            reinterpret_cast<float4*>(out + base * 64)[q] = *reinterpret_cast<const float4*>(tile + r * kLd + ((q & 15) << 2));
    }
}

// The 1-D parameters of a set (norm vectors), every tensor a run of rows of 64 elements: transform,
// top-k and pack of all of them in one launch, each tensor read where it lies.  Two forms, the same bits (of a NaN but
// for its payload); the launcher's rule says where each is the faster one.
//
// The tensor that group `grp` of the set belongs to (tensor t has ceil(rows / 64) groups), `grp` becoming the group within
// it: one load per lane and a prefix sum over the tensors' group counts - a scan of the table is a chain of dependent
// loads, and took longer than the rest of the launch.  false where the set has no such group.
__device__ __forceinline__ bool find_group(const tplr_tensor_desc* __restrict__ table, int n_tensors, int lane, int& t, int& grp) {
    for (int t0 = 0; t0 < n_tensors; t0 += 64) {  // (64 tensors a turn)
        const uint32_t groups = t0 + lane < n_tensors ? static_cast<uint32_t>((table[t0 + lane].x_chunks + 63) >> 6) : 0u;
        const uint32_t incl = wave_incl_scan_u32(groups);
        const uint64_t behind = __ballot(incl > static_cast<uint32_t>(grp));
        if (behind) {
            const int at = __builtin_ctzll(behind);
            grp -= static_cast<int>(__builtin_amdgcn_readlane(incl - groups, at));
            t = t0 + at;
            return true;
        }
        grp -= static_cast<int>(__builtin_amdgcn_readlane(incl, 63));
    }
    return false;
}

// A wave takes four rows of one tensor: the transform and its scale exactly as k_dct1d applies them, then each row sorted
// across the lanes.  What bounds it is the chain of one wave, which is short.  The 25 norm vectors of a 150M model (300
// rows) take 8.3 us, in the other form 9.7 us.
template <bool kUseDct>
__global__ __launch_bounds__(256) void k_encode_rows(const tplr_tensor_desc* __restrict__ table, int n_tensors, int64_t first_group,
                                                     int k, uint8_t* __restrict__ idx12, float* __restrict__ val) {
    constexpr int kPerWave = 4, kPerGroup = 64 / (4 * kPerWave);  // workgroups per group of 64 rows
    __shared__ __align__(16) float tile_all[4][kPerWave * kLd];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    float* const tile = tile_all[wv];
    int t, grp = static_cast<int>(first_group + blockIdx.x / kPerGroup);
    if (!find_group(table, n_tensors, lane, t, grp)) return;
    const tplr_tensor_desc d = table[t];
    const int first = grp * 64 + (static_cast<int>(blockIdx.x % kPerGroup) * 4 + wv) * kPerWave;  // this wave's first row
    const int left = d.x_chunks - first;
    if (left <= 0) return;  // wave-uniform
    load_rows<kPerWave>((const gfloat*)d.dense + static_cast<int64_t>(first) * 64, left, tile, lane);
    if (kUseDct) transform_rows<kPerWave>(tile, lane, 0);
    const int64_t row = d.chunk_begin + first;
#pragma unroll
    for (int r = 0; r < kPerWave; ++r) {
        const Selected s = sort_row<false>(tile[r * kLd + lane], 0.f, true, false);
        if (r < left) emit_selected<false>(s, lane, k, row + r, idx12, val);
    }
}

// A wave takes 64 rows of one tensor, a row per lane: every lane transforms its own, sorts its 64 coefficients in
// registers with a bitonic network and writes its row's payload, the k leading indices and their values fetched back from
// the tile.  No lane idles in the transform and the network needs no exchange between lanes; what bounds it is its stores,
// 2.5 k of them a row and each to a line of its own, and that a short set leaves most SIMDs without a wave.
template <bool kUseDct>
__global__ __launch_bounds__(64) void k_encode_rows_lane(const tplr_tensor_desc* __restrict__ table, int n_tensors,
                                                         int64_t first_group, int k, uint8_t* __restrict__ idx12,
                                                         float* __restrict__ val) {
    __shared__ __align__(16) float tile[64 * kLd];
    const int lane = threadIdx.x;
    int t, grp = static_cast<int>(first_group + blockIdx.x);
    if (!find_group(table, n_tensors, lane, t, grp)) return;
    const tplr_tensor_desc d = table[t];
    const int left = d.x_chunks - grp * 64;  // rows from this group's first to the tensor's end
    load_rows<64>((const gfloat*)d.dense + static_cast<int64_t>(grp) * 4096, left, tile, lane);
    float w[64];
    tile_rows_to_regs(w, tile, lane);
    if (kUseDct) {  // (as transform_rows, with the result kept)
        dct64_fwd(w);
#pragma unroll
        for (int d = 0; d < 64; ++d) w[d] *= 0.17677669529663687f;
    }
    wave_lds_fence();
    regs_to_tile_rows(w, tile, lane);
    // Keys (magnitude bits, 63 - index) ordered as unsigned 64-bit integers - held as doubles: for positive,
    // normal, finite doubles the two orders are the same, and a compare-exchange is then one v_max_f64 and one
    // v_min_f64.  One is added to the exponent field so that a zero magnitude is a normal double, and NaNs share
    // a magnitude key just below where that addition would reach the doubles' own infinities and NaNs.
    double key[64];
#pragma unroll
    for (int e = 0; e < 64; ++e) {
        const uint32_t a = __builtin_bit_cast(uint32_t, w[e]) & 0x7fffffffu;
        const uint32_t mag = (a > 0x7f800000u ? 0x7fdfffffu : a) + 0x00100000u;
        key[e] = __builtin_bit_cast(double, (static_cast<uint64_t>(mag) << 32) | static_cast<uint32_t>(63 - e));
    }
    // bitonic sort, descending
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int i = 0; i < 64; ++i) {
                const int l = i ^ stride;
                if (l > i) {
                    const bool up = (i & size) != 0 && size < 64;  // this run ascends
                    const double a = key[i], b = key[l];
                    const double hi = __builtin_fmax(a, b), lo = __builtin_fmin(a, b);
                    key[i] = up ? lo : hi;
                    key[l] = up ? hi : lo;
                }
            }
        }
    }
    wave_lds_fence();
    if (lane >= left) return;
    const int64_t row = d.chunk_begin + static_cast<int64_t>(grp) * 64 + lane;
    float* vrow = val + row * k;
    uint8_t* irow = idx12 + row * (k + (k >> 1));
    const float* mine = tile + lane * kLd;
#pragma unroll
    for (int j = 0; j < 64; j += 2) {
        if (j < k) {  // k is even
            const uint32_t i0 = 63u - static_cast<uint32_t>(__builtin_bit_cast(uint64_t, key[j]));
            const uint32_t i1 = 63u - static_cast<uint32_t>(__builtin_bit_cast(uint64_t, key[j + 1]));
            vrow[j] = mine[i0];
            vrow[j + 1] = mine[i1];
            const uint32_t pair = i0 | (i1 << 12);
            uint8_t* o = irow + 3 * (j >> 1);
            o[0] = static_cast<uint8_t>(pair);
            o[1] = static_cast<uint8_t>(pair >> 8);
            o[2] = static_cast<uint8_t>(pair >> 16);
        }
    }
}

// =========================================================================================
// scatters into rows
// =========================================================================================
// One peer's packed rows into zeroed rows of any length (decompress of chunks with other edges), at most 64 entries a
// row: a workgroup of four waves clears a row in LDS, its first wave adds the entries (one per lane, requested before
// the clearing), all store it, 16 bytes a lane where rows align.  An entry's slot first takes its lane's number: a lane
// that reads back another's has met a repeated index (no top-k makes them), and that row's entries are then gathered
// by their first lane, in entry order, and averaged - what scatter_reduce_ "mean" leaves (src/tplr/compress.py:472-474).
// 1000 rows of 3000 take 8.3 us, a wave per row 9.5 us; with a counter per element and every lane compared with every
// other for each row 13.6 us.
template <bool kVec>
__global__ __launch_bounds__(256) void k_scatter_rows_packed(const uint8_t* __restrict__ idx12, const float* __restrict__ val,
                                                             int k, int row_len, int reduce_mode, float* __restrict__ out,
                                                             int32_t* __restrict__ err, int32_t* __restrict__ flag) {
    __shared__ __align__(16) float acc[TPLR_MAX_ROW];
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t row = blockIdx.x;
    int me = -1;
    float a = 0.f;
    if (tid < k) {  // (k <= 64: the first wave)
        me = static_cast<int>(load_idx12((const gbyte*)idx12 + row * (k + (k >> 1)), tid));
        a = val[row * k + tid];
    }
#pragma unroll
    for (int q = 0; q < TPLR_MAX_ROW / 1024; ++q)
        reinterpret_cast<float4*>(acc)[q * 256 + tid] = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    if (tid < 64) {
        if (me >= row_len) {
            if (err) atomicMax(err, me);
            if (flag) *flag = 1;  // (pinned host memory: a plain store)
            me = -1;
        }
        if (me >= 0) acc[me] = __uint_as_float(static_cast<uint32_t>(lane));
        wave_lds_fence();
        const bool clash = me >= 0 && __float_as_uint(acc[me]) != static_cast<uint32_t>(lane);
        if (__ballot(clash) != 0) {  // wave-uniform
            float sum = 0.f, n = 0.f;
            bool first = true;
            for (int i = 0; i < 64; ++i) {
                const int other = __shfl(me, i);
                const float x = __shfl(a, i);
                if (other == me) {
                    first = first && i >= lane;
                    sum += x;
                    n += 1.f;
                }
            }
            if (me >= 0 && first) acc[me] = (reduce_mode == TPLR_REDUCE_MEAN && n > 1.f) ? sum / n : sum;
        } else if (me >= 0) {
            acc[me] = 0.f + a;
        }
    }
    __syncthreads();
    float* orow = out + row * row_len;
    if (kVec) {
#pragma unroll
        for (int q = 0; q < TPLR_MAX_ROW / 1024; ++q)
            if (q * 256 + tid < row_len / 4)
                reinterpret_cast<float4*>(orow)[q * 256 + tid] = reinterpret_cast<const float4*>(acc)[q * 256 + tid];
    } else {
#pragma unroll
        for (int i = 0; i < TPLR_MAX_ROW / 256; ++i)
            if (i * 256 + tid < row_len) orow[i * 256 + tid] = acc[i * 256 + tid];
    }
}

// Does every one of n_pairs packed pairs of indices lie below row_len?  Every workgroup takes a run of them and tells the host in
// a word of pinned memory of its own (1: no) while the scatter behind it still runs: the caller has to know before it returns,
// and waiting for the scatter itself left the device idle until the next call's launch (20 us of the 66 us that a 3000 x 1000
// parameter took there and back).  A few workgroups: their words cross to the host one by one.  1000 rows of 32 entries 3 us.
__global__ __launch_bounds__(1024) void k_check_rows(const uint8_t* __restrict__ idx12, int64_t n_pairs, int row_len,
                                                     uint32_t* __restrict__ words) {
    __shared__ uint32_t wave_max[16];
    const int64_t p0 = n_pairs * blockIdx.x / gridDim.x;
    n_pairs = n_pairs * (blockIdx.x + 1) / gridDim.x - p0;
    const int tid = threadIdx.x;
    uint32_t most = 0;
    auto take = [&](uint32_t pair) {
        const uint32_t a = pair & 0xfffu, b = (pair >> 12) & 0xfffu;
        most = a > most ? a : most;
        most = b > most ? b : most;
    };
    const gbyte* src = (const gbyte*)idx12 + 3 * p0;
    const int64_t quads = n_pairs >> 2;  // four pairs are twelve bytes
#pragma unroll 4
    for (int64_t q = tid; q < quads; q += 1024) {
        const uint32_t w0 = *(const gu32*)(src + 12 * q), w1 = *(const gu32*)(src + 12 * q + 4), w2 = *(const gu32*)(src + 12 * q + 8);
        take(w0), take(w0 >> 24 | w1 << 8), take(w1 >> 16 | w2 << 16), take(w2 >> 8);
    }
    if (tid < (n_pairs & 3)) {
        const gbyte* p = src + 3 * (4 * quads + tid);
        take(p[0] | static_cast<uint32_t>(p[1]) << 8 | static_cast<uint32_t>(p[2]) << 16);
    }
    most = wave_max_u32(most);
    if ((tid & 63) == 0) wave_max[tid >> 6] = most;
    __syncthreads();
    if (tid < 64) {
        most = wave_max_u32(wave_max[tid & 15]);
        if (tid == 0)
            __hip_atomic_store(words + blockIdx.x, most < static_cast<uint32_t>(row_len) ? 0u : 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// generic rows (unpacked indices, more than 64 entries a row): exact source-order accumulation
__global__ __launch_bounds__(64) void k_scatter_rows(const uint8_t* __restrict__ idx12,
                                                     const int64_t* __restrict__ idx64,
                                                     const float* __restrict__ val, int64_t k_per_row,
                                                     int row_len, int reduce_mode, float* __restrict__ out,
                                                     int32_t* __restrict__ err) {
    __shared__ float acc[TPLR_MAX_ROW];
    __shared__ uint32_t cnt[TPLR_MAX_ROW];
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    for (int i = lane; i < row_len; i += 64) {
        acc[i] = 0.f;
        cnt[i] = 0;
    }
    __syncthreads();
    const uint8_t* irow = idx12 ? idx12 + row * (k_per_row + (k_per_row >> 1)) : nullptr;
    for (int64_t j0 = 0; j0 < k_per_row; j0 += 64) {
        const int64_t j = j0 + lane;
        int64_t ix = -1;
        float a = 0.f;
        if (j < k_per_row) {
            ix = idx12 ? static_cast<int64_t>(load_idx12(irow, static_cast<int>(j))) : idx64[row * k_per_row + j];
            a = val[row * k_per_row + j];
            if (ix < 0 || ix >= row_len) {
                if (err) atomicMax(err, ix < 0 || ix > 0x7fffffff ? 0x7fffffff : static_cast<int32_t>(ix));
                ix = -1;
            }
        }
        // rank among earlier lanes of this batch that hit the same destination
        const int me = static_cast<int>(ix);
        int rank = 0;
        for (int i = 0; i < 63; ++i) {
            const int other = __shfl(me, i);
            rank += (i < lane && other == me && me >= 0) ? 1 : 0;
        }
        int maxrank = rank;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(maxrank, off);
            maxrank = o > maxrank ? o : maxrank;
        }
        for (int r = 0; r <= maxrank; ++r) {
            if (me >= 0 && rank == r) {
                acc[me] += a;
                cnt[me] += 1;
            }
            __syncthreads();
        }
    }
    float* orow = out + row * row_len;
    for (int i = lane; i < row_len; i += 64) {
        const uint32_t c = cnt[i];
        const float s = acc[i];
        orow[i] = (reduce_mode == TPLR_REDUCE_MEAN && c > 1) ? s / static_cast<float>(c) : s;
    }
}

}  // namespace tplr

using namespace tplr;

extern "C" {

int tplr_dct1d(const float* d_in, int64_t n_vec, int inverse, float* d_out, void* stream) {
    if (n_vec < 0) return TPLR_E_BADARG;
    if (n_vec == 0) return 0;
    if (!d_in || !d_out) return TPLR_E_BADARG;
    // four rows per wave up to four waves per SIMD of the device, 64 beyond (see load_rows)
    if (n_vec <= 16384)
        hipLaunchKernelGGL(k_dct1d<4>, dim3(static_cast<unsigned>((n_vec + 3) / 4)), dim3(64), 0,
                           static_cast<hipStream_t>(stream), d_in, n_vec, inverse, d_out);
    else
        hipLaunchKernelGGL(k_dct1d<64>, dim3(static_cast<unsigned>((n_vec + 63) / 64)), dim3(64), 0,
                           static_cast<hipStream_t>(stream), d_in, n_vec, inverse, d_out);
    return launch_status();
}

int tplr_topk_pack(const float* d_coef, int64_t n_rows, int64_t row_len, int k, uint8_t* d_idx12,
                   float* d_val, void* stream) {
    if (n_rows < 0 || row_len < 1 || k < 2 || (k & 1) || k > row_len) return TPLR_E_BADARG;
    if (row_len > TPLR_MAX_ROW) return TPLR_E_TOOMANY;
    if (n_rows == 0) return 0;
    if (!d_coef || !d_idx12 || !d_val) return TPLR_E_BADARG;
    const int rl = static_cast<int>(row_len);
    if (rl <= 128) {
        const dim3 grid(static_cast<unsigned>((n_rows + 3) / 4)), block(256);
        if (rl <= 64)
            hipLaunchKernelGGL(k_topk_short<false>, grid, block, 0, static_cast<hipStream_t>(stream), d_coef, n_rows, rl, k,
                               d_idx12, d_val);
        else
            hipLaunchKernelGGL(k_topk_short<true>, grid, block, 0, static_cast<hipStream_t>(stream), d_coef, n_rows, rl, k,
                               d_idx12, d_val);
        return launch_status();
    }
    if (k > kCandCap)
        hipLaunchKernelGGL(k_topk_rows_sorted, dim3(grid8(n_rows)), dim3(256), 0, static_cast<hipStream_t>(stream),
                           d_coef, n_rows, rl, k, d_idx12, d_val);
    else if (rl < 4096)
        hipLaunchKernelGGL(k > 32 ? k_topk_rows_any<true> : k_topk_rows_any<false>, dim3(grid8(n_rows)), dim3(64), 0,
                           static_cast<hipStream_t>(stream), d_coef, n_rows, rl, k, d_idx12, d_val);
    else
        hipLaunchKernelGGL(k > 32 ? k_topk_rows<true> : k_topk_rows<false>, dim3(grid8(n_rows)), dim3(64), 0,
                           static_cast<hipStream_t>(stream), d_coef, n_rows, k, d_idx12, d_val);
    return launch_status();
}

int tplr_encode_rows_batch(const tplr_tensor_desc* d_desc, int n_tensors, int64_t total_groups, int k, int use_dct,
                           uint8_t* d_idx12, float* d_val, void* stream) {
    if (!d_desc || n_tensors < 1 || total_groups < 0 || !d_idx12 || !d_val || k < 2 || (k & 1) || k > 64)
        return TPLR_E_BADARG;
    if (total_groups == 0) return 0;
    if (total_groups > 0x7fffffff) return TPLR_E_TOOMANY;
    // Four rows a wave : a row a lane, in us.  With the transform 16 384 rows (256 groups) k = 2 10.5 : 8.8, k = 32 11.0 : 11.4;
    // 24 576 rows k = 32 15.8 : 13.4, k = 48 16.2 : 17.6; 65 536 rows k = 2 32.5 : 9.6, k = 48 33.9 : 31.0, k = 64 34.7 : 38.7; 2^20
    // rows k = 2 474 : 198, k = 48 489 : 473.  Few groups leave most compute units' instruction caches cold, which
    // costs the four-row form more: 8 tensors of 16 rows k = 32 10.5 : 9.6, 16 groups 9.9 : 9.6 - but 32 groups 9.3 : 9.7, 25
    // tensors of 12 rows 8.3 : 9.7, 8192 rows 7.9 : 10.2, a single row 6.1 : 8.6.  Without the transform 16 384 rows k = 2 7.2 : 7.5,
    // 24 576 rows k = 2 9.2 : 7.7, k = 24 9.8 : 10.3, 65 536 rows k = 24 19.6 : 15.6, k = 32 19.9 : 20.1, 2^20 rows k = 24 243 : 265.
    const int64_t n = total_groups;
    const int most = !use_dct ? (n > 256 ? 24 : 0) : n >= 1024 ? 48 : n >= 384 ? 32 : n >= 256 ? 24 : n >= 2 && n <= 16 ? 32 : 0;
    if (k <= most) {
        constexpr int64_t kPiece = 4 * kMaxGroups256;  // groups of one launch: 64 threads each
        for (int64_t g = 0; g < total_groups; g += kPiece) {
            const int64_t count = total_groups - g < kPiece ? total_groups - g : kPiece;
            hipLaunchKernelGGL(use_dct ? k_encode_rows_lane<true> : k_encode_rows_lane<false>, dim3(static_cast<unsigned>(count)), dim3(64),
                               0, static_cast<hipStream_t>(stream), d_desc, n_tensors, g, k, d_idx12, d_val);
        }
        return launch_status();
    }
    constexpr int64_t kPiece = kMaxGroups256 / 4;  // groups of one launch: four workgroups of 256 threads each
    for (int64_t g = 0; g < total_groups; g += kPiece) {
        const int64_t count = total_groups - g < kPiece ? total_groups - g : kPiece;
        hipLaunchKernelGGL(use_dct ? k_encode_rows<true> : k_encode_rows<false>, dim3(static_cast<unsigned>(count * 4)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), d_desc, n_tensors, g, k, d_idx12, d_val);
    }
    return launch_status();
}

// (a workgroup of 256 per row, and a launch has fewer than 2^32 threads: more rows than kMaxGroups256 go in several)
static int scatter_packed(const uint8_t* d_idx12, const float* d_val, int64_t n_rows, int k, int row_len, int reduce_mode,
                          float* d_out, int32_t* d_err, int32_t* flag, void* stream) {
    const bool vec = (row_len & 3) == 0 && (reinterpret_cast<uintptr_t>(d_out) & 15) == 0;
    for (int64_t r = 0; r < n_rows; r += kMaxGroups256) {
        const int64_t rows = n_rows - r < kMaxGroups256 ? n_rows - r : kMaxGroups256;
        hipLaunchKernelGGL(vec ? k_scatter_rows_packed<true> : k_scatter_rows_packed<false>, dim3(static_cast<unsigned>(rows)),
                           dim3(256), 0, static_cast<hipStream_t>(stream), d_idx12 + r * (k + (k >> 1)), d_val + r * k, k, row_len,
                           reduce_mode, d_out + r * row_len, d_err, flag);
    }
    return launch_status();
}

int tplr_decompress_rows(const uint8_t* d_idx12, const float* d_val, int64_t n_rows, int k, int64_t row_len, float* d_out,
                         int32_t* flag, void* stream) {
    if (!d_idx12 || !d_val || !d_out || n_rows < 0 || row_len < 1 || k < 2) return TPLR_E_BADARG;
    if (k & 1) return TPLR_E_ODD;
    if (k > 64 || row_len > TPLR_MAX_ROW || n_rows > 0x7fffffff) return TPLR_E_TOOMANY;
    if (n_rows == 0) return 0;
    return scatter_packed(d_idx12, d_val, n_rows, k, static_cast<int>(row_len), TPLR_REDUCE_MEAN, d_out, nullptr, flag, stream);
}

int tplr_check_rows(const uint8_t* d_idx12, int64_t n_rows, int k, int64_t row_len, uint32_t* words, int n_words, void* stream) {
    if (!d_idx12 || !words || n_words < 1 || n_words > 65535 || n_rows < 1 || k < 2 || row_len < 1) return TPLR_E_BADARG;
    if (k & 1) return TPLR_E_ODD;
    if (row_len > TPLR_MAX_ROW) return TPLR_E_TOOMANY;
    hipLaunchKernelGGL(k_check_rows, dim3(static_cast<unsigned>(n_words)), dim3(1024), 0, static_cast<hipStream_t>(stream), d_idx12, n_rows * (k / 2),
                       static_cast<int>(row_len), words);
    return launch_status();
}

int tplr_scatter_rows(const uint8_t* d_idx12, const int64_t* d_idx64, const float* d_val, int64_t n_rows,
                      int64_t k_per_row, int64_t row_len, int reduce_mode, float* d_out, int32_t* d_err,
                      void* stream) {
    if (n_rows < 0 || k_per_row < 0 || row_len < 1 || (!d_idx12 == !d_idx64) || !d_val || !d_out ||
        (reduce_mode != TPLR_REDUCE_MEAN && reduce_mode != TPLR_REDUCE_SUM))
        return TPLR_E_BADARG;
    if (d_idx12 && (k_per_row & 1)) return TPLR_E_ODD;
    if (row_len > TPLR_MAX_ROW) return TPLR_E_TOOMANY;
    if (n_rows == 0) return 0;
    if (d_idx12 && k_per_row <= 64) {
        return scatter_packed(d_idx12, d_val, n_rows, static_cast<int>(k_per_row), static_cast<int>(row_len), reduce_mode, d_out,
                              d_err, nullptr, stream);
    }
    hipLaunchKernelGGL(k_scatter_rows, dim3(static_cast<unsigned>(n_rows)), dim3(64), 0,
                       static_cast<hipStream_t>(stream), d_idx12, d_idx64, d_val, k_per_row,
                       static_cast<int>(row_len), reduce_mode, d_out, d_err);
    return launch_status();
}

}  // extern "C"
