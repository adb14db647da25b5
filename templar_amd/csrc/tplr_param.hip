// One parameter's payloads into its chunks: what the reference's per-parameter calls batch_decompress and decompress
// leave before the transform (src/tplr/compress.py:425-580), a chunk spread over the four waves of a workgroup.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/tplr_hip.h"
#include "tplr_chunk.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

constexpr int kParamPeers = 24;  // payloads of one launch
constexpr int kParamNorms = 64;  // norms that one wave ranks
// Which way a parameter's chunks go: a chunk per workgroup of four waves (k_aggregate_param), a chunk per wave
// (k_aggregate_chunk), or k_decode_aggregate's persistent teams.
//  - While the workgroups of four waves are one resident round (4 to 7 of a compute unit, by their LDS), a chunk's chain is
//    what counts, and four waves share it.  In us against a wave per chunk, k = 32: 1024 chunks of five peers 6.5 : 7.2, 1536 of
//    five 7.5 : 7.7 and 1664 9.5 : 8.3; k = 48: 1280 of thirteen 9.9 : 10.4 and 1344 12.1 : 10.4; k = 64: 1024 of twenty 11.2 : 11.6 and 1088 14.2 :
//    12.3.  One or two peers' few entries leave it ahead into chunks beyond: 4096 of one 13.0 : 13.6, of two 13.4 : 13.8; 59 136 of
//    one 169 : 173.
//  - Into chunks a wave per chunk stays ahead of the teams: 4096 of twenty (k = 64) 26.6 : 21.3, payloads from memory 27.8 :
//    22.1; 16 384 of four 60 : 54 / 65 : 60, 59 136 of fifteen 272 : 240 / 291 : 254 (of five 218 : 196, but 228 : 245).
//  - Into rows up to 8192: 8192 of four 33 : 21 / 33 : 22, of fifteen 37.6 : 28.0 / 40.7 : 39.1; but the teams store rows of 1 KB
//    together: 16 384 of fifteen 60.5 : 71.4 / 66.4 : 79.0, 59 136 of ten 228 : 243 / 255 : 240.  Of one or two peers
//    the chunks by themselves stay ahead for longer: 12 288 of one 46.5 : 30.2, of two 46.7 : 30.8, 24 576 of one 95 : 85.
constexpr int64_t kFourWaveFewPeers = 61440, kFewPeersRows = 24576, kRowChunks = 8192;  // chunks times peers, twice; chunks

struct ParamPeer {
    const uint8_t* idx;
    const void* val;  // fp32 values, or codes
};
struct ParamPeers {
    ParamPeer peer[kParamPeers];  // those past the last repeat it: a wave fetches its peers' pointers without looking
};

// The aggregate of one parameter's chunks, without the transform.  A workgroup of four waves takes one chunk and wave w
// its rows 16 w .. 16 w + 15.  What bounds it is the chain of one wave - payload, scatters in peer order, mean, stores -
// and the device's stores: a 2048 x 2048 parameter has one chunk per SIMD, where k_decode_aggregate's persistent waves
// clear, fill and store 64 rows each by themselves and k_clip_scales is a launch of its own in front of them.
// The waves request the payloads of every fourth peer while they clear their rows and hand them over through
// LDS, the last wave the clip factors with them (made from the norms: cheaper than a launch); then each walks all entries in peer order and keeps those of its own rows.  One instruction adds one peer's entries: an
// exchange that leaves a mark in the slot until the sum is written back, as in k_decode_aggregate, tells of a repeated
// index in a peer's row, and the wave then does its rows again with every entry in its turn (exact).
// Measured, clip factors included, chunked: 2048 x 2048, 15 peers of k = 32 8.9 us (two launches of the general kernels
// 12.3); 8192 x 2048 from one peer's codes, k = 64, 12.1 us (19.8).  Its compute units' LDS pipelines are what fills up
// first (three LDS instructions a step).
// kUnits: peers staged (the launcher rounds up); kCodes: values are a quantiser's codes, lookup[code] + shift (:637-643).
template <int kUnits, bool kCodes>
__global__ __launch_bounds__(256) void k_aggregate_param(const ParamPeers pp, const float* __restrict__ factors,
                                                         const float* __restrict__ norms, int n_norms, int P, int k,
                                                         const float* __restrict__ lookup, const float* __restrict__ shift,
                                                         int n_bins, int X, int64_t n_chunks, int64_t ld,
                                                         float* __restrict__ out) {
    static_assert(kUnits % 4 == 0, "every wave stages a quarter of the peers");
    constexpr int kMine = kUnits / 4;
    constexpr uint32_t kMark = 0xffffffffu;  // (a NaN: the sum in a slot has these bits only if a peer sent them)
    __shared__ __align__(16) float sums[4096];
    __shared__ __align__(16) uint32_t counts[1024];  // four coefficients to a word
    __shared__ __align__(8) uint2 entries[kUnits][64];
    __shared__ float factor[kUnits];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t chunk = xcd_contiguous(blockIdx.x, gridDim.x);
    if (chunk >= n_chunks) return;  // the whole workgroup

    // (lanes without an entry read entry 0, units without a peer the last peer's: a load behind a branch would be
    // waited for there)
    const bool lane_on = lane < k;
    const int le = lane_on ? lane : 0;
    const int64_t at_idx = chunk * (k + (k >> 1)) + 3 * (le >> 1) + (le & 1), at_val = chunk * k + le;
    uint32_t ix[kMine], bits[kMine];
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const ParamPeer& from = pp.peer[wv + 4 * i];
        ix[i] = *(const gu16*)((const gbyte*)from.idx + at_idx);
        if constexpr (kCodes)
            bits[i] = ((const gbyte*)from.val)[at_val];
        else
            bits[i] = __float_as_uint(((const gfloat*)from.val)[at_val]);
    }
    // the last wave, whose share of the payloads is the smallest, makes the clip factors
    if (wv == 3 && (norms || factors)) {  // wave-uniform
        float f;
        if (norms)
            f = lane_clip_factor(norms[lane < n_norms ? lane : 0], n_norms, lane);
        else
            f = factors[lane < P ? lane : 0];
        if (lane < kUnits) factor[lane] = f;
    }
    float* const rows = sums + wv * 1024;
    uint32_t* const cnt = counts + wv * 256;
    auto clear = [&] {
#pragma unroll
        for (int q = 0; q < 4; ++q) reinterpret_cast<float4*>(rows)[q * 64 + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
        reinterpret_cast<uint4*>(cnt)[lane] = make_uint4(0u, 0u, 0u, 0u);
    };
    clear();
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int p = wv + 4 * i;
        float a = __uint_as_float(bits[i]);
        if constexpr (kCodes) {
            const uint32_t c = bits[i] < static_cast<uint32_t>(n_bins) ? bits[i] : static_cast<uint32_t>(n_bins - 1);
            a = lookup[c] + *shift;
        }
        const uint32_t e = (le & 1) ? ix[i] >> 4 : ix[i] & 0xfffu;
        entries[p][lane] = make_uint2(p < P && lane_on ? e : kMark, __float_as_uint(a));  // (kMark: in no wave's rows)
    }
    __syncthreads();

    const bool scaled = norms || factors;
    const float mine = scaled && lane < kUnits ? factor[lane] : 1.0f;
    // peer p's value times its factor
    auto value = [&](uint32_t v, int p) {
        const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine), p));
        return __uint_as_float(v) * f;
    };
    // (all entries are fetched before the first is added: a step then waits for its exchange alone)
    uint2 e[kUnits];
#pragma unroll
    for (int p = 0; p < kUnits; ++p) e[p] = entries[p][lane];
    uint32_t seen = 0;
#pragma unroll
    for (int p = 0; p < kUnits; ++p) {
        const uint32_t s = e[p].x;
        if ((s >> 10) == static_cast<uint32_t>(wv)) {  // (none of a unit past the last peer)
            const uint32_t old = __hip_atomic_exchange(reinterpret_cast<uint32_t*>(sums + s), kMark, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_WAVEFRONT);
            __hip_atomic_fetch_add(&counts[s >> 2], 1u << ((s & 3u) * 8u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            seen = seen > old ? seen : old;
            sums[s] = __uint_as_float(old) + value(e[p].y, p);
        }
        wave_lds_fence();
    }
    if (__ballot(seen == kMark) != 0) {  // wave-uniform
        clear();
        wave_lds_fence();
        // counts saturate their byte only beyond 255 contributions; P rows of k <= 64 entries may hold more
        // repeats, so they are carried as floats in the entries' order, sums first
        float total[16];
#pragma unroll 1
        for (int phase = 0; phase < 2; ++phase) {
#pragma unroll 1
            for (int p = 0; p < P; ++p) {
                const uint2 e = entries[p][lane];
                const uint32_t s = e.x & 1023u;
                const bool here = (e.x >> 10) == static_cast<uint32_t>(wv);
                const float x = phase ? 1.0f : value(e.y, p);
                const int me = here ? static_cast<int>(s) : -1;
                int rank = 0;  // among the earlier lanes that name the same coefficient; one rank per turn
                for (int i = 0; i < 63; ++i) {
                    const int other = __shfl(me, i);
                    rank += (i < lane && other == me && here) ? 1 : 0;
                }
                const int turns = static_cast<int>(wave_max_u32(static_cast<uint32_t>(rank)));
                for (int r = 0; r <= turns; ++r) {
                    if (here && rank == r) rows[s] = rows[s] + x;
                    wave_lds_fence();
                }
            }
            if (phase == 0) {
#pragma unroll
                for (int q = 0; q < 16; ++q) total[q] = rows[q * 64 + lane];
                wave_lds_fence();
                clear();
                wave_lds_fence();
            }
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const float n = rows[q * 64 + lane];
            rows[q * 64 + lane] = n > 1.0f ? total[q] / n : total[q];
        }
        wave_lds_fence();  // (the counts stay zero: what is read below is the mean already)
    }

    const int64_t y = chunk / X, xc = chunk - y * X;
    float* dst = out + (ld ? (y * 64 + wv * 16) * ld + xc * 64 : chunk * 4096 + wv * 1024);
    const int64_t step = ld ? ld : 64;
    const int r0 = lane >> 4, col = (lane & 15) << 2;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float4 v = reinterpret_cast<const float4*>(rows)[q * 64 + lane];
        const uint32_t c = cnt[q * 64 + lane];
        if (c & 0xfefefefeu) {  // a coefficient that more than one peer sent
            auto mean = [&](float s, int b) {
                const uint32_t n = (c >> b) & 255u;
                return n > 1u ? s / static_cast<float>(n) : s;
            };
            v.x = mean(v.x, 0), v.y = mean(v.y, 8), v.z = mean(v.z, 16), v.w = mean(v.w, 24);
        }
        *reinterpret_cast<float4*>(dst + (q * 4 + r0) * step + col) = v;
    }
}

// The same aggregate with a chunk per wave, for more work than k_aggregate_param's.  The chunk goes through LDS in halves of
// 32 rows and leaves for memory half by half; sixteen waves of a compute unit (10 KB of LDS, 128 registers) have their
// payloads requested at once, where k_decode_aggregate's persistent eight take their chunks in turn and every wave of
// k_aggregate_param walks all entries of its chunk to keep a quarter of them.  What bounds it is the LDS instructions of the
// scatter, three for each peer and half, and the stores.  4096 chunks of 20 peers, k = 64, clip factors included 21.3 us, where
// the persistent kernel took 26.6 (the stores alone 11).  Short-lived workgroups of one wave: teams of two and four were not
// faster (a chunk's result is 16 KB in one piece).
template <int kUnits>
__global__ __launch_bounds__(64, 4) void k_aggregate_chunk(const ParamPeers pp, const float* __restrict__ factors,
                                                           const float* __restrict__ norms, int n_norms, int P, int k, int X,
                                                           int64_t n_chunks, int64_t ld, float* __restrict__ out) {
    constexpr uint32_t kMark = 0xffffffffu;         // (as in k_aggregate_param)
    constexpr int kBits = kUnits <= 15 ? 4 : 8;     // of a counter
    constexpr int kCntWords = kHalfWords * kBits / 32;
    __shared__ __align__(16) float tile[kHalfWords];
    __shared__ __align__(16) uint32_t cnt[kCntWords];
    const int lane = threadIdx.x;
    const int64_t chunk = xcd_contiguous(blockIdx.x, gridDim.x);
    if (chunk >= n_chunks) return;
    const bool lane_on = lane < k;
    const int le = lane_on ? lane : 0;
    const int64_t at_idx = uniform64(chunk * (k + (k >> 1))), at_val = uniform64(chunk * k);
    const uint32_t io = 3u * (static_cast<uint32_t>(le) >> 1) + (le & 1);
    uint32_t pos[kUnits];
    float val[kUnits];
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
        pos[u] = *(const gu16*)((const gbyte*)pp.peer[u].idx + at_idx + io);
        val[u] = ((const gfloat*)pp.peer[u].val + at_val)[le];
    }
    float sc = 1.0f;  // lane p: peer p's factor
    if (norms)        // wave-uniform
        sc = lane_clip_factor(norms[lane < n_norms ? lane : 0], n_norms, lane);
    else if (factors)
        sc = factors[lane < P ? lane : 0];
    auto factor_of = [&](int p) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sc), p)); };
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
        const uint32_t e = (le & 1) ? pos[u] >> 4 : pos[u] & 0xfffu;
        pos[u] = lane_on && u < P ? half_pos(e) << 2 : 0xffffu;  // in bytes; the last of them in neither half
        val[u] *= factor_of(u);
    }
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 8; ++q) reinterpret_cast<float4*>(tile)[q * 64 + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = 0; q < kCntWords / 256; ++q) reinterpret_cast<uint4*>(cnt)[q * 64 + lane] = make_uint4(0u, 0u, 0u, 0u);
        wave_lds_fence();
    };
    // half a chunk with every entry in its turn: sums, then counts, then means
    auto exact_half = [&](uint32_t half) __attribute__((always_inline)) {
        float4 total[8];
#pragma unroll 1
        for (int phase = 0; phase < 2; ++phase) {
            clear();
#pragma unroll 1
            for (int p = 0; p < P; ++p) {
                const uint32_t w = *(const gu16*)((const gbyte*)pp.peer[p].idx + at_idx + io);
                const uint32_t e = half_pos((le & 1) ? w >> 4 : w & 0xfffu);
                float x = ((const gfloat*)pp.peer[p].val + at_val)[le] * factor_of(p);
                if (phase) x = 1.0f;
                const bool here = lane_on && (e >> 11) == half;
                const int me = here ? static_cast<int>(e & 2047u) : -1;
                int rank = 0;  // among the earlier lanes that name the same coefficient; one rank per turn
                for (int i = 0; i < 63; ++i) {
                    const int other = __shfl(me, i);
                    rank += (i < lane && other == me && here) ? 1 : 0;
                }
                const int turns = static_cast<int>(wave_max_u32(static_cast<uint32_t>(rank)));
                for (int r = 0; r <= turns; ++r) {
                    if (here && rank == r) tile[me] = tile[me] + x;
                    wave_lds_fence();
                }
            }
            if (phase == 0) {
#pragma unroll
                for (int q = 0; q < 8; ++q) total[q] = reinterpret_cast<const float4*>(tile)[q * 64 + lane];
                wave_lds_fence();
            }
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            float4 n = reinterpret_cast<const float4*>(tile)[q * 64 + lane];
            auto one = [](float s, float c) { return c > 1.0f ? s / c : s; };
            n.x = one(total[q].x, n.x), n.y = one(total[q].y, n.y), n.z = one(total[q].z, n.z), n.w = one(total[q].w, n.w);
            reinterpret_cast<float4*>(tile)[q * 64 + lane] = n;
        }
        wave_lds_fence();
    };
    const int64_t y = chunk / X, xc = chunk - y * X;
    float* const dst = out + (ld ? y * 64 * ld + xc * 64 : chunk * 4096);
    const int64_t step = ld ? ld : 64;
    const int r0 = lane >> 4, c4 = lane & 15;
    auto half_chunk = [&](auto ht) __attribute__((always_inline)) {
        constexpr uint32_t half = decltype(ht)::value;
        clear();
        uint32_t seen = 0;
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            // (a copy the optimiser cannot see through, or it keeps what it derives from the position across the halves)
            uint32_t at = pos[u];
            asm volatile("" : "+v"(at));
            if ((at >> 13) == half) {
                float* const t = reinterpret_cast<float*>(reinterpret_cast<char*>(tile) + (at & 8191u));
                const uint32_t old = __hip_atomic_exchange(reinterpret_cast<uint32_t*>(t), kMark, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_WAVEFRONT);
                if constexpr (kBits == 4)
                    __hip_atomic_fetch_add(&cnt[(at >> 5) & 255u], 1u << (at & 28u), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WAVEFRONT);
                else
                    __hip_atomic_fetch_add(&cnt[(at >> 4) & 511u], 1u << ((at << 1) & 24u), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WAVEFRONT);
                seen = seen > old ? seen : old;
                *t = __uint_as_float(old) + val[u];
            }
        }
        wave_lds_fence();
        if (__builtin_expect(__ballot(seen == kMark) != 0, 0)) {  // wave-uniform
            exact_half(half);
        } else {
            if constexpr (kBits == 4)
                half_means4(tile, cnt, lane);
            else
                half_means8(tile, cnt, lane);
            wave_lds_fence();
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int row = q * 4 + r0;
            const float4 v = reinterpret_cast<const float4*>(tile)[row * 16 + (c4 ^ (row & 15))];
            *reinterpret_cast<float4*>(dst + (static_cast<int64_t>(half * 32 + row)) * step + c4 * 4) = v;
        }
        wave_lds_fence();
    };
    half_chunk(std::integral_constant<uint32_t, 0>{});
    half_chunk(std::integral_constant<uint32_t, 1>{});
}

template <bool kCodes>
static int launch_param(const ParamPeers& pp, const float* factors, const float* norms, int n_norms, int P, int k,
                        const float* lookup, const float* shift, int n_bins, int64_t X, int64_t n, int64_t ld, float* out,
                        void* stream) {
    auto kernel = k_aggregate_param<4, kCodes>;
    if constexpr (!kCodes)
        kernel = P <= 4 ? k_aggregate_param<4, false> : P <= 8 ? k_aggregate_param<8, false>
               : P <= 16 ? k_aggregate_param<16, false> : k_aggregate_param<24, false>;
    hipLaunchKernelGGL(kernel, dim3(grid8(n)), dim3(256), 0, static_cast<hipStream_t>(stream), pp, factors, norms, n_norms, P, k,
                       lookup, shift, n_bins, static_cast<int>(X), n, ld, out);
    return launch_status();
}

// chunks that k_aggregate_param's workgroups hold at a time
static int64_t four_wave_round(int P) {
    constexpr int64_t any = int64_t{1} << 40;
    if (P <= 4) {
        static const int r = persistent_grid(k_aggregate_param<4, false>, any, 256);
        return r;
    }
    if (P <= 8) {
        static const int r = persistent_grid(k_aggregate_param<8, false>, any, 256);
        return r;
    }
    if (P <= 16) {
        static const int r = persistent_grid(k_aggregate_param<16, false>, any, 256);
        return r;
    }
    static const int r = persistent_grid(k_aggregate_param<24, false>, any, 256);
    return r;
}

// (the launcher's form with room for the peers at hand: units without one still take part in every step)
static int launch_chunk(const ParamPeers& pp, const float* factors, const float* norms, int n_norms, int P, int k, int64_t X,
                        int64_t n, int64_t ld, float* out, void* stream) {
    auto kernel = P <= 4    ? k_aggregate_chunk<4>
                  : P <= 8  ? k_aggregate_chunk<8>
                  : P <= 12 ? k_aggregate_chunk<12>
                  : P <= 15 ? k_aggregate_chunk<15>
                  : P <= 20 ? k_aggregate_chunk<20>
                            : k_aggregate_chunk<24>;
    hipLaunchKernelGGL(kernel, dim3(grid8(n)), dim3(64), 0, static_cast<hipStream_t>(stream), pp, factors, norms, n_norms, P, k,
                       static_cast<int>(X), n, ld, out);
    return launch_status();
}

// Chunks (Y, X, 64, 64) into the (64 Y, 64 X) tensor they are cut from: decode without the transform (src/tplr/compress.py:281).
// A workgroup takes 32 rows of a band of chunks, 256 columns wide: a wave reads 256 bytes of four chunks and writes 1 KB of a
// row, eight rows requested before the first is stored; stores past the caches, which the result would only pass through.
// It is bound by memory: 2048 x 8192 19.6 us, 6.9 TB/s read and written (torch's strided copy 22-26); 2048 x 2048 6.3 (7.9);
// rows per workgroup and whether a wave's rows are the chunk's or the tensor's matter by 5 %.
__global__ __launch_bounds__(256) void k_unchunk(const v4f* __restrict__ chunks, int X, int tiles, int64_t n_groups, v4f* __restrict__ out) {
    const int64_t g = xcd_contiguous(blockIdx.x, gridDim.x);
    if (g >= n_groups) return;
    const int64_t half = g & 1, t = g >> 1, y = t / tiles;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int col = static_cast<int>(t - y * tiles) * 256 + lane * 4;  // (fewer than 2^31 columns)
    if (col >= X * 64) return;
    const int64_t C = static_cast<int64_t>(X) * 64;
    const int row0 = static_cast<int>(half) * 32 + wv;
    const v4f* src = chunks + (((y * X + (col >> 6)) * 4096 + row0 * 64 + (col & 63)) >> 2);
    v4f* dst = out + (((y * 64 + row0) * C + col) >> 2);
    v4f v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = src[i * 64];
#pragma unroll
    for (int i = 0; i < 8; ++i) __builtin_nontemporal_store(v[i], dst + i * C);
}

}  // namespace tplr

using namespace tplr;

extern "C" int tplr_aggregate_param(const uint8_t* const* h_idx12, const float* const* h_val, const float* d_norms, int n_norms,
                                    float* d_scale, int n_peers, int k, int64_t R, int64_t C, float* d_out, int64_t ld_out,
                                    void* stream) {
    if (!h_idx12 || !h_val || !d_out || n_peers < 1 || k < 2 || (k & 1) || k > 4096 || R < 0 || C < 0 || n_norms < 0 ||
        (d_norms && (n_norms < n_peers || !d_scale)))
        return TPLR_E_BADARG;
    if (n_peers > TPLR_MAX_PEERS || n_norms > TPLR_MAX_PEERS) return TPLR_E_TOOMANY;
    if ((R % 64) || (C % 64)) return TPLR_E_SHAPE;
    if (ld_out != 0 && ld_out < C) return TPLR_E_BADARG;
    const int64_t n = (R / 64) * (C / 64);
    if (n == 0) return 0;
    if (C / 64 > 0x7fffffff || R / 64 > 0x7fffffff || ld_out > (int64_t{1} << 23)) return TPLR_E_TOOMANY;
    const bool few = n_peers <= 2 && n * n_peers <= (ld_out ? kFewPeersRows : kFourWaveFewPeers);
    if (n_peers <= kParamPeers && k <= 64 && n_norms <= kParamNorms && (few || n <= (ld_out ? kRowChunks : kMaxGroups256)) &&
        (ld_out & 3) == 0 && (reinterpret_cast<uintptr_t>(d_out) & 15) == 0) {
        ParamPeers pp = {};
        for (int p = 0; p < n_peers; ++p) {
            if (!h_idx12[p] || !h_val[p]) return TPLR_E_BADARG;
        }
        for (int p = 0; p < kParamPeers; ++p) {
            const int u = p < n_peers ? p : n_peers - 1;
            pp.peer[p] = {h_idx12[u], h_val[u]};
        }
        if (n <= four_wave_round(n_peers) || (few && !ld_out))
            return launch_param<false>(pp, d_scale, d_norms, n_norms, n_peers, k, nullptr, nullptr, 0, C / 64, n, ld_out, d_out, stream);
        return launch_chunk(pp, d_scale, d_norms, n_norms, n_peers, k, C / 64, n, ld_out, d_out, stream);
    }
    if (d_norms && n_peers <= kParamPeers && k <= 64 && n_norms <= kParamNorms)
        return aggregate_from_norms(h_idx12, h_val, d_norms, n_norms, n_peers, k, R, C, d_out, ld_out, stream);
    if (d_norms)
        if (int s = tplr_clip_scales(d_norms, n_norms, 0, d_scale, nullptr, stream)) return s;
    return tplr_decode_aggregate(h_idx12, h_val, d_scale, n_peers, k, R, C, TPLR_REDUCE_MEAN, 0, 0, d_out, ld_out, nullptr, stream);
}

extern "C" int tplr_decompress_codes(const uint8_t* d_idx12, const uint8_t* d_codes, const float* d_lookup, const float* d_shift,
                                     int n_bins, int k, int64_t R, int64_t C, float* d_out, int64_t ld_out, void* stream) {
    if (!d_idx12 || !d_codes || !d_lookup || !d_shift || !d_out || n_bins < 1 || n_bins > 256 || k < 2 || (k & 1) || R < 0 || C < 0)
        return TPLR_E_BADARG;
    if (k > 64) return TPLR_E_TOOMANY;
    if ((R % 64) || (C % 64)) return TPLR_E_SHAPE;
    if ((ld_out != 0 && ld_out < C) || (ld_out & 3) || (reinterpret_cast<uintptr_t>(d_out) & 15)) return TPLR_E_BADARG;
    const int64_t n = (R / 64) * (C / 64);
    if (n == 0) return 0;
    if (n > kMaxGroups256) return TPLR_E_TOOMANY;
    ParamPeers pp = {};
    for (ParamPeer& p : pp.peer) p = {d_idx12, d_codes};
    return launch_param<true>(pp, nullptr, nullptr, 0, 1, k, d_lookup, d_shift, n_bins, C / 64, n, ld_out, d_out, stream);
}

extern "C" int tplr_unchunk(const float* d_chunks, int64_t R, int64_t C, float* d_out, void* stream) {
    if (int st = check_2d(d_chunks, d_out, R, C)) return st;
    if ((reinterpret_cast<uintptr_t>(d_chunks) & 15) || (reinterpret_cast<uintptr_t>(d_out) & 15)) return TPLR_E_BADARG;
    if (R == 0 || C == 0) return 0;
    const int64_t tiles = (C + 255) / 256, groups = R / 64 * tiles * 2;
    if (C > 0x7fffff00 || groups > kMaxGroups256) return TPLR_E_TOOMANY;
    hipLaunchKernelGGL(k_unchunk, dim3(grid8(groups)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       reinterpret_cast<const v4f*>(d_chunks), static_cast<int>(C / 64), static_cast<int>(tiles), groups,
                       reinterpret_cast<v4f*>(d_out));
    return launch_status();
}
