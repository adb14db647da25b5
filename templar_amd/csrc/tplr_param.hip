// One parameter's payloads into its chunks: what the reference's per-parameter calls batch_decompress and decompress
// leave before the transform (src/tplr/compress.py:425-580), a chunk spread over the four waves of a workgroup.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tplr_hip.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

constexpr int kParamPeers = 24;  // payloads of one launch
constexpr int kParamNorms = 64;  // norms that one wave ranks
// Chunks times peers up to which a chunk per workgroup is the faster way, into chunked results and into rows: beyond it
// the scatters, of which every wave issues all and keeps a quarter, fill the compute units' LDS pipelines; and the
// persistent kernel's teams store rows of 1 KB together, but no such rows into chunks.  Clip factors and aggregate in us, this
// kernel against k_decode_aggregate that makes the factors itself, chunked: 1024 chunks of 15 peers 8.9 : 11.5, of 20
// (k = 64) 10.7 : 13.3, 4096 of 5 15.2 : 18.7, of 15 22.1 : 22.5, 16 384 of 4 58.7 : 62.5 - but 2048 of 20 (k = 64) 17.0 : 16.5, 4096
// of 20 28.9 : 27.1.  Into rows: 1024 of 15 9.2 : 10.7, 4096 of 5 15.9 : 18.4 - but 2048 of 15 14.1 : 12.8, of 12 13.2 : 12.5.
constexpr int64_t kParamWorkChunks = 61440, kParamWorkRows = 24576;

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
    if (n_peers <= kParamPeers && k <= 64 && n_norms <= kParamNorms && n * n_peers <= (ld_out ? kParamWorkRows : kParamWorkChunks) && (ld_out & 3) == 0 &&
        (reinterpret_cast<uintptr_t>(d_out) & 15) == 0) {
        ParamPeers pp = {};
        for (int p = 0; p < n_peers; ++p) {
            if (!h_idx12[p] || !h_val[p]) return TPLR_E_BADARG;
        }
        for (int p = 0; p < kParamPeers; ++p) {
            const int u = p < n_peers ? p : n_peers - 1;
            pp.peer[p] = {h_idx12[u], h_val[u]};
        }
        return launch_param<false>(pp, d_scale, d_norms, n_norms, n_peers, k, nullptr, nullptr, 0, C / 64, n, ld_out, d_out, stream);
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
