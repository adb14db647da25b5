// Decode of payloads with the transform, a chunk per wave: aggregate, evaluation update, outer step.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/tplr_hip.h"
#include "tplr_chunk.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

// Up to fifteen peers' payloads into chunks, through the inverse transform: the aggregate of k_decode_aggregate (same bits), and
// with kSubtract dst - result and its guard against results that are not finite.
//
// A wave takes one chunk, a workgroup four neighbouring ones, and ends: the hardware puts the next chunk where one has
// ended, so that loads, arithmetic and stores of a compute unit's waves overlap whatever their pace, and a set's last round
// is as full as the others.  What that needs is waves: the chunk goes through LDS in halves of 32 rows (9 KB a wave),
// scattered, averaged and read into registers one after the other, and three waves fit a SIMD where k_decode_aggregate has
// two, its next chunks' payloads in the registers of the third.  Against that stand the payload's way from memory, which
// nothing hides here, and a chain of LDS round trips per peer and half.
// Subtracting, what bounds it is the loads and stores (1520 us alone) and this form is the faster one throughout.  In us, before
// and now: one peer, the 294 144 chunks of a 1B set 1722 -> 1545, a 150M model's 39 648 274 -> 225; eight peers of k = 64 1890 -> 1725,
// fifteen 2222 -> 1915; one 2048 x 2048 tensor from four 19 -> 15.  The team stores together (1544, each wave by itself 1570).
// Not subtracting, payloads not in any cache: one peer 972 -> 940 and 154 -> 138; for more see decode_chunks_serves.
constexpr int kChunkPeers = 15;  // what four bits count
struct ChunkPeers {
    const uint8_t* idx[kChunkPeers];
    const float* val[kChunkPeers];  // (those past the last repeat it)
};

template <int kUnits, bool kSubtract>
__global__ __launch_bounds__(256, 3) void k_decode_chunk(const ChunkPeers pp, const float* __restrict__ scale, int P, int k,
                                                       const tplr_tensor_desc* __restrict__ table, const tplr_tensor_desc single,
                                                       int n_tensors, int64_t first, int64_t end, int mean, int with_sum,
                                                       float* __restrict__ stats, int32_t* __restrict__ guard) {
    constexpr int T = 4;
    constexpr int kCntWords = kUnits > 1 ? kHalfWords / 8 : 4;  // four bits a coefficient
    constexpr uint32_t kMark = 0xffffffffu;  // (a NaN: a sum has these bits only if a peer sent them)
    __shared__ __align__(16) float tile_all[T][kHalfWords];
    __shared__ __align__(16) uint32_t cnt_all[T][kCntWords];
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    float* const tile = tile_all[wv];
    uint32_t* const cnt = cnt_all[wv];
    const int lane = threadIdx.x & 63;
    const int64_t g = first + xcd_contiguous(blockIdx.x, gridDim.x) * T + wv;
    if (g >= end) return;  // wave-uniform

    // ---- the payload: lane j holds entry j of every peer (lanes without one reload entry 0 and stay out of it)
    const bool lane_on = lane < k;
    const int le = lane_on ? lane : 0;
    const int64_t at_idx = uniform64(g * (k + (k >> 1))), at_val = uniform64(g * k);
    const uint32_t io = 3u * (static_cast<uint32_t>(le) >> 1) + (le & 1);
    uint32_t pos[kUnits];
    float val[kUnits];
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
        pos[u] = *(const gu16*)((const gbyte*)pp.idx[u] + at_idx + io);
        val[u] = ((const gfloat*)pp.val[u] + at_val)[le];
    }
    const Place at = place_of(table, single, n_tensors, g);
    const int pl = lane < P ? lane : P - 1;
    // (the transform below is 32x the orthonormal one: its input carries the exact 2^-5)
    const float sc = (scale ? scale[static_cast<int64_t>(at.t) * P + pl] : 1.0f) * kDctPow2Scale;
    auto factor_of = [&](int p) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sc), p)); };
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
        const uint32_t e = (le & 1) ? pos[u] >> 4 : pos[u] & 0xfffu;
        pos[u] = lane_on && u < P ? half_pos(e) << 2 : 0xffffu;  // in bytes; the last of them in neither half
        val[u] *= factor_of(u);
    }

    auto clear = [&] {
#pragma unroll
        for (int q = 0; q < 8; ++q) reinterpret_cast<float4*>(tile)[q * 64 + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = 0; q < kCntWords / 256; ++q) reinterpret_cast<uint4*>(cnt)[q * 64 + lane] = make_uint4(0u, 0u, 0u, 0u);
        wave_lds_fence();
    };
    // sums of half a chunk with every entry in its turn, then counts, then means
    auto exact_half = [&](uint32_t half) __attribute__((always_inline)) {
        float4 total[8];
#pragma unroll 1
        for (int phase = 0; phase < 2; ++phase) {
            clear();
#pragma unroll 1
            for (int p = 0; p < P; ++p) {
                const uint32_t w = *(const gu16*)((const gbyte*)pp.idx[p] + at_idx + io);
                const uint32_t e = half_pos((le & 1) ? w >> 4 : w & 0xfffu);
                float x = ((const gfloat*)pp.val[p] + at_val)[le] * factor_of(p);
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
            auto one = [&](float s, float c) { return mean && c > 1.0f ? s / c : s; };
            n.x = one(total[q].x, n.x), n.y = one(total[q].y, n.y), n.z = one(total[q].z, n.z), n.w = one(total[q].w, n.w);
            reinterpret_cast<float4*>(tile)[q * 64 + lane] = n;
        }
        wave_lds_fence();
    };
    // the coefficients of one half into the tile
    auto gather_half = [&](auto ht) __attribute__((always_inline)) {
        constexpr uint32_t half = decltype(ht)::value;
        clear();
        uint32_t seen = 0;
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            if ((pos[u] >> 13) == half) {
                float* const t = reinterpret_cast<float*>(reinterpret_cast<char*>(tile) + (pos[u] & 8191u));
                const uint32_t old = __hip_atomic_exchange(reinterpret_cast<uint32_t*>(t), kMark, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_WAVEFRONT);
                // (one peer sends a coefficient once, or the exact path has it)
                if constexpr (kUnits > 1)
                    __hip_atomic_fetch_add(&cnt[(pos[u] >> 5) & 255u], 1u << (pos[u] & 28u), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WAVEFRONT);
                seen = seen > old ? seen : old;
                *t = __uint_as_float(old) + val[u];
            }
        }
        wave_lds_fence();
        if (__builtin_expect(__ballot(seen == kMark) != 0, 0)) {  // wave-uniform
            exact_half(half);
        } else if (kUnits > 1 && mean) {
            half_means4(tile, cnt, lane);
            wave_lds_fence();
        }
    };

    float v[64], before[64];
    {
        float w[64];
        gather_half(std::integral_constant<uint32_t, 0>{});
        if (lane < 32) half_rows_to_regs(w, tile, lane & 31);
        wave_lds_fence();
        gather_half(std::integral_constant<uint32_t, 1>{});
        if (lane >= 32) half_rows_to_regs(w, tile, lane & 31);
        wave_lds_fence();
        dct64_inv(w);  // along d: w[l] = sum_d Y[lane][d] F[l][d]
        if (lane < 32) regs_to_half_rows(w, tile, lane & 31);
        wave_lds_fence();
        half_cols_to_regs<0>(v, tile, lane);
        wave_lds_fence();
        if (lane >= 32) regs_to_half_rows(w, tile, lane & 31);
        wave_lds_fence();
        half_cols_to_regs<1>(v, tile, lane);
    }
    // (the destination's rows arrive during the second pass)
    if constexpr (kSubtract) load_chunk_rows(before, (const void*)at.chunk0, at.ld, lane);
    dct64_inv(v);  // along b: v[k] = sum_b Z[b][lane] F[k][b]
    if (stats) {  // wave-uniform
        float ss = 0.f, sm = 0.f;
#pragma unroll
        for (int r = 0; r < 64; ++r) ss = __builtin_fmaf(v[r], v[r], ss);
        ss = wave_sum_f32(ss);
        if (with_sum) {
#pragma unroll
            for (int r = 0; r < 64; ++r) sm += v[r];
            sm = wave_sum_f32(sm);
            if (lane == 0) stats[2 * g] = ss, stats[2 * g + 1] = sm;
        } else if (lane == 0) {
            stats[g] = ss;
        }
    }
    bool drop = false;
    if constexpr (kSubtract) {
        if (guard) {  // wave-uniform
            float z = 0.f;
#pragma unroll
            for (int r = 0; r < 64; ++r) z = __builtin_fmaf(v[r], 0.0f, z);
            drop = __ballot(z != z) != 0;
            if (drop && lane == 0) guard[at.t] = 1;
        }
#pragma unroll
        for (int r = 0; r < 64; ++r) v[r] = before[r] - v[r];
    }
    // (a bare barrier: nothing is handed over, and a wave that has ended is not waited for)
    if constexpr (kSubtract) __builtin_amdgcn_s_barrier();
    store_chunk_rows(v, (void*)at.chunk0, at.ld, lane, drop);
}

template <int kUnits, bool kSubtract>
static int launch_chunks(const ChunkPeers& pp, const float* d_scale, int n_peers, int k, const tplr_tensor_desc* d_desc,
                      const tplr_tensor_desc& single, int n_tensors, int64_t total, int mean, int with_sum, float* d_stats,
                      int32_t* d_guard, void* stream) {
    constexpr int64_t piece = kMaxGroups256 * 4;  // chunks of one launch
    for (int64_t first = 0; first < total; first += piece) {
        const int64_t end = total - first < piece ? total : first + piece;
        hipLaunchKernelGGL((k_decode_chunk<kUnits, kSubtract>), dim3(grid8((end - first + 3) / 4)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), pp, d_scale, n_peers, k, d_desc, single, n_tensors, first, end, mean,
                           with_sum, d_stats, d_guard);
    }
    return launch_status();
}

// Without the subtraction, payloads coming from memory, in us k_decode_aggregate against this form (k = 32 / 64): 1024 chunks of
// four peers 11.9 : 9.3 / 12.2 : 9.4, of fifteen 14.0 : 11.6 / 15.3 : 12.3; 4096 of four 23.9 : 21.9 / 24.5 : 22.8, of fifteen 27.5 : 27.1 /
// 29.6 : 28.6; 8192 of four 40.2 : 37.9 / 41.6 : 39.4, of fifteen 46.9 : 47.5 / 50.8 : 50.4; but 16 384 of two 66.9 : 67.0 / 69.5 : 68.6, of eight
// 72.5 : 76.2 / 75.1 : 80.5, 294 144 of two 980 : 1032 / 1074 : 1062, of fifteen 1216 : 1344 / 1255 : 1364.  (Between, where the other's rounds come out
// badly, this one is ahead for a few peers: 39 648 of four 162 : 157 / 169 : 164.)
bool decode_chunks_serves(int n_peers, int k, int64_t total, bool subtract) {
    return n_peers <= kChunkPeers && k <= 64 && (subtract || n_peers == 1 || total <= 8192);
}

int decode_chunks(const uint8_t* const* h_idx12, const float* const* h_val, const float* d_scale, int n_peers, int k,
                  const tplr_tensor_desc* d_desc, const tplr_tensor_desc& single, int n_tensors, int64_t total, bool subtract,
                  bool mean, bool with_sum, float* d_stats, int32_t* d_guard, void* stream) {
    ChunkPeers pp;
    for (int u = 0; u < kChunkPeers; ++u) {
        pp.idx[u] = h_idx12[u < n_peers ? u : n_peers - 1];
        pp.val[u] = h_val[u < n_peers ? u : n_peers - 1];
    }
    auto launch = n_peers == 1    ? subtract ? launch_chunks<1, true> : launch_chunks<1, false>
                  : n_peers == 2  ? subtract ? launch_chunks<2, true> : launch_chunks<2, false>
                  : n_peers <= 4  ? subtract ? launch_chunks<4, true> : launch_chunks<4, false>
                  : n_peers <= 8  ? subtract ? launch_chunks<8, true> : launch_chunks<8, false>
                  : n_peers <= 12 ? subtract ? launch_chunks<12, true> : launch_chunks<12, false>
                                  : subtract ? launch_chunks<15, true> : launch_chunks<15, false>;
    return launch(pp, d_scale, n_peers, k, d_desc, single, n_tensors, total, mean, with_sum, d_stats, d_guard, stream);
}

// What the updates' launches multiply their values by, and what an outer step reports, where a chain of elementwise launches of
// 4-5 us each would stand around a launch of one or two milliseconds.
//
// Per tensor the peers' factors times lr; NaN, which keeps every chunk of the tensor as it is and flags it, where one of them
// is not finite and positive (nothing then vouches for the gradient), or where `bad` names a code outside its quantiser.
__global__ __launch_bounds__(64) void k_outer_factors(const float* __restrict__ scale, int P, float lr,
                                                      const int32_t* __restrict__ bad, float* __restrict__ factor) {
    const int64_t row = static_cast<int64_t>(blockIdx.x) * P;
    bool unsound = bad && *bad != 0;
    for (int p = threadIdx.x; p < P; p += 64) {
        const float f = scale[row + p];
        unsound = unsound || !(f > 0.f) || __builtin_isinf(f);
    }
    const bool keep = __ballot(unsound) != 0;
    for (int p = threadIdx.x; p < P; p += 64) factor[row + p] = keep ? __builtin_nanf("") : scale[row + p] * lr;
}

// factor_t = alpha * min(1, clip_t / (norm_t + 1e-8)), the norm from n_partials partial sums of squares (added in double);
// without partial sums alpha * clip_t
__global__ __launch_bounds__(64) void k_update_factors(const float* __restrict__ partials, int n_partials,
                                                       const float* __restrict__ clip, float alpha, int n_tensors,
                                                       float* __restrict__ factor) {
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t >= n_tensors) return;
    float f = clip[t];
    if (n_partials > 0) {
        double ss = 0.0;
        for (int i = 0; i < n_partials; ++i) ss += static_cast<double>(partials[static_cast<int64_t>(t) * n_partials + i]);
        f = f / (static_cast<float>(__builtin_sqrt(ss)) + 1e-8f);
        f = f > 1.0f ? 1.0f : f;  // clamp(max=1); NaN propagates as in torch.clamp
    }
    factor[t] = alpha * f;
}

// figures of lr * gradient {norm, mean, all finite, sum of squares} -> those of the gradient, each rounded once (lr^2 in single
// precision would be rounded itself, and is zero from 1e-23 down)
__global__ __launch_bounds__(64) void k_outer_stats(float4* __restrict__ stats, int n_tensors, float lr) {
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t >= n_tensors) return;
    float4 v = stats[t];
    v.x /= __builtin_fabsf(lr), v.y /= lr;
    v.w = static_cast<float>(v.w / (static_cast<double>(lr) * lr));
    stats[t] = v;
}

}  // namespace tplr

using namespace tplr;

extern "C" int tplr_outer_factors(const float* d_scale, int n_tensors, int n_peers, float lr, const int32_t* d_bad, float* d_factor,
                                  void* stream) {
    if (!d_scale || !d_factor || n_tensors < 1 || n_peers < 1) return TPLR_E_BADARG;
    hipLaunchKernelGGL(k_outer_factors, dim3(static_cast<unsigned>(n_tensors)), dim3(64), 0, static_cast<hipStream_t>(stream), d_scale,
                       n_peers, lr, d_bad, d_factor);
    return launch_status();
}

extern "C" int tplr_update_factors(const float* d_partials, int n_partials, const float* d_clip, float alpha, int n_tensors,
                                   float* d_factor, void* stream) {
    if (!d_clip || !d_factor || n_tensors < 1 || n_partials < 0 || (n_partials > 0 && !d_partials)) return TPLR_E_BADARG;
    hipLaunchKernelGGL(k_update_factors, dim3((static_cast<unsigned>(n_tensors) + 63) / 64), dim3(64), 0, static_cast<hipStream_t>(stream),
                       d_partials, n_partials, d_clip, alpha, n_tensors, d_factor);
    return launch_status();
}

extern "C" int tplr_outer_stats(float* d_stats, int n_tensors, float lr, void* stream) {
    if (!d_stats || n_tensors < 1 || (reinterpret_cast<uintptr_t>(d_stats) & 15)) return TPLR_E_BADARG;
    hipLaunchKernelGGL(k_outer_stats, dim3((static_cast<unsigned>(n_tensors) + 63) / 64), dim3(64), 0, static_cast<hipStream_t>(stream),
                       reinterpret_cast<float4*>(d_stats), n_tensors, lr);
    return launch_status();
}
