// Fused encode (rows, transform, top-k select, pack): single tensors and batches.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tplr_hip.h"
#include "tplr_chunk.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

// Persistent fused encode: every wave walks its slice of the chunk list.  The kernel is bound by
// vector-ALU issue and by the latencies between its phases, so it is shaped for residency -
// 8.5 KB + 1 KB of LDS and a register budget that admits three to four waves per SIMD - and
// leaves the overlap of one wave's row loads with the other waves' arithmetic to the hardware.
// The three waves of a SIMD pass its issue slots round: the arbiter alone serves the oldest wave first, so
// that the workgroups dispatched last run behind all the way and the launch waits for them.  Each wave
// therefore steps through the priority levels 0, 1, 2 chunk by chunk, the three dispatch layers of a full
// grid one step apart, and changes level once its rows are requested (4 % off the launch; the level
// values, the direction and a change at another phase or every other chunk matter less than 1 %).
// Every other encode is k_encode_chunk's, below; this form is for sets with the transform that fit one round of waves or
// fill many (see walks), where what counts is that a wave has nothing to wait for: 879 us for the 115 tensors of a 1B set
// (k = 32), against 928 with a look-up of its tensor in every wave at three waves per SIMD.
template <bool kTwo>
__global__ __launch_bounds__(64, 3) void k_encode_topk_pack(const tplr_tensor_desc* __restrict__ table, int n_tensors, int64_t total,
                                                            int k, uint8_t* __restrict__ idx12, float* __restrict__ val) {
    __shared__ __align__(16) float buf[kHalfFloats];
    __shared__ uint64_t cand[kCandCap];
    const int lane = threadIdx.x;
    int64_t g0, g1;
    my_range(total, g0, g1);
    if (g0 >= g1) return;
    Cursor c;
    cursor_seek(c, table, tplr_tensor_desc{}, n_tensors, g0);
#if TPLR_DCT_MATRIX_CORES
    float ca[16] = {};
    load_dct4_operand(ca, lane);
#endif
    int turn = static_cast<int>(blockIdx.x * 3u / gridDim.x);  // the dispatch layer of a full grid; wave-uniform
    for (int64_t g = g0; g < g1; ++g) {
        float v[64], w[64];
        load_chunk_cols(v, c, lane);
        if (g + 1 < g1) cursor_next(c, g + 1);
        set_wave_priority(turn);
        turn = turn == 2 ? 0 : turn + 1;
#if TPLR_DCT_MATRIX_CORES
        dct64_fwd_matrix(v, ca);
        transpose_via_half(v, w, buf, lane);
        dct64_fwd_matrix(w, ca);
#else
        chunk_forward<true>(v, w, buf, lane);
#endif
        const Selected s = select_topk<kTwo, false>(w, buf, cand, lane, k, kDctPow2Scale);
        emit_selected<kTwo>(s, lane, k, g, idx12, val);
    }
}

// Measurement aid: the memory side of the encode alone - the same grid, chunk ranges and row loads, nothing else
// (the 64 values of a lane are added up so that the loads are not dropped, and the sum never leaves the wave).
__global__ __launch_bounds__(64, 3) void k_calib_encode(const tplr_tensor_desc* __restrict__ table,
                                                        const tplr_tensor_desc single, int n_tensors, int64_t total,
                                                        float* __restrict__ sink) {
    const int lane = threadIdx.x;
    int64_t g0, g1;
    my_range(total, g0, g1);
    if (g0 >= g1) return;
    Cursor c;
    cursor_seek(c, table, single, n_tensors, g0);
    float s = 0.0f;
    for (int64_t g = g0; g < g1; ++g) {
        float v[64];
        load_chunk_cols(v, c, lane);
        if (g + 1 < g1) cursor_next(c, g + 1);
#pragma unroll
        for (int r = 0; r < 64; ++r) s += v[r];
    }
    if (__float_as_uint(s) == 0x7fedcba9u && sink) sink[0] = s;  // (a NaN pattern no sum produces)
}

// One chunk per wave, kTeam neighbouring chunks per workgroup (with the transform single waves).  Without the transform it is bound by memory and by the
// latencies of the select: four waves per SIMD (112 registers, the exact search's among them; 10 KB of LDS a wave
// is just what sixteen waves of a compute unit may have); with it by vector-ALU issue, three waves.  Workgroups are
// short-lived: the hardware puts the next chunk where one has ended, so no wave waits for a slower one, and a wave's loads
// overlap the others' arithmetic.  As one resident round of waves that walk ranges of the chunk list, with 4096 chunks over
// 3072 waves for instance, most of the device idled through the second chunk.  In us, before and now: one tensor without the
// transform 8192 x 2048, k = 64 20.8 -> 17.4, 8192 x 8192 60 -> 48, k = 32 51 -> 44; with it 8192 x 8192 62 -> 56; the 1B set's 294 144
// chunks without it, k = 32 795 -> 750, k = 64 841 -> 790; its miner step of two launches, k = 64 with four-bin codes 3436 -> 3165.
// kEf: the miner's momentum update rides on the load (src/tplr/neurons.py:151-152): the chunk of
// the error-feedback tensor becomes ef * decay + grad (two roundings, as mul_ then add_), is
// written back in place and is what gets encoded.  Rows written together are served sooner: teams of four there, but single waves
// (of the same kernel) while there are fewer chunks than SIMDs, which then share no compute unit's LDS and fetches: with the
// transform 64 chunks 10.2 -> 8.6 us / 11.4 -> 9.7, 768 12.3 -> 11.7 / 13.2 -> 12.6; 2048 23.3 : 24.4, 4096 40.4 : 42.2.
template <bool kUseDct, bool kEf>
constexpr int encode_team() { return kEf ? 4 : kUseDct ? 1 : 2; }

template <bool kTwo, bool kUseDct, bool kEf>
__global__ __launch_bounds__((64 * encode_team<kUseDct, kEf>()), kUseDct || kEf ? 3 : 4) void k_encode_chunk(
    const tplr_tensor_desc* __restrict__ table, const tplr_tensor_desc single, int n_tensors, int64_t first, int64_t end, int k,
    uint8_t* __restrict__ idx12, float* __restrict__ val, const tplr_tensor_desc* __restrict__ grad_table, float decay, int team) {
    constexpr int T = encode_team<kUseDct, kEf>();
    // team: waves of this launch's workgroups, at most T (with the momentum update; otherwise T)
    __shared__ __align__(16) float buf_all[T][kHalfFloats];
    __shared__ uint64_t cand_all[T][kCandCap];
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));  // wave of the team
    float* const buf = buf_all[wv];
    uint64_t* const cand = cand_all[wv];
    const int lane = threadIdx.x & 63;
    const int64_t g = first + xcd_contiguous(blockIdx.x, gridDim.x) * (kEf ? team : T) + wv;
    if (g >= end) return;  // wave-uniform; the waves of a team never wait for one another
    const Place at = place_of(table, single, n_tensors, g);
    float v[64], w[64];
    load_chunk_rows(v, (const void*)at.chunk0, at.ld, lane);
    if constexpr (kEf) {
        const Place from = place_of(grad_table, single, n_tensors, g);
        load_chunk_rows(w, (const void*)from.chunk0, from.ld, lane);
#pragma unroll
        for (int r = 0; r < 64; ++r) {
            const float m = v[r] * decay;
            v[r] = m + w[r];
        }
        store_chunk_rows(v, (void*)at.chunk0, at.ld, lane);
    }
    // Untransformed gradients often differ in scale from row to row or column to column;
    // the select's threshold statistic is then taken in both directions.  (Coefficients of
    // the transform are mixed across both and one direction is as good as two.)
    uint32_t c1 = 0, c2 = 0;
    if (!kUseDct) lane_stats<kTwo>(v, c1, c2);
#if TPLR_DCT_MATRIX_CORES
    float ca[16] = {};
    if (kUseDct) load_dct4_operand(ca, lane);
    if (kUseDct) dct64_fwd_matrix(v, ca);
    transpose_via_half(v, w, buf, lane);
    if (kUseDct) dct64_fwd_matrix(w, ca);
#else
    chunk_forward<kUseDct>(v, w, buf, lane);
#endif
    const Selected s = select_topk<kTwo, !kUseDct, kUseDct || kEf>(w, buf, cand, lane, k, kUseDct ? kDctPow2Scale : 1.0f, c1, c2);
    emit_selected<kTwo>(s, lane, k, g, idx12, val);
}

// d_desc null: one tensor, `single`; d_grad_desc: the momentum update on the load
template <bool kTwo, bool kUseDct, bool kEf = false>
static int launch_chunks(const tplr_tensor_desc* d_desc, const tplr_tensor_desc& single, int n_tensors, int64_t total, int k,
                         uint8_t* d_idx12, float* d_val, void* stream, const tplr_tensor_desc* d_grad_desc = nullptr,
                         float decay = 0.f) {
    constexpr int kSimds = 1024;
    const int team = kEf && total < kSimds ? 1 : encode_team<kUseDct, kEf>();
    const int64_t piece = kMaxGroups256 * team;  // chunks of one launch
    for (int64_t first = 0; first < total; first += piece) {
        const int64_t end = total - first < piece ? total : first + piece;
        hipLaunchKernelGGL((k_encode_chunk<kTwo, kUseDct, kEf>), dim3(grid8((end - first + team - 1) / team)), dim3(64 * team), 0,
                           static_cast<hipStream_t>(stream), d_desc, single, n_tensors, first, end, k, d_idx12, d_val, d_grad_desc,
                           decay, team);
    }
    return launch_status();
}

// A set with the transform: ranges of the chunk list for one resident round of waves, or a chunk per wave?  The ranges differ
// by a chunk, which the whole device waits for - with a handful of chunks a wave that is most of the last round - where the
// other looks up every chunk's tensor.  In us, ranges against a chunk per wave (k = 32 / 64): 2560 chunks 16.6 : 18.1 / 18.4 : 19.6; 5120
// 28.3 : 27.6 / 32.2 : 30.5; 10 240 43.7 : 40.7 / 51.7 : 47.8; 15 360 57.4 : 56.5 / 67.9 : 65.0; 20 480 72.7 : 75.5 / 88.4 : 80.7; 61 440 194 : 195 / 223 :
// 219; 294 144 879 : 928 / 1015 : 1040.
template <bool kTwo>
static bool walks(int64_t total, int& resident) {
    static const int waves = persistent_grid(k_encode_topk_pack<kTwo>, int64_t{1} << 40);
    resident = waves;
    return total <= waves || total > static_cast<int64_t>(waves) * (kTwo ? 20 : 5);
}

template <bool kTwo>
static int launch_set(const tplr_tensor_desc* d_desc, int n_tensors, int64_t total, int k, uint8_t* d_idx12, float* d_val,
                      void* stream) {
    int resident;
    if (!walks<kTwo>(total, resident))
        return launch_chunks<kTwo, true>(d_desc, tplr_tensor_desc{}, n_tensors, total, k, d_idx12, d_val, stream);
    const int64_t need = ((total + 7) / 8) * 8;
    hipLaunchKernelGGL(k_encode_topk_pack<kTwo>, dim3(static_cast<unsigned>(need < resident ? need : resident)), dim3(64), 0,
                       static_cast<hipStream_t>(stream), d_desc, n_tensors, total, k, d_idx12, d_val);
    return launch_status();
}

}  // namespace tplr

using namespace tplr;

extern "C" int tplr_encode_topk_pack(const float* d_x, int64_t R, int64_t C, int64_t ld_x, int k, int use_dct, uint8_t* d_idx12,
                                     float* d_val, void* stream) {
    if (int s = check_2d(d_x, d_val, R, C)) return s;
    if (!d_idx12 || ld_x < C || k < 2 || (k & 1) || k > kCandCap) return TPLR_E_BADARG;
    const int64_t n = (R / 64) * (C / 64);
    if (n == 0) return 0;
    if (C / 64 > 0x7fffffff || R / 64 > 0x7fffffff || !ld_ok(ld_x)) return TPLR_E_TOOMANY;
    tplr_tensor_desc single;
    single.dense = const_cast<float*>(d_x);
    single.ld = ld_x;
    single.chunk_begin = 0;
    single.x_chunks = static_cast<int32_t>(C / 64);
    single.y_chunks = static_cast<int32_t>(R / 64);
    if (k > 32)
        return use_dct ? launch_chunks<true, true>(nullptr, single, 1, n, k, d_idx12, d_val, stream)
                       : launch_chunks<true, false>(nullptr, single, 1, n, k, d_idx12, d_val, stream);
    return use_dct ? launch_chunks<false, true>(nullptr, single, 1, n, k, d_idx12, d_val, stream)
                   : launch_chunks<false, false>(nullptr, single, 1, n, k, d_idx12, d_val, stream);
}

extern "C" int tplr_encode_topk_pack_batch(const tplr_tensor_desc* d_desc, int n_tensors, int64_t total_chunks, int k, int use_dct,
                                           uint8_t* d_idx12, float* d_val, void* stream) {
    if (!d_desc || n_tensors < 1 || total_chunks < 0 || !d_idx12 || !d_val || k < 2 || (k & 1) || k > kCandCap)
        return TPLR_E_BADARG;
    if (total_chunks == 0) return 0;
    const tplr_tensor_desc none = {};
    if (use_dct)
        return k > 32 ? launch_set<true>(d_desc, n_tensors, total_chunks, k, d_idx12, d_val, stream)
                      : launch_set<false>(d_desc, n_tensors, total_chunks, k, d_idx12, d_val, stream);
    return k > 32 ? launch_chunks<true, false>(d_desc, none, n_tensors, total_chunks, k, d_idx12, d_val, stream)
                  : launch_chunks<false, false>(d_desc, none, n_tensors, total_chunks, k, d_idx12, d_val, stream);
}

extern "C" int tplr_ef_encode_topk_pack_batch(const tplr_tensor_desc* d_ef_desc, const tplr_tensor_desc* d_grad_desc, int n_tensors,
                                              int64_t total_chunks, float decay, int k, int use_dct, uint8_t* d_idx12, float* d_val,
                                              void* stream) {
    if (!d_ef_desc || !d_grad_desc || n_tensors < 1 || total_chunks < 0 || !d_idx12 || !d_val || k < 2 || (k & 1) || k > kCandCap)
        return TPLR_E_BADARG;
    if (total_chunks == 0) return 0;
    const tplr_tensor_desc none = {};
#define TPLR_EF(TWO, DCT) \
    launch_chunks<TWO, DCT, true>(d_ef_desc, none, n_tensors, total_chunks, k, d_idx12, d_val, stream, d_grad_desc, decay)
    if (k > 32) return use_dct ? TPLR_EF(true, true) : TPLR_EF(true, false);
    return use_dct ? TPLR_EF(false, true) : TPLR_EF(false, false);
#undef TPLR_EF
}

extern "C" int tplr_calib_encode(const tplr_tensor_desc* d_desc, int n_tensors, int64_t total_chunks, void* stream) {
    if (!d_desc || n_tensors < 1 || total_chunks < 0) return TPLR_E_BADARG;
    if (total_chunks == 0) return 0;
    static int resident = 0;
    if (resident == 0) resident = persistent_grid(k_encode_topk_pack<false>, int64_t{1} << 40);  // the grid it stands in for
    const int64_t need = ((total_chunks + 7) / 8) * 8;
    tplr_tensor_desc none = {};
    hipLaunchKernelGGL(k_calib_encode, dim3(static_cast<unsigned>(need < resident ? need : resident)), dim3(64), 0,
                       static_cast<hipStream_t>(stream), d_desc, none, n_tensors, total_chunks,
                       static_cast<float*>(nullptr));
    return launch_status();
}
