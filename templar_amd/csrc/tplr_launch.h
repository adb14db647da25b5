// Host-side launch helpers shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tplr_hip.h"

namespace tplr {

inline int launch_status() {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

// workgroups of 256 threads in one launch, which has fewer than 2^32 threads
constexpr int64_t kMaxGroups256 = 0xfffff0;

inline unsigned grid8(int64_t n) { return static_cast<unsigned>(((n + 7) / 8) * 8); }

inline int check_2d(const void* a, const void* b, int64_t R, int64_t C) {
    if (!a || !b || R < 0 || C < 0) return TPLR_E_BADARG;
    if ((R % 64) || (C % 64)) return TPLR_E_SHAPE;
    return 0;
}

// chunk rows are addressed with 32-bit byte offsets (63 rows * ld * 4 bytes)
inline bool ld_ok(int64_t ld) { return ld > 0 && ld <= (int64_t{1} << 23); }

// persistent grids: exactly one resident set of workgroups of `threads` threads (one wave, or a team of
// waves), as the occupancy calculator reports it for the kernel at hand (registers or LDS bound it); a
// larger grid would leave a second, mostly empty round
template <typename Kernel>
int persistent_grid(Kernel kernel, int64_t total, int threads = 64) {
    int n_cu = 256, per_cu = 0, dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
        n_cu = v;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess || per_cu < 1)
        per_cu = threads > 64 ? 2 : 4;
    int64_t g = static_cast<int64_t>(n_cu) * per_cu;
    g = g < 8 ? 8 : (g / 8) * 8;
    const int64_t need = ((total + 7) / 8) * 8;
    return static_cast<int>(need < g ? need : g);
}

// The aggregate with the transform, a chunk per wave, where that is the way to go (mean: as the reference, otherwise the sum;
// with_sum: d_stats takes two floats a chunk, otherwise the sum of squares alone), subtract: dst - result, chunks whose
// result is not finite left and their tensors flagged in d_guard.  single: the tensor where d_desc is null.  The arguments
// checked by the caller.
bool decode_chunks_serves(int n_peers, int k, int64_t total, bool subtract);
int decode_chunks(const uint8_t* const* h_idx12, const float* const* h_val, const float* d_scale, int n_peers, int k,
                  const tplr_tensor_desc* d_desc, const tplr_tensor_desc& single, int n_tensors, int64_t total, bool subtract,
                  bool mean, bool with_sum, float* d_stats, int32_t* d_guard, void* stream);

// The persistent aggregate of one parameter (k <= 64, at most 24 peers, mean, no transform) with the clip factors made from
// n_norms <= 64 norms inside the launch; the arguments checked by the caller (tplr_aggregate_param).
int aggregate_from_norms(const uint8_t* const* h_idx12, const float* const* h_val, const float* d_norms, int n_norms, int n_peers,
                         int k, int64_t R, int64_t C, float* d_out, int64_t ld_out, void* stream);

}  // namespace tplr
