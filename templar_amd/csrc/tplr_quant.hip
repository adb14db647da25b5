// The statistical quantiser over the values sent (TopKCompressor._quantize_values and _dequantize_values,
// src/tplr/compress.py:582-644).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "../../include/tplr_hip.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

// Three launches over slices of every tensor: the moments, the codes with per-bin sums, the tables.  Of one tensor with up to
// eight bins two: the workgroup that finishes its codes last makes the table, which saves a launch of 4 us.  With more bins
// that workgroup would read up to a megabyte by itself, its lanes 4 KB apart: of 262 144 values a whole call with 256 bins
// takes 98.9 us that way and 17.6 us with a wave per bin, with 64 bins 32.9 and 17.6.  Partial sums are
// carried in double, kept per (tensor, slice) in a caller-provided workspace and added in a fixed order by whoever
// needs the total, so every workgroup of a tensor derives the same shift and scale.
// Workspace layout (doubles): moments[T][S][2], then bins[T][S][2 * n_bins] (sums, counts).
//
// The moments are taken about the tensor's first value, where value - first is exact in double: sum (x - first) and
// sum (x - first)^2 in one pass over the values give the mean and, about the rounded mean, the sum of squares of the
// centred values (:594-597) - zero exactly for a constant tensor, as the reference's second pass has it, and otherwise
// with the thirteen digits that are left of a double when the first value lies ten standard deviations out.  Where the
// first value is not finite they are taken about zero: the mean of values with one infinity is that infinity (:594).
struct QuantSlice {
    const float4* v;
    uchar4* q;
    int64_t n4;   // float4 groups in this slice
    int64_t n;    // values in the whole tensor
    float first;  // the tensor's first value, or zero
    int t, s;
};

// what the moments of n values from v[0] on are taken about
__device__ __forceinline__ float quant_pivot(const float* v, int64_t n) {
    const float x = n > 0 ? *v : 0.f;
    return __builtin_fabsf(x) < __builtin_inff() ? x : 0.f;  // (NaN: zero)
}

// (`table` null: `single` is the one tensor)
__device__ __forceinline__ QuantSlice quant_slice(const float* val, uint8_t* codes, const tplr_tensor_desc* table,
                                                   const tplr_tensor_desc& single, int k, int S) {
    QuantSlice qs;
    qs.t = blockIdx.x / S;
    qs.s = blockIdx.x - qs.t * S;
    const tplr_tensor_desc d = table ? table[qs.t] : single;
    const int64_t rows = static_cast<int64_t>(d.x_chunks) * d.y_chunks;
    const int64_t r0 = rows * qs.s / S, r1 = rows * (qs.s + 1) / S;
    qs.v = reinterpret_cast<const float4*>(val + (d.chunk_begin + r0) * k);
    qs.q = codes ? reinterpret_cast<uchar4*>(codes + (d.chunk_begin + r0) * k) : nullptr;
    qs.n4 = (r1 - r0) * k >> 2;  // k is a multiple of 4
    qs.n = rows * k;
    qs.first = quant_pivot(val + d.chunk_begin * k, rows);
    return qs;
}

// shift and scale of tensor t from its slices' moments; the whole wave takes part
__device__ __forceinline__ void quant_shift_scale(const double* work, int t, int S, int64_t n, float first, int n_bins,
                                                  float range_in_sigmas, float& shift, float& scale) {
    const double2* m = reinterpret_cast<const double2*>(work) + static_cast<int64_t>(t) * S;
    double s1 = 0.0, s2 = 0.0;
    for (int i = threadIdx.x & 63; i < S; i += 64) s1 += m[i].x, s2 += m[i].y;
    s1 = wave_sum_f64(s1);
    s2 = wave_sum_f64(s2);
    const double cnt = static_cast<double>(n);
    shift = static_cast<float>(static_cast<double>(first) + s1 / cnt);                  // :594
    const double off = static_cast<double>(shift) - static_cast<double>(first);
    double ss = s2 - 2.0 * off * s1 + cnt * off * off;  // sum (x - shift)^2
    ss = ss < 0.0 ? 0.0 : ss;
    const float sd = static_cast<float>(sqrt(ss) / sqrt(cnt - 1.0));                    // :597
    const float sc = range_in_sigmas * sd / static_cast<float>(n_bins);                 // :598
    scale = (sc == 0.f || sc != sc || __builtin_isinf(sc)) ? 1.0f : sc;                 // :599-600
}

// Doubles that another workgroup of the same launch reads: stored to and loaded from where the whole device sees them.
// (Ordinary stores with a release and an acquire around them write back and invalidate an XCD's whole L2 per workgroup:
// 20 us for 256 of them.)
__device__ __forceinline__ void device_store(double* p, double x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double device_load(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the mean of bin `bin` from the slices' sums and counts, dealt over the lanes of a wave (:619)
__device__ __forceinline__ float quant_bin_mean(const double* bins, int S, int n_bins, int bin) {
    double sum = 0.0, cnt = 0.0;
    for (int s = threadIdx.x & 63; s < S; s += 64)
        sum += device_load(bins + s * 2 * n_bins + bin), cnt += device_load(bins + s * 2 * n_bins + n_bins + bin);
    sum = wave_sum_f64(sum);
    cnt = wave_sum_f64(cnt);
    return cnt > 0.0 ? static_cast<float>(sum / cnt) : 0.f;
}

// One tensor's results where its codes are made (k_quant_codes), instead of a launch of their own.
struct QuantOne {
    uint32_t* done;  // slices finished, zeroed by k_quant_moments; null: k_quant_tables makes the table
    float *shift, *scale, *lookup;  // null: k_quant_tables stores all
};

__global__ __launch_bounds__(256) void k_quant_moments(const float* __restrict__ val, int k,
                                                       const tplr_tensor_desc* __restrict__ table,
                                                       const tplr_tensor_desc single, int S,
                                                       double* __restrict__ work, uint32_t* __restrict__ done) {
    __shared__ double part[2][4];
    const int tid = threadIdx.x;
    if (done && blockIdx.x == 0 && tid == 0) *done = 0u;
    const QuantSlice qs = quant_slice(val, nullptr, table, single, k, S);
    const double first = static_cast<double>(qs.first);
    double s1 = 0.0, s2 = 0.0;
    for (int64_t i = tid; i < qs.n4; i += 256) {
        const float4 x = qs.v[i];
        const double a = x.x - first, b = x.y - first, c = x.z - first, e = x.w - first;
        s1 += (a + b) + (c + e);
        s2 += (a * a + b * b) + (c * c + e * e);
    }
    s1 = wave_sum_f64(s1);
    s2 = wave_sum_f64(s2);
    if ((tid & 63) == 0) part[0][tid >> 6] = s1, part[1][tid >> 6] = s2;
    __syncthreads();
    if (tid < 2) work[2 * static_cast<int64_t>(blockIdx.x) + tid] = (part[tid][0] + part[tid][1]) + (part[tid][2] + part[tid][3]);
}

// kBins: a handful of bins (templar runs four), 4 or 8 of them kept in registers per thread, no contended atomics;
// 0: up to 256 bins in LDS.  A thread adds its value to every bin, zero to all but one: four times two instructions a
// value with four bins, where the eight-bin form with counts in double took 89 us for the 1B set's 19 million values
// and this one 60 us (one parameter of 262 144 values: 19.3 us in 16 slices, now 5.5 in 256).
template <int kBins>
__global__ __launch_bounds__(256) void k_quant_codes(const float* __restrict__ val, int k,
                                                     const tplr_tensor_desc* __restrict__ table,
                                                     const tplr_tensor_desc single, int T, int S, int n_bins,
                                                     float range_in_sigmas, uint8_t* __restrict__ codes,
                                                     double* __restrict__ work, const QuantOne one) {
    const int tid = threadIdx.x;
    const QuantSlice qs = quant_slice(val, codes, table, single, k, S);
    float shift, scale;
    quant_shift_scale(work, qs.t, S, qs.n, qs.first, n_bins, range_in_sigmas, shift, scale);
    if (one.scale && blockIdx.x == 0 && tid == 0) {
        *one.shift = shift;
        // (the caller may be watching for it in pinned host memory while this launch goes on)
        __hip_atomic_store(one.scale, scale, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    double* out = work + 2 * static_cast<int64_t>(T) * S + static_cast<int64_t>(blockIdx.x) * 2 * n_bins;
    const float offset = static_cast<float>(n_bins / 2), top = static_cast<float>(n_bins - 1);
    auto code = [&](float x, float& c) {
        c = x - shift;                                  // :595
        float r = __builtin_rintf(c / scale + offset);  // :604-605, ties to even as torch.round
        r = r < 0.f ? 0.f : r;
        r = r > top ? top : r;                          // :606
        return static_cast<uint32_t>(r);
    };
    if constexpr (kBins > 0) {
        __shared__ double sums[4][kBins];
        __shared__ uint32_t counts[4][kBins];
        double s[kBins];
        uint32_t n[kBins];
#pragma unroll
        for (int b = 0; b < kBins; ++b) s[b] = 0.0, n[b] = 0u;
        auto tally = [&](uint32_t q, float c) {  // :614-617
#pragma unroll
            for (int b = 0; b < kBins; ++b) {
                const bool in = q == static_cast<uint32_t>(b);
                s[b] += static_cast<double>(in ? c : 0.f);
                n[b] += in ? 1u : 0u;
            }
        };
        for (int64_t i = tid; i < qs.n4; i += 256) {
            const float4 x = qs.v[i];
            float c0, c1, c2, c3;
            const uint32_t q0 = code(x.x, c0), q1 = code(x.y, c1), q2 = code(x.z, c2), q3 = code(x.w, c3);
            qs.q[i] = make_uchar4(static_cast<unsigned char>(q0), static_cast<unsigned char>(q1),
                                  static_cast<unsigned char>(q2), static_cast<unsigned char>(q3));
            tally(q0, c0), tally(q1, c1), tally(q2, c2), tally(q3, c3);
        }
#pragma unroll
        for (int b = 0; b < kBins; ++b) {
            const double sum = wave_sum_f64(s[b]);
            const uint32_t cnt = wave_sum_u32(n[b]);
            if ((tid & 63) == 0) sums[tid >> 6][b] = sum, counts[tid >> 6][b] = cnt;
        }
        __syncthreads();
        if (tid < n_bins) {
            device_store(out + tid, (sums[0][tid] + sums[1][tid]) + (sums[2][tid] + sums[3][tid]));
            device_store(out + n_bins + tid, static_cast<double>(counts[0][tid] + counts[1][tid] + counts[2][tid] + counts[3][tid]));
        }
    } else {
        __shared__ double bin_sum[256];
        __shared__ unsigned int bin_cnt[256];
        bin_sum[tid] = 0.0, bin_cnt[tid] = 0u;
        __syncthreads();
        for (int64_t i = tid; i < qs.n4; i += 256) {
            const float4 x = qs.v[i];
            float c0, c1, c2, c3;
            const uint32_t q0 = code(x.x, c0), q1 = code(x.y, c1), q2 = code(x.z, c2), q3 = code(x.w, c3);
            qs.q[i] = make_uchar4(static_cast<unsigned char>(q0), static_cast<unsigned char>(q1),
                                  static_cast<unsigned char>(q2), static_cast<unsigned char>(q3));
            atomicAdd(&bin_sum[q0], static_cast<double>(c0)), atomicAdd(&bin_cnt[q0], 1u);  // :614-617
            atomicAdd(&bin_sum[q1], static_cast<double>(c1)), atomicAdd(&bin_cnt[q1], 1u);
            atomicAdd(&bin_sum[q2], static_cast<double>(c2)), atomicAdd(&bin_cnt[q2], 1u);
            atomicAdd(&bin_sum[q3], static_cast<double>(c3)), atomicAdd(&bin_cnt[q3], 1u);
        }
        __syncthreads();
        if (tid < n_bins) device_store(out + tid, bin_sum[tid]), device_store(out + n_bins + tid, static_cast<double>(bin_cnt[tid]));
    }
    if (one.done) {  // uniform: the workgroup that finishes last, whichever that is, makes the table
        __shared__ uint32_t before;
        // every wave's sums have reached the device's memory before the workgroup's arrival is counted
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) before = __hip_atomic_fetch_add(one.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (before == static_cast<uint32_t>(S) - 1u) {  // (so all have arrived, and the loads below are behind that)
            const double* bins = work + 2 * static_cast<int64_t>(T) * S;
            for (int bin = tid >> 6; bin < n_bins; bin += 4) {
                const float mean = quant_bin_mean(bins, S, n_bins, bin);
                if ((tid & 63) == 0) one.lookup[bin] = mean;
            }
        }
    }
}

// One wave per bin of tensor blockIdx.y, and bin 0's the scalars (null: they are stored already).
__global__ __launch_bounds__(64) void k_quant_tables(const float* __restrict__ val, const tplr_tensor_desc* __restrict__ table,
                                                     const tplr_tensor_desc single, int k, int T, int S, int n_bins, float range_in_sigmas,
                                                     const double* __restrict__ work, float* __restrict__ shift_out,
                                                     float* __restrict__ scale_out, float* __restrict__ lookup) {
    const int t = blockIdx.y, bin = blockIdx.x, lane = threadIdx.x;
    const float mean = quant_bin_mean(work + 2 * static_cast<int64_t>(T) * S + static_cast<int64_t>(t) * S * 2 * n_bins, S, n_bins, bin);
    if (lane == 0) lookup[static_cast<int64_t>(t) * n_bins + bin] = mean;
    if (bin == 0 && scale_out) {  // wave-uniform
        const tplr_tensor_desc d = table ? table[t] : single;
        const int64_t n = static_cast<int64_t>(d.x_chunks) * d.y_chunks * k;
        float shift, scale;
        quant_shift_scale(work, t, S, n, quant_pivot(val + d.chunk_begin * k, n), n_bins, range_in_sigmas, shift, scale);
        if (lane == 0) shift_out[t] = shift, scale_out[t] = scale;
    }
}

// De-quantise one peer's flat payload of 8-bit codes: value = lookup[t][code] + shift[t], the
// tensor t found from the row id (:637-643 for every parameter of the set at once).  Four codes per thread.
__global__ __launch_bounds__(256) void k_dequantize_batch(const uint8_t* __restrict__ q,
                                                          const float* __restrict__ lookup,
                                                          const float* __restrict__ shift, int n_bins, int k,
                                                          const tplr_tensor_desc* __restrict__ table, int n_tensors,
                                                          int64_t n4, float* __restrict__ val) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n4; i += stride) {
        const int64_t row = (i * 4) / k;  // k is a multiple of 4 here: the four codes share a row
        int lo = 0, hi = n_tensors;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (table[mid].chunk_begin <= row)
                lo = mid;
            else
                hi = mid;
        }
        const uchar4 c = reinterpret_cast<const uchar4*>(q)[i];
        const float* lk = lookup + static_cast<int64_t>(lo) * n_bins;
        const float sh = shift[lo];
        float4 o;
        o.x = lk[c.x < n_bins ? c.x : n_bins - 1] + sh;
        o.y = lk[c.y < n_bins ? c.y : n_bins - 1] + sh;
        o.z = lk[c.z < n_bins ? c.z : n_bins - 1] + sh;
        o.w = lk[c.w < n_bins ? c.w : n_bins - 1] + sh;
        reinterpret_cast<float4*>(val)[i] = o;
    }
}

struct DeqPtrs {
    const uint8_t* codes[TPLR_MAX_PEERS];
    float* out[TPLR_MAX_PEERS];
};

// One parameter's codes of P peers, each with its own lookup and shift: block row p serves peer p.
__global__ __launch_bounds__(256) void k_dequantize_peers(const DeqPtrs pp, int64_t n4,
                                                          const float* __restrict__ lookup,
                                                          const float* __restrict__ shift, int n_bins) {
    const int p = blockIdx.y;
    const uchar4* q = reinterpret_cast<const uchar4*>(pp.codes[p]);
    float4* o = reinterpret_cast<float4*>(pp.out[p]);
    const float* lk = lookup + static_cast<int64_t>(p) * n_bins;
    const float sh = shift[p];
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n4; i += stride) {
        const uchar4 c = q[i];
        float4 r;
        r.x = lk[c.x < n_bins ? c.x : n_bins - 1] + sh;
        r.y = lk[c.y < n_bins ? c.y : n_bins - 1] + sh;
        r.z = lk[c.z < n_bins ? c.z : n_bins - 1] + sh;
        r.w = lk[c.w < n_bins ? c.w : n_bins - 1] + sh;
        o[i] = r;
    }
}

// The same with every peer's lookup and shift where they lie, up to kListPeers of them per launch.
constexpr int kListPeers = 32;
struct DeqLists {
    const uint8_t* codes[kListPeers];
    const float* lookup[kListPeers];
    const float* shift[kListPeers];
    float* out[kListPeers];
};

__global__ __launch_bounds__(256) void k_dequantize_lists(const DeqLists pp, int64_t n4, int n_bins) {
    const int p = blockIdx.y;
    const uchar4* q = reinterpret_cast<const uchar4*>(pp.codes[p]);
    float4* o = reinterpret_cast<float4*>(pp.out[p]);
    const float* lk = pp.lookup[p];
    const float sh = *pp.shift[p];
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n4; i += stride) {
        const uchar4 c = q[i];
        float4 r;
        r.x = lk[c.x < n_bins ? c.x : n_bins - 1] + sh;
        r.y = lk[c.y < n_bins ? c.y : n_bins - 1] + sh;
        r.z = lk[c.z < n_bins ? c.z : n_bins - 1] + sh;
        r.w = lk[c.w < n_bins ? c.w : n_bins - 1] + sh;
        o[i] = r;
    }
}

// `one`: a single tensor (its descriptor `single`) with d_shift and d_scale stored early
static int launch_quantize(const float* d_val, int k, const tplr_tensor_desc* d_desc, const tplr_tensor_desc& single, int n_tensors, int n_bins,
                           float range_in_sigmas, int n_slices, double* d_work, uint8_t* d_codes, float* d_shift,
                           float* d_scale, float* d_lookup, void* stream, bool one = false) {
    const dim3 grid(static_cast<unsigned>(n_tensors) * n_slices), block(256);
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint32_t* done = one && n_bins <= 8 ? reinterpret_cast<uint32_t*>(d_work + static_cast<int64_t>(n_slices) * (2 + 2 * n_bins)) : nullptr;
    const QuantOne results = {done, one ? d_shift : nullptr, one ? d_scale : nullptr, one ? d_lookup : nullptr};
    hipLaunchKernelGGL(k_quant_moments, grid, block, 0, st, d_val, k, d_desc, single, n_slices, d_work, done);
    hipLaunchKernelGGL(n_bins <= 4 ? k_quant_codes<4> : n_bins <= 8 ? k_quant_codes<8> : k_quant_codes<0>, grid, block, 0, st,
                       d_val, k, d_desc, single, n_tensors, n_slices, n_bins, range_in_sigmas, d_codes, d_work, results);
    if (!done)
        hipLaunchKernelGGL(k_quant_tables, dim3(static_cast<unsigned>(n_bins), static_cast<unsigned>(n_tensors)), dim3(64), 0, st,
                           d_val, d_desc, single, k, n_tensors, n_slices, n_bins, range_in_sigmas, d_work, one ? nullptr : d_shift,
                           one ? nullptr : d_scale, d_lookup);
    return launch_status();
}

static int check_quantize(const float* d_val, int k, const tplr_tensor_desc* d_desc, int n_tensors, int n_bins,
                          int n_slices, const uint8_t* d_codes, const float* d_shift, const float* d_scale,
                          const float* d_lookup, bool one = false) {
    if (!d_val || (!d_desc && !one) || !d_codes || !d_shift || !d_scale || !d_lookup || n_tensors < 1 || k < 4 || (k & 3) ||
        n_bins < 1 || n_bins > 256 || n_slices < 1 || n_slices > 1024)
        return TPLR_E_BADARG;
    if ((reinterpret_cast<uintptr_t>(d_val) & 15) || (reinterpret_cast<uintptr_t>(d_codes) & 3)) return TPLR_E_BADARG;
    if (static_cast<int64_t>(n_tensors) * n_slices > 0x7fffffff) return TPLR_E_TOOMANY;
    return 0;
}

}  // namespace tplr

using namespace tplr;

extern "C" {

int tplr_dequantize_peers(const uint8_t* const* h_codes, int n_peers, int64_t n, const float* d_lookup,
                          const float* d_shift, int n_bins, float* const* h_out, void* stream) {
    if (!h_codes || !h_out || !d_lookup || !d_shift || n_peers < 1 || n < 0 || (n & 3) || n_bins < 1 || n_bins > 256)
        return TPLR_E_BADARG;
    if (n_peers > TPLR_MAX_PEERS) return TPLR_E_TOOMANY;
    if (n == 0) return 0;
    DeqPtrs pp;
    for (int p = 0; p < TPLR_MAX_PEERS; ++p) {
        pp.codes[p] = p < n_peers ? h_codes[p] : nullptr;
        pp.out[p] = p < n_peers ? h_out[p] : nullptr;
        if (p < n_peers && (!pp.codes[p] || !pp.out[p] || (reinterpret_cast<uintptr_t>(pp.codes[p]) & 3) ||
                            (reinterpret_cast<uintptr_t>(pp.out[p]) & 15)))
            return TPLR_E_BADARG;
    }
    const int64_t n4 = n >> 2;
    int64_t bx = (n4 + 255) / 256;
    bx = bx > 2048 ? 2048 : bx;
    hipLaunchKernelGGL(k_dequantize_peers, dim3(static_cast<unsigned>(bx), static_cast<unsigned>(n_peers)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), pp, n4, d_lookup, d_shift, n_bins);
    return launch_status();
}

int tplr_dequantize_lists(const uint8_t* const* h_codes, int n_peers, int64_t n, const float* const* h_lookup,
                          const float* const* h_shift, int n_bins, float* const* h_out, void* stream) {
    if (!h_codes || !h_out || !h_lookup || !h_shift || n_peers < 1 || n < 0 || (n & 3) || n_bins < 1 || n_bins > 256)
        return TPLR_E_BADARG;
    if (n_peers > TPLR_MAX_PEERS) return TPLR_E_TOOMANY;
    if (n == 0) return 0;
    for (int p = 0; p < n_peers; ++p)
        if (!h_codes[p] || !h_out[p] || !h_lookup[p] || !h_shift[p] || (reinterpret_cast<uintptr_t>(h_codes[p]) & 3) ||
            (reinterpret_cast<uintptr_t>(h_out[p]) & 15))
            return TPLR_E_BADARG;
    const int64_t n4 = n >> 2;
    int64_t bx = (n4 + 255) / 256;
    bx = bx > 2048 ? 2048 : bx;
    for (int p0 = 0; p0 < n_peers; p0 += kListPeers) {
        DeqLists pp = {};
        const int count = n_peers - p0 < kListPeers ? n_peers - p0 : kListPeers;
        for (int p = 0; p < count; ++p) {
            pp.codes[p] = h_codes[p0 + p];
            pp.lookup[p] = h_lookup[p0 + p];
            pp.shift[p] = h_shift[p0 + p];
            pp.out[p] = h_out[p0 + p];
        }
        hipLaunchKernelGGL(k_dequantize_lists, dim3(static_cast<unsigned>(bx), static_cast<unsigned>(count)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), pp, n4, n_bins);
    }
    return launch_status();
}

int tplr_quantize_batch(const float* d_val, int k, const tplr_tensor_desc* d_desc, int n_tensors, int n_bins,
                        float range_in_sigmas, int n_slices, double* d_work, uint8_t* d_codes, float* d_shift,
                        float* d_scale, float* d_lookup, void* stream) {
    if (!d_work || (reinterpret_cast<uintptr_t>(d_work) & 7)) return TPLR_E_BADARG;
    if (int s = check_quantize(d_val, k, d_desc, n_tensors, n_bins, n_slices, d_codes, d_shift, d_scale, d_lookup))
        return s;
    return launch_quantize(d_val, k, d_desc, tplr_tensor_desc{}, n_tensors, n_bins, range_in_sigmas, n_slices, d_work, d_codes, d_shift,
                           d_scale, d_lookup, stream);
}

int tplr_quantize(const float* d_val, int64_t n, int n_bins, float range_in_sigmas, int n_slices, double* d_work,
                  uint8_t* d_codes, float* d_shift, float* d_scale, float* d_lookup, void* stream) {
    if (!d_work || (reinterpret_cast<uintptr_t>(d_work) & 7) || n < 4 || (n & 3)) return TPLR_E_BADARG;
    if (int s = check_quantize(d_val, 4, nullptr, 1, n_bins, n_slices, d_codes, d_shift, d_scale, d_lookup, true)) return s;
    if (n / 4 > 0x7fffffff) return TPLR_E_TOOMANY;
    tplr_tensor_desc single = {};
    single.x_chunks = static_cast<int32_t>(n / 4);  // rows of four values
    single.y_chunks = 1;
    return launch_quantize(d_val, 4, nullptr, single, 1, n_bins, range_in_sigmas, n_slices, d_work, d_codes, d_shift, d_scale,
                           d_lookup, stream, true);
}

int tplr_dequantize_batch(const uint8_t* d_codes, const float* d_lookup, const float* d_shift, int n_bins, int k,
                          const tplr_tensor_desc* d_desc, int n_tensors, int64_t total_rows, float* d_val,
                          void* stream) {
    if (!d_codes || !d_lookup || !d_shift || !d_desc || !d_val || n_bins < 1 || n_bins > 256 || k < 4 || (k & 3) ||
        n_tensors < 1 || total_rows < 0)
        return TPLR_E_BADARG;
    if ((reinterpret_cast<uintptr_t>(d_codes) & 3) || (reinterpret_cast<uintptr_t>(d_val) & 15)) return TPLR_E_BADARG;
    if (total_rows == 0) return 0;
    const int64_t n4 = total_rows * k / 4;
    const int64_t blocks = (n4 + 255) / 256;
    hipLaunchKernelGGL(k_dequantize_batch, dim3(static_cast<unsigned>(blocks < 65536 ? blocks : 65536)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), d_codes, d_lookup, d_shift, n_bins, k, d_desc, n_tensors, n4,
                       d_val);
    return launch_status();
}

}  // extern "C"

// ---- the quantiser without a caller-provided workspace ----------------------------------------
// The partial sums of tplr_quantize_batch live in a file-scope device array instead.  The array's
// name is a host-side handle, not a device address: its address on the current device comes from
// hipGetSymbolAddress, once per device, and only that pointer is handed to kernels.
static __device__ __align__(256) double scratch[TPLR_STATIC_WORK_DOUBLES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex scratch_lock;
double* scratch_ptr[kMaxDevices];  // per device: every GPU holds its own copy of the array

// the array's address on the current device; nullptr with *status set when it cannot be had
double* scratch_on_current_device(int* status) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *status = static_cast<int>(e);
        return nullptr;
    }
    if (dev < 0 || dev >= kMaxDevices) {
        *status = TPLR_E_TOOMANY;
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(scratch_lock);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            *status = e != hipSuccess ? static_cast<int>(e) : TPLR_E_BADARG;
            return nullptr;
        }
        scratch_ptr[dev] = static_cast<double*>(p);
    }
    return scratch_ptr[dev];
}
}  // namespace

extern "C" {

int64_t tplr_static_work_bytes(void) { return static_cast<int64_t>(TPLR_STATIC_WORK_DOUBLES) * 8; }

int tplr_quantize_batch_static(const float* d_val, int k, const tplr_tensor_desc* d_desc, int n_tensors, int n_bins,
                               float range_in_sigmas, int n_slices, uint8_t* d_codes, float* d_shift, float* d_scale,
                               float* d_lookup, void* stream) {
    if (int s = check_quantize(d_val, k, d_desc, n_tensors, n_bins, n_slices, d_codes, d_shift, d_scale, d_lookup))
        return s;
    const int64_t need = static_cast<int64_t>(n_tensors) * n_slices * (2 + 2 * static_cast<int64_t>(n_bins));
    if (need > TPLR_STATIC_WORK_DOUBLES) return TPLR_E_WORKSPACE;
    int status = 0;
    double* work = scratch_on_current_device(&status);
    if (!work) return status;
    return launch_quantize(d_val, k, d_desc, tplr_tensor_desc{}, n_tensors, n_bins, range_in_sigmas, n_slices, work, d_codes, d_shift,
                           d_scale, d_lookup, stream);
}

}  // extern "C"
