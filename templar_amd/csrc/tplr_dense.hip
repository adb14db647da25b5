// Dense per-chunk contraction with the caller's bases: chunk edges other than 64, transforms whose norm is not
// "ortho", and ChunkingTransformer.einsum_2d with any matrices (src/tplr/compress.py:186-222).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tplr_hip.h"
#include "tplr_device.h"
#include "tplr_launch.h"

namespace tplr {

typedef float v4acc __attribute__((ext_vector_type(4)));

// O = Bh^T X Bw per chunk on the fp32 matrix instructions (16x16x4: operand A lane l holds A[l%16][l/16], operand B
// B[l/16][l%16], the result's register r holds D[4(l/16)+r][l%16]).
//
// What bounds it: (h + w) multiply-adds per element are 110 for a 60 x 50 chunk, 28 flop per byte moved, above the
// balance of the vector ALU (without packed operations 78 Tflop/s) and about at that of the matrix cores in fp32
// (157 Tflop/s): the 3000 x 1000 tensor's 0.7 Gflop are 4.5 us there and its 24 MB about as long in memory.
//
// Layout: a workgroup of four waves takes kStack chunks at a time, so that four 16-row strips are there for the four
// waves in either pass whatever the chunk's size (edges up to 16 and 32 stack four and two chunks; kMT, kNT: tiles
// of 16 rows and columns, 1, 2 or 4).  Pass 1: wave w makes rows 16 (w mod kMT) .. of T = Bh^T X, its strip of Bh
// in kMT * 4 registers for the whole launch, X staged in LDS (zero outside the chunk, so that padded steps of the
// contraction add nothing); T goes to LDS.  Pass 2: wave w makes columns 16 (w mod kNT) .. of T Bw, its strip of Bw in
// registers.  Row strides: X is read four rows by sixteen columns at a time (stride 16 mod 64 words: four distinct
// quarters of the banks), T sixteen rows by four columns (stride 4 mod 64).  The next chunks' rows are requested
// before pass 1 and arrive during the arithmetic.  Tile counts are template arguments, so that the contraction is
// straight-line code but for the last tile's steps: a branch per step of four, with the 64-bit divisions that found a
// chunk's place, made the launch four times slower.
//
// Measured: 3000 x 1000 in chunks of 60 x 50 14.4 us (one chunk per scalar-FMA workgroup, both bases staged for each:
// 79 us), 4500 x 3780 in chunks of 60 x 63 46-50 us, 85 Tflop/s.  At three or four waves per SIMD the small one is a
// single round of workgroups: its time is the matrix work of a compute unit's four chunks (7 us) between the first
// rows' arrival and the last stores.
template <int kMT, int kNT>
__global__ __launch_bounds__(256, 3) void k_dense2d(const float* __restrict__ in, int64_t C, int X, int h, int w,
                                                    const float* __restrict__ bh, const float* __restrict__ bw,
                                                    int in_chunked, int out_chunked, int n_chunks,
                                                    float* __restrict__ out) {
    constexpr int kMS = kMT == 3 ? 4 : kMT, kNS = kNT == 3 ? 4 : kNT;  // strips, idle ones included
    constexpr int kStack = kMS < kNS ? 4 / kMS : 4 / kNS;
    constexpr int kRowsPer = 16 * kMT;                        // rows of LDS per chunk
    constexpr int kRows = kStack * kRowsPer;
    constexpr int kLx = kNS == 4 ? 80 : kNS == 2 ? 48 : 16;   // row stride of X
    constexpr int kLt = 16 * kNS + 4;                         // row stride of T
    constexpr int kPerInstr = 4 / kNS;                        // chunk rows per load instruction of a wave
    constexpr int kStep = 4 * kPerInstr;                      // rows per load of the four waves
    static_assert(kRowsPer % kStep == 0, "a load of the four waves stays inside one chunk");
    constexpr int kLoads = kRowsPer / kStep;                  // per chunk
    __shared__ float sx[kRows * kLx];
    __shared__ float st[kRows * kLt];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int l16 = lane & 15, lq = lane >> 4;
    const int hw = h * w;
    const int groups = (n_chunks + kStack - 1) / kStack;

    // a chunk's place: (first element, row stride) in the row-major or the chunked layout
    auto place = [&](int chunk, int chunked) -> int64_t {
        if (chunked) return static_cast<int64_t>(chunk) * hw;
        const int y = static_cast<int>(static_cast<unsigned>(chunk) / static_cast<unsigned>(X));
        return static_cast<int64_t>(y) * h * C + static_cast<int64_t>(chunk - y * X) * w;
    };
    // (T past the chunk's columns is zero times Bh: kept at zero where Bh holds an infinity)
    const bool last_in = 16 * (kNT - 1) + l16 < w;
    // this lane's place in a load: column `col` of row i * kStep + wv * kPerInstr + sub of a chunk
    const int col = lane % (16 * kNS), sub = lane / (16 * kNS);
    float pre[kStack][kLoads];
    auto request = [&](int grp) {
        const int64_t ld = in_chunked ? w : C;
#pragma unroll
        for (int c = 0; c < kStack; ++c) {
            const int chunk = grp * kStack + c;  // wave-uniform
            const int rows = chunk < n_chunks ? h : 0;
            const float* row = in + place(chunk < n_chunks ? chunk : 0, in_chunked) + wv * kPerInstr * ld;
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                const int r = i * kStep + wv * kPerInstr;  // wave-uniform
                float x = 0.f;
                if constexpr (kPerInstr == 1) {
                    // a row past the chunk gets a range of zero bytes, a column past it fails the range check: zero
                    const __amdgpu_buffer_rsrc_t rs =
                        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, r < rows ? w * 4 : 0, 0x00020000);
                    x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, col * 4, 0, 0));
                } else if (r + sub < rows && col < w) {
                    x = row[sub * ld + col];
                }
                pre[c][i] = x;
                row += kStep * ld;
            }
        }
    };

    int grp = blockIdx.x;
    request(grp);
    // the bases' strips: Bh[k][16 mt + l16] for k = 4 s + lq, Bw[k][16 nt + l16] likewise; zero outside
    const int mt = wv % kMS, nt = wv % kNS;
    float a1[4 * kMT], b2[4 * kNT];
#pragma unroll
    for (int s = 0; s < 4 * kMT; ++s) {
        const int k = 4 * s + lq, b = 16 * mt + l16;
        a1[s] = k < h && b < h ? bh[k * h + b] : 0.f;
    }
#pragma unroll
    for (int s = 0; s < 4 * kNT; ++s) {
        const int k = 4 * s + lq, d = 16 * nt + l16;
        b2[s] = k < w && d < w ? bw[k * w + d] : 0.f;
    }
    for (; grp < groups; grp += gridDim.x) {
        // (the sizes as this turn sees them, copies the optimiser cannot see through: it would keep every row's
        // offset and every comparison below in scalar registers across the loop, and spill them)
        asm volatile("" : "+s"(h), "+s"(w), "+s"(C));
#pragma unroll
        for (int c = 0; c < kStack; ++c)
#pragma unroll
            for (int i = 0; i < kLoads; ++i) sx[(c * kRowsPer + i * kStep + wv * kPerInstr + sub) * kLx + col] = pre[c][i];
        __syncthreads();
        if (grp + static_cast<int>(gridDim.x) < groups) request(grp + gridDim.x);
        if (kMT != 3 || mt < 3) {  // wave-uniform
#pragma unroll
            for (int c0 = 0; c0 < kStack; c0 += 4 / kMS) {
                const int c = c0 + wv / kMS;
                v4acc acc[kNT];
#pragma unroll
                for (int n = 0; n < kNT; ++n) acc[n] = v4acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 4 * kMT; ++s) {
                    if (s > 4 * kMT - 4 && 4 * s >= h) break;  // wave-uniform: the last tile's steps past the chunk
#pragma unroll
                    for (int n = 0; n < kNT; ++n)
                        acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            a1[s], sx[(c * kRowsPer + 4 * s + lq) * kLx + 16 * n + l16], acc[n], 0, 0, 0);
                }
#pragma unroll
                for (int n = 0; n < kNT; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        st[(c * kRowsPer + 16 * mt + 4 * lq + r) * kLt + 16 * n + l16] = n + 1 < kNT || last_in ? acc[n][r] : 0.f;
            }
        }
        __syncthreads();
        if (kNT != 3 || nt < 3) {  // wave-uniform
#pragma unroll
            for (int c0 = 0; c0 < kStack; c0 += 4 / kNS) {
                const int c = c0 + wv / kNS, chunk = grp * kStack + c;
                v4acc acc[kMT];
#pragma unroll
                for (int m = 0; m < kMT; ++m) acc[m] = v4acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 4 * kNT; ++s) {
                    if (s > 4 * kNT - 4 && 4 * s >= w) break;
#pragma unroll
                    for (int m = 0; m < kMT; ++m)
                        acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            st[(c * kRowsPer + 16 * m + l16) * kLt + 4 * s + lq], b2[s], acc[m], 0, 0, 0);
                }
                if (chunk < n_chunks) {  // wave-uniform
                    const int64_t ld = out_chunked ? w : C;
                    const int d = 16 * nt + l16;
                    if (d < w) {
                        float* o = out + place(chunk, out_chunked) + 4 * lq * ld + d;
#pragma unroll
                        for (int m = 0; m < kMT; ++m)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (m + 1 < kMT || 16 * m + 4 * lq + r < h) o[(16 * m + r) * ld] = acc[m][r];
                    }
                }
            }
        }
    }
}

// One-row chunks (a 1-D parameter, a dimension that is prime): rows of w elements lying one after the other in either
// layout, out = bh[0] * (row Bw).  A wave takes 16 rows, its operands straight from memory - a parameter of this
// kind is a few thousand elements, and what counts is the number of dependent trips to memory.
template <int kNT>
__global__ __launch_bounds__(64) void k_dense_rows(const float* __restrict__ in, int64_t n_rows, int w,
                                                   const float* __restrict__ bh, const float* __restrict__ bw,
                                                   float* __restrict__ out) {
    const int lane = threadIdx.x, l16 = lane & 15, lq = lane >> 4;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * 16;
    const bool row_in = row0 + l16 < n_rows;
    const float factor = bh[0];
    float a[4 * kNT];
#pragma unroll
    for (int s = 0; s < 4 * kNT; ++s) a[s] = row_in && 4 * s + lq < w ? in[(row0 + l16) * w + 4 * s + lq] * factor : 0.f;
    v4acc acc[kNT];
#pragma unroll
    for (int n = 0; n < kNT; ++n) acc[n] = v4acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4 * kNT; ++s) {
#pragma unroll
        for (int n = 0; n < kNT; ++n) {
            const int k = 4 * s + lq, d = 16 * n + l16;
            acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], k < w && d < w ? bw[k * w + d] : 0.f, acc[n], 0, 0, 0);
        }
    }
#pragma unroll
    for (int n = 0; n < kNT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = row0 + 4 * lq + r;
            const int d = 16 * n + l16;
            if (row < n_rows && d < w) out[row * w + d] = acc[n][r];
        }
}

template <int kMT, int kNT>
static int launch_dense2d(const float* d_in, int64_t C, int h, int w, const float* d_bh, const float* d_bw, int in_chunked,
                          int out_chunked, int64_t n, float* d_out, void* stream) {
    constexpr int kMS = kMT == 3 ? 4 : kMT, kNS = kNT == 3 ? 4 : kNT;
    constexpr int kStack = kMS < kNS ? 4 / kMS : 4 / kNS;
    static const int resident = persistent_grid(k_dense2d<kMT, kNT>, int64_t{1} << 40, 256);
    const int64_t groups = (n + kStack - 1) / kStack;
    hipLaunchKernelGGL((k_dense2d<kMT, kNT>), dim3(static_cast<unsigned>(groups < resident ? groups : resident)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), d_in, C, static_cast<int>(C / w), h, w, d_bh, d_bw, in_chunked,
                       out_chunked, static_cast<int>(n), d_out);
    return launch_status();
}

}  // namespace tplr

using namespace tplr;

extern "C" int tplr_dct2d_dense(const float* d_in, int64_t R, int64_t C, int h, int w, const float* d_bh,
                                const float* d_bw, int in_chunked, int out_chunked, float* d_out, void* stream) {
    if (!d_in || !d_out || !d_bh || !d_bw || R < 0 || C < 0 || h < 1 || w < 1 || h > 64 || w > 64)
        return TPLR_E_BADARG;
    if ((R % h) || (C % w)) return TPLR_E_SHAPE;
    const int64_t n = (R / h) * (C / w);
    if (n == 0) return 0;
    if (n > 0x7fff0000) return TPLR_E_TOOMANY;  // chunks are counted in 32 bits (and a grid has fewer workgroups)
    const int mt = (h + 15) / 16, nt = (w + 15) / 16;  // tiles of 16
    if (h == 1) {  // one-row chunks lie one after the other in both layouts
        const dim3 grid(static_cast<unsigned>((n + 15) / 16)), block(64);
        const hipStream_t st = static_cast<hipStream_t>(stream);
        if (nt == 1)
            hipLaunchKernelGGL(k_dense_rows<1>, grid, block, 0, st, d_in, n, w, d_bh, d_bw, d_out);
        else if (nt == 2)
            hipLaunchKernelGGL(k_dense_rows<2>, grid, block, 0, st, d_in, n, w, d_bh, d_bw, d_out);
        else
            hipLaunchKernelGGL(k_dense_rows<4>, grid, block, 0, st, d_in, n, w, d_bh, d_bw, d_out);
        return launch_status();
    }
#define TPLR_DENSE(MT, NT) \
    case 4 * MT + NT: return launch_dense2d<MT, NT>(d_in, C, h, w, d_bh, d_bw, in_chunked, out_chunked, n, d_out, stream);
    switch (4 * mt + nt) {
        TPLR_DENSE(1, 1) TPLR_DENSE(1, 2) TPLR_DENSE(1, 3) TPLR_DENSE(1, 4)
        TPLR_DENSE(2, 1) TPLR_DENSE(2, 2) TPLR_DENSE(2, 3) TPLR_DENSE(2, 4)
        TPLR_DENSE(3, 1) TPLR_DENSE(3, 2) TPLR_DENSE(3, 3) TPLR_DENSE(3, 4)
        TPLR_DENSE(4, 1) TPLR_DENSE(4, 2) TPLR_DENSE(4, 3) TPLR_DENSE(4, 4)
    }
#undef TPLR_DENSE
    return TPLR_E_BADARG;
}
