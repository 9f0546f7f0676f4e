// Projections of a decode step's few rows: out[m][n] = sum over k of x[m][k] * w[n][k], 16-bit operands, fp32 sums, one rounding.
//
// A step of a small batch reads the whole weight matrix for a handful of rows (the fused projection of the 8B-shaped layer: 50 MB for 4
// rows).  A wave owns two weight rows and requests eight 1 KB slices of each at once - 16 KB a wave, three waves a SIMD at 6 144 rows, and
// most of the matrix is in flight or used -; the rows of x lie in LDS, a 16-byte piece of them serves both weight rows; products are
// two-element dot products, summed across the wave once per row.  (Matrix instructions would idle: a loaded weight takes part in `rows` multiply-adds.)
// What bounds it: at one row the read (4.3 TB/s), at four and more each workgroup's copy of x to LDS before its first product.
// us from a recorded graph, weights from memory, this and the library's product: 4 x 4 096 x 6 144 14.4 / 14.8, x 4 096 10.1 / 14.8, 1 row x 6 144
// 11.6 / 14.5, 2 x 6 144 x 8 192 22.1 / 23.5, 8 x 4 096 x 6 144 21.1 / 14.5.  Up to eight rows all the same: launched one by one, as the eager step
// does, the library's product takes 20 us of host time, this 3 (layer of batch 4, one tile, 16 steps 1 317 -> 815 us; six rows 6.5 us more of the device
// than the library, 34 less of the host).
#include "cq_common.h"

namespace cq {

typedef uint32_t U4 __attribute__((ext_vector_type(4)));

constexpr int kRowSlices = 8;    // 512-channel slices of a weight row in flight
constexpr int kMostRows = 8;
constexpr int kMostX = 64 * 1024;   // bytes of x in LDS

template <typename DT, int M>
__global__ __launch_bounds__(256) void linear_rows_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ out,
                                                          int64_t ldx, int rows, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    U4* xs = reinterpret_cast<U4*>(smem);   // [M][K / 8]
    const int tid = threadIdx.x, lane = tid & 63;
    const int n0 = (static_cast<int>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(tid >> 6)) * 2;   // (N is a multiple of 8)
    const int k8 = K >> 3, slices = K >> 9;
    // x first: it is waited for first
    for (int m = 0; m < rows; ++m) {
        const U4* xg = reinterpret_cast<const U4*>(x + m * ldx);
        for (int i = tid; i < k8; i += 256) xs[m * k8 + i] = xg[i];
    }
    const U4* w0 = reinterpret_cast<const U4*>(w) + static_cast<int64_t>(n0) * k8 + lane;
    U4 a[2][kRowSlices];
    auto request = [&](int c, int i) {   // (slices past the end repeat the last one and are not used)
        const int at = min(c + i, slices - 1) * 64;
        a[0][i] = w0[at];
        a[1][i] = w0[k8 + at];
    };
#pragma unroll
    for (int i = 0; i < kRowSlices; ++i) request(0, i);
    __syncthreads();
    float acc[2 * M];
#pragma unroll
    for (int i = 0; i < 2 * M; ++i) acc[i] = 0.f;
    for (int c = 0; c < slices; c += kRowSlices) {
#pragma unroll
        for (int i = 0; i < kRowSlices; ++i) {
            if (c + i >= slices) break;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const U4 xv = xs[min(m, rows - 1) * k8 + (c + i) * 64 + lane];   // (M is `rows` or the next size: rows past it repeat the last)
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[r * M + m] = dot2<DT>(a[r][i][j], xv[j], acc[r * M + m]);
            }
            if (c + kRowSlices < slices) request(c + kRowSlices, i);
        }
    }
    wave_reduce_n<2 * M>(acc, OpSum(), 0.f);
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * M; ++i) v = lane == i ? acc[i] : v;
    const int r = lane / M, m = lane % M;
    if (lane < 2 * M && m < rows) store_elem<DT>(out, static_cast<int64_t>(m) * N + n0 + r, v);
}

template <typename DT, int M>
static int launch_linear(const void* x, int64_t ldx, const void* w, void* out, int rows, int N, int K, hipStream_t st) {
    hipLaunchKernelGGL((linear_rows_kernel<DT, M>), dim3(N / 8), dim3(256), static_cast<size_t>(rows) * K * 2, st,
                       static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(out), ldx, rows, N, K);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

template <typename DT>
static int launch_linear_rows(const void* x, int64_t ldx, const void* w, void* out, int rows, int N, int K, hipStream_t st) {
    if (rows == 1) return launch_linear<DT, 1>(x, ldx, w, out, rows, N, K, st);
    if (rows == 2) return launch_linear<DT, 2>(x, ldx, w, out, rows, N, K, st);
    if (rows <= 4) return launch_linear<DT, 4>(x, ldx, w, out, rows, N, K, st);
    return launch_linear<DT, 8>(x, ldx, w, out, rows, N, K, st);
}

}  // namespace cq

extern "C" {

int cq_linear_rows_takes(int M, int K, int N) {
    return M >= 1 && M <= cq::kMostRows && K >= 2048 && K % 512 == 0 && static_cast<int64_t>(M) * K * 2 <= cq::kMostX && N >= 8 && N % 8 == 0;
}

int cq_linear_rows(const void* x, int64_t ldx, int dtype, int M, int K, const void* w, int N, void* out, cq_stream_t stream) {
    if (!x || !w || !out) return CQ_ERR_NULL;
    if (dtype != CQ_BF16 && dtype != CQ_FP16) return CQ_ERR_DTYPE;
    if (!cq_linear_rows_takes(M, K, N)) return CQ_ERR_UNSUPPORTED;
    if (!cq::aligned16(x) || !cq::aligned16(w) || ldx % 8) return CQ_ERR_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return dtype == CQ_BF16 ? cq::launch_linear_rows<cq::BF16>(x, ldx, w, out, M, N, K, st) : cq::launch_linear_rows<cq::FP16>(x, ldx, w, out, M, N, K, st);
}

}  // extern "C"
