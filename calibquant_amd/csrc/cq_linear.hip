// Projections of a decode step's few rows: out[m][n] = sum over k of x[m][k] * w[n][k], 16-bit operands, fp32 sums, one rounding.
//
// A step of a small batch reads the whole weight matrix for a handful of rows (the fused projection of the 8B-shaped layer: 50 MB for 4 rows).
// From three rows on (linear_tiles_kernel): a workgroup of eight waves owns one, two or three tiles of eight weight rows, a wave an eighth of the
// channels; it requests its part of the weights and of x straight into matrix operands, eight 1 KB pieces of each tile in flight, and waits for
// nothing before its first product.  A 16 x 16 x 32 product takes 64 channels of eight rows and eight columns: rows and columns 8 .. 15 hold the same
// weight and x rows, 32 channels on, and the two diagonal 8 x 8 blocks are the sums (the other two are not used; the matrix units idle either way).
// So an instruction reads whole 128-byte lines, and up to eight rows of x take the same instructions as one.  The waves' blocks meet in LDS.
// One and two rows (linear_rows_kernel): a wave owns two weight rows and reads 1 KB of one row at a time, eight of each in flight; x lies in LDS, products
// are two-element dot products.  Where the memory-side cache holds the weights that is the faster read (1 x 4 096 x 4 096 4.5, the tiles 6.4), but x's copy
// comes before the first product and every row of x adds its dot products.
// What bounds it: launch and the read (4.3 TB/s at 4 x 4 096 x 6 144).
// Measured, us from a recorded graph, weights from memory (from the cache): dot products / tiles / the library's product:
//   4 x 4 096 x 6 144 12.9 (10.3) / 11.7 (9.9) / 15.2 (10.9); x 4 096 10.2 (7.1) / 8.8 (7.2) / 15.5 (11.4)
//   8 x 4 096 x 6 144 19.2 (17.8) / 12.0 (10.2) / 14.4 (11.0); x 4 096 13.0 (10.8) / 9.2 (7.8) / 15.5 (11.5)
//   4 x 6 144 x 8 192 23.5 (20.9) / 23.8 (21.2) / 23.9 (17.4); x 6 144 19.1 (17.0) / 19.4 (16.3) / 18.3 (14.6)
//   2 x 6 144 x 8 192 21.0 (18.1) / 23.6 (19.8) / 24.1 (17.3); 2 x 4 096 x 6 144 11.7 (8.9) / 11.6 (10.0) / 15.3 (10.9)
//   1 x 4 096 x 6 144 10.9 (8.2) / 10.7 (9.2) / 14.2 (10.7)
// Launched one by one, as the eager step does, the library's product takes 20 us of host time, this 3.  cq_linear_rows_pays() has the sizes a step takes it for.
#include "cq_common.h"

namespace cq {

constexpr int kRowSlices = 8;       // 512-channel slices of a weight row in flight
constexpr int kMostX = 64 * 1024;   // bytes of x in LDS

template <typename DT, int M>
__global__ __launch_bounds__(256) void linear_rows_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ out,
                                                          int64_t ldx, int N, int K) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    U4* xs = reinterpret_cast<U4*>(smem);   // [M][K / 8]
    const int tid = threadIdx.x, lane = tid & 63;
    const int n0 = (static_cast<int>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(tid >> 6)) * 2;   // (N is a multiple of 8)
    const int k8 = K >> 3, slices = K >> 9;
    // x first: it is waited for first
    for (int m = 0; m < M; ++m) {
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
                const U4 xv = xs[m * k8 + (c + i) * 64 + lane];
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
    if (lane < 2 * M) store_elem<DT>(out, static_cast<int64_t>(lane % M) * N + n0 + lane / M, v);
}

template <typename DT, int M>
static int launch_rows(const void* x, int64_t ldx, const void* w, void* out, int N, int K, hipStream_t st) {
    hipLaunchKernelGGL((linear_rows_kernel<DT, M>), dim3(N / 8), dim3(256), static_cast<size_t>(M) * K * 2, st, static_cast<const uint16_t*>(x),
                       static_cast<const uint16_t*>(w), static_cast<uint16_t*>(out), ldx, N, K);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

constexpr int kLinearWaves = 8;
constexpr int kLinearFlight = 8;   // pieces of 64 channels in flight
constexpr int kMostRows = 8;

template <typename DT, int kTiles>
__global__ __launch_bounds__(64 * kLinearWaves) void linear_tiles_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                                        uint16_t* __restrict__ out, int64_t ldx, int rows, int N, int K) {
    __shared__ F4 part[2 * kLinearWaves][8][2 * kTiles];   // [wave, diagonal block][row of x][weight row / 4]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = static_cast<int>(blockIdx.x) * (8 * kTiles);   // (N is a multiple of it)
    const int pieces = K >> 9;   // of this wave: K / 64 / 8, exactly
    const int row = lane & 7, block = (lane >> 3) & 1, quad = lane >> 4;
    const int at = wave * pieces * 64 + block * 32 + quad * 8;   // first channel of this lane
    const uint16_t* wp = w + static_cast<int64_t>(n0 + row) * K + at;
    const uint16_t* xp = x + min(row, rows - 1) * ldx + at;   // (columns past the last row of x repeat it and are not stored)
    U4 a[kTiles][kLinearFlight], b[kLinearFlight];
    auto request = [&](int p, int i) {   // (pieces past the end repeat the last one and are not used)
        const int o = min(p, pieces - 1) * 64;
#pragma unroll
        for (int t = 0; t < kTiles; ++t) a[t][i] = *reinterpret_cast<const U4*>(wp + static_cast<int64_t>(t) * 8 * K + o);
        b[i] = *reinterpret_cast<const U4*>(xp + o);
    };
#pragma unroll
    for (int i = 0; i < kLinearFlight; ++i) request(i, i);
    F4 acc[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) acc[t] = F4{0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < pieces; p += kLinearFlight) {
#pragma unroll
        for (int i = 0; i < kLinearFlight; ++i) {
            if (p + i >= pieces) break;
#pragma unroll
            for (int t = 0; t < kTiles; ++t) acc[t] = mfma16<DT>(a[t][i], b[i], acc[t]);
            if (p + kLinearFlight < pieces) request(p + kLinearFlight + i, i);
        }
    }
    // a lane holds weight rows 4 quad + 0 .. 3 of column lane % 16; the diagonal blocks: quads 0, 1 of columns 0 .. 7 and quads 2, 3 of 8 .. 15
    if ((quad >> 1) == block) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) part[2 * wave + block][row][2 * t + (quad & 1)] = acc[t];
    }
    __syncthreads();
    if (tid < 64 * kTiles) {
        const int m = tid / (8 * kTiles), n = tid % (8 * kTiles);
        float v = 0.f;
#pragma unroll
        for (int s = 0; s < 2 * kLinearWaves; ++s) v += reinterpret_cast<const float*>(&part[s][m][0])[n];
        if (m < rows) store_elem<DT>(out, static_cast<int64_t>(m) * N + n0 + n, v);
    }
}

template <typename DT, int kTiles>
static int launch_tiles(const void* x, int64_t ldx, const void* w, void* out, int rows, int N, int K, hipStream_t st) {
    hipLaunchKernelGGL((linear_tiles_kernel<DT, kTiles>), dim3(N / (8 * kTiles)), dim3(64 * kLinearWaves), 0, st, static_cast<const uint16_t*>(x),
                       static_cast<const uint16_t*>(w), static_cast<uint16_t*>(out), ldx, rows, N, K);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

// Tiles of a workgroup: as many as leave the fullest compute unit with no more rows than fewer tiles would (a launch lasts as long as that one),
// because a workgroup's tiles share its reads of x.  us with one, two, three tiles, weights from memory: 4 x 4 096 x 6 144 12.1, 12.8, 11.4 (768, 384, 256
// workgroups on 256 compute units), 8 rows 13.9, 14.0, 11.6; 8 x 4 096 x 4 096 9.9, 8.6; 4 x 6 144 x 8 192 26.9, 23.8 (four tiles: 23.9); 3 x 2 048 x 1 024 5.0, 6.7.
static int linear_tiles(int N) {
    constexpr int kUnits = 256;
    int best = 1, least = 0;
    for (int t = 1; t <= 3; ++t) {
        if (N % (8 * t) != 0) continue;
        const int fullest = (N / (8 * t) + kUnits - 1) / kUnits * t;
        if (t == 1 || fullest <= least) best = t, least = fullest;
    }
    return best;
}

template <typename DT>
static int launch_linear_rows(const void* x, int64_t ldx, const void* w, void* out, int rows, int N, int K, hipStream_t st) {
    if (rows <= 2 && static_cast<int64_t>(rows) * K * 2 <= kMostX)
        return rows == 1 ? launch_rows<DT, 1>(x, ldx, w, out, N, K, st) : launch_rows<DT, 2>(x, ldx, w, out, N, K, st);
    switch (linear_tiles(N)) {
        case 3: return launch_tiles<DT, 3>(x, ldx, w, out, rows, N, K, st);
        case 2: return launch_tiles<DT, 2>(x, ldx, w, out, rows, N, K, st);
        default: return launch_tiles<DT, 1>(x, ldx, w, out, rows, N, K, st);
    }
}

}  // namespace cq

extern "C" {

int cq_linear_rows_takes(int M, int K, int N) {
    return M >= 1 && M <= cq::kMostRows && K >= 2048 && K % 512 == 0 && N >= 8 && N % 8 == 0;
}

// Where the product is no slower on the device than the library's, weights from memory (a model's weights do not fit the cache, and from some hundred
// megabytes of them on the device bounds the step, not the host).  us, this / the library's:
//   one row 16 384 x 4 096 29.8 / 30.1, two 6 144 x 8 192 20.5 / 23.8, x 6 144 16.8 / 18.1 (7 168 x 7 168 22.2 / 21.4)
//   three to eight: 4 096 channels are eight pieces a wave, all in flight at once; more come in turns of eight, whose last one is padded with repeats
//   (eight rows 5 120 x 5 120 24.0 / 14.4, 6 144 x 8 192 26.1 / 23.9, x 6 144 20.2 / 18.1; the 26B-shaped model's step 1.8 % slower); fewer
//   leave several turns of workgroups too short each (2 048 x 12 288 19.5 / 15.9, 2 560 x 16 384 26.2 / 19.7; x 4 096 7.9 / 10.5, 8.2 / 11.2;
//   4 096 x 16 384 26.4 / 32.6, at the least 4 096 x 14 336 29.3 / 29.0).
int cq_linear_rows_pays(int M, int K, int N) {
    if (!cq_linear_rows_takes(M, K, N)) return 0;
    if (M <= 2) return K <= (M == 1 ? 16384 : 6144);
    return K == 4096 || (K < 4096 && N <= 4096);
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
