// Prefill quantise-and-pack for gfx950, and the unfused quant()/encode()
// operators of the reference surface.
//
// Per-channel statistics need a column reduction over the token axis.  Rows of 128 channels go through the one-pass
// kernel below, which keeps them in registers between the reduction and the codes.  What that does not take (other
// widths, the unpacked codes of quant(), token axes beyond its part counts) is three launches on one stream:
//   1. partial min/max per (batch, head, token chunk, channel)  - reads x once
//   2. statistics: combine the chunks, run the storage-dtype op chain
//      and, per channel, the input thresholds at which the code steps up
//   3. emit: re-read x, compare against the thresholds, pack the codes
// Every arithmetic step that the reference performs as a separate torch op on
// a 16-bit tensor is rounded to that dtype here (rnd<DT>), and divisions are
// IEEE (__fdiv_rn); contraction is off so no multiply-add is fused.
//
// For a positive finite scale the code is a non-decreasing step function of the
// input (division by a positive number, adding a constant, rounding, clamping are
// all monotone), so it is fixed by L thresholds per channel: the smallest storage
// value that yields code k.  The statistics kernel finds them by bisection over
// the ordered 16-bit values, evaluating the exact op chain, and the emit kernel
// only compares - the per-element IEEE division would otherwise bound the pass.
#include "cq_common.h"

#include <algorithm>
#include <atomic>

#include <type_traits>

#pragma clang fp contract(off)

namespace cq {

constexpr int kQThreads = 256;
constexpr int kQUnroll = 4;   // rows in flight per thread in the chunked kernels

struct QuantGeom {
    int B, T, H, D;
    int64_t sb, st, sh;   // element strides of x
    int nchunk, chunk;    // token chunks
    FastDiv dH;           // divisor H
    FastDiv dTB;          // per-token quantiser: workgroup passes per (batch, head)
    int shared_stats;     // non-zero: one row of statistics / thresholds serves every (batch, head) (whole-tensor mode)
    // One-pass kernel: `parts` workgroups share a (batch, head) pair, `part_rows` token rows each, and, if there are
    // several, exchange their channel minima / maxima through `rec` inside the launch: [pair * parts + part][two channels]
    // records of two 64-bit words: the minima as 16-bit keys, below the call's epoch xor the maxima; the maxima, below its
    // complement xor the minima.  A record is valid by itself - 64 bits of it must fit, and a word of it beside one that the
    // workspace held before does not - and nothing has to be cleared.  The wait
    // for the other parts is bounded (spin_limit polls); what is not there by then is read from x again (rows_again()), so the
    // result does not depend on the workgroups being resident together.  spin_limit 0: a part goes on with what it has and
    // sets *status (pinned host memory).
    int parts, part_rows;
    FastDiv dP;           // divisor `parts`
    unsigned long long* rec;
    uint32_t epoch;
    int spin_limit;
    int* status;
};

static inline int pick_chunks(int B, int T, int H) {
    int64_t bh = static_cast<int64_t>(B) * H;
    int64_t want = (4096 + bh - 1) / bh;
    int64_t cap = T / 64 > 1 ? T / 64 : 1;
    int64_t n = want < cap ? want : cap;
    if (n > 256) n = 256;
    if (n < 1) n = 1;
    return static_cast<int>(n);
}

// Extremes that keep a NaN, as torch's reductions and the one-pass kernel below do (one instruction each, as fminf / fmaxf).
__device__ __forceinline__ float ext_min(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float ext_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }
struct OpExtMin { __device__ __forceinline__ float operator()(float a, float b) const { return ext_min(a, b); } };
struct OpExtMax { __device__ __forceinline__ float operator()(float a, float b) const { return ext_max(a, b); } };

// ---- 1. partial min / max -------------------------------------------------
// grid (nchunk, H, B), 256 threads.  A row of D elements is covered by D/8
// adjacent lanes with one 16-byte load each; 256/(D/8) rows per iteration.
template <typename DT>
__global__ __launch_bounds__(kQThreads) void minmax_partial_kernel(const uint16_t* __restrict__ x, QuantGeom g,
                                                                  float* __restrict__ part) {
    const int lpr = g.D >> 3;
    const int rows_per_iter = kQThreads / lpr;
    const int lane = threadIdx.x % lpr;
    const int row = threadIdx.x / lpr;
    const int c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int t0 = c * g.chunk;
    const int t1 = min(g.T, t0 + g.chunk);
    const uint16_t* base = x + b * g.sb + h * g.sh + lane * 8;

    float mn[8], mx[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) { mn[i] = INFINITY; mx[i] = -INFINITY; }
    // four rows in flight per thread; rows past the chunk re-read its last row (harmless for min / max)
    for (int tb = t0 + row; tb < t1; tb += kQUnroll * rows_per_iter) {
        uint4 v[kQUnroll];
#pragma unroll
        for (int u = 0; u < kQUnroll; ++u)
            v[u] = *reinterpret_cast<const uint4*>(base + min(tb + u * rows_per_iter, t1 - 1) * g.st);
#pragma unroll
        for (int u = 0; u < kQUnroll; ++u) {
            float f[8];
            unpack8<DT>(v[u], f);
#pragma unroll
            for (int i = 0; i < 8; ++i) { mn[i] = ext_min(mn[i], f[i]); mx[i] = ext_max(mx[i], f[i]); }
        }
    }
    __shared__ float smn[kQThreads * 8];
    __shared__ float smx[kQThreads * 8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        smn[(row * lpr + lane) * 8 + i] = mn[i];
        smx[(row * lpr + lane) * 8 + i] = mx[i];
    }
    __syncthreads();
    // thread d (< D) folds the rows_per_iter partial rows of channel d
    for (int d = threadIdx.x; d < g.D; d += kQThreads) {
        float a = INFINITY, z = -INFINITY;
        for (int r = 0; r < rows_per_iter; ++r) {
            a = ext_min(a, smn[r * g.D + d]);
            z = ext_max(z, smx[r * g.D + d]);
        }
        float* o = part + ((static_cast<int64_t>(b) * g.H + h) * g.nchunk + c) * 2 * g.D;
        o[d] = a;
        o[g.D + d] = z;
    }
}

// One element of calibquant.py:36: round(clamp(x / scale + zero_point, 0, L)).
// Returns the rounded value; NaN stays NaN (the reference's LUT search then
// finds no match and yields index 0).
template <typename DT>
__device__ __forceinline__ float quant_value(float x, float s, float zp, float levels) {
    float y = rnd<DT>(__fdiv_rn(x, s));
    y = rnd<DT>(y + zp);
    if (y != y) return y;
    y = fminf(fmaxf(y, 0.0f), levels);
    return rintf(y);
}

// Monotone map between the 16-bit storage patterns and integers: order of the keys =
// order of the values (-inf lowest, +inf highest; NaN patterns lie outside [kKeyLo, kKeyHi]).
template <typename DT> struct Keys;
template <> struct Keys<BF16> { static constexpr int lo = -0x7f80, hi = 0x7f80; };
template <> struct Keys<FP16> { static constexpr int lo = -0x7c00, hi = 0x7c00; };
template <typename DT>
__device__ __forceinline__ float key_value(int key) {   // key >= 0: pattern key; key < 0: sign bit + (-key)
    const uint32_t bits = key >= 0 ? static_cast<uint32_t>(key) : (0x8000u | static_cast<uint32_t>(-key));
    return Cvt<DT>::to_float(bits);
}

// ---- 2. statistics ---------------------------------------------------------
// grid (B*H), 1024 threads = 1024/D parts x D channels: thread (p, d) folds every (1024/D)-th chunk
// partial of channel d; after the fold, part 0 writes the statistics and parts 1..3 search one
// threshold each.
// The op chain of calibquant.py:27-34 with one rounding per op; `tensor / python_scalar` is
// a multiply by the fp32 reciprocal, as torch's device kernel does.
constexpr int kStatThreads = 1024;
template <typename DT>
__global__ void stats_kernel(const float* __restrict__ part, QuantGeom g, float clip, float levels,
                             uint16_t* __restrict__ scale, uint16_t* __restrict__ zero, float* __restrict__ thr) {
    const int bh = blockIdx.x;
    const int d = threadIdx.x % g.D;
    const int pt = threadIdx.x / g.D;
    const int nparts = kStatThreads / g.D;   // >= 4 for D <= 256
    __shared__ float sh[2 * kStatThreads];   // [part][2][D]
    float a = INFINITY, z = -INFINITY;
    const float* p = part + static_cast<int64_t>(bh) * g.nchunk * 2 * g.D;
#pragma unroll 4
    for (int c = pt; c < g.nchunk; c += nparts) {   // independent loads: four pairs in flight
        a = ext_min(a, p[c * 2 * g.D + d]);
        z = ext_max(z, p[c * 2 * g.D + g.D + d]);
    }
    sh[(pt * 2) * g.D + d] = a;
    sh[(pt * 2 + 1) * g.D + d] = z;
    __syncthreads();
    for (int q = 0; q < nparts; ++q) {
        a = ext_min(a, sh[(q * 2) * g.D + d]);
        z = ext_max(z, sh[(q * 2 + 1) * g.D + d]);
    }
    const float x_min = rnd<DT>(a * clip);
    const float x_max = rnd<DT>(z * clip);
    const float diff = rnd<DT>(x_max - x_min);
    const float inv_levels = __fdiv_rn(1.0f, levels);
    const float s = rnd<DT>(diff * inv_levels);
    const float zp = rnd<DT>(__fdiv_rn(-x_min, s));
    // thresholds thr[k-1] = smallest storage value whose code is >= k (k = 1..L), kept as
    // [k][channel].  NaN in thr[0]: the step-function argument does not hold for this channel
    // (scale not positive and finite, or zero-point NaN) and emit evaluates the chain itself.
    float* o = thr + static_cast<int64_t>(bh) * 3 * g.D + d;
    const bool monotone = s > 0.0f && s < INFINITY && zp == zp;
    if (pt == 0) {
        scale[static_cast<int64_t>(bh) * g.D + d] = static_cast<uint16_t>(Cvt<DT>::from_float(s));
        zero[static_cast<int64_t>(bh) * g.D + d] = static_cast<uint16_t>(Cvt<DT>::from_float(zp));
        return;
    }
    if (pt > 3) return;
    const int nlev = static_cast<int>(levels);
    const int k = pt;   // this thread's level
    float t = NAN;      // no value reaches code k
    if (monotone && k <= nlev) {
        int lo = Keys<DT>::lo, hi = Keys<DT>::hi;   // invariant: code(lo) < k (or lo is the floor), answer in (lo, hi]
        if (quant_value<DT>(key_value<DT>(hi), s, zp, levels) >= static_cast<float>(k)) {
            if (quant_value<DT>(key_value<DT>(lo), s, zp, levels) >= static_cast<float>(k)) {
                hi = lo;
            } else {
                while (hi - lo > 1) {
                    const int mid = lo + (hi - lo) / 2;
                    if (quant_value<DT>(key_value<DT>(mid), s, zp, levels) >= static_cast<float>(k)) hi = mid;
                    else lo = mid;
                }
            }
            t = key_value<DT>(hi);
        }
    }
    // thr[1] distinguishes "not monotone" (non-NaN) from "code 1 unreachable" (NaN)
    if (!monotone) t = (k == 2) ? 1.0f : NAN;
    o[(k - 1) * g.D] = t;
}

// Whole-tensor statistics (`per_channel=False`, calibquant.py:29-31: x.min() * scale, x.max() * scale):
// one 1024-thread workgroup folds every chunk partial into a single (min, max), runs the same op chain
// and threshold search as above, and writes one row of D identical statistics / thresholds that the
// emit kernel reads for every (batch, head), plus the two scalars the caller gets back.
template <typename DT>
__global__ __launch_bounds__(kStatThreads) void tensor_stats_kernel(const float* __restrict__ part, int64_t npairs, int D,
                                                                    float clip, float levels,
                                                                    uint16_t* __restrict__ scale_row,
                                                                    uint16_t* __restrict__ zero_row,
                                                                    float* __restrict__ thr_row,
                                                                    uint16_t* __restrict__ scale1,
                                                                    uint16_t* __restrict__ zero1) {
    __shared__ float smn[kStatThreads / kWave], smx[kStatThreads / kWave];
    __shared__ float st[2 + 3];   // scale, zero-point, thresholds
    const int tid = threadIdx.x;
    float a = INFINITY, z = -INFINITY;
    const int64_t n = npairs * 2 * D;
    for (int64_t e = tid; e < n; e += kStatThreads) {
        const float v = part[e];
        if ((e / D) & 1) z = ext_max(z, v); else a = ext_min(a, v);   // [pair][min row | max row][D]
    }
    a = wave_reduce(a, OpExtMin(), INFINITY);
    z = wave_reduce(z, OpExtMax(), -INFINITY);
    if ((tid & 63) == 0) { smn[tid >> 6] = a; smx[tid >> 6] = z; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 0; w < kStatThreads / kWave; ++w) { a = ext_min(a, smn[w]); z = ext_max(z, smx[w]); }
        const float x_min = rnd<DT>(a * clip);
        const float x_max = rnd<DT>(z * clip);
        const float diff = rnd<DT>(x_max - x_min);
        const float s = rnd<DT>(diff * __fdiv_rn(1.0f, levels));
        st[0] = s;
        st[1] = rnd<DT>(__fdiv_rn(-x_min, s));
    }
    __syncthreads();
    const float s = st[0], zp = st[1];
    const bool monotone = s > 0.0f && s < INFINITY && zp == zp;
    const int nlev = static_cast<int>(levels);
    if (tid < 3) {
        const int k = tid + 1;
        float t = NAN;
        if (monotone && k <= nlev) {
            int lo = Keys<DT>::lo, hi = Keys<DT>::hi;
            if (quant_value<DT>(key_value<DT>(hi), s, zp, levels) >= static_cast<float>(k)) {
                if (quant_value<DT>(key_value<DT>(lo), s, zp, levels) >= static_cast<float>(k)) {
                    hi = lo;
                } else {
                    while (hi - lo > 1) {
                        const int mid = lo + (hi - lo) / 2;
                        if (quant_value<DT>(key_value<DT>(mid), s, zp, levels) >= static_cast<float>(k)) hi = mid;
                        else lo = mid;
                    }
                }
                t = key_value<DT>(hi);
            }
        }
        if (!monotone) t = (k == 2) ? 1.0f : NAN;   // same marker as stats_kernel: emit evaluates the chain itself
        st[2 + tid] = t;
    }
    __syncthreads();
    for (int d = tid; d < D; d += kStatThreads) {
        scale_row[d] = static_cast<uint16_t>(Cvt<DT>::from_float(s));
        zero_row[d] = static_cast<uint16_t>(Cvt<DT>::from_float(zp));
        thr_row[d] = st[2];
        thr_row[D + d] = st[3];
        thr_row[2 * D + d] = st[4];
    }
    if (tid == 0) {
        scale1[0] = static_cast<uint16_t>(Cvt<DT>::from_float(s));
        zero1[0] = static_cast<uint16_t>(Cvt<DT>::from_float(zp));
    }
}

// ---- 3. emit -----------------------------------------------------------------
// XQ = false: packed codes (B, H, T, D*BITS/8).  XQ = true: the unpacked code
// values as storage-dtype numbers in a contiguous (B, T, H, D) tensor.
template <typename DT, int BITS, bool XQ>
__global__ __launch_bounds__(kQThreads) void emit_kernel(const uint16_t* __restrict__ x, QuantGeom g,
                                                        const uint16_t* __restrict__ scale,
                                                        const uint16_t* __restrict__ zero,
                                                        const float* __restrict__ thr,
                                                        uint8_t* __restrict__ codes, uint16_t* __restrict__ xq) {
    const int lpr = g.D >> 3;
    const int rows_per_iter = kQThreads / lpr;
    const int lane = threadIdx.x % lpr;
    const int row = threadIdx.x / lpr;
    // chunks are walked in the reverse order of the min / max launch: what that launch read last is
    // still in the memory-side cache when this one starts
    const int c = gridDim.x - 1 - blockIdx.x, h = gridDim.y - 1 - blockIdx.y, b = gridDim.z - 1 - blockIdx.z;
    const int t0 = c * g.chunk;
    const int t1 = min(g.T, t0 + g.chunk);
    const uint16_t* base = x + b * g.sb + h * g.sh + lane * 8;
    const int64_t bh = static_cast<int64_t>(b) * g.H + h;
    const int64_t sbh = g.shared_stats ? 0 : bh;   // row of the statistics / threshold arrays
    constexpr float levels = static_cast<float>((1 << BITS) - 1);

    float s[8], zp[8];
    {
        uint4 sv = *reinterpret_cast<const uint4*>(scale + sbh * g.D + lane * 8);
        uint4 zv = *reinterpret_cast<const uint4*>(zero + sbh * g.D + lane * 8);
        unpack8<DT>(sv, s);
        unpack8<DT>(zv, zp);
    }
    // thresholds of this lane's 8 channels (all three levels are loaded, as vectors, whatever BITS is);
    // `slow`: a channel without the step-function property
    float th[3][8];
    bool slow = false;
    {
        const float4* tp = reinterpret_cast<const float4*>(thr + sbh * 3 * g.D + lane * 8);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float4 a = tp[k * (g.D >> 2)], c4 = tp[k * (g.D >> 2) + 1];
            th[k][0] = a.x; th[k][1] = a.y; th[k][2] = a.z; th[k][3] = a.w;
            th[k][4] = c4.x; th[k][5] = c4.y; th[k][6] = c4.z; th[k][7] = c4.w;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) slow = slow | ((th[0][i] != th[0][i]) & (th[1][i] == th[1][i]));
    }
    const int nb = g.D * BITS / 8;  // bytes per packed row
    // dword stores: the lanes of a quad sit in one row (16 or 32 lanes per row) and combine their bytes
    const bool wide = !XQ && (lpr % 4) == 0 && (reinterpret_cast<uintptr_t>(codes) & 3u) == 0;
    const int64_t step = rows_per_iter * g.st;
    const uint16_t* rp = base + (t0 + row) * g.st;
    const uint16_t* last = base + (t1 - 1) * g.st;   // rows past the chunk re-read its last row
    for (int tb = t0 + row; tb < t1; tb += kQUnroll * rows_per_iter, rp += kQUnroll * step) {
        uint4 v[kQUnroll];   // four rows in flight per thread
#pragma unroll
        for (int u = 0; u < kQUnroll; ++u)
            v[u] = *reinterpret_cast<const uint4*>(tb + u * rows_per_iter < t1 ? rp + u * step : last);
#pragma unroll
        for (int u = 0; u < kQUnroll; ++u) {
            const int t = tb + u * rows_per_iter;
            if (t >= t1) break;   // uniform over the lanes of a row
            float f[8];
            unpack8<DT>(v[u], f);
            if constexpr (XQ) {
                float qv[8];
                if (!slow) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        qv[i] = (f[i] >= th[0][i]) ? 1.0f : 0.0f;
                        if constexpr (BITS == 2) {
                            qv[i] += (f[i] >= th[1][i]) ? 1.0f : 0.0f;
                            qv[i] += (f[i] >= th[2][i]) ? 1.0f : 0.0f;
                        }
                        qv[i] = (f[i] != f[i]) ? f[i] : qv[i];   // a NaN input stays NaN in x_q
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) qv[i] = quant_value<DT>(f[i], s[i], zp[i], levels);
                }
                uint32_t w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    w[i] = Cvt<DT>::from_float(qv[2 * i]) | (Cvt<DT>::from_float(qv[2 * i + 1]) << 16);
                uint16_t* o = xq + ((static_cast<int64_t>(b) * g.T + t) * g.H + h) * g.D + lane * 8;
                *reinterpret_cast<uint4*>(o) = make_uint4(w[0], w[1], w[2], w[3]);
            } else {
                uint32_t code[8];
                if (!slow) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {   // a NaN input compares false: code 0
                        code[i] = (f[i] >= th[0][i]) ? 1u : 0u;
                        if constexpr (BITS == 2) {
                            code[i] += (f[i] >= th[1][i]) ? 1u : 0u;
                            code[i] += (f[i] >= th[2][i]) ? 1u : 0u;
                        }
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float qv = quant_value<DT>(f[i], s[i], zp[i], levels);
                        code[i] = (qv != qv) ? 0u : static_cast<uint32_t>(qv);
                    }
                }
                uint8_t* o = codes + (bh * g.T + t) * nb;
                if constexpr (BITS == 1) {
                    uint32_t byte = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) byte |= code[i] << (7 - i);
                    if (wide) {
                        int w = static_cast<int>(byte << (8 * (lane & 3)));
                        w |= dpp_move_i<0xB1>(w, 0);
                        w |= dpp_move_i<0x4E>(w, 0);
                        if ((lane & 3) == 0) *reinterpret_cast<uint32_t*>(o + lane) = static_cast<uint32_t>(w);
                    } else {
                        o[lane] = static_cast<uint8_t>(byte);
                    }
                } else {
                    const uint32_t b0 = (code[0] << 6) | (code[1] << 4) | (code[2] << 2) | code[3];
                    const uint32_t b1 = (code[4] << 6) | (code[5] << 4) | (code[6] << 2) | code[7];
                    const uint32_t half = b0 | (b1 << 8);
                    if (wide) {
                        int w = static_cast<int>(half << (16 * (lane & 1)));
                        w |= dpp_move_i<0xB1>(w, 0);
                        if ((lane & 1) == 0) *reinterpret_cast<uint32_t*>(o + 2 * lane) = static_cast<uint32_t>(w);
                    } else {
                        reinterpret_cast<uint16_t*>(o)[lane] = static_cast<uint16_t>(half);
                    }
                }
            }
        }
    }
}

// ---- one-pass quantise and pack ------------------------------------------------------------
// A 256-thread workgroup owns a run of token rows of one (batch, head) pair: whole rows of 128 channels (256 bytes, LPR = 16
// lanes a row), or, where there is little to do, a quarter of the channels (64 bytes, LPR = 4), 16 bytes x up to 52 rows per
// thread, which stay in registers between the min / max and the emit, so x is read from HBM once.  A longer token axis is
// shared by several workgroups (SPLIT), which exchange their channels' extremes inside the launch.
// thread = (row r = tid / LPR of a pass of 256 / LPR rows, 16-byte piece tid % LPR).
// Two workgroups are resident per compute unit (one wave per SIMD and 256 registers each), the next part's rows are
// requested while this one's are packed.
//
// What bounds it: memory.  Batch 64 x 3 328 tokens x 8 heads, 1 bit, 464 MB, us: the strided key block of a fused projection 106
// -> 92, then 88 with the parts' records read once for two channels (4 registers spilled instead of 13); a contiguous tensor 129 -> 93, 2 bits
// 130 -> 106; the loads alone 75, the code stores 10 - 12 more whatever their form (a streaming kernel without any structure: 64 and 75).  Against a 1 024-thread workgroup per compute unit that
// owned 64-byte quarters of 3 328 rows:
//  - whole rows instead of 64-byte pieces: a contiguous tensor 129 -> 103 (its pieces lay 2 KB apart, on few channels);
//  - non-temporal loads (every line is used once, by one workgroup): 97 -> 89; with 40 or more rows per thread, which is what
//    split_plan() gives large tensors and small ones of few channels.  us ordinary / non-temporal, from memory (and where the
//    memory-side cache holds the tensor): 70 x 831 x 2 heads 9.3 / 9.5 (7.9 / 8.4), 25 x 600 x 8 10.2 / 9.6 (7.0 / 7.5), 21 x 1 700 x 8
//    22.5 / 21.5 (20.7 / 19.5), 64 x 1 664 x 8 57 / 51 (49 / 50), 16 x 9 984 x 8 86 / 78;
//  - codes from packed 16-bit comparisons (EmitPlan), about 15 vector instructions per 8 elements instead of 24;
//  - the threshold search by inverting the op chain (threshold_key) instead of four rounds of 16-ary search.
// More and smaller workgroups (3 x 24 rows, 4 x 16 or 20, 2 x 28) measured 99 to 127: the folds, the exchange and the
// thresholds are paid per part.  Delaying every second workgroup's start so that the two of a unit run out of step: no change.
// Small and long shapes: 1 x 64 tokens x 8 heads 6.0 -> 3.5, 1 x 3 328 12 -> 6.2, 8 x 1 024 7.6 -> 6.5, 64 x 256 37 -> 8.5,
// 1 x 32 768 36 -> 22.5, 16 x 9 984 strided 105 -> 75, contiguous 109 -> 73.
constexpr int kFThreads = 256;
constexpr int kFRows = 52;                  // rows per thread at most
constexpr int kFMaxT = 3328;                // token axis at most with the rotary embedding fused in
constexpr int kFResident = 2;               // workgroups per compute unit of the persistent launch
constexpr int kFGridDefault = 256;          // compute units when no device can be asked: a whole MI355X

// Rotary embedding fused into the pass (ROPE): x is the un-rotated key block; every row is rotated as it
// arrives - rnd(rnd(x * cos) + rotate_half(x) * sin), the arithmetic of the ops the reference runs on the
// whole key tensor before it quantises the image slice (patch_internvl.py:125-134, 258-260, 295-297) - the
// rotated row is written out once (the prefill attention and the caller's cache need it) and quantised from
// the registers.  A channel d pairs with d + 64: the partner's raw values are eight lanes away.
struct RopeArgs {
    const uint16_t* cos;      // (table_rows, 128) in the storage dtype
    const uint16_t* sin;
    const int64_t* pos;       // position id of (b, t) at pos[b * pos_sb + t * pos_st]; NULL: pos0 + t
    int64_t pos_sb, pos_st, pos0, table_rows;
    uint16_t* out;            // rotated rows, (B, T, H, 128) through element strides
    int64_t ob, ot, oh;
    // cq_rope_rows_grouped: every head is a group of `gn` rows, `gs` elements apart in x and `og` in out
    int gn = 1;
    int64_t gs = 0, og = 0;
};

typedef uint32_t U4 __attribute__((ext_vector_type(4)));
typedef short S2 __attribute__((ext_vector_type(2)));
typedef unsigned short US2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_max_s(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(S2, a), __builtin_bit_cast(S2, b))); }
__device__ __forceinline__ uint32_t pk_max_u(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(US2, a), __builtin_bit_cast(US2, b))); }
__device__ __forceinline__ uint32_t pk_min_s(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(S2, a), __builtin_bit_cast(S2, b))); }
__device__ __forceinline__ uint32_t pk_min_u(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(US2, a), __builtin_bit_cast(US2, b))); }
__device__ __forceinline__ uint32_t pk_sub_sat(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(S2, a), __builtin_bit_cast(S2, b))); }
__device__ __forceinline__ uint32_t pk_sign(uint32_t a) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(S2, a) >> 15); }   // 0xffff where negative
__device__ __forceinline__ uint32_t quad_xor(uint32_t v, std::integral_constant<int, 1>) { return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0xB1, 0xf, 0xf, true)); }
__device__ __forceinline__ uint32_t quad_xor(uint32_t v, std::integral_constant<int, 2>) { return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x4E, 0xf, 0xf, true)); }

// The codes of a lane's eight channels of one row, four elements an instruction or two, from the raw 16-bit words.
// Both storage types are sign-magnitude, so "x >= threshold" is an integer comparison of the words: the sign of a
// saturating packed subtraction, which v_perm_b32 spreads over a byte per element (its selectors 8 .. 11) and a
// four-byte dot product with the fields' weights (2^7 .. 2^0 for one bit) turns into the packed byte, modulo 256.
// NaN inputs are kept out by the caller (sanitize()).
// One bit: for a positive threshold the signed words compare as the values do (c = 0: the code is 1 where the
// difference is not negative); for one <= 0 the unsigned words do, in reverse (c = 0x8000: 1 where it is).  Two bits: x is
// made monotone once, y = x < 0 ? x ^ 0x7fff : x, and compared three times.
template <int BITS> struct EmitPlan;
template <> struct EmitPlan<1> {
    uint32_t t[4], c[4], w[2];
    int init;
    __device__ __forceinline__ void load(const uint16_t (*thr)[128], const uint16_t* flip, int c0) {
        const U4 tv = *reinterpret_cast<const U4*>(&thr[0][c0]), cv = *reinterpret_cast<const U4*>(flip + c0);
#pragma unroll
        for (int i = 0; i < 4; ++i) { t[i] = tv[i]; c[i] = cv[i]; }
        const uint32_t n0 = __builtin_amdgcn_perm(c[1], c[0], 0x0b0a0908u), n1 = __builtin_amdgcn_perm(c[3], c[2], 0x0b0a0908u);
        w[0] = (n0 & 0xf0e0c080u) | (~n0 & 0x10204080u);
        w[1] = (n1 & 0xfffefcf8u) | (~n1 & 0x01020408u);
        init = __builtin_amdgcn_sdot4(static_cast<int>(~n1), static_cast<int>(0xfffefcf8u),
                                      __builtin_amdgcn_sdot4(static_cast<int>(~n0), static_cast<int>(0xf0e0c080u), 0, false), false);
    }
    __device__ __forceinline__ uint32_t byte(const U4& x) const {   // bits 0 .. 7 are the packed byte
        uint32_t d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = pk_sub_sat(x[i] ^ c[i], t[i]);
        const uint32_t p0 = __builtin_amdgcn_perm(d[1], d[0], 0x0b0a0908u), p1 = __builtin_amdgcn_perm(d[3], d[2], 0x0b0a0908u);
        return static_cast<uint32_t>(__builtin_amdgcn_sdot4(static_cast<int>(p1), static_cast<int>(w[1]),
                                                            __builtin_amdgcn_sdot4(static_cast<int>(p0), static_cast<int>(w[0]), init, false), false));
    }
};
template <> struct EmitPlan<2> {
    uint32_t t[3][4];
    __device__ __forceinline__ void load(const uint16_t (*thr)[128], const uint16_t*, int c0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const U4 tv = *reinterpret_cast<const U4*>(&thr[k][c0]);
#pragma unroll
            for (int i = 0; i < 4; ++i) t[k][i] = tv[i];
        }
    }
    __device__ __forceinline__ void bytes(const U4& x, uint32_t& b0, uint32_t& b1) const {   // bits 0 .. 7 of either
        uint32_t y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = x[i] ^ (pk_sign(x[i]) & 0x7fff7fffu);
        int a0 = 255, a1 = 255;   // 3 * (64 + 16 + 4 + 1): every level reached, less what is not
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint32_t d[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) d[i] = pk_sub_sat(y[i], t[k][i]);
            a0 = __builtin_amdgcn_sdot4(static_cast<int>(__builtin_amdgcn_perm(d[1], d[0], 0x0b0a0908u)), 0x01041040, a0, false);
            a1 = __builtin_amdgcn_sdot4(static_cast<int>(__builtin_amdgcn_perm(d[3], d[2], 0x0b0a0908u)), 0x01041040, a1, false);
        }
        b0 = static_cast<uint32_t>(a0);
        b1 = static_cast<uint32_t>(a1);
    }
};

// NaN elements of a piece become -infinity, which every threshold leaves below it: code 0, as a comparison of floats gives
template <typename DT> __device__ __forceinline__ void sanitize(U4& x) {
    constexpr uint32_t kInf2 = static_cast<uint32_t>(Keys<DT>::hi) * 0x10001u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // negative halves where the magnitude is beyond infinity's, spread over the half; in place (the assembly keeps
        // the compiler from giving the result of this rarely taken branch registers of its own)
        uint32_t m = pk_sub_sat(kInf2, x[i] & 0x7fff7fffu), w = x[i];
        asm("v_pk_ashrrev_i16 %1, 15, %1 op_sel_hi:[0,1]\n\tv_bfi_b32 %0, %1, %2, %0" : "+v"(w), "+v"(m) : "v"(0x80008000u | kInf2));
        x[i] = w;
    }
}

// The smallest key (Keys<DT>) whose code is at least k, kNoKey if no value reaches it, for a lane pair that shares a
// channel (odd: its second lane).  The op chain is inverted in fp32 - the value of y that rounds up to code k,
// the quotient that rounds to it after the zero-point, the input that divides to that - which lands within a step or
// two; the exact chain at four keys around the guess then decides, and a bisection over all keys does where they do not
// bracket the step (degenerate statistics, values near zero).  The code is a non-decreasing function of x for every (scale,
// zero-point) the chain can produce - also for scale 0 (x / 0 is -inf, NaN, +inf in that order and NaN maps to code 0)
// and for NaN statistics (every code 0).
constexpr int kNoKey = 0x7fff;
template <typename DT> __device__ __forceinline__ int value_key(float f) {   // nearest storage value
    const int p = static_cast<int>(Cvt<DT>::from_float(f) & 0xffffu);
    return (p & 0x8000) ? -(p & 0x7fff) : p;
}
template <typename DT> __device__ __forceinline__ int key_from(float f, bool strict) {   // the smallest one not below f, or above it
    const int k = value_key<DT>(f);
    const float v = key_value<DT>(k);
    return v < f || (strict && v == f) ? k + 1 : k;
}
template <typename DT>
__device__ __forceinline__ int threshold_key(float s, float zp, float levels, int k, bool odd) {
    const int half = value_key<DT>(static_cast<float>(k) - 0.5f);          // y at a tie: it rounds to the even code
    const int ck = (k & 1) ? half + 1 : half;
    const float m = 0.5f * (key_value<DT>(ck - 1) + key_value<DT>(ck));    // what rounds to ck or above
    const int yk = key_from<DT>(m - zp, (k & 1) != 0);                     // (the tie between ck - 1 and ck goes to the even word)
    const float q = 0.5f * (key_value<DT>(yk - 1) + key_value<DT>(yk));
    const int guess = key_from<DT>(q * s, false);
    const int first = min(max(guess - 2, Keys<DT>::lo), Keys<DT>::hi - 3);
    auto reaches = [&](int key) { return quant_value<DT>(key_value<DT>(key), s, zp, levels) >= static_cast<float>(k); };
    const int k0 = first + (odd ? 2 : 0);
    int seen = (reaches(k0) ? 1 : 0) + (reaches(k0 + 1) ? 1 : 0);          // of this lane's two keys
    seen += dpp_move_i<0xB1>(seen, 0);
    int key = first + 4 - seen;
    if (__ballot(seen == 0 || seen == 4)) {
        int lo = Keys<DT>::lo - 1, hi = Keys<DT>::hi;   // code(lo) < k (lo may be the virtual floor), answer in (lo, hi]
        const bool reach = reaches(hi);
        while (hi - lo > 1) {   // (as many rounds in every lane)
            const int mid = (lo + hi) >> 1;
            if (reaches(mid)) hi = mid; else lo = mid;
        }
        if (seen == 0 || seen == 4) key = reach ? hi : kNoKey;
    }
    return key;
}

// Two neighbouring channels of the token rows [t, end) of a pair, read (and rotated) again, folded onto the minima and maxima.
template <typename DT, bool ROPE>
__device__ __forceinline__ void rows_again(const uint16_t* x, const QuantGeom& g, const RopeArgs& ra, int bh, int channel, int t, int end,
                                           uint32_t& a2, uint32_t& z2) {
    const uint32_t b = g.dH.quot(static_cast<uint32_t>(bh)), h = static_cast<uint32_t>(bh) - b * g.dH.div;
    const uint16_t* col = x + static_cast<int64_t>(b) * g.sb + static_cast<int64_t>(h) * g.sh;
    auto word = [](const uint16_t* p) { return *reinterpret_cast<const uint32_t*>(p); };
    auto take = [&](uint32_t v) {
        v ^= pk_sign(v) & 0x7fff7fffu;
        a2 = pk_min_s(a2, v);
        z2 = pk_max_s(z2, v);
    };
    if constexpr (ROPE) {
        const uint32_t sign = channel < 64 ? 0x80008000u : 0u;   // of rotate_half
#pragma unroll 1
        for (; t < end; ++t) {
            const uint16_t* xp = col + static_cast<int64_t>(t) * g.st;
            const int64_t pl = ra.pos ? ra.pos[static_cast<int64_t>(b) * ra.pos_sb + static_cast<int64_t>(t) * ra.pos_st] : ra.pos0 + t;
            const int64_t ps = (pl < 0 ? 0 : pl >= ra.table_rows ? ra.table_rows - 1 : pl) * 128 + channel;
            const uint32_t v = word(xp + channel), y = word(xp + (channel ^ 64)) ^ sign, cw = word(ra.cos + ps), sw = word(ra.sin + ps);
            take(Cvt<DT>::from_float(rnd<DT>(Cvt<DT>::lo(v) * Cvt<DT>::lo(cw)) + Cvt<DT>::lo(y) * Cvt<DT>::lo(sw)) |
                 Cvt<DT>::from_float(rnd<DT>(Cvt<DT>::hi(v) * Cvt<DT>::hi(cw)) + Cvt<DT>::hi(y) * Cvt<DT>::hi(sw)) << 16);
        }
    } else {
        const uint16_t* p = col + static_cast<int64_t>(t) * g.st + channel;
#pragma unroll 1
        for (int rows = end - t; rows > 0; --rows, p += g.st) take(word(p));
    }
}

// The parts of a pair (or quarter) are consecutive ids; a workgroup walks ids blockIdx.x, blockIdx.x + gridDim.x, ... in increasing
// order.  With all workgroups resident, whoever waits for another part waits for a workgroup whose earlier ids belong to
// the same or earlier pairs, so no two wait for each other; where they are not (other streams' kernels, compute-unit masks), a wait
// ends after its bound and the missing rows are read again.
template <typename DT, int BITS, int NR, int LPR = 16, bool ROPE = false, bool SPLIT = false>   // NR: rows per thread
__global__ __launch_bounds__(kFThreads, kFResident) void fused_pack_kernel(const uint16_t* __restrict__ x, QuantGeom g, float clip,
                                                              uint16_t* __restrict__ scale,
                                                              uint16_t* __restrict__ zero,
                                                              uint8_t* __restrict__ codes, RopeArgs ra) {
    static_assert(NR % 4 == 0, "rows are packed and stored four at a time");
    constexpr int L = (1 << BITS) - 1;
    constexpr float levels = static_cast<float>(L);
    static_assert(LPR == 16 || (LPR == 4 && !ROPE), "whole rows or quarters");
    constexpr int kFPass = kFThreads / LPR;            // rows that one load of all threads covers
    constexpr int kChan = 8 * LPR;                     // channels of the workgroup
    constexpr int kLG = kFThreads / (kChan / 2);       // lanes that fold a pair of channels
    constexpr int kLC = kLG / 2;                       // lanes per channel after that
    constexpr bool kStream = LPR == 16 && NR >= 40;
    // the threads' extremes as monotone 16-bit keys, two channels a word (the row pitch spreads what a wave reads together
    // over the banks)
    constexpr int kPitch = LPR == 16 ? 80 : 20;
    __shared__ __attribute__((aligned(16))) uint32_t part_mn[kFPass][kPitch];
    __shared__ __attribute__((aligned(16))) uint32_t part_mx[kFPass][kPitch];
    __shared__ __attribute__((aligned(16))) uint16_t s_thr[L][128];   // thresholds as EmitPlan compares them
    __shared__ __attribute__((aligned(16))) uint16_t s_flip[128];
    const int tid = threadIdx.x, q4 = tid & 3;
    const int piece = tid % LPR, row = tid / LPR;
    const int npairs = g.B * g.H;
    const int nids = npairs * (16 / LPR) * g.parts;   // (below 2^31 with the grid added: split_plan())
    // id = slice * parts + part; slice = quarter * pairs + pair: with eight heads the quarters of a pair, which share its
    // lines of x and of the codes, come to lie on one die (ids a multiple of 8 apart)
    auto slice_of = [&](int id) { return SPLIT ? static_cast<int>(g.dP.quot(static_cast<uint32_t>(id))) : id; };
    auto quarter_of = [&](int slice) { return LPR == 16 ? 0 : (slice >= npairs) + (slice >= 2 * npairs) + (slice >= 3 * npairs); };
    auto first_of = [&](int id) { return SPLIT ? (id - slice_of(id) * g.parts) * g.part_rows : 0; };  // first row of the id's part
    auto rows_of = [&](int id) { return SPLIT ? min(g.T - first_of(id), g.part_rows) : g.T; };        // rows of it
    auto base_of = [&](int id) -> const unsigned char* {
        const int slice = slice_of(id), quarter = quarter_of(slice);
        const uint32_t bh = static_cast<uint32_t>(slice - quarter * npairs);
        const uint32_t b = g.dH.quot(bh), h = bh - b * g.dH.div;
        return reinterpret_cast<const unsigned char*>(x + static_cast<int64_t>(b) * g.sb + static_cast<int64_t>(h) * g.sh +
                                                      static_cast<int64_t>(first_of(id)) * g.st + quarter * 32);
    };
    // A load takes its address as a scalar base (part, pass of rows) + a vector offset that is the same for every
    // full pass; the last pass has an offset of its own, whose rows past the end repeat the last one (min / max unchanged,
    // never written), and the passes behind it repeat the last pass.
    const uint32_t st_bytes = static_cast<uint32_t>(g.st) * 2u;   // (the host checks that it is below 2^24)
    const uint32_t pass_bytes = st_bytes * kFPass;
    const uint32_t off_full = static_cast<uint32_t>(__umul24(static_cast<uint32_t>(row), st_bytes)) + piece * 16;
    auto tail_offset = [&](int len) -> uint32_t {
        return static_cast<uint32_t>(__umul24(static_cast<uint32_t>(min(row, (len - 1) & (kFPass - 1))), st_bytes)) + piece * 16;
    };
    auto load_row = [&](const unsigned char* base, uint32_t pass_bytes, int i, int last_pass, uint32_t off_full, uint32_t off_last) -> U4 {
        const unsigned char* p = base + static_cast<uint64_t>(static_cast<uint32_t>(min(i, last_pass))) * pass_bytes;
        const U4* q = reinterpret_cast<const U4*>(p + (i < last_pass ? off_full : off_last));
        if constexpr (kStream) return __builtin_nontemporal_load(q);
        else return *q;
    };
    int id = blockIdx.x;
    if (id >= nids) return;   // (the whole workgroup)
    U4 v[NR];
    {
        const unsigned char* base = base_of(id);
        const int len0 = rows_of(id);
        const uint32_t off_last = tail_offset(len0);
#pragma unroll
        for (int i = 0; i < NR; ++i) v[i] = load_row(base, pass_bytes, i, (len0 - 1) / kFPass, off_full, off_last);
    }
    // While a part's rows are emitted, every row's registers are refilled with the same row of the workgroup's next
    // part: its loads are in flight during the emit and its min / max pass starts without a wait.
    for (;;) {
    const int slice = slice_of(id), quarter = quarter_of(slice);
    const int bh = slice - quarter * npairs;
    const int next_id = id + static_cast<int>(gridDim.x);
    const bool has_next = next_id < nids;
    const int t_first = first_of(id), t_len = rows_of(id);
    if constexpr (ROPE) {
        const uint32_t bb = g.dH.quot(static_cast<uint32_t>(bh)), hh = static_cast<uint32_t>(bh) - bb * g.dH.div;
        int row_i = row;   // opaque: the rows' addresses are worked out anew for each part, not kept across the loop
        asm volatile("" : "+v"(row_i));
        const int rope_last = (t_len - 1) / kFPass, row_l = min(row_i, (t_len - 1) & (kFPass - 1));
        auto row_of = [&](int i) { return t_first + min(i, rope_last) * kFPass + (i < rope_last ? row_i : row_l); };   // the row that v[i] holds
        uint16_t* orow = ra.out + static_cast<int64_t>(bb) * ra.ob + static_cast<int64_t>(hh) * ra.oh + piece * 8;
        const int64_t* pos_p = ra.pos ? ra.pos + static_cast<int64_t>(bb) * ra.pos_sb : reinterpret_cast<const int64_t*>(ra.cos);
        const int64_t pos_st = ra.pos ? ra.pos_st : 0;
        const int64_t trow_max = ra.table_rows - 1;
        const uint32_t ysign = piece >= 8 ? 0u : 0x80008000u;   // rotate_half(x) = (-x2, x1): the lower half takes minus its partner
        // the table rows of GR rows at a time are requested before the first of them is used: every request
        // is a round trip to the L2, and one row after the other would make a part wait for NR of them in turn
        constexpr int GR = 2;
#pragma unroll
        for (int i0 = 0; i0 < NR; i0 += GR) {
            U4 cw[GR], sw[GR];
#pragma unroll
            for (int k = 0; k < GR; ++k) {
                const int t = row_of(i0 + k);
                // no control flow around the loads (the compiler then requests a group's rows side by side):
                // without a position tensor the load reads a valid dummy and the select takes pos0 + t
                const int64_t pv = pos_p[static_cast<int64_t>(t) * pos_st];
                const int64_t pl = ra.pos ? pv : ra.pos0 + t;
                // clamped to the table in 32 bits (the host checks table_rows < 2^24)
                const uint32_t ps = static_cast<uint32_t>(pl < 0 ? 0 : (pl > trow_max ? trow_max : pl));
                cw[k] = *reinterpret_cast<const U4*>(ra.cos + __umul24(ps, 128u) + piece * 8);
                sw[k] = *reinterpret_cast<const U4*>(ra.sin + __umul24(ps, 128u) + piece * 8);
            }
#pragma unroll
            for (int k = 0; k < GR; ++k) {
                const int i = i0 + k;
                const int t = row_of(i);
                U4 pw;   // the partner's raw piece: the lane eight away holds channel d +- 64 of the same row
#pragma unroll
                for (int w = 0; w < 4; ++w) pw[w] = static_cast<uint32_t>(dpp_move_i<0x128>(static_cast<int>(v[i][w]), 0)) ^ ysign;   // row_ror:8
                U4 r4;
#pragma unroll
                for (int w = 0; w < 4; ++w) {   // a word (two elements) at a time: few values live at once
                    const float x0 = Cvt<DT>::lo(v[i][w]), x1 = Cvt<DT>::hi(v[i][w]);
                    const float y0 = Cvt<DT>::lo(pw[w]), y1 = Cvt<DT>::hi(pw[w]);
                    const float c0 = Cvt<DT>::lo(cw[k][w]), c1 = Cvt<DT>::hi(cw[k][w]);
                    const float s0 = Cvt<DT>::lo(sw[k][w]), s1 = Cvt<DT>::hi(sw[k][w]);
                    const uint32_t o0 = Cvt<DT>::from_float(rnd<DT>(x0 * c0) + y0 * s0);   // y carries the sign of rotate_half
                    const uint32_t o1 = Cvt<DT>::from_float(rnd<DT>(x1 * c1) + y1 * s1);
                    r4[w] = o0 | (o1 << 16);
                }
                v[i] = r4;
                // unconditional store: a row past the end repeats an earlier one, so what is written twice is written with the same bits
                *reinterpret_cast<U4*>(orow + static_cast<int64_t>(t) * ra.ot) = r4;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // Both storage types are sign-magnitude, so the extremes of a column follow from packed 16-bit integer folds of the
    // raw words, two elements per instruction and no unpacking: as signed integers the non-negative values are in
    // value order (the signed maximum is the largest of them, if there is one); as unsigned integers the negative
    // values lie above every non-negative one, in order of magnitude (the unsigned maximum is the most negative value,
    // if there is one).  A column of one sign among the thread's rows needs a third fold (the unsigned minimum: the
    // smallest non-negative value, or with negatives only the one nearest to zero), which a wave
    // without such a column leaves out.  -0 counts as negative and orders below +0.
    uint32_t k_smax[4], k_umin[4], k_umax[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) { k_smax[w] = v[0][w]; k_umax[w] = v[0][w]; }
#pragma unroll
    for (int i = 1; i < NR; ++i) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            k_smax[w] = pk_max_s(k_smax[w], v[i][w]);
            k_umax[w] = pk_max_u(k_umax[w], v[i][w]);
        }
    }
    uint32_t one_sign = 0, top_s = k_smax[0], top_u = k_umax[0];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        one_sign |= k_smax[w] | ~k_umax[w];
        top_s = pk_max_s(top_s, k_smax[w]);
        top_u = pk_max_u(top_u, k_umax[w]);
        k_umin[w] = 0xffffffffu;
    }
    if (__ballot((one_sign & 0x80008000u) != 0)) {
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int w = 0; w < 4; ++w) k_umin[w] = pk_min_u(k_umin[w], v[i][w]);
    }
    // a NaN of either sign is beyond the infinity of that sign
    constexpr int kInf = Keys<DT>::hi;
    const bool nan_here = static_cast<short>(top_s) > kInf || static_cast<short>(top_s >> 16) > kInf ||
                          (top_u & 0xffffu) > (0x8000u | kInf) || (top_u >> 16) > (0x8000u | kInf);
    if (__ballot(nan_here)) {   // (its channel's statistics are NaN and the codes 0, as the ops give; other channels are not touched)
#pragma unroll
        for (int i = 0; i < NR; ++i) sanitize<DT>(v[i]);
    }
    // the thread's extremes as monotone keys: y = x < 0 ? x ^ 0x7fff : x
    {
        U4 mn, mx;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t neg = pk_sign(k_umax[w]), pos = ~pk_sign(k_smax[w]);   // there is a negative / a non-negative value
            const uint32_t lo = (neg & k_umax[w]) | (~neg & k_umin[w]), hi = (pos & k_smax[w]) | (~pos & k_umin[w]);
            mn[w] = lo ^ (pk_sign(lo) & 0x7fff7fffu);
            mx[w] = hi ^ (pk_sign(hi) & 0x7fff7fffu);
        }
        *reinterpret_cast<U4*>(&part_mn[row][piece * 4]) = mn;
        *reinterpret_cast<U4*>(&part_mx[row][piece * 4]) = mx;
    }
    __syncthreads();
    // kLG lanes fold the partials of two channels, four each; then kLC lanes have a channel, run the statistics chain (all: the
    // same instructions) and search the thresholds.
    {
        const int pair2 = tid / kLG, lg = tid % kLG;   // channels 2 * pair2, 2 * pair2 + 1
        uint32_t a2 = part_mn[lg][pair2], z2 = part_mx[lg][pair2];
#pragma unroll
        for (int j = 1; j < kFPass / kLG; ++j) {
            a2 = pk_min_s(a2, part_mn[lg + kLG * j][pair2]);
            z2 = pk_max_s(z2, part_mx[lg + kLG * j][pair2]);
        }
        auto across = [&](auto ctrl) {
            a2 = pk_min_s(a2, static_cast<uint32_t>(dpp_move_i<decltype(ctrl)::value>(static_cast<int>(a2), 0)));
            z2 = pk_max_s(z2, static_cast<uint32_t>(dpp_move_i<decltype(ctrl)::value>(static_cast<int>(z2), 0)));
        };
        auto fold_lanes = [&] {
            across(std::integral_constant<int, 0xB1>{});       // lane ^ 1
            across(std::integral_constant<int, 0x4E>{});       // lane ^ 2
            if constexpr (kLG == 16) {
                across(std::integral_constant<int, 0x141>{});  // mirrored in eight lanes
                across(std::integral_constant<int, 0x140>{});  // ... in sixteen
            }
        };
        fold_lanes();
        if constexpr (SPLIT) {
            // This part's extremes of the two channels go out as one self-validating record; then the records of all parts
            // are polled (device-scope loads, a bounded number of times; each of the channels' lanes takes every kLG-th
            // part, two at a time) and folded.  The other parts are being worked on right now by other workgroups of this launch,
            // unless something else holds the compute units they need.
            unsigned long long* first = g.rec + static_cast<int64_t>(slice) * g.parts * kChan;   // (two words for two channels)
            if (lg == 0) {
                unsigned long long* mine = first + static_cast<uint32_t>((id - slice * g.parts) * kChan + 2 * pair2);
                __hip_atomic_store(mine, static_cast<unsigned long long>(g.epoch ^ z2) << 32 | a2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(mine + 1, static_cast<unsigned long long>(~g.epoch ^ a2) << 32 | z2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            auto whole = [&](unsigned long long lo, unsigned long long hi) {
                return (static_cast<uint32_t>(lo >> 32) ^ static_cast<uint32_t>(hi)) == g.epoch && (static_cast<uint32_t>(hi >> 32) ^ static_cast<uint32_t>(lo)) == ~g.epoch;
            };
            int polls = 0;
            for (int base = 0; base < g.parts; base += 2 * kLG) {
                const bool two = base + kLG < g.parts;
                unsigned long long lo[2], hi[2];   // past the end the last part again
                bool all = false;
                while (!all && polls < g.spin_limit) {
                    if (polls) __builtin_amdgcn_s_sleep(1);
                    ++polls;
                    all = true;
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        if (k && !two) continue;
                        unsigned long long* theirs = first + static_cast<uint32_t>(min(base + k * kLG + lg, g.parts - 1) * kChan + 2 * pair2);
                        lo[k] = __hip_atomic_load(theirs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        hi[k] = __hip_atomic_load(theirs + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        if (k == 0 || two) all = all && whole(lo[k], hi[k]);
                }
                if (!all) { polls = -1; break; }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    if (k && !two) continue;
                    a2 = pk_min_s(a2, static_cast<uint32_t>(lo[k]));
                    z2 = pk_max_s(z2, static_cast<uint32_t>(hi[k]));
                }
            }
            if (polls < 0) {
                if (g.spin_limit <= 0) {   // this call's result is not valid
                    if (g.status) __hip_atomic_store(g.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                } else {
                    // Not all of them within the bound: what is still not there of the lane's parts it reads itself.
#pragma unroll 1
                    for (int p = lg; p < g.parts; p += kLG) {
                        unsigned long long* theirs = first + static_cast<uint32_t>(p * kChan + 2 * pair2);
                        const unsigned long long lo = __hip_atomic_load(theirs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        const unsigned long long hi = __hip_atomic_load(theirs + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (whole(lo, hi)) {
                            a2 = pk_min_s(a2, static_cast<uint32_t>(lo));
                            z2 = pk_max_s(z2, static_cast<uint32_t>(hi));
                        } else {
                            rows_again<DT, ROPE>(x, g, ra, bh, quarter * 32 + 2 * pair2, p * g.part_rows, min(g.T, (p + 1) * g.part_rows), a2, z2);
                        }
                    }
                }
            }
            fold_lanes();
        }
        const int c = 2 * pair2 + lg / kLC, lc = lg % kLC;
        const bool odd = (lc & 1) != 0, lead = lc == 0;
        const uint32_t ext = lg / kLC ? (z2 & 0xffff0000u) | (a2 >> 16) : (z2 << 16) | (a2 & 0xffffu);   // the channel's maximum, minimum
        auto bits_of = [](uint32_t key) { return (key & 0x8000u) ? key ^ 0x7fffu : key; };   // (16 bits) the monotone map is its own inverse
        const float x_min = rnd<DT>(Cvt<DT>::to_float(bits_of(ext & 0xffffu)) * clip);
        const float x_max = rnd<DT>(Cvt<DT>::to_float(bits_of(ext >> 16)) * clip);
        const float diff = rnd<DT>(x_max - x_min);
        const float sc = rnd<DT>(diff * __fdiv_rn(1.0f, levels));
        const float zp = rnd<DT>(__fdiv_rn(-x_min, sc));
        if (lead && (!SPLIT || t_first == 0)) {   // (one of the parts writes them)
            const int64_t o = static_cast<int64_t>(bh) * 128 + quarter * 32 + c;
            scale[o] = static_cast<uint16_t>(Cvt<DT>::from_float(sc));
            zero[o] = static_cast<uint16_t>(Cvt<DT>::from_float(zp));
        }
#pragma unroll
        for (int k = 1; k <= L; ++k) {
            const int key = threshold_key<DT>(sc, zp, levels, k, odd);
            if (lead) {
                // as EmitPlan compares: two bits, monotone words (-0 is one below +0, and belongs to a threshold of 0);
                // one bit, signed words above 0 and reversed magnitudes up to it
                if constexpr (BITS == 2) s_thr[k - 1][c] = static_cast<uint16_t>(key > 0 ? key : key - 1);
                else {
                    s_thr[0][c] = static_cast<uint16_t>(key > 0 ? key : 1 - key);
                    s_flip[c] = static_cast<uint16_t>(key <= 0 ? 0x8000 : 0);
                }
            }
        }
    }
    __syncthreads();
    EmitPlan<BITS> ep;
    ep.load(s_thr, s_flip, piece * 8);
    const unsigned char* next_base = base_of(has_next ? next_id : id);
    const int next_len = rows_of(has_next ? next_id : id);
    // opaque: what the rows' addresses are made of; they are worked out anew for each part, not kept across the loop
    int next_last = (next_len - 1) / kFPass;
    uint32_t next_full = off_full, next_off = tail_offset(next_len), next_pass = pass_bytes;
    int t_out = q4 * kFPass + row;
    asm volatile("" : "+v"(next_full), "+v"(next_off), "+v"(t_out), "+s"(next_last), "+s"(next_pass));
    constexpr int nb = 128 * BITS / 8;   // bytes per packed row
    // lane q of a quad ends with row 4 j + q's bytes of all four pieces of the quad
    uint8_t* orow = codes + (static_cast<int64_t>(bh) * g.T + t_first) * nb + (quarter + (piece >> 2)) * (nb / 4);
    const uint32_t sel1 = (q4 & 1) ? 0x03070105u : 0x06020400u, sel2 = (q4 & 2) ? 0x03020706u : 0x05040100u;
    auto emit = [&](auto refill) {
#pragma unroll
        for (int i0 = 0; i0 < NR; i0 += 4) {
            uint32_t b[4][BITS];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if constexpr (BITS == 1) b[k][0] = ep.byte(v[i0 + k]);
                else ep.bytes(v[i0 + k], b[k][0], b[k][1]);
                // the row is packed: its registers take the same row of the next part
                if constexpr (decltype(refill)::value) v[i0 + k] = load_row(next_base, next_pass, i0 + k, next_last, next_full, next_off);
            }
            if constexpr (BITS == 1) {
                uint32_t w = __builtin_amdgcn_perm(b[1][0], b[0][0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[3][0], b[2][0], 0x04000c0cu);
                w = __builtin_amdgcn_perm(quad_xor(w, std::integral_constant<int, 1>{}), w, sel1);   // rows 0, 2 / 1, 3 of a lane pair
                w = __builtin_amdgcn_perm(quad_xor(w, std::integral_constant<int, 2>{}), w, sel2);   // row q4 of the quad
                if (t_out < t_len - i0 * kFPass)
                    __builtin_nontemporal_store(w, reinterpret_cast<uint32_t*>(orow + i0 * kFPass * nb + static_cast<uint32_t>(t_out) * nb));
            } else {
                // two bytes a row and lane: rows 0, 1 and 2, 3 in a word each
                uint32_t w01 = __builtin_amdgcn_perm(b[0][1], b[0][0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[1][1], b[1][0], 0x04000c0cu);
                uint32_t w23 = __builtin_amdgcn_perm(b[2][1], b[2][0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[3][1], b[3][0], 0x04000c0cu);
                const uint32_t selh = (q4 & 1) ? 0x03020706u : 0x05040100u;   // of a lane pair: row 0 (2) for the even lane, 1 (3) for the odd
                w01 = __builtin_amdgcn_perm(quad_xor(w01, std::integral_constant<int, 1>{}), w01, selh);
                w23 = __builtin_amdgcn_perm(quad_xor(w23, std::integral_constant<int, 1>{}), w23, selh);
                const bool up = (q4 & 2) != 0;
                const uint32_t keep = up ? w23 : w01, got = quad_xor(up ? w01 : w23, std::integral_constant<int, 2>{});
                if (t_out < t_len - i0 * kFPass) {
                    uint32_t* o = reinterpret_cast<uint32_t*>(orow + i0 * kFPass * nb + static_cast<uint32_t>(t_out) * nb);
                    __builtin_nontemporal_store(up ? got : keep, o);   // (the codes are 4-byte aligned at least)
                    __builtin_nontemporal_store(up ? keep : got, o + 1);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (!has_next) {
        emit(std::false_type{});
        return;
    }
    emit(std::true_type{});
    id = next_id;
    }
}

// rows per thread of the instantiation for `need` passes: whole rows, quarters, with the rotary embedding
static constexpr int fused_rows(int need, int lpr, bool rope) {
    if (rope) return need <= 8 ? 8 : need <= 16 ? 16 : need <= 32 ? 32 : kFRows;
    if (lpr == 4) return need <= 4 ? 4 : need <= 8 ? 8 : need <= 16 ? 16 : need <= 32 ? 32 : kFRows;
    return need <= 4 ? 4 : need <= 8 ? 8 : need <= 16 ? 16 : need <= 24 ? 24 : need <= 32 ? 32 : need <= 40 ? 40 : kFRows;
}
template <typename DT, int BITS, int LPR, bool ROPE, bool SPLIT>
static void launch_fused_rows(int nr, dim3 grid, hipStream_t st, const uint16_t* xp, const QuantGeom& g, float clip,
                              uint16_t* sp, uint16_t* zp, uint8_t* codes, const RopeArgs& ra) {
    auto go = [&](auto n) {
        constexpr int NR = decltype(n)::value;
        if constexpr (fused_rows(NR, LPR, ROPE) == NR)   // (no instantiation that the choice above does not name)
            hipLaunchKernelGGL((fused_pack_kernel<DT, BITS, NR, LPR, ROPE, SPLIT>), grid, dim3(kFThreads), 0, st, xp, g, clip, sp, zp, codes, ra);
    };
    switch (nr) {
        case 4: go(std::integral_constant<int, 4>{}); break;
        case 8: go(std::integral_constant<int, 8>{}); break;
        case 16: go(std::integral_constant<int, 16>{}); break;
        case 24: go(std::integral_constant<int, 24>{}); break;
        case 32: go(std::integral_constant<int, 32>{}); break;
        case 40: go(std::integral_constant<int, 40>{}); break;
        default: go(std::integral_constant<int, kFRows>{}); break;
    }
}

// Compute units of the current device, asked once per process.
static int persistent_units() {
    static std::atomic<int> cached{0};
    int n = cached.load(std::memory_order_relaxed);
    if (n > 0) return n;
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu < 1) {
        (void)hipGetLastError();   // not an error of the caller's
        cu = kFGridDefault;
    }
    cached.store(cu, std::memory_order_relaxed);
    return cu;
}

// ---- how the work is cut ------------------------------------------------------------------------------------
// Lanes per row, parts of the token axis, rows per part, rows per thread, workgroups of the launch.  Among the rows
// per thread that give a part count that fits (at most 128; quarters only where all of them are resident at once) the one
// that is expected to take the least, in hundredths of a microsecond: for each turn of a compute unit 0.08 us per row of
// a thread and 0.4 us of folds and thresholds, a little more with the 52 rows that leave no register over; with several parts 1 us
// for the exchange and what polling the other parts costs.  Fitted to 29 shapes, contiguous and strided, timed with every part
// count that fits: 4 % from the best on average, 42 % for the worst (6 x 2 700 x 8 heads contiguous, from memory).
// Why quarters at all, us of whole rows (best part count) / quarters: 4 x 320 x 8 heads 4.7 / 3.8, 1 x 1 024 4.9 / 4.2,
// 8 x 1 024 7.2 / 6.4, 1 x 32 768 x 2 heads 11.8 / 8.3 (fewer channels to exchange per part).  The quarters of a pair share
// its 128-byte lines, and lie on one die only if the pairs are a multiple of eight; otherwise two dies fetch every line,
// which a row then costs more the more of the chip asks for them (up to 0.2 us): 15 x 2 590 x 4 heads 12.2 / 17.5,
// 30 x 3 300 x 2 heads 14.3 / 19.8, 19 x 1 994 x 2 heads 7.1 / 9.0; 1 x 12 171 x 4 heads, 64 workgroups, 10.3 / 8.2.
// With the rotary embedding a row costs ten times as much, and of two workgroups on a compute unit the second takes little less
// than the first, us, rows per thread 52 / 32 / 16 / 8: 6 x 3 328 x 8 heads 42 / 31 / 33 / 37, 64 x 1 300 x 2 heads 41 / 31 / 33 / 35,
// 40 x 600 x 4 heads 31 / 28 / 19 / 23, 64 x 3 328 x 8 heads 263 / 292 / 298 / 374 (18 shapes: 1 % from the best on average,
// 12 % for the worst).
struct SplitPlan { int lpr, parts, part_rows, nr, grid; };
constexpr int kFMostParts = 128;
static bool split_plan(int64_t pairs, int T, bool rope, SplitPlan* sp) {
    const int cu = persistent_units();
    const int64_t room = static_cast<int64_t>(cu) * kFResident;
    int64_t best = -1;
    for (int lpr = 16; lpr >= (rope ? 16 : 4); lpr -= 12) {
        const int pass = kFThreads / lpr;
        const int64_t slices = pairs * (16 / lpr);
        for (int n = 4; n <= kFRows; n = n < 8 ? 8 : n < 40 ? n + 8 : n + 12) {
            if (fused_rows(n, lpr, rope) != n) continue;
            // the fewest parts that n rows per thread hold (more of them only cost more); none of them empty
            const int least = (T - 1) / (n * pass) + 1, rows = (T - 1) / least + 1, p = (T - 1) / rows + 1;
            if (p > kFMostParts || p > room || slices * p > 0x7fffffff - room || (lpr == 4 && slices * p > room)) continue;   // (a pair's parts are resident together)
            const int64_t turns = (slices * p + cu - 1) / cu;                                  // per compute unit
            const int64_t row = lpr == 4 && pairs % 8 ? 8 + std::min<int64_t>(12, slices * p / 16) : 8;
            const int64_t work = rope ? turns / 2 * (100 * n + 400) + turns % 2 * (65 * n + 300)
                                      : turns * (row * n + (lpr == 16 && n == kFRows ? 65 : 40));
            const int64_t cost = work + (p > 1 ? 100 + (rope ? 10 : 5) * p : 0);
            if (best < 0 || cost < best) {
                best = cost;
                *sp = SplitPlan{lpr, p, rows, n, static_cast<int>(slices * p < room ? slices * p : room)};
            }
        }
    }
    return best >= 0;
}
// records that the parts exchange (a pair's channels are the same number in whole rows and in quarters)
static size_t split_records_bytes(int64_t pairs, int parts) { return static_cast<size_t>(pairs) * parts * 128 * sizeof(unsigned long long); }

template <typename DT> static void launch_rope_rows(const uint16_t* x, const QuantGeom& g, const RopeArgs& ra, hipStream_t st);

__global__ __launch_bounds__(256) void clear_records_kernel(unsigned long long* rec, int64_t n) {
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) rec[i] = 0ull;
}

// A part that waits in vain reads the others' rows itself.  Only with the bound set to 0 (cq_quantize_pack_wait_polls) do
// parts go on alone and set a word of pinned host memory (one per device, allocated at the first such call outside a stream
// capture, never freed): the next call on the device reports CQ_ERR_LAUNCH once, and the process goes on with three
// launches.
constexpr int kQMaxDevices = 64;
static std::atomic<int*> g_qstatus[kQMaxDevices];
static std::atomic<bool> g_split_off{false};
static std::atomic<uint32_t> g_qepoch{0x51ab0000u};
static std::atomic<int> g_qspin{1 << 12};   // polls of about a microsecond each

static int* split_status_word(hipStream_t st) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kQMaxDevices) return nullptr;
    int* p = g_qstatus[dev].load(std::memory_order_acquire);
    if (p) return p;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;   // not while the stream is being recorded
    if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return nullptr;
    }
    void* raw = nullptr;
    if (hipHostMalloc(&raw, 64, hipHostMallocDefault) != hipSuccess || !raw) {
        (void)hipGetLastError();
        return nullptr;
    }
    *static_cast<volatile int*>(raw) = 0;
    int* expected = nullptr;
    if (!g_qstatus[dev].compare_exchange_strong(expected, static_cast<int*>(raw), std::memory_order_acq_rel)) {
        (void)hipHostFree(raw);   // another host thread was first
        return expected;
    }
    return static_cast<int*>(raw);
}

static bool one_pass_shape(const QuantGeom& g, const uint8_t* codes) {
    return g.D == 128 && (reinterpret_cast<uintptr_t>(codes) & 3u) == 0 &&
           static_cast<int64_t>(g.B) * g.H < (static_cast<int64_t>(1) << 25) &&   // 32-bit ids
           g.st > 0 && g.st * 2 < (1 << 24);   // 32-bit row offsets inside a pass
}

// Rotated rows that overwrite rows of x: parts that may read each other's rows of x again do not take that.
static bool rope_overlaps(const uint16_t* x, const QuantGeom& g, const RopeArgs& ra) {
    auto span = [&](const uint16_t* p, int64_t sb, int64_t st, int64_t sh, uintptr_t* lo, uintptr_t* hi) {
        int64_t a = 0, z = 128;
        const int64_t ends[3] = {(g.B - 1) * sb, (g.T - 1) * st, (g.H - 1) * sh};
        for (int64_t e : ends) (e < 0 ? a : z) += e;
        *lo = reinterpret_cast<uintptr_t>(p) + static_cast<uintptr_t>(a * 2);
        *hi = reinterpret_cast<uintptr_t>(p) + static_cast<uintptr_t>(z * 2);
    };
    uintptr_t x0, x1, o0, o1;
    span(x, g.sb, g.st, g.sh, &x0, &x1);
    span(ra.out, ra.ob, ra.ot, ra.oh, &o0, &o1);
    return x0 < o1 && o0 < x1;
}

template <typename DT>
static int run_quant(const void* x, QuantGeom g, int bits, float clip, uint8_t* codes, void* xq, void* scale,
                     void* zero, float* ws, hipStream_t st, const RopeArgs* rope = nullptr) {
    dim3 grid(g.nchunk, g.H, g.B);
    const uint16_t* xp = static_cast<const uint16_t*>(x);
    uint16_t* sp = static_cast<uint16_t*>(scale);
    uint16_t* zp = static_cast<uint16_t*>(zero);
    if (rope && (xq || g.T > kFMaxT || !one_pass_shape(g, codes))) return CQ_ERR_UNSUPPORTED;
    SplitPlan spl;
    // (a negative clip factor swaps minimum and maximum: the code then falls with x, which the thresholds do not cover)
    if (!xq && clip >= 0.0f && one_pass_shape(g, codes) && split_plan(static_cast<int64_t>(g.B) * g.H, g.T, rope != nullptr, &spl) &&
        !(rope && spl.parts > 1 && rope_overlaps(xp, g, *rope))) {
        const int spin = g_qspin.load(std::memory_order_relaxed);
        int* status = nullptr;
        if (spl.parts > 1 && spin == 0) {
            status = g_split_off.load(std::memory_order_relaxed) ? nullptr : split_status_word(st);
            if (status && *static_cast<volatile int*>(status) != 0) {
                *static_cast<volatile int*>(status) = 0;
                g_split_off.store(true, std::memory_order_relaxed);
                return CQ_ERR_LAUNCH;   // an earlier split pass did not complete: its output is not valid
            }
        }
        if (spl.parts == 1 || spin > 0 || status) {
            g.parts = spl.parts;
            g.part_rows = spl.part_rows;
            g.dP.set(static_cast<uint32_t>(spl.parts));
            g.rec = reinterpret_cast<unsigned long long*>(ws);
            if (spl.parts > 1) {
                uint32_t ep = g_qepoch.fetch_add(1, std::memory_order_relaxed) + 1;
                g.epoch = ep ? ep : g_qepoch.fetch_add(1, std::memory_order_relaxed) + 1;
            }
            g.spin_limit = spin;
            g.status = status;
            if (spl.parts > 1) {
                // A recorded launch comes back with the same epoch: its records are emptied first, in the recording too.
                // (0 is never an epoch)
                hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
                if (hipStreamIsCapturing(st, &cs) != hipSuccess) (void)hipGetLastError();
                else if (cs != hipStreamCaptureStatusNone) {
                    const int64_t n = static_cast<int64_t>(g.B) * g.H * spl.parts * 128;
                    const int64_t blocks = (n + 255) / 256;
                    hipLaunchKernelGGL(clear_records_kernel, dim3(static_cast<unsigned>(blocks < 1024 ? blocks : 1024)), dim3(256), 0, st, g.rec, n);
                    CQ_LAUNCH_CHECK();
                }
            }
            const dim3 fgrid(static_cast<unsigned>(spl.grid));
            const RopeArgs ra = rope ? *rope : RopeArgs{};
            auto launch = [&](auto b, auto l, auto r) {
                constexpr int B_ = decltype(b)::value, L_ = decltype(l)::value;
                constexpr bool R_ = decltype(r)::value;
                if (spl.parts > 1) launch_fused_rows<DT, B_, L_, R_, true>(spl.nr, fgrid, st, xp, g, clip, sp, zp, codes, ra);
                else launch_fused_rows<DT, B_, L_, R_, false>(spl.nr, fgrid, st, xp, g, clip, sp, zp, codes, ra);
            };
            auto with_bits = [&](auto b) {
                if (rope) launch(b, std::integral_constant<int, 16>{}, std::true_type{});
                else if (spl.lpr == 16) launch(b, std::integral_constant<int, 16>{}, std::false_type{});
                else launch(b, std::integral_constant<int, 4>{}, std::false_type{});
            };
            if (bits == 1) with_bits(std::integral_constant<int, 1>{});
            else with_bits(std::integral_constant<int, 2>{});
            CQ_LAUNCH_CHECK();
            return CQ_OK;
        }
    }
    if (rope) {
        // no exchange inside a launch: the rotated rows first, then the three launches on them
        launch_rope_rows<DT>(xp, g, *rope, st);
        CQ_LAUNCH_CHECK();
        xp = rope->out;
        g.sb = rope->ob; g.st = rope->ot; g.sh = rope->oh;
    }
    hipLaunchKernelGGL(minmax_partial_kernel<DT>, grid, dim3(kQThreads), 0, st, xp, g, ws);
    CQ_LAUNCH_CHECK();
    const float levels = static_cast<float>((1 << bits) - 1);
    float* thr = ws + static_cast<size_t>(g.B) * g.H * g.nchunk * 2 * g.D;
    hipLaunchKernelGGL(stats_kernel<DT>, dim3(g.B * g.H), dim3(kStatThreads), 0, st, ws, g, clip, levels, sp, zp, thr);
    CQ_LAUNCH_CHECK();
    uint16_t* xqp = static_cast<uint16_t*>(xq);
    if (xq) {
        if (bits == 1)
            hipLaunchKernelGGL((emit_kernel<DT, 1, true>), grid, dim3(kQThreads), 0, st, xp, g, sp, zp, thr, codes, xqp);
        else
            hipLaunchKernelGGL((emit_kernel<DT, 2, true>), grid, dim3(kQThreads), 0, st, xp, g, sp, zp, thr, codes, xqp);
    } else {
        if (bits == 1)
            hipLaunchKernelGGL((emit_kernel<DT, 1, false>), grid, dim3(kQThreads), 0, st, xp, g, sp, zp, thr, codes, xqp);
        else
            hipLaunchKernelGGL((emit_kernel<DT, 2, false>), grid, dim3(kQThreads), 0, st, xp, g, sp, zp, thr, codes, xqp);
    }
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

// quant(per_channel=False): partial min / max, whole-tensor statistics, emit of the unpacked codes.
template <typename DT>
static int run_quant_tensor(const void* x, QuantGeom g, int bits, float clip, void* xq, void* scale1, void* zero1,
                            float* ws, hipStream_t st) {
    dim3 grid(g.nchunk, g.H, g.B);
    const uint16_t* xp = static_cast<const uint16_t*>(x);
    hipLaunchKernelGGL(minmax_partial_kernel<DT>, grid, dim3(kQThreads), 0, st, xp, g, ws);
    CQ_LAUNCH_CHECK();
    const float levels = static_cast<float>((1 << bits) - 1);
    const int64_t npairs = static_cast<int64_t>(g.B) * g.H * g.nchunk;
    float* thr = ws + static_cast<size_t>(npairs) * 2 * g.D;            // 3 * D thresholds
    uint16_t* srow = reinterpret_cast<uint16_t*>(thr + 3 * g.D);         // D scales, then D zero-points
    uint16_t* zrow = srow + g.D;
    hipLaunchKernelGGL(tensor_stats_kernel<DT>, dim3(1), dim3(kStatThreads), 0, st, ws, npairs, g.D, clip, levels, srow,
                       zrow, thr, static_cast<uint16_t*>(scale1), static_cast<uint16_t*>(zero1));
    CQ_LAUNCH_CHECK();
    g.shared_stats = 1;
    uint16_t* xqp = static_cast<uint16_t*>(xq);
    if (bits == 1)
        hipLaunchKernelGGL((emit_kernel<DT, 1, true>), grid, dim3(kQThreads), 0, st, xp, g, srow, zrow, thr, nullptr, xqp);
    else
        hipLaunchKernelGGL((emit_kernel<DT, 2, true>), grid, dim3(kQThreads), 0, st, xp, g, srow, zrow, thr, nullptr, xqp);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

static int quant_entry(const void* x, int dtype, int B, int T, int H, int D, int64_t sb, int64_t st, int64_t sh,
                       int bits, float clip, uint8_t* codes, void* xq, void* scale, void* zero, void* ws,
                       size_t ws_bytes, cq_stream_t stream, const RopeArgs* rope = nullptr) {
    if (!x || !scale || !zero || (!codes && !xq)) return CQ_ERR_NULL;
    if (dtype != CQ_BF16 && dtype != CQ_FP16) return CQ_ERR_DTYPE;
    if (bits != 1 && bits != 2) return CQ_ERR_UNSUPPORTED;
    if (B < 1 || T < 1 || H < 1 || (D != 64 && D != 128 && D != 256)) return CQ_ERR_SHAPE;
    if (H > 65535 || B > 65535) return CQ_ERR_SHAPE;
    if ((sb % 8) || (st % 8) || (sh % 8) || !aligned16(x) || !aligned16(scale) || !aligned16(zero) ||
        (xq && !aligned16(xq)) || (codes && (reinterpret_cast<uintptr_t>(codes) & 1u)))
        return CQ_ERR_ALIGN;
    const size_t need = cq_quantize_pack_workspace(B, T, H, D);
    if (!ws || ws_bytes < need || !aligned16(ws)) return CQ_ERR_WORKSPACE;
    QuantGeom g = {};
    g.B = B; g.T = T; g.H = H; g.D = D;
    g.sb = sb; g.st = st; g.sh = sh;
    g.nchunk = pick_chunks(B, T, H);
    g.chunk = (T + g.nchunk - 1) / g.nchunk;
    g.dH.set(static_cast<uint32_t>(H));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == CQ_BF16)
        return run_quant<BF16>(x, g, bits, clip, codes, xq, scale, zero, static_cast<float*>(ws), s, rope);
    return run_quant<FP16>(x, g, bits, clip, codes, xq, scale, zero, static_cast<float*>(ws), s, rope);
}

// Rotary embedding of the rows of a (B, T, H, 128) view, the same arithmetic as above: one thread per
// (row, head, 8 channels of the lower half and the matching 8 of the upper half).
template <typename DT>
__global__ __launch_bounds__(256) void rope_rows_kernel(const uint16_t* __restrict__ x, QuantGeom g, RopeArgs ra) {
    typedef uint32_t U4 __attribute__((ext_vector_type(4)));
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t total = static_cast<int64_t>(g.B) * g.T * g.H * ra.gn * 8;
    if (gid >= total) return;
    const int p8 = static_cast<int>(gid & 7);
    int64_t r = gid >> 3;
    const int gq = static_cast<int>(r % ra.gn); r /= ra.gn;
    const int h = static_cast<int>(r % g.H); r /= g.H;
    const int t = static_cast<int>(r % g.T);
    const int b = static_cast<int>(r / g.T);
    const uint16_t* xr = x + b * g.sb + static_cast<int64_t>(t) * g.st + static_cast<int64_t>(h) * g.sh + gq * ra.gs + p8 * 8;
    int64_t ps = ra.pos ? ra.pos[b * ra.pos_sb + static_cast<int64_t>(t) * ra.pos_st] : ra.pos0 + t;
    ps = ps < 0 ? 0 : (ps >= ra.table_rows ? ra.table_rows - 1 : ps);
    const U4 lo = *reinterpret_cast<const U4*>(xr), hi = *reinterpret_cast<const U4*>(xr + 64);
    const U4 cl = *reinterpret_cast<const U4*>(ra.cos + ps * 128 + p8 * 8), ch = *reinterpret_cast<const U4*>(ra.cos + ps * 128 + 64 + p8 * 8);
    const U4 sl = *reinterpret_cast<const U4*>(ra.sin + ps * 128 + p8 * 8), sh = *reinterpret_cast<const U4*>(ra.sin + ps * 128 + 64 + p8 * 8);
    float x1[8], x2[8], c1[8], c2[8], s1[8], s2[8];
    unpack8<DT>(lo, x1); unpack8<DT>(hi, x2); unpack8<DT>(cl, c1); unpack8<DT>(ch, c2); unpack8<DT>(sl, s1); unpack8<DT>(sh, s2);
    uint32_t o1[8], o2[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        o1[j] = Cvt<DT>::from_float(rnd<DT>(x1[j] * c1[j]) + (-x2[j]) * s1[j]);
        o2[j] = Cvt<DT>::from_float(rnd<DT>(x2[j] * c2[j]) + x1[j] * s2[j]);
    }
    U4 r1, r2;
#pragma unroll
    for (int w = 0; w < 4; ++w) { r1[w] = o1[2 * w] | (o1[2 * w + 1] << 16); r2[w] = o2[2 * w] | (o2[2 * w + 1] << 16); }
    uint16_t* orow = ra.out + b * ra.ob + static_cast<int64_t>(t) * ra.ot + static_cast<int64_t>(h) * ra.oh + gq * ra.og + p8 * 8;
    *reinterpret_cast<U4*>(orow) = r1;
    *reinterpret_cast<U4*>(orow + 64) = r2;
}

template <typename DT> static void launch_rope_rows(const uint16_t* x, const QuantGeom& g, const RopeArgs& ra, hipStream_t st) {
    const int64_t blocks = (static_cast<int64_t>(g.B) * g.T * g.H * ra.gn * 8 + 255) / 256;   // (the callers keep it below 2^31)
    hipLaunchKernelGGL(rope_rows_kernel<DT>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, x, g, ra);
}

static int check_rope(const void* cos_table, const void* sin_table, int64_t table_rows, const int64_t* pos,
                      void* out, int64_t ob, int64_t ot, int64_t oh, int D) {
    if (!cos_table || !sin_table || !out) return CQ_ERR_NULL;
    if (D != 128) return CQ_ERR_UNSUPPORTED;
    if (table_rows < 1 || table_rows >= (1 << 24)) return CQ_ERR_SHAPE;
    if (!aligned16(cos_table) || !aligned16(sin_table) || !aligned16(out) || (ob % 8) || (ot % 8) || (oh % 8) ||
        (pos && (reinterpret_cast<uintptr_t>(pos) & 7u)))
        return CQ_ERR_ALIGN;
    return CQ_OK;
}

// ---- per-token value quantiser --------------------------------------------------------
// The reference's `triton_quantize_and_pack_along_last_dim` (qjl/new_pack.py:53-82): for every
// token and every group of 32 consecutive channels min and max, scale = (max - min) / L,
// code = round(clamp((x - min) / scale, 0, L)), every op rounded to the storage dtype
// (`tensor / python int` multiplies by the fp32 reciprocal; `div_` by the scale tensor is an
// IEEE division), 32/BITS codes per int32 word with the first code in the lowest bits.
// GROUPED: a lane owns a group, so nothing is worked out twice and consecutive lanes write consecutive words and statistics;
// the rows come in whole (16 lanes a row) and go through LDS, where a lane picks up its group's 64 bytes.  Otherwise, for
// inputs of a few thousand rows, four lanes share a group: less work in a row per lane, no LDS.
// One pass over x, its lines used once (GROUPED: non-temporal).
// Batch 64 x 3 328 tokens x 8 heads, us, four lanes a group with a branch per element for degenerate scales -> this:
// strided view of a fused projection 117 -> 96 at 1 bit, 134 -> 93 at 2 bits, contiguous 114 -> 86 (491 MB: 5.7 TB/s); what
// bounded it was some 86 vector instructions for 8 elements, 45 now.  With the group's 64 bytes as four loads per lane
// instead of through LDS: 126 and 133 (lines asked for four times).
template <typename DT> struct Ties;   // half a step of the storage type above 0.5, below 1.5, above 2.5: where rounding moves on
template <> struct Ties<BF16> { static constexpr float a = 0.5f + 0.001953125f, b = 1.5f - 0.00390625f, c = 2.5f + 0.0078125f; };
template <> struct Ties<FP16> { static constexpr float a = 0.5f + 0.000244140625f, b = 1.5f - 0.00048828125f, c = 2.5f + 0.0009765625f; };

// w = 2 w + (f >= t) over f[7] .. f[0]: each comparison leaves its lane mask in a scalar register pair of its own and the
// add takes it as the carry-in.  The compares come first, so every mask is read at least two instructions after it is
// written, as this chip requires of a vector instruction that reads a scalar register written by another.
__device__ __forceinline__ uint32_t shift_in8(uint32_t w, const float* f, float t) {
    unsigned long long m0, m1, m2, m3, m4, m5, m6, m7;
    asm volatile(
        "v_cmp_le_f32_e64 %[m7], %[t], %[f7]\n\t"
        "v_cmp_le_f32_e64 %[m6], %[t], %[f6]\n\t"
        "v_cmp_le_f32_e64 %[m5], %[t], %[f5]\n\t"
        "v_cmp_le_f32_e64 %[m4], %[t], %[f4]\n\t"
        "v_cmp_le_f32_e64 %[m3], %[t], %[f3]\n\t"
        "v_cmp_le_f32_e64 %[m2], %[t], %[f2]\n\t"
        "v_cmp_le_f32_e64 %[m1], %[t], %[f1]\n\t"
        "v_cmp_le_f32_e64 %[m0], %[t], %[f0]\n\t"
        "v_addc_co_u32_e64 %[w], %[m7], %[w], %[w], %[m7]\n\t"
        "v_addc_co_u32_e64 %[w], %[m6], %[w], %[w], %[m6]\n\t"
        "v_addc_co_u32_e64 %[w], %[m5], %[w], %[w], %[m5]\n\t"
        "v_addc_co_u32_e64 %[w], %[m4], %[w], %[w], %[m4]\n\t"
        "v_addc_co_u32_e64 %[w], %[m3], %[w], %[w], %[m3]\n\t"
        "v_addc_co_u32_e64 %[w], %[m2], %[w], %[w], %[m2]\n\t"
        "v_addc_co_u32_e64 %[w], %[m1], %[w], %[w], %[m1]\n\t"
        "v_addc_co_u32_e64 %[w], %[m0], %[w], %[w], %[m0]"
        : [w] "+v"(w), [m0] "=&s"(m0), [m1] "=&s"(m1), [m2] "=&s"(m2), [m3] "=&s"(m3), [m4] "=&s"(m4), [m5] "=&s"(m5),
          [m6] "=&s"(m6), [m7] "=&s"(m7)
        : [t] "v"(t), [f0] "v"(f[0]), [f1] "v"(f[1]), [f2] "v"(f[2]), [f3] "v"(f[3]), [f4] "v"(f[4]), [f5] "v"(f[5]),
          [f6] "v"(f[6]), [f7] "v"(f[7]));
    return w;
}
// w = 4 w + the number of thresholds t1 <= t2 <= t3 that f reaches, over f[3] .. f[0]: the code's upper bit is "t2 reached",
// its lower one "t1 and not t2, or t3", which the scalar unit works out from the masks
__device__ __forceinline__ uint32_t shift_in4x2(uint32_t w, const float* f, float t1, float t2, float t3) {
    unsigned long long a0, a1, a2, a3, b0, b1, b2, b3, c0, c1, c2, c3;
    asm volatile(
        "v_cmp_le_f32_e64 %[a3], %[t1], %[f3]\n\t"
        "v_cmp_le_f32_e64 %[b3], %[t2], %[f3]\n\t"
        "v_cmp_le_f32_e64 %[c3], %[t3], %[f3]\n\t"
        "v_cmp_le_f32_e64 %[a2], %[t1], %[f2]\n\t"
        "v_cmp_le_f32_e64 %[b2], %[t2], %[f2]\n\t"
        "v_cmp_le_f32_e64 %[c2], %[t3], %[f2]\n\t"
        "s_andn2_b64 %[a3], %[a3], %[b3]\n\t"
        "v_cmp_le_f32_e64 %[a1], %[t1], %[f1]\n\t"
        "s_or_b64 %[a3], %[a3], %[c3]\n\t"
        "v_cmp_le_f32_e64 %[b1], %[t2], %[f1]\n\t"
        "s_andn2_b64 %[a2], %[a2], %[b2]\n\t"
        "v_cmp_le_f32_e64 %[c1], %[t3], %[f1]\n\t"
        "s_or_b64 %[a2], %[a2], %[c2]\n\t"
        "v_cmp_le_f32_e64 %[a0], %[t1], %[f0]\n\t"
        "v_cmp_le_f32_e64 %[b0], %[t2], %[f0]\n\t"
        "v_cmp_le_f32_e64 %[c0], %[t3], %[f0]\n\t"
        "s_andn2_b64 %[a1], %[a1], %[b1]\n\t"
        "v_addc_co_u32_e64 %[w], %[b3], %[w], %[w], %[b3]\n\t"
        "s_or_b64 %[a1], %[a1], %[c1]\n\t"
        "v_addc_co_u32_e64 %[w], %[a3], %[w], %[w], %[a3]\n\t"
        "s_andn2_b64 %[a0], %[a0], %[b0]\n\t"
        "v_addc_co_u32_e64 %[w], %[b2], %[w], %[w], %[b2]\n\t"
        "s_or_b64 %[a0], %[a0], %[c0]\n\t"
        "v_addc_co_u32_e64 %[w], %[a2], %[w], %[w], %[a2]\n\t"
        "v_addc_co_u32_e64 %[w], %[b1], %[w], %[w], %[b1]\n\t"
        "v_addc_co_u32_e64 %[w], %[a1], %[w], %[w], %[a1]\n\t"
        "v_addc_co_u32_e64 %[w], %[b0], %[w], %[w], %[b0]\n\t"
        "v_addc_co_u32_e64 %[w], %[a0], %[w], %[w], %[a0]"
        : [w] "+v"(w), [a0] "=&s"(a0), [a1] "=&s"(a1), [a2] "=&s"(a2), [a3] "=&s"(a3), [b0] "=&s"(b0), [b1] "=&s"(b1),
          [b2] "=&s"(b2), [b3] "=&s"(b3), [c0] "=&s"(c0), [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3)
        : [t1] "v"(t1), [t2] "v"(t2), [t3] "v"(t3), [f0] "v"(f[0]), [f1] "v"(f[1]), [f2] "v"(f[2]), [f3] "v"(f[3])
        : "scc");
    return w;
}

constexpr int token_rows(bool grouped) { return kQThreads / (grouped ? 4 : 16); }   // tokens per workgroup pass
template <typename DT, int BITS, bool GROUPED>
__global__ __launch_bounds__(kQThreads) void token_pack_kernel(const uint16_t* __restrict__ x, QuantGeom g,
                                                               int32_t* __restrict__ words,
                                                               uint16_t* __restrict__ scale,
                                                               uint16_t* __restrict__ mins) {
    constexpr float levels = static_cast<float>((1 << BITS) - 1);
    constexpr int kRows = token_rows(GROUPED);
    constexpr int kPieces = GROUPED ? 4 : 1;   // 16-byte pieces of a group per lane
    constexpr int kElems = 8 * kPieces;
    __shared__ __attribute__((aligned(16))) unsigned char tile[kQThreads / kWave][GROUPED ? 16 * 256 : 16];   // a wave's 16 token rows
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // A lane reads its group's pieces starting with a different one in each of four rows, so that 16 lanes meet all banks
    // once; the packed words are rotated back.
    const int turn = GROUPED ? (lane >> 2) & 3 : 0;
    const float inv_levels = __fdiv_rn(1.0f, levels);
    // A workgroup pass is 64 (16) consecutive tokens of one (batch, head).  Consecutive workgroups take the heads of the
    // same tokens, then the next ones: what is in flight on the device at any moment then covers whole token
    // rows of x.  (Walking the output order (b, h, t) instead, everything in flight reads the same 256-byte column of
    // its token rows - one head - and a contiguous (B, T, H, D) input then keeps a fraction of the memory channels
    // busy.)
    const uint32_t ntb = g.dTB.div;                                   // token blocks per (batch, head)
    const int64_t nblk = static_cast<int64_t>(g.B) * g.H * ntb;      // (the host keeps this below 2^31)
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        const uint32_t b32 = static_cast<uint32_t>(blk);
        const uint32_t bt = g.dH.quot(b32);                           // (b, token block)
        const int h = static_cast<int>(b32 - bt * g.dH.div);
        const uint32_t bq = g.dTB.quot(bt);
        const int b = static_cast<int>(bq);
        const int t0 = static_cast<int>(bt - bq * ntb) * kRows;
        const int r = static_cast<int>(threadIdx.x) / (GROUPED ? 4 : 16);   // the lane's row
        const uint16_t* xb = x + static_cast<int64_t>(b) * g.sb + static_cast<int64_t>(t0) * g.st + static_cast<int64_t>(h) * g.sh;
        U4 v[kPieces];
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int row = GROUPED ? wv * 16 + 4 * i + (lane >> 4) : r;
            const U4* p = reinterpret_cast<const U4*>(xb + min(row, g.T - 1 - t0) * g.st + (lane & 15) * 8);   // rows past the end repeat the last one
            if constexpr (GROUPED) v[i] = __builtin_nontemporal_load(p);
            else v[i] = *p;
        }
        if constexpr (GROUPED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<U4*>(tile[wv] + i * 1024 + lane * 16) = v[i];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const U4*>(tile[wv] + lane * 64 + ((i + turn) & 3) * 16);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        float f[kElems];
#pragma unroll
        for (int i = 0; i < kPieces; ++i) unpack8<DT>(v[i], f + 8 * i);
        float mn = f[0], mx = f[0];
#pragma unroll
        for (int i = 1; i < kElems; ++i) { mn = fminf(mn, f[i]); mx = fmaxf(mx, f[i]); }
        if constexpr (!GROUPED) {
            mn = quad_reduce(mn, OpMin(), INFINITY);
            mx = quad_reduce(mx, OpMax(), -INFINITY);
        }
        const float s = rnd<DT>(rnd<DT>(mx - mn) * inv_levels);
        uint32_t w[GROUPED ? BITS : 1];   // (four lanes a group: the lane's 8 or 16 bits)
        if (__ballot(!(s > 0.0f && s < INFINITY)) == 0) {
            // The code steps up where y = storage(fp32(d / s)), d = storage(x - min), crosses 0.5 (exclusive), 1.5
            // (inclusive), 2.5 (exclusive) under round-half-even, i.e. where fp32(d / s) crosses the midpoint m to the
            // neighbouring storage value.  d and s have 8 (11) significant bits and m at most 10 (12), so s * m is exact
            // in fp32 and d / s is either exactly m or further from it than fp32 rounding can move it: the comparison
            // d > s * m (or >=) decides exactly what the division would, without dividing.
            const float m1 = s * Ties<DT>::a, m2 = s * Ties<DT>::b, m3 = s * Ties<DT>::c;
            float y1, y2, y3;
            if constexpr (std::is_same<DT, BF16>::value) {
                // ... and d = bf16(y), y = fp32(x - min) >= 0, is a monotone function of y, so each of those comparisons is
                // one comparison of y itself: with u the smallest bf16 value that satisfies it (the one above m for ">", m
                // rounded up for ">="), bf16(y) >= u exactly when y lies above the midpoint between u and the bf16 value
                // below it, or on it if u is the even one of the two (round-half-even).  In the bit patterns of positive
                // floats that midpoint is u - 0x8000, also across a power of two.
                auto from = [](float m, bool inclusive) -> float {
                    const uint32_t mb = __float_as_uint(m);
                    const uint32_t ub = inclusive ? ((mb + 0xffffu) & 0xffff0000u) : ((mb & 0xffff0000u) + 0x10000u);
                    const uint32_t mid = ub - 0x8000u;
                    return __uint_as_float((ub & 0x10000u) ? mid + 1u : mid);
                };
                y1 = from(m1, false); y2 = from(m2, true); y3 = from(m3, false);
            } else {   // the next float above m, for ">"
                y1 = __uint_as_float(__float_as_uint(m1) + 1u); y2 = m2; y3 = __uint_as_float(__float_as_uint(m3) + 1u);
            }
#pragma unroll
            for (int i = 0; i < kElems; ++i) {
                f[i] -= mn;
                if constexpr (!std::is_same<DT, BF16>::value) f[i] = rnd<DT>(f[i]);
            }
            constexpr int kWords = GROUPED ? BITS : 1, kPer = kElems / kWords;
#pragma unroll
            for (int k = 0; k < kWords; ++k) {
                w[k] = 0;
                if constexpr (BITS == 1) {
#pragma unroll
                    for (int i = kPer - 8; i >= 0; i -= 8) w[k] = shift_in8(w[k], f + i, y1);
                } else {
#pragma unroll
                    for (int i = kPer - 4; i >= 0; i -= 4) w[k] = shift_in4x2(w[k], f + kPer * k + i, y1, y2, y3);
                }
            }
        } else {   // a group of equal values, or an infinity: as the ops say
            constexpr int kWords = GROUPED ? BITS : 1, kPer = kElems / kWords;
#pragma unroll
            for (int k = 0; k < kWords; ++k) {
                w[k] = 0;
#pragma unroll 1
                for (int i = 0; i < kPer; ++i) {
                    const uint32_t word = v[(k * kPer + i) / 8][(i % 8) / 2];
                    const float e = (i & 1) ? Cvt<DT>::hi(word) : Cvt<DT>::lo(word);
                    const float q = rnd<DT>(__fdiv_rn(rnd<DT>(e - mn), s));
                    if (q == q) w[k] |= static_cast<uint32_t>(rintf(fminf(fmaxf(q, 0.0f), levels))) << (BITS * i);
                }
            }
        }
        const int64_t row0 = (static_cast<int64_t>(b) * g.H + h) * g.T + t0;   // output row order (b, h, t)
        if constexpr (!GROUPED) {
            const int64_t gidx = (row0 + r) * 4 + (lane >> 2 & 3);
            const int q4 = lane & 3;
            if (r < g.T - t0) {
                if constexpr (BITS == 1) {
                    uint32_t o = w[0] << (8 * q4);   // 8 bits per lane, 32 per quad: one word
                    o |= quad_xor(o, std::integral_constant<int, 1>{});
                    o |= quad_xor(o, std::integral_constant<int, 2>{});
                    if (q4 == 0) words[gidx] = static_cast<int32_t>(o);
                } else {
                    // 16 bits per lane: lanes (0,1) and (2,3) of the quad make the group's two words
                    const uint32_t o = w[0] | quad_xor(w[0], std::integral_constant<int, 1>{}) << 16;
                    if ((q4 & 1) == 0) words[gidx * 2 + (q4 >> 1)] = static_cast<int32_t>(o);
                }
                if (q4 == 0) {
                    scale[gidx] = static_cast<uint16_t>(Cvt<DT>::from_float(s));
                    mins[gidx] = static_cast<uint16_t>(Cvt<DT>::from_float(mn));
                }
            }
        } else {
            if constexpr (BITS == 1) {
                w[0] = __builtin_amdgcn_alignbit(w[0], w[0], (32 - 8 * turn) & 31);
            } else {
                const bool swap = (turn & 2) != 0, half = (turn & 1) != 0;
                const uint32_t lo = swap ? w[BITS - 1] : w[0], hi = swap ? w[0] : w[BITS - 1];
                w[0] = half ? __builtin_amdgcn_alignbit(lo, hi, 16) : lo;
                w[BITS - 1] = half ? __builtin_amdgcn_alignbit(hi, lo, 16) : hi;
            }
            if (r < g.T - t0) {
                const int64_t gidx = row0 * 4 + static_cast<int>(threadIdx.x);
                if constexpr (BITS == 1) __builtin_nontemporal_store(static_cast<int32_t>(w[0]), words + gidx);
                else {
                    __builtin_nontemporal_store(static_cast<int32_t>(w[0]), words + gidx * 2);
                    __builtin_nontemporal_store(static_cast<int32_t>(w[BITS - 1]), words + gidx * 2 + 1);
                }
                __builtin_nontemporal_store(static_cast<uint16_t>(Cvt<DT>::from_float(s)), scale + gidx);
                __builtin_nontemporal_store(static_cast<uint16_t>(Cvt<DT>::from_float(mn)), mins + gidx);
            }
        }
    }
}

// ---- encode() ---------------------------------------------------------------------
template <typename IT>
__device__ __forceinline__ uint32_t index_of(const IT* p, int64_t i);
template <> __device__ __forceinline__ uint32_t index_of<int64_t>(const int64_t* p, int64_t i) { return static_cast<uint32_t>(p[i]); }
template <> __device__ __forceinline__ uint32_t index_of<int32_t>(const int32_t* p, int64_t i) { return static_cast<uint32_t>(p[i]); }
template <> __device__ __forceinline__ uint32_t index_of<uint8_t>(const uint8_t* p, int64_t i) { return p[i]; }
struct Bf16Tag { uint16_t v; };
struct Fp16Tag { uint16_t v; };
template <> __device__ __forceinline__ uint32_t index_of<Bf16Tag>(const Bf16Tag* p, int64_t i) {
    float f = bf16_bits_to_float(p[i].v);
    return (f != f) ? 0u : static_cast<uint32_t>(static_cast<int>(f));
}
template <> __device__ __forceinline__ uint32_t index_of<Fp16Tag>(const Fp16Tag* p, int64_t i) {
    float f = fp16_bits_to_float(p[i].v);
    return (f != f) ? 0u : static_cast<uint32_t>(static_cast<int>(f));
}

template <typename IT, int BITS>
__global__ void encode_kernel(const IT* __restrict__ idx, int64_t nbytes, uint8_t* __restrict__ out) {
    constexpr int dpe = 8 / BITS;
    constexpr uint32_t m = (1u << BITS) - 1u;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < nbytes;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        uint32_t byte = 0;
#pragma unroll
        for (int k = 0; k < dpe; ++k) byte |= (index_of<IT>(idx, i * dpe + k) & m) << (BITS * (dpe - 1 - k));
        out[i] = static_cast<uint8_t>(byte);
    }
}

template <typename IT>
static int run_encode(const void* idx, int64_t nbytes, int bits, uint8_t* out, hipStream_t st) {
    int64_t blocks = (nbytes + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (bits == 1)
        hipLaunchKernelGGL((encode_kernel<IT, 1>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           static_cast<const IT*>(idx), nbytes, out);
    else
        hipLaunchKernelGGL((encode_kernel<IT, 2>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           static_cast<const IT*>(idx), nbytes, out);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

}  // namespace cq

extern "C" {

size_t cq_quantize_pack_workspace(int B, int T, int H, int D) {
    if (B < 1 || T < 1 || H < 1 || D < 1) return 0;
    // partial min / max per chunk, then three thresholds per channel (+ one row of statistics in the
    // storage dtype for the whole-tensor mode of cq_quant_tensor)
    size_t need = (static_cast<size_t>(B) * H * (static_cast<size_t>(cq::pick_chunks(B, T, H)) * 2 + 3) + 4) * D * sizeof(float);
    // (the records that the parts of a split slice exchange, when the one-pass kernel takes a long token axis)
    cq::SplitPlan spl;
    for (int rope = 0; rope < 2; ++rope) {
        if (D != 128 || !cq::split_plan(static_cast<int64_t>(B) * H, T, rope != 0, &spl) || spl.parts == 1) continue;
        const size_t rec = cq::split_records_bytes(static_cast<int64_t>(B) * H, spl.parts);
        if (rec > need) need = rec;
    }
    return need;
}

int cq_quantize_pack_plan(int B, int T, int H, int rope, cq_quantize_plan* plan) {
    if (!plan) return CQ_ERR_NULL;
    if (B < 1 || T < 1 || H < 1) return CQ_ERR_SHAPE;
    cq::SplitPlan spl;
    if ((rope && T > cq::kFMaxT) || !cq::split_plan(static_cast<int64_t>(B) * H, T, rope != 0, &spl)) return CQ_ERR_UNSUPPORTED;
    plan->channels = 8 * spl.lpr;
    plan->rows_per_thread = spl.nr;
    plan->parts = spl.parts;
    plan->part_rows = spl.part_rows;
    plan->workgroups = spl.grid;
    return CQ_OK;
}

int cq_quantize_pack_wait_polls(int polls) {
    const int before = cq::g_qspin.load(std::memory_order_relaxed);
    if (polls >= 0) {
        cq::g_qspin.store(polls, std::memory_order_relaxed);
        cq::g_split_off.store(false, std::memory_order_relaxed);
    }
    return before;
}

int cq_quantize_pack(const void* x, int dtype, int B, int T, int H, int D, int64_t stride_b, int64_t stride_t,
                     int64_t stride_h, int bits, float clip, uint8_t* codes, void* scale, void* zero,
                     void* workspace, size_t workspace_bytes, cq_stream_t stream) {
    if (!codes) return CQ_ERR_NULL;
    return cq::quant_entry(x, dtype, B, T, H, D, stride_b, stride_t, stride_h, bits, clip, codes, nullptr, scale,
                           zero, workspace, workspace_bytes, stream);
}

int cq_rope_quantize_pack(const void* x, int dtype, int B, int T, int H, int D, int64_t stride_b, int64_t stride_t,
                          int64_t stride_h, const void* cos_table, const void* sin_table, int64_t table_rows,
                          const int64_t* pos, int64_t pos_stride_b, int64_t pos_stride_t, int64_t pos0,
                          void* x_rot, int64_t rot_stride_b, int64_t rot_stride_t, int64_t rot_stride_h,
                          int bits, float clip, uint8_t* codes, void* scale, void* zero,
                          void* workspace, size_t workspace_bytes, cq_stream_t stream) {
    if (!codes) return CQ_ERR_NULL;
    int rc = cq::check_rope(cos_table, sin_table, table_rows, pos, x_rot, rot_stride_b, rot_stride_t, rot_stride_h, D);
    if (rc != CQ_OK) return rc;
    cq::RopeArgs ra;
    ra.cos = static_cast<const uint16_t*>(cos_table); ra.sin = static_cast<const uint16_t*>(sin_table);
    ra.pos = pos; ra.pos_sb = pos_stride_b; ra.pos_st = pos_stride_t; ra.pos0 = pos0; ra.table_rows = table_rows;
    ra.out = static_cast<uint16_t*>(x_rot); ra.ob = rot_stride_b; ra.ot = rot_stride_t; ra.oh = rot_stride_h;
    return cq::quant_entry(x, dtype, B, T, H, D, stride_b, stride_t, stride_h, bits, clip, codes, nullptr, scale,
                           zero, workspace, workspace_bytes, stream, &ra);
}

int cq_rope_rows(const void* x, int dtype, int B, int T, int H, int D, int64_t stride_b, int64_t stride_t,
                 int64_t stride_h, const void* cos_table, const void* sin_table, int64_t table_rows,
                 const int64_t* pos, int64_t pos_stride_b, int64_t pos_stride_t, int64_t pos0,
                 void* x_rot, int64_t rot_stride_b, int64_t rot_stride_t, int64_t rot_stride_h, cq_stream_t stream) {
    return cq_rope_rows_grouped(x, dtype, B, T, H, 1, D, stride_b, stride_t, stride_h, 0, cos_table, sin_table, table_rows,
                                pos, pos_stride_b, pos_stride_t, pos0, x_rot, rot_stride_b, rot_stride_t, rot_stride_h, 0,
                                stream);
}

int cq_rope_rows_grouped(const void* x, int dtype, int B, int T, int H, int G, int D, int64_t stride_b, int64_t stride_t,
                         int64_t stride_h, int64_t stride_g, const void* cos_table, const void* sin_table,
                         int64_t table_rows, const int64_t* pos, int64_t pos_stride_b, int64_t pos_stride_t, int64_t pos0,
                         void* x_rot, int64_t rot_stride_b, int64_t rot_stride_t, int64_t rot_stride_h,
                         int64_t rot_stride_g, cq_stream_t stream) {
    if (!x) return CQ_ERR_NULL;
    if (dtype != CQ_BF16 && dtype != CQ_FP16) return CQ_ERR_DTYPE;
    if (B < 1 || T < 1 || H < 1 || G < 1) return CQ_ERR_SHAPE;
    int rc = cq::check_rope(cos_table, sin_table, table_rows, pos, x_rot, rot_stride_b, rot_stride_t, rot_stride_h, D);
    if (rc != CQ_OK) return rc;
    if ((stride_b % 8) || (stride_t % 8) || (stride_h % 8) || (stride_g % 8) || (rot_stride_g % 8) || !cq::aligned16(x))
        return CQ_ERR_ALIGN;
    cq::QuantGeom g = {};
    g.B = B; g.T = T; g.H = H; g.D = D; g.sb = stride_b; g.st = stride_t; g.sh = stride_h;
    cq::RopeArgs ra;
    ra.cos = static_cast<const uint16_t*>(cos_table); ra.sin = static_cast<const uint16_t*>(sin_table);
    ra.pos = pos; ra.pos_sb = pos_stride_b; ra.pos_st = pos_stride_t; ra.pos0 = pos0; ra.table_rows = table_rows;
    ra.out = static_cast<uint16_t*>(x_rot); ra.ob = rot_stride_b; ra.ot = rot_stride_t; ra.oh = rot_stride_h;
    ra.gn = G; ra.gs = stride_g; ra.og = rot_stride_g;
    const int64_t total = static_cast<int64_t>(B) * T * H * G * 8;
    const int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7fffffff) return CQ_ERR_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint16_t* xp = static_cast<const uint16_t*>(x);
    if (dtype == CQ_BF16) cq::launch_rope_rows<cq::BF16>(xp, g, ra, st);
    else cq::launch_rope_rows<cq::FP16>(xp, g, ra, st);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

int cq_quantize_pack_token(const void* x, int dtype, int B, int T, int H, int D, int64_t stride_b, int64_t stride_t,
                           int64_t stride_h, int bits, int group_size, int32_t* words, void* scale, void* mins,
                           cq_stream_t stream) {
    if (!x || !words || !scale || !mins) return CQ_ERR_NULL;
    if (dtype != CQ_BF16 && dtype != CQ_FP16) return CQ_ERR_DTYPE;
    if ((bits != 1 && bits != 2) || group_size != 32 || D != 128) return CQ_ERR_UNSUPPORTED;
    if (B < 1 || T < 1 || H < 1) return CQ_ERR_SHAPE;
    if ((stride_b % 8) || (stride_t % 8) || (stride_h % 8) || !cq::aligned16(x) ||
        (reinterpret_cast<uintptr_t>(words) & 3u) || (reinterpret_cast<uintptr_t>(scale) & 1u) ||
        (reinterpret_cast<uintptr_t>(mins) & 1u))
        return CQ_ERR_ALIGN;
    cq::QuantGeom g = {};
    g.B = B; g.T = T; g.H = H; g.D = D;
    g.sb = stride_b; g.st = stride_t; g.sh = stride_h;
    g.nchunk = 1; g.chunk = T;
    g.dH.set(static_cast<uint32_t>(H));
    // A lane per group from 56 K rows on, where it has enough workgroups to fill the chip: us, four lanes a group / one (bf16, 1 bit),
    // 24 x 150 tokens x 8 heads 3.8 / 4.3, 3 x 1 700 4.3 / 4.6, 2 x 3 328 5.0 / 4.9 (2 bits 5.9 / 6.0, fp16 5.0 / 5.3), 4 x 2 000 5.8 / 5.3 (2 bits
    // 6.8 / 6.2, fp16 5.9 / 5.6), 4 x 3 328 8.9 / 7.2, 1 x 32 768 17.8 / 14.6, 64 x 3 328 strided 109 / 92.
    const bool grouped = static_cast<int64_t>(B) * T * H >= 56 * 1024;
    const int64_t ntb = (static_cast<int64_t>(T) + cq::token_rows(grouped) - 1) / cq::token_rows(grouped);
    g.dTB.set(static_cast<uint32_t>(ntb));
    const int64_t nblk = static_cast<int64_t>(B) * H * ntb;
    if (nblk > 0x7fffffff) return CQ_ERR_SHAPE;
    int64_t blocks = nblk;
    if (blocks > (1 << 20)) blocks = 1 << 20;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint16_t* xp = static_cast<const uint16_t*>(x);
    uint16_t* sp = static_cast<uint16_t*>(scale);
    uint16_t* mp = static_cast<uint16_t*>(mins);
    const dim3 grid(static_cast<unsigned>(blocks)), block(cq::kQThreads);
    auto launch = [&](auto dt, auto b, auto gr) {
        hipLaunchKernelGGL((cq::token_pack_kernel<decltype(dt), decltype(b)::value, decltype(gr)::value>), grid, block, 0, st, xp, g, words, sp, mp);
    };
    auto with_bits = [&](auto dt, auto gr) {
        if (bits == 1) launch(dt, std::integral_constant<int, 1>{}, gr);
        else launch(dt, std::integral_constant<int, 2>{}, gr);
    };
    auto with_type = [&](auto gr) {
        if (dtype == CQ_BF16) with_bits(cq::BF16{}, gr);
        else with_bits(cq::FP16{}, gr);
    };
    if (grouped) with_type(std::true_type{});
    else with_type(std::false_type{});
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

int cq_quant(const void* x, int dtype, int B, int T, int H, int D, int64_t stride_b, int64_t stride_t,
             int64_t stride_h, int bits, float clip, void* x_q, void* scale, void* zero, void* workspace,
             size_t workspace_bytes, cq_stream_t stream) {
    if (!x_q) return CQ_ERR_NULL;
    return cq::quant_entry(x, dtype, B, T, H, D, stride_b, stride_t, stride_h, bits, clip, nullptr, x_q, scale,
                           zero, workspace, workspace_bytes, stream);
}

int cq_quant_tensor(const void* x, int dtype, int B, int T, int H, int D, int64_t stride_b, int64_t stride_t,
                    int64_t stride_h, int bits, float clip, void* x_q, void* scale1, void* zero1, void* workspace,
                    size_t workspace_bytes, cq_stream_t stream) {
    if (!x || !x_q || !scale1 || !zero1) return CQ_ERR_NULL;
    if (dtype != CQ_BF16 && dtype != CQ_FP16) return CQ_ERR_DTYPE;
    if (bits != 1 && bits != 2) return CQ_ERR_UNSUPPORTED;
    if (B < 1 || T < 1 || H < 1 || (D != 64 && D != 128 && D != 256)) return CQ_ERR_SHAPE;
    if (H > 65535 || B > 65535) return CQ_ERR_SHAPE;
    if ((stride_b % 8) || (stride_t % 8) || (stride_h % 8) || !cq::aligned16(x) || !cq::aligned16(x_q) ||
        (reinterpret_cast<uintptr_t>(scale1) & 1u) || (reinterpret_cast<uintptr_t>(zero1) & 1u))
        return CQ_ERR_ALIGN;
    const size_t need = cq_quantize_pack_workspace(B, T, H, D);
    if (!workspace || workspace_bytes < need || !cq::aligned16(workspace)) return CQ_ERR_WORKSPACE;
    cq::QuantGeom g = {};
    g.B = B; g.T = T; g.H = H; g.D = D;
    g.sb = stride_b; g.st = stride_t; g.sh = stride_h;
    g.nchunk = cq::pick_chunks(B, T, H);
    g.chunk = (T + g.nchunk - 1) / g.nchunk;
    g.dH.set(static_cast<uint32_t>(H));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == CQ_BF16)
        return cq::run_quant_tensor<cq::BF16>(x, g, bits, clip, x_q, scale1, zero1, static_cast<float*>(workspace), s);
    return cq::run_quant_tensor<cq::FP16>(x, g, bits, clip, x_q, scale1, zero1, static_cast<float*>(workspace), s);
}

int cq_encode(const void* idx, int idx_dtype, int64_t rows, int D, int bits, uint8_t* out, cq_stream_t stream) {
    if (!idx || !out) return CQ_ERR_NULL;
    if (bits != 1 && bits != 2) return CQ_ERR_UNSUPPORTED;
    if (rows < 0 || D < 1 || (D % (8 / bits)) != 0) return CQ_ERR_SHAPE;
    if (rows == 0) return CQ_OK;
    const int64_t nbytes = rows * (D * bits / 8);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (idx_dtype) {
        case CQ_I64: return cq::run_encode<int64_t>(idx, nbytes, bits, out, s);
        case CQ_I32: return cq::run_encode<int32_t>(idx, nbytes, bits, out, s);
        case CQ_U8: return cq::run_encode<uint8_t>(idx, nbytes, bits, out, s);
        case CQ_BF16: return cq::run_encode<cq::Bf16Tag>(idx, nbytes, bits, out, s);
        case CQ_FP16: return cq::run_encode<cq::Fp16Tag>(idx, nbytes, bits, out, s);
        default: return CQ_ERR_DTYPE;
    }
}

}  // extern "C"
