// Fused decode attention over bit-packed K/V for gfx950 (MI355X).
//
// One workgroup (1024 threads, or 512 threads with two workgroups resident per compute
// unit when there are more units than compute units) owns one (batch, kv-head,
// head-group, token-chunk) unit and runs the whole step for HPB query heads that share
// the kv-head:
//
//   loads    the packed K rows are requested at kernel entry, the first block of
//            packed V rows behind them (half before the logits, half as the K
//            registers free up), the window's first K rows ahead of the packed V rows and
//            its V rows behind them: each stream is in flight while the phase before
//            its consumer runs, and no phase starts behind a queue of requests
//            it does not need.  (The window's rows at entry, or ahead of the logits: the packed K rows
//            wait behind them.  us, batch 64 x 3 328 + 128 19.3 -> 20.8, 16 x 9 984 + 105 17.8 -> 19.1.)
//   K side   the codes are small integers: q.s_k goes onto a fixed-point grid, eight 4-bit digits and a sign a value, and a
//            tile's logits are exact products of 6-bit and 4-bit floats (see "the step on the matrix cores" below); the
//            fp16/bf16 K tensor is never materialised.  A thread keeps its logits in registers, the last rounds' in LDS.
//   stats    min / max of the image logits (calibration), then e = exp(w' - M).
//   V side   e (times the token's group scale, for per-token values) as four byte digits against the packed V rows,
//            on 8-bit integer products.  Per-channel scale / zero-point are applied once at the end.
//   residual the full-precision rows run last as an online-softmax flash-decode in
//            the same workgroup, on 16-bit products with the weights in three parts, and are merged at the end.
//
// When the chunk does not cover all T tokens (long context or small batch)
// a first launch computes every chunk's logits and publishes the per-chunk min / max;
// the main launch recomputes its chunk's logits, exponentiates against the global min / max and writes an (m, l, acc)
// partial; the last workgroup of a unit to get there combines the unit's partials.  Where all the chunks' workgroups
// fit the device at once, one launch does both: the chunks exchange their min / max inside it.
#pragma once
#include "cq_common.h"
#include "cq_digits.h"

// The kernels below lean on behaviour of this architecture family that the HIP memory model does not
// promise (see the in-launch merge of the chunked step) and on its LDS size, DPP controls and
// instruction set: refuse to build device code for anything else.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the decode kernels are written for gfx950"
#endif

#include <type_traits>

namespace cq {

constexpr int kD = 128;
// 16-byte pieces of packed K and V rows in flight per thread, and of the V rows how many are requested
// ahead of the logits
constexpr int kMatrixK = 4, kMatrixV = 4, kMatrixE = 2;
constexpr int kLdsMax = 160 * 1024;
constexpr int kDefaultUnits = 256; // compute units of a whole MI355X, assumed when no device can be asked
constexpr int kRegPair = 8;        // rounds of logits a thread of a 512-thread workgroup keeps in registers (4 096 tokens)
constexpr int kRegTwoBit = 4;      // ... of a 1024-thread workgroup with per-token values and a short chunk (4 096 tokens)
constexpr int kRegLong = 10;       // ... of a 1024-thread workgroup that holds a long chunk in one launch (10 240 tokens)
constexpr int kRegMost = 16;       // ... of the longest chunks a plan for fewer than four heads per unit can have (16 384 tokens)
constexpr float kLog2e = 1.4426950408889634f;

// Profiling build (-DCQ_PHASE_STOPS, `python -m calibquant_amd.build --phase-stops`; only the headline
// instantiation is compiled): a launch can be told to end at a phase boundary (environment variable
// CQ_DECODE_PHASE_STOP = k, read per call), so that whole-launch hardware counters of runs with successive
// k give per-phase counts by subtraction.  The shipped library has none of this.
#ifdef CQ_PHASE_STOPS
#define CQ_PHASE(k) do { if (g.stop == (k)) return; } while (0)
#else
#define CQ_PHASE(k) do { } while (0)
#endif


template <int N> struct alignas(N * 4) Vec { float v[N]; };
typedef uint32_t U2 __attribute__((ext_vector_type(2)));
typedef uint32_t Pair16 __attribute__((aligned(2)));   // two 16-bit values wherever they lie: q and the statistics need no alignment

// Of a launch's rounds of logits, how many (the last ones) a thread keeps in LDS of its own instead of registers: all of them in registers
// leave too few for the products' operands and the rows in flight, and a spilled row waits for its load (batch 64 18.4 -> 22.0 us with 16
// registers spilled).  16 bytes a lane, written and read once each: no bank conflicts, no vector instruction.  The same LDS holds a tile of the window's rows later.
constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int parked_rounds(bool vtok, int nt, int rounds) {
    if (vtok || rounds <= 4) return 0;
    if (rounds > 10) return nt == 512 ? 7 : 6;
    return nt == 512 ? 4 : 5;
}

// ... and the bytes of it (static LDS, beside the dynamic): at least a tile of 128 window rows; two for 1 024 threads, which have the
// LDS to themselves and take the tiles in turn: no barrier between the values of one and the rows of the next
constexpr int kWindowTile = 128 * 256;
constexpr int parked_lds(bool vtok, int nt, int rounds) { return cmax(parked_rounds(vtok, nt, rounds) * nt * 16, nt == 1024 ? 2 * kWindowTile : kWindowTile); }

struct DecodeGeom {
    const void* q;
    const uint8_t* ck;
    const uint8_t* cv;
    const void *ks, *kz, *vs, *vz;
    const void *kres, *vres;
    int64_t rs_b, rs_h, rs_r;
    const float* mask;
    int64_t mask_sb;
    void* out;
    const int32_t* r_dev;   // optional: residual row count read at run time (R is then the capacity)
    float* mm;    // [B][Hq][nsplit][2] chunk logit min / max
    float* part;  // [B][Hq][nx][kD + 2] partials (m, l, acc)
    int* cnt;     // chunked step in two launches: [unit] count of the unit's chunks (+ residual unit) that have written
                  // their partial; the one that finds all the others done merges them
    // Chunked step in ONE launch (every chunk's workgroup resident at once): the chunks of a unit exchange their
    // logit min / max inside the launch.  rec: [unit][head][chunk][2] 64-bit records, a float (min, then max)
    // in the lower half and the call's epoch in the upper half - a record is valid by itself, so a chunk
    // publishes with plain write-through stores and waits for nothing, and the others poll the records
    // (whatever an earlier call or an uninitialised workspace left there has another epoch).  done: [unit][chunk] words
    // (in the place of the two-launch form's min / max), and done_res [unit] for the window's workgroup (in
    // that of its counters), set to done_tag() of the epoch when the workgroup's partial is written: the unit's first workgroup
    // waits for them and merges.  status: host-visible word that a workgroup sets
    // when it gives up waiting (spin_limit polls); NULL: nowhere to report.
    unsigned long long* rec;
    unsigned long long* done;
    unsigned long long* done_res;
    int* status;
    uint32_t epoch;
    int fused;
    int stream;   // launch_streams()
    int spin_limit;
#ifdef CQ_PHASE_STOPS
    int stop;     // phase boundary at which the launch ends (-1: runs to the end)
#endif
    int B, Hq, Hkv, T, R, S;
    int nsplit, chunk, nx;
    int calib;
    float off_max, off_min;
    FastDiv d_ng, d_nx, d_hkv;   // divisors of the unit decomposition: head groups, chunks (+ residual unit), kv heads
    int G;        // query heads per kv head
    int ncu;      // paired launch whose workgroups are all resident from the start (at most two per compute unit):
                  // the number of compute units (the two workgroups of a unit are told apart by it); else 0
};


// VTOK: values quantised per token and per group of 32 channels (scale * code + minimum, codes in little-endian
// 32-bit words, first channel in the lowest bits) instead of per channel.
// Region A of the LDS holds the query's digits while the logits are worked out, then one 64-token tile of weights and of
// packed V rows per wave, later the folds' partials; the words a whole workgroup shares lie behind it.
template <int BITS, int HPB, bool VTOK = false, int NT_ = 1024> struct Lay {
    static constexpr int kNT = NT_;                 // threads per workgroup
    static constexpr int kNW = kNT / kWave;         // waves per workgroup
    // residual window: tiles of 128 rows for either workgroup size - a 512-thread workgroup puts 4 lanes on a
    // row (32 channels each), a 1024-thread one 8 (16 channels each)
    static constexpr int LPR = kNT / 128;           // lanes per residual row
    static constexpr int kResTile = kNT / LPR;      // residual rows per tile
    static constexpr int NKP = 16 / LPR;            // 16-byte pieces of a row per lane
    static constexpr int RPW = kResTile / kNW;      // rows of a tile whose values one wave multiplies
    static constexpr int NB = 16 * BITS;            // bytes per packed row
    static constexpr int KR = kMatrixK / BITS;      // K token rounds in flight per thread
    // bytes of a wave's tile: weights, then packed V rows (VTOK: weights and rows of one channel group, statistics)
    static constexpr int MXT = VTOK ? 2560 : (1 + BITS) * 1024;
    static constexpr int kRegionA = cmax(kNW * MXT, kNW * kD * HPB * 4);
    // shared words, in floats (what is read as vectors first: each of these starts on 16 bytes)
    static constexpr int F_QRAW = 0;                          // HPB*kD raw 16-bit q
    static constexpr int F_SRES = F_QRAW + HPB * kD / 2;      // kResTile*HPB: logits of a tile of the window
    static constexpr int F_PRES = F_SRES + kResTile * HPB;    // kResTile*HPB: the waves' closing sums
    static constexpr int F_VSZ = F_PRES + kResTile * HPB;     // 2*kD: value scale, zero-point
    static constexpr int F_QSZ = F_VSZ + (VTOK ? 0 : 2 * kD); // [head]: value of one grid step, zero-point sum
    static constexpr int F_RED = F_QSZ + 2 * HPB;             // minima, maxima, masked maxima; from 4*HPB the chunks' fold and its flag
    static constexpr int F_STAT = F_RED + 8 * HPB;            // 8*HPB: per-head softmax state
    static constexpr int F_END = F_STAT + 8 * HPB;
    static_assert(kNW * 5 * HPB <= kResTile * HPB, "the waves' closing sums fit the window's weights");
    static constexpr int kLds = kRegionA + (F_END * 4 + 255) / 256 * 256;
};

// Tokens a chunk of a plan may have, for units of hpb heads in 1 024 threads.  These are what the LDS tables of an earlier
// form of the kernel left room for (the limits of the forms below are of the same kind); the instantiations hold more, up to
// launch_rounds() * threads.
constexpr int plan_chunk(int bits, bool vtok, int hpb) {
    if (vtok) return bits == 1 ? (hpb == 4 ? 3520 : hpb == 2 ? 4480 : 4736) : (hpb == 2 ? 4672 : 5120);
    return bits == 1 ? (hpb == 4 ? 4480 : hpb == 2 ? 10560 : 16384) : (hpb == 4 ? 4096 : hpb == 2 ? 10176 : 16384);
}
constexpr int kPlanLong = 10048;                     // four heads at 1 bit, where that saves the chunks
constexpr int kPlanPair4 = 4096, kPlanPair2 = 4736;  // 512 threads: four heads, two heads (1 bit)

// Launches whose packed rows (and per-token statistics) are most of the 256 MB memory-side cache or more, each read by one
// unit: hardly anything of them would be found there again, and non-temporal loads stream faster.  us at 3 328 + 128 tokens,
// ordinary / non-temporal, with the rows from memory (a model's other layers in between) and, in brackets, the same call repeated:
// 1 bit, 123 MB 45.2 / 43.4 (39.2 / 41.0), 150 MB 52.3 / 51.0 (46.5 / 48.3), 177 MB 61.0 / 58.5 (56.4 / 55.6), batch 256, 218 MB, 71.9 / 69.5
// (72.8 / 65.5); with per-token values 82 MB 34.2 / 33.9 (31.3 / 32.7), 164 MB 66.6 / 64.7 (60.3 / 62.8), 204 MB 82.6 / 81.7 (80.6 / 80.0); 2 bits,
// 109 MB 26.9 / 27.5 (23.3 / 27.0), 218 MB 52.2 / 52.5 (45.9 / 51.5), 245 MB 63.5 / 61.3 (60.9 / 61.2), 436 MB 101.0 / 101.5 (101.3 / 99.8), with
// per-token values no difference at any size.  So the lines are 168 MiB and, at 2 bits, 228 MiB: from there on neither gets
// slower.  Where two units share the rows: 16 x 9 984 with two units per kv head 20.5 / 21.9; in chunks: 8 x 32 768 (67 MB)
// 26.7 / 28.0.  Instantiated for the forms that such launches take (four heads per unit).
constexpr bool stream_form(int bits, bool vtok, int hpb, int nt) { return hpb == 4 && (vtok ? bits == 1 : nt == 512); }
inline bool launch_streams(int bits, bool vtok, int hpb, int nt, int groups, int nsplit, int64_t tokens) {   // tokens: over all (batch, kv head) pairs
    return stream_form(bits, vtok, hpb, nt) && groups == 1 && nsplit == 1 &&
           tokens * (32 * bits + (vtok ? 16 : 0)) >= (static_cast<int64_t>(bits == 1 ? 168 : 228) << 20);
}

// What a launch of units of hpb heads in nt threads runs with: the rounds of logits its instantiation keeps in
// registers for chunks of at most `chunk` tokens, and its dynamic LDS.  Launches pick by the first and check themselves
// against both (cq_decode_matrix.h); cq_decode_attn_plan reports them.
constexpr int launch_rounds(bool vtok, int hpb, int nt, int chunk) {
    if (vtok) return chunk <= kRegTwoBit * nt ? kRegTwoBit : kRegPair;
    if (hpb == 4) return nt == 512 ? kRegPair : kRegLong;
    const int few = nt == 512 ? kRegPair : kRegLong;
    return chunk <= few * nt ? few : kRegMost;
}
template <int BITS, bool VTOK, int NT> constexpr int launch_lds(int hpb) {
    return hpb == 4 ? Lay<BITS, 4, VTOK, NT>::kLds : hpb == 2 ? Lay<BITS, 2, VTOK, NT>::kLds : Lay<BITS, 1, VTOK, NT>::kLds;
}
inline int launch_lds(int bits, bool vtok, int hpb, int nt) {
    if (vtok) return bits == 1 ? launch_lds<1, true, 1024>(hpb) : launch_lds<2, true, 1024>(hpb);
    if (nt == 512) return bits == 1 ? launch_lds<1, false, 512>(hpb) : launch_lds<2, false, 512>(hpb);
    return bits == 1 ? launch_lds<1, false, 1024>(hpb) : launch_lds<2, false, 1024>(hpb);
}

// Unit decomposition of a 1-D grid.  Consecutive work ids share packed codes
// (head groups of one kv-head), so when the grid is a multiple of the 8 XCDs
// the hardware's round-robin placement is undone to keep them on one L2.
__device__ __forceinline__ int virtual_block_id() {
    const int n = gridDim.x;
    const int l = blockIdx.x;
    if ((n & 7) == 0) return (l & 7) * (n >> 3) + (l >> 3);
    return l;
}

typedef short S4 __attribute__((ext_vector_type(4)));
// A weight 0 <= p <= 1 in three 16-bit parts, p = kPartUnit * (part 0 + kPartScale * part 1 + kPartScale^2 * part 2): bf16 holds 8 bits in each, all
// 24; fp16 11, the weight and the lower parts scaled up so that none is lost to its small exponents (to 2^-61 of a weight of 1).  Part 0 is 0 only
// where the weight is, and so infinite times an infinite value (a weight below 2^-39 takes fp16's smallest number, part 1 what that is too much).
template <typename DT> constexpr float kPartScale = std::is_same<DT, FP16>::value ? 1.f / 4096.f : 1.f;
template <typename DT> constexpr float kPartUnit = std::is_same<DT, FP16>::value ? 1.f / 16384.f : 1.f;
template <typename DT> __device__ __forceinline__ void split_weight(float p, uint32_t* o) {
    if constexpr (std::is_same<DT, FP16>::value) p *= 16384.f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if constexpr (std::is_same<DT, BF16>::value) {
            const uint32_t b = __float_as_uint(p) & 0xffff0000u;
            o[i] = b >> 16;
            p -= __uint_as_float(b);
        } else {
            o[i] = Cvt<DT>::from_float(p);
            if (i == 0) o[0] = max(o[0], min(__float_as_uint(p), 1u));
            p = (p - Cvt<DT>::to_float(o[i])) * 4096.f;
        }
    }
}

// A float handed from one workgroup to another inside a launch: device-scope atomic store.
__device__ __forceinline__ void publish(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The partials of a unit are announced in a word each, not counted: read-modify-writes are executed at the memory side
// whatever scope they name (about 2 us a round trip, those on one address one after the other; with
// a compare-and-swap counter that a unit's workgroups retried on, us, counter -> words: 8 chunks a unit (8 x 32 768) 27.5 ->
// 25.0, 16 (4 x 16 384 + 200, 2 bits) 40.4 -> 25.2, 32 (1 x 32 768 + 100) 68.6 -> 20.7).  The first wave of the
// unit's first workgroup polls the others' words, as many times as the caller's bound says (every other workgroup ends
// without waiting for this one, so the bound only matters where they are not all resident together).
// Whoever is last leaves the unit's words empty, because a recorded launch comes back with the same epoch.  That is the
// first workgroup if its wait succeeds.  If not, it takes the words over with another mark and leaves the number of
// workgroups still to come in its own word; one that finds the mark as it announces itself counts down, and the last clears.
// (Announcing by exchange, whose result nothing waits for but the workgroup's own end, instead of by a store: no difference.)
// A word is the epoch and its complement, so nothing else that a workspace may hold passes for one.
__device__ __forceinline__ unsigned long long* done_word(const DecodeGeom& g, int64_t unit, int split) {
    return split < g.nsplit ? g.done + unit * g.nsplit + split : g.done_res + unit;
}
__device__ __forceinline__ unsigned long long done_tag(uint32_t epoch) { return static_cast<unsigned long long>(epoch) << 32 | static_cast<uint32_t>(~epoch); }
__device__ __forceinline__ unsigned long long left_tag(uint32_t epoch) { return static_cast<unsigned long long>(epoch) << 32 | epoch; }

// The single-launch chunked step's hand-over words of one unit back to empty, by `nt` threads, once every other workgroup is past them.
template <int HPB>
__device__ __forceinline__ void clear_handover(const DecodeGeom& g, int64_t unit, int tid, int nt) {
    for (int i = tid; i < HPB * g.nsplit * 2; i += nt)
        __hip_atomic_store(g.rec + unit * HPB * g.nsplit * 2 + i, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int i = tid; i <= g.nsplit; i += nt) __hip_atomic_store(done_word(g, unit, i), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// One thread of a workgroup other than the unit's first, when its partial (if it has one) is written.
template <int HPB>
__device__ __forceinline__ void announce(const DecodeGeom& g, int64_t unit, int split) {
    if (__hip_atomic_exchange(done_word(g, unit, split), done_tag(g.epoch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != left_tag(g.epoch)) return;
    if (__hip_atomic_fetch_add(g.done + unit * g.nsplit, ~0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 1ull) clear_handover<HPB>(g, unit, 0, 1);
}
// One wave of the unit's first workgroup: true when every other one has announced itself; false when the bound is used
// up, and the unit's words are no longer this workgroup's business.
__device__ __forceinline__ bool others_done(const DecodeGeom& g, int64_t unit, int lane) {
    for (int it = 0; it < g.spin_limit; ++it) {
        bool all = true;
        for (int s = 1 + lane; s < g.nx; s += 64)
            all = all && __hip_atomic_load(done_word(g, unit, s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == done_tag(g.epoch);
        if (__builtin_amdgcn_ballot_w64(!all) == 0) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    // The count is in place (its exchange has returned) before the first mark is.
    unsigned long long* count = g.done + unit * g.nsplit;
    if (lane == 0) __hip_atomic_exchange(count, static_cast<unsigned long long>(g.nx), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    int here = 1;   // this workgroup and those that came before the mark
    for (int s0 = 1; s0 < g.nx; s0 += 64) {
        const int s = s0 + lane;
        const bool came = s < g.nx && __hip_atomic_exchange(done_word(g, unit, s), left_tag(g.epoch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == done_tag(g.epoch);
        here += __builtin_popcountll(__builtin_amdgcn_ballot_w64(came));
    }
    bool last = false;
    if (lane == 0) last = __hip_atomic_fetch_add(count, ~0ull * static_cast<unsigned>(here), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == static_cast<unsigned long long>(here);
    return __builtin_amdgcn_ballot_w64(last) != 0;   // (all of them are past their words after all)
}

// ---- the step on the matrix cores --------------------------------------------------------------
// The codes are small integers, so both contractions run exactly on the matrix cores: what is not
// an integer - q.s_k, and the softmax weights - is put on a 32-bit fixed-point grid of its own maximum and split into
// digits.  The 16 rows of a tile are four heads times four digits (pairs of digits), the columns are tokens (logits)
// or byte columns of the packed V rows (sums), and a lane of the result holds the sums of one head:
// exact integers, put together in fp32.
// Values: 8-bit integer products (16 x 16 x 64), weights as four signed byte digits, packed V bytes masked in place - a code then counts 2^s,
// which the closing fold takes back.  Logits: 6-bit by 4-bit float products (16 x 16 x 128) take a token's 128 channels at twice the rate and
// expand packed codes to half bytes, 5 instructions per 32 codes where byte fields take 9 (two bits: 3 per 16, 5).  The digits
// then have 4 bits, so as many products are issued either way (2 x 4 per 64 tokens), but their sums come as floats that three
// multiply-adds put together, without integer shifts and conversions: 53 vector instructions per 64 tokens and four heads for 66.
// (8-bit floats on the left, which need no packing of digits, halve the rate.  The codes' rows loaded as the products read them,
// 4 bytes of four rows to a lane, save the exchange between lanes, but a quarter of a load's lanes then covers 16 rows: batch 64 18.2 -> 20.0.)
// What bounds it: a wave issues 53 vector instructions per 64 tokens and four heads for the logits, 70 for weights and values, and 16
// products, which vector instructions of other waves do not overlap with here (8 integer products and 64 ANDs of four waves a
// SIMD take the sum of their times).  At batch 256 that keeps the SIMDs busy for nine tenths of a launch.
// Measured, us per step in turn on one box, against 8-bit integer products for the logits, the window on dot products, logits all in
// registers and rounds that are skipped one by one: batch 64 x 3 328 + 128 18.6 -> 17.7, 2 bits 27.5 -> 27.0; batch 256 x 3 328 52.7 -> 51.6,
// x 300 + 40 32.7 -> 27.3; 16 x 9 984 + 105, six heads 19.5 -> 18.8; 8 x 32 768 in chunks 24.2 -> 22.6; batch 1 and 6 no difference.
// Error against 64 bits: a weight is off by 2^-31 at most and exact from 2^-7 on (weight_digits()); a channel's q.s_k by 2^(s - 32) of the head's
// largest (s = 0 .. 2), then the fp32 roundings.  fp16 outputs lie 1.9e-4 to 2.3e-4 from 64 bits, bf16 1.5e-3 to 1.8e-3, which is their own
// rounding (sixteen shapes, the same to four digits as with integer products).
typedef int I4 __attribute__((ext_vector_type(4)));
typedef int I2 __attribute__((ext_vector_type(2)));

// The logits' operands.  Right: packed codes as 4-bit floats (E2M1), eight to a dword, masked in place: the fields of a half byte
// read 0.5, 1 and 2 - the topmost would be the sign and is moved to the lowest place; a 2-bit code in the lower half of one reads
// half its value, the upper is moved down.  Left: a channel's q.s_k on a 32-bit grid of the head's largest, divided by what its field counts,
// as a sign and eight 4-bit digits in 6-bit floats (E2M3, where 0 .. 15 eighths are the codes 0 .. 15): rows (head, pair of
// digits), the lower and the upper digit of a pair one product each, 16 apart by the product's own scale.  All sums are whole
// numbers of sixteenths below 2^24, exact in fp32.
// k order: lane (x, kg) has dword kg of a packed row (two bits: dwords kg and 4 + kg).
// A wave prepares a head, a lane two neighbouring channels (query_pair() * 2 and the next): their fields are neighbours as well.  Lanes that
// differ in bits 0, 1, 3 hold the eight nibbles of the same two dwords.
template <int BITS> __device__ __forceinline__ int query_pair(int lane) {
    const int j = ((lane & 3) | ((lane >> 1) & 4)) ^ 1, b2 = (lane >> 2) & 1;   // (nibble n of a dword is the higher of a byte's halves for odd n, the earlier channels)
    return (lane & 0x30) | (BITS == 1 ? (j << 1) | b2 : (b2 << 3) | j);
}

// 4 nibbles (of the lower 16 bits) -> 24 bits, two empty bits above each
__device__ __forceinline__ uint32_t spread6(uint32_t x) {
    const uint32_t t = (x & 0xffu) | ((x << 4) & ~0xffu);
    return ((t & 0x00f00fu) | ((t << 2) & ~0x00f00fu)) & 0x3cf3cfu;
}

// Eight lanes' numbers to 48 bits of codes: lane n ends with digit n of all of them, in nibble order.  (The butterfly of an 8 x 8 transposition of
// nibbles; `neg`: the signs of the wave's lanes.)
struct Codes { uint32_t lo, hi; };   // 24 bits each
__device__ __forceinline__ Codes digit_codes(int x, int lane) {
    uint32_t w = static_cast<uint32_t>(x < 0 ? -x : x);
    const uint64_t neg = __builtin_amdgcn_ballot_w64(x < 0);
    uint32_t t = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w), 0xB1, 0xf, 0xf, true));    // lane ^ 1
    t = __builtin_amdgcn_alignbit(t, t, (lane & 1) ? 4 : 28);
    const uint32_t own = (lane & 1) ? 0xf0f0f0f0u : 0x0f0f0f0fu;
    w = (w & own) | (t & ~own);
    t = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w), 0x4E, 0xf, 0xf, true));             // lane ^ 2
    w = __builtin_amdgcn_perm(t, w, (lane & 2) ? 0x03070105u : 0x06020400u);
    t = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w), 0x128, 0xf, 0xf, true));            // lane ^ 8
    w = __builtin_amdgcn_perm(t, w, (lane & 8) ? 0x03020706u : 0x05040100u);
    // (bit i of four times 0x108420 stands at i + 5 k + 5, once each: those at 6 i + 5 are kept)
    const uint32_t sg = static_cast<uint32_t>(neg >> (lane & 0x34));
    return {spread6(w) | (((sg & 15u) * 0x108420u) & 0x820820u), spread6(w >> 16) | ((((sg >> 8) & 15u) * 0x108420u) & 0x820820u)};
}

// One head of q.s_k into the left operand, by one wave.  qs: a lane's two channels.  In LDS: [lower, upper digits][lane] 24 bytes.
// scale: (value of one step of the result, zero-point sum).
constexpr int kQueryHalf = 64 * 24;
template <int BITS>
__device__ __forceinline__ void matrix_query(const float* qs, float qz, int h, int lane, unsigned char* operand, float* scale) {
    const int top = wave_max_key(max(__builtin_bit_cast(int, qs[0]) & 0x7fffffff, __builtin_bit_cast(int, qs[1]) & 0x7fffffff));
    const float zs = wave_sum(qz);
    // the largest value lies in [2^(e-1), 2^e); a head that is all but zero keeps a grid of 2^-91
    const int e = max((top >> 23) - 126, -60);
    const float grid = __builtin_bit_cast(float, (31 - e + 127) << 23);
    // fields of the pair: at 1 bit 3 and 2, or 1 and 0; they count 2^shift, shift = 0, 2, 1, 0
    const bool low = lane & 4;
    const float c0 = BITS == 1 && low ? grid * 0.5f : grid, c1 = BITS == 1 && !low ? grid * 0.25f : grid;
    const Codes odd = digit_codes(__float2int_rn(qs[0] * c0), lane), even = digit_codes(__float2int_rn(qs[1] * c1), lane);
    const int digit = (lane & 3) | ((lane >> 1) & 4);
    const int kg = BITS == 1 ? lane >> 4 : ((lane >> 4) & 1) * 2 + (low ? 1 : 0), part = BITS == 1 ? (low ? 0 : 1) : lane >> 5;   // k block, and which half of its 24 bytes
    uint32_t* o = reinterpret_cast<uint32_t*>(operand + (digit & 1) * kQueryHalf + (kg * 16 + 4 * h + (digit >> 1)) * 24 + part * 12);
    o[0] = even.lo | (even.hi << 24);
    o[1] = (even.hi >> 8) | (odd.lo << 16);
    o[2] = (odd.lo >> 16) | (odd.hi << 8);
    if (lane == 0) {
        // an infinity or a NaN anywhere in the head makes all its logits NaN, as a floating-point sum would
        // (results count 16 grid steps: a digit is held as eighths, the lowest field as a half)
        scale[2 * h] = top >= 0x7f800000 ? __builtin_nanf("") : __builtin_bit_cast(float, (e - 31 + 4 + 127) << 23);
        scale[2 * h + 1] = zs;
    }
}

typedef int I8 __attribute__((ext_vector_type(8)));
struct QueryOperand { I8 lower, upper; };   // (6-bit floats: six dwords of each)
__device__ __forceinline__ QueryOperand load_query(const unsigned char* regA, int lane) {
    QueryOperand o;
    const U2* p = reinterpret_cast<const U2*>(regA) + 3 * lane;
    const U2 l0 = p[0], l1 = p[1], l2 = p[2], u0 = p[192], u1 = p[193], u2 = p[194];
    o.lower = I8{static_cast<int>(l0.x), static_cast<int>(l0.y), static_cast<int>(l1.x), static_cast<int>(l1.y), static_cast<int>(l2.x), static_cast<int>(l2.y), 0, 0};
    o.upper = I8{static_cast<int>(u0.x), static_cast<int>(u0.y), static_cast<int>(u1.x), static_cast<int>(u1.y), static_cast<int>(u2.x), static_cast<int>(u2.y), 0, 0};
    return o;
}

// Logits of 64 tokens, one row per lane: a 4 x 4 exchange of dwords between the four groups of 16 lanes gives lane
// (x, kg) dword kg of the tokens x, 16 + x, 32 + x, 48 + x - the right operand of four 16-token tiles.  The results are in steps of
// the query's grid, before the zero-point: logit = result * step - zero-point sum, which the minima and maxima take (the map is
// monotone) and the exponent's factor carries.
template <int BITS>
__device__ __forceinline__ void matrix_logits(const uint4* c, const QueryOperand& a, float* out) {
    uint32_t w[BITS][4];
#pragma unroll
    for (int s = 0; s < BITS; ++s) {
        const auto x01 = __builtin_amdgcn_permlane16_swap(c[s].x, c[s].y, false, false);
        const auto x23 = __builtin_amdgcn_permlane16_swap(c[s].z, c[s].w, false, false);
        const auto y02 = __builtin_amdgcn_permlane32_swap(x01[0], x23[0], false, false);
        const auto y13 = __builtin_amdgcn_permlane32_swap(x01[1], x23[1], false, false);
        w[s][0] = y02[0]; w[s][2] = y02[1]; w[s][1] = y13[0]; w[s][3] = y13[1];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t u = w[0][j], v = w[BITS - 1][j];
        I8 f;
        if constexpr (BITS == 1)
            f = I8{static_cast<int>(u & 0x11111111u), static_cast<int>(u & 0x22222222u), static_cast<int>(u & 0x44444444u), static_cast<int>((u >> 3) & 0x11111111u), 0, 0, 0, 0};
        else
            f = I8{static_cast<int>(u & 0x33333333u), static_cast<int>((u >> 2) & 0x33333333u), static_cast<int>(v & 0x33333333u), static_cast<int>((v >> 2) & 0x33333333u), 0, 0, 0, 0};
        F4 acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a.lower, f, F4{0.f, 0.f, 0.f, 0.f}, 2, 4, 0, 0x7f, 0, 0x7f);
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a.upper, f, acc, 2, 4, 0, 0x83, 0, 0x7f);   // x 2^4
        const float lo = __builtin_fmaf(acc[1], 256.f, acc[0]), hi = __builtin_fmaf(acc[3], 256.f, acc[2]);
        out[j] = __builtin_fmaf(hi, 65536.f, lo);
    }
}

// Eight rows of one byte column per lane: of a [row][16 bytes] tile in LDS, lane x of 16 gets byte x of eight rows
__device__ __forceinline__ I2 column8(const unsigned char* p) {
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) I2*)(p));
}

// The fields of a packed V byte in place, each sum counting 2^shift (the fold takes it back); the byte itself instead of
// the topmost, as a signed number - at 1 bit -128 b7 + the others; at 2 bits, with the top bit flipped, the byte less 128, which
// needs the sum of the weights as well (accumulator 8).  One AND or XOR per four codes less than a shift and four masks.
template <int BITS> __device__ __forceinline__ constexpr int value_mask(int i) {
    if (BITS == 1) return i < 7 ? 0x01010101 << i : 0;
    return i < 3 ? 0x03030303 << (2 * i) : static_cast<int>(0x80808080u);
}

// Weighted code sums of 64 tokens.  The weights (lane: head lane / 16, tokens 16 j + x) go through the wave's LDS tile
// as [token][head] words, i.e. rows of 16 digit bytes, the packed V rows as they are, [token][16 bytes]; both come
// back by columns, 16 tokens of one column per lane.  first: there are no sums yet.
template <int BITS>
__device__ __forceinline__ void matrix_values(unsigned char* tile, const float* e, const U4* v, I4* acc, bool first) {
    const int lane = threadIdx.x & 63, x = lane & 15, k = lane >> 4;
#pragma unroll
    for (int s = 0; s < BITS; ++s) *reinterpret_cast<U4*>(tile + (1 + s) * 1024 + lane * 16) = v[s];
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t*>(tile + (16 * j + x) * 16 + 4 * k) = weight_digits(e[j], 1073741824.f);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const unsigned char* col = tile + (16 * k + (x >> 1)) * 16 + (x & 1) * 8;
    const I2 e0 = column8(col), e1 = column8(col + 128);
    const I4 a = {e0[0], e0[1], e1[0], e1[1]};
#pragma unroll
    for (int s = 0; s < BITS; ++s) {
        const I2 v0 = column8(col + (1 + s) * 1024), v1 = column8(col + (1 + s) * 1024 + 128);
        const int w[4] = {v0[0], v0[1], v1[0], v1[1]};
        constexpr int NF = 8 / BITS;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            const int m = value_mask<BITS>(i);
            I4 f;
#pragma unroll
            for (int r = 0; r < 4; ++r) f[r] = i < NF - 1 ? w[r] & m : w[r] ^ m;
            acc[s * NF + i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, f, first ? I4{0, 0, 0, 0} : acc[s * NF + i], 0, 0, 0);
        }
    }
    if constexpr (BITS == 2) acc[8] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, I4{0x01010101, 0x01010101, 0x01010101, 0x01010101}, first ? I4{0, 0, 0, 0} : acc[8], 0, 0, 0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the lane's sums (one head, byte column x) as floats in channel order (sums of digits are whole numbers below 2^28)
template <int BITS> __device__ __forceinline__ void matrix_fold(const I4* acc, float* out, int x, int swz) {
    constexpr int NF = 8 / BITS;
#pragma unroll
    for (int s = 0; s < BITS; ++s) {
        I4 top = -acc[s * NF + NF - 1];
        if constexpr (BITS == 1) {
#pragma unroll
            for (int i = 0; i < NF - 1; ++i) top += acc[i];                     // 128 x the topmost field's sums
        } else {
            top = 128 * acc[8] - top;                                           // the unsigned bytes' sums
#pragma unroll
            for (int i = 0; i < NF - 1; ++i) top -= acc[s * NF + i];            // 64 x
        }
        Vec<4> o[NF / 4];
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            const I4 a = i < NF - 1 ? acc[s * NF + i] : top;
            float r = static_cast<float>(a[3]);
#pragma unroll
            for (int p = 2; p >= 0; --p) r = __builtin_fmaf(r, 256.f, static_cast<float>(a[p]));
            const float unit = 1.f / (1073741824.f * static_cast<float>(1 << (BITS * i)));
            o[(NF - 1 - i) / 4].v[(NF - 1 - i) % 4] = r * unit;   // first channel of a byte in its top bits
        }
#pragma unroll
        for (int q = 0; q < NF / 4; ++q) *reinterpret_cast<Vec<4>*>(out + (((16 * s + x) * NF + 4 * q) ^ swz)) = o[q];
    }
}

// Per-token values: a weight is e * scale[token][group of 32 channels], so every group has a left operand of its own.
// The right operand is arranged for it: a group's 4 (8) bytes of a row, read back by columns as 8 rows x 8 bytes (at 1 bit
// the four bytes twice), meet in lane x as byte x mod 4 (8), and the lane keeps the field x / 4 (x / 8) of it and, from the
// byte shifted by four, the one half a byte higher: 16 columns of the result are 16 channels, two MFMAs are a group.
// The grid is a head's own largest e * scale of the group among the wave's tokens - the weighted scale, because a token
// without weight (masked, or out of this head's sight) may have a scale of any size; sums of e * minimum stay in fp32.
// Measured at batch 64 x 3 328 + 128, 1 bit, us per step in turn on one box: look-up form 58.6, this one 38.9 (1 024 threads,
// one workgroup per compute unit: the four groups' operands, converted and read back one after the other, are what bounds
// it).  Grids of the scales alone, as wide as the least weighted token makes them, were within 1 % there and 2.5 % faster in
// the middle of 60 shapes.
// Weights and scales have 32 bits here, the look-up tables held their products and short sums as fp16.
// st: the lane's own token's scales and minima (layout of `stats` below); pw: the head's grid, 2^(30 - e) per group.
template <int BITS, typename DT>
__device__ __forceinline__ void matrix_values_token(unsigned char* tile, const float* e, const U4* v, U4 st, const float* pw,
                                                    float* cm, I4* acc) {
    const int lane = threadIdx.x & 63, x = lane & 15, k = lane >> 4;
    unsigned char* rows = tile + 1024;    // [token][8 bytes]
    unsigned char* stats = tile + 1536;   // [token][scales 0 1, minima 0 1, scales 2 3, minima 2 3]
    *reinterpret_cast<U4*>(stats + lane * 16) = st;
    const uint32_t mask = BITS == 1 ? 0x01010101u << (x >> 2) : 0x03030303u << (2 * (x >> 3));
    const unsigned char* col = tile + (16 * k + (x >> 1)) * 16 + (x & 1) * 8;
    const unsigned char* rcol = rows + (16 * k + (x >> 1)) * 8;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float sc[4][2];                       // [16 j + x][group of the pair]: e * scale
#pragma unroll
    for (int gi = 0; gi < 4; ++gi) {
        if (gi % 2 == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const U2 t = *reinterpret_cast<const U2*>(stats + (16 * j + x) * 16 + 4 * gi);
                sc[j][0] = e[j] * Cvt<DT>::lo(t.x);
                sc[j][1] = e[j] * Cvt<DT>::hi(t.x);
                cm[gi] = __builtin_fmaf(e[j], Cvt<DT>::lo(t.y), cm[gi]);
                cm[gi + 1] = __builtin_fmaf(e[j], Cvt<DT>::hi(t.y), cm[gi + 1]);
            }
        }
        U2 w2;
        if constexpr (BITS == 1) { w2.x = v[0][gi]; w2.y = v[0][gi]; }
        else { w2.x = v[gi >> 1][2 * (gi & 1)]; w2.y = v[gi >> 1][2 * (gi & 1) + 1]; }
        *reinterpret_cast<U2*>(rows + lane * 8) = w2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // (at most 2^30: the grid comes from this very product)
            *reinterpret_cast<uint32_t*>(tile + (16 * j + x) * 16 + 4 * k) = weight_digits(sc[j][gi % 2], pw[gi]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const I2 e0 = column8(col), e1 = column8(col + 128), v0 = column8(rcol), v1 = column8(rcol + 64);
        const I4 a = {e0[0], e0[1], e1[0], e1[1]};
        const uint32_t w[4] = {static_cast<uint32_t>(v0[0]), static_cast<uint32_t>(v0[1]), static_cast<uint32_t>(v1[0]), static_cast<uint32_t>(v1[1])};
        I4 f0, f1;
#pragma unroll
        for (int r = 0; r < 4; ++r) { f0[r] = static_cast<int>(w[r] & mask); f1[r] = static_cast<int>((w[r] >> 4) & mask); }
        acc[2 * gi] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, f0, acc[2 * gi], 0, 0, 0);
        acc[2 * gi + 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, f1, acc[2 * gi + 1], 0, 0, 0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// A dword of every lane's own token to the lanes that hold the token's weights: o[j] is that of token 16 j + x
__device__ __forceinline__ void token_rows(uint32_t v, uint32_t* o) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false), b = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
    o[0] = a[0]; o[1] = a[1]; o[2] = b[0]; o[3] = b[1];
}

// The largest |e * scale| of every group so far, as bit patterns (unsigned: a NaN is larger than any number).
// scales: the lane's own token's
template <typename DT> __device__ __forceinline__ void token_tops(const float* e, U2 scales, uint32_t* top) {
    uint32_t s01[4], s23[4];
    token_rows(scales.x & 0x7fff7fffu, s01);
    token_rows(scales.y & 0x7fff7fffu, s23);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        top[0] = max(top[0], __builtin_bit_cast(uint32_t, e[j] * Cvt<DT>::lo(s01[j])));
        top[1] = max(top[1], __builtin_bit_cast(uint32_t, e[j] * Cvt<DT>::hi(s01[j])));
        top[2] = max(top[2], __builtin_bit_cast(uint32_t, e[j] * Cvt<DT>::lo(s23[j])));
        top[3] = max(top[3], __builtin_bit_cast(uint32_t, e[j] * Cvt<DT>::hi(s23[j])));
    }
}

// its sums as floats in channel order; pw: the grids
template <int BITS> __device__ __forceinline__ void matrix_fold_token(const I4* acc, const float* pw, float* out, int x, int swz) {
    const int byte = BITS == 1 ? x & 3 : x & 7, f = BITS == 1 ? x >> 2 : x >> 3;
    const float field = __builtin_bit_cast(float, (127 - BITS * f) << 23);   // the field counts 2^(BITS f)
#pragma unroll
    for (int gi = 0; gi < 4; ++gi) {
        // the value of one grid step: 1 / pw, or the NaN that stands for a group with an infinity or a NaN in it
        const float unit = pw[gi] != pw[gi] ? pw[gi] : __builtin_bit_cast(float, (254 << 23) - __builtin_bit_cast(int, pw[gi]));
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const I4 a = acc[2 * gi + q];
            float r = static_cast<float>(a[3]);
#pragma unroll
            for (int p = 2; p >= 0; --p) r = __builtin_fmaf(r, 256.f, static_cast<float>(a[p]));
            out[(32 * gi + byte * (8 / BITS) + f + q * (4 / BITS)) ^ swz] = r * field * unit;
        }
    }
}

enum Extras { kNoExtras, kDeviceRows, kMasked };

// CHUNKED: the launch is one of the two of a chunked step (the min/max launch always is); a single launch carries
// none of their code.  EXTRAS: the call has an additive mask (kMasked), or may have a residual row count read from device memory (kDeviceRows;
// never both); a call with neither runs an instantiation without their code (the kernel sits at the register limit of its occupancy,
// and code that never runs still costs registers).  The two apart, because a mask's first values are requested ahead: nine loads a lane that
// a row count, or a chunked launch without a mask, does not need.  Measured, us, one form for both / two: 4 x 733 + 258, per-token values, row count
// 11.14 / 10.60; 16 x 9 984 + 105, six heads, row count 18.12 / 17.66; fifteen shapes with a row count 4.8 % less.
// (A chunked launch with a mask gains nothing from the early request and loses nothing: fifty shapes within 0.1 %.)
// STREAM: the packed rows are read with non-temporal loads (see launch_streams()).
// NH: query heads a unit serves, at most HPB.  Operands and partials are laid out HPB heads wide either way; with
// NH = 3 the fourth head's rows are padding - six query heads per kv-head (InternLM2-20B) make two exact units of
// three instead of two units of four that carry two padding heads between them.
template <int BITS, int HPB, typename DT, bool MINMAX_ONLY, bool VTOK = false, int NT = 1024, int REGL = 0,
          bool CHUNKED = MINMAX_ONLY, Extras EXTRAS = kNoExtras, int NH = HPB, bool STREAM = false>
// (four waves per SIMD - at most 128 VGPRs - for either workgroup size: two 512-thread workgroups per compute
// unit are only resident together within that)
__global__ __launch_bounds__(NT, 4) void decode_kernel(DecodeGeom g) {
    using L = Lay<BITS, HPB, VTOK, NT>;
    constexpr int NB = L::NB;
    constexpr int kNT = L::kNT, kNW = L::kNW, kResTile = L::kResTile;
    extern __shared__ __attribute__((aligned(256))) unsigned char smem[];
    constexpr int PARK = MINMAX_ONLY ? 0 : parked_rounds(VTOK, NT, REGL), RR = REGL - PARK;
    __shared__ F4 parked[MINMAX_ONLY ? 1 : parked_lds(VTOK, NT, REGL) / 16];
    unsigned char* regA = smem;
    float* fx = reinterpret_cast<float*>(smem + L::kRegionA);
    float* qsz = fx + L::F_QSZ;
    float* red = fx + L::F_RED;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = tid >> 6;
    const int G = g.G;
    // Wave priorities of the paired launch (two 512-thread workgroups per compute unit, all of them resident from
    // the first cycle).  Left to the hardware's own arbitration the workgroup that was dispatched first gets most of
    // the issue slots, and the other one ends alone on the unit with too few waves to hide its latencies.  So the
    // short, latency-bound phases (set-up, reductions) go above the throughput phases, the first workgroup ahead in
    // the logits and the second in the packed-V loop.  Measured with and without, us per step at 3 328 + 128 tokens:
    // batch 33, 2 bits 21.1 -> 19.8; batch 40 19.3 -> 18.6; batch 64, 2 bits 27.4 -> 26.6, 1 bit 21.3 -> 21.2; two heads
    // per unit 17.8 -> 18.1.  Launches with more workgroups than fit at once start their later workgroups as earlier
    // ones end, which staggers them by itself; there the priorities are left alone.
    // `second`: the workgroup that shares its unit with an older one (workgroups are handed out unit by
    // unit, g.ncu at a time).
    const bool prio_on = NT == 512 && g.ncu > 0;
    const bool second = prio_on && blockIdx.x >= static_cast<unsigned>(g.ncu);
    auto phase_priority = [&](auto phase_c) {
        constexpr int PH = decltype(phase_c)::value;   // 0 set-up, 1 logits, 2 min/max .. mask, 3 exp and packed V, 4 folds, window, merge
        if constexpr (NT == 512) {
            if (prio_on) {
                if constexpr (PH == 0 || PH == 2) __builtin_amdgcn_s_setprio(2);
                else if constexpr (PH == 1) { if (second) __builtin_amdgcn_s_setprio(0); else __builtin_amdgcn_s_setprio(1); }
                else if constexpr (PH == 3) { if (second) __builtin_amdgcn_s_setprio(2); else __builtin_amdgcn_s_setprio(1); }
                else __builtin_amdgcn_s_setprio(0);
            }
        }
    };
    // (unconditional at entry - with no later change every wave simply runs at this priority - so that no branch
    // on a kernel argument stands between the wave's start and the loads of the other arguments: all of them are
    // then requested in one go instead of in two round trips)
    if constexpr (NT == 512) __builtin_amdgcn_s_setprio(2);

    uint32_t vb = static_cast<uint32_t>(virtual_block_id());
    uint32_t qn = g.d_ng.quot(vb);
    const int hg = static_cast<int>(vb - qn * g.d_ng.div); vb = qn;
    qn = g.d_nx.quot(vb);
    const int split = static_cast<int>(vb - qn * g.d_nx.div); vb = qn;
    qn = g.d_hkv.quot(vb);
    const int hkv = static_cast<int>(vb - qn * g.d_hkv.div);
    const int b = static_cast<int>(qn);
    static_assert(NH >= 1 && NH <= HPB, "heads per unit");
    const int hq0 = hkv * G + hg * NH;
    const int nh = min(NH, G - hg * NH);   // query heads of this unit; the rest of its NH heads are padding
    const int64_t bh = static_cast<int64_t>(b) * g.Hkv + hkv;

    const bool img_unit = split < g.nsplit && g.T > 0;
    const int R = (EXTRAS == kDeviceRows && g.r_dev) ? min(*g.r_dev, g.R) : g.R;   // rows in the residual window
    const bool do_res = !MINMAX_ONLY && R > 0 && (!CHUNKED || split == g.nsplit);
    const int t0 = img_unit ? split * g.chunk : 0;
    const int n = img_unit ? min(g.T, t0 + g.chunk) - t0 : 0;
    const float inv_sqrt_d = 0.08838834764831845f;  // 1/sqrt(128)

    // ---- entry: the few elements phase 0 needs are requested first; the packed K rows follow
    // phase 0, packed V rows and the residual tile later still (see the file header).
    // Loads are unconditional with clamped (always valid) addresses: no divergent
    // control flow around them, so the compiler can wait on exactly the counter value
    // each consumer needs.
    // A unit without packed tokens or without residual rows aims the unused streams
    // at q (always mapped, at least 256 bytes) and never looks at what comes back.
    const bool has_img = n > 0;
    const int64_t unit = bh * static_cast<int64_t>(g.d_ng.div) + hg;
    // wave h < HPB: head h of q and the keys' statistics; the last wave: the values'
    const int wvu = __builtin_amdgcn_readfirstlane(wv);
    const int pair = query_pair<BITS>(lane);   // the two channels this lane sets up
    uint32_t q_raw, s_raw, z_raw;
    {
        const int h = min(min(wvu, HPB - 1), nh - 1);   // a padding head repeats the last real one
        const Pair16* qp = reinterpret_cast<const Pair16*>(static_cast<const uint16_t*>(g.q) + (static_cast<int64_t>(b) * g.Hq + hq0 + h) * kD);
        const bool vstat = !VTOK && wvu == kNW - 1;
        const Pair16* sp = has_img ? reinterpret_cast<const Pair16*>(static_cast<const uint16_t*>(vstat ? g.vs : g.ks) + bh * kD) : qp;
        const Pair16* zp = has_img ? reinterpret_cast<const Pair16*>(static_cast<const uint16_t*>(vstat ? g.vz : g.kz) + bh * kD) : qp;
        q_raw = qp[pair];
        s_raw = sp[pair];
        z_raw = zp[pair];
    }
    static_assert(HPB < kNW, "a wave is left for the values' statistics");
    // Two heads or one: few units (or few heads), where a launch lasts as long as its phases in a row; dot products straight from the loaded rows
    // are the shorter chain (us, 2 x 800 + 250, 16 / 4 heads 8.0 for 8.3; 1 x 300 + 60 6.25 for 6.45).
    constexpr bool kDotWindow = HPB <= 2;
    const int64_t code_off = has_img ? (bh * g.T + t0) * NB : 0;   // one offset for both code streams
    const uint4* ckp = reinterpret_cast<const uint4*>(has_img ? g.ck + code_off : static_cast<const uint8_t*>(g.q));
    const uint4* cvp = reinterpret_cast<const uint4*>((has_img ? g.cv : static_cast<const uint8_t*>(g.q)) + code_off);
    const int last_row = has_img ? n - 1 : 0;
    // residual tile: a thread loads a slice of a K and of a V row (row = tid / LPR, 128 / LPR elements); a wave's rows go through its own
    // part of the LDS
    constexpr int LPR = L::LPR, NKP = L::NKP, RPW = L::RPW;
    const int lq = tid % LPR, krow = tid / LPR;
    // (the strides are read where the other kernel arguments are, not behind the branch that needs them: one
    // round trip to the argument block instead of one more)
    // (a single launch: every workgroup has a window; of a chunked launch only the residual units do)
    int64_t arg_rs_b = g.rs_b, arg_rs_h = g.rs_h, arg_rs_r = g.rs_r;
    if constexpr (!CHUNKED) asm volatile("" : "+s"(arg_rs_b), "+s"(arg_rs_h), "+s"(arg_rs_r));
    const int64_t res_off = do_res ? b * arg_rs_b + hkv * arg_rs_h : 0;   // one offset for both windows
    const uint16_t* kb = static_cast<const uint16_t*>(do_res ? g.kres : g.q) + res_off;
    const uint16_t* vbp = static_cast<const uint16_t*>(do_res ? g.vres : g.q) + res_off;
    const int last_r = do_res ? R - 1 : 0;
    const int64_t rs_r = do_res ? arg_rs_r : 0;
    U4 rk[NKP], rv[NKP];
    auto load_res = [&](const uint16_t* base, int r0, U4* o) {   // rows past R re-read row R-1 (their weight is 0)
        const uint16_t* p = base + min(r0 + krow, last_r) * rs_r + lq * 8;
#pragma unroll
        for (int i = 0; i < NKP; ++i) o[i] = *reinterpret_cast<const U4*>(p + i * (LPR * 8));   // piece i * LPR + lq
    };

    // The first packed K rows are requested behind q and the statistics, before either is looked at: they arrive while q
    // goes onto its grid.  (us, requested after that: 3 328 + 128 tokens, batch 64, 1 bit 20.4 -> 20.0, per-token values
    // 36.7 -> 35.7; 16 x 9 984 20.8 -> 20.3; batch 1 and 6 within 1 %.)
    __builtin_amdgcn_sched_barrier(0);
    // Round r's row of a thread: a scalar base and the thread's offset in the round, both kept inside the chunk (rounds and
    // rows past its end repeat the last row).
    auto row_at = [&](const void* p, int r) {
        const int r0 = min(r * kNT, last_row);
        return reinterpret_cast<const unsigned char*>(p) + static_cast<int64_t>(r0) * NB + min(static_cast<uint32_t>(tid) * NB, static_cast<uint32_t>(last_row - r0) * NB);
    };
    uint4 kc[L::KR][BITS];
    auto request_k = [&](int r) {
        const U4* p = reinterpret_cast<const U4*>(row_at(ckp, r));
#pragma unroll
        for (int i = 0; i < BITS; ++i) kc[r % L::KR][i] = __builtin_bit_cast(uint4, STREAM ? __builtin_nontemporal_load(p + i) : p[i]);
    };
#pragma unroll
    for (int r = 0; r < L::KR; ++r) request_k(r);
    __builtin_amdgcn_sched_barrier(0);

    CQ_PHASE(1);   // prologue, requests of q, the statistics and the first packed K rows
    // ---- phase 0: q onto its grid ---------------------------------------------------
    if (wvu < HPB) {
        reinterpret_cast<uint32_t*>(fx + L::F_QRAW)[wvu * (kD / 2) + pair] = q_raw;
        if (n > 0) {
            const float qs[2] = {Cvt<DT>::lo(q_raw) * inv_sqrt_d * Cvt<DT>::lo(s_raw), Cvt<DT>::hi(q_raw) * inv_sqrt_d * Cvt<DT>::hi(s_raw)};
            matrix_query<BITS>(qs, qs[0] * Cvt<DT>::lo(z_raw) + qs[1] * Cvt<DT>::hi(z_raw), wvu, lane, regA, qsz);
        }
    }
    if (!VTOK && n > 0 && wvu == kNW - 1) {
        *reinterpret_cast<Vec<2>*>(fx + L::F_VSZ + 2 * pair) = Vec<2>{{Cvt<DT>::lo(s_raw), Cvt<DT>::hi(s_raw)}};
        *reinterpret_cast<Vec<2>*>(fx + L::F_VSZ + kD + 2 * pair) = Vec<2>{{Cvt<DT>::lo(z_raw), Cvt<DT>::hi(z_raw)}};
    }
    if (tid < 3 * HPB) reinterpret_cast<int*>(red)[tid] = static_cast<int>(0x80000000u);   // the meeting words of the waves' minima and maxima
    // Chunked launch: the chunks' logit min / max, lane s the pair of chunk s for every head (all in flight
    // together; they are folded across the wave where the calibration needs them).
    struct alignas(8) MinMax { float lo, hi; };
    MinMax mraw[HPB];
    // Logits: round rd's 64 tokens of a wave start at 64 * wv + rd * kNT; lane (x, h) = (lane & 15, lane >> 4) has the
    // logits of head h for the tokens 16 j + x of them
    float lx[RR][4];
    auto get_logits = [&](int rd, float* o) {
        if (rd < RR) {
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = lx[rd < RR ? rd : 0][j];
        } else {
            const F4 v = parked[(rd - RR) * NT + tid];
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = v[j];
        }
    };
    auto put_logits = [&](int rd, const float* o) {
        if (rd < RR) {
#pragma unroll
            for (int j = 0; j < 4; ++j) lx[rd < RR ? rd : 0][j] = o[j];
        } else {
            parked[(rd - RR) * NT + tid] = F4{o[0], o[1], o[2], o[3]};
        }
    };
    if constexpr (!MINMAX_ONLY) {
        if (CHUNKED && has_img && !g.fused) {
#pragma unroll
            for (int h = 0; h < HPB; ++h) {
                const MinMax* p = reinterpret_cast<const MinMax*>(g.mm) +
                                  (static_cast<int64_t>(b) * g.Hq + hq0 + min(h, nh - 1)) * g.nsplit;
                mraw[h] = p[min(lane, g.nsplit - 1)];
            }
        }
    }
    __syncthreads();

    float* stat = fx + L::F_STAT;   // [alpha | m_res | l_res | m_img | l_img][HPB]
    float o_res = 0.f;
    float mn = INFINITY, mx = -INFINITY;   // of the lane's head (hl)
    // First block of packed V rows: half of it is requested here, behind the packed K rows, the
    // rest as the K registers free up, so it has arrived when the logits are done.
    constexpr int kVF = VTOK ? (REGL > 4 ? 1 : 2) * BITS : kMatrixV;   // 16-byte pieces of packed V rows in flight per thread
    U4 vc[kVF];
    auto request_v = [&](int slot, int piece) {   // piece: round * BITS + 16-byte piece of the row
        const U4* p = reinterpret_cast<const U4*>(row_at(cvp, piece / BITS)) + piece % BITS;
        vc[slot] = STREAM ? __builtin_nontemporal_load(p) : *p;
    };
    constexpr int kVEarly = VTOK ? BITS : kMatrixE;
    if constexpr (!MINMAX_ONLY) {
#pragma unroll
        for (int r = 0; r < kVEarly; ++r) request_v(r, r);
    }
    // The mask's values of the first rounds and of the window's first tile, ahead of the phases that add them.  (No mask: q, always mapped.)
    constexpr int kMaskAhead = EXTRAS == kMasked ? (REGL < 2 ? REGL : 2) : 0;
    const bool masked = EXTRAS == kMasked && g.mask;
    const float* mask_img = masked && n > 0 ? g.mask + b * g.mask_sb + g.S + t0 : reinterpret_cast<const float*>(g.q);
    const float* mask_win = masked ? g.mask + b * g.mask_sb : reinterpret_cast<const float*>(g.q);
    float mask_v[kMaskAhead ? kMaskAhead : 1][4], mask_w = 0.f;
    if constexpr (kMaskAhead > 0) {
        const int top = masked && n > 0 ? n - 1 : 0;
#pragma unroll
        for (int r = 0; r < kMaskAhead; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) mask_v[r][j] = mask_img[min((tid & ~63) + r * kNT + 16 * j + (lane & 15), top)];
        const int r = min(wv * RPW + (lane & 15) % RPW, last_r);
        mask_w = mask_win[masked && do_res ? (r < g.S ? r : g.T + r) : 0];
    }

    CQ_PHASE(2);   // q on its grid
    // the wave's first token, and the head whose results this lane holds (lanes beyond the unit's heads repeat
    // the last one)
    const int wt0 = __builtin_amdgcn_readfirstlane(tid);
    const int hl = min(lane >> 4, HPB - 1);
    // per-token values: the chunk's scales and minima, four 16-bit values a token
    const U2* vsp = reinterpret_cast<const U2*>(has_img ? static_cast<const uint16_t*>(g.vs) + (bh * g.T + t0) * 4 : static_cast<const uint16_t*>(g.q));
    const U2* vmp = reinterpret_cast<const U2*>(has_img ? static_cast<const uint16_t*>(g.vz) + (bh * g.T + t0) * 4 : static_cast<const uint16_t*>(g.q));
    U2 ts[VTOK && !MINMAX_ONLY ? REGL : 1];   // the scales of the lane's own tokens
    if (has_img) {
        const QueryOperand aq = load_query(regA, lane);
        float lo = INFINITY, hi = -INFINITY;
        phase_priority(std::integral_constant<int, 1>{});
#pragma unroll
        for (int rd = 0; rd < REGL; ++rd) {
            // (left at the wave's end, not skipped round by round: a wait then counts every load issued since its own)
            if (wt0 + rd * kNT >= n) break;
            float l[4];
            matrix_logits<BITS>(kc[rd % L::KR], aq, l);
            if (rd + L::KR < REGL) request_k(rd + L::KR);
            if (!MINMAX_ONLY) put_logits(rd, l);
#pragma unroll
            for (int j = 0; j < 4; ++j) { lo = fminf(lo, l[j]); hi = fmaxf(hi, l[j]); }
            __builtin_amdgcn_sched_barrier(0);
            if (!MINMAX_ONLY && rd < kVF - kVEarly) request_v(kVEarly + rd, kVEarly + rd);   // the rest of the first packed V rows
        }
        phase_priority(std::integral_constant<int, 2>{});
        if constexpr (VTOK && !MINMAX_ONLY) {   // they arrive during the min / max and the calibration
#pragma unroll
            for (int rd = 0; rd < REGL; ++rd) ts[rd] = vsp[min(tid + rd * kNT, n - 1)];
        }
        // the waves' minima and maxima meet in LDS, from one lane per head
        const int klo = row_max_key(float_key(-lo)), khi = row_max_key(float_key(hi));
        int* redi = reinterpret_cast<int*>(red);
        if ((lane & 15) == 0 && (lane >> 4) < HPB) {
            __hip_atomic_fetch_max(redi + hl, klo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_max(redi + HPB + hl, khi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __syncthreads();
        mn = -key_float(redi[hl]);
        mx = key_float(redi[HPB + hl]);
    }

    CQ_PHASE(4);   // block min / max
    const bool speaks = wv == 0 && (lane & 15) == 0 && (lane >> 4) < nh;   // one lane per real head, for what a workgroup writes per head
    if constexpr (MINMAX_ONLY) {
        if (n > 0 && speaks) {
            float* o = g.mm + ((static_cast<int64_t>(b) * g.Hq + hq0 + hl) * g.nsplit + split) * 2;
            o[0] = mn;
            o[1] = mx;
        }
        if (split == 0 && tid == 0) g.cnt[unit] = 0;   // the main launch counts the unit's partials from 0
        return;
    } else {
        float m_img = -INFINITY;   // of the lane's head
        // From here a lane of the first eight waves owns channel `od` of head `hl`: as the window's products leave them
        const int od = 16 * wv + (lane & 15);
        const bool owns = wv < 8 && (lane >> 4) < HPB;
        float o_img = 0.f;

        if constexpr (CHUNKED) {
            // One launch: this chunk's min / max go out now (write-through stores that nothing waits for); the other
            // chunks' are collected further down.
            // (padding heads repeat the last real one: every head of the unit's layout has its records)
            if (g.fused && has_img && wv == 0 && (lane & 15) == 0 && (lane >> 4) < HPB) {
                unsigned long long* o = g.rec + ((unit * HPB + hl) * g.nsplit + split) * 2;
                const unsigned long long tag = static_cast<unsigned long long>(g.epoch) << 32;
                __hip_atomic_store(o, tag | __float_as_uint(mn), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(o + 1, tag | __float_as_uint(mx), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }

        if (n > 0) {
            // ---- phase 4: calibration + exp ---------------------------------------------
            if constexpr (CHUNKED) {
                if (g.fused) {
                    // Wait until every chunk of the unit has published: the first wave polls the records, lane s
                    // those of chunk s, a bounded number of times (workgroups that are not all resident together -
                    // a smaller device than planned for - must not spin for ever; giving up ends this workgroup
                    // without a result and tells the host), folds them and leaves the unit's min / max in LDS.
                    float* fold = red + 4 * HPB;           // 2 * HPB floats, then whether the wait succeeded
                    int* flag = reinterpret_cast<int*>(fold + 2 * HPB);
                    if (wv == 0) {
                        const unsigned long long* pr = g.rec + ((unit * HPB) * g.nsplit + min(lane, g.nsplit - 1)) * 2;
                        float mm2[2 * HPB];
                        bool ok = false;
                        for (int it = 0; it < g.spin_limit && !ok; ++it) {
                            bool valid = true;
#pragma unroll
                            for (int h = 0; h < HPB; ++h) {
                                const unsigned long long lo = __hip_atomic_load(pr + h * g.nsplit * 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                const unsigned long long hi = __hip_atomic_load(pr + h * g.nsplit * 2 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                valid = valid && static_cast<uint32_t>(lo >> 32) == g.epoch && static_cast<uint32_t>(hi >> 32) == g.epoch;
                                mm2[h] = -__uint_as_float(static_cast<uint32_t>(lo));
                                mm2[HPB + h] = __uint_as_float(static_cast<uint32_t>(hi));
                            }
                            ok = __builtin_amdgcn_ballot_w64(!valid) == 0;
                            if (!ok) __builtin_amdgcn_s_sleep(2);
                        }
                        wave_reduce_n<2 * HPB>(mm2, OpMax(), -INFINITY);
                        if (lane == 0) {
#pragma unroll
                            for (int i = 0; i < 2 * HPB; ++i) fold[i] = mm2[i];
                            *flag = ok ? 1 : 0;
                            if (!ok && g.status) __hip_atomic_store(g.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        }
                    }
                    __syncthreads();
                    if (!*flag) {
                        // Given up: no result from this workgroup, but it still announces itself, so that the unit's
                        // hand-over words are left empty and a replay of this very launch (same epoch)
                        // does not take this launch's records for its own.
                        if (split != 0) {
                            if (tid == 0) announce<HPB>(g, unit, split);
                            return;
                        }
                        int* last = reinterpret_cast<int*>(red);
                        if (wv == 0) {
                            const bool ok = others_done(g, unit, lane);
                            if (lane == 0) *last = ok ? 1 : 0;
                        }
                        __syncthreads();
                        if (*last) clear_handover<HPB>(g, unit, tid, kNT);
                        return;
                    }
                    mn = -fold[hl];
                    mx = fold[HPB + hl];
                } else {
                // one fold for both: max of (-min, max) over the chunks
                float mm2[2 * HPB];
#pragma unroll
                for (int h = 0; h < HPB; ++h) {
                    mm2[h] = -mraw[h].lo;
                    mm2[HPB + h] = mraw[h].hi;
                    const MinMax* p = reinterpret_cast<const MinMax*>(g.mm) +
                                      (static_cast<int64_t>(b) * g.Hq + hq0 + min(h, nh - 1)) * g.nsplit;
                    for (int s = lane + 64; s < g.nsplit; s += 64) {   // (more than 64 chunks)
                        const MinMax v = p[s];
                        mm2[h] = fmaxf(mm2[h], -v.lo);
                        mm2[HPB + h] = fmaxf(mm2[HPB + h], v.hi);
                    }
                }
                wave_reduce_n<2 * HPB>(mm2, OpMax(), -INFINITY);
                mn = -mm2[0];
                mx = mm2[HPB];
#pragma unroll
                for (int h = 1; h < HPB; ++h) { mn = hl == h ? -mm2[h] : mn; mx = hl == h ? mm2[HPB + h] : mx; }
                }
            }
            // Up to here minima and maxima are in grid steps before the zero-point, as the logits stay; the calibration takes
            // the logits themselves (all chunks of a unit have the same step and zero-point sum: the same query and statistics).
            // Every lane works out its own head's.
            const float step = qsz[2 * hl], zs = qsz[2 * hl + 1];
            // The range is that of the grid steps: the difference of the two logits carries their roundings, and a slope from it does
            // not fit the steps where the logits differ by little beside their size.
            const float range = (mx - mn) * step;
            float slope = 1.0f, tmin = __builtin_fmaf(mn, step, -zs);
            if (g.calib) {
                tmin += g.off_min;
                // (the hardware reciprocal, one unit in the last place: far inside the tolerance of the map)
                slope = (range + (g.off_max - g.off_min)) * __builtin_amdgcn_rcpf(range + 1e-8f);
            }
            // e = exp(x - M) with x = (w - mn) * slope + tmin, as exp2((w - peak) * ea): `peak` is the logit whose x is M, so no
            // weight is above 1 - which the fixed-point weights rely on - however large the logits are or far from 0 they lie
            // (a constant that takes M back is off by M's own rounding), and a degenerate logit range, whose slope is
            // ~1e8, meets the exact zero of (w - peak).
            float eal, pkl;
            if (masked) {
                const float sl = slope * step;
                float top = -INFINITY;
#pragma unroll
                for (int rd = 0; rd < REGL; ++rd) {
                    if (wt0 + rd * kNT < n) {
                        float l[4];
                        get_logits(rd, l);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float mv = rd < kMaskAhead ? mask_v[rd < kMaskAhead ? rd : 0][j] : mask_img[min(wt0 + rd * kNT + 16 * j + (lane & 15), n - 1)];
                            l[j] = (l[j] - mn) * sl + tmin + mv;
                            top = fmaxf(top, l[j]);
                        }
                        put_logits(rd, l);
                    }
                }
                const int kt = row_max_key(float_key(top));
                int* redi = reinterpret_cast<int*>(red + 2 * HPB);
                if ((lane & 15) == 0 && (lane >> 4) < HPB)
                    __hip_atomic_fetch_max(redi + hl, kt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __syncthreads();
                m_img = key_float(redi[hl]);
                eal = kLog2e;
                pkl = m_img;
                if (m_img == -INFINITY) { eal = 1.f; pkl = INFINITY; }   // every position masked out
            } else {
                m_img = fmaxf(tmin, range * slope + tmin);
                eal = slope * kLog2e * step;
                pkl = slope < 0.f ? mn : mx;
                if (m_img == -INFINITY) { eal = 1.f; pkl = INFINITY; }
            }
            float lsum = 0.f;
            I4 acc[BITS == 2 && !VTOK ? 9 : 8];
            if (VTOK || wt0 >= n) {   // (else the first round starts them)
#pragma unroll
                for (int i = 0; i < (BITS == 2 && !VTOK ? 9 : 8); ++i) acc[i] = I4{0, 0, 0, 0};
            }
            unsigned char* et = regA + wv * L::MXT;
            constexpr int KV = kVF / BITS;   // rounds of packed V rows in flight
            U2 ssc[VTOK ? KV : 1], smin[VTOK ? KV : 1];   // VTOK: the statistics of the lane's own tokens, as many rounds ahead
            float cm[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (VTOK) {
#pragma unroll
                for (int r = 0; r < KV; ++r) {
                    ssc[r] = ts[r];
                    smin[r] = vmp[min(tid + r * kNT, n - 1)];
                }
            }
            if constexpr (!kDotWindow) load_res(kb, 0, rk);   // the first tile of the window: its K rows arrive during the packed V rows
            phase_priority(std::integral_constant<int, 3>{});
            auto weights = [&](int rd, float* e) {   // of round rd's tile
                const int tw = wt0 + rd * kNT;
                get_logits(rd, e);
#pragma unroll
                for (int j = 0; j < 4; ++j) e[j] = __builtin_amdgcn_exp2f((e[j] - pkl) * eal);
                if (tw + kWave > n) {   // the chunk's last tile: what is past the end weighs nothing
#pragma unroll
                    for (int j = 0; j < 4; ++j) e[j] = tw + 16 * j + (lane & 15) < n ? e[j] : 0.f;
                }
            };
            float vpw[4] = {0.f, 0.f, 0.f, 0.f};   // VTOK: the grids of the lane's head
            if constexpr (VTOK) {
                uint32_t top[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int rd = 0; rd < REGL; ++rd) {
                    if (wt0 + rd * kNT < n) {
                        weights(rd, lx[rd]);   // (in place: the logits are not needed any more)
                        token_tops<DT>(lx[rd], ts[rd], top);
                    }
                }
#pragma unroll
                for (int gi = 0; gi < 4; ++gi) {
                    const int bits = row_max_key(static_cast<int>(top[gi] & 0x7fffffffu));
                    const int e = max((bits >> 23) - 126, -90);   // the largest lies in [2^(e-1), 2^e)
                    // an infinity or a NaN among them makes the head's sums of the group NaN
                    vpw[gi] = bits >= 0x7f800000 ? __builtin_nanf("") : __builtin_bit_cast(float, (30 - e + 127) << 23);
                }
            }
#pragma unroll
            for (int rd = 0; rd < REGL; ++rd) {
                if (wt0 + rd * kNT >= n) break;
                float e[4];
                if constexpr (VTOK) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) e[j] = lx[rd][j];
                } else {
                    weights(rd, e);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) lsum += e[j];
                if constexpr (VTOK) {
                    const U2 a = ssc[rd % KV], m = smin[rd % KV];
                    matrix_values_token<BITS, DT>(et, e, vc + (rd % KV) * BITS, U4{a.x, m.x, a.y, m.y}, vpw, cm, acc);
                } else {
                    matrix_values<BITS>(et, e, vc + (rd % KV) * BITS, acc, rd == 0);
                }
                __builtin_amdgcn_sched_barrier(0);   // one round at a time: interleaved, they do not fit the registers
                if (rd + KV < REGL) {
#pragma unroll
                    for (int i = 0; i < BITS; ++i) request_v((rd % KV) * BITS + i, (rd + KV) * BITS + i);
                    if constexpr (VTOK) {
                        ssc[rd % KV] = vsp[min(tid + (rd + KV) * kNT, n - 1)];
                        smin[rd % KV] = vmp[min(tid + (rd + KV) * kNT, n - 1)];
                    }
                }
            }
            phase_priority(std::integral_constant<int, 4>{});
            if constexpr (kDotWindow) load_res(kb, 0, rk);
            else load_res(vbp, 0, rv);   // ... its V rows: in flight during the fold and the window's logits
            float* lpart = fx + L::F_PRES;   // the waves' sums of e (not in `red`, which a slower wave may still read)
            lsum = row_reduce(lsum, OpSum(), 0.f);
            constexpr int kParts = VTOK ? 5 : 1;     // VTOK: and of e * minimum per channel group
            if constexpr (VTOK) {
#pragma unroll
                for (int gi = 0; gi < 4; ++gi) cm[gi] = row_reduce(cm[gi], OpSum(), 0.f);
            }
            if ((lane & 15) == 0 && (lane >> 4) < HPB) {
                lpart[wv * kParts * HPB + hl] = lsum;
                if constexpr (VTOK) {
#pragma unroll
                    for (int gi = 0; gi < 4; ++gi) lpart[(wv * kParts + 1 + gi) * HPB + hl] = cm[gi];
                }
            }
            // a wave's sums, [head][channel], take the place of its own tile: nobody else reads or writes there
            static_assert(HPB * kD * 4 <= L::MXT, "a wave's sums fit its tile");
            const float* redv = reinterpret_cast<const float*>(regA);
            if ((lane >> 4) < HPB) {
                float* o = reinterpret_cast<float*>(et) + hl * kD;   // (channels in the order channel ^ 16 * head: the fold reads them without bank conflicts)
                if constexpr (VTOK) matrix_fold_token<BITS>(acc, vpw, o, lane & 15, hl << 4);
                else matrix_fold<BITS>(acc, o, lane & 15, hl << 4);
            }
            __syncthreads();
            if (owns) {
                const int h = hl, d = od;
                float a = 0.f, lh = 0.f;
#pragma unroll
                for (int w = 0; w < kNW; ++w) { a += redv[w * (L::MXT / 4) + h * kD + (d ^ (h << 4))]; lh += lpart[w * kParts * HPB + h]; }
                if constexpr (VTOK) {
                    float cmin = 0.f;
#pragma unroll
                    for (int w = 0; w < kNW; ++w) cmin += lpart[(w * kParts + 1 + (d >> 5)) * HPB + h];
                    o_img = a + cmin;
                } else {
                    o_img = fx[L::F_VSZ + d] * (a - fx[L::F_VSZ + kD + d] * lh);
                }
                if (d == 0) stat[4 * HPB + h] = lh;
            }
            // (no barrier: what was read here - the sums, the waves' sums of e - is next written behind barriers of the
            // window, and `stat` is read behind the one of the merge)
        }

        if (n == 0) {
            load_res(kb, 0, rk);
            if constexpr (!kDotWindow) load_res(vbp, 0, rv);
        }
        CQ_PHASE(8);   // fold of the packed part
        // ---- phase 6: full-precision residual rows, online softmax.  Runs last: its first
        // tile is requested when the packed-V phase ends and arrives during that phase's fold.
#pragma unroll
        for (int h = 0; h < HPB; ++h) {
            if (tid == h) {
                stat[HPB + h] = -INFINITY;
                stat[2 * HPB + h] = 0.f;
            }
        }
        if (do_res) {
            if constexpr (kDotWindow) {
                float m_run = -INFINITY, l_run = 0.f;
                float* sres = fx + L::F_SRES;
                float* pres = fx + L::F_PRES;
                // raw 16-bit q, [head][kD], read per head as two 16-byte LDS loads
                const uint4* q128 = reinterpret_cast<const uint4*>(fx + L::F_QRAW);
                float accv[2][HPB];   // the lane's channel pair
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int h = 0; h < HPB; ++h) accv[k][h] = 0.f;

                for (int r0 = 0; r0 < R; r0 += kResTile) {
                    const bool more = r0 + kResTile < R;
                    const int r = r0 + krow;
                    uint32_t vw[RPW];   // the tile's value words, a channel pair of the wave's rows: in flight while its logits and weights are worked out
#pragma unroll
                    for (int i = 0; i < RPW; ++i) vw[i] = *reinterpret_cast<const uint32_t*>(vbp + min(r0 + wvu * RPW + i, last_r) * rs_r + 2 * lane);
                    float dot[HPB];
#pragma unroll
                    for (int h = NH; h < HPB; ++h) dot[h] = 0.f;
#pragma unroll
                    for (int h = 0; h < NH; ++h) {
                        float a = 0.f;
#pragma unroll
                        for (int i = 0; i < NKP; ++i) {
                            const uint4 qa = q128[h * (kD / 8) + i * LPR + lq];
                            a = dot2<DT>(qa.x, rk[i].x, a); a = dot2<DT>(qa.y, rk[i].y, a);
                            a = dot2<DT>(qa.z, rk[i].z, a); a = dot2<DT>(qa.w, rk[i].w, a);
                        }
                        dot[h] = (LPR == 4 ? quad_reduce(a, OpSum(), 0.f) : oct_reduce(a, OpSum(), 0.f)) * inv_sqrt_d;
                    }
                    if (more) load_res(kb, r0 + kResTile, rk);   // next tile's K slice, in place
                    if (lq == 0) {
                        float mv = 0.f;
                        if (masked && r < R) mv = mask_win[r < g.S ? r : g.T + r];
#pragma unroll
                        for (int h = 0; h < HPB; ++h) sres[krow * HPB + h] = (r < R) ? dot[h] + mv : -INFINITY;
                    }
                    __syncthreads();
                    if (wv < NH) {   // wave h keeps the running softmax state of head h
                        const int h = wv;
                        constexpr int kRL = kResTile / kWave;   // tile rows per lane
                        float sv[kRL], smax = -INFINITY;
#pragma unroll
                        for (int i = 0; i < kRL; ++i) {
                            sv[i] = sres[(lane + i * kWave) * HPB + h];
                            smax = fmaxf(smax, sv[i]);
                        }
                        const float mnew = fmaxf(m_run, wave_max(smax));
                        const bool dead = (mnew == -INFINITY);
                        float psum = 0.f;
#pragma unroll
                        for (int i = 0; i < kRL; ++i) {
                            const float pi = dead ? 0.f : __expf(sv[i] - mnew);
                            pres[(lane + i * kWave) * HPB + h] = pi;
                            psum += pi;
                        }
                        const float al = dead ? 1.0f : __expf(m_run - mnew);
                        l_run = l_run * al + wave_sum(psum);
                        m_run = mnew;
                        if (lane == 0) { stat[h] = al; stat[HPB + h] = m_run; stat[2 * HPB + h] = l_run; }
                    }
                    __syncthreads();
                    if (r0 > 0) {
#pragma unroll
                        for (int h = 0; h < NH; ++h) {
                            const float al = stat[h];
                            accv[0][h] *= al;
                            accv[1][h] *= al;
                        }
                    }
#pragma unroll
                    for (int i = 0; i < RPW; ++i) {
                        const float f0 = Cvt<DT>::lo(vw[i]), f1 = Cvt<DT>::hi(vw[i]);
                        const Vec<HPB> p = reinterpret_cast<const Vec<HPB>*>(pres)[wvu * RPW + i];   // the row's weights (0 past R), one address per wave
#pragma unroll
                        for (int h = 0; h < NH; ++h) {
                            accv[0][h] = __builtin_fmaf(p.v[h], f0, accv[0][h]);
                            accv[1][h] = __builtin_fmaf(p.v[h], f1, accv[1][h]);
                        }
                    }
                }
                // (regA was last read by the packed part's sum, behind which lie the tiles' barriers)
                float* red2 = reinterpret_cast<float*>(regA);  // [wave][head][kD]: the fold reads consecutive words
#pragma unroll
                for (int h = 0; h < HPB; ++h) {
                    Vec<2> a2;
                    a2.v[0] = accv[0][h]; a2.v[1] = accv[1][h];
                    *reinterpret_cast<Vec<2>*>(red2 + (wv * HPB + h) * kD + 2 * lane) = a2;
                }
                __syncthreads();
                if (owns) {
#pragma unroll
                    for (int w = 0; w < kNW; ++w) o_res += red2[(w * HPB + hl) * kD + od];
                }
            } else {
                float m_run = -INFINITY, l_run = 0.f;
                float* sres = fx + L::F_SRES;
                unsigned char* tile_rows = reinterpret_cast<unsigned char*>(parked);
                unsigned char* wrows = tile_rows + wv * 1024;   // a wave's rows: four to 1 KB, NT * 16 apart
                auto row_piece = [&](int row, int piece) { return (row >> 2) * (NT * 16) + (row & 3) * 256 + ((piece ^ row) << 4); };
                auto park_rows = [&](const U4* v) {
#pragma unroll
                    for (int i = 0; i < NKP; ++i) *reinterpret_cast<U4*>(wrows + row_piece(lane / LPR, i * LPR + lq)) = v[i];
                };
                const int x = lane & 15, kg = lane >> 4;
                const unsigned char* q16 = smem + L::kRegionA + L::F_QRAW * 4 + min(x >> 2, HPB - 1) * (kD * 2) + kg * 16;   // left operand: rows 4 h .. 4 h + 3 are head h
                constexpr int kPB = 272;   // bytes of a row of weight parts: 128 window rows and 16 bytes against bank conflicts
                unsigned char* parts = regA;    // [4 * head + part][window row], read by the fold above before the tile's first barrier
                static_assert(16 * kPB <= L::kRegionA, "the weights' parts fit region A");
                F4 racc = {0.f, 0.f, 0.f, 0.f};

                for (int r0 = 0; r0 < R; r0 += kResTile) {
                    const bool more = r0 + kResTile < R;
                    if (r0 > 0) {
                        if constexpr (NT == 1024) {
                            const int other = (r0 / kResTile) % 2 ? kWindowTile : -kWindowTile;
                            tile_rows += other;
                            wrows += other;
                        } else {
                            __syncthreads();   // (the values of the tile before are read)
                        }
                    }
                    park_rows(rk);
                    if (more) load_res(kb, r0 + kResTile, rk);
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    F4 dot = {0.f, 0.f, 0.f, 0.f};
                    const int xr = x % RPW;   // (waves of eight rows: columns 8 .. 15 repeat them)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        dot = mfma16<DT>(*reinterpret_cast<const U4*>(q16 + 64 * s), *reinterpret_cast<const U4*>(wrows + row_piece(xr, 4 * s + kg)), dot);
                    if (x < RPW && kg < HPB) {
                        const int r = r0 + wv * RPW + x;
                        float w = dot[0] * inv_sqrt_d;
                        if (masked && r < R) w += r0 == 0 ? mask_w : mask_win[r < g.S ? r : g.T + r];
                        sres[(wv * RPW + x) * HPB + kg] = r < R ? w : -INFINITY;
                    }
                    __syncthreads();
                    if (wv < NH) {   // wave h keeps the running softmax state of head h; a lane two neighbouring rows
                        const int h = wv;
                        const float s0 = sres[2 * lane * HPB + h], s1 = sres[(2 * lane + 1) * HPB + h];
                        const float mnew = fmaxf(m_run, wave_max(fmaxf(s0, s1)));
                        const bool dead = (mnew == -INFINITY);
                        const float p0 = dead ? 0.f : __expf(s0 - mnew), p1 = dead ? 0.f : __expf(s1 - mnew);
                        uint32_t w0[3], w1[3];
                        split_weight<DT>(p0, w0);
                        split_weight<DT>(p1, w1);
#pragma unroll
                        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint32_t*>(parts + (4 * h + i) * kPB + 4 * lane) = w0[i] | (w1[i] << 16);
                        const float al = dead ? 1.0f : __expf(m_run - mnew);
                        l_run = l_run * al + wave_sum(p0 + p1);
                        m_run = mnew;
                        if (lane == 0) { stat[h] = al; stat[HPB + h] = m_run; stat[2 * HPB + h] = l_run; }
                    }
                    park_rows(rv);   // (over the wave's K rows; behind the weights, so that these do not wait for the values)
                    if (more) load_res(vbp, r0 + kResTile, rv);
                    __syncthreads();
                    if (wv < 8) {   // 16 channels of all heads: a wave each
                        if (r0 > 0) racc *= stat[hl];
#pragma unroll
                        for (int s = 0; s < kResTile / 32; ++s) {
                            const U4 w = *reinterpret_cast<const U4*>(parts + x * kPB + 64 * s + 16 * kg);
                            U4 v;
#pragma unroll
                            for (int t = 0; t < 2; ++t) {   // rows 32 s + 8 kg + 4 t + 0 .. 3: column x of four rows
                                const int row = (8 * kg + 4 * t + (x >> 2)) % RPW;
                                const unsigned char* o = tile_rows + ((32 * s + 8 * kg) / RPW) * 1024 +
                                                         row_piece(row, 2 * wv + ((x >> 1) & 1)) + (x & 1) * 8;
                                const U2 c = __builtin_bit_cast(U2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) S4*)(o)));
                                v[2 * t] = c.x; v[2 * t + 1] = c.y;
                            }
                            racc = mfma16<DT>(w, v, racc);
                        }
                    }
                }
                o_res = racc[0];
                // (an infinite sum stays one: 0, a lower part's, times an infinite value would make it a NaN)
                if (__builtin_fabsf(o_res) != INFINITY) o_res += kPartScale<DT> * (racc[1] + kPartScale<DT> * racc[2]);
                o_res *= kPartUnit<DT>;
            }
        }

        if (speaks) {
            stat[3 * HPB + hl] = m_img;
            if (n == 0) stat[4 * HPB + hl] = 0.f;
        }
        CQ_PHASE(9);   // residual window
        // ---- phase 7: merge / write ---------------------------------------------------------
        __syncthreads();
        if (owns && hl < nh) {
            const int h = hl, d = od;
            const float mr = stat[HPB + h], lr = stat[2 * HPB + h];
            const float mi = stat[3 * HPB + h], li = stat[4 * HPB + h];
            const int64_t row = static_cast<int64_t>(b) * g.Hq + hq0 + h;
            if constexpr (!CHUNKED) {
                const float mf = fmaxf(mi, mr);
                const float wi = (mi == -INFINITY) ? 0.f : __expf(mi - mf);
                const float wr = (mr == -INFINITY) ? 0.f : __expf(mr - mf);
                const float num = o_img * wi + o_res * wr;
                const float den = li * wi + lr * wr;
                store_elem<DT>(g.out, row * kD + d, num * __builtin_amdgcn_rcpf(den));
            } else {
                float* p = g.part + (row * g.nx + split) * (kD + 2);
                const bool is_img = split < g.nsplit;
                if (d == 0) { publish(p, is_img ? mi : mr); publish(p + 1, is_img ? li : lr); }
                publish(p + 2 + d, is_img ? o_img : o_res);
            }
        }
        if constexpr (CHUNKED) {
            // The unit's chunks (and its residual unit) each leave an (m, l, acc) partial.  Two launches: the workgroup that
            // finds all the others' already counted combines them; one launch: the first chunk's, when the others have
            // announced theirs.  The partials are device-scope atomic stores
            // (written through to the level all compute units share, so no cache has to be written back as a
            // whole): every thread waits for its own stores to complete, the barrier collects the workgroup,
            // then one thread counts or announces.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            int* last = reinterpret_cast<int*>(red);
            if (g.fused) {
                if (split != 0) {
                    if (tid == 0) announce<HPB>(g, unit, split);
                    return;
                }
                if (wv == 0) {
                    const bool ok = others_done(g, unit, lane);
                    if (lane == 0) {
                        *last = ok ? 1 : 0;
                        if (!ok && g.status) __hip_atomic_store(g.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
                }
            } else if (tid == 0) {
                *last = __hip_atomic_fetch_add(g.cnt + unit, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g.nx - 1;
            }
            __syncthreads();
            if (*last) {
                // the reader: one acquire drops this compute unit's and this die's cached copies of what other
                // dies wrote, after which ordinary loads (issued together, unlike atomic ones) see the partials
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                if (tid < nh * kD) {
                    const int h = tid / kD, d = tid % kD;
                    const int64_t row = static_cast<int64_t>(b) * g.Hq + hq0 + h;
                    const float* p = g.part + row * g.nx * (kD + 2);
                    // eight partials at a time, their loads in flight together; running (m, num, den)
                    float m = -INFINITY, num = 0.f, den = 0.f;
                    for (int s0 = 0; s0 < g.nx; s0 += 8) {
                        float ms[8], ls[8], as[8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            const float* q = p + min(s0 + k, g.nx - 1) * (kD + 2);
                            ms[k] = q[0]; ls[k] = q[1]; as[k] = q[2 + d];
                        }
                        float mb = m;
#pragma unroll
                        for (int k = 0; k < 8; ++k) mb = fmaxf(mb, (s0 + k < g.nx) ? ms[k] : -INFINITY);
                        const float keep = (m == -INFINITY) ? 0.f : __expf(m - mb);
                        num *= keep; den *= keep;
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            const float w = (s0 + k < g.nx && ms[k] != -INFINITY) ? __expf(ms[k] - mb) : 0.f;
                            den += ls[k] * w;
                            num += as[k] * w;
                        }
                        m = mb;
                    }
                    store_elem<DT>(g.out, row * kD + d, num / den);
                }
                // every other workgroup of the unit is past the hand-over words
                if (g.fused) clear_handover<HPB>(g, unit, tid, kNT);
            }
        }
    }
}

// The min/max launch of a two-launch chunked step: no residual unit.
static inline DecodeGeom minmax_geometry(const DecodeGeom& g) {
    DecodeGeom g1 = g;
    g1.nx = g.nsplit;
    g1.d_nx.set(static_cast<uint32_t>(g.nsplit));
    return g1;
}

}  // namespace cq
