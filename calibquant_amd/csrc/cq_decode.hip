// Host side of the fused decode attention step (kernels: cq_decode_kernel.h): plans, launches, entry points.
#include "cq_decode_kernel.h"

#include <atomic>
#include <cstdlib>

#ifdef CQ_PHASE_STOPS
#include "cq_decode_matrix.h"
#endif

namespace cq {

// Launches the matrix-core form (one source file per storage type: cq_decode_matrix_*.hip).
template <typename DT>
int launch_matrix(const DecodeGeom& g, int bits, int hpb, int nh, int nt, unsigned units, hipStream_t st);
// ... with per-token values (cq_decode_matrix_token_*.hip)
template <typename DT>
int launch_matrix_token(const DecodeGeom& g, int bits, int hpb, int nt, unsigned units, hipStream_t st);

// ---- the chunked step in one launch: host side ------------------------------------------------------
// A word of pinned host memory per device that a workgroup sets when it gives up waiting for the other
// chunks of its unit (allocated once, at the first such call on the device; never freed).  The next chunked
// call on that device finds it set, reports CQ_ERR_LAUNCH once and the process goes on with two launches.
constexpr int kMaxDevices = 64;
static std::atomic<int*> g_status[kMaxDevices];
static std::atomic<bool> g_fused_off{false};      // set by a give-up; cleared by cq_decode_attn_wait_polls
static std::atomic<bool> g_fused_wanted{true};    // cq_decode_attn_single_launch
static std::atomic<uint32_t> g_epoch{0x5eed0000u};
static std::atomic<int> g_spin_limit{1 << 18};   // polls of about a microsecond each

// Compute units of the current device (a partitioned device reports its own share), asked once per
// process; kDefaultUnits when there is no device to ask (a host that only plans).
static int pair_units() {
    static std::atomic<int> cached{0};
    int n = cached.load(std::memory_order_relaxed);
    if (n > 0) return n;
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu < 1) {
        (void)hipGetLastError();   // not an error of the caller's
        cu = kDefaultUnits;
    }
    cached.store(cu, std::memory_order_relaxed);
    return cu;
}

// head groups per kv head; the last one may be partly padding (its spare heads repeat its last query head
// and write nothing)
static inline int ngroups(int G, int hpb) { return (G + hpb - 1) / hpb; }

struct Plan {
    int hpb, nh, nt, nsplit, chunk, nx;   // hpb: heads an entry is wide; nh: heads a unit serves
    bool fused;   // chunked step in one launch: every chunk's workgroup fits the device at once
    size_t ws_mm, ws_part, ws_cnt;   // chunked launch: min / max, partials, counters
};

// units of nh heads (entries hpb wide) in workgroups of nt threads, chunks of at most maxc tokens
static void plan_for(const cq_decode_args* a, Plan* p, int hpb, int nh, int nt, int maxc) {
    const int G = a->Hq / a->Hkv;
    const int64_t units = static_cast<int64_t>(a->B) * a->Hkv * ngroups(G, nh);
    int nsplit = 1;
    if (a->T > 0) {
        const int need = (a->T + maxc - 1) / maxc;
        nsplit = need;
        if (a->force_splits > 0) {
            nsplit = a->force_splits > need ? a->force_splits : need;
        } else if (units < 192 && need > 1) {
            // too few units to fill the device and T does not fit one unit anyway: more, smaller chunks.
            // (A T that fits one unit is never chunked: the min/max launch's second pass over the packed
            // K rows and the merge cost more than the idle compute units, at any batch size.)
            int64_t want = (512 + units - 1) / units;
            int64_t most = a->T / 1024 > 1 ? a->T / 1024 : 1;
            if (want > most) want = most;
            if (want > nsplit) nsplit = static_cast<int>(want);
        }
    }
    int chunk = a->T > 0 ? ((a->T + nsplit - 1) / nsplit + 63) / 64 * 64 : 64;
    if (chunk > maxc) chunk = maxc;
    nsplit = a->T > 0 ? (a->T + chunk - 1) / chunk : 1;
    p->hpb = hpb;
    p->nh = nh;
    p->nt = nt;
    p->nsplit = nsplit;
    p->chunk = chunk;
    p->nx = nsplit + ((nsplit > 1 && a->R > 0) ? 1 : 0);
    const size_t rows = static_cast<size_t>(a->B) * a->Hq;
    p->ws_mm = nsplit > 1 ? ((rows * nsplit * 2 * sizeof(float) + 255) / 256 * 256) : 0;
    p->ws_part = nsplit > 1 ? (rows * p->nx * (kD + 2) * sizeof(float) + 255) / 256 * 256 : 0;
    // counters: [unit] partials written (one launch: the window's announcement), then the min / max records of that form
    p->ws_cnt = nsplit > 1 ? (static_cast<size_t>(units) * sizeof(unsigned long long) + 255) / 256 * 256 +
                                 static_cast<size_t>(units) * hpb * nsplit * 16 : 0;
    p->fused = false;
}

static int make_plan(const cq_decode_args* a, Plan* p) {
    if (!a) return CQ_ERR_NULL;
    const int kPairUnits = pair_units();
    if (a->dtype != CQ_BF16 && a->dtype != CQ_FP16) return CQ_ERR_DTYPE;
    if (a->bits != 1 && a->bits != 2) return CQ_ERR_UNSUPPORTED;
    if (a->D != kD) return CQ_ERR_UNSUPPORTED;
    if (a->B < 1 || a->Hq < 1 || a->Hkv < 1 || a->Hq % a->Hkv) return CQ_ERR_SHAPE;
    if (a->T < 0 || a->R < 0 || (a->T == 0 && a->R == 0)) return CQ_ERR_SHAPE;
    if (a->sprompt_len < 0 || a->sprompt_len > a->R) return CQ_ERR_SHAPE;
    const int G = a->Hq / a->Hkv;
    if (a->v_mode != CQ_V_PER_CHANNEL && a->v_mode != CQ_V_PER_TOKEN) return CQ_ERR_UNSUPPORTED;
    const bool vtok = a->v_mode == CQ_V_PER_TOKEN;
    // heads a unit with four-wide entries serves: three when that divides the group exactly and four does not
    // (G = 3, 6, 9: exact units instead of a padded last one; per-channel values only)
    const int nh4 = (!vtok && G % 3 == 0 && G % 4 != 0) ? 3 : 4;
    auto plan = [&](Plan* o, int hpb, int nh) { plan_for(a, o, hpb, nh, 1024, plan_chunk(a->bits, vtok, hpb)); };
    // G = 3, 5, 6, 7, ...: units of four heads with the last one partly padding (two units per kv head at
    // G = 6) do less work than units of two heads or one (three or six of them, each walking all the packed rows).
    // Per-token values at 2 bits: two heads per unit, padded for odd G (there is no form with four).
    if (vtok && a->bits == 2) plan(p, G >= 2 ? 2 : 1, G >= 2 ? 2 : 1);
    else if (G > 2) plan(p, 4, nh4);
    else plan(p, G, G);
    if (!vtok && a->force_splits == 0 && p->hpb >= 2) {
        // Four heads per unit at 1 bit, enough units to fill the device, and T beyond the chunk: the longer chunk may
        // still hold all T tokens in one launch, which saves the min/max launch's second pass over the packed K rows.
        const int64_t units = static_cast<int64_t>(a->B) * a->Hkv * ngroups(G, p->nh);
        Plan q;
        if (a->bits == 1 && p->hpb == 4 && p->nsplit > 1 && units >= kPairUnits * 3 / 4) {
            plan_for(a, &q, 4, nh4, 1024, kPlanLong);
            if (q.nsplit == 1) *p = q;
        }
        // More units than compute units: 512-thread workgroups, two resident per compute unit, need fewer
        // instructions per unit than one 1024-thread workgroup after the other (half as many waves pay
        // the per-wave set-up, reductions and folds).  Single launch: only if their chunk also holds all T tokens.
        // Chunked launch (four heads per unit): the chunks are units of their own.
        if (p->hpb == 4 || a->bits == 1) {
            plan_for(a, &q, p->hpb, p->nh, 512, p->hpb == 4 ? kPlanPair4 : kPlanPair2);
            const bool single = p->nsplit == 1 && q.nsplit == 1 && units > kPairUnits;
            const bool chunked = p->hpb == 4 && p->nsplit > 1 && q.nsplit > 1 && units * q.nsplit > kPairUnits;
            if (single || chunked) *p = q;
        }
    }
    // A handful of units leave most compute units idle, and a launch then lasts as long as one unit: with one head to a unit
    // it is a shorter chain, and there are compute units for four times as many.  us from a recorded graph, one / two / four heads a unit, 32 / 8 heads:
    // 2 x 700 + 60 6.50 / 6.77 / 6.78, 2 x 3 328 + 128 9.50 / 9.63 / 9.60, 8 x 3 328 + 128 10.30 / 9.92 / 9.75, 10 x 3 328 + 128 18.1 / 10.1 / 9.8.
    // (Two heads from 33 to 64 units of four: within 2 % of four heads either way.  The line is from the look-up form: 15.5 for 18.8.)
    if (a->force_splits == 0 && p->nsplit == 1 && p->hpb == 4) {
        const int64_t u4 = static_cast<int64_t>(a->B) * a->Hkv * ngroups(G, p->nh);
        const int h = u4 <= 32 ? 1 : (u4 <= 64 && G % 2 == 0) ? 2 : 4;
        Plan q = *p;
        if (h < 4) plan(&q, h, h);
        if (q.nsplit == 1) *p = q;
    }
    const int64_t blocks = static_cast<int64_t>(a->B) * a->Hkv * ngroups(G, p->nh) * p->nx;
    if (blocks > 0x7fffffff) return CQ_ERR_SHAPE;
    // Chunked, and every chunk's workgroup resident at once (two 512-thread workgroups per compute unit, one of
    // 1024): one launch, the chunks exchange their min / max inside it and keep their logits - no second read of
    // the packed K rows, no logits buffer.  (The residual units wait for nobody and make room as they end.)
    if (p->nsplit > 1) {
        const int64_t waiting = static_cast<int64_t>(a->B) * a->Hkv * ngroups(G, p->nh) * p->nsplit;
        const int64_t room = static_cast<int64_t>(kPairUnits) * (p->nt == 512 && launch_lds(a->bits, vtok, p->hpb, p->nt) + parked_lds(vtok, p->nt, launch_rounds(vtok, p->hpb, p->nt, p->chunk)) <= kLdsMax / 2 ? 2 : 1);
        // (one lane per chunk polls)
        if (waiting <= room && p->nsplit <= 64 && g_fused_wanted.load(std::memory_order_relaxed)) p->fused = true;
    }
    return CQ_OK;
}

// The geometry's derived fields for units of nh heads in workgroups of nt threads.
static DecodeGeom unit_geometry(const DecodeGeom& g, int nh, int nt) {
    DecodeGeom gm = g;
    gm.G = g.Hq / g.Hkv;
    const int64_t blocks = static_cast<int64_t>(g.B) * g.Hkv * ngroups(gm.G, nh) * g.nx;
    gm.ncu = (nt == 512 && !g.fused && blocks <= 2 * static_cast<int64_t>(pair_units())) ? pair_units() : 0;
    gm.d_ng.set(static_cast<uint32_t>(ngroups(gm.G, nh)));
    gm.d_nx.set(static_cast<uint32_t>(g.nx));
    gm.d_hkv.set(static_cast<uint32_t>(g.Hkv));
    return gm;
}

template <typename DT>
static int dispatch(const DecodeGeom& g, const Plan& p, int bits, bool vtok, hipStream_t st) {
    DecodeGeom gm = unit_geometry(g, p.nh, p.nt);
    gm.stream = launch_streams(bits, vtok, p.hpb, p.nt, ngroups(gm.G, p.nh), g.nsplit, static_cast<int64_t>(g.B) * g.Hkv * g.T);
    const unsigned units = static_cast<unsigned>(g.B) * g.Hkv * ngroups(gm.G, p.nh);
#ifdef CQ_PHASE_STOPS
    if (vtok || !std::is_same<DT, BF16>::value || bits != 1 || p.hpb != 4 || p.nh != 4 || p.nt != 512 || g.nsplit > 1)
        return CQ_ERR_UNSUPPORTED;
    return launch_matrix_one<1, 4, BF16, false, 512, kRegPair, false, kNoExtras, 4>(gm, units, st);
#else
    return vtok ? launch_matrix_token<DT>(gm, bits, p.hpb, p.nt, units, st)
                : launch_matrix<DT>(gm, bits, p.hpb, p.nh, p.nt, units, st);
#endif
}

// ---- static scratch for callers that cannot allocate --------------------------------------------
// The chunked path's workspace (per-chunk logit min / max, flash-decoding partials) in a file-scope
// device array: every GPU the library runs on holds its own copy, at its own address, until the
// process ends.  Host code never uses the array's name as an address: the device address is asked
// for once per device (with that device current) and kept.
constexpr size_t kScratchBytes = static_cast<size_t>(8) << 20;
// (`used`: no kernel names the array - they get its address as an argument - so nothing else keeps it in the code object)
static __device__ __align__(256) __attribute__((used)) unsigned char scratch[kScratchBytes];

static std::atomic<void*> g_scratch_ptr[kMaxDevices];

static int scratch_address(void** out) {
    int dev = 0;
    CQ_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return CQ_ERR_UNSUPPORTED;
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        CQ_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return CQ_ERR_LAUNCH;
        g_scratch_ptr[dev].store(p, std::memory_order_release);   // every caller on this device gets the same address
    }
    *out = p;
    return CQ_OK;
}

static int* fused_status_word(hipStream_t st) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    int* p = g_status[dev].load(std::memory_order_acquire);
    if (p) return p;
    // not while the stream is being recorded: an allocation would end the recording
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
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
    if (!g_status[dev].compare_exchange_strong(expected, static_cast<int*>(raw), std::memory_order_acq_rel)) {
        (void)hipHostFree(raw);   // another host thread was first
        return expected;
    }
    return static_cast<int*>(raw);
}

static int decode_entry(const cq_decode_args* a, void* workspace, size_t workspace_bytes, bool static_scratch,
                        cq_stream_t stream) {
    Plan p;
    int rc = make_plan(a, &p);
    if (rc != CQ_OK) return rc;
    if (!a->q || !a->out) return CQ_ERR_NULL;
    if (a->T > 0 && (!a->codes_k || !a->codes_v || !a->k_scale || !a->k_zero || !a->v_scale || !a->v_zero))
        return CQ_ERR_NULL;
    if (a->R > 0 && (!a->k_res || !a->v_res)) return CQ_ERR_NULL;
    if (a->r_dev && a->mask) return CQ_ERR_UNSUPPORTED;   // the mask's length would have to follow the count
    if (a->r_dev && (reinterpret_cast<uintptr_t>(a->r_dev) & 3)) return CQ_ERR_ALIGN;
    if (a->T > 0 && (!aligned16(a->codes_k) || !aligned16(a->codes_v))) return CQ_ERR_ALIGN;
    if (a->R > 0 && (!aligned16(a->k_res) || !aligned16(a->v_res) || (a->res_stride_b % 8) ||
                     (a->res_stride_h % 8) || (a->res_stride_r % 8)))
        return CQ_ERR_ALIGN;
    const size_t need = p.ws_mm + p.ws_part + p.ws_cnt;
    // One launch when the plan allows it, the caller's own workspace is used (the static entry point allocates
    // nothing, not even the status word) and no earlier launch of this process gave up waiting.
    int* status = nullptr;
    bool fused = p.fused && !static_scratch && !g_fused_off.load(std::memory_order_relaxed);
    if (fused) {
        status = fused_status_word(static_cast<hipStream_t>(stream));
        if (!status) {
            fused = false;
        } else if (*static_cast<volatile int*>(status) != 0) {
            *static_cast<volatile int*>(status) = 0;
            g_fused_off.store(true, std::memory_order_relaxed);
            return CQ_ERR_LAUNCH;   // an earlier single-launch step did not complete: its output is not valid
        }
    }
    if (static_scratch) {
        if (need > kScratchBytes) return CQ_ERR_SCRATCH_LIMIT;
        workspace = nullptr;
        if (need) {
            rc = scratch_address(&workspace);
            if (rc != CQ_OK) return rc;
        }
    } else if (need && (!workspace || workspace_bytes < need || !aligned16(workspace))) {
        return CQ_ERR_WORKSPACE;
    }

    DecodeGeom g;
    g.q = a->q; g.ck = a->codes_k; g.cv = a->codes_v;
    g.ks = a->k_scale; g.kz = a->k_zero; g.vs = a->v_scale; g.vz = a->v_zero;
    g.kres = a->k_res; g.vres = a->v_res;
    g.rs_b = a->res_stride_b; g.rs_h = a->res_stride_h; g.rs_r = a->res_stride_r;
    g.mask = a->mask; g.mask_sb = a->mask_stride_b;
    g.r_dev = a->r_dev;
    g.out = a->out;
    g.mm = static_cast<float*>(workspace);
    g.part = need ? reinterpret_cast<float*>(static_cast<char*>(workspace) + p.ws_mm) : nullptr;
    g.cnt = need ? reinterpret_cast<int*>(static_cast<char*>(workspace) + p.ws_mm + p.ws_part) : nullptr;
    {
        const int G = a->Hq / a->Hkv;
        const size_t units = static_cast<size_t>(a->B) * a->Hkv * ngroups(G, p.nh);
        char* c0 = reinterpret_cast<char*>(g.cnt);
        g.done = reinterpret_cast<unsigned long long*>(workspace);
        g.done_res = reinterpret_cast<unsigned long long*>(c0);
        g.rec = reinterpret_cast<unsigned long long*>(c0 + (units * sizeof(unsigned long long) + 255) / 256 * 256);
    }
#ifdef CQ_PHASE_STOPS
    {
        const char* e = getenv("CQ_DECODE_PHASE_STOP");
        g.stop = e ? atoi(e) : -1;
    }
#endif
    g.fused = fused ? 1 : 0;
    g.status = status;
    g.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    uint32_t ep = g_epoch.fetch_add(1, std::memory_order_relaxed) + 1;
    g.epoch = ep ? ep : g_epoch.fetch_add(1, std::memory_order_relaxed) + 1;   // (0 is never an epoch)
    g.B = a->B; g.Hq = a->Hq; g.Hkv = a->Hkv; g.T = a->T; g.R = a->R; g.S = a->sprompt_len;
    g.nsplit = p.nsplit; g.chunk = p.chunk; g.nx = p.nx;
    g.calib = a->calibrate; g.off_max = a->calib_off_max; g.off_min = a->calib_off_min;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool vtok = a->v_mode == CQ_V_PER_TOKEN;
    if (a->dtype == CQ_BF16) return dispatch<BF16>(g, p, a->bits, vtok, st);
    return dispatch<FP16>(g, p, a->bits, vtok, st);
}

}  // namespace cq

extern "C" {

size_t cq_decode_attn_workspace(const cq_decode_args* args) {
    cq::Plan p;
    if (cq::make_plan(args, &p) != CQ_OK) return 0;
    return p.ws_mm + p.ws_part + p.ws_cnt;
}

int cq_decode_attn_single_launch(int enable) {
    const int before = cq::g_fused_wanted.load(std::memory_order_relaxed) ? 1 : 0;
    if (enable >= 0) cq::g_fused_wanted.store(enable != 0, std::memory_order_relaxed);
    return before;
}

int cq_decode_attn_gave_up(void) {
    for (int dev = 0; dev < cq::kMaxDevices; ++dev) {
        const int* p = cq::g_status[dev].load(std::memory_order_acquire);
        if (p && *static_cast<const volatile int*>(p) != 0) return 1;
    }
    return 0;
}

int cq_decode_attn_wait_polls(int polls) {
    const int before = cq::g_spin_limit.load(std::memory_order_relaxed);
    if (polls >= 0) {
        cq::g_spin_limit.store(polls, std::memory_order_relaxed);
        cq::g_fused_off.store(false, std::memory_order_relaxed);
    }
    return before;
}

int cq_decode_attn_plan(const cq_decode_args* args, cq_decode_plan* plan) {
    if (!plan) return CQ_ERR_NULL;
    cq::Plan p;
    const int rc = cq::make_plan(args, &p);
    if (rc != CQ_OK) return rc;
    plan->threads = p.nt;
    plan->heads_per_unit = p.nh;
    plan->chunks = p.nsplit;
    plan->chunk_tokens = args->T > 0 ? p.chunk : 0;
    plan->launches = (p.nsplit > 1 && !p.fused) ? 2 : 1;
    const bool vtok = args->v_mode == CQ_V_PER_TOKEN;
    plan->lds_bytes = cq::launch_lds(args->bits, vtok, p.hpb, p.nt);
    plan->register_logits = cq::launch_rounds(vtok, p.hpb, p.nt, p.chunk);
    return CQ_OK;
}

int cq_decode_attn(const cq_decode_args* a, cq_stream_t stream) {
    if (!a) return CQ_ERR_NULL;
    return cq::decode_entry(a, a->workspace, a->workspace_bytes, false, stream);
}

size_t cq_decode_attn_static_limit(void) { return cq::kScratchBytes; }

int cq_decode_attn_static(const cq_decode_args* a, cq_stream_t stream) {
    if (!a) return CQ_ERR_NULL;
    return cq::decode_entry(a, nullptr, 0, true, stream);
}

}  // extern "C"
