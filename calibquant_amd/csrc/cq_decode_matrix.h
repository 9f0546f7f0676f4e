// Launches of the matrix-core form of the decode step (kernel: cq_decode_kernel.h).
#pragma once
#include "cq_decode_kernel.h"

#include <atomic>

namespace cq {

template <int BITS, int HPB, typename DT, bool VTOK, int NT, int REGL, bool CHUNKED, Extras EXTRAS, int NH>
static int launch_matrix_one(const DecodeGeom& g, unsigned units, hipStream_t st) {
    constexpr int lds = Lay<BITS, HPB, VTOK, NT>::kLds;
    static_assert(lds <= 64 * 1024, "no raised dynamic-LDS limit needed");
    static_assert(lds + parked_lds(VTOK, NT, REGL) <= kLdsMax / (NT == 512 ? 2 : 1), "two 512-thread workgroups share a compute unit");
    static_assert(lds == launch_lds<BITS, VTOK, NT>(HPB), "the LDS that plans report");
    if (launch_rounds(VTOK, HPB, NT, g.chunk) != REGL || g.chunk > REGL * NT) return CQ_ERR_UNSUPPORTED;   // (a token too many would be left out of the sum)
    if constexpr (CHUNKED) {
        if (!g.fused) {
            const DecodeGeom g1 = minmax_geometry(g);   // (this launch never looks at values)
            constexpr int lds1 = Lay<BITS, HPB, false, NT>::kLds;
            hipLaunchKernelGGL((decode_kernel<BITS, HPB, DT, true, false, NT, REGL, true, kNoExtras, NH>),
                               dim3(units * g.nsplit), dim3(NT), lds1, st, g1);
            CQ_LAUNCH_CHECK();
        }
    }
    if constexpr (!CHUNKED && stream_form(BITS, VTOK, HPB, NT)) {
        if (g.stream) {
            hipLaunchKernelGGL((decode_kernel<BITS, HPB, DT, false, VTOK, NT, REGL, CHUNKED, EXTRAS, NH, true>), dim3(units * g.nx),
                               dim3(NT), lds, st, g);
            CQ_LAUNCH_CHECK();
            return CQ_OK;
        }
    }
    hipLaunchKernelGGL((decode_kernel<BITS, HPB, DT, false, VTOK, NT, REGL, CHUNKED, EXTRAS, NH>), dim3(units * g.nx),
                       dim3(NT), lds, st, g);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

// A chunked launch has two instantiations: with the mask, and with the row count (which may be absent).  All kernels keep within the 128
// registers, except chunked ones of sixteen rounds with a mask (4 to 32 spilled: two heads, or one at 2 bits) and the fp16 form of per-token values with
// two heads and eight rounds, chunked without a mask (4).
// SINGLE: no plan chunks such units.
template <int BITS, int HPB, typename DT, int NT, int REGL, int NH = HPB, bool VTOK = false, bool SINGLE = false>
static int launch_matrix_unit(const DecodeGeom& g, unsigned units, hipStream_t st) {
    if constexpr (SINGLE) { if (g.nsplit > 1) return CQ_ERR_UNSUPPORTED; }
    else if (g.nsplit > 1) return g.mask ? launch_matrix_one<BITS, HPB, DT, VTOK, NT, REGL, true, kMasked, NH>(g, units, st)
                                         : launch_matrix_one<BITS, HPB, DT, VTOK, NT, REGL, true, kDeviceRows, NH>(g, units, st);
    if (g.mask) return launch_matrix_one<BITS, HPB, DT, VTOK, NT, REGL, false, kMasked, NH>(g, units, st);
    if (g.r_dev) return launch_matrix_one<BITS, HPB, DT, VTOK, NT, REGL, false, kDeviceRows, NH>(g, units, st);
    return launch_matrix_one<BITS, HPB, DT, VTOK, NT, REGL, false, kNoExtras, NH>(g, units, st);
}

template <int BITS, typename DT>
static int launch_matrix_bits(const DecodeGeom& g, int hpb, int nh, int nt, unsigned units, hipStream_t st) {
    const bool most = launch_rounds(false, hpb, nt, g.chunk) == kRegMost;
    if (nt == 512) {
        if (hpb == 4 && nh == 3) return launch_matrix_unit<BITS, 4, DT, 512, kRegPair, 3>(g, units, st);
        if (hpb == 4) return launch_matrix_unit<BITS, 4, DT, 512, kRegPair>(g, units, st);
        if constexpr (BITS == 1) {   // (two bits: two heads per unit only where there are few units)
            if (hpb == 2) return most ? launch_matrix_unit<BITS, 2, DT, 512, kRegMost, 2, false, true>(g, units, st)
                                      : launch_matrix_unit<BITS, 2, DT, 512, kRegPair, 2, false, true>(g, units, st);
        }
        return CQ_ERR_UNSUPPORTED;
    }
    if (hpb == 4 && nh == 3) return launch_matrix_unit<BITS, 4, DT, 1024, kRegLong, 3>(g, units, st);
    if (hpb == 4) return launch_matrix_unit<BITS, 4, DT, 1024, kRegLong>(g, units, st);
    if (hpb == 2) return most ? launch_matrix_unit<BITS, 2, DT, 1024, kRegMost>(g, units, st)
                              : launch_matrix_unit<BITS, 2, DT, 1024, kRegLong>(g, units, st);
    return most ? launch_matrix_unit<BITS, 1, DT, 1024, kRegMost>(g, units, st)
                : launch_matrix_unit<BITS, 1, DT, 1024, kRegLong>(g, units, st);
}

// nt threads per workgroup, g.chunk tokens at most: the plan's (cq_decode.hip: make_plan)
template <typename DT>
int launch_matrix(const DecodeGeom& g, int bits, int hpb, int nh, int nt, unsigned units, hipStream_t st) {
    return bits == 1 ? launch_matrix_bits<1, DT>(g, hpb, nh, nt, units, st) : launch_matrix_bits<2, DT>(g, hpb, nh, nt, units, st);
}

// Per-token values: 1 024 threads, four heads at 1 bit at most, two at 2 bits.  Four rounds of logits for chunks of up to
// 4 096 tokens (the sixteen registers more of eight rounds do not fit beside the statistics of the values), eight above.
template <int BITS, int HPB, typename DT>
static int launch_token_unit(const DecodeGeom& g, unsigned units, hipStream_t st) {
    constexpr int most = plan_chunk(BITS, true, HPB);
    static_assert(most <= kRegPair * 1024, "the plan's chunks fit eight rounds");
    if (launch_rounds(true, HPB, 1024, g.chunk) == kRegTwoBit)
        return launch_matrix_unit<BITS, HPB, DT, 1024, kRegTwoBit, HPB, true>(g, units, st);
    if constexpr (most > kRegTwoBit * 1024) return launch_matrix_unit<BITS, HPB, DT, 1024, kRegPair, HPB, true>(g, units, st);
    return CQ_ERR_UNSUPPORTED;
}

template <typename DT>
int launch_matrix_token(const DecodeGeom& g, int bits, int hpb, int nt, unsigned units, hipStream_t st) {
    if (nt != 1024 || (bits == 2 && hpb == 4)) return CQ_ERR_UNSUPPORTED;
    if (bits == 2) return hpb == 2 ? launch_token_unit<2, 2, DT>(g, units, st) : launch_token_unit<2, 1, DT>(g, units, st);
    if (hpb == 4) return launch_token_unit<1, 4, DT>(g, units, st);
    return hpb == 2 ? launch_token_unit<1, 2, DT>(g, units, st) : launch_token_unit<1, 1, DT>(g, units, st);
}

}  // namespace cq
