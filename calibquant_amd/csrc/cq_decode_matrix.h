// Launches of the matrix-core form of the decode step (kernel: cq_decode_kernel.h, template flag MX).
#pragma once
#include "cq_decode_kernel.h"

#include <atomic>

namespace cq {

template <int BITS, int HPB, typename DT, int NT, int REGL, bool CHUNKED, bool EXTRAS, int NH>
static int launch_matrix_one(const DecodeGeom& g, unsigned units, hipStream_t st) {
    constexpr int lds = Lay<BITS, HPB, false, NT, REGL, true>::lds_bytes(0);
    static_assert(lds <= 64 * 1024, "no raised dynamic-LDS limit needed; two 512-thread workgroups share a compute unit");
    if constexpr (CHUNKED) {
        if (!g.fused) {
            const DecodeGeom g1 = minmax_geometry(g, 0);
            hipLaunchKernelGGL((decode_kernel<BITS, HPB, DT, true, false, NT, REGL, true, false, NH, true>),
                               dim3(units * g.nsplit), dim3(NT), lds, st, g1);
            CQ_LAUNCH_CHECK();
        }
    }
    hipLaunchKernelGGL((decode_kernel<BITS, HPB, DT, false, false, NT, REGL, CHUNKED, EXTRAS, NH, true>), dim3(units * g.nx),
                       dim3(NT), lds, st, g);
    CQ_LAUNCH_CHECK();
    return CQ_OK;
}

// A chunked launch has one instantiation: what the mask and the row count cost it in registers, it has to spare.
template <int BITS, int HPB, typename DT, int NT, int REGL, int NH = HPB>
static int launch_matrix_unit(const DecodeGeom& g, unsigned units, hipStream_t st) {
    if (g.nsplit > 1) return launch_matrix_one<BITS, HPB, DT, NT, REGL, true, true, NH>(g, units, st);
    if (g.mask || g.r_dev) return launch_matrix_one<BITS, HPB, DT, NT, REGL, false, true, NH>(g, units, st);
    return launch_matrix_one<BITS, HPB, DT, NT, REGL, false, false, NH>(g, units, st);
}

template <int BITS, typename DT>
static int launch_matrix_bits(const DecodeGeom& g, int hpb, int nh, int nt, unsigned units, hipStream_t st) {
    if (nt == 512) {
        if (hpb == 4 && nh == 3) return launch_matrix_unit<BITS, 4, DT, 512, kRegPair, 3>(g, units, st);
        if (hpb == 4) return launch_matrix_unit<BITS, 4, DT, 512, kRegPair>(g, units, st);
        if (g.chunk <= kRegPair * 512) return launch_matrix_unit<BITS, 2, DT, 512, kRegPair>(g, units, st);
        return launch_matrix_unit<BITS, 2, DT, 512, kRegMost>(g, units, st);
    }
    if (hpb == 4 && nh == 3) return launch_matrix_unit<BITS, 4, DT, 1024, kRegLong, 3>(g, units, st);
    if (hpb == 4) return launch_matrix_unit<BITS, 4, DT, 1024, kRegLong>(g, units, st);
    if (g.chunk <= kRegLong * 1024)
        return hpb == 2 ? launch_matrix_unit<BITS, 2, DT, 1024, kRegLong>(g, units, st)
                        : launch_matrix_unit<BITS, 1, DT, 1024, kRegLong>(g, units, st);
    return hpb == 2 ? launch_matrix_unit<BITS, 2, DT, 1024, kRegMost>(g, units, st)
                    : launch_matrix_unit<BITS, 1, DT, 1024, kRegMost>(g, units, st);
}

// nt threads per workgroup, g.chunk tokens at most: the plan's (cq_decode.hip: make_plan), whose layouts hold no more
// tokens than the instantiation picked here - checked, because a token too many would be left out of the sum
template <typename DT>
int launch_matrix(const DecodeGeom& g, int bits, int hpb, int nh, int nt, unsigned units, hipStream_t st) {
    const int rounds = hpb == 4 ? (nt == 512 ? kRegPair : kRegLong) : kRegMost;
    if (g.chunk > rounds * nt || (nt == 512 && hpb == 1)) return CQ_ERR_UNSUPPORTED;
    return bits == 1 ? launch_matrix_bits<1, DT>(g, hpb, nh, nt, units, st) : launch_matrix_bits<2, DT>(g, hpb, nh, nt, units, st);
}

}  // namespace cq
