// The matrix-core form of the decode step for fp16 inputs and per-token values.
#include "cq_decode_matrix.h"

namespace cq {
template int launch_matrix_token<FP16>(const DecodeGeom& g, int bits, int hpb, int nt, unsigned units, hipStream_t st);
}  // namespace cq
