// Instances of the medium-M GEMM with bf16 activations.
#include "gemm_kwave.h"

namespace pw4 {

KwaveFn kwave_bf16(int stype, bool zp, int rt, int ct) { return pick_type<true>(stype, zp, rt, ct); }

}  // namespace pw4
