// Instances of the medium-M GEMM with fp16 activations.
#include "gemm_kwave.h"

namespace pw4 {

KwaveFn kwave_f16(int stype, bool zp, int rt, int ct) { return pick_type<false>(stype, zp, rt, ct); }

}  // namespace pw4
