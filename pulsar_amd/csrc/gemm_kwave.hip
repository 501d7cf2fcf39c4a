// Launch of the medium-M GEMM (kernel: gemm_kwave.h; its instances are built by
// gemm_kwave_f16.hip and gemm_kwave_bf16.hip).
#include <algorithm>

#include "w4a16_common.h"
#include "w4a16_kernels.h"

namespace pw4 {

bool kwave_ok(int64_t N, int64_t K, int64_t G, int sbytes) {
    // 32-bit buffer ranges: a row tile of x, the weight words, the scales
    return K > 0 && K % 64 == 0 && G > 0 && G % 64 == 0 && N % 8 == 0 && K <= (int64_t{1} << 22) &&
           round_up(N, kMarlinBN) * K / 2 <= INT32_MAX && K / G * N * sbytes <= INT32_MAX && N * 4 <= INT32_MAX;
}

int kwave_tile_floats(int rt, int ct) { return rt * ct * 1024; }

hipError_t launch_kwave(int xtype, int stype, bool zp, int rt, const KwaveArgs& args, hipStream_t stream,
                        KernelEvents ev) {
    KwaveArgs a = args;
    const int ct = kwave_col_tiles(a.nb);
    const KwaveFn fn = xtype == X_BF16 ? kwave_bf16(stype, zp, rt, ct) : kwave_f16(stype, zp, rt, ct);
    // what the kernel's indexing rests on
    if (fn == nullptr || a.nb <= 0 || a.nb > 128 || a.nb % 16 != 0 || a.splits < 1 || a.splits > 65535 ||
        a.chunks_per_split < 1 || !kwave_ok(a.N, a.K, a.G, stype == S_F32 ? 4 : 2) || a.K % a.G != 0 ||
        (int64_t)a.chunks_per_split * a.splits < a.nchunks || (a.splits > 1 && (a.partial == nullptr || a.counters == nullptr)) ||
        (a.silu && a.N % 16 != 0)) {
        return hipErrorInvalidValue;
    }
    a.nchunks = a.K / 64;
    a.Kg = a.K / a.G;
    a.cpg = a.G / 64;
    a.cpg_recip = a.cpg > 1 ? (uint32_t)(((uint64_t{1} << 32) + a.cpg - 1) / a.cpg) : 0;
    a.ncols = (int)round_up(a.N, kMarlinBN);
    a.w_bytes = (uint32_t)((int64_t)a.ncols * a.K / 2);
    a.num_m = (int)ceil_div(a.M, 32 * rt);
    a.num_n = (int)ceil_div(a.N, a.nb);
    // runs of two chunks (one 128-K quant group) where they cost no wave a chunk more than single ones
    const int n = std::min(a.chunks_per_split, a.nchunks);
    a.run_log2 = ceil_div(n, 16) * 2 <= ceil_div(n, 8) ? 1 : 0;
    const int64_t nwg = (int64_t)a.num_m * a.num_n;
    if (nwg > INT32_MAX) return hipErrorInvalidValue;
    launch_kernel(fn, dim3((unsigned)nwg, (unsigned)a.splits), dim3(kKwaveThreads), 0, stream, ev.start, ev.stop, a);
    return hipGetLastError();
}

}  // namespace pw4
