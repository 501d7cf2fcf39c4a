// W4A16 GEMM for medium M on the MARLIN layout: y[M,N] = x[M,K] @ dequant(W)^T,
// fp16 or bf16 activations, K and the group size multiples of 64.
//
// Work split.  A workgroup of eight waves owns a tile of up to 32 * RT rows by
// nb <= 32 * C columns over one K slice (the planner gives whole column tiles, a
// pinned plan any multiple of 16); the waves split the slice's 64-K chunks
// between them, and every wave computes the whole tile over its own chunks.  So a weight word is loaded and dequantized by exactly one wave, an
// activation fragment is read from LDS once and used for all C column tiles,
// and no wave waits for another before the end: each has its own LDS ring of
// activations and its own register ring of weight words.  The eight partial
// tiles meet in LDS once, at the end of the slice.
//
// Streaming.  Per chunk a wave issues 4 * RT LDS copies of x (1 KB each: eight
// rows of 128 bytes), one or two of scales (and zero points), and C 16-byte
// weight loads per lane.  Copies and loads are buffer instructions: rows past M
// and chunks past the slice are out of the resource's range, so they read
// nothing.  The stages of the LDS ring are separate LDS variables: the
// compiler then knows which copy a read of a stage depends on, and its vmcnt
// waits leave the rest of the ring in flight.  (With one array, or through
// global_load_lds, it waits for every outstanding copy.)
//
// Math.  One 64-K chunk of 32 columns is four v_mfma_f32_32x32x16 per 32 rows:
// lane (c = l%32, h = l/32) holds the four words of column c in the chunk's
// tile h, and pair s of those words is the K run 32h + [8s, 8s + 8) of MFMA s.
// B = u - z, exact in fp16 and in bf16.  The group scale is applied in fp32 to
// the accumulators: with s_g a column's scale in group g, the running sum is
// multiplied by s_(g-1) / s_g when group g starts and by the last group's scale
// at the end (a group whose scale is zero adds zero and is skipped).
//
// Range.  The running sum is y / s_g, which fp32 does not hold for every input that
// y fits: scales far apart or (bf16) very large x overflow it.  A workgroup whose sums
// come out infinite or NaN where x is finite computes its slice again, each chunk's
// products scaled by themselves, and a scale out of range (scale_in_range) makes them
// NaN.  fp16 x cannot get there within that range, so fp16 x with fp16 scales has no
// check; the others look behind their stores.
//
// K slices across workgroups (small N): every workgroup writes its fp32 tile
// and the last to arrive for a tile (arrival counter) sums the slices in slice
// order, stores y and resets the counter.
//
// What bounds it.  At M = 32 the weight stream beside the x copies: LDS copies move 32
// bytes a clock per CU and return in order with the weights, so x costs as much as
// weights do, which is why tiles are as wide as the registers allow (gate_up
// 4096 x 28672: 18.6 us, of which the MFMAs fill 22% of the SIMDs' time and VALU issue
// 44%).  With two row tiles, and bf16's exact dequant, the issue itself: gate_up M = 64
// 37% and 47% with fp16 x, 29% and 70% with bf16.
// Graph periods on one MI355X, fp16 x, us, before (decode kernel up to M = 32,
// 128-row prefill tiles past it, with their combine) / this kernel:
//   gate_up 4096 x 28672   M = 24 27.0 / 18.1, M = 32 29.2 / 18.7, M = 64 42.6 / 24.2
//   down 14336 x 4096      M = 32 24.3 / 13.6, M = 64 31.8 / 18.1, M = 256 43.4 / 39.8
//   qkv 4096 x 6144        M = 32 11.0 / 9.2, M = 64 21.1 / 10.8, M = 256 27.5 / 20.2
//   o 4096 x 4096          M = 64 18.8 / 8.6, M = 256 24.3 / 14.0, M = 512 31.5 / 23.0
//   70B down 28672 x 8192  M = 32 64.8 / 34.3, M = 64 68.5 / 45.0
//   70B gate_up 8192 x 57344  M = 20 95.9 / 57.0, M = 32 125 / 62.4
// bf16 x: gate_up M = 64 41.9 / 26.9, down M = 64 35.0 / 19.0, qkv M = 256 27.7 / 24.2.
//
// Reference counterpart: w4a16_marlin_kernel at BM = 32 and 64
// (pulsar-core/src/kernels/w4a16_marlin.cu:197-304).
#pragma once

#include <type_traits>
#include <utility>

#include "w4a16_common.h"
#include "w4a16_kernels.h"

namespace pw4 {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kKwaveThreads;
static_assert(kThreads == kWaves * 64, "launch_kwave's block");
constexpr int kScaleSlot = 768;  // per wave and stage: 512 bytes of scales, 256 of zero-point words

// Scales the running sum takes: 2^-41 <= |s| < 2^23 (infinities and NaN make their sums so
// by themselves).  Two of them are less than 2^64 apart, so with fp16 x (2^16, times 15,
// over K <= 2^22) it stays below 2^106.  Written so that its constants are inline ones:
// the loop has no register for others.
__device__ __forceinline__ bool scale_in_range(float s) {
    return (uint32_t)(__builtin_amdgcn_frexp_expf(s) + 40) < 64u;
}

// Ring depth in chunks: LDS stages of x (RT * 4 KB per wave each, 128 KB in all)
// and register sets of weight words.
constexpr int ring_depth(int rt) { return rt == 1 ? 4 : 2; }

typedef __attribute__((address_space(3))) void lds_void;

template <int I>
using Int = std::integral_constant<int, I>;

template <typename F, int... I>
__device__ __forceinline__ void unroll_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(Int<I>{}), ...);
}

// (a & mask) | b; mask in an SGPR and b in a VGPR, so that it is one v_and_or_b32
__device__ __forceinline__ uint32_t bfi(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | b; }

template <bool BF16, typename ST, bool ZP, int RT, int C>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void kwave_kernel(const KwaveArgs a) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass needs the stub only, and drops a body it cannot check
    constexpr int D = ring_depth(RT);
    constexpr int kStage = RT * 4096;  // bytes of x per wave and stage
    __shared__ __attribute__((aligned(1024))) uint8_t xs0[kWaves * kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t xs1[kWaves * kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t xs2[D > 2 ? kWaves * kStage : 16];
    __shared__ __attribute__((aligned(1024))) uint8_t xs3[D > 2 ? kWaves * kStage : 16];
    __shared__ __attribute__((aligned(256))) uint8_t ss0[kWaves * kScaleSlot];
    __shared__ __attribute__((aligned(256))) uint8_t ss1[kWaves * kScaleSlot];
    __shared__ __attribute__((aligned(256))) uint8_t ss2[D > 2 ? kWaves * kScaleSlot : 16];
    __shared__ __attribute__((aligned(256))) uint8_t ss3[D > 2 ? kWaves * kScaleSlot : 16];
    __shared__ int s_last, s_over;
    __shared__ uint32_t s_bad[RT];  // rows whose sums are infinite or NaN
    auto xs = [&](auto i) -> uint8_t* {
        constexpr int I = decltype(i)::value;
        if constexpr (I == 0) return xs0;
        if constexpr (I == 1) return xs1;
        if constexpr (I == 2) return xs2;
        if constexpr (I == 3) return xs3;
    };
    auto ss = [&](auto i) -> uint8_t* {
        constexpr int I = decltype(i)::value;
        if constexpr (I == 0) return ss0;
        if constexpr (I == 1) return ss1;
        if constexpr (I == 2) return ss2;
        if constexpr (I == 3) return ss3;
    };

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int c = lane & 31, h = lane >> 5;
    const int M = a.M, N = a.N, K = a.K;

    // ---- tile: consecutive tiles share an XCD, row tiles of one column tile first
    const int nwg = a.num_m * a.num_n;
    int tile;
    {
        const int b = blockIdx.x, xcd = b & 7, q = nwg >> 3, r = nwg & 7;
        tile = xcd * q + min(xcd, r) + (b >> 3);
    }
    const int tn = tile / a.num_m, tm = tile - tn * a.num_m;
    const int m0 = tm * 32 * RT, n0 = tn * a.nb;
    const int split = blockIdx.y;
    const int c0 = split * a.chunks_per_split;
    const int c1 = min(c0 + a.chunks_per_split, a.nchunks);
    // this wave's chunks: runs of 2^run_log2 chunks, eight waves apart
    const int rl = a.run_log2;
    auto chunk_at = [&](int j) { return c0 + ((((j >> rl) << 3) + wave) << rl) + (j & ((1 << rl) - 1)); };

    // ---- ring refills ---------------------------------------------------------
    // (out-of-range refills read nothing: num_records 0)
    const int rows = min(M - m0, 32 * RT);
    const uint16_t* xt = a.x + (int64_t)m0 * K;
    const int x_range = rows * K * 2;
    // lane l copies 16-byte unit l % 8 (swizzled by row) of row l / 8 of each eight;
    // the swizzle of rows 8i.. depends on i's parity alone
    uint32_t x_off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = i * 8 + (lane >> 3);
        x_off[i] = (uint32_t)row * (uint32_t)(K * 2) + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    constexpr int kScaleCopies = sizeof(ST) == 4 && C > 2 ? 2 : 1;
    uint32_t s_off[kScaleCopies];
#pragma unroll
    for (int i = 0; i < kScaleCopies; ++i) {
        s_off[i] = sizeof(ST) == 4 ? (uint32_t)min(n0 + i * 64 + lane, N - 1) * 4u
                                   : (uint32_t)min(n0 + 2 * lane, N - 2) * 2u;  // N even
    }
    const int nw = N >> 3;
    const uint32_t z_off = (uint32_t)min((n0 >> 3) + lane, nw - 1) * 4u;
    uint32_t w_off[C];  // this lane's 16 bytes of each column tile's chunk 0
#pragma unroll
    for (int ct = 0; ct < C; ++ct) {
        // columns past the tile re-read its last one (their results are dropped)
        const int n = min(n0 + min(ct * 32 + c, a.nb - 1), a.ncols - 1);
        w_off[ct] = ((uint32_t)(n >> 6) * (uint32_t)a.nchunks * kChunkWords + (uint32_t)(h * 256 + (n & 63) * 4)) * 4u;
    }
    auto group_of = [&](int kc) { return a.cpg == 1 ? kc : (int)__umulhi((uint32_t)kc, a.cpg_recip); };
    // A chunk's refill is kCopies LDS copies (x, scales, zero points) and C weight loads.
    u32x4 wq[D][C];
    constexpr int kXC = RT * 4, kCopies = kXC + kScaleCopies + (ZP ? 1 : 0);
    struct Refill {
        int x_range, x_at, s_range, s_at, z_range, z_at, w_range, w_at;
    };
    auto prepare_refill = [&](int j) {
        Refill f;
        const int kc = chunk_at(j);
        const bool ok = kc < c1;
        const int g = ok ? group_of(kc) : 0;
        const int sb = N * (int)sizeof(ST);
        f.x_range = ok ? x_range : 0;
        f.x_at = ok ? kc * 128 : 0;
        f.s_range = ok ? a.Kg * sb : 0;
        f.s_at = g * sb;
        f.z_range = ok ? a.Kg * nw * 4 : 0;
        f.z_at = g * nw * 4;
        f.w_range = ok ? (int)a.w_bytes : 0;
        f.w_at = ok ? kc * (kChunkWords * 4) : 0;
        return f;
    };
    auto copy = [&](const Refill& f, auto ic, auto st) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i < kXC) {
            const __amdgpu_buffer_rsrc_t rx =
                __builtin_amdgcn_make_buffer_rsrc((void*)xt, (short)0, f.x_range, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(xs(st) + wave * kStage + i * 1024), 16,
                                                     (int)x_off[i & 1] + (i & ~1) * (K * 16), f.x_at, 0, 0);
        } else if constexpr (i < kXC + kScaleCopies) {
            constexpr int k = i - kXC;
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc((void*)a.scales, (short)0, f.s_range, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(ss(st) + wave * kScaleSlot + k * 256), 4,
                                                     (int)s_off[k], f.s_at, 0, 0);
        } else {
            const __amdgpu_buffer_rsrc_t rz =
                __builtin_amdgcn_make_buffer_rsrc((void*)a.qzeros, (short)0, f.z_range, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rz, (lds_void*)(ss(st) + wave * kScaleSlot + 512), 4, (int)z_off,
                                                     f.z_at, 0, 0);
        }
    };
    auto copies = [&](const Refill& f, auto lo, auto hi, auto st) {  // [lo, hi) of them
        constexpr int L = decltype(lo)::value, H = decltype(hi)::value;
        if constexpr (L < H) {
            unroll_seq([&](auto i) { copy(f, Int<L + decltype(i)::value>{}, st); },
                       std::make_integer_sequence<int, H - L>{});
        }
    };
    auto load_w = [&](const Refill& f, int ct, auto st) {
        const __amdgpu_buffer_rsrc_t rw =
            __builtin_amdgcn_make_buffer_rsrc((void*)a.w, (short)0, f.w_range, 0x00020000);
        // (2: non-temporal)
        wq[decltype(st)::value][ct] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)w_off[ct], f.w_at, 2);
    };

    f32x16 acc[RT][C];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < C; ++ct)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[rt][ct][e] = 0.f;
    float s_run[C];
#pragma unroll
    for (int ct = 0; ct < C; ++ct) s_run[ct] = 1.f;

    // splice constants in VGPRs (the masks come in SGPRs)
    uint32_t k1024, k64;
    asm volatile("v_mov_b32 %0, %1" : "=v"(k1024) : "s"(0x64006400u));
    asm volatile("v_mov_b32 %0, %1" : "=v"(k64) : "s"(0x54005400u));

    // ---- one chunk --------------------------------------------------------------
    auto step = [&](int j, auto st, auto refills) {
        constexpr int I = decltype(st)::value;
        constexpr bool kRefills = decltype(refills)::value;
        const uint8_t* xa = xs(st) + wave * kStage;
        const uint8_t* sa = ss(st) + wave * kScaleSlot;
        u32x4 av[4][RT];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int row = rt * 32 + c;
                av[s][rt] = *reinterpret_cast<const u32x4*>(xa + row * 128 + (((4 * h + s) ^ ((row >> 1) & 7)) * 16));
            }
        float sf[C];
        uint32_t zw[C];
#pragma unroll
        for (int ct = 0; ct < C; ++ct) {
            const int cl = ct * 32 + c;
            if constexpr (sizeof(ST) == 4) {
                sf[ct] = *reinterpret_cast<const float*>(sa + cl * 4);
            } else {
                sf[ct] = (float)*reinterpret_cast<const _Float16*>(sa + cl * 2);
            }
            zw[ct] = 8u;
            if constexpr (ZP) zw[ct] = (*reinterpret_cast<const uint32_t*>(sa + 512 + (cl >> 3) * 4) >> (4 * (cl & 7))) & 0xfu;
        }
        // the stage is in registers (the reads have returned), so its refill may go out
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        Refill rf{};
        if constexpr (kRefills) rf = prepare_refill(j + D);

        // scales: a column whose scale is zero in this group takes u = z and keeps its running scale
        bool zero = false;
#pragma unroll
        for (int ct = 0; ct < C; ++ct) zero |= sf[ct] == 0.f;
        if (__builtin_expect(__ballot(zero) != 0, 0)) {
#pragma unroll
            for (int ct = 0; ct < C; ++ct) {
                const bool t = sf[ct] == 0.f;
                sf[ct] = t ? s_run[ct] : sf[ct];
                const uint32_t zz = zw[ct] * 0x11111111u;
#pragma unroll
                for (int tg = 0; tg < 4; ++tg) wq[I][ct][tg] = t ? zz : wq[I][ct][tg];
            }
        }
        const int kc = chunk_at(j);
        // (the first chunk multiplies zeros)
        if (kc < c1 && (j == 0 || group_of(kc) != group_of(chunk_at(j - 1)))) {
#pragma unroll
            for (int ct = 0; ct < C; ++ct) {
                float r = s_run[ct] * __builtin_amdgcn_rcpf(sf[ct]);
                // (NaN sums are what the end of the slice looks for)
                if constexpr (sizeof(ST) == 4) r = scale_in_range(sf[ct]) ? r : __builtin_bit_cast(float, 0xffffffffu);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[rt][ct][e] *= r;
                s_run[ct] = sf[ct];
            }
        }
        // the zero point in both halves; 1024 + z and 64 + z are spliced where they are
        // used, which costs one operation per fragment and holds no registers
        uint32_t zz[C];
        float zf[C];
#pragma unroll
        for (int ct = 0; ct < C; ++ct) {
            zz[ct] = zw[ct] * 0x10001u;
            zf[ct] = (float)zw[ct];
        }
        auto dequant = [&](int s, int ct) {
            u32x4 bv;
#pragma unroll
            for (int tg = 0; tg < 4; ++tg) {
                const uint32_t q = wq[I][ct][tg];
                if constexpr (BF16) {
                    // nibble at bit 4s of a half word spliced into 2^(23 - 4s): exact
                    // 2^(23 - 4s) + u in fp32, and u - z exact in bf16's high half
                    const float base = (float)(1 << (23 - 4 * s));
                    const uint32_t bb = __builtin_bit_cast(uint32_t, base);
                    const float zc = base + zf[ct];
                    const float lo = __builtin_bit_cast(float, (q & (0xfu << (4 * s))) | bb) - zc;
                    const float hi = __builtin_bit_cast(float, ((q >> 16) & (0xfu << (4 * s))) | bb) - zc;
                    bv[tg] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo),
                                                   0x07060302u);
                } else {
                    const uint32_t v = s < 2 ? q : q >> 8;
                    bv[tg] = (s & 1) ? as_u32(as_h2(bfi(a.masks.hi, v, k64)) - as_h2(k64 | (zz[ct] << 4)))
                                     : as_u32(as_h2(bfi(a.masks.lo, v, k1024)) - as_h2(k1024 | zz[ct]));
                }
            }
            return bv;
        };
        // The refill goes out between the MFMAs: in one burst it would fill the CU's
        // address path and hold the wave up before its arithmetic.  Copies during
        // MFMAs 0-2, each weight load behind the last use of its registers.
        unroll_seq(
            [&](auto ic) {
                constexpr int i = decltype(ic)::value, s = i / C, ct = i % C;
                const u32x4 bv = dequant(s, ct);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt][ct] = mfma32x32x16<BF16>(av[s][rt], bv, acc[rt][ct]);
                if constexpr (!kRefills) {
                } else if constexpr (s < 3) {
                    copies(rf, Int<kCopies * i / (3 * C)>{}, Int<kCopies * (i + 1) / (3 * C)>{}, st);
                } else {
                    load_w(rf, ct, st);
                }
                __builtin_amdgcn_sched_barrier(0);
            },
            std::make_integer_sequence<int, 4 * C>{});
    };

    // ---- the slice ----------------------------------------------------------------
    unroll_seq(
        [&](auto st) {
            const Refill f = prepare_refill(decltype(st)::value);
            copies(f, Int<0>{}, Int<kCopies>{}, st);
            for (int ct = 0; ct < C; ++ct) load_w(f, ct, st);
            __builtin_amdgcn_sched_barrier(0);
        },
        std::make_integer_sequence<int, D>{});
    // Waves w and w + 4 share a SIMD: one of them goes ahead where both could issue, so that
    // they do not run their dequant and their MFMAs in step (1-3% over the sizes above).
    if (wave >= kWaves / 2) __builtin_amdgcn_s_setprio(2);
    const int nw_chunks = [&] {
        // chunks of this wave: whole rounds of eight runs, then its part of the last round
        const int n = max(c1 - c0, 0), round = 8 << rl;
        const int full = n / round, rest = n - full * round;
        return (full << rl) + min(max(rest - (wave << rl), 0), 1 << rl);
    }();
    // Whole rounds of the ring (refills past the wave's last chunk are out of range: from
    // nowhere), then the last chunks without refills.  Leaving a round in the middle, or
    // skipping a refill, would merge ring states, and the waits after it drain the ring.
    int j = 0;
    for (; j + D <= nw_chunks; j += D) {
        unroll_seq([&](auto st) { step(j + decltype(st)::value, st, std::true_type{}); },
                   std::make_integer_sequence<int, D>{});
    }
    unroll_seq(
        [&](auto st) {
            if (j + decltype(st)::value < nw_chunks) step(j + decltype(st)::value, st, std::false_type{});
        },
        std::make_integer_sequence<int, D - 1>{});

    // ---- the slice once more, each chunk's products scaled by themselves -------------
    // (B of bf16 x is (u - z) / 1024, still exact, so that a chunk's sum is no larger than
    // its largest x; plain loads: no measured workload comes here).  It takes its arguments
    // and its lane index anew, or the compiler holds what it derives from them in registers
    // through the whole slice: bf16 x, fp32 scales, zero points, gate_up M = 64 30.6 -> 33.1 us.
    auto rescan = [&]() {
        const KwaveArgs* p = reinterpret_cast<const KwaveArgs*>((const void*)__builtin_amdgcn_kernarg_segment_ptr());
        asm volatile("" : "+s"(p));
        int ln = threadIdx.x;
        asm volatile("" : "+v"(ln));
        const int c = ln & 31, h = (ln >> 5) & 1, wave = __builtin_amdgcn_readfirstlane(ln >> 6);
        const int64_t N = p->N, K = p->K;
        constexpr float kDown = BF16 ? 0x1p-10f : 1.f, kUp = 1.f / kDown;
#pragma unroll
        for (int ct = 0; ct < C; ++ct) {
            s_run[ct] = 1.f;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[rt][ct][e] = 0.f;
        }
        const int end = min((split + 1) * p->chunks_per_split, p->nchunks);
#pragma unroll 1
        for (int kc = split * p->chunks_per_split + wave; kc < end; kc += kWaves) {
            const int64_t g = kc / p->cpg;
#pragma unroll
            for (int ct = 0; ct < C; ++ct) {
                const int n = min(n0 + ct * 32 + c, (int)N - 1);
                const float s = (float)reinterpret_cast<const ST*>(p->scales)[g * N + n];
                uint32_t z = 8u;
                if constexpr (ZP) z = (p->qzeros[g * (N >> 3) + (n >> 3)] >> (4 * (n & 7))) & 0xfu;
                const u32x4 q = *reinterpret_cast<const u32x4*>(
                    p->w + ((int64_t)(n >> 6) * p->nchunks + kc) * kChunkWords + h * 256 + (n & 63) * 4);
                auto weight = [&](uint32_t u) { return ((float)(u & 0xfu) - (float)z) * kDown; };
                u32x4 bv[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int tg = 0; tg < 4; ++tg) {
                        const uint32_t lo = f32_to_out<BF16>(weight(q[tg] >> (4 * i)));
                        const uint32_t hi = f32_to_out<BF16>(weight(q[tg] >> (16 + 4 * i)));
                        bv[i][tg] = lo | hi << 16;
                    }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const uint16_t* xr = p->x + min(m0 + rt * 32 + c, p->M - 1) * K + kc * 64 + h * 32;
                    f32x16 t;
#pragma unroll
                    for (int e = 0; e < 16; ++e) t[e] = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        t = mfma32x32x16<BF16>(*reinterpret_cast<const u32x4*>(xr + 8 * i), bv[i], t);
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[rt][ct][e] += t[e] * s * kUp;
                }
            }
        }
    };

    // ---- sum of the waves in LDS, over the freed stages ----------------------------
    // A wave's accumulators are 16-byte quads (four rows of a column),
    // [tile][e / 4][lane]; quad q of the tile is summed by thread q % 512.
    constexpr int kTileBytes = RT * C * 4096;           // of one wave
    constexpr int kArray = kWaves * kStage;             // of one LDS variable
    constexpr bool kTwoPhase = kTileBytes * kWaves > kArray * D;
    constexpr int kParts = kTwoPhase ? kWaves / 2 : kWaves;  // partial tiles in LDS at a time
    static_assert(kTileBytes * kParts <= kArray * D && kArray % kTileBytes == 0, "the sum fits the stages");
    auto region = [&](int w) -> uint8_t* {
        const int at = w * kTileBytes, arr = at / kArray, off = at - arr * kArray;
        if constexpr (D > 2) {
            return (arr == 0 ? xs0 : arr == 1 ? xs1 : arr == 2 ? xs2 : xs3) + off;
        } else {
            return (arr == 0 ? xs0 : xs1) + off;
        }
    };
    auto put = [&](uint8_t* to) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < C; ++ct)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const f32x4 v{acc[rt][ct][4 * e4], acc[rt][ct][4 * e4 + 1], acc[rt][ct][4 * e4 + 2],
                                  acc[rt][ct][4 * e4 + 3]};
                    *reinterpret_cast<f32x4*>(to + (((rt * C + ct) * 4 + e4) * 64 + lane) * 16) = v;
                }
    };
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies into LDS are done (those past its chunks too)
    if (tid < RT) s_bad[tid] = 0;
    if (tid == 0) s_over = 0;
    constexpr int kQuads = RT * C * 256;
    constexpr int QT = (kQuads + kThreads - 1) / kThreads;  // quads per thread
    f32x4 sum[QT];
    auto add_waves = [&]() {
#pragma unroll
        for (int ct = 0; ct < C; ++ct)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[rt][ct][e] *= s_run[ct];
        __syncthreads();
        if constexpr (kTwoPhase) {
            if (wave >= kParts) put(region(wave - kParts));
            __syncthreads();
            if (wave < kParts) {
                const uint8_t* from = region(wave);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int ct = 0; ct < C; ++ct)
#pragma unroll
                        for (int e4 = 0; e4 < 4; ++e4) {
                            const f32x4 v =
                                *reinterpret_cast<const f32x4*>(from + (((rt * C + ct) * 4 + e4) * 64 + lane) * 16);
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[rt][ct][4 * e4 + e] += v[e];
                        }
            }
            // (a wave overwrites only the region it read)
            if (wave < kParts) put(region(wave));
        } else {
            put(region(wave));
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            const int q = tid + i * kThreads;
            if (kQuads % kThreads != 0 && q >= kQuads) break;
            f32x4 v[kParts];
#pragma unroll
            for (int w = 0; w < kParts; ++w) v[w] = *reinterpret_cast<const f32x4*>(region(w) + q * 16);
            sum[i] = v[0];
#pragma unroll
            for (int w = 1; w < kParts; ++w) sum[i] += v[w];
        }
    };
    add_waves();

    // ---- output -----------------------------------------------------------------------
    auto store = [&](int q, const f32x4& v) {
        const int ln = q & 63, e4 = (q >> 6) & 3, t = q >> 8;  // t = rt * C + ct
        const int rt = t / C, ct = t - rt * C;
        const int cl = ct * 32 + (ln & 31);
        const int n = n0 + cl;
        const int m = m0 + rt * 32 + 8 * e4 + 4 * (ln >> 5);
        if (a.silu) {
            // gate|up interleaved by 8: a gate lane takes its up value from lane ^ 8
            const int nh = N >> 1;
            f32x4 up;
#pragma unroll
            for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(v[e], 8);
            if (cl < a.nb && n < N && (n & 8) == 0) {
                const int on = (n >> 4 << 3) | (n & 7);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (m + e < M) a.y[(int64_t)(m + e) * nh + on] = f32_to_out<BF16>(silu_mul(v[e], up[e]));
            }
            return;
        }
        if (cl < a.nb && n < N) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (m + e < M) {
                    a.y[(int64_t)(m + e) * N + n] = f32_to_out<BF16>(v[e]);
                    if (a.y32) a.y32[(int64_t)(m + e) * N + n] = v[e];
                }
        }
    };
    auto store_sums = [&]() {
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            const int q = tid + i * kThreads;
            if (kQuads % kThreads != 0 && q >= kQuads) break;
            store(q, sum[i]);
        }
    };
    constexpr bool kCheck = BF16 || sizeof(ST) == 4;  // (see Range)
    auto look = [&]() {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            if (kQuads % kThreads != 0 && tid + i * kThreads >= kQuads) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) bad |= !(__builtin_fabsf(sum[i][e]) <= 0x1.fffffep127f);
        }
        if (__builtin_expect(__ballot(bad) != 0, 0)) {
#pragma unroll
            for (int i = 0; i < QT; ++i) {
                const int q = tid + i * kThreads;
                if (kQuads % kThreads != 0 && q >= kQuads) break;
                uint32_t rows4 = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) rows4 |= (uint32_t)!(__builtin_fabsf(sum[i][e]) <= 0x1.fffffep127f) << e;
                if (rows4) atomicOr(&s_bad[q / (C * 256)], rows4 << (8 * ((q >> 6) & 3) + 4 * ((q & 63) >> 5)));
            }
        }
    };
    // Whether a row of s_bad is finite in x (an infinity or NaN of x belongs in its row's
    // sums, and is there already).  Every wave looks at every eighth row.
    auto overflowed = [&]() {
        constexpr uint32_t kInf = BF16 ? 0x7f80u : 0x7c00u;
        const KwaveArgs* p = reinterpret_cast<const KwaveArgs*>((const void*)__builtin_amdgcn_kernarg_segment_ptr());
        asm volatile("" : "+s"(p));
        int ln = threadIdx.x;
        asm volatile("" : "+v"(ln));
        const int begin = split * p->chunks_per_split, end = min(begin + p->chunks_per_split, p->nchunks);
#pragma unroll 1
        for (int r = __builtin_amdgcn_readfirstlane(ln >> 6); r < 32 * RT; r += kWaves) {
            if (!((s_bad[r >> 5] >> (r & 31)) & 1u) || m0 + r >= p->M) continue;
            const u32x4* xr = reinterpret_cast<const u32x4*>(p->x + (int64_t)(m0 + r) * p->K);
            bool inf = false;
#pragma unroll 1
            for (int i = begin * 8 + (ln & 63); i < end * 8; i += 64) {
                const u32x4 v = xr[i];
#pragma unroll
                for (int j = 0; j < 4; ++j) inf |= (v[j] & kInf) == kInf || ((v[j] >> 16) & kInf) == kInf;
            }
            if (__ballot(inf) == 0 && (ln & 63) == 0) s_over = 1;
        }
        __syncthreads();  // (s_bad stays as it is: a wave may still be at its any_bad)
        return __builtin_amdgcn_readfirstlane(s_over) != 0;
    };
    auto any_bad = [&]() {
        uint32_t v = 0;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) v |= s_bad[rt];
        return __builtin_amdgcn_readfirstlane(v) != 0;
    };
    if (a.partial == nullptr) {
        store_sums();
        if constexpr (kCheck) {
            look();
            __syncthreads();  // (and every wave has read the regions)
            if (__builtin_expect(any_bad(), 0) && overflowed()) {
                rescan();
                add_waves();
                store_sums();
            }
        }
        return;
    }
    // K slices: device-scope stores and loads (written through to and read from
    // the device's coherence point); every wave waits for its stores before the
    // barrier ahead of the counter, so the last arriver sees every slice.
    auto part = [&](int sp, int q) {
        return reinterpret_cast<uint64_t*>(a.partial + (((int64_t)tile * a.splits + sp) * kQuads + q) * 4);
    };
    auto write_part = [&]() {
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            const int q = tid + i * kThreads;
            if (kQuads % kThreads != 0 && q >= kQuads) break;
            uint64_t* p = part(split, q);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint64_t v = (uint64_t)__builtin_bit_cast(uint32_t, (float)sum[i][2 * e]) |
                                   ((uint64_t)__builtin_bit_cast(uint32_t, (float)sum[i][2 * e + 1]) << 32);
                __hip_atomic_store(p + e, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if constexpr (kCheck) look();
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    };
    write_part();
    if constexpr (kCheck) {
        if (__builtin_expect(any_bad(), 0) && overflowed()) {
            rescan();
            add_waves();
            write_part();
        }
    }
    if (tid == 0) {
        s_last = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                 a.splits - 1;
    }
    __syncthreads();
    if (!s_last) return;
#pragma unroll
    for (int i = 0; i < QT; ++i) sum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int sp0 = 0; sp0 < a.splits; sp0 += 4) {
        uint64_t v[4][QT][2];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int sp = min(sp0 + b, a.splits - 1);  // (past the last: re-read, not added)
#pragma unroll
            for (int i = 0; i < QT; ++i) {
                const int q = min(tid + i * kThreads, kQuads - 1);
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    v[b][i][e] = __hip_atomic_load(part(sp, q) + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (sp0 + b >= a.splits) break;
#pragma unroll
            for (int i = 0; i < QT; ++i)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    sum[i][2 * e] += __builtin_bit_cast(float, (uint32_t)v[b][i][e]);
                    sum[i][2 * e + 1] += __builtin_bit_cast(float, (uint32_t)(v[b][i][e] >> 32));
                }
        }
    }
    store_sums();
    if (tid == 0) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}

template <bool BF16, typename ST, bool ZP>
KwaveFn pick_tile(int rt, int ct) {
    if (rt == 1) {
        if (ct == 1) return kwave_kernel<BF16, ST, ZP, 1, 1>;
        if (ct == 2) return kwave_kernel<BF16, ST, ZP, 1, 2>;
        if (ct == 4) return kwave_kernel<BF16, ST, ZP, 1, 4>;
    }
    if (rt == 2) {
        if (ct == 1) return kwave_kernel<BF16, ST, ZP, 2, 1>;
        if (ct == 2) return kwave_kernel<BF16, ST, ZP, 2, 2>;
        if (ct == 4) return kwave_kernel<BF16, ST, ZP, 2, 4>;
    }
    return nullptr;
}

// The kernel for a scale type, zero points and tile (rt 1 or 2, ct 1, 2 or 4), or null.
template <bool BF16>
KwaveFn pick_type(int stype, bool zp, int rt, int ct) {
    if (stype == S_F32) return zp ? pick_tile<BF16, float, true>(rt, ct) : pick_tile<BF16, float, false>(rt, ct);
    return zp ? pick_tile<BF16, _Float16, true>(rt, ct) : pick_tile<BF16, _Float16, false>(rt, ct);
}

}  // namespace
}  // namespace pw4
