"""The medium-M GEMM (gemm_kwave.h): eight K waves per tile, sums through LDS, K slices summed by
the last workgroup to arrive.

PW4_KWAVE="<row tiles>,<columns>,<slices>" pins its tile, so that every edge is reached: one and
two 32-row tiles, full and ragged; 16 to 128 columns on 1, 2 and 4 column tiles, with tiles that
straddle the 64-column weight blocks; waves without a chunk, uneven waves, several ring rounds;
slices of unequal length.  The bars are those of every GEMM test (w4a16_case), against the fp32
oracle.
"""

import ctypes
import os

import numpy as np
import pytest
import torch

import pulsar_amd
from pulsar_amd import ops
from pw4_capi import DTYPE_BF16, DTYPE_F16, PW4_NOALLOC_SCRATCH_BYTES, declare
from w4a16_case import baseline_case, check


def describe(m, k, n, g=128, dtype=DTYPE_F16, layout=1, perm=0, splits=0):
    lib = pulsar_amd.capi()
    lib.pw4_medium_plan_describe.argtypes = [ctypes.c_int] * 6 + [ctypes.c_int64] * 5 + [ctypes.c_char_p, ctypes.c_size_t]
    buf = ctypes.create_string_buffer(160)
    rc = lib.pw4_medium_plan_describe(layout, dtype, DTYPE_F16, 0, perm, 0, m, n, k, g, splits, buf, len(buf))
    assert rc == 0, rc
    return buf.value.decode()


@pytest.fixture
def pin():
    old = os.environ.pop("PW4_KWAVE", None)

    def set_(v):
        if v is None:
            os.environ.pop("PW4_KWAVE", None)
        else:
            os.environ["PW4_KWAVE"] = v

    yield set_
    set_(old)


def _run(c, g, sdtype, act, sym, offset=0):
    g_idx = torch.from_numpy(c.g_idx).cuda() if act else None
    wm, perm = ops.repack_w4a16_gptq(c.qweight(), g_idx, g)
    s = torch.from_numpy(np.ascontiguousarray(c.scale_nk.T)).to(sdtype).cuda()
    if offset:  # the same values at an address that is not a multiple of four
        buf = torch.empty(s.numel() + offset, dtype=sdtype, device="cuda")
        buf[offset:].copy_(s.reshape(-1))
        s = buf[offset:].view(s.shape)
    return ops.gemm_w4a16_gptq(c.x, wm, s, None if sym else c.qzeros(), perm if act else None, g)


# (pin, m, n, k, g)
CASES = [
    ("1,16,1", 17, 64, 64, 64),       # one chunk: seven waves without one
    ("1,32,1", 32, 96, 512, 64),      # one chunk a wave
    ("1,48,1", 31, 200, 1088, 64),    # 17 chunks; tiles straddle the 64-column blocks, ragged N
    ("1,112,1", 33, 456, 2304, 256),  # two row tiles of 32, the second of one row; 36 chunks
    ("1,128,3", 20, 1000, 4096, 128),  # 22 + 22 + 20 chunks
    ("2,16,2", 64, 128, 1024, 128),
    ("2,64,1", 65, 320, 4160, 64),    # a second row tile of one row; 65 chunks
    ("2,96,1", 63, 520, 768, 128),
    ("2,112,5", 130, 904, 2560, 128),
    ("2,128,8", 48, 136, 8192, 128),
    ("1,64,1", 33, 256, 1152, 192),   # three chunks a group: the group index of a chunk is no shift
    ("2,128,2", 70, 264, 3840, 192),
    ("1,32,3", 24, 72, 2560, 320),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sdtype,sym,act", [(torch.float16, True, False), (torch.float32, False, True),
                                            (torch.float16, False, True), (torch.float32, True, False)])
@pytest.mark.parametrize("plan,m,n,k,g", CASES)
def test_kwave_plans(pin, plan, m, n, k, g, dtype, sdtype, sym, act):
    c = baseline_case(m, n, k, g, dtype=dtype, seed=m * 3 + n, symmetric=sym, act_order=act)
    pin(plan)
    y = _run(c, g, sdtype, act, sym)
    check(y, c.y_ref, dtype, f"{plan} m={m} n={n} k={k} g={g} {dtype}")
    for _ in range(3):  # the counters are left zero, and the sum does not depend on arrival
        assert torch.equal(_run(c, g, sdtype, act, sym), y)


def _silu(y):
    t = y.astype(np.float64).reshape(y.shape[0], -1, 2, 8)
    return (t[:, :, 0] / (1.0 + np.exp(-t[:, :, 0])) * t[:, :, 1]).reshape(y.shape[0], -1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sym,act", [(True, False), (False, True)])
@pytest.mark.parametrize("plan,m,n,k", [("1,32,1", 9, 48, 512), ("1,48,1", 31, 208, 1024), ("2,64,2", 65, 320, 2048),
                                        ("2,112,1", 47, 464, 768), ("1,128,1", 33, 144, 1024),
                                        ("2,128,3", 130, 912, 2560)])
def test_kwave_silu(pin, plan, m, n, k, sym, act, dtype):
    """The gate in the kernel's store, unsplit and behind the sum of K slices; tiles whose last
    columns, and rows, are past the output."""
    c = baseline_case(m, n, k, 128, dtype=dtype, seed=m + n, symmetric=sym, act_order=act)
    wm, perm = ops.repack_w4a16_gptq(c.qweight(), torch.from_numpy(c.g_idx).cuda() if act else None, 128)
    pin(plan)
    y = ops.gemm_w4a16_silu_mul(c.x, wm, c.scale(torch.float16, kn=True), None if sym else c.qzeros(),
                                perm if act else None, 128)
    assert y.shape == (m, n // 2)
    check(y, _silu(c.y_ref), dtype, f"{plan} m={m} n={n} k={k} {dtype}", abs_excess=False)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("plan,m,n,k,g", [("1,32,1", 33, 96, 512, 64), ("2,64,2", 64, 320, 2048, 128),
                                          ("2,128,1", 130, 520, 1088, 64), ("1,128,3", 48, 136, 4096, 128)])
def test_kwave_packed(pin, plan, m, n, k, g, dtype):
    """Packed weights past the decode sizes: repacked into the workspace, behind the partial tiles."""
    c = baseline_case(m, n, k, g, dtype=dtype, seed=m + k)
    pin(plan)
    assert describe(m, k, n, g, layout=0).endswith("repack")
    y = ops.gemm_w4a16(c.x, c.ct_packed(), c.scale(), g)
    check(y, c.y_ref, dtype, f"{plan} m={m} n={n} k={k} g={g} {dtype}")
    assert torch.equal(ops.gemm_w4a16(c.x, c.ct_packed(), c.scale(), g), y)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(64, 512, 2048), (16, 512, 1024)])
def test_workspace_too_small_for_the_slices(pin, monkeypatch, m, n, k):
    """K slices need scratch; without enough of it the call runs its decode or prefill plan, which
    here needs none, bit for bit as if the medium-M kernel were kept out."""
    g = 128
    c = baseline_case(m, n, k, g, seed=m)
    wm, _ = ops.repack_w4a16_gptq(c.qweight(), None, g)
    s = c.scale(torch.float16, kn=True)
    lib = declare(pulsar_amd.capi())
    monkeypatch.setenv("PW4_PREFILL_SPLITS", "1")

    def call(nbytes):
        y = torch.empty(m, n, dtype=torch.float16, device="cuda")
        ws = torch.zeros(max(nbytes, 1), dtype=torch.uint8, device="cuda")
        rc = lib.pw4_gemm_w4a16_marlin(c.x.data_ptr(), DTYPE_F16, wm.data_ptr(), s.data_ptr(), DTYPE_F16, None, None,
                                       y.data_ptr(), m, n, k, g, 0, ws.data_ptr() if nbytes else None, nbytes,
                                       torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc == 0, rc
        return y

    pin("0")
    assert lib.pw4_gemm_w4a16_marlin_workspace_size(m, n, k, g, 0, 0) == 0
    other = call(0)
    pin("2,64,2")
    need = lib.pw4_gemm_w4a16_marlin_workspace_size(m, n, k, g, 0, 0)
    assert need > 0
    full = call(need)
    check(full, c.y_ref, torch.float16, "on its slices")
    for nbytes in (need - 256, 1 << 20, 0):
        assert torch.equal(call(nbytes), other), nbytes
    assert torch.equal(call(need), full)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("plan", ["1,64,1", "2,128,2"])
def test_zero_and_negative_scales(pin, plan, dtype):
    """A group whose scale is zero adds nothing (wherever it lies in a wave's chunks), and
    negative scales are as good as positive ones."""
    m, n, k, g = 40, 256, 2048, 128
    c = baseline_case(m, n, k, g, dtype=dtype, seed=5)
    rng = np.random.default_rng(7)
    s = c.scale_nk * np.where(rng.random(c.scale_nk.shape) < 0.5, -1, 1)
    s[rng.random(s.shape) < 0.4] = 0.0
    s[3] = 0.0       # a column without any weight
    s[5, 1:] = 0.0   # the first group alone
    s[6, :-1] = 0.0  # the last group alone
    c.scale_nk = s.astype(np.float32)
    w = (c.u.astype(np.float32) - 8) * np.repeat(c.scale_nk, g, axis=1)
    ref = c.x.float().cpu().numpy() @ w.T
    pin(plan)
    y = _run(c, g, torch.float32, False, True)
    check(y, ref, dtype, f"{plan} {dtype}")
    assert (y[:, 3] == 0).all()


def _ref64(c, g):
    """x @ dequant(W)^T in 64 bits, for scales and activations whose fp32 sums could overflow."""
    w = (c.u.astype(np.float64) - c.z.T.repeat(g, axis=1)) * np.repeat(c.scale_nk.astype(np.float64), g, axis=1)
    return c.x.double().cpu().numpy() @ w.T


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sym", [True, False])
@pytest.mark.parametrize("low", [2.0 ** -40, 2.0 ** -45, 2.0 ** -119, 1e-40, 2.0 ** 45])
@pytest.mark.parametrize("plan", ["1,64,1", "2,128,2", "1,128,3", "2,32,1"])
def test_scales_far_from_their_neighbours(pin, plan, low, sym, dtype):
    """A group whose scale is many powers of two below (or above) the others': the sum behind it,
    in its units, is past fp32, but y is not."""
    if low > 1 and dtype == torch.float16:
        pytest.skip("activations of 2^-45 are not fp16 values")
    m, n, k, g = 40, 256, 2048, 128
    c = baseline_case(m, n, k, g, dtype=dtype, seed=11, symmetric=sym)
    s = np.full_like(c.scale_nk, 16.0)
    s[:, 5] = low
    s[7, 1:] = low      # all groups but the first, or the last
    s[9, :-1] = low
    s[11] = low         # every group
    s[13, 3:] = 0.0
    c.scale_nk = s.astype(np.float32)
    if low > 1:  # y of ordinary size again
        c.x = (c.x.float() * 2.0 ** -45).to(dtype)
    ref = _ref64(c, g)
    pin(plan)
    y = _run(c, g, torch.float32, False, sym)
    cols = [i for i in range(n) if i not in (11, 7, 9)] if low > 1 else list(range(n))
    check(y[:, cols], ref[:, cols], dtype, f"{plan} low={low} {dtype}", abs_excess=False)
    for i in (7, 9, 11):  # against their own size: their sums may be far from the others'
        r = ref[:, i]
        if np.abs(r).max() > 1e-37 and dtype == torch.bfloat16 or np.abs(r).max() > 1e-2:
            assert np.abs(y[:, i].double().cpu().numpy() - r).max() <= 2e-2 * np.abs(r).max(), (i, low)


@pytest.mark.gpu
@pytest.mark.parametrize("sdtype,sym", [(torch.float16, True), (torch.float32, False)])
@pytest.mark.parametrize("plan", ["1,64,1", "2,128,2"])
def test_large_bf16_activations(pin, plan, sdtype, sym):
    """Activations near bf16's largest, scaled by a power of two: the same result, scaled."""
    m, n, k, g = 40, 256, 2048, 128
    c = baseline_case(m, n, k, g, dtype=torch.bfloat16, seed=12, symmetric=sym)
    pin(plan)
    y = _run(c, g, sdtype, False, sym)
    check(y, c.y_ref, torch.bfloat16, plan)
    c.x = (c.x.float() * 2.0 ** 121).to(torch.bfloat16)
    assert c.x.isfinite().all()
    scaled = _run(c, g, sdtype, False, sym).double() * 2.0 ** -121
    check(scaled, c.y_ref, torch.bfloat16, plan + " scaled")


@pytest.mark.gpu
@pytest.mark.parametrize("plan", ["1,64,1", "2,128,2"])
def test_overflow_beside_rows_that_are_infinite_by_themselves(pin, plan):
    """Rows whose x holds an infinity or NaN need no second look; rows that overflow beside them
    do, in the same tile and in others, for large bf16 x and for scales far apart."""
    m, n, k, g = 72, 256, 2048, 128
    bad = {3: float("inf"), 40: float("nan"), 71: float("-inf")}
    keep = [i for i in range(m) if i not in bad]
    pin(plan)
    for dtype in (torch.bfloat16, torch.float16):
        c = baseline_case(m, n, k, g, dtype=dtype, seed=31)
        if dtype == torch.bfloat16:
            c.x = (c.x.float() * 2.0 ** 121).to(dtype)
            for row, v in bad.items():
                c.x[row, 17 * row] = v
            y = _run(c, g, torch.float16, False, True)
            check(y[keep].double() * 2.0 ** -121, c.y_ref[keep], dtype, f"{plan} large x")
            assert not y[list(bad)].isfinite().any()
            c = baseline_case(m, n, k, g, dtype=dtype, seed=31)
        s = np.full_like(c.scale_nk, 16.0)
        s[:, 5] = 2.0 ** -119
        c.scale_nk = s
        ref = _ref64(c, g)
        for row, v in bad.items():
            c.x[row, 17 * row] = v
        y = _run(c, g, torch.float32, False, True)
        check(y[keep], ref[keep], dtype, f"{plan} {dtype} scales", abs_excess=False)
        assert not y[list(bad)].isfinite().any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_infinite_and_nan_rows_stay_in_their_rows(pin, dtype):
    m, n, k, g = 48, 192, 1024, 128
    c = baseline_case(m, n, k, g, dtype=dtype, seed=9)
    c.x[7, 100] = float("inf")
    c.x[40, 900] = float("nan")
    pin("2,64,2")
    y = _run(c, g, torch.float16, False, True).float()
    keep = torch.ones(m, dtype=torch.bool)
    keep[[7, 40]] = False
    check(y[keep].to(dtype), c.y_ref[keep.numpy()], dtype, "the other rows")
    assert y[40].isnan().all()
    u = torch.from_numpy(c.u[:, 100].astype(np.int64)).cuda() - 8  # inf * weight: its sign, or NaN for 0
    assert torch.equal(y[7][u > 0], torch.full_like(y[7][u > 0], float("inf")))
    assert torch.equal(y[7][u < 0], torch.full_like(y[7][u < 0], float("-inf")))
    assert y[7][u == 0].isnan().all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,g", [(32, 6144, 4096, 128), (100, 520, 4160, 64)])
def test_default_plan_and_unaligned_scales(pin, m, n, k, g, dtype):
    """The plan the library picks by itself, and the call it does not take: fp16 scales at an odd
    2-byte address run on the decode or prefill plan, with the same result up to rounding."""
    c = baseline_case(m, n, k, g, dtype=dtype, seed=m)
    pin(None)
    assert describe(m, k, n, g, DTYPE_BF16 if dtype == torch.bfloat16 else DTYPE_F16).startswith("kwave")
    for offset in (0, 1):
        check(_run(c, g, torch.float16, False, True, offset), c.y_ref, dtype, f"m={m} offset={offset}")


@pytest.mark.gpu
def test_no_alloc_call_whose_slices_do_not_fit_its_scratch(pin):
    """16-column tiles take 32 columns of partial tile each: eight slices of 200 x 4096 need 59 MB
    beside the 16 MB zero region, more than the no-alloc scratch.  The call runs its other plan."""
    m, n, k, g = 200, 4096, 4096, 128
    c = baseline_case(m, n, k, g, seed=21)
    wm, _ = ops.repack_w4a16_gptq(c.qweight(), None, g)
    s = c.scale(torch.float16, kn=True)
    lib = declare(pulsar_amd.capi())
    pin("1,16,8")
    assert lib.pw4_gemm_w4a16_marlin_workspace_size(m, n, k, g, 0, 0) > PW4_NOALLOC_SCRATCH_BYTES
    y = torch.empty(m, n, dtype=torch.float16, device="cuda")
    rc = lib.pw4_gemm_w4a16_marlin_noalloc(c.x.data_ptr(), DTYPE_F16, wm.data_ptr(), s.data_ptr(), DTYPE_F16, None,
                                           None, y.data_ptr(), m, n, k, g, 0,
                                           torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    check(y, c.y_ref, torch.float16, "no-alloc")


@pytest.mark.parametrize("m,k,n,kwave", [
    # us on MI355X, graph periods, fp16 x: K-wave / the decode or prefill plan
    (24, 4096, 6144, True),    # 9.0 / 10.7
    (17, 4096, 4096, False),   # 7.8 / 7.7
    (32, 4096, 28672, True),   # 19.9 / 29.0
    (32, 14336, 4096, True),   # 14.9 / 24.3
    (64, 4096, 4096, True),    # 9.2 / 19.0
    (128, 14336, 4096, True),  # 25.7 / 35.3
    (256, 4096, 6144, True),   # 20.9 / 28.3
    (256, 4096, 28672, False),  # 85 / 65.6
    (4096, 4096, 28672, False),
    (16, 4096, 28672, False),  # 18.2 / 16.0
    (17, 4096, 28672, True),   # 18.3 / 26.6
    (20, 8192, 57344, True),   # 54.5 / 91.7, two rounds of tiles
    (1024, 4096, 4096, False),  # 47.2 / 45.9, two rounds of tiles
    (8, 4096, 4096, False),
])
def test_planner(pin, m, k, n, kwave):
    pin(None)
    assert (describe(m, k, n) != "none") == kwave, describe(m, k, n)


@pytest.mark.parametrize("m,k,n,g,dtype,kwave", [
    # the same on small layers, where a launch and the units' ends are most of the decode kernel's
    # time: K-wave / decode
    (9, 2048, 2560, 64, DTYPE_BF16, False),    # 6.1 / 4.4
    (9, 3072, 4096, 64, DTYPE_F16, False),     # 6.7 / 5.0
    (16, 512, 1024, 64, DTYPE_F16, False),     # 4.2 / 3.5
    (32, 1024, 4096, 128, DTYPE_BF16, False),  # 5.3 / 4.3
    (32, 1536, 2560, 64, DTYPE_BF16, False),   # 5.9 / 5.3
    (9, 8192, 8192, 64, DTYPE_BF16, True),     # 14.3 / 16.7 (M = 10)
    (13, 14336, 4096, 64, DTYPE_BF16, True),   # 14.3 / 16.4
])
def test_planner_on_small_layers(pin, m, k, n, g, dtype, kwave):
    pin(None)
    assert (describe(m, k, n, g, dtype) != "none") == kwave, describe(m, k, n, g, dtype)


@pytest.mark.parametrize("m,k,n,dtype,kwave", [
    # few columns and many rows, where every XCD reads all of x: K-wave / prefill tiles
    (2048, 12288, 512, DTYPE_F16, False),   # 58.4 / 40.2
    (4096, 8192, 128, DTYPE_BF16, False),   # 41.3 / 29.2
    (1500, 8192, 512, DTYPE_F16, False),    # 34.6 / 27.7
    (2048, 8192, 1024, DTYPE_F16, False),
    (1024, 16384, 512, DTYPE_F16, False),   # 47.4 / 37.2
    (2048, 4096, 1024, DTYPE_F16, True),    # 29.0 / 32.0
])
def test_planner_on_narrow_layers(pin, m, k, n, dtype, kwave):
    pin(None)
    assert (describe(m, k, n, 128, dtype) != "none") == kwave, describe(m, k, n, 128, dtype)


def test_planner_keeps_what_the_kernel_does_not_take(pin):
    pin(None)
    assert describe(64, 4096, 4096, splits=2) == "none"   # a forced K split
    assert describe(64, 4096, 4096, g=32) == "none"       # groups inside a chunk
    assert describe(64, 4128, 4096, g=32) == "none"
    assert describe(64, 4096, 4100) == "none"             # N % 8
    assert describe(64, 0, 4096) == "none"
    assert describe(32, 4096, 4096, layout=0) == "none"   # packed words at decode sizes
    assert describe(64, 4096, 4096, layout=0).endswith("repack")
    # K / 64 below eight chunks still has a plan
    assert describe(2000, 64, 512, g=64) in ("none", "kwave rows=64 nb=128 splits=1")
