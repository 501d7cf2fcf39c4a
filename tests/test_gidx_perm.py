"""The act-order permutation at the edges of its variants: spans of one batch held in registers
(K up to 4096, and 16384 with 16-byte loads), the two-walk spans past them, and the status from
the counting workgroup, which takes 16384 groups at a time."""

import numpy as np
import pytest
import torch

from pulsar_amd import ops

pytestmark = pytest.mark.gpu

# (K, G): K = 262160 has 16385 groups
SIZES = [(16, 16), (4096, 16), (4112, 16), (16384, 128), (16512, 128), (262144, 16), (262160, 16)]


def _g_idx(k, g, seed):
    return np.random.default_rng(seed).permutation(np.arange(k, dtype=np.int32) // g)


def _perm(g_idx, g, offset):
    k = len(g_idx)
    buf = torch.empty(k + offset, dtype=torch.int32, device="cuda")
    buf[offset:].copy_(torch.from_numpy(g_idx))
    qw = torch.zeros(k // 8, 8, dtype=torch.int32, device="cuda")
    return ops.repack_w4a16_gptq(qw, buf[offset:], g)[1]


@pytest.mark.parametrize("offset", [0, 1])  # 1: not 16-byte aligned
@pytest.mark.parametrize("k,g", SIZES)
def test_perm_is_the_stable_argsort(k, g, offset):
    gi = _g_idx(k, g, k + offset)
    want = np.argsort(gi, kind="stable").astype(np.int32)
    for _ in range(2):
        assert np.array_equal(_perm(gi, g, offset).cpu().numpy(), want)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("k,g", SIZES)
def test_bad_groupings_are_refused(k, g, offset):
    ngroups = k // g
    gi = _g_idx(k, g, k)
    for at, value in ((0, -1), (k - 1, ngroups), (k // 2, (int(gi[k // 2]) + 1) % ngroups),
                      (0, ngroups - 1 if gi[0] != ngroups - 1 else 0)):
        bad = gi.copy()
        bad[at] = value
        if np.array_equal(bad, gi):  # a single group cannot be moved to another
            continue
        with pytest.raises(RuntimeError, match="g_idx"):
            _perm(bad, g, offset)
    assert np.array_equal(_perm(gi, g, offset).cpu().numpy(), np.argsort(gi, kind="stable"))


def test_refused_under_capture():
    """The host reads the status, so the call cannot be captured: it raises before it records
    anything, and the capture around it stays whole."""
    k, g = 4096, 128
    gi = _g_idx(k, g, 3)
    qw = torch.zeros(k // 8, 64, dtype=torch.int32, device="cuda")
    t = torch.from_numpy(gi).cuda()
    x = torch.arange(64, dtype=torch.float32, device="cuda")
    ops.repack_w4a16_gptq(qw, t, g)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captured"):
            ops.repack_w4a16_gptq(qw, t, g)
        y = x * 2
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, x * 2)
    assert np.array_equal(_perm(gi, g, 0).cpu().numpy(), np.argsort(gi, kind="stable"))
