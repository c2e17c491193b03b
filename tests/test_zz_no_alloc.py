"""gchi_tc_count_noalloc: triangle counting with no workspace and no
allocation (its counters live in a library-owned device array).  Called
through the C ABI and checked against gchi_tc_count on the same oriented
adjacency, bit-exact, on two calls in a row with the second input smaller
(the shared array keeps the first call's counts, which must not leak into the
second); sizes beyond the array's limit are refused."""
import ctypes

import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu


def _prep(dev, scale, ef, seed):
    s, d = graphs.rmat_pairs(scale, ef, seed)
    keep = s != d
    a, b = np.minimum(s[keep], d[keep]), np.maximum(s[keep], d[keep])
    key = np.unique((a.astype(np.uint64) << np.uint64(32)) | b.astype(np.uint64))
    hs = (key >> np.uint64(32)).astype(np.uint32)
    hd = (key & np.uint64(0xffffffff)).astype(np.uint32)
    n = int(max(hs.max(), hd.max())) + 1
    return dev.TrianglePrep(dev.to_dev_u32(hs), dev.to_dev_u32(hd), n), n


def _noalloc(dev, prep, n):
    import torch
    pv = dev.empty_u32(n)
    tot = torch.zeros(1, dtype=torch.int64, device="cuda")
    ovf = torch.zeros(1, dtype=torch.int32, device="cuda")
    dev.check(dev.lib().gchi_tc_count_noalloc(dev.dptr(prep.off), dev.dptr(prep.adj), n, dev.dptr(pv), dev.dptr(tot),
                                              dev.dptr(ovf), dev.stream()), "tc_count_noalloc")
    return pv, tot, ovf


def test_tc_count_noalloc_equals_workspace_form(dev):
    big, nb = _prep(dev, 16, 16, 4)
    small, ns = _prep(dev, 11, 8, 6)
    assert ns < nb
    for prep, n in ((big, nb), (small, ns)):
        pv_w, tot_w, ovf_w = prep.count()
        pv_n, tot_n, ovf_n = _noalloc(dev, prep, n)
        np.testing.assert_array_equal(dev.to_host_u32(pv_n, n), dev.to_host_u32(pv_w, n))
        assert int(tot_n.item()) == int(tot_w.item()) > 0
        assert int(ovf_n.item()) == int(ovf_w.item()) == 0
    # again on the big graph after the small one: the same counts
    pv_n, tot_n, _ = _noalloc(dev, big, nb)
    pv_w, tot_w, _ = big.count()
    np.testing.assert_array_equal(dev.to_host_u32(pv_n, nb), dev.to_host_u32(pv_w, nb))
    assert int(tot_n.item()) == int(tot_w.item())


@pytest.mark.parametrize("n", [64, 65, 66, 512, 513, 514, 600, 1024, 1025, 1026, 1100])
def test_tc_count_noalloc_complete_graphs(dev, n):
    """K_n: rows of every length up to n - 1, around the lines between the tail
    kernel (up to 64 entries here), the hash kernel (up to 1024) and the search
    kernel, whose longer rows do not fit its LDS stage."""
    a, b = np.triu_indices(n, 1)
    prep = dev.TrianglePrep(dev.to_dev_u32(a.astype(np.uint32)), dev.to_dev_u32(b.astype(np.uint32)), n)
    rows = np.diff(dev.to_host_u32(prep.off, n + 1).astype(np.int64))
    assert rows.max() == n - 1
    pv, tot, ovf = _noalloc(dev, prep, n)
    assert int(tot.item()) == n * (n - 1) * (n - 2) // 6 and int(ovf.item()) == 0
    assert (dev.to_host_u32(pv, n) == (n - 1) * (n - 2) // 2).all()


def test_tc_count_noalloc_dense_rows_are_not_searched(dev):
    """36M pairs in rows of up to 599 entries take about a millisecond through the
    hash kernel; searched one by one they took 225."""
    import time

    import torch
    n = 600
    a, b = np.triu_indices(n, 1)
    prep = dev.TrianglePrep(dev.to_dev_u32(a.astype(np.uint32)), dev.to_dev_u32(b.astype(np.uint32)), n)
    best = 1.0
    for _ in range(3):
        torch.cuda.synchronize()
        t = time.perf_counter()
        _noalloc(dev, prep, n)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    assert best < 0.03


def test_tc_count_noalloc_refuses_oversize(dev):
    L = dev.lib()
    one = ctypes.c_void_p(1)
    assert L.gchi_tc_count_noalloc(one, one, (1 << 22) + 1, one, one, one, None) == -1
    buf = ctypes.create_string_buffer(256)
    L.gchi_last_error(buf, 256)
    assert b"GCHI_TC_NOALLOC_MAX_VERTICES" in buf.value
