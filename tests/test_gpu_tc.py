"""GPU parity of triangle counting: vertexmap, per-vertex counts and total
bit-exact vs the reference's trianglecounting output (golden) and the oracle."""
import numpy as np
import pytest

import graphs
import oracle

pytestmark = pytest.mark.gpu


def run_tc(dev, src, dst, n):
    prep = dev.TrianglePrep(dev.to_dev_u32(src), dev.to_dev_u32(dst), n)
    pv, tot, ovf = prep.count()
    return prep, dev.to_host_u32(pv, n), int(tot.item()), int(ovf.item())


@pytest.mark.parametrize("case", graphs.TC_CASES, ids=[c["name"] for c in graphs.TC_CASES])
def test_tc_vs_reference_golden(dev, manifest, golden, case):
    src, dst, n = graphs.make(case)
    prep, pv, tot, ovf = run_tc(dev, src, dst, n)
    assert ovf == 0
    g = manifest[case["name"]]
    assert tot == g["total"]
    np.testing.assert_array_equal(dev.to_host_u32(prep.vertexmap, n), golden[f"{case['name']}__vertexmap"])
    np.testing.assert_array_equal(pv, golden[f"{case['name']}__tc_pervertex"])


def test_tc_duplicates_and_reciprocal_edges(dev):
    # the same triangle given with reversed and repeated edges counts once
    src = np.array([0, 1, 2, 1, 0, 2, 3], np.uint32)
    dst = np.array([1, 2, 0, 0, 2, 1, 3], np.uint32)
    prep, pv, tot, ovf = run_tc(dev, src, dst, 4)
    assert tot == 1 and prep.noriented == 3
    vm = dev.to_host_u32(prep.vertexmap, 4)
    for v in range(3):
        assert pv[vm[v]] == 1
    assert pv[vm[3]] == 0


def test_tc_lists_of_the_core(dev):
    # K_1100: oriented lists of up to 1,099 entries, all in the core (lists as long
    # outside it: test_tc_rows_long_outside_the_core; without a core:
    # test_tc_count_noalloc_complete_graphs)
    n = 1100
    a, b = np.triu_indices(n, 1)
    prep, pv, tot, ovf = run_tc(dev, a.astype(np.uint32), b.astype(np.uint32), n)
    assert tot == n * (n - 1) * (n - 2) // 6
    assert (pv == (n - 1) * (n - 2) // 2).all()


def test_tc_scale21_vs_oracle(dev):
    """The TC workload: simple undirected R-MAT scale 21 (edge factor 16, seed 4)."""
    case = {"name": "tc_rmat21", "rmat": (21, 16, 4), "simple": True}
    src, dst, n = graphs.make(case)
    prep, pv, tot, ovf = run_tc(dev, src, dst, n)
    vm, opv, otot = oracle.triangles(n, src, dst)
    print(f"\nscale21 TC: N={n} E={len(src)} oriented={prep.noriented} triangles={otot}")
    assert tot == otot
    np.testing.assert_array_equal(dev.to_host_u32(prep.vertexmap, n), vm)
    np.testing.assert_array_equal(pv, opv)


@pytest.mark.parametrize("n", [3, 65, 66, 129, 131, 1500, 4097, 4200])
def test_tc_complete_graphs(dev, n):
    """K_n around the sizes of the counting kernels: rows of 64 and 65 core
    entries (list / bitmap), a core smaller than, equal to and larger than the
    4096 highest ranks, more bitmaps per wavefront than its bit planes hold."""
    a, b = np.triu_indices(n, 1)
    prep, pv, tot, ovf = run_tc(dev, a.astype(np.uint32), b.astype(np.uint32), n)
    assert ovf == 0 and tot == n * (n - 1) * (n - 2) // 6
    assert (pv == (n - 1) * (n - 2) // 2).all()


@pytest.mark.parametrize("n,hubs,p,extra", [(5000, 200, 0.9, 40000), (17000, 700, 0.5, 60000),
                                            (40000, 4200, 0.05, 200000), (150000, 300, 0.7, 500000)])
def test_tc_core_and_tail_vs_oracle(dev, n, hubs, p, extra):
    """Dense hubs, random edges to them and a sparse rest: triangles with none,
    one, two and all vertices in the core, bitmapped and listed rows, credits
    counted in LDS and in global memory; the same counts from the form without
    a workspace (no core kernel)."""
    import torch
    rng = np.random.default_rng(n)
    a, b = np.triu_indices(hubs, 1)
    k = rng.random(len(a)) < p
    s = [a[k], rng.integers(0, hubs, extra), rng.integers(0, n, extra)]
    d = [b[k], rng.integers(0, n, extra), rng.integers(0, n, extra)]
    base = rng.integers(0, n - 3, 5000)  # triangles of the tail
    s += [base, base, base + 1]
    d += [base + 1, base + 2, base + 2]
    ids = rng.permutation(n)
    s, d = ids[np.concatenate(s)], ids[np.concatenate(d)]
    src, dst = graphs.preprocess(s, d, simple=True)
    prep, pv, tot, ovf = run_tc(dev, src, dst, n)
    vm, opv, otot = oracle.triangles(n, src, dst)
    assert tot == otot and ovf == 0
    np.testing.assert_array_equal(pv, opv)
    q = dev.empty_u32(n)
    t2 = torch.zeros(1, dtype=torch.int64, device="cuda")
    o2 = torch.zeros(1, dtype=torch.int32, device="cuda")
    dev.check(dev.lib().gchi_tc_count_noalloc(dev.dptr(prep.off), dev.dptr(prep.adj), n, dev.dptr(q), dev.dptr(t2),
                                              dev.dptr(o2), dev.stream()), "tc_count_noalloc")
    assert int(t2.item()) == otot
    np.testing.assert_array_equal(dev.to_host_u32(q, n), opv)


@pytest.mark.parametrize("n", [31, 32, 63, 64, 65, 95, 96, 100, 127, 128])
def test_tc_workgroups_of_small_graphs(dev, n):
    """Vertex counts around one, two and three workgroups of the core kernel, whose
    workspace holds a block of credits for each."""
    import ctypes
    a, b = np.triu_indices(n, 1)
    prep, pv, tot, ovf = run_tc(dev, a.astype(np.uint32), b.astype(np.uint32), n)
    assert ovf == 0 and tot == n * (n - 1) * (n - 2) // 6
    assert (pv == (n - 1) * (n - 2) // 2).all()
    nb = ctypes.c_size_t()
    dev.check(dev.lib().gchi_tc_count_workspace(n, ctypes.byref(nb)))
    assert nb.value >= max(1, n // 32) * 65536


def test_tc_rows_long_outside_the_core(dev):
    """K_5150: 1,054 vertices below the 4,096 of the core, whose rows hold up to
    1,053 entries outside it, so the tail, hash and search kernels all count
    beside the core kernel."""
    n, core = 5150, 4096
    a, b = np.triu_indices(n, 1)
    prep, pv, tot, ovf = run_tc(dev, a.astype(np.uint32), b.astype(np.uint32), n)
    adj, off = dev.to_host_u32(prep.adj, prep.noriented), dev.to_host_u32(prep.off, n + 1).astype(np.int64)
    outside = np.add.reduceat(adj < n - core, off[:-2])  # the last vertex has no row
    assert (outside > 1024).any() and ((outside > 512) & (outside <= 1024)).any()
    assert (outside[outside > 0] <= 512).any()
    assert ovf == 0 and tot == n * (n - 1) * (n - 2) // 6
    assert (pv == (n - 1) * (n - 2) // 2).all()


def test_tc_long_core_rows_below_the_bitmaps(dev):
    """40,000 vertices with 70 to 130 edges each into 4,000 hubs and some among
    themselves: vertices below the 16,384 bitmapped ranks whose rows hold more than
    64 core entries, walked entry by entry against a's bitmap."""
    import torch
    n, hubs, rows, core = 40000, 4000, 16384, 4096
    rng = np.random.default_rng(40000)
    low = np.arange(hubs, n)
    deg = rng.integers(70, 131, len(low))
    s = [np.repeat(low, deg), rng.integers(hubs, n, 80000)]
    d = [rng.integers(0, hubs, int(deg.sum())), rng.integers(hubs, n, 80000)]
    ids = rng.permutation(n)
    src, dst = graphs.preprocess(ids[np.concatenate(s)], ids[np.concatenate(d)], simple=True)
    prep, pv, tot, ovf = run_tc(dev, src, dst, n)
    adj, off = dev.to_host_u32(prep.adj, prep.noriented), dev.to_host_u32(prep.off, n + 1).astype(np.int64)
    entries = np.concatenate([[0], np.cumsum(adj >= n - core)])
    long_rows = (entries[off[1:]] - entries[off[:-1]] > 64) & (np.arange(n) < n - rows)
    assert long_rows[adj].sum() > 10000  # such a row is the b of a pair that often
    vm, opv, otot = oracle.triangles(n, src, dst)
    assert tot == otot and ovf == 0
    np.testing.assert_array_equal(pv, opv)
    q = dev.empty_u32(n)
    t2 = torch.zeros(1, dtype=torch.int64, device="cuda")
    o2 = torch.zeros(1, dtype=torch.int32, device="cuda")
    dev.check(dev.lib().gchi_tc_count_noalloc(dev.dptr(prep.off), dev.dptr(prep.adj), n, dev.dptr(q), dev.dptr(t2),
                                              dev.dptr(o2), dev.stream()), "tc_count_noalloc")
    assert int(t2.item()) == otot
    np.testing.assert_array_equal(dev.to_host_u32(q, n), opv)
