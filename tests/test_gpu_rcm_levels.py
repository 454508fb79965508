"""Sizes where the ordering's walk and the relabelling change paths: levels above one work-group's
8192 edges, children sorted by a lane (up to 64), in LDS and in memory (8192), a wave's children
beyond its 512 staged, adjacency lists cut into segments of 512 (with a vertex of more than 2048
neighbours), and rows sorted by a wave (64), by a work-group (4096) or by keys."""
import numpy as np
import pytest

import vcsr_mc_amd as vm
from golden_io import csr_from_edges
from gpu_util import dev, say
from test_gpu_rcm import gpu_apply, gpu_rcm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    (10, 16, 17, 63, 64, 65, 300, 511, 512, 513, 9000),
    (1, 8190, 8191, 8192, 8193, 8194, 2),
    tuple([0, 70, 0, 600, 3] * 40),
    (60000, 66, 5),
    (2045, 2046, 2047, 2048, 511, 512, 513, 1),
    (2049, 1023, 1024, 1025, 510, 0, 64, 65, 4095, 4096, 4097),
    tuple([2500, 0, 1, 700] * 12),
])
def test_hub_levels(orc, sizes):
    """A centre joined to hubs with the given numbers of leaves, the leaves with 0 to 5 pendant
    vertices each (many equal degrees), in a random numbering, beside a second component."""
    rng = np.random.default_rng(sum(sizes))
    edges, n = [], 1 + len(sizes)
    for h, k in enumerate(sizes):
        edges.append((0, 1 + h))
        for leaf in range(n, n + k):
            edges.append((1 + h, leaf))
        n += k
    pend = rng.integers(0, 6, n)
    pend[:1 + len(sizes)] = 0
    src = np.repeat(np.arange(n), pend)
    dst = n + np.arange(src.size)
    n += src.size
    e = np.concatenate([np.array(edges, np.int64), np.stack([src, dst], 1),
                        np.array([[n, n + 1], [n + 1, n + 2]])])
    n += 3
    e = rng.permutation(n)[e]
    e = e[rng.permutation(len(e))]
    rp, col = csr_from_edges(n, n, [tuple(x) for x in e])
    say("hub levels", sizes[:4], n, col.size)
    assert np.array_equal(gpu_rcm(rp, col, n, n), orc.rcm_order(rp, col, n, n))


@pytest.mark.parametrize("hubs,n,spread", [(1, 70000, 1), (4, 40000, 1), (30, 20000, 40),
                                           (3, 100000, 2000), (200, 30000, 7)])
def test_shared_hubs(orc, hubs, n, spread):
    """Hubs joined to most vertices, which all compete for them: lists cut into segments, groups split
    in several passes and, with degrees that lie far apart (`spread`), in parts of unlike sizes."""
    rng = np.random.default_rng(hubs * 7 + spread)
    e = []
    for k in range(hubs):
        leaves = rng.choice(n, int(n * rng.uniform(0.3, 1.0)), replace=False)
        e.append(np.stack([np.full(leaves.size, k), leaves], 1))
    # edges among the leaves, their number falling off steeply from vertex to vertex
    k = np.minimum(spread, (spread / (1 + rng.permutation(n) % 997)).astype(np.int64))
    src = np.repeat(np.arange(n), k)
    e.append(np.stack([src, rng.integers(0, n, src.size)], 1))
    e = np.concatenate(e)
    key = np.unique(rng.permutation(n)[e] @ np.array([n, 1]))
    rp = np.searchsorted(key, n * np.arange(n + 1)).astype(np.int32)
    col = (key % n).astype(np.int32)
    say("shared hubs", hubs, n, spread, col.size)
    assert np.array_equal(gpu_rcm(rp, col, n, n), orc.rcm_order(rp, col, n, n))


@pytest.mark.parametrize("longest", [64, 65, 4096, 4097])
@pytest.mark.parametrize("O", [7, 8])
def test_relabel_row_lengths(longest, O):
    """Rows of 0, 1, 63 .. 65 and `longest` nonzeros in any column order, against numpy; then the
    same with one column repeated in the longest row, which is refused and changes nothing."""
    rng = np.random.default_rng(longest)
    N = 6000
    lens = [0, 1, 63, min(64, longest), min(65, longest), 2, longest, 0, 129 if longest > 129 else 3]
    rp = np.zeros(len(lens) + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    col = np.concatenate([rng.choice(N, k, replace=False) for k in lens]).astype(np.int32)
    val = rng.uniform(-1, 1, col.size).astype(np.float32)
    pos = rng.permutation(N).astype(np.int32)
    B = rng.uniform(-1, 1, (N, O)).astype(np.float32)
    say("relabel rows", longest, O)
    c2, v2, B2 = gpu_apply(rp, col, val, len(lens), N, pos, B, O)
    for r in range(len(lens)):
        s = slice(rp[r], rp[r + 1])
        at = np.argsort(pos[col[s]], kind="stable")
        assert np.array_equal(c2[s], pos[col[s]][at]) and np.array_equal(v2[s], val[s][at]), r
    want = np.empty_like(B)
    want[pos] = B
    assert np.array_equal(B2, want)
    bad = col.copy()
    bad[rp[7] - 1] = bad[rp[6]]
    dc, dv = dev(bad), dev(val)
    with pytest.raises(vm.VCSRMCError) as e:
        vm.apply_column_permutation_device(dev(rp), dc, dv, len(lens), N, dev(pos))
    assert e.value.status == vm.ERR_UNSORTED
    assert np.array_equal(dc.cpu().numpy(), bad) and np.array_equal(dv.cpu().numpy(), val)
