"""Every form of the tree search (1, 4, 8 or 16 lanes per query) against the oracle, at the sizes where
they can go wrong: partial groups and blocks, leaves of none to several hundred points (record-group
boxes from 64), paths shorter and longer than a group, list widths at their edges, exact ties, and
queries with NaN, infinite and huge rows.  The results are exact, so equality is bit for bit."""
import numpy as np
import pytest
import torch

import oracle
import torch_kdtree_amd as tk
from tests._util import assert_same, gpu_query, nonfinite_queries, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 2, 3, 8])
@pytest.mark.parametrize("lattice", [False, True])
def test_lanes_match_oracle(cuda, dtype, d, lattice):
    rng = np.random.default_rng(4100 + d + 10 * lattice)
    # (points, levels): one point; fewer points than leaves; small leaves; 16 and 17 levels; leaves of 100 and 500
    for n, levels in ((1, 1), (37, 6), (3000, 7), (65536, 16), (70001, 17), (3200, 5), (4000, 3)):
        if lattice:  # many exact ties, queries on points
            ref = rng.integers(0, 9, (n, d)).astype(dtype)
            qry = rng.integers(-1, 10, (129, d)).astype(dtype)
        else:
            ref = (rng.standard_normal((n, d)) * 1e3).astype(dtype)
            qry = nonfinite_queries(rng, 129, d, dtype)
        tree = tk.build_kd_tree(torch.from_numpy(ref), device=cuda, levels=levels)
        low = tk.build_kd_tree(torch.from_numpy(ref), device=cuda, levels=levels, tie_break="lower_index")
        ot, sh = oracle_for(tree), tree.kdtree.get_shuffled_inds()
        for k, lanes in ((1, (1, 4, 8, 16)), (4, (4,)), (5, (1, 4, 8)), (8, (4, 8)), (9, (8, 16)), (16, (1, 8, 16)),
                         (17, (1, 16)), (32, (16,)), (33, (16,)), (64, (16,)), (65, (16,)), (128, (16,))):
            if k > n:
                continue
            od, oi = ot.search(qry, k)
            bd, bi = oracle.bruteforce(ref, qry, k)
            for ln in lanes:
                what = "n %d levels %d k %d lanes %d " % (n, levels, k, ln)
                tree.kdtree.set_lanes(ln)
                dist, sidx, oidx = gpu_query(tree, qry, k, cuda)
                assert_same(dist, od, what + "distances")
                assert_same(sidx, oi, what + "structured indices")
                assert_same(oidx, sh[oi].astype(np.int64), what + "original indices")
                low.kdtree.set_lanes(ln)
                dist, sidx, oidx = gpu_query(low, qry, k, cuda)
                assert_same(dist, bd, what + "lower-index distances")
                assert_same(oidx, bi.astype(np.int64), what + "lower-index indices")


@pytest.mark.parametrize("nq", [1, 15, 17, 24001, 100001, 700001])
def test_lanes_rule_keeps_results(cuda, nq):
    """The rule's own choice on either side of its size limits, with and without a presort, against 16
    lanes."""
    rng = np.random.default_rng(4200 + nq)
    ref = rng.random((30000, 3)).astype(np.float32)
    q = torch.from_numpy(rng.random((nq, 3)).astype(np.float32)).to(cuda)
    tree = tk.build_kd_tree(torch.from_numpy(ref), device=cuda, levels="auto")
    for k in (3, 8, 16, 20):
        tree.kdtree.set_lanes(16)
        tree.presort = "off"
        want = [t.clone() for t in tree.query(q, nr_nns_searches=k)]
        tree.kdtree.set_lanes(0)
        for presort in ("auto", "off", "leaf", "morton"):
            tree.presort = presort
            got = tree.query(q, nr_nns_searches=k)
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (k, presort)


def test_lanes_argument(cuda):
    tree = tk.build_kd_tree(torch.rand(100, 3), device=cuda)
    for bad in (-1, 2, 3, 32):
        with pytest.raises(RuntimeError):
            tree.kdtree.set_lanes(bad)
