"""The search with one lane a query, which only large calls take by themselves, asked for by name: launch
variants, the lower-index policy's lists with lanes that meet ties beside lanes that meet none, record-group boxes,
unaligned output rows, presorts, partial wavefronts and NaN rows, at every d.  Results are exact, so equality is
bit for bit, against the oracle (reference policy) and brute force (lower-index policy)."""
import numpy as np
import pytest
import torch

import oracle
import torch_kdtree_amd as tk
from torch_kdtree_amd import torch_knn
from tests._util import assert_same, gpu_query, oracle_for, with_nan_rows

pytestmark = pytest.mark.gpu


def _tree(ref, cuda, levels, tie="reference", mode=0, **kw):
    tree = tk.build_kd_tree(torch.from_numpy(ref), device=cuda, levels=levels, tie_break=tie, **kw)
    tree.kdtree.set_lanes(1)
    tree.kdtree.set_lower_list(mode)
    return tree


def _sparse_duplicates(rng, n, q, d, dtype):
    """Too few duplicated points for the upload's sample: a few lanes of a wavefront meet exact ties."""
    ref = (rng.standard_normal((n, d)) * 1e3).astype(dtype)
    dup = ref[rng.choice(n, 24, replace=False)]
    ref = np.concatenate([ref, dup])[rng.permutation(n + 24)]
    qry = (rng.standard_normal((q, d)) * 1e3).astype(dtype)
    qry[::97] = ref[rng.choice(len(ref), len(qry[::97]), replace=False)]
    qry[5:5 + 24 * 40:40] = dup
    return ref, qry


@pytest.mark.parametrize("tie,mode", [("reference", 0), ("lower_index", 0), ("lower_index", 1), ("lower_index", 2)])
@pytest.mark.parametrize("k", [5, 6, 8, 13, 16])
def test_variants_with_one_lane(cuda, tie, mode, k):
    rng = np.random.default_rng(7100 + k)
    ref, qry = _sparse_duplicates(rng, 40_000, 20_000, 3, np.float32)
    base = _tree(ref, cuda, 11, tie, mode)
    if tie == "reference":
        od, oi = oracle_for(base).search(qry, k)
        oi = base.kdtree.get_shuffled_inds()[oi]
    else:
        assert not base.kdtree.get_lower_list()[1]
        od, oi = oracle.bruteforce(ref, qry, k)
    for v in range(len(torch_knn.tree_variants())):
        tree = _tree(ref, cuda, 11, tie, mode, variant=v)
        dist, _, oidx = gpu_query(tree, qry, k, cuda)
        assert tree.kdtree.get_variant() == v
        assert_same(dist, od, "variant %d distances" % v)
        assert_same(oidx, oi.astype(np.int64), "variant %d indices" % v)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 2, 3, 8])
@pytest.mark.parametrize("levels", [9, 4])
def test_lists_and_leaves_with_one_lane(cuda, dtype, d, levels):
    """Small leaves and leaves of 375 points (record-group boxes); queries in full and partial wavefronts; NaN rows."""
    rng = np.random.default_rng(7200 + d)
    clouds = {"sparse": _sparse_duplicates(rng, 6000, 1501, d, dtype),
              "lattice": (rng.integers(0, 5, (6000, d)).astype(dtype),
                          (rng.integers(0, 5, (1501, d)) + 0.5 * rng.integers(0, 2, (1501, d))).astype(dtype))}
    for name, (ref, qry) in clouds.items():
        qry, _ = with_nan_rows(qry, rng, frac=0.02)
        refp = _tree(ref, cuda, levels)
        ot, sh = oracle_for(refp), refp.kdtree.get_shuffled_inds()
        for k in (1, 2, 4, 5, 8, 12, 16, 29, 32):
            what = "%s k %d " % (name, k)
            od, oi = ot.search(qry, k)
            dist, sidx, oidx = gpu_query(refp, qry, k, cuda)
            assert_same(dist, od, what + "distances")
            assert_same(sidx, oi, what + "structured indices")
            assert_same(oidx, sh[oi].astype(np.int64), what + "indices")
            bd, bi = oracle.bruteforce(ref, qry, k)
            for mode in (0, 1, 2):
                low = _tree(ref, cuda, levels, "lower_index", mode)
                dist, sidx, oidx = gpu_query(low, qry, k, cuda)
                assert_same(dist, bd, what + "mode %d distances" % mode)
                assert_same(oidx, bi.astype(np.int64), what + "mode %d indices" % mode)
                assert_same(low.kdtree.get_shuffled_inds()[sidx], bi, what + "mode %d structured" % mode)


@pytest.mark.parametrize("tie", ["reference", "lower_index"])
@pytest.mark.parametrize("d", [1, 2, 3, 8])
def test_unaligned_rows_and_presorts_with_one_lane(cuda, d, tie):
    rng = np.random.default_rng(7300 + d)
    ref, qry = _sparse_duplicates(rng, 20_000, 5003, d, np.float32)
    q = torch.from_numpy(qry).to(cuda)
    tree = _tree(ref, cuda, 9, tie)
    for k in (4, 8, 16, 31, 32):
        tree.presort = "off"
        d0, s0, o0 = gpu_query(tree, qry, k, cuda)
        for presort in ("auto", "morton", "leaf", "off"):
            tree.presort = presort
            bd = torch.empty(q.shape[0] * k + 1, dtype=torch.float32, device=cuda)[1:].view(-1, k)
            bi = torch.empty(q.shape[0] * k + 1, dtype=torch.int32, device=cuda)[1:].view(-1, k)
            dd, oo = tree.query(q, nr_nns_searches=k, result_dists=bd, result_idx=bi)
            assert_same(dd.cpu().numpy(), d0, "k %d %s distances" % (k, presort))
            assert_same(bi.cpu().numpy(), s0, "k %d %s structured indices" % (k, presort))
            assert_same(oo.cpu().numpy(), o0, "k %d %s indices" % (k, presort))
