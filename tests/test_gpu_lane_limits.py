"""The lane rule's choice on either side of the sizes where one lane a query takes over from groups, against 16
lanes without a presort: few and many points, each number of axes, lists that k fills and that it does not,
both tie policies.  The results are the same bits."""
import pytest
import torch

import torch_kdtree_amd as tk

pytestmark = pytest.mark.gpu
F, D = torch.float32, torch.float64

# dtype, d, points, k, tie policy, last size of the groups
_LIMITS = [
    (F, 1, 3_000, 16, "reference", 600_000), (F, 1, 50_000, 32, "lower_index", 180_000),
    (F, 2, 3_000, 8, "reference", 1_000_000), (F, 2, 50_000, 16, "reference", 450_000),
    (F, 2, 50_000, 20, "reference", 480_000), (F, 3, 9_999, 16, "lower_index", 180_000),
    (F, 3, 10_000, 16, "reference", 1_000_000), (F, 3, 9_999, 32, "reference", 200_000),
    (F, 3, 10_000, 32, "reference", 650_000), (F, 3, 60_000, 8, "reference", 1_500_000),
    (D, 2, 3_000, 16, "reference", 300_000), (D, 3, 3_000, 24, "reference", 300_000),
    (D, 3, 60_000, 8, "lower_index", 1_750_000), (D, 1, 3_000, 32, "lower_index", 1_000_000),
    (F, 8, 999, 2, "reference", 249_750), (F, 8, 4_999, 32, "reference", 1_249_750),
    (F, 8, 999, 5, "lower_index", 799_200), (D, 8, 999, 16, "reference", 49_950), (D, 8, 700, 6, "lower_index", 280_000),
]


@pytest.mark.parametrize("dtype,d,n,k,tie,last", _LIMITS)
def test_one_lane_takes_over(cuda, dtype, d, n, k, tie, last):
    g = torch.Generator(device=cuda).manual_seed(n + k)
    ref = torch.rand((n, d), generator=g, device=cuda, dtype=dtype)
    if tie == "reference":  # (some exact ties)
        ref[: n // 20] = ref[n // 20: 2 * (n // 20)]
    q = torch.rand((last + 1, d), generator=g, device=cuda, dtype=dtype)
    tree = tk.build_kd_tree(ref, levels="auto", tie_break=tie)
    tree.kdtree.set_lanes(16)
    tree.presort = "off"
    want_d, want_i = tree.query(q, nr_nns_searches=k)
    tree.kdtree.set_lanes(0)
    tree.presort = "auto"
    for nq in (last, last + 1):
        got_d, got_i = tree.query(q[:nq], nr_nns_searches=k)
        assert torch.equal(got_d, want_d[:nq]) and torch.equal(got_i, want_i[:nq]), nq


# dtype, d, points, levels, k, last size of the groups: one pair of leaves, leaves of hundreds, thousands and a few points
_LEAVES = [(F, 1, 150, 1, 1, 24_000), (F, 3, 150, 1, 8, 70_000), (F, 2, 150, 1, 32, 100_000), (D, 1, 150, 1, 16, 70_000),
           (F, 1, 64_000, 7, 4, 120_000), (F, 1, 64_000, 7, 16, 80_000), (F, 1, 64_000, 4, 1, 45_000), (D, 1, 64_000, 4, 1, 24_000),
           (F, 1, 64_000, 4, 8, 75_000), (F, 2, 64_000, 8, 8, 240_000), (F, 2, 64_000, 4, 16, 150_000),
           (F, 3, 64_000, 14, 16, 500_000), (D, 3, 64_000, 14, 8, 600_000), (F, 1, 64_000, 15, 8, 1_200_000)]


@pytest.mark.parametrize("dtype,d,n,levels,k,last", _LEAVES)
def test_one_lane_takes_over_by_leaf(cuda, dtype, d, n, levels, k, last):
    g = torch.Generator(device=cuda).manual_seed(n + levels)
    ref = torch.rand((n, d), generator=g, device=cuda, dtype=dtype)
    q = torch.rand((last + 1, d), generator=g, device=cuda, dtype=dtype)
    tree = tk.build_kd_tree(ref, levels=levels)
    tree.kdtree.set_lanes(16)
    tree.presort = "off"
    want_d, want_i = tree.query(q, nr_nns_searches=k)
    tree.kdtree.set_lanes(0)
    tree.presort = "auto"
    for nq in (last, last + 1):
        got_d, got_i = tree.query(q[:nq], nr_nns_searches=k)
        assert torch.equal(got_d, want_d[:nq]) and torch.equal(got_i, want_i[:nq]), nq
