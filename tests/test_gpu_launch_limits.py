"""Calls whose lanes or words together would pass the 2^32 threads of one launch."""
import numpy as np
import pytest
import torch

import oracle
import torch_kdtree_amd as tk
from tests._util import assert_same

pytestmark = pytest.mark.gpu


def test_group_search_of_more_than_2_28_queries(cuda):
    """d = 8, 16 lanes a query: rows at the start, around the slices' borders and at the end."""
    n = (1 << 28) + 3000
    rng = np.random.default_rng(2808)
    ref = rng.standard_normal((300, 8)).astype(np.float32)
    tree = tk.build_kd_tree(torch.from_numpy(ref), device=cuda, levels=5)
    q = torch.randn((n, 8), generator=torch.Generator(device=cuda).manual_seed(8), device=cuda)
    dist, inds = tree.query(q, nr_nns_searches=1)
    picks = np.unique(np.concatenate([np.arange(b - 300, b + 300) for b in (300, 1 << 27, 1 << 28, n - 300)]))
    sel = torch.from_numpy(picks).to(cuda)
    qs, got_d, got_i = q[sel].cpu().numpy(), dist[sel].cpu().numpy(), inds[sel].cpu().numpy()
    del q, dist, inds
    torch.cuda.empty_cache()
    od, oi = oracle.OracleTree(ref, 5).search(qs, 1)
    assert_same(got_d, od, "distances")
    assert_same(got_i, tree.kdtree.get_shuffled_inds()[oi].astype(np.int64), "indices")


def test_device_tree_of_2_32_coordinate_words(cuda):
    """The largest GPU build in the widest records (2^28 points of 8 doubles): its structured points and
    indices come from the device tree, one word of 2^32 after the other."""
    n, levels = 1 << 28, 4
    if torch.cuda.mem_get_info()[0] < (120 << 30):
        pytest.skip("needs 120 GB of GPU memory")
    ref = torch.rand((n, 8), dtype=torch.float64, generator=torch.Generator(device=cuda).manual_seed(9), device=cuda)
    tree = tk.build_kd_tree(ref, levels=levels, builder="gpu")
    seen = torch.zeros(n, dtype=torch.bool, device=cuda)
    for s in range(0, n, 1 << 24):
        idx = tree.shuffled_ind[s:s + (1 << 24)]
        assert torch.equal(tree.structured_points[s:s + (1 << 24)], ref[idx]), s
        seen[idx] = True
    assert bool(seen.all())
    del ref, tree, seen, idx
    torch.cuda.empty_cache()
