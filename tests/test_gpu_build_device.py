"""A tree that the GPU build left on the GPU against the same tree written to a file, loaded and uploaded
from the host: structured points, index maps, nodes, the choice of the lower-index list, and query
results under both policies.  Sizes around the node sort in LDS (nodes of at most 4,096 points), leaves
of 0 to 2, 16, 64 and more points (record-group boxes from 64), and one leaf pair of everything; with
ties, repeated points, and infinite coordinates."""
import numpy as np
import pytest
import torch

import oracle
import torch_kdtree_amd as tk
from tests._util import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 2, 3, 8])
@pytest.mark.parametrize("kind", ["normal", "lattice", "repeated", "inf"])
def test_device_tree_equals_uploaded_tree(cuda, tmp_path, dtype, d, kind):
    rng = np.random.default_rng(5100 + d)
    for n, levels in ((1, 1), (3, 2), (2047, 11), (2049, 3), (4096, 12), (4097, 1), (20_000, 8), (70_001, 6)):
        pts = (rng.standard_normal((n, d)) * 1e3).astype(dtype)
        if kind == "lattice":
            pts = rng.integers(-9, 10, (n, d)).astype(dtype)
        elif kind == "repeated":
            pts[n // 2:] = pts[:n - n // 2]
        elif kind == "inf":
            pts[n // 3, d - 1] = np.inf
        built = tk.build_kd_tree(torch.from_numpy(pts), device=cuda, levels=levels, builder="gpu")
        path = str(tmp_path / "t.bin")
        built.save(path)
        loaded = tk.load_kd_tree(path, device=cuda)
        what = "n %d levels %d " % (n, levels)
        assert built.kdtree.is_finite() == loaded.kdtree.is_finite() == bool(np.isfinite(pts).all())
        assert built.kdtree.get_lower_list() == loaded.kdtree.get_lower_list(), what
        assert torch.equal(built.structured_points, loaded.structured_points), what
        assert torch.equal(built.shuffled_ind, loaded.shuffled_ind), what
        assert_same(built.structured_points.cpu().numpy(), built.kdtree.get_structured_points(), what + "points")
        assert_same(built.structured_points.cpu().numpy(), pts[built.shuffled_ind.cpu().numpy()], what + "indices")
        q_np = np.concatenate([pts[:60], (rng.standard_normal((60, d)) * 1e3).astype(dtype)])
        q = torch.from_numpy(q_np).to(cuda)
        for k in (1, 16, 40):
            if k > n:
                continue
            for tie in ("reference", "lower_index"):
                built.tie_break = loaded.tie_break = tie
                db, ib = built.query(q, nr_nns_searches=k)
                dl, il = loaded.query(q, nr_nns_searches=k)
                assert_same(db.cpu().numpy(), dl.cpu().numpy(), what + "k %d %s distances" % (k, tie))
                assert torch.equal(ib, il), (what, k, tie)
            bd, bi = oracle.bruteforce(pts, q_np, k)
            assert_same(ib.cpu().numpy(), bi.astype(np.int64), what + "k %d brute force" % k)
