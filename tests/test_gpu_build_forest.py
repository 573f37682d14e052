"""Forests whose trees leave the sorts over the whole array at different depths: big clouds beside small ones,
down to leaves of one point and none.  Every tree equals the one that the single build makes of its cloud."""
import numpy as np
import pytest
import torch

import torch_kdtree_amd as tk
from tests._util import assert_same

pytestmark = pytest.mark.gpu


def _forest_equals_single_builds(cuda, clouds, levels, check):
    dtype = clouds[0].dtype
    batch = tk.build_kd_tree_batch([torch.from_numpy(c).to(cuda) for c in clouds], device=cuda, levels=levels,
                                   builder="gpu")
    picked = [clouds[c][:40] for c in range(len(clouds))]
    dists, inds = batch.query([torch.from_numpy(p).to(cuda) for p in picked], [min(5, len(c)) for c in clouds])
    for c in check:
        one = tk.build_kd_tree(torch.from_numpy(clouds[c]), device=cuda, levels=levels[c], builder="gpu")
        d, i = one.query(torch.from_numpy(picked[c]).to(cuda), nr_nns_searches=min(5, len(clouds[c])))
        what = "cloud %d (%d points, %d levels, %s) " % (c, len(clouds[c]), levels[c], dtype)
        assert_same(dists[c].cpu().numpy(), d.cpu().numpy(), what + "distances")
        assert_same(inds[c].cpu().numpy(), i.cpu().numpy(), what + "indices")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 3, 8])
@pytest.mark.parametrize("lattice", [False, True])
def test_small_clouds_beside_big_ones(cuda, dtype, d, lattice):
    rng = np.random.default_rng(5200 + d)
    # (points, levels): tails from depth 5, 0 (of 1 to 4,096 points), 1 and 3, and one tree without a tail
    shapes = ((70_001, 12), (1, 1), (2, 2), (3, 2), (4, 3), (37, 6), (255, 8), (256, 9), (257, 9), (2048, 12), (4096, 13),
              (4097, 13), (20_000, 15), (30_000, 2))
    clouds = [(rng.integers(0, 9, (n, d)) if lattice else rng.standard_normal((n, d)) * 1e3).astype(dtype)
              for n, _ in shapes]
    _forest_equals_single_builds(cuda, clouds, [lv for _, lv in shapes], range(len(shapes)))


def test_more_tail_nodes_than_one_launch_would_take(cuda):
    """A cloud of 2^24 points and 1,024 of 4,096 points in leaves of one and none: taken to the big cloud's
    depth, the small ones' 2^22 nodes with a workgroup each would be a launch of 2^32 threads."""
    rng = np.random.default_rng(5300)
    clouds = [rng.random((1 << 24, 1), dtype=np.float32)] + [rng.random((4096, 1), dtype=np.float32) for _ in range(1024)]
    _forest_equals_single_builds(cuda, clouds, [13] + [13] * 1024, (1, 513, 1024))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,levels", [(4095, 5), (8191, 4), (8192, 4), (8193, 4), (8193, 14), (16_383, 3), (16_385, 6)])
def test_nodes_around_the_workgroup_size(cuda, dtype, n, levels):
    """Nodes of just under, exactly and just over 4,096 points, which one workgroup sorts to the leaves: the tree is
    the host build's, point by point (no two coordinates are equal)."""
    rng = np.random.default_rng(n + levels)
    pts = np.stack([rng.permutation(n) for _ in range(3)], axis=1).astype(dtype)
    host = tk.build_kd_tree(torch.from_numpy(pts), device="cpu", levels=levels)
    built = tk.build_kd_tree(torch.from_numpy(pts), device=cuda, levels=levels, builder="gpu")
    assert_same(built.structured_points.cpu().numpy(), host.structured_points.numpy(), "structured points")
    assert_same(built.shuffled_ind.cpu().numpy(), host.shuffled_ind.numpy(), "indices")
    for a, b, what in zip(built.kdtree.get_nodes(), host.kdtree.get_nodes(), ("axis", "split", "leaf offsets")):
        assert_same(a, b, what)
