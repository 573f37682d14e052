"""autotune.tune measures the launch variants where they run: its variant queries take one lane each, whatever
the size of the call, and a tree that it does not return keeps no such choice."""
import pytest
import torch

from torch_kdtree_amd import autotune, nn_distance

pytestmark = pytest.mark.gpu


class _Spy:
    """A tree handle that notes the lanes and variant set when a query runs."""

    def __init__(self, tree, log):
        self._tree, self._log, self._lanes, self._variant = tree, log, 0, 0

    def set_lanes(self, lanes):
        self._lanes = lanes
        self._tree.set_lanes(lanes)

    def set_variant(self, variant):
        self._variant = variant
        self._tree.set_variant(variant)

    def query(self, *args, **kwargs):
        self._log.append((self._lanes, self._variant))
        return self._tree.query(*args, **kwargs)

    def __getattr__(self, name):
        return getattr(self._tree, name)


@pytest.mark.parametrize("tie", ["reference", "lower_index"])
def test_variants_are_timed_with_one_lane(cuda, tmp_path, monkeypatch, tie):
    monkeypatch.setenv("TORCH_KDTREE_AMD_TUNING", str(tmp_path / "tuning.json"))
    log = []
    init = nn_distance.TorchKDTree.__init__

    def spied(self, *args, **kwargs):
        init(self, *args, **kwargs)
        self.kdtree = _Spy(self.kdtree, log)

    monkeypatch.setattr(nn_distance.TorchKDTree, "__init__", spied)
    g = torch.Generator(device=cuda).manual_seed(5)
    ref, qry = (torch.rand((n, 3), generator=g, device=cuda) for n in (50_000, 20_000))
    out = autotune.tune(ref, qry, 12, leaf_sizes=(32,), repeats=1, tie_break=tie)
    variants = sorted(out["measured_variants"])
    assert len(variants) > 1
    for v in variants[1:]:
        assert (1, v) in log and all(lanes == 1 for lanes, w in log if w == v), log
    assert (1, 0) in log
