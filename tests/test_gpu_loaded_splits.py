"""A tree image whose split values do not bound their points (no build makes one; its checksum is right, so it
loads): GPU queries under the reference policy follow the reference's walk, as the host search does."""
import struct

import numpy as np
import pytest
import torch

import torch_kdtree_amd as tk

pytestmark = pytest.mark.gpu
_HEADER = 8 + 4 * 4 + 8


def _fnv1a(data):
    h = 1469598103934665603
    for b in data:
        h = ((h ^ b) * 1099511628211) & 0xffffffffffffffff
    return h


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("moved", [0.0, 0.05])
def test_splits_off_their_points(cuda, tmp_path, dtype, moved):
    rng = np.random.default_rng(17)
    ref, qry = rng.random((900, 3)).astype(dtype), torch.from_numpy(rng.random((300, 3)).astype(dtype))
    levels, path = 5, str(tmp_path / "tree.bin")
    tk.build_kd_tree(torch.from_numpy(ref), levels=levels).save(path)
    data = bytearray(open(path, "rb").read())
    n = (1 << levels) - 1
    split = np.frombuffer(bytes(data[_HEADER:_HEADER + n * ref.itemsize]), dtype=dtype)
    split = (split + moved * rng.uniform(-1, 1, n)).astype(dtype)
    data[_HEADER:_HEADER + n * ref.itemsize] = split.tobytes()
    data[-8:] = struct.pack("<Q", _fnv1a(data[:-8]))
    open(path, "wb").write(data)
    host, gpu = tk.load_kd_tree(path, device="cpu"), tk.load_kd_tree(path, device=cuda)
    for k in (1, 5, 16, 40):
        want_d, want_i = host.query(qry, nr_nns_searches=k)
        for lanes in (0, 1, 16):
            gpu.kdtree.set_lanes(lanes)
            got_d, got_i = gpu.query(qry.to(cuda), nr_nns_searches=k)
            assert torch.equal(got_d.cpu(), want_d) and torch.equal(got_i.cpu(), want_i), (k, lanes)
