"""The first getter of a tree that the GPU build left on the GPU, which fills its host arrays."""
import threading

import numpy as np
import pytest
import torch

import torch_kdtree_amd as tk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tie", ["reference", "lower_index"])
def test_first_getter_beside_queries(cuda, tie):
    """Several threads query, each on its own stream, while others ask for the host arrays."""
    g = torch.Generator(device=cuda).manual_seed(4)
    ref = torch.rand((200_000, 3), generator=g, device=cuda)
    q = torch.rand((2_000, 3), generator=g, device=cuda)
    tree = tk.build_kd_tree(ref, builder="gpu", tie_break=tie)
    want = tree.query(q, nr_nns_searches=6)
    points = tree.structured_points.cpu().numpy()
    torch.cuda.synchronize()
    go, errors = threading.Barrier(6), []

    def queries():
        try:
            stream = torch.cuda.Stream()
            go.wait()
            with torch.cuda.stream(stream):
                outs = [tree.query(q, nr_nns_searches=6) for _ in range(50)]
            stream.synchronize()
            assert all(torch.equal(a, b) for o in outs for a, b in zip(o, want))
        except Exception as e:  # noqa: BLE001 - reported by the test's own thread
            errors.append(e)

    def getter():
        try:
            go.wait()
            assert np.array_equal(tree.kdtree.get_structured_points(), points)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=f) for f in (queries,) * 4 + (getter,) * 2]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("getter", ["get_structured_points", "get_nodes", "save"])
def test_first_getter_during_a_capture(cuda, tmp_path, getter):
    """A stream is being captured meanwhile: the capture goes on, and the captured query replays."""
    g = torch.Generator(device=cuda).manual_seed(3)
    ref = torch.rand((20_000, 3), generator=g, device=cuda)
    q = torch.rand((500, 3), generator=g, device=cuda)
    tree = tk.build_kd_tree(ref, builder="gpu")
    want_d, want_i = tree.query(q, nr_nns_searches=4)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        d, i = tree.query(q, nr_nns_searches=4)
        if getter == "save":
            tree.kdtree.save(str(tmp_path / "t.bin"))
        else:
            got = getattr(tree.kdtree, getter)()
    for _ in range(3):
        d.fill_(-1)
        i.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(d, want_d) and torch.equal(i, want_i)
    points = tree.structured_points.cpu().numpy()
    if getter == "save":
        loaded = tk.load_kd_tree(str(tmp_path / "t.bin"))
        assert np.array_equal(loaded.structured_points.numpy(), points)
    elif getter == "get_structured_points":
        assert np.array_equal(got, points)
    else:
        assert got[2][0] == 0 and got[2][-1] == 20_000
