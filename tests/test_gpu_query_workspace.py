"""A caller's own workspace of tk_knn_query_gpu: the size that tk_knn_query_gpu_workspace names serves every k, and
one byte less is refused, also for a k whose search takes no presort at that size."""
import ctypes
import os

import pytest
import torch

import torch_kdtree_amd as tk

pytestmark = pytest.mark.gpu
_LIB = os.path.join(os.path.dirname(os.path.abspath(tk.__file__)), "libtorch_kdtree_amd.so")


@pytest.mark.parametrize("d", [3, 8])
@pytest.mark.parametrize("nq", [4_096, 50_000, 800_000])
def test_workspace_size(cuda, d, nq):
    lib, vp, sz = ctypes.CDLL(_LIB), ctypes.c_void_p, ctypes.c_size_t
    lib.tk_last_error.restype = ctypes.c_char_p
    lib.tk_tree_build.argtypes = [vp, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, vp]
    lib.tk_tree_upload.argtypes, lib.tk_tree_free.argtypes, lib.tk_tree_free.restype = [vp, ctypes.c_int], [vp], None
    lib.tk_knn_query_gpu.argtypes = [vp, vp, ctypes.c_int64, ctypes.c_int, vp, vp, vp, ctypes.c_int, ctypes.c_int, vp, sz, vp]
    lib.tk_knn_query_gpu_workspace.argtypes = [vp, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int, vp]
    ref = torch.rand((20_000, d), generator=torch.Generator().manual_seed(d))
    q = torch.rand((nq, d), generator=torch.Generator(device=cuda).manual_seed(nq), device=cuda)
    tree, need = vp(), sz()
    assert lib.tk_tree_build(ref.data_ptr(), 20_000, d, 0, 9, 0, ctypes.byref(tree)) == 0, lib.tk_last_error()
    try:
        assert lib.tk_tree_upload(tree, 0) == 0, lib.tk_last_error()
        stream = torch.cuda.current_stream().cuda_stream
        for k in (1, 8, 16, 33):
            assert lib.tk_knn_query_gpu_workspace(tree, nq, k, 0, -1, ctypes.byref(need)) == 0
            assert need.value > 0
            outs = []
            for ws_bytes in (None, need.value):
                out = (torch.empty((nq, k), device=cuda), torch.empty((nq, k), dtype=torch.int32, device=cuda),
                       torch.empty((nq, k), dtype=torch.int64, device=cuda))
                ws = torch.empty(ws_bytes or 0, dtype=torch.uint8, device=cuda)
                rc = lib.tk_knn_query_gpu(tree, q.data_ptr(), nq, k, *(t.data_ptr() for t in out), 0, -1,
                                          ws.data_ptr() if ws_bytes else None, ws_bytes or 0, stream)
                assert rc == 0, lib.tk_last_error()
                outs.append(out)
            assert all(torch.equal(a, b) for a, b in zip(*outs))
            rc = lib.tk_knn_query_gpu(tree, q.data_ptr(), nq, k, *(t.data_ptr() for t in outs[0]), 0, -1, ws.data_ptr(),
                                      need.value - 1, stream)
            assert rc != 0 and b"workspace" in lib.tk_last_error(), k
    finally:
        torch.cuda.synchronize()
        lib.tk_tree_free(tree)
