"""A batch over trees among which one comes from an image whose split values do not bound their points (no
build makes one; it loads, its checksum being right): under the reference policy the batch follows the
reference's walk there, so that every cloud's results equal the host search of the same tree bit for bit, in
each launch form, with the gradients of those neighbours; under the lower-index policy they equal brute
force."""
import ctypes
import os
import struct

import numpy as np
import pytest
import torch

import oracle
import torch_kdtree_amd as tk
from tests._util import assert_same

pytestmark = pytest.mark.gpu
_LIB = os.path.join(os.path.dirname(os.path.abspath(tk.__file__)), "libtorch_kdtree_amd.so")
_HEADER = 8 + 4 * 4 + 8


def _fnv1a(data):
    h = 1469598103934665603
    for b in data:
        h = ((h ^ b) * 1099511628211) & 0xffffffffffffffff
    return h


def _lib():
    lib = ctypes.CDLL(_LIB)
    vp = ctypes.c_void_p
    lib.tk_last_error.restype = ctypes.c_char_p
    lib.tk_tree_load.argtypes = [ctypes.c_char_p, ctypes.POINTER(vp)]
    lib.tk_tree_free.argtypes = lib.tk_batch_free.argtypes = [vp]
    lib.tk_tree_free.restype = lib.tk_batch_free.restype = None
    lib.tk_batch_create.argtypes = [vp, ctypes.c_int, vp, vp, ctypes.c_int, ctypes.c_int, ctypes.POINTER(vp)]
    lib.tk_batch_set_persistent.argtypes = [vp, ctypes.c_int]
    lib.tk_batch_forward.argtypes = [vp] * 6
    lib.tk_batch_capture.argtypes = [vp] * 9
    lib.tk_batch_launch.argtypes = [vp, vp]
    return lib


def _image(path, ref, levels, moved, rng):
    """The tree of ref written to path, its split values moved by up to `moved`."""
    tk.build_kd_tree(torch.from_numpy(ref), levels=levels).save(path)
    if moved:
        data = bytearray(open(path, "rb").read())
        n = (1 << levels) - 1
        split = np.frombuffer(bytes(data[_HEADER:_HEADER + n * ref.itemsize]), dtype=ref.dtype)
        split = (split + moved * rng.uniform(-1, 1, n)).astype(ref.dtype)
        data[_HEADER:_HEADER + n * ref.itemsize] = split.tobytes()
        data[-8:] = struct.pack("<Q", _fnv1a(data[:-8]))
        open(path, "wb").write(data)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 2, 3, 8])
@pytest.mark.parametrize("tie", ["reference", "lower_index"])
def test_batch_over_splits_off_their_points(cuda, tmp_path, dtype, d, tie):
    lib, vp = _lib(), ctypes.c_void_p
    rng = np.random.default_rng(600 + d)

    def check(rc):
        assert rc == 0, lib.tk_last_error().decode()

    tdt = torch.float32 if dtype == np.float32 else torch.float64
    nq, ks, moved = (200, 129, 64), (5, 32, 1), (0.3, 0.0, 0.1)
    refs = [rng.random((n, d)).astype(dtype) for n in (900, 300, 2500)]
    qrys = [rng.random((n, d)).astype(dtype) for n in nq]
    qrys[1][3, d - 1] = np.nan
    hosts, handles = [], (vp * 3)()
    try:
        for c, ref in enumerate(refs):
            path = str(tmp_path / ("t%d.bin" % c))
            _image(path, ref, (5, 3, 7)[c], moved[c], rng)
            hosts.append(tk.load_kd_tree(path, device="cpu"))
            h = vp()
            check(lib.tk_tree_load(path.encode(), ctypes.byref(h)))
            handles[c] = h.value
        q = torch.from_numpy(np.concatenate(qrys)).to(cuda)
        w = torch.rand(sum(n * k for n, k in zip(nq, ks)), dtype=tdt, device=cuda)
        for form in ("ranges", "persistent", "captured"):
            plan = vp()
            check(lib.tk_batch_create(handles, 3, (ctypes.c_int64 * 3)(*nq), (ctypes.c_int32 * 3)(*ks),
                                      int(tie == "lower_index"), 0, ctypes.byref(plan)))
            try:
                dist, idx = torch.empty_like(w), torch.empty(w.numel(), dtype=torch.int32, device=cuda)
                orig = torch.empty(w.numel(), dtype=torch.int64, device=cuda)
                gq = torch.empty_like(q)
                gr = torch.empty((sum(len(r) for r in refs), d), dtype=tdt, device=cuda)
                stream = torch.cuda.current_stream().cuda_stream
                check(lib.tk_batch_set_persistent(plan, int(form == "persistent")))
                if form == "captured":
                    check(lib.tk_batch_capture(plan, q.data_ptr(), dist.data_ptr(), idx.data_ptr(), orig.data_ptr(),
                                               w.data_ptr(), gq.data_ptr(), gr.data_ptr(), stream))
                    for _ in range(3):
                        for t in (dist, idx, orig, gq, gr):
                            t.fill_(-1)
                        check(lib.tk_batch_launch(plan, stream))
                else:
                    check(lib.tk_batch_forward(plan, q.data_ptr(), dist.data_ptr(), idx.data_ptr(), orig.data_ptr(),
                                               stream))
                torch.cuda.synchronize()
            finally:
                lib.tk_batch_free(plan)
            ob = qb = 0
            for c in range(3):
                n, k = nq[c], ks[c]
                got_d = dist[ob:ob + n * k].view(n, k).cpu().numpy()
                got_i = orig[ob:ob + n * k].view(n, k).cpu().numpy()
                what = "%s cloud %d " % (form, c)
                if tie == "reference":
                    want_d, want_i = (t.numpy() for t in hosts[c].query(torch.from_numpy(qrys[c]), nr_nns_searches=k))
                else:
                    want_d, want_i = oracle.bruteforce(refs[c], qrys[c], k)
                assert_same(got_d, want_d, what + "distances")
                assert_same(got_i, want_i.astype(np.int64), what + "indices")
                if form == "captured" and c != 1:  # (cloud 1 has a NaN row)
                    g = w[ob:ob + n * k].view(n, k).cpu().numpy()
                    acc = np.zeros((n, d), dtype)
                    for j in range(k):
                        diff = qrys[c] - refs[c][want_i[:, j]]
                        acc = acc + g[:, j:j + 1] * (diff + diff)
                    assert_same(gq[qb:qb + n].cpu().numpy(), acc, what + "dL/dq")
                ob, qb = ob + n * k, qb + n
    finally:
        for h in handles:
            if h:
                lib.tk_tree_free(h)
