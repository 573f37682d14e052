"""The backward's row accesses: 16 bytes at a time where k is a multiple of 8 and the rows lie on 16 bytes,
one element at a time elsewhere.  The gradients are the same bits either way, and those of a float64 sum."""
import pytest
import torch

from torch_kdtree_amd import torch_knn

pytestmark = pytest.mark.gpu


def _at(x, pad):
    """x in a buffer of its own, `pad` elements past a 16-byte boundary."""
    buf = torch.empty(x.numel() + 4, dtype=x.dtype, device=x.device)
    v = buf[pad:pad + x.numel()].view(x.shape)
    v.copy_(x)
    assert buf.data_ptr() % 16 == 0
    return v


def _backward(q, ref, idx, g):
    dq, dr = torch.empty_like(q), torch.empty_like(ref)
    torch_knn.knn_backward(q.data_ptr(), ref.data_ptr(), q.shape[0], ref.shape[0], q.shape[1],
                           "float64" if q.dtype == torch.float64 else "float32", idx.shape[1], idx.data_ptr(),
                           g.data_ptr(), dq.data_ptr(), dr.data_ptr(), torch.cuda.current_stream().cuda_stream)
    return dq, dr


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("d", [1, 3, 8])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 16, 40])
def test_rows_aligned_or_not(cuda, dtype, d, k):
    n, nq = 301, 1021
    gen = torch.Generator(device=cuda).manual_seed(1000 * d + k)
    ref = torch.rand((n, d), generator=gen, device=cuda, dtype=dtype)
    q = torch.rand((nq, d), generator=gen, device=cuda, dtype=dtype)
    idx = torch.randint(0, n, (nq, k), generator=gen, device=cuda)
    g = torch.randn((nq, k), generator=gen, device=cuda, dtype=dtype)
    dq, dr = _backward(q, ref, _at(idx, 0), _at(g, 0))
    for pi, pg in ((1, 0), (0, 1), (1, 1)):
        dq1, dr1 = _backward(q, ref, _at(idx, pi), _at(g, pg))
        assert torch.equal(dq, dq1) and torch.equal(dr, dr1)
    term = g.double()[..., None] * 2 * (q.double()[:, None] - ref.double()[idx])
    eps = torch.finfo(dtype).eps
    mag = term.abs()
    # (a sum of m terms, each with three roundings: at most (m + 3) eps of the sum of the magnitudes)
    assert ((dq.double() - term.sum(1)).abs() <= (k + 3) * eps * mag.sum(1) + 1e-300).all()
    want = torch.zeros((n, d), dtype=torch.float64, device=cuda)
    size, cnt = torch.zeros_like(want), torch.zeros(n, dtype=torch.float64, device=cuda)
    flat = idx.reshape(-1)
    want.index_add_(0, flat, -term.reshape(-1, d))
    size.index_add_(0, flat, mag.reshape(-1, d))
    cnt.index_add_(0, flat, torch.ones_like(flat, dtype=torch.float64))
    assert ((dr.double() - want).abs() <= (cnt[:, None] + 3) * eps * size + 1e-300).all()
