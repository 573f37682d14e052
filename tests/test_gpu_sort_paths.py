"""The radix sort's paths against torch's stable sort: one workgroup (up to 4,096 pairs), look-back passes (up
to 2^19 pairs), and three launches a pass."""
import pytest
import torch

from torch_kdtree_amd import torch_knn

pytestmark = pytest.mark.gpu


def _launch(k, v, ko, vo, key_bits):
    torch_knn.sort_pairs(k.data_ptr(), v.data_ptr(), ko.data_ptr(), vo.data_ptr(), k.numel(), key_bits,
                         torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("n", [4096, 4097, 131_072, 131_073, 1 << 21, (1 << 21) + 1, 5_000_003])
@pytest.mark.parametrize("key_bits,spread", [(8, 8), (20, 20), (24, 3), (31, 31)])
def test_sort_paths(cuda, n, key_bits, spread):
    g = torch.Generator(device=cuda).manual_seed(n + key_bits)
    k = torch.randint(0, 1 << spread, (n,), generator=g, device=cuda)
    if spread < 8:  # few distinct values in the highest digit, long runs of equal keys
        k = k << (key_bits - spread)
    v = torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device=cuda).int()
    k = k.int()
    ko, vo = torch.empty_like(k), torch.empty_like(v)
    want, perm = torch.sort(k, stable=True)
    for _ in range(2):
        ko.fill_(-1)
        vo.fill_(0)
        _launch(k, v, ko, vo, key_bits)
        assert torch.equal(ko, want) and torch.equal(vo, v[perm])
