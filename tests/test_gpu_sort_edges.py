"""The radix sort where one of its forms hands over to the next, against torch's stable sort: one workgroup up
to 4,096 pairs; look-back with tiles of 2,048 pairs, whose passes sum the counts themselves up to 32 tiles
(65,536 pairs), up to 2^19 pairs; three launches a pass beyond.  With values and without (they are then the
pairs' indices, as the presort, the backward and the batch ask for), and with no bits to sort by."""
import pytest
import torch

from torch_kdtree_amd import torch_knn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4096, 4097, 65_536, 65_537, 1 << 19, (1 << 19) + 1, (1 << 21) + 1])
@pytest.mark.parametrize("key_bits", [0, 5, 8, 16, 20, 31])
@pytest.mark.parametrize("values", [True, False])
def test_sort_hand_overs(cuda, n, key_bits, values):
    g = torch.Generator(device=cuda).manual_seed(n + key_bits)
    k = torch.randint(0, 1 << max(key_bits, 1), (n,), generator=g, device=cuda).int()
    v = torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device=cuda).int()
    ko, vo = torch.empty_like(k), torch.empty_like(v)
    if key_bits:
        want, perm = torch.sort(k, stable=True)
    else:
        want, perm = k, torch.arange(n, device=cuda)
    for _ in range(2):
        ko.fill_(-1)
        vo.fill_(-1)
        torch_knn.sort_pairs(k.data_ptr(), v.data_ptr() if values else 0, ko.data_ptr(), vo.data_ptr(), n, key_bits,
                             torch.cuda.current_stream().cuda_stream)
        assert torch.equal(ko, want)
        assert torch.equal(vo, v[perm] if values else perm.int())
