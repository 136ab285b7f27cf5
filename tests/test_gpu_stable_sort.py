"""mm_stable_sort and the CSR of its keys against torch's stable sort: sizes around a wave, a tile and one, two and
three digits, keys that are all equal and keys that miss most of the range; exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [0, 1, 63, 65, 4096, 4097, 300001])
@pytest.mark.parametrize("n", [1, 2, 256, 257, 65537, 20000003])
def test_stable_sort(E, n):
    from mace_onegpu.fused_conv import csr_of_sorted, stable_sort
    g = torch.Generator().manual_seed(E + n)
    wide = torch.randint(0, n, (E,), generator=g, dtype=torch.int32)
    for keys in (wide, torch.full_like(wide, n - 1), wide // 3):
        ref, perm = torch.sort(keys, stable=True)
        k, p = stable_sort(keys.cuda(), n)
        assert torch.equal(k.cpu(), ref) and torch.equal(p.cpu().long(), perm)
    rowptr = csr_of_sorted(k, n)
    assert torch.equal(rowptr.cpu(), torch.searchsorted(ref, torch.arange(n + 1, dtype=torch.int32)).int())
