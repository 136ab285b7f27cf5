"""mm_species_lists at row counts around its threads, waves and 4,096-row tiles, with absent species; exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 5, 255, 257, 4095, 4097, 20001])
@pytest.mark.parametrize("S", [1, 3, 16])
def test_species_lists(n, S):
    from mace_onegpu import _lib
    spec = torch.randint(0, S, (n,), generator=torch.Generator().manual_seed(n + S), dtype=torch.int32)
    spec[spec == 1] = 0
    lists = torch.full((S, n + 2), -7, dtype=torch.int32, device="cuda")
    counts = torch.full((S,), -7, dtype=torch.int32, device="cuda")
    _lib.K.mm_species_lists(spec.cuda(), n, S, lists, n + 2, counts, _lib.stream())
    for s in range(S):
        rows = torch.nonzero(spec == s).squeeze(1).int()
        assert int(counts[s]) == rows.numel()
        assert torch.equal(lists[s, :rows.numel()].cpu(), rows) and bool((lists[s, rows.numel():] == -7).all())
