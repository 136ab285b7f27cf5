"""mm_chunk_topology against the tensor form of chunk_topology (run on the CPU): node list and local senders of chunks
at the edges of its 32-atom words and 32,768-atom blocks, without edges, with every atom a sender, and bad senders."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,a,b,E", [(1, 0, 1, 3), (31, 5, 9, 0), (32, 0, 32, 70), (33, 32, 33, 40), (64, 10, 20, 5000),
                                      (32767, 100, 4000, 20000), (32768, 0, 1, 200000), (32769, 32768, 32769, 1500),
                                      (100001, 33333, 66666, 400001)])
def test_chunk_topology_matches_tensor_form(nt, a, b, E):
    from mace_onegpu.receiver_chunk_mace import chunk_topology
    g = torch.Generator().manual_seed(nt + E)
    pj = torch.randint(0, nt, (E + 7,), generator=g, dtype=torch.int32)
    e0, e1 = 3, 3 + E
    loc, flag = torch.full((nt,), -1, dtype=torch.int32), torch.zeros(nt, dtype=torch.bool)
    nodes, ls = chunk_topology(a, b, e0, e1, pj, loc, flag)
    for _ in range(2):
        n2, l2 = chunk_topology(a, b, e0, e1, pj.cuda(), loc.cuda(), flag.cuda())
        assert n2.dtype == torch.int32 and l2.dtype == torch.int32
        assert torch.equal(n2.cpu(), nodes) and torch.equal(l2.cpu(), ls)
    for bad in (-1, nt):
        if E:
            wrong = pj.clone()
            wrong[e1 - 1] = bad
            with pytest.raises(IndexError, match="senders of receivers"):
                chunk_topology(a, b, e0, e1, wrong.cuda(), loc.cuda(), flag.cuda())


@pytest.mark.parametrize("unsorted", [False, True])
def test_pair_batch_matches_cpu(unsorted):
    from mace_onegpu.mliap_threepass import _PairBatch

    class Data:
        pass
    g = torch.Generator().manual_seed(5)
    d, P, nl, nt = Data(), 3001, 97, 130
    d.pair_i = torch.randint(0, nl, (P,), generator=g)
    if not unsorted:
        d.pair_i = torch.sort(d.pair_i).values
    d.pair_j, d.rij = torch.randint(0, nt, (P,), generator=g), torch.randn(P, 3, generator=g, dtype=torch.float64)
    cpu, gpu = _PairBatch(d, nl, nt, torch.device("cpu"), True), _PairBatch(d, nl, nt, torch.device("cuda"), True)
    assert (cpu.perm is None) == (gpu.perm is None) == (not unsorted)
    for k in ("pair_i", "pair_j", "rij", "rowptr"):
        assert torch.equal(getattr(cpu, k), getattr(gpu, k).to("cpu", getattr(cpu, k).dtype))
    assert (cpu.rowptr_host == gpu.rowptr_host).all()
    for bad in (-1, nl):
        d.pair_i = torch.sort(d.pair_i).values
        d.pair_i[0 if bad < 0 else -1] = bad
        with pytest.raises(ValueError, match="local atom"):
            _PairBatch(d, nl, nt, torch.device("cuda"), False)
