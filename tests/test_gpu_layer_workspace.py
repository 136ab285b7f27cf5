"""The chunk workspace of FastLayers (marked gpu): what a first pass allocates and gives back."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def chunk(model):
    """(system, a chunk of 700 of the 1,536 atoms of a water box with its topology, species columns)."""
    from mace_onegpu import systems
    from mace_onegpu.receiver_chunk_mace import ReceiverChunkMACE, System
    pos, box, Z = systems.water_box(512, seed=4)
    s = System(pos, box, Z - 1, 6.0, "cuda")
    s.build_neighbors()
    ev = ReceiverChunkMACE(model, chunk=700, device="cuda")
    return s, ev.graphs(s)[0], ev.fl.cols


def _layers(model, cols, **kw):
    from mace_onegpu.fast_layers import FastLayers
    return FastLayers(model, cols, device="cuda", **kw)


def test_first_workspace_keeps_the_cache_and_layer_1_takes_no_sender_slots(model, chunk, monkeypatch):
    """A workspace that replaces none does not empty the allocator's cache (milliseconds of a first pass), a larger one
    does; the sender slots come with the first pass B."""
    s, g, cols = chunk
    fl = _layers(model, cols)
    emptied = []
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: emptied.append(1))
    H1 = torch.empty(s.N, 512, device="cuda")
    PF, eat = torch.zeros(g.nE, 3, device="cuda"), torch.zeros(s.N, dtype=torch.float64, device="cuda")
    fl.pass_a(g, H1)
    fl.pass_c(g, torch.zeros_like(H1), PF, eat)
    assert not emptied and not {"e_slot", "g_send", "g_n"} & set(fl.ws)
    H1 = torch.zeros_like(H1)
    fl.pass_b(g, H1, torch.zeros_like(H1), PF, eat)
    assert not emptied and fl.ws["e_slot"].numel() >= g.nE + 64
    old = fl.ws
    fl.workspace(g.nC + 1, g.n_nodes, g.nE)
    assert len(emptied) == 1 and fl.ws is not old and "e_slot" not in fl.ws
    torch.cuda.synchronize()


@pytest.mark.parametrize("deterministic", [False, True])
def test_pass_b_with_tables_beyond_32_bits(model, chunk, deterministic):
    """pass_b takes the per-harmonic kernels where one channel block's tables exceed 32-bit addresses (bwd_vec False): 17
    numbers per partial row instead of 3, and a workspace that holds them.  Both forms agree to 2e-6 in the 2-norm (an
    error of 7e-7 each against 64 bits) and write nothing behind the chunk's pair forces."""
    s, g, cols = chunk
    gen = torch.Generator(device="cuda").manual_seed(3)
    H1 = torch.randn(s.N, 512, generator=gen, device="cuda")
    out = {}
    for vec in (True, False):
        fl = _layers(model, cols, deterministic=deterministic)
        assert fl.bwd_vec
        fl.bwd_vec = vec
        ws = fl.prepare(g)
        assert ws["part"].numel() >= 8 * ws["E"] * (3 if vec else 17)
        # a guard behind the partials: the buffer is replaced by the front of a longer one
        n = ws["part"].numel()
        room = torch.full((n + 1024,), 7.0, device="cuda")
        ws["part"] = room[:n]
        PF = torch.full((g.nE + 64, 3), 5.0, device="cuda")
        G1, eat = torch.zeros(s.N, 512, device="cuda"), torch.zeros(s.N, dtype=torch.float64, device="cuda")
        print(f"case bwd_vec {vec} deterministic {deterministic}: {g.nE} edges", flush=True)
        fl.pass_b(g, H1, G1, PF, eat)
        torch.cuda.synchronize()
        assert bool((room[n:] == 7.0).all()) and bool((PF[g.nE:] == 5.0).all())
        out[vec] = (PF[:g.nE].double(), G1.double(), eat)
    assert torch.equal(out[True][2], out[False][2])
    for a, b in zip(out[True][:2], out[False][:2]):
        assert float((a - b).norm() / b.norm()) <= 2e-6
