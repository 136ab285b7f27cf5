"""The cell-list kernel at the edges of its tiles (marked gpu), bit for bit against the plain-C restatement: cells
with no, one and more than 64 atoms, more candidates than one LDS stage (1024) and than the mask words the count pass
keeps, receivers that are not a multiple of a workgroup's 16, thinly filled boxes (a wave per receiver) up to 2^24
cells (more than a launch with a workgroup per cell takes), and the brute-force scan of boxes under three cells."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

R = 6.0


def _box(name):
    rng = np.random.default_rng(5)
    L = np.array([25.0, 19.0, 31.0])
    if name == "sparse":                       # mostly empty cells
        return rng.uniform(0, L, (37, 3)), L
    if name == "single":
        return np.array([[1.0, 2.0, 3.0]]), L
    if name == "dense_corner":                 # one crowded cell (wrapping around the origin) among sparse ones
        return np.concatenate([rng.uniform(-2.5, 2.5, (1500, 3)), rng.uniform(0, L, (300, 3))]), L
    if name == "even":                         # about 100 atoms per cell: 2,700 candidates
        return rng.uniform(0, L, (100 * 4 * 3 * 5, 3)), L
    if name == "vacuum":                       # a crowded and a thin cluster in 18 x 16 x 21 cells, one wrapping around
        L = np.array([109.0, 97.0, 127.0])
        return np.concatenate([rng.uniform(-9, 9, (2500, 3)), rng.normal(60.0, 12.0, (1200, 3))]), L
    if name == "most_cells":                   # 1024 x 1024 x 16 cells
        L = np.array([6144.5, 6144.5, 96.5])
        return np.concatenate([rng.uniform(0, L, (500, 3)), rng.uniform(-6, 6, (100, 3))]), L
    if name == "slab":                         # two cells along one axis: every atom is a candidate
        L = np.array([14.0, 40.0, 33.0])
        return rng.uniform(0, L, (1031, 3)), L
    raise ValueError(name)


@pytest.mark.parametrize("name", ["single", "sparse", "dense_corner", "even", "vacuum", "most_cells", "slab"])
def test_bit_exact_with_the_c_oracle(name):
    from mace_onegpu.receiver_chunk_mace import System
    from oracle import nlist_c
    pos, L = _box(name)
    perm, pos_s, NN, rowptr, send = nlist_c.neighbor_list(pos, L, R)
    for words in (None, 0, 3):                 # the default mask words, none, and too few for most cells
        s = System(pos, L, np.zeros(len(pos), dtype=int), R, "cuda")
        if words is not None:
            s._mask_words = lambda brute, ncells: words
        print(f"case {name}: {len(pos)} atoms, mask words {words}", flush=True)
        s.build_neighbors()
        torch.cuda.synchronize()
        assert np.array_equal(s.perm.cpu().numpy(), perm) and np.array_equal(s.pos.cpu().numpy(), pos_s)
        assert np.array_equal(s.NN.cpu().numpy(), NN) and np.array_equal(s.rowptr.cpu().numpy(), rowptr)
        assert np.array_equal(s.send.cpu().numpy(), send)


def test_no_atoms():
    from mace_onegpu.receiver_chunk_mace import System
    for L in ([25.0, 19.0, 31.0], [14.0, 40.0, 33.0]):       # by cells and brute force
        s = System(np.zeros((0, 3)), np.array(L), np.zeros(0, dtype=int), R, "cuda")
        assert s.build_neighbors() == 0
        assert s.rowptr.tolist() == [0] and s.send.numel() == 0 and s.NN.numel() == 0
