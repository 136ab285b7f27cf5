"""The explicit-weight convolution where the waves of a workgroup share a receiver's edges, and where they do not, and
its index preparation (marked gpu): mean degrees on both sides of the rule, receivers of 0 .. 5 edges (waves without a
share), one hub, index types and layouts, and the errors for indices out of range.  Against the fp64 oracle; the bar is
2e-5 of the largest value, as for the other cases of these kernels."""
import numpy as np
import pytest
import torch

from mace_onegpu.fused_conv import ChannelwiseTP, FusedConvTP, receiver_csr

pytestmark = pytest.mark.gpu

C = 128
DEGREES = {"short": [0, 1, 2, 3, 5], "long": [0, 1, 18, 31, 64, 65], "hub": [0] * 20 + [331]}


def _graph(name, n, seed):
    rng = np.random.default_rng(seed)
    deg = rng.choice(DEGREES[name], n)
    deg[0] = max(DEGREES[name])
    recv = np.repeat(np.arange(n), deg)
    return torch.from_numpy(np.stack([rng.integers(0, n, len(recv)), recv]))


@pytest.mark.parametrize("in_ls", [(0,), (0, 1), (0, 1, 2, 3)])
@pytest.mark.parametrize("name", sorted(DEGREES))
def test_against_the_oracle(in_ls, name):
    from mace_onegpu import o3
    from oracle import mace_ref
    desc, n = ChannelwiseTP(in_ls), 23
    ei = _graph(name, n, 1)
    E = ei.shape[1]
    print(f"case {desc} {name}: {E} edges", flush=True)
    g = torch.Generator().manual_seed(2)
    x = [torch.randn(r, c, generator=g, dtype=torch.float64).float().double().requires_grad_(True)
         for r, c in ((n, desc.nX * C), (E, 16), (E, desc.nW * C))]
    mid = mace_ref.channelwise_tp(x[2].reshape(E, desc.nW, C), x[0].reshape(n, desc.nX, C), x[1], ei[0],
                                  desc.table["paths"], desc.table["in_ls"], o3.coupling)
    ref = mace_ref.scatter_sum(mid, ei[1], n).reshape(n, desc.nO * C)
    R = torch.randn(ref.shape, generator=g, dtype=torch.float64).float().double()
    gref = torch.autograd.grad((ref * R).sum(), x)
    xd = [t.detach().float().cuda().requires_grad_(True) for t in x]
    out = FusedConvTP(desc, desc.weight_numel)(*xd, ei.cuda())
    got = torch.autograd.grad(out, xd, R.float().cuda())
    for a, b in zip((out, *got), (ref, *gref)):
        a, b = a.detach().double().cpu(), b.detach()
        assert float((a - b).abs().max()) <= 2e-5 * float(b.abs().max())


@pytest.mark.parametrize("E", [1, 2, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("layout", ["int64", "int32", "int16", "columns", "unsorted"])
def test_receiver_csr(E, layout):
    rng = np.random.default_rng(E)
    n = 300
    recv = np.sort(rng.integers(3, n - 40, E))
    if layout == "unsorted":
        recv = rng.permutation(recv)
    ei = torch.from_numpy(np.stack([rng.integers(0, n, E), recv])).cuda()
    if layout in ("int32", "int16"):
        ei = ei.to(getattr(torch, layout))
    if layout == "columns":
        ei = ei.t().contiguous().t()
    rowptr, eid, send = receiver_csr(ei, n, n)
    assert np.array_equal(rowptr.cpu().numpy(), np.searchsorted(np.sort(recv), np.arange(n + 1)))
    assert torch.equal(send.cpu().long(), ei[0].cpu().long())
    if layout == "unsorted" and (np.diff(recv) < 0).any():
        assert np.array_equal(eid.cpu().numpy(), np.argsort(recv, kind="stable"))
    else:
        assert eid is None


@pytest.mark.parametrize("row,value", [(0, -1), (0, 7), (0, 2 ** 32), (1, -1), (1, 7), (1, 2 ** 32 + 2)])
def test_indices_out_of_range(row, value):
    ei = torch.tensor([[0, 1, 6], [0, 3, 6]]).cuda()
    ei[row, 1] = value
    with pytest.raises(IndexError, match="sender" if row == 0 else "receiver"):
        receiver_csr(ei, 7, 7)


def test_more_receivers_than_one_launch_takes_workgroups():
    """2^24 receivers of 4 edges (a mean degree at which a workgroup shares a receiver's edges): a workgroup each would
    be 2^32 threads, more than a launch takes.  All edges read one row of each operand, so every output row is the
    same; four equal fp32 products, the bar is an ulp of their sum for each of the 3 roundings."""
    from mace_onegpu._lib import stream
    d = ChannelwiseTP([0], 0, (0,))
    fwd, _ = d.kernels(edge_count=True)
    n = 2 ** 24
    g = torch.Generator().manual_seed(0)
    X, W, Y = (torch.randn(1, k, generator=g) for k in (C, C, 16))
    i32 = dict(dtype=torch.int32, device="cuda")
    rowptr, zeros = torch.arange(0, 4 * n + 1, 4, **i32), torch.zeros(4 * n, **i32)
    out = torch.empty(n, C, device="cuda")
    fwd(4 * n, rowptr, n, zeros, zeros, Y.cuda(), 16, W.cuda(), C, X.cuda(), C, out, C, stream())
    ref = 4 * d.table["terms"][0][4] * (X * W * Y[:, :1]).double()
    assert bool((out == out[0]).all())
    assert float(((out[:1].double().cpu() - ref) / ref).abs().max()) <= 3 * 2.0 ** -23
