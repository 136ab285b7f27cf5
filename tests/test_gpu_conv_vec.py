"""The layer-2 backward on the matrix cores (mm_sender_slots, mm_conv2_bwd_vec, mm_conv2_bwd_vec_det, mm_edge_grad_vec)
at the edges of its tiles (marked gpu), against fp64 autograd: receivers around multiples of the 16-edge tile, empty
ones and a short last group, more distinct senders than LDS slots, more edges than a group's slot list, directions at
and next to the poles of the polar frame, cotangents from 1e-30 to 1e20 with channels of zeros, lengths below the table
start; and non-finite cotangents, which must stay visible.

Bars: sums of up to a few thousand products against fp64, 1e-5 of the largest value, as for the per-harmonic kernels; and
5e-7 in the 2-norm, where the independent errors of a value's factors (operands of 2^-23, some ten fp32 roundings of 2^-24
at most, a third of that rms) add up to about 2e-7."""
import numpy as np
import pytest
import torch

from test_gpu_conv_kernels import C, _case, _terms

pytestmark = pytest.mark.gpu

CASES = {"tiles": (71, 900, 0, True, [1, 2, 15, 16, 17, 31, 32, 33, 48, 90]),
         "scattered": (37, 4000, 240, False, None),          # distinct senders of a group beyond the slots
         "long": (9, 4000, 0, False, [400, 401, 7]),          # a group beyond the slot list's edges
         "single": (2, 5, 0, False, [3])}                    # (_case leaves every 7th receiver empty)


def _reference(cs, tp, inv_h):
    """dL/dX [n, 4, C] and dL/dvec [E, 3] (vec = r u, spline coordinate t with dt/dr = inv_h where t is not -0)."""
    from oracle import mace_ref
    f = lambda a: torch.tensor(a, dtype=torch.float64).float().double()
    E, nC = len(cs["send"]), len(cs["rowptr"]) - 1
    recv = torch.repeat_interleave(torch.arange(nC), torch.from_numpy(np.diff(cs["rowptr"])).long())
    send = torch.from_numpy(cs["send"]).long()
    tabc = f(cs["tab"]).permute(1, 2, 0, 3, 4).reshape(cs["NR"], 10, C, 4)[torch.from_numpy(cs["row"]).long()]
    u, r, t0 = f(cs["u"]), f(cs["r"]), f(cs["t"])
    vec = (u * r[:, None]).requires_grad_(True)
    length = vec.norm(dim=1)
    below = torch.from_numpy(np.signbit(cs["t"]))
    t = t0 + torch.where(below, torch.zeros_like(r), inv_h * (length - length.detach()))
    tt = t[:, None, None]
    W = tabc[..., 0] + tt * (tabc[..., 1] + tt * (tabc[..., 2] + tt * tabc[..., 3]))
    X = f(cs["X"]).view(-1, 4, C).requires_grad_(True)
    Y = mace_ref.sh(vec)
    gA = f(cs["gA"]).view(nC, 40, C)[recv]
    loss = 0
    for (w, k, m, o, coef) in tp["terms"]:
        loss = loss + (coef * W[:, w] * X[send][:, k] * Y[:, m:m + 1] * gA[:, o]).sum()
    gX, gv = torch.autograd.grad(loss, [X, vec])
    return gX, gv


def _run(cs, inv_h, det=False):
    from mace_onegpu.codegen import GROUP, SLOTS
    from mace_onegpu.fast_layers import sender_csr
    from mace_onegpu._lib import K, stream
    from mace_onegpu.receiver_chunk_mace import ChunkGraph
    E, nC, n = len(cs["send"]), len(cs["rowptr"]) - 1, len(cs["X"])
    f32 = dict(dtype=torch.float32, device="cuda")
    pk = torch.empty(E, 4, **f32)
    pk[:, 0], pk[:, 3] = torch.tensor(cs["t"], **f32), 0.0
    pk.view(torch.int32)[:, 1] = torch.tensor(cs["row"], dtype=torch.int32, device="cuda")
    send = torch.tensor(cs["send"], dtype=torch.int32, device="cuda")
    pk.view(torch.int32)[:, 2] = send
    eu = torch.cat([torch.tensor(cs["u"], **f32), torch.tensor(cs["r"], **f32)[:, None]], 1).contiguous()
    rp = torch.tensor(cs["rowptr"], dtype=torch.int32, device="cuda")
    X, tab, gA = (torch.tensor(cs[k], **f32).contiguous() for k in ("X", "tab", "gA"))
    part = torch.full((8, E * 3 + 5), float("nan"), **f32)
    args = (rp, nC, pk, eu, X, 4 * C, tab, 1, cs["NR"] + 1, inv_h, gA, part, E * 3 + 5)
    if det:
        g = ChunkGraph()
        g.ls, g.nE, g.n_nodes = send, E, n
        gXe, gX = torch.full((E, 4 * C), float("nan"), **f32), torch.full((n, 4 * C), float("nan"), **f32)
        K.mm_conv2_bwd_vec_det(*args, gXe, stream())
        K.mm_gather_rows_csr(*sender_csr(g), gXe, 4 * C, 4 * C, gX, 4 * C, n, stream())
    else:
        ng = (nC + GROUP - 1) // GROUP
        slots = (torch.full((E + 64,), 77, dtype=torch.uint8, device="cuda"),
                 torch.full((ng * SLOTS,), -1, dtype=torch.int32, device="cuda"),
                 torch.full((ng,), -1, dtype=torch.int32, device="cuda"))
        K.mm_sender_slots(rp, nC, send, *slots, stream())
        es, gs, gn = (t.cpu() for t in slots)
        for q in range(ng):                    # every edge's slot names its sender; each sender one slot
            a, b = int(cs["rowptr"][q * GROUP]), int(cs["rowptr"][min(q * GROUP + GROUP, nC)])
            used = gs[q * SLOTS:q * SLOTS + int(gn[q])].long()
            assert 0 <= int(gn[q]) <= SLOTS and len(torch.unique(used)) == len(used)
            has = es[a:b] != 255
            assert torch.equal(used[es[a:b][has].long()], torch.from_numpy(cs["send"][a:b]).long()[has])
        gX = torch.zeros(n, 4 * C, **f32)
        K.mm_conv2_bwd_vec(*args, gX, *slots, stream())
    assert torch.isnan(part[:, E * 3:]).all()
    pf = torch.full((E, 3), float("nan"), **f32)
    K.mm_edge_grad_vec(E, None, part, E * 3 + 5, 8, None, None, None, eu, pf, 0, stream())
    torch.cuda.synchronize()
    return gX.view(n, 8, 4, 16).permute(0, 2, 1, 3).reshape(n, 4, C), pf


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e20])
def test_against_fp64_autograd(name, scale):
    nC, n, dmax, local, degrees = CASES[name]
    cs = _case(3, nC, n, dmax, local, degrees=degrees)
    E = len(cs["send"])
    u = cs["u"]
    u[0::5] = [0.0, 0.0, 1.0]
    u[1::5] = [0.0, 0.0, -1.0]
    u[2::5] = [3e-9, -4e-9, 1.0]
    u[3::5] = [0.6, 0.8, 0.0]
    cs["t"][::3] = -0.0
    cs["gA"] *= scale
    cs["gA"].reshape(nC, 40, C)[:, :, ::7] = 0
    if nC > 2:
        cs["gA"][-1] = 0
    print(f"case {name} scale {scale}: {E} edges", flush=True)
    inv_h = 3.0
    gX_r, gv_r = _reference(cs, _terms(), inv_h)
    for det in (False, True):
        gX, pf = _run(cs, inv_h, det)
        for got, ref in ((gX, gX_r), (pf, gv_r)):
            got = got.double().cpu()
            assert torch.isfinite(got).all()
            assert float((got - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
            rel = float((got - ref).norm() / ref.norm())
            print(f"  det {det}: relative error {rel:.2e}", flush=True)
            assert rel <= 5e-7


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_non_finite_cotangents_stay_visible(bad):
    cs = _case(3, 9, 50, 0, False, degrees=[5])
    cs["rowptr"] = np.arange(10, dtype=np.int32) * 5
    cs["send"] = np.tile(np.arange(5, dtype=np.int32), 9)
    for k in ("u", "r", "t", "row", "dens"):
        cs[k] = np.resize(cs[k], (45,) + cs[k].shape[1:])
    cs["gA"].reshape(9, 40, C)[4, 17, 30] = bad
    gX, pf = _run(cs, 3.0)
    assert not torch.isfinite(pf[20:25]).all(1).any()              # every edge of the receiver
    assert torch.isfinite(pf[:20]).all() and torch.isfinite(pf[25:]).all()
    assert not torch.isfinite(gX[:5, :, 30]).all(1).any()          # every one of its senders
