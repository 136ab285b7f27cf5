"""mm_linear over row counts around its 32-row stages, its 1,024-row workgroups and the rule that groups four stages per
weight load, with one and several sources, row gathers, accumulation and output rows that are only float-aligned,
against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 33, 1023, 2081, 9001])
@pytest.mark.parametrize("n_src", [1, 2, 3])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_linear_rows_and_sources(rows, n_src, accumulate):
    from mace_onegpu import _lib
    from mace_onegpu.fast_layers import LinPlan, mfma_block
    g = torch.Generator().manual_seed(rows + n_src)
    n_comp = 8
    Ws = [torch.randn(128, 128, generator=g, dtype=torch.float64) for _ in range(4)]
    W = torch.cat([mfma_block(w.float()) for w in Ws]).cuda()
    # component j: the sources j .. j + n_src - 1 with different weight blocks; the last component has one source
    srcs = [[(128 * ((j + q) % n_comp), (j + q) % 4) for q in range(n_src if j < n_comp - 1 else 1)]
            for j in range(n_comp)]
    plan = LinPlan([(1 + 128 * j, s) for j, s in enumerate(srcs)])
    n_in, stride = rows + 5, 128 * n_comp + 3
    x = torch.randn(n_in, 128 * n_comp, generator=g)
    perm = torch.randperm(n_in, generator=g)[:rows]
    scale = torch.rand(rows, generator=g)
    out0 = torch.randn(rows + 1, stride, generator=g)
    out = out0.cuda()
    _lib.K.mm_linear(x.cuda(), 128 * n_comp, perm.int().cuda(), out, stride, None, W, scale.cuda(), 0, None, None, 0, 1,
                     0, rows, accumulate, plan.n, plan.nsrc, plan.inoff, plan.widx, plan.outoff, 0, _lib.stream())
    out = out.cpu()
    xd, ref = x[perm].double(), out0.double()
    bound = torch.zeros_like(ref)
    for j, src in enumerate(srcs):
        cols = slice(1 + 128 * j, 129 + 128 * j)
        y = sum(xd[:, o:o + 128] @ Ws[w].float().double() for o, w in src) * scale.double()[:, None]
        a = sum(xd[:, o:o + 128].abs() @ Ws[w].abs() for o, w in src) * scale.double()[:, None]
        old = ref[:rows, cols] * accumulate
        # per product: three omitted bf16 products (3 * 2^-24) and the remainders of the operands (2 * 2^-27); six
        # partial sums of 128 n_src products accumulated in fp32, of which the rounding errors add like a random walk
        # (sqrt of the number of additions, 32 products per instruction); scale and sum: one rounding each
        n_add = 6 * 4 * len(src)
        bound[:rows, cols] = a * 2 ** -24 * (3 + 0.25 + 4 * n_add ** 0.5) + 2 ** -23 * (old.abs() + y.abs())
        ref[:rows, cols] = old + y
    err = (out.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound.clamp_min(1e-300)).max())   # nothing else was written
