"""GPU parity of the strided f32-MFMA GEMM at the edges of its tiles, chunks
and of the three ways it reads an operand (pieces along k, along the rows,
single elements), against f64."""
import numpy as np
import pytest

from helpers import draw, make_layer, rel_l2, to_dev, to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,S,H", [(1, 1, 1), (31, 33, 5), (64, 32, 64), (65, 97, 130), (513, 36, 260), (40, 1024, 12),
                                   (2100, 768, 260), (1027, 1030, 34), (3300, 1000, 900), (65, 1800, 1792)])
def test_graft_gemm_kinds(dev, M, S, H):
    """The six graft GEMMs: every pair of operand orientations, lengths off the
    chunks and pieces, few tiles (many wavefronts per tile) to several 64 x 64
    tiles per CU. Operands are bf16 or rounded to it, so products are exact;
    f32 sums: rel-L2 within 1e-6 per doubling of the number of terms."""
    import torch
    from glt_amd import _ffi as F, ops
    g = torch.Generator(device="cuda").manual_seed(M + S + H)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    delta, xs, xh = rnd(S, H), rnd(M, S).bfloat16(), rnd(M, H).bfloat16()
    dys, dyh = rnd(M, S), rnd(M, H)
    r = lambda t: t.bfloat16().double()
    cases = [(F.GEMM_EXPAND_FWD, (M, S), H, dict(a=xh, lda=H, delta=delta), lambda: r(xh) @ r(delta).t()),
             (F.GEMM_CONTRACT_FWD, (M, H), S, dict(a=xs, lda=S, delta=delta), lambda: r(xs) @ r(delta)),
             (F.GEMM_EXPAND_WGRAD, (S, H), M, dict(a=xh, lda=H, dy=dys), lambda: r(dys).t() @ r(xh)),
             (F.GEMM_CONTRACT_WGRAD, (S, H), M, dict(a=xs, lda=S, dy=dyh), lambda: r(xs).t() @ r(dyh)),
             (F.GEMM_EXPAND_IGRAD, (M, H), S, dict(delta=delta, dy=dys), lambda: r(dys) @ r(delta)),
             (F.GEMM_CONTRACT_IGRAD, (M, S), H, dict(delta=delta, dy=dyh), lambda: r(dyh) @ r(delta).t())]
    for kind, shape, terms, args, ref in cases:
        out = rnd(*shape)
        want = 0.5 * ref() + 2.0 * out.double()
        ops.graft_gemm(kind, M, S, H, out, alpha=0.5, beta=2.0, **args)
        assert rel_l2(to_np(out), want.cpu().numpy()) <= 1e-6 * max(1.0, np.log2(terms)), kind


@pytest.mark.parametrize("M,D,I,pl", [(33, 100, 130, [(7, 31, 3, 90), (130, 33, 0, 100)]),
                                      (130, 256, 320, [(64, 96, 32, 64), (320, 64, 0, 256)]),
                                      (1601, 512, 704, [(5, 64, 0, 512)])])
def test_f32_mlp(dev, M, D, I, pl):
    """The f32 layer forward and backward with odd, in-place and appended
    slices, from a few tiles to several 64 x 64 tiles per CU."""
    import torch
    from glt_amd import ops, synth
    N = max([I] + [i0 + s for i0, s, _, _ in pl])
    wg, wu, wd, sl = make_layer(D, I, N, pl, False)
    x = draw((M, D), 100, synth.TID_X, 0, 1, False)
    dy = draw((M, D), 200, synth.TID_DY, 0, 1, False)
    f = torch.float32
    base = ops.BaseMLP(to_dev(wg, f), to_dev(wu, f), to_dev(wd, f))
    gs = [ops.GraftSlice(s["i0"], s["s"], s["h0"], s["h"], *(to_dev(s[p], f) for p in ("gate", "up", "down"))) for s in sl]
    xd, dyd = to_dev(x, f), to_dev(dy, f)
    y, g, u, inter = ops.mlp_forward(base, gs, xd, N)
    dx, grads = ops.mlp_backward(base, gs, xd, dyd, N, g, u, inter)
    rg, ru, ri, ry = O.mlp_fwd(x, wg, wu, wd, N, sl, bf16=False)
    rdx, rgr = O.mlp_bwd(x, wg, wu, wd, N, sl, rg, ru, ri, dy, bf16=False)
    for name, t, r in (("g", g, rg), ("u", u, ru), ("inter", inter, ri), ("y", y, ry), ("dx", dx, rdx)):
        assert rel_l2(to_np(t), r) <= 1e-5, name
    for j in range(len(pl)):
        for p in range(3):
            assert rel_l2(to_np(grads[j][p]), rgr[j][p]) <= 1e-5, (j, p)


def test_more_tiles_than_a_grid_dimension_holds(dev):
    """A gate/up launch of 2^24 + 2 tiles (2^29 + 64 rows of one column): y of
    every row, x holding one of four values."""
    import torch
    from glt_amd import ops
    M = (1 << 29) + 64
    one = torch.full((1, 1), 1.0, device="cuda")
    base = ops.BaseMLP(one, one, one)
    vals = torch.tensor([-2.0, 0.5, 1.0, 3.0], device="cuda")
    x = vals.repeat(M // 4).view(M, 1)
    y, _, _, inter = ops.mlp_forward(base, [], x, 1, save=False)
    ref, _, _, _ = ops.mlp_forward(base, [], vals.view(4, 1).contiguous(), 1, save=False)
    assert torch.equal(y.view(M // 4, 4), ref.view(1, 4).expand(M // 4, 4))
    want = torch.nn.functional.silu(vals.double()) * vals.double()
    assert rel_l2(to_np(ref.view(-1)), want.cpu().numpy()) <= 1e-6


def test_reductions_past_two_to_the_thirty(dev):
    """One output over more than 2^30 terms: zeros but for a few terms at both
    ends and in the middle, summed exactly."""
    import torch
    from glt_amd import _ffi as F, ops
    H = (1 << 30) + 44
    a = torch.zeros((1, H), dtype=torch.bfloat16, device="cuda")
    delta = torch.zeros((1, H), device="cuda")
    want = 0.0
    for k, t in enumerate((0, 1, 255, 256, H // 2, (1 << 30) - 1, 1 << 30, H - 2, H - 1)):
        a[0, t], delta[0, t] = k + 1, 2.0 ** k
        want += (k + 1) * 2.0 ** k
    out = torch.empty((1, 1), device="cuda")
    ops.graft_gemm(F.GEMM_EXPAND_FWD, 1, 1, H, out, a=a, lda=H, delta=delta)
    assert out.item() == want
