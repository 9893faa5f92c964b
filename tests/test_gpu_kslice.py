"""GPU parity of the small-tile MFMA GEMM: launches of few tiles, at the edges of
its tile shapes (32 x 32 to 128 x 256), with reductions whose K-steps do not
divide evenly over the unrolled steps."""
import numpy as np
import pytest

from helpers import assert_bf16_budget, draw, make_layer, rel_l2, to_dev, to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 31, 33, 64, 65, 129, 200, 257, 400])
@pytest.mark.parametrize("K,V", [(64, 2048), (704, 4104), (1088, 16000)])
def test_head_both_ways(dev, M, K, V):
    """LM head (bf16 out, K = 1, 11 or 17 steps; V ends inside a tile) and its
    backward (f32 out, K = V padded to whole steps where V is a multiple of 64,
    else the strided kernel) against f64. One bf16 rounding; f32 sums of exact
    products: rel-L2 within 1e-6 per doubling of the number of terms."""
    import torch
    from glt_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * 7919 + K)
    x = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    w = torch.randn((V, K), generator=g, device="cuda").mul_(0.05).bfloat16()
    y = ops.lm_head_fwd(x, w)
    assert_bf16_budget(to_np(y), (x.double() @ w.double().t()).cpu().numpy(), q=1, what="logits")
    if K >= 512:  # K output columns
        gr = torch.randn((M, V), generator=g, device="cuda").bfloat16()
        dx = ops.lm_head_bwd(gr, w)
        assert rel_l2(to_np(dx), (gr.double() @ w.double()).cpu().numpy()) <= 1e-6 * np.log2(V)


@pytest.mark.parametrize("M", [1, 32, 63, 65, 128, 129])
def test_weights_past_the_cache(dev, M):
    """One row of tiles (up to 128 rows) over more than 128 MiB of weights,
    which are loaded non-temporally: LM head and the dual gate/up launch."""
    import torch
    from glt_amd import ops
    K, V = 4160, 16264
    assert V * K * 2 > 128 << 20
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    w = torch.randn((V, K), generator=g, device="cuda").mul_(0.05).bfloat16()
    assert_bf16_budget(to_np(ops.lm_head_fwd(x, w)), (x.double() @ w.double().t()).cpu().numpy(), q=1, what="logits")
    wg, wu = w[:8128], w[8128:2 * 8128].contiguous()
    wd = torch.randn((K, 8128), generator=g, device="cuda").mul_(0.05).bfloat16()
    _, gt, up, inter = ops.mlp_forward(ops.BaseMLP(wg, wu, wd), [], x, 8128)
    rg, ru = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    assert_bf16_budget(to_np(gt), rg.cpu().numpy(), q=1, what="gate")
    assert_bf16_budget(to_np(up), ru.cpu().numpy(), q=1, what="up")
    ri = torch.nn.functional.silu(rg) * ru
    assert_bf16_budget(to_np(inter), ri.cpu().numpy(), q=3, what="inter")


@pytest.mark.parametrize("M", [7, 40, 70, 130, 300, 520])
def test_mlp_slices(dev, M):
    """Forward and backward with an in-place slice over base columns, one with
    an H offset and an appended one (tiles of two and three K-segments, tiles
    with none), residual output included."""
    import torch
    from glt_amd import ops, synth
    D, I = 1024, 3008
    pl = [(64, 192, 0, 1024), (1024, 128, 512, 448), (I, 192, 0, 1024)]
    N = I + 192 + 64  # the last 64 columns have no segment
    wg, wu, wd, sl = make_layer(D, I, N, pl, True)
    dt = torch.bfloat16
    x = draw((M, D), 100, synth.TID_X, 0, 1, True)
    dy = draw((M, D), 200, synth.TID_DY, 0, 1, True)
    base = ops.BaseMLP(to_dev(wg, dt), to_dev(wu, dt), to_dev(wd, dt))
    gs = [ops.GraftSlice(s["i0"], s["s"], s["h0"], s["h"], *(to_dev(s[p], torch.float32) for p in ("gate", "up", "down")))
          .pack() for s in sl]
    xd, dyd = to_dev(x, dt), to_dev(dy, dt)
    y, g, u, inter = ops.mlp_forward(base, gs, xd, N)
    dx, grads = ops.mlp_backward(base, gs, xd, dyd, N, g, u, inter)
    res = xd.clone()
    ops.mlp_forward(base, gs, xd, N, residual=res)
    torch.cuda.synchronize()
    rg, ru, ri, ry = O.mlp_fwd(x, wg, wu, wd, N, sl)
    rdx, rgr = O.mlp_bwd(x, wg, wu, wd, N, sl, rg, ru, ri, dy)
    for name, t, r, q in (("g", g, rg, 2), ("u", u, ru, 2), ("inter", inter, ri, 3), ("y", y, ry, 4), ("dx", dx, rdx, 4)):
        assert_bf16_budget(to_np(t), r, q=q, what=name)
    assert torch.equal(res, (xd.float() + y.float()).bfloat16())  # the rounded output, added and rounded
    assert np.all(to_np(inter)[:, I + 192:] == 0)
    # over few tokens the roundings of the saved operand do not average out:
    # inter carries three (gate, up, their product), dgate / dup four (gate,
    # up, the gradient of both and its own), and its sum with exact x or dy none
    for j in range(len(pl)):
        for p in range(3):
            assert_bf16_budget(to_np(grads[j][p]), rgr[j][p], q=4, what=f"slice {j} projection {p}")


@pytest.mark.parametrize("M", [1, 63, 65, 191, 1000])
def test_ragged_weight_gradients(dev, M):
    """Token counts off the 64-token steps of the weight-gradient GEMM, whose
    operands are then padded with zeros: gradients of a slice with an H offset
    and an appended one against f64 sums of the saved activations, from a bf16
    and an f32 upstream gradient (the same bits: the values are bf16)."""
    import torch
    from glt_amd import ops
    D, I = 512, 1024
    pl = [(128, 192, 64, 384), (I, 128, 0, 512)]
    N = I + 128
    wg, wu, wd, sl = make_layer(D, I, N, pl, True)
    dt = torch.bfloat16
    base = ops.BaseMLP(to_dev(wg, dt), to_dev(wu, dt), to_dev(wd, dt))
    gs = [ops.GraftSlice(s["i0"], s["s"], s["h0"], s["h"], *(to_dev(s[p], torch.float32) for p in ("gate", "up", "down")))
          .pack() for s in sl]
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, D), generator=g, device="cuda").to(dt)
    dy = torch.randn((M, D), generator=g, device="cuda").to(dt)
    y, gp, up, inter = ops.mlp_forward(base, gs, x, N)
    nbytes = ops.mlp_backward_workspace(base, gs, M, N) + 2 * M * D + 512  # dy f32: its bf16 copy too
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")     # stale NaN bits in the padding
    dx, grads = ops.mlp_backward(base, gs, x, dy, N, gp, up, inter, workspace=ws)
    dx32, grads32 = ops.mlp_backward(base, gs, x, dy.float(), N, gp, up, inter, workspace=ws)
    assert torch.equal(dx, dx32)
    dg, du = ops.gate_up_bwd((dy.float() @ torch.cat([base.down.float(), torch.zeros(D, 128, device="cuda")], 1)
                              + _graft_rows(gs, dy, N)), gp, up)
    for j, s in enumerate(gs):
        cols, hs = slice(s.i_start, s.i_start + s.s), slice(s.h_start, s.h_start + s.h)
        for p, (a, b) in enumerate(((dg, x), (du, x), (inter, dy))):
            ref = (a[:, cols].double().t() @ b[:, hs].double()).cpu().numpy()
            # dgate / dup enter the sums rounded to bf16, inter as saved
            assert_bf16_budget(to_np(grads[j][p]), ref, q=1, what=f"slice {j} projection {p}")
            assert torch.equal(grads[j][p], grads32[j][p])


@pytest.mark.parametrize("M", [65, 128])
@pytest.mark.parametrize("what,recompute", [("gate", False), ("up", False), ("down", False), ("inter", False),
                                            ("gate", True), ("down", True)])
def test_weight_gradients_off_16_bytes(dev, M, what, recompute):
    """A gradient buffer 4 bytes, or the saved inter 2, past a 16-byte boundary:
    the same bf16 operands, read by the strided kernel or its scalar transpose.
    f32 sums of exact products: rel-L2 within 1e-6 per doubling of the number of terms, and
    nothing written around the buffer."""
    import ctypes
    import torch
    from glt_amd import _ffi as F, ops
    D, I, S, H0, H = 512, 1024, 128, 64, 384
    N = I + S
    g = torch.Generator(device="cuda").manual_seed(M)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").mul_(0.02)
    bf = torch.bfloat16
    base = ops.BaseMLP(rn(I, D).to(bf), rn(I, D).to(bf), rn(D, I).to(bf))
    gs = [ops.GraftSlice(I, S, H0, H, rn(S, H), rn(S, H), rn(S, H)).pack()]
    x, dy = rn(M, D).mul_(50).to(bf), rn(M, D).mul_(50).to(bf)
    _, gp, up, inter = ops.mlp_forward(base, gs, x, N)
    dx0, g0 = ops.mlp_backward(base, gs, x, dy, N, gp, up, inter)

    d, keep = ops._desc(base, gs, M, N, True, recompute=recompute)
    n = F.load().glt_mlp_bwd_workspace_size(ctypes.byref(d))
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    store = [torch.full((S * H + 8,), 7.0, device="cuda") for _ in range(3)]
    off = [1 if name == what else 0 for name in ("gate", "up", "down")]
    garr = (F.GraftGrads * 1)()
    garr[0] = F.GraftGrads(*(t.data_ptr() + 4 * o for t, o in zip(store, off)))
    if what == "inter":
        odd = torch.empty(M * N + 1, dtype=bf, device="cuda")
        odd[1:] = inter.reshape(-1)
        inter = odd[1:]
    dx = torch.empty_like(dx0)
    b = base.c_struct()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    F.call("glt_mlp_bwd", ctypes.byref(d), ctypes.byref(b), p(x), p(dy), p(gp), p(up), p(inter), p(dx), garr, p(ws), n,
           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert torch.equal(dx, dx0)
    for t, o, ref in zip(store, off, g0[0]):
        assert rel_l2(to_np(t[o:o + S * H]), to_np(ref).reshape(-1)) <= 1e-6 * np.log2(M)
        assert torch.all(t[:o] == 7.0) and torch.all(t[o + S * H:] == 7.0)


def _graft_rows(gs, dy, N):
    import torch
    out = torch.zeros((dy.shape[0], N), device="cuda")
    for s in gs:
        out[:, s.i_start:s.i_start + s.s] += dy[:, s.h_start:s.h_start + s.h].float() @ s.down.bfloat16().float().t()
    return out
