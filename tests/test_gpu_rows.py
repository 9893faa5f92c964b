"""A token's outputs depend on that token alone: the same bits whatever the
tokens beside it in the call, hence also whichever GEMM kernel and tile shape a
call of that size takes. The exact logits hash of an eval set therefore does
not depend on how the set is cut into batches."""
import pytest

from helpers import make_layer, to_dev

pytestmark = pytest.mark.gpu

MS = (1, 8, 33, 64, 100, 154, 200, 257, 384, 512, 777, 1024, 2048)


def _bits(t):
    import torch
    return t.view(torch.int16 if t.element_size() == 2 else torch.int32)


@pytest.mark.parametrize("D,I,pl", [
    (2048, 11008, [(2752, 2752, 0, 2048)]),                   # in place
    (4096, 6144, [(6144, 256, 0, 4096), (6400, 64, 64, 448)]),  # appended; part of the hidden columns
])
def test_mlp(dev, D, I, pl):
    """Forward (saved, unsaved and residual form) and the backward's dx of the
    first M of 4608 tokens, against the call on all of them."""
    import torch
    from glt_amd import ops
    N = max([I] + [i0 + s for i0, s, _, _ in pl])
    wg, wu, wd, sl = make_layer(D, I, N, pl, True)
    dt = torch.bfloat16
    base = ops.BaseMLP(to_dev(wg, dt), to_dev(wu, dt), to_dev(wd, dt))
    gs = [ops.GraftSlice(s["i0"], s["s"], s["h0"], s["h"], *(to_dev(s[p], torch.float32) for p in ("gate", "up", "down")))
          .pack() for s in sl]
    g = torch.Generator(device="cuda").manual_seed(D)
    x = torch.randn((4608, D), generator=g, device="cuda").to(dt)
    dy = torch.randn((4608, D), generator=g, device="cuda").to(dt)

    def run(M):
        xs, res = x[:M].contiguous(), dy[:M].clone()
        y, gp, up, inter = ops.mlp_forward(base, gs, xs, N)
        dx, _ = ops.mlp_backward(base, gs, xs, dy[:M].contiguous(), N, gp, up, inter)
        ops.mlp_forward(base, gs, xs, N, residual=res)
        y2, _, _, inter2 = ops.mlp_forward(base, gs, xs, N, save=False)
        assert torch.equal(_bits(y), _bits(y2)) and torch.equal(_bits(inter), _bits(inter2)), M
        return dict(y=y, gate=gp, up=up, inter=inter, dx=dx, residual=res)

    full = run(4608)
    for M in MS:
        part = run(M)
        for k in full:
            assert torch.equal(_bits(full[k][:M]), _bits(part[k])), (k, M)


@pytest.mark.parametrize("V,D", [(32000, 2048), (4104, 1088)])
def test_head(dev, V, D):
    import torch
    from glt_amd import ops
    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.randn((4608, D), generator=g, device="cuda").bfloat16()
    w = torch.randn((V, D), generator=g, device="cuda").mul_(0.05).bfloat16()
    gr = torch.randn((2100, V), generator=g, device="cuda").bfloat16()
    y, dx = ops.lm_head_fwd(x, w), ops.lm_head_bwd(gr, w)
    for M in MS:
        assert torch.equal(_bits(ops.lm_head_fwd(x[:M].contiguous(), w)), _bits(y[:M])), M
        if V % 64 == 0:
            assert torch.equal(_bits(ops.lm_head_bwd(gr[:M].contiguous(), w)), _bits(dx[:M])), M


@pytest.mark.parametrize("I,M", [(8448, 8), (8448, 48), (8448, 100), (17408, 100)])
def test_mlp_weights_past_the_cache(dev, I, M):
    """Gate/up of 138 and 285 MB, and dX's as much, which one row of tiles (32 x
    32, 64 x 64, 128 x 64 and 128 x 128) loads non-temporally, against 600 tokens,
    which do not."""
    import torch
    from glt_amd import ops
    D = 4096
    g = torch.Generator(device="cuda").manual_seed(I)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").mul_(0.02).bfloat16()
    base = ops.BaseMLP(rn(I, D), rn(I, D), rn(D, I))
    x, dy = rn(600, D).mul_(50), rn(600, D).mul_(50)

    def run(n):
        _, gp, up, inter = ops.mlp_forward(base, [], x[:n].contiguous(), I)
        dx, _ = ops.mlp_backward(base, [], x[:n].contiguous(), dy[:n].contiguous(), I, gp, up, inter)
        return gp, up, inter, dx

    for a, b in zip(run(600), run(M)):
        assert torch.equal(_bits(a[:M]), _bits(b))


@pytest.mark.parametrize("V", [32000, 49152])
def test_head_weights_past_the_cache(dev, V):
    """The same of an LM head: 64 x 64 to 128 x 256 tiles."""
    import torch
    from glt_amd import ops
    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.randn((600, 4096), generator=g, device="cuda").bfloat16()
    w = torch.randn((V, 4096), generator=g, device="cuda").mul_(0.05).bfloat16()
    y = ops.lm_head_fwd(x, w)
    for M in (5, 48, 100):
        assert torch.equal(_bits(ops.lm_head_fwd(x[:M].contiguous(), w)), _bits(y[:M])), M


@pytest.mark.parametrize("D,I,pl,bf16", [
    (512, 1408, [(1408, 256, 0, 512)], False),
    (260, 390, [(7, 31, 3, 90), (390, 33, 0, 260)], False),
    (360, 500, [(500, 40, 0, 360)], True),  # not whole 64-K steps: the strided kernel
])
def test_strided_mlp(dev, D, I, pl, bf16):
    """The f32 path, and bf16 shapes off the fragment layout: from one tile to
    several 64 x 64 tiles per CU."""
    import torch
    from glt_amd import ops
    N = max([I] + [i0 + s for i0, s, _, _ in pl])
    wg, wu, wd, sl = make_layer(D, I, N, pl, bf16)
    dt = torch.bfloat16 if bf16 else torch.float32
    base = ops.BaseMLP(to_dev(wg, dt), to_dev(wu, dt), to_dev(wd, dt))
    gs = [ops.GraftSlice(s["i0"], s["s"], s["h0"], s["h"], *(to_dev(s[p], torch.float32) for p in ("gate", "up", "down")))
          .pack() for s in sl]
    g = torch.Generator(device="cuda").manual_seed(D)
    x = torch.randn((8300, D), generator=g, device="cuda").to(dt)
    dy = torch.randn((8300, D), generator=g, device="cuda").to(dt)

    def run(M):
        y, gp, up, inter = ops.mlp_forward(base, gs, x[:M].contiguous(), N)
        dx, _ = ops.mlp_backward(base, gs, x[:M].contiguous(), dy[:M].contiguous(), N, gp, up, inter)
        res = dy[:M].clone()
        ops.mlp_forward(base, gs, x[:M].contiguous(), N, residual=res)
        return dict(y=y, gate=gp, up=up, inter=inter, dx=dx, residual=res)

    full = run(8300)
    for M in MS:
        part = run(M)
        for k in full:
            assert torch.equal(_bits(full[k][:M]), _bits(part[k])), (k, M)


def test_eval_hash_of_any_batches(dev):
    """A model's logits over eight sequences, hashed as one batch and as batches
    of three, one and four."""
    import torch
    from glt_amd import ops
    D, I, S, V, T, H = 512, 1408, 256, 3200, 77, 4
    wg, wu, wd, sl = make_layer(D, I, I + S, [(I, S, 0, D)], True)
    dt = torch.bfloat16
    base = ops.BaseMLP(to_dev(wg, dt), to_dev(wu, dt), to_dev(wd, dt))
    gs = [ops.GraftSlice(sl[0]["i0"], S, 0, D, *(to_dev(sl[0][p], torch.float32) for p in ("gate", "up", "down"))).pack()]
    g = torch.Generator(device="cuda").manual_seed(T)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").mul_(0.05).to(dt)
    att = [rn(H * 128, D), rn(2 * 128, D), rn(2 * 128, D), rn(D, H * 128)]
    one = torch.ones(D, dtype=dt, device="cuda")
    embed, head = rn(V, D), rn(V, D)
    ids = torch.randint(0, V, (8, T), generator=g, device="cuda", dtype=torch.int32)

    def logits(rows):
        layer = ops.DecoderLayer(rows.shape[0], T, H, 2, *att, one, one, base, gs, I + S, rope_theta=10000.0, rms_eps=1e-5)
        return ops.Model([layer], embed, one, head).forward(rows).view(-1, V)

    def batches(cuts):
        out = []
        for rows in torch.split(ids, cuts):
            out.append((logits(rows.contiguous()), rows.contiguous()))
        return ops.eval_batches(out)["logits_hash"]

    assert batches([8]) == batches([3, 1, 4]) == batches([1] * 8)


@pytest.mark.parametrize("K", [1088, 1090])  # the MFMA path; the strided kernel
@pytest.mark.parametrize("M", [8, 64, 200, 512])
def test_infinities_and_nan_stay_in_their_rows(dev, M, K):
    """A row of infinities, one of NaN and one of the type's largest values
    leave every other row's bits as they are, and give what f32 sums give."""
    import torch
    from glt_amd import ops
    V = 4104
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    w = torch.randn((V, K), generator=g, device="cuda").mul_(0.05).bfloat16()
    bad = x.clone()
    bad[1], bad[3], bad[M - 2] = float("inf"), float("nan"), torch.finfo(torch.bfloat16).max
    y, z = ops.lm_head_fwd(x, w), ops.lm_head_fwd(bad, w)
    rows = [m for m in range(M) if m not in (1, 3, M - 2)]
    assert torch.equal(_bits(y[rows]), _bits(z[rows]))
    # infinity times weights of both signs; the largest value's products, all finite, sum past the range or not
    assert torch.all(torch.isnan(z[3])) and not torch.any(torch.isfinite(z[1]))
    ref = bad[M - 2].double() @ w.double().t()
    far = ref.abs() > 2 * torch.finfo(torch.float32).max
    assert far.any() and torch.all(~torch.isfinite(z[M - 2][far]))
