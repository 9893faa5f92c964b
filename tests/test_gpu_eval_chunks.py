"""Shadow-eval statistics and logits hash over every cut of the rows into
chunks (1024 to 16 per row), rows that start off 16 bytes, and rows shorter
than their chunks, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,V,ld", [(1, 1, 1, 1), (1, 2, 7, 9), (1, 3, 50257, 50257), (1, 5, 16392, 16400),
                                      (2, 130, 4099, 4099), (3, 400, 515, 520), (4, 4099, 33, 33), (2, 8200, 24, 24)])
def test_eval_stats_cuts(dev, B, T, V, ld):
    """Hash exact; sums are f64 on both sides; nll within the f32 rounding of
    max + log(sum exp) - label, 2^-22 of its terms per row."""
    import torch
    from glt_amd import ops
    g = torch.Generator().manual_seed(B * T + V)
    full = (torch.randn((B * T, ld), generator=g) * 3).bfloat16()
    ids = torch.randint(0, V, (B, T), generator=g, dtype=torch.int32)
    logits = full.cuda()[:, :V]
    h0 = 0x9E3779B97F4A7C15
    x = full[:, :V].float().numpy().reshape(B, T, V)
    for h in (O.FNV_BASIS, h0):
        r = ops.eval_stats(logits, ids.cuda(), h)
        ref = O.eval_stats(x, ids.numpy(), h) if T > 1 else None
        assert r["logits_hash"] == O.eval_hash_reference(x.reshape(B * T, V), h)
        assert r["count"] == B * (T - 1)
        assert abs(r["logits_sum"] - float(x.astype(np.float64).sum())) <= 1e-12 * float(np.abs(x).astype(np.float64).sum())
        assert abs(r["logits_sumsq"] - float((x.astype(np.float64) ** 2).sum())) <= 1e-12 * float((x.astype(np.float64) ** 2).sum())
        if ref:
            assert abs(r["total_nll"] - ref["total_nll"]) <= 2.0 ** -22 * (np.log(V) + 4 * np.abs(x).max()) * B * T


@pytest.mark.parametrize("V", [33, 32, 4099, 4096])
def test_logits_at_the_ends_of_the_range(dev, V):
    """Rows that hold the type's largest value, only its lowest, a mask of the
    lowest and of -inf beside ordinary logits, and rows of infinities: nll as
    max + log(sum exp(x - max)) - label gives it in f64, within f32 rounding of
    its terms, NaN where that is NaN."""
    import torch
    from glt_amd import ops
    big = torch.finfo(torch.bfloat16).max
    g = torch.Generator().manual_seed(V)
    base = (torch.randn((2, V), generator=g) * 3).bfloat16()
    rows = []
    for kind in range(8):
        r = base.clone()
        if kind == 0: r[0, V // 2] = big
        if kind == 1: r[0] = -big
        if kind == 2: r[0, ::2] = -big
        if kind == 3: r[0, 1::2] = -float("inf")
        if kind == 4: r[0, 1:] = -float("inf")
        if kind == 5: r[0] = -float("inf")
        if kind == 6: r[0, V - 1] = float("inf")
        if kind == 7: r[0] = torch.where(r[0] > 0, 1.5e38, -1.5e38)
        rows.append(r)
    for kind, r in enumerate(rows):
        for label in (0, V - 2):
            ids = torch.tensor([[0, label]], dtype=torch.int32)
            got = ops.eval_stats(r.cuda(), ids.cuda())
            z = r[0].double()
            m = z.max()
            want = (m + torch.log(torch.exp(z - m).sum()) - z[label]).item()
            nll = got["total_nll"]
            if want != want:
                assert nll != nll, (kind, label, nll)
            elif abs(want) == float("inf"):
                assert nll == want, (kind, label, nll)
            else:
                terms = abs(m.item()) + abs(z[label].item()) + np.log(V)
                assert abs(nll - want) <= 2.0 ** -22 * terms, (kind, label, nll, want)


def test_workspace_of_the_largest_batch(dev):
    """One workspace, sized once for the longest batch, for shorter batches
    whose rows are cut into more chunks: hash against the oracle, and the bytes
    past the workspace untouched."""
    import ctypes
    import torch
    from glt_amd import _ffi as F
    lib = F.load()
    V, largest = 40, 2052
    n, guard = lib.glt_eval_stats_workspace_size(1, largest), 4 << 20
    ws = torch.full((n + guard,), 0x5A, dtype=torch.uint8, device="cuda")
    g = torch.Generator().manual_seed(V)
    logits = (torch.randn((largest, V), generator=g) * 3).bfloat16()
    ids = torch.randint(0, V, (largest,), generator=g, dtype=torch.int32)
    ld, di = logits.cuda(), ids.cuda()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    for T in (largest, 2048, 1024, 257, 256, 1):
        r = F.EvalResult()
        assert lib.glt_eval_stats_workspace_size(1, T) <= n
        F.call("glt_eval_stats", p(ld), V, p(di), 1, T, V, F.EVAL_HASH_REFERENCE, O.FNV_BASIS, ctypes.byref(r), p(ws), n,
               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert r.logits_hash == O.eval_hash_reference(logits[:T].float().numpy(), O.FNV_BASIS), T
        assert r.count == T - 1
    assert torch.all(ws[n:] == 0x5A).item()
