"""The library's work as its users call it: sizes, inputs, one pass, and what
a pass cannot do without.

Every case is one kind of call with its sizes:

* train_step   RMSNorm, grafted MLP forward, graft-only backward with the
               norm's backward, clipped AdamW: one optimizer step of one
               layer's graft (bf16, f32 upstream gradient).
* mlp_fwd      the grafted MLP forward alone, nothing saved (inference).
* mlp_f32      the f32 path, forward and graft-only backward.
* layer        a decoder layer's forward and its MLP's backward by
               recompute, as a training step with recompute runs it.
* attention    causal GQA attention of ragged sequences.
* model        embedding, decoder layers, final norm, LM head: the logits of
               a prompt.
* head_loss    LM head, masked cross-entropy with its gradient, and the
               gradient back through the head.
* eval         the shadow-eval statistics and logits hash of a batch.
* bake         shadow_bake materialising grafted base matrices.

listed() holds one to three sizes of each kind, draw() spreads over the
ranges they stand for.
"""
import ctypes

import torch

from glt_amd import _ffi as F
from glt_amd import ops

DEV = "cuda"
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
EPS = 1e-5
THETA = 500000.0
HD = 128
LR, B1, B2, AEPS, WD, CLIP = 1e-4, 0.9, 0.999, 1e-8, 0.01, 1.0


# ------------------------------------------------------------------ cases
def listed():
    """Sizes of this repository's benchmark, tests and configurations, and
    ragged ones between them. `slices` lists a layer's graft slices as
    "i_start:s:h_start:h"."""
    return [
        # the benchmark's step: 8 x 2048 tokens, one appended slice
        dict(name="train_step_16384", kind="train_step", M=16384, D=4096, I=14336, slices="14336:1024:0:4096"),
        # a packed batch of documents that fills no tile: odd token count
        dict(name="train_step_1999", kind="train_step", M=1999, D=4096, I=14336, slices="14336:1024:0:4096"),
        # the reference's default hidden size and slice (2048, 11008, 2752), the
        # slice in place over existing neurons, one short sequence
        dict(name="train_step_512_inplace", kind="train_step", M=512, D=2048, I=11008, slices="2752:2752:0:2048"),
        # the f32 configuration: 4 x 128 tokens, hidden 512, base 1408, slice 256
        dict(name="mlp_f32_512", kind="mlp_f32", M=512, D=512, I=1408, slices="1408:256:0:512"),
        # a handful of tokens at inference: bound by the weights and launches
        dict(name="mlp_fwd_8", kind="mlp_fwd", M=8, D=4096, I=14336, slices="14336:1024:0:4096"),
        # a prompt through four stacked slices
        dict(name="mlp_fwd_200_stacked", kind="mlp_fwd", M=200, D=4096, I=14336,
             slices="14336:512:0:4096,14848:512:0:4096,15360:512:0:4096,15872:512:0:4096"),
        # the decoder layer of the benchmark, forward and recompute backward
        dict(name="layer_2x4096", kind="layer", B=2, T=4096, D=4096, I=14336, Hq=32, Hkv=8,
             slices="14336:1024:0:4096"),
        # ragged sequences
        dict(name="attention_3x1531", kind="attention", B=3, T=1531, Hq=32, Hkv=8),
        # two short prompts through a whole (two-layer) model to logits
        dict(name="model_2x77", kind="model", B=2, T=77, D=4096, I=14336, Hq=32, Hkv=8, V=128256, L=2,
             slices="14336:1024:0:4096"),
        # the loss end of a training step
        dict(name="head_loss_4x500", kind="head_loss", B=4, T=500, D=4096, V=128256),
        # a shadow-eval batch of short texts
        dict(name="eval_4x512", kind="eval", B=4, T=512, V=128256),
        # four layers' matrices baked with one appended slice
        dict(name="bake_4", kind="bake", L=4, D=4096, I=14336, N=15360, placements="14336:1024:0:4096",
             graft="f32"),
    ]


def _log_int(rng, lo, hi):
    """Log-uniform, every second one odd or otherwise unaligned."""
    import math
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v if rng.random() < 0.5 or v < 256 else v // 64 * 64))


def _mlp_dims(rng):
    """(D, I) and slices: the two model widths here, one to four slices of a
    multiple of 64 neurons, appended or in place."""
    D, I = rng.choice([(4096, 14336), (2048, 11008)])
    n = rng.choice([1, 1, 1, 2, 4])
    s = 64 * rng.randint(2, 16)
    if rng.random() < 0.3:  # in place over existing neurons
        i0 = 64 * rng.randint(0, (I - n * s) // 64)
    else:
        i0 = I
    return D, I, ",".join("%d:%d:0:%d" % (i0 + j * s, s, D) for j in range(n))


def draw(rng):
    kind = rng.choice(["train_step", "train_step", "mlp_fwd", "mlp_fwd", "mlp_f32", "layer", "attention", "model",
                       "head_loss", "eval", "bake"])
    if kind == "train_step":
        D, I, sl = _mlp_dims(rng)
        return dict(kind=kind, M=_log_int(rng, 64, 12288), D=D, I=I, slices=sl)
    if kind == "mlp_fwd":
        D, I, sl = _mlp_dims(rng)
        return dict(kind=kind, M=_log_int(rng, 1, 8192), D=D, I=I, slices=sl)
    if kind == "mlp_f32":
        D, I = 64 * rng.randint(4, 16), 64 * rng.randint(8, 44)
        s = 32 * rng.randint(2, 12)
        i0 = I if rng.random() < 0.7 else rng.randint(0, I - s)
        return dict(kind=kind, M=_log_int(rng, 64, 2048), D=D, I=I, slices="%d:%d:0:%d" % (i0, s, D))
    if kind == "layer":
        D, I, sl = _mlp_dims(rng)
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, T=_log_int(rng, 64, 8192 // B), D=D, I=I, Hq=D // HD, Hkv=rng.choice([4, 8]),
                    slices=sl)
    if kind == "attention":
        B = rng.randint(1, 8)
        Hkv = rng.choice([4, 8])
        return dict(kind=kind, B=B, T=_log_int(rng, 32, 16384 // B), Hq=Hkv * rng.choice([1, 2, 4]), Hkv=Hkv)
    if kind == "model":
        D, I, sl = _mlp_dims(rng)
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, T=_log_int(rng, 8, 1024 // B), D=D, I=I, Hq=D // HD, Hkv=rng.choice([4, 8]),
                    V=rng.choice([32000, 49152, 128256]), L=rng.randint(1, 3), slices=sl)
    if kind == "head_loss":
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, T=_log_int(rng, 32, 4096 // B), D=rng.choice([2048, 4096]),
                    V=rng.choice([32000, 49152, 128256]))
    if kind == "eval":
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, T=_log_int(rng, 16, 8192 // B), V=rng.choice([32000, 50257, 128256]))
    D, I = rng.choice([(4096, 14336), (2048, 11008)])
    s = 64 * rng.randint(2, 32)
    h = D if rng.random() < 0.5 else rng.randint(D // 4, D)  # a slice may cover part of the hidden columns
    app = rng.random() < 0.6
    i0 = I if app else rng.randint(0, I - s)
    return dict(kind="bake", L=rng.randint(1, 4), D=D, I=I, N=I + s if app else I,
                placements="%d:%d:%d:%d" % (i0, s, rng.randint(0, D - h), h), graft=rng.choice(["f32", "bf16"]))


def _slices(text):
    return [tuple(int(v) for v in s.split(":")) for s in text.split(",")]


def _width(case):
    """N: the base neurons and the appended ones."""
    return max([case["I"]] + [i0 + s for i0, s, _, _ in _slices(case["slices"])])


# ----------------------------------------------------------------- inputs
class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)

    def normal(self, shape, std=1.0, mean=0.0, dtype=BF):
        t = torch.empty(shape, dtype=F32, device=DEV)
        t.normal_(mean, std, generator=self.g)
        return t if dtype == F32 else t.to(dtype)

    def ints(self, shape, hi, dtype=torch.int32):
        return torch.randint(0, hi, shape, generator=self.g, device=DEV, dtype=torch.int64).to(dtype)


def _mlp_inputs(d, case, dtype=BF):
    """Base weights and slice masters of one MLP (weights ~ N(0, 0.02))."""
    D, I = case["D"], case["I"]
    w = [d.normal((I, D), 0.02, dtype=dtype), d.normal((I, D), 0.02, dtype=dtype), d.normal((D, I), 0.02, dtype=dtype)]
    masters = [d.normal((3, s, h), 0.02, dtype=F32) for _, s, _, h in _slices(case["slices"])]
    return w, masters


def _mlp_objects(case, w, masters):
    base = ops.BaseMLP(*w)
    sl = [ops.GraftSlice(i0, s, h0, h, m[0], m[1], m[2])
          for (i0, s, h0, h), m in zip(_slices(case["slices"]), masters)]
    if w[0].dtype == BF:
        for s in sl:
            s.pack()
    return base, sl


def _layer_inputs(d, case):
    D, nq, nk = case["D"], case["Hq"] * HD, case["Hkv"] * HD
    att = [d.normal((nq, D), 0.02), d.normal((nk, D), 0.02), d.normal((nk, D), 0.02), d.normal((D, nq), 0.02),
           d.normal(D, 0.02, 1.0), d.normal(D, 0.02, 1.0)]
    return att, _mlp_inputs(d, case)


def _inputs(case, seed):
    """The tensors of a case, the same for prepare() and exact()."""
    d, kind = _Draw(seed), case["kind"]
    if kind == "train_step":
        M, D = case["M"], case["D"]
        return dict(x=d.normal((M, D)), gamma=d.normal(D, 0.02, 1.0), dy=d.normal((M, D), dtype=F32),
                    mlp=_mlp_inputs(d, case))
    if kind == "mlp_fwd":
        return dict(x=d.normal((case["M"], case["D"])), mlp=_mlp_inputs(d, case))
    if kind == "mlp_f32":
        M, D = case["M"], case["D"]
        return dict(x=d.normal((M, D), dtype=F32), dy=d.normal((M, D), dtype=F32), mlp=_mlp_inputs(d, case, F32))
    if kind == "layer":
        M, D = case["B"] * case["T"], case["D"]
        return dict(x=d.normal((M, D)), dy=d.normal((M, D), dtype=F32), layer=_layer_inputs(d, case))
    if kind == "attention":
        B, T = case["B"], case["T"]
        return dict(q=d.normal((B, T, case["Hq"], HD)), k=d.normal((B, T, case["Hkv"], HD)),
                    v=d.normal((B, T, case["Hkv"], HD)))
    if kind == "model":
        D, V = case["D"], case["V"]
        return dict(layers=[_layer_inputs(d, case) for _ in range(case["L"])], embed=d.normal((V, D)),
                    final=d.normal(D, 0.02, 1.0), head=d.normal((V, D), 0.02), ids=d.ints((case["B"], case["T"]), V))
    if kind == "head_loss":
        B, T, D, V = case["B"], case["T"], case["D"], case["V"]
        return dict(x=d.normal((B * T, D)), head=d.normal((V, D), 0.02), ids=d.ints((B, T), V),
                    ood=(d.ints((B, T), 3) == 0).to(torch.int32))  # a third of the positions excluded
    if kind == "eval":
        B, T, V = case["B"], case["T"], case["V"]
        return dict(logits=d.normal((B * T, V), 2.0), ids=d.ints((B, T), V))
    L, D, I = case["L"], case["D"], case["I"]
    gd = F32 if case["graft"] == "f32" else BF
    return dict(gate=[d.normal((I, D), 0.02) for _ in range(L)], up=[d.normal((I, D), 0.02) for _ in range(L)],
                down=[d.normal((D, I), 0.02) for _ in range(L)],
                grafts=[[d.normal((3, s, h), 0.02, dtype=gd) for _ in range(L)]
                        for _, s, _, h in _slices(case["placements"])])


# ---------------------------------------------------------------- prepare
def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    s["kind"] = kind
    if kind == "train_step":
        _prepare_step(case, s)
    elif kind in ("mlp_fwd", "mlp_f32"):
        s["N"] = _width(case)
        s["base"], s["slices"] = _mlp_objects(case, *s.pop("mlp"))
        if kind == "mlp_f32":
            s["ws"] = torch.empty(ops.mlp_backward_workspace(s["base"], s["slices"], case["M"], s["N"]),
                                  dtype=torch.uint8, device=DEV)
    elif kind == "layer":
        s["layer"] = _layer_object(case, *s["layer"])
        s["N"] = _width(case)
        s["ws"] = torch.empty(_recompute_ws(case, s["layer"], s["N"]), dtype=torch.uint8, device=DEV)
    elif kind == "model":
        layers = [_layer_object(case, *li) for li in s.pop("layers")]
        s["model"] = ops.Model(layers, s["embed"], s["final"], s["head"])
    elif kind == "head_loss":
        s["prepared"] = torch.empty(F.load().glt_lm_head_prepared_size(case["V"], case["D"]), dtype=torch.uint8,
                                    device=DEV)
        F.call("glt_lm_head_prepare", _p(s["head"]), case["V"], case["D"], _p(s["prepared"]), ops._stream())
        s["B"], s["T"] = case["B"], case["T"]
    elif kind == "bake":
        D, I, N, L = case["D"], case["I"], case["N"], case["L"]
        s["dims"] = dict(D=D, I=I, N=N)
        s["placements"] = _slices(case["placements"])
        for name, shape in (("gate_out", (N, D)), ("up_out", (N, D)), ("down_out", (D, N))):
            s[name] = [torch.empty(shape, dtype=BF, device=DEV) for _ in range(L)]
    return s


def _layer_object(case, att, mlp):
    base, sl = _mlp_objects(case, *mlp)
    return ops.DecoderLayer(case["B"], case["T"], case["Hq"], case["Hkv"], *att, base, sl, _width(case),
                            rope_theta=THETA, rms_eps=EPS)


def _recompute_ws(case, layer, N):
    d, _keep = ops._desc(layer.base, layer.slices, case["B"] * case["T"], N, True, recompute=True, dy_f32=True)
    return F.load().glt_mlp_bwd_workspace_size(ctypes.byref(d))


def _prepare_step(case, s):
    """Buffers and descriptors of the C ABI, allocated once as a training
    program does."""
    M, D, N = case["M"], case["D"], _width(case)
    w, masters = s.pop("mlp")
    base, sl = _mlp_objects(case, w, masters)
    n, lib = len(sl), F.load()
    new = lambda shape, dt: torch.empty(shape, dtype=dt, device=DEV)
    s.update(base=base, slices=sl, masters=masters, M=M, D=D, N=N, i=0,
             grads=[torch.zeros_like(m) for m in masters], m=[torch.zeros_like(m) for m in masters],
             v=[torch.zeros_like(m) for m in masters],
             xn=new((M, D), BF), var=new(M, F32), y=new((M, D), BF), g=new((M, N), BF), u=new((M, N), BF),
             inter=new((M, N), BF), dx=new((M, D), F32), dx_norm=new((M, D), F32))
    s["arr"] = ops._slices_array(sl)
    s["desc"] = F.MlpDesc(M, D, case["I"], N, F.DTYPE_BF16, F.MLP_EXPLICIT | F.MLP_DY_F32, n, s["arr"], None)
    s["bw"] = base.c_struct()
    s["ws"] = new(lib.glt_mlp_bwd_workspace_size(ctypes.byref(s["desc"])), torch.uint8)
    s["clip_ws"] = new(lib.glt_adamw_workspace_size(0), torch.uint8)
    s["gg"] = (F.GraftGrads * n)(*[F.GraftGrads(g[0].data_ptr(), g[1].data_ptr(), g[2].data_ptr())
                                   for g in s["grads"]])
    for k in ("grads", "m", "v"):
        s[k + "_ptr"] = F.ptr_array([t.data_ptr() for t in s[k]])
    s["packed_ptr"] = F.ptr_array([x.packed.data_ptr() for x in sl])


# -------------------------------------------------------------------- run
def run(s):
    return _RUN[s["kind"]](s)


def _run_step(s):
    st = ops._stream()
    M, D, desc, bw = s["M"], s["D"], ctypes.byref(s["desc"]), ctypes.byref(s["bw"])
    F.call("glt_rmsnorm_fwd", _p(s["x"]), _p(s["gamma"]), _p(s["xn"]), _p(s["var"]), M, D, EPS, st)
    F.call("glt_mlp_fwd", desc, bw, _p(s["xn"]), _p(s["y"]), _p(s["g"]), _p(s["u"]), _p(s["inter"]), st)
    F.call("glt_mlp_rmsnorm_bwd", desc, bw, _p(s["xn"]), _p(s["dy"]), _p(s["g"]), _p(s["u"]), _p(s["inter"]),
           _p(s["dx"]), s["gg"], _p(s["ws"]), s["ws"].numel(), _p(s["x"]), _p(s["gamma"]), _p(s["var"]), EPS,
           _p(s["dx_norm"]), st)
    F.call("glt_adamw_graft_step", s["arr"], len(s["slices"]), s["grads_ptr"], s["m_ptr"], s["v_ptr"],
           s["packed_ptr"], 7, s["i"], LR, B1, B2, AEPS, WD, CLIP, _p(s["clip_ws"]), s["clip_ws"].numel(), st)
    s["i"] += 1
    return dict(y=s["y"], dx=s["dx"], dx_norm=s["dx_norm"], grads=s["grads"], masters=s["masters"], m=s["m"],
                v=s["v"])


def _run_mlp_fwd(s):
    y, _, _, inter = ops.mlp_forward(s["base"], s["slices"], s["x"], s["N"], save=False)
    return dict(y=y, inter=inter)


def _run_mlp_f32(s):
    y, g, u, inter = ops.mlp_forward(s["base"], s["slices"], s["x"], s["N"])
    dx, grads = ops.mlp_backward(s["base"], s["slices"], s["x"], s["dy"], s["N"], g, u, inter, workspace=s["ws"])
    return dict(y=y, dx=dx, grads=grads)


def _run_layer(s):
    layer = s["layer"]
    x, x_ffn, var = layer.forward(s["x"].clone())  # the layer updates its input in place
    dx, grads = ops.mlp_backward(layer.base, layer.slices, x_ffn, s["dy"], s["N"], recompute=True,
                                 workspace=s["ws"])
    return dict(x=x, x_ffn=x_ffn, dx=dx, grads=grads)


def _run_attention(s):
    return ops.attention(s["q"], s["k"], s["v"])


def _run_model(s):
    return s["model"].forward(s["ids"])


def _run_head_loss(s):
    B, T = s["B"], s["T"]
    logits = ops.lm_head_fwd(s["x"], s["head"], s["prepared"])
    V = logits.shape[1]
    stats, grad, ce = ops.masked_ce(logits.view(B, T, V), s["ids"], s["ood"], ce_per_token=True)
    dx = ops.lm_head_bwd(grad.view(B * T, V), s["head"], s["prepared"])
    return dict(logits=logits, stats=stats, grad=grad, ce=ce, dx=dx)


def _run_eval(s):
    r = ops.eval_stats(s["logits"], s["ids"])
    r["logits_hash"] = ctypes.c_int64(r["logits_hash"]).value  # the same 64 bits, signed
    return r


def _run_bake(s):
    state = F.ModelState(0)
    ops.shadow_bake(state, s["gate"], s["up"], s["down"], s["grafts"], s["placements"], materialize=True,
                    gate_out=s["gate_out"], up_out=s["up_out"], down_out=s["down_out"], **s["dims"])
    return dict(gate=s["gate_out"], up=s["up_out"], down=s["down_out"])


_RUN = {"train_step": _run_step, "mlp_fwd": _run_mlp_fwd, "mlp_f32": _run_mlp_f32, "layer": _run_layer,
        "attention": _run_attention, "model": _run_model, "head_loss": _run_head_loss, "eval": _run_eval,
        "bake": _run_bake}


# ------------------------------------------------------------------- work
def _mlp_work(case, M, fwd, bwd, save, es=2):
    """(bytes, flops) of the MLP's parts: each weight, activation and
    gradient read or written once."""
    D, I, N = case["D"], case["I"], _width(case)
    sl = _slices(case["slices"])
    cols = I * D + sum(s * h for _, s, _, h in sl)  # weight elements of one projection
    b = f = 0
    if fwd:
        f += 2 * M * cols * 3
        b += 3 * cols * es + 2 * M * D * es + (3 if save else 1) * M * N * es
    if bwd:
        f += 2 * M * cols * 3 + 3 * sum(2 * M * s * h for _, s, _, h in sl)
        b += 3 * cols * es + M * D * (es + 4 + 4) + 3 * M * N * es + 3 * 4 * sum(s * h for _, s, _, h in sl)
    return b, f


def _layer_fwd_work(case, M):
    D, nq, nk, T = case["D"], case["Hq"] * HD, case["Hkv"] * HD, case["T"]
    b, f = _mlp_work(case, M, True, False, False)
    w = D * (2 * nq + 2 * nk)
    f += 2 * M * w + 2 * M * T * nq  # causal: half of 4 * T^2 * nq per sequence
    b += w * 2 + 2 * M * D * 2
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "train_step":
        M, D = case["M"], case["D"]
        b, f = _mlp_work(case, M, True, True, True)
        b += 2 * M * D * 2 + M * D * (2 + 4)  # the norm forward, and its backward beside dx
        b += 28 * 3 * sum(s * h for _, s, _, h in _slices(case["slices"]))  # AdamW's masters, moments, gradients
    elif kind == "mlp_fwd":
        b, f = _mlp_work(case, case["M"], True, False, False)
    elif kind == "mlp_f32":
        b, f = _mlp_work(case, case["M"], True, True, True, es=4)
    elif kind == "layer":
        M = case["B"] * case["T"]
        b, f = _layer_fwd_work(case, M)
        b2, f2 = _mlp_work(case, M, False, True, False)
        N = _width(case)
        f += f2 + 2 * (f2 - 3 * sum(2 * M * s * h for _, s, _, h in _slices(case["slices"]))) // 3  # gate/up again
        b += b2 - 3 * M * N * 2
    elif kind == "attention":
        B, T, Hq, Hkv = case["B"], case["T"], case["Hq"], case["Hkv"]
        b, f = 2 * B * T * HD * (2 * Hq + 2 * Hkv), 2 * B * T * T * Hq * HD
    elif kind == "model":
        M, D, V = case["B"] * case["T"], case["D"], case["V"]
        b, f = _layer_fwd_work(case, M)
        b, f = b * case["L"] + V * D * 2 + M * (V + D) * 2, f * case["L"] + 2 * M * V * D
    elif kind == "head_loss":
        M, D, V = case["B"] * case["T"], case["D"], case["V"]
        b, f = V * D * 2 + M * D * (2 + 4) + 2 * M * V * 2, 4 * M * V * D
    elif kind == "eval":
        b, f = case["B"] * case["T"] * case["V"] * 2, 0
    else:
        D, I, N, L = case["D"], case["I"], case["N"], case["L"]
        g = 4 if case["graft"] == "f32" else 2
        b = L * 3 * (2 * I * D + 2 * N * D + g * sum(s * h for _, s, _, h in _slices(case["placements"])))
        f = 0
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the distance measured between the path and its
    64-bit result (bf16 kinds), or between two orders of its f32 sums."""
    kind = case["kind"]
    if kind == "bake":
        return "exact"  # one f32 add per element, rounded once
    return {"rel": {"train_step": 1.5e-2, "mlp_fwd": 1.2e-2, "mlp_f32": 5e-6, "layer": 2e-2, "attention": 8e-3,
                    "model": 4e-2, "head_loss": 8e-3, "eval": 1e-5}[kind]}


# ------------------------------------------------------------------ exact
def _norm64(x, w):
    var = (x * x).mean(-1, keepdim=True)
    return x * torch.rsqrt(var + EPS) * w, var


def _weights64(case, mlp):
    """Base with every slice added: gate/up [N, D], down [D, N] in f64."""
    (wg, wu, wd), masters = mlp
    N, D, I = _width(case), case["D"], case["I"]
    G, U, Dn = (torch.zeros((N, D), dtype=F64, device=DEV) for _ in range(3))
    G[:I], U[:I], Dn[:I] = wg.double(), wu.double(), wd.double().t()
    for (i0, s, h0, h), m in zip(_slices(case["slices"]), masters):
        md = (m if wg.dtype == F32 else m.to(BF)).double()
        G[i0:i0 + s, h0:h0 + h] += md[0]
        U[i0:i0 + s, h0:h0 + h] += md[1]
        Dn[i0:i0 + s, h0:h0 + h] += md[2]
    return G, U, Dn


def _mlp64(x, W):
    G, U, Dn = W
    g, u = x @ G.t(), x @ U.t()
    inter = torch.nn.functional.silu(g) * u
    return inter @ Dn, g, u, inter


def _mlp_bwd64(case, x, dy, W, g, u, inter):
    G, U, Dn = W
    di = dy @ Dn.t()
    sg = torch.sigmoid(g)
    dg, du = di * u * (sg * (1 + g * (1 - sg))), di * (g * sg)
    del di, sg
    dx = dg @ G + du @ U
    grads = []
    for i0, s, h0, h in _slices(case["slices"]):
        xs, ds = x[:, h0:h0 + h], dy[:, h0:h0 + h]
        grads.append([dg[:, i0:i0 + s].t() @ xs, du[:, i0:i0 + s].t() @ xs, inter[:, i0:i0 + s].t() @ ds])
    return dx, grads


def _rope64(t):
    """t [B, T, H, 128] rotated in halves."""
    T, half = t.shape[1], HD // 2
    inv = 1.0 / (THETA ** (torch.arange(half, dtype=F64, device=DEV) * 2 / HD))
    ang = torch.arange(T, dtype=F64, device=DEV)[:, None] * inv[None]
    c, s = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
    a, b = t[..., :half], t[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention64(q, k, v):
    B, T, Hq, _ = q.shape
    rep = Hq // k.shape[2]
    out = torch.empty_like(q)
    future = torch.ones((T, T), dtype=torch.bool, device=DEV).triu(1)
    for b in range(B):
        for h in range(Hq):
            s = (q[b, :, h] @ k[b, :, h // rep].t()) * HD ** -0.5
            s = torch.softmax(s.masked_fill_(future, float("-inf")), -1)
            out[b, :, h] = s @ v[b, :, h // rep]
    return out


def _layer64(case, x, att, mlp):
    """x [M, D] -> layer output, MLP input and (weights, saved activations)."""
    B, T, Hq, Hkv = case["B"], case["T"], case["Hq"], case["Hkv"]
    wq, wk, wv, wo, ln_in, ln_post = (t.double() for t in att)
    xn, _ = _norm64(x, ln_in)
    q = _rope64((xn @ wq.t()).view(B, T, Hq, HD))
    k = _rope64((xn @ wk.t()).view(B, T, Hkv, HD))
    v = (xn @ wv.t()).view(B, T, Hkv, HD)
    x = x + _attention64(q, k, v).view(B * T, Hq * HD) @ wo.t()
    x_ffn, _ = _norm64(x, ln_post)
    W = _weights64(case, mlp)
    y, g, u, inter = _mlp64(x_ffn, W)
    return x + y, x_ffn, (W, g, u, inter)


def exact(case, seed):
    kind = case["kind"]
    t = _inputs(case, seed)
    if kind == "train_step":
        x, gamma, dy = t["x"].double(), t["gamma"].double(), t["dy"].double()
        W = _weights64(case, t["mlp"])
        xn, var = _norm64(x, gamma)
        y, g, u, inter = _mlp64(xn, W)
        dx, grads = _mlp_bwd64(case, xn, dy, W, g, u, inter)
        del g, u, inter, W
        r = torch.rsqrt(var + EPS)
        dxn = dx * r * gamma - x * ((dx * x * gamma).mean(-1, keepdim=True) * r ** 3)
        grads = [torch.stack(gs) for gs in grads]
        norm = torch.sqrt(sum((gs * gs).sum() for gs in grads) + 1e-8)
        sc = torch.where(norm > CLIP, CLIP / norm, torch.ones_like(norm))
        w, m, v = [], [], []
        for gs, w0 in zip(grads, t["mlp"][1]):
            w0 = w0.double()
            m.append((1 - B1) * gs * sc)
            v.append((1 - B2) * (gs * sc) ** 2)
            w.append(w0 - LR * (m[-1] / (1 - B1)) / (torch.sqrt(v[-1] / (1 - B2)) + AEPS) - LR * WD * w0)
        return dict(y=y, dx=dx, dx_norm=dxn, grads=grads, masters=w, m=m, v=v)
    if kind == "mlp_fwd":
        y, _, _, inter = _mlp64(t["x"].double(), _weights64(case, t["mlp"]))
        return dict(y=y, inter=inter)
    if kind == "mlp_f32":
        x, dy = t["x"].double(), t["dy"].double()
        W = _weights64(case, t["mlp"])
        y, g, u, inter = _mlp64(x, W)
        dx, grads = _mlp_bwd64(case, x, dy, W, g, u, inter)
        return dict(y=y, dx=dx, grads=grads)
    if kind == "layer":
        x, x_ffn, (W, g, u, inter) = _layer64(case, t["x"].double(), *t["layer"])
        dx, grads = _mlp_bwd64(case, x_ffn, t["dy"].double(), W, g, u, inter)
        return dict(x=x, x_ffn=x_ffn, dx=dx, grads=grads)
    if kind == "attention":
        return _attention64(t["q"].double(), t["k"].double(), t["v"].double())
    if kind == "model":
        x = t["embed"].double()[t["ids"].reshape(-1).long()]
        for li in t["layers"]:
            x, _, _ = _layer64(case, x, *li)
        x, _ = _norm64(x, t["final"].double())
        return x @ t["head"].double().t()
    if kind == "head_loss":
        return _head_loss64(case, t)
    if kind == "eval":
        return _eval64(case, t)
    D, I, N = case["D"], case["I"], case["N"]
    out = dict(gate=[], up=[], down=[])
    for l in range(case["L"]):
        for p, name in enumerate(("gate", "up", "down")):
            full = torch.zeros((N, D), dtype=F64, device=DEV)
            full[:I] = t[name][l].double().t() if p == 2 else t[name][l].double()
            for j, (i0, s, h0, h) in enumerate(_slices(case["placements"])):
                full[i0:i0 + s, h0:h0 + h] += t["grafts"][j][l][p].double()
            out[name].append(full.t().contiguous() if p == 2 else full)
    return out


def _head_loss64(case, t):
    B, T, V = case["B"], case["T"], case["V"]
    head = t["head"].double()
    logits = t["x"].double() @ head.t()
    ids = t["ids"].long()
    z = logits.view(B, T, V)[:, :T - 1].reshape(-1, V)
    lab = ids[:, 1:].reshape(-1)
    mask = (t["ood"][:, 1:].reshape(-1) == 0).double()
    n = mask.sum().clamp(min=1.0)
    rows = torch.arange(lab.numel(), device=DEV)
    lse = torch.logsumexp(z, -1)
    xl = z[rows, lab]
    ce = lse - xl
    g = torch.softmax(z, -1)
    pl = g[rows, lab].clone()
    g[rows, lab] -= 1.0
    g *= (mask / n)[:, None]
    grad = torch.zeros((B, T, V), dtype=F64, device=DEV)
    grad[:, :T - 1] = g.view(B, T - 1, V)
    del g, z
    stats = torch.stack([(ce * mask).sum() / n, (xl * mask).sum() / n, (pl * mask).sum() / n, n])
    return dict(logits=logits, stats=stats, grad=grad, ce=ce, dx=grad.view(B * T, V) @ head)


def _eval64(case, t):
    B, T, V = case["B"], case["T"], case["V"]
    ids = t["ids"].long()
    s = s2 = nll = 0.0
    for b in range(B):
        z = t["logits"].view(B, T, V)[b].double()
        s, s2 = s + float(z.sum()), s2 + float((z * z).sum())
        if T > 1:
            z = z[:T - 1]
            nll += float((torch.logsumexp(z, -1) - z.gather(1, ids[b, 1:, None])[:, 0]).sum())
    n = B * (T - 1)
    return {"total_nll": nll, "count": n, "ce": nll / max(n, 1), "logits_sum": s, "logits_sumsq": s2,
            "logits_hash": None}
