"""Timing cases of the attention path: what a host program has this library do, through the entry points it calls.

A case is one pass over inputs that are already on the device, with the layers, handles and models a program keeps:

  block     a training step of a transformer block (``TransformerBlockLayer``): parameter gradients cleared, forward,
            backward; GPT style (LayerNorm, MLP) or Llama style (RMSNorm, rotary attention, gated MLP), float or double
            base type, attention through the explicit chain (the layer's default) or the attention handle
  head      a training step of a language model's output: inner product to the vocabulary, softmax, both backward
  mlp       a training step of a block's MLP kept in 16-bit storage: inner product, activation, inner product
  attn      inference of a causal self attention layer over whole sequences (prefill), its fused form
  cross     inference of a multi-head attention layer over padded batches (encoder self attention, cross attention,
            decoder self attention under a per-sequence mask)
  decode    one decode step of an attention layer over its key / value cache: projection of one token per sequence,
            rotation, append, attention over the cached positions, output projection
  generate  the llama2 engine: a prompt pass and greedy decoding, ids in and ids out
"""
import ctypes
import math
import os
import random  # noqa: F401  (draw takes a random.Random)
import tempfile

import numpy as np
import torch

from mycaffe_amd import checkpoint
from mycaffe_amd.cudadnn import CudaDnn, CudaDnnDouble
from mycaffe_amd.layers import (ActivationLayer, Blob, CausalSelfAttentionLayer, InnerProductLayer, MultiheadAttentionLayer,
                                SoftmaxLayer, TransformerBlockLayer)
from mycaffe_amd.llm_inference import LlmInference

# model shapes of the benchmark and the tests
LLAMA_110M = dict(dim=768, hidden_dim=2048, n_layers=12, n_heads=12, n_kv_heads=12, vocab_size=32000, seq_len=1024)
LLAMA_15M = dict(dim=288, hidden_dim=768, n_layers=6, n_heads=6, n_kv_heads=6, vocab_size=32000, seq_len=256)
LLAMA_GQA = dict(dim=256, hidden_dim=512, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=512, seq_len=512)
MODELS = {"110m": LLAMA_110M, "15m": LLAMA_15M, "gqa": LLAMA_GQA}


def listed():
    return [
        # the smallest block there is (the golden fixtures' shape): nothing but calls, as in a unit test or a toy model
        dict(name="block_f32_tiny", kind="block", base="float", style="gpt", act="relu", sdpa=False, B=1, T=4, C=3, H=3, hidden=12),
        # GPT-2 small's block at its training shape, the layer's default attention (explicit chain)
        dict(name="block_f32_gpt", kind="block", base="float", style="gpt", act="relu", sdpa=False, B=8, T=1024, C=768, H=12, hidden=3072),
        # the same block through the attention handle, GELU, sequences that are no power of two
        dict(name="block_f32_gpt_fused", kind="block", base="float", style="gpt", act="gelu_bert", sdpa=True, B=4, T=700, C=768, H=12, hidden=3072),
        # a block of a 15M-parameter Llama: narrow, heads of 48
        dict(name="block_f32_llama", kind="block", base="float", style="llama", act="silu", sdpa=False, B=4, T=256, C=288, H=6, hidden=768),
        # the double base type, as gradient checks and precision studies use it
        dict(name="block_f64_gpt", kind="block", base="double", style="gpt", act="relu", sdpa=False, B=2, T=128, C=256, H=4, hidden=1024),
        # logits and softmax of a batch of positions over a 32000-word vocabulary
        dict(name="head_f32", kind="head", rows=1000, C=768, V=32000),
        # GPT-2 small's MLP, 16-bit storage
        dict(name="mlp_bf16", kind="mlp", rows=8000, C=768, hidden=3072, act="gelu_bert"),
        # prefill of GPT-2 small's attention layer, 16-bit storage
        dict(name="attn_bf16", kind="attn", half=True, rope=False, B=8, T=1024, C=768, H=12),
        # cross attention of an encoder-decoder over padded batches
        dict(name="cross_bf16", kind="cross", half=True, mask="key", B=32, Tq=128, Tk=256, C=512, H=8),
        # a decode step of a 7B-wide attention layer, eight sequences of 2048 cached positions
        dict(name="decode_bf16", kind="decode", half=True, B=8, L=2048, H=32, hs=128),
        # one user generating from the 110M model; a batch of sixteen from 16-bit weights
        dict(name="generate_f32_b1", kind="generate", model="110m", half=False, kv_half=False, B=1, prompt=128, new=64),
        dict(name="generate_bf16_b16", kind="generate", model="110m", half=True, kv_half=False, B=16, prompt=128, new=32),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "head", "mlp", "attn", "cross", "decode", "generate"])
    if kind == "block":
        style = rng.choice(["gpt", "gpt", "llama"])
        base = rng.choice(["float", "float", "double"])
        hs = rng.choice([16, 32, 48, 64, 64])
        H = rng.randint(1, 12 if base == "float" else 6)
        T = _log(rng, 8, 1024 if base == "float" else 192)
        B = _log(rng, 1, max(1, min(16, (8192 if base == "float" else 512) // T)))
        C = H * hs
        hidden = 4 * C if style == "gpt" else 64 * ((8 * C // 3 + 63) // 64)
        return dict(kind=kind, base=base, style=style, act="silu" if style == "llama" else rng.choice(["relu", "gelu", "gelu_bert"]),
                    sdpa=rng.random() < 0.5, B=B, T=T, C=C, H=H, hidden=hidden)
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 16, 2048), C=rng.choice([288, 512, 768]), V=_log(rng, 1000, 32000))
    if kind == "mlp":
        C = rng.choice([256, 288, 384, 512, 768, 1024])
        return dict(kind=kind, rows=_log(rng, 32, 8192), C=C, hidden=4 * C, act=rng.choice(["relu", "gelu_bert", "silu"]))
    if kind == "attn":
        hs = rng.choice([48, 64, 64, 128])
        H = rng.randint(2, 16)
        T = _log(rng, 16, 2048)
        return dict(kind=kind, half=rng.random() < 0.7, rope=rng.random() < 0.5, B=_log(rng, 1, max(1, min(32, 8192 // T))), T=T, C=H * hs, H=H)
    if kind == "cross":
        mask = rng.choice(["key", "key", "batch"])
        Tk = _log(rng, 16, 512)
        Tq = Tk if mask == "batch" else _log(rng, 16, 512)
        H = rng.choice([4, 8, 8, 12])
        return dict(kind=kind, half=rng.random() < 0.7, mask=mask, B=_log(rng, 2, 32), Tq=Tq, Tk=Tk, C=64 * H, H=H)
    if kind == "decode":
        H, hs = rng.choice([(12, 64), (16, 64), (16, 128), (32, 128)])
        return dict(kind=kind, half=rng.random() < 0.7, B=_log(rng, 1, 32), L=_log(rng, 64, 4096), H=H, hs=hs)
    model = rng.choice(["110m", "15m", "15m", "gqa"])
    half = rng.random() < 0.5
    return dict(kind="generate", model=model, half=half, kv_half=half and rng.random() < 0.5, B=_log(rng, 1, 16), prompt=_log(rng, 4, 128),
                new=_log(rng, 8, 48))


# ---- what a program keeps: one device context per base type, its layers, their blobs -----------------------------------
_contexts = {}


def _cuda(base="float"):
    if base not in _contexts:
        _contexts[base] = CudaDnnDouble(0) if base == "double" else CudaDnn(0)
    return _contexts[base]


class _Owner:
    """Frees what a state holds once neither the state nor a view of its memory is left."""

    def __init__(self, cuda, *things):
        self.cuda, self.things = cuda, list(things)

    def _free(self, o, seen):
        if id(o) in seen or o is self.cuda:
            return
        seen.add(id(o))
        if isinstance(o, Blob):
            o.Dispose()
        elif isinstance(o, LlmInference):
            o.CleanUp()
        elif isinstance(o, int):
            self.cuda.FreeMemory(o)
        elif callable(o):
            o()
        elif isinstance(o, (list, tuple)):
            for v in o:
                self._free(v, seen)
        elif type(o).__module__ == Blob.__module__:
            d = vars(o)
            for name, free in (("hAttn", self.cuda.FreeAttn), ("hRope", self.cuda.FreeRope), ("hLayerNorm", self.cuda.FreeLayerNorm)):
                if d.get(name):
                    free(d[name])
            for h in d.get("_handles", ()):
                self.cuda.FreeMemory(h)
            for v in d.values():
                for w in v.values() if isinstance(v, dict) else v if isinstance(v, list) else [v]:
                    if type(w).__module__ == Blob.__module__:
                        self._free(w, seen)

    def __del__(self):
        seen = set()
        for t in self.things:
            try:
                self._free(t, seen)
            except Exception:
                pass


class _Memory:
    """Device memory behind a handle, for torch (no copy); keeps its owner alive."""

    def __init__(self, owner, handle, shape, half=False):
        cuda = owner.cuda
        name = "Internal_GetPointerDouble" if cuda.DTYPE is np.float64 else "Internal_GetPointerFloat"
        get = getattr(cuda._lib, name)
        get.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_void_p)]
        p = ctypes.c_void_p()
        if get(0, cuda.m_hKernel, int(handle), ctypes.byref(p)) != 0 or not p.value:
            raise RuntimeError("no address behind memory handle %d" % handle)
        self.owner = owner
        kind = "<i2" if half else "<f8" if cuda.DTYPE is np.float64 else "<f4"
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (p.value, False), "version": 2}


def _view(owner, handle, shape, half=False):
    t = torch.as_tensor(_Memory(owner, handle, shape, half), device="cuda")
    return t.view(torch.bfloat16) if half else t


def _normal(rng, shape, std=1.0):
    return rng.standard_normal(shape, dtype=np.float32) * np.float32(std)


def _blob(cuda, values, half=False):
    b = Blob(cuda, values.shape, half)
    b.mutable_cpu_data = values
    return b


def _clear(cuda, params):
    """The solver's ClearParamDiffs."""
    for p in params:
        cuda.set(p.count(), p.gpu_diff, 0.0)


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, np.random.default_rng(seed))


def run(state):
    return state["run"](state)


# ---- block -------------------------------------------------------------------------------------------------------------
def _prepare_block(c, rng):
    cuda = _cuda(c["base"])
    B, T, C, hid, llama = c["B"], c["T"], c["C"], c["hidden"], c["style"] == "llama"
    x, top = _blob(cuda, _normal(rng, (B, T, C))), Blob(cuda)
    layer = TransformerBlockLayer(cuda, c["H"], C, T, c["act"], not llama, 1e-5, c["sdpa"], training=True, enable_llama_style_head=llama,
                                  hidden_dim=hid)
    p = dict(attn_weight=_normal(rng, (3 * C, C), 0.3 / math.sqrt(C)), attn_proj_weight=_normal(rng, (C, C), 0.3 / math.sqrt(C)),
             fc_weight=_normal(rng, (hid, C), 0.5 / math.sqrt(C)), proj_weight=_normal(rng, (C, hid), 0.5 / math.sqrt(hid)))
    if llama:
        p.update(fc2_weight=_normal(rng, (hid, C), 0.5 / math.sqrt(C)), rms1_weight=1 + _normal(rng, (C,), 0.1), rms2_weight=1 + _normal(rng, (C,), 0.1))
    else:
        p.update(attn_bias=_normal(rng, (3 * C,), 0.1), attn_proj_bias=_normal(rng, (C,), 0.1), fc_bias=_normal(rng, (hid,), 0.1),
                 proj_bias=_normal(rng, (C,), 0.1))
    layer.Setup(x, p)
    params = layer.attn1.c_attn.blobs + layer.attn1.c_proj.blobs + layer.fc1.blobs + layer.proj.blobs
    if llama:
        params = params + layer.fc2.blobs + layer.norm1.blobs + layer.norm2.blobs
    top.Reshape(B, T, C)
    top.mutable_cpu_diff = _normal(rng, (B, T, C))
    owner = _Owner(cuda, x, top, layer)
    outs = [_view(owner, top.gpu_data, (B, T, C)), _view(owner, x.gpu_diff, (B, T, C))] + [_view(owner, b.gpu_diff, b.shape_) for b in params]
    return dict(run=_run_block, owner=owner, cuda=cuda, layer=layer, x=x, top=top, params=params, outs=outs)


def _run_block(s):
    _clear(s["cuda"], s["params"])
    s["layer"].Forward(s["x"], s["top"])
    s["layer"].Backward(s["top"], s["x"])
    return s["outs"]


# ---- head --------------------------------------------------------------------------------------------------------------
def _prepare_head(c, rng):
    cuda = _cuda()
    M, C, V = c["rows"], c["C"], c["V"]
    x, logits, prob = _blob(cuda, _normal(rng, (1, M, C))), Blob(cuda), Blob(cuda)
    ip, softmax = InnerProductLayer(cuda, V, False), SoftmaxLayer(cuda, -1)
    ip.Setup(x, _normal(rng, (V, C), 1.0 / math.sqrt(C)))
    prob.Reshape(1, M, V)
    prob.mutable_cpu_diff = _normal(rng, (1, M, V))
    owner = _Owner(cuda, x, logits, prob, ip, softmax)
    outs = [_view(owner, prob.gpu_data, (M, V)), _view(owner, x.gpu_diff, (M, C)), _view(owner, ip.blobs[0].gpu_diff, (V, C))]
    return dict(run=_run_head, owner=owner, cuda=cuda, x=x, logits=logits, prob=prob, ip=ip, softmax=softmax, outs=outs)


def _run_head(s):
    _clear(s["cuda"], s["ip"].blobs)
    s["ip"].Forward(s["x"], s["logits"])
    s["softmax"].Forward(s["logits"], s["prob"])
    s["softmax"].Backward(s["prob"], s["logits"])
    s["ip"].Backward(s["logits"], s["x"])
    return s["outs"]


# ---- mlp ---------------------------------------------------------------------------------------------------------------
def _prepare_mlp(c, rng):
    cuda = _cuda()
    M, C, hid = c["rows"], c["C"], c["hidden"]
    x, h, a, y = _blob(cuda, _normal(rng, (1, M, C)), True), Blob(cuda, half=True), Blob(cuda, half=True), Blob(cuda, half=True)
    fc, act, proj = InnerProductLayer(cuda, hid, True, 2, True), ActivationLayer(cuda, c["act"]), InnerProductLayer(cuda, C, True, 2, True)
    fc.Setup(x, _normal(rng, (hid, C), 1.0 / math.sqrt(C)), _normal(rng, (hid,), 0.1))
    a.Reshape(1, M, hid)
    proj.Setup(a, _normal(rng, (C, hid), 1.0 / math.sqrt(hid)), _normal(rng, (C,), 0.1))
    y.Reshape(1, M, C)
    y.mutable_cpu_diff = _normal(rng, (1, M, C))
    owner = _Owner(cuda, x, h, a, y, fc, act, proj)
    params = fc.blobs + proj.blobs
    outs = [_view(owner, y.gpu_data, (M, C), True), _view(owner, x.gpu_diff, (M, C), True)] + [_view(owner, b.gpu_diff, b.shape_, True) for b in params]
    return dict(run=_run_mlp, owner=owner, cuda=cuda, x=x, h=h, a=a, y=y, fc=fc, act=act, proj=proj, params=params, outs=outs)


def _run_mlp(s):
    _clear(s["cuda"], s["params"])
    s["fc"].Forward(s["x"], s["h"])
    s["act"].Forward(s["h"], s["a"])
    s["proj"].Forward(s["a"], s["y"])
    s["proj"].Backward(s["y"], s["a"])
    s["act"].Backward(s["a"], s["h"])
    s["fc"].Backward(s["h"], s["x"])
    return s["outs"]


# ---- attn --------------------------------------------------------------------------------------------------------------
def _prepare_attn(c, rng):
    cuda = _cuda()
    B, T, C, half = c["B"], c["T"], c["C"], c["half"]
    x, top = _blob(cuda, _normal(rng, (B, T, C)), half), Blob(cuda, half=half)
    layer = CausalSelfAttentionLayer(cuda, c["H"], C, T, True, True, c["rope"], half=half, fused_qkv_heads=True)
    layer.Setup(x, _normal(rng, (3 * C, C), 1.0 / math.sqrt(C)), _normal(rng, (3 * C,), 0.1), _normal(rng, (C, C), 1.0 / math.sqrt(C)),
                _normal(rng, (C,), 0.1))
    top.Reshape(B, T, C)
    owner = _Owner(cuda, x, top, layer)
    return dict(run=_run_attn, owner=owner, layer=layer, x=x, top=top, outs=_view(owner, top.gpu_data, (B, T, C), half))


def _run_attn(s):
    s["layer"].Forward(s["x"], s["top"])
    return s["outs"]


# ---- cross -------------------------------------------------------------------------------------------------------------
def _prepare_cross(c, rng):
    cuda = _cuda()
    B, Tq, Tk, C, half = c["B"], c["Tq"], c["Tk"], c["C"], c["half"]
    layer = MultiheadAttentionLayer(cuda, c["H"], C, max(Tq, Tk), True, True, half=half, fuse_batch_qk_mask=True)
    q = _blob(cuda, _normal(rng, (B, Tq, C)), half)
    k = q if c["mask"] == "batch" else _blob(cuda, _normal(rng, (B, Tk, C)), half)
    valid = rng.integers(max(1, Tk // 8), Tk + 1, B)
    mask = (np.arange(Tk)[None, :] < valid[:, None]).astype(np.float32)
    if c["mask"] == "batch":
        mask = (mask[:, None, :] * np.tril(np.ones((Tq, Tk), np.float32))[None]).astype(np.float32)
    w = {}
    for n in "qkvo":
        w["w" + n], w["b" + n] = _normal(rng, (C, C), 1.0 / math.sqrt(C)), _normal(rng, (C,), 0.1)
    layer.Setup(q, k, k, w)
    m, top = _blob(cuda, mask), Blob(cuda, half=half)
    top.Reshape(B, Tq, C)
    owner = _Owner(cuda, q, k, m, top, layer)
    return dict(run=_run_cross, owner=owner, layer=layer, q=q, k=k, m=m, top=top, outs=_view(owner, top.gpu_data, (B, Tq, C), half))


def _run_cross(s):
    s["layer"].Forward(s["q"], s["k"], s["k"], s["m"], s["top"])
    return s["outs"]


# ---- decode ------------------------------------------------------------------------------------------------------------
def _prepare_decode(c, rng):
    cuda = _cuda()
    B, L, H, hs, half = c["B"], c["L"], c["H"], c["hs"], c["half"]
    C, n = H * hs, B * H * L * hs
    put = lambda a: cuda.AllocMemory(a, bHalfSize=half)  # noqa: E731
    h = dict(x=put(_normal(rng, B * C)), w=put(_normal(rng, 3 * C * C, 1.0 / math.sqrt(C))), b=put(_normal(rng, 3 * C, 0.1)),
             wo=put(_normal(rng, C * C, 1.0 / math.sqrt(C))), bo=put(_normal(rng, C, 0.1)))
    for name in ("q", "kn", "vn", "y", "out"):
        h[name] = cuda.AllocMemory(B * C, bHalfSize=half)
    for name in ("kc", "vc"):
        # earlier positions: a block of random values, repeated
        block = _normal(rng, min(n, (1 << 20) + 8))
        src, h[name] = put(block), cuda.AllocMemory(n, bHalfSize=half)
        cuda.copy(block.size, src, h[name])
        have = block.size
        while have < n:
            more = min(have, n - have)
            cuda.copy(more, h[name], h[name], 0, have)
            have += more
        cuda.FreeMemory(src)
    h["rope"] = cuda.CreateRope(0, 0, B * C, B, L, H, hs, 10000.0)
    rope = h["rope"]
    owner = _Owner(cuda, *[v for k, v in h.items() if k != "rope"], lambda: cuda.FreeRope(rope))
    outs = [_view(owner, h["out"], (B, C), half)] + [_view(owner, h[k], (B, H, L, hs), half) for k in ("kc", "vc")]
    return dict(run=_run_decode, owner=owner, cuda=cuda, case=c, h=h, outs=outs)


def _run_decode(s):
    cuda, h, c = s["cuda"], s["h"], s["case"]
    B, L, H, hs = c["B"], c["L"], c["H"], c["hs"]
    cuda.QkvProjHeads(B, 1, H, hs, h["x"], h["w"], h["b"], h["q"], h["kn"], h["vn"])
    cuda.AttnDecodeForward(B, H, H, hs, L, h["q"], h["kc"], h["vc"], h["y"], H * L * hs, L * hs, hs, 0.0, h["rope"], h["kn"], h["vn"])
    cuda.LinearForward(B, H * hs, H * hs, h["y"], h["wo"], h["bo"], h["out"])
    return s["outs"]


# ---- generate ----------------------------------------------------------------------------------------------------------
def _checkpoint(model):
    """A model file of that shape with random weights, written once."""
    cfg = MODELS[model]
    path = os.path.join(tempfile.gettempdir(), "mycaffe_amd_cases_%d_%s.bin" % (os.getuid(), model))
    if not os.path.exists(path):
        gen = torch.Generator(device="cuda").manual_seed(7)
        std = 0.08 if model == "gqa" else 0.02
        parts = []
        for name, shape in checkpoint.tensor_shapes(cfg, False):
            t = torch.ones(shape, device="cuda") if name.startswith("rms") else torch.randn(shape, generator=gen, device="cuda") * std
            parts.append(t.reshape(-1).cpu().numpy())
        part = "%s.%d" % (path, os.getpid())
        checkpoint.write_v1(part, cfg, np.concatenate(parts), False)
        os.replace(part, path)
    return path


def _prepare_generate(c, rng):
    cuda = _cuda()
    inf = LlmInference(cuda)
    inf.Initialize(fTemperature=0.0)
    inf.SetOption(1, 1 if c["half"] else 0)       # weights kept in 16 bits
    inf.SetOption(8, 1 if c["kv_half"] else 0)    # caches kept in 16 bits
    inf.Load(_checkpoint(c["model"]))
    prompts = rng.integers(3, MODELS[c["model"]]["vocab_size"], (c["B"], c["prompt"]))
    return dict(run=_run_generate, owner=_Owner(cuda, inf), inf=inf, prompts=prompts, total=c["prompt"] + c["new"])


def _run_generate(s):
    p = s["prompts"]
    return s["inf"].GenerateIds(p[0], s["total"]) if len(p) == 1 else s["inf"].GenerateBatch(p, s["total"])


# ---- what a pass cannot do without -------------------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind == "block":
        es = 8 if c["base"] == "double" else 4
        M, C, hid = c["B"] * c["T"], c["C"], c["hidden"]
        weights = 4 * C * C + (3 if c["style"] == "llama" else 2) * C * hid
        attention = 2 * c["B"] * c["T"] * (c["T"] + 1) * C             # two products, the causal half
        # backward: twice the products; x, its gradient, top and its gradient; every weight read, every gradient written
        return dict(flops=3.0 * (2 * M * weights + attention), bytes=float(es * (4 * M * C + 2 * weights)))
    if kind == "head":
        M, C, V = c["rows"], c["C"], c["V"]
        return dict(flops=6.0 * M * C * V, bytes=4.0 * (2 * M * C + 2 * V * C + 2 * M * V))
    if kind == "mlp":
        M, C, hid = c["rows"], c["C"], c["hidden"]
        return dict(flops=12.0 * M * C * hid, bytes=2.0 * (4 * M * C + 4 * C * hid))
    es = 2 if c.get("half") else 4
    if kind == "attn":
        M, C = c["B"] * c["T"], c["C"]
        return dict(flops=8.0 * M * C * C + 2.0 * c["B"] * c["T"] * (c["T"] + 1) * C, bytes=float(es * (2 * M * C + 4 * C * C)))
    if kind == "cross":
        Mq, Mk, C = c["B"] * c["Tq"], c["B"] * c["Tk"], c["C"]
        return dict(flops=4.0 * C * C * (Mq + Mk) + 4.0 * c["B"] * c["Tq"] * c["Tk"] * C,
                    bytes=float(es * (2 * Mq * C + (Mk * C if c["mask"] == "key" else 0) + 4 * C * C)))
    if kind == "decode":
        C = c["H"] * c["hs"]
        return dict(flops=8.0 * c["B"] * C * C + 4.0 * c["B"] * c["L"] * C, bytes=float(es * (4 * C * C + 2 * c["B"] * c["L"] * C + 2 * c["B"] * C)))
    m = MODELS[c["model"]]
    kvd = m["dim"] // m["n_heads"] * m["n_kv_heads"]
    per_layer = (m["dim"] + 2 * kvd) * m["dim"] + m["dim"] * m["dim"] + 3 * m["hidden_dim"] * m["dim"]
    matrices = m["n_layers"] * per_layer + m["vocab_size"] * m["dim"]
    # every step reads all weights once and each sequence's cache; the prompt pass reads the weights once more
    positions = sum(range(c["prompt"] + 1, c["prompt"] + c["new"] + 1))
    cache = 2.0 * c["B"] * m["n_layers"] * kvd * positions * (2 if c["kv_half"] else 4)
    return dict(flops=2.0 * matrices * c["B"] * (c["prompt"] + c["new"]), bytes=float((c["new"] + 1) * matrices * es + cache))


def tolerance(case):
    if case["kind"] == "generate":
        # ids; where two logits are equal to the last bits, one sequence may go on from the other of the two
        return {"rel": 0.0, "differ": 0.01}
    if case["kind"] == "block" and case["base"] == "double":
        return {"rel": 1e-12}
    if case["kind"] == "mlp" or case.get("half"):
        return {"rel": 1e-2}
    return {"rel": 1e-5}
