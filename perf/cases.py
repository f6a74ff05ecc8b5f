"""The calls whose time on the GPU matters to a program that decodes or
prefills a mixture-of-experts model with llmpager_amd.

Six kinds of pass, each through the public entry points:

  moe     MoeLayer.forward of every layer of a group of layers, each with its
          own weights, tokens and residual (what a model runs per decode step
          or prefill chunk; the attention blocks between them left out), eager
          or replayed as one captured graph
  mla     Kernels.mla_attn_decode_batch over the latent caches of several
          layers: sequences of different lengths in caches of one capacity
  attn    the attention block of several layers: rmsnorm_gemv (q, k, v), then
          attn_block (norms, rope, cache append, attention, output projection)
  step    DecodeStep.run: one token through a whole (shortened) model with
          its lm_head, to logits
  launch  the same decode layer by the launchers that each stand for one
          kernels.rs call, the experts through q4g64_gemv_batch
  paged   one token after the other through layers whose experts do not all
          fit their VRAM slots: route, read the picks back, request them from
          the pager, resolve, run the experts, release

Shapes are those of the repository's bench and tests: Qwen3-30B-A3B (hidden
2048, 128 experts of 768, top 8), Qwen3-235B-A22B (hidden 4096, experts of
1536) and DeepSeek-V2-Lite (hidden 2048, 64 experts of 1408, top 6, a shared
MLP of 2816; MLA with a 512 + 64 latent).  Layers are stacked so that a pass
reads more than the 256 MB memory-side cache holds, as a whole model does."""
from __future__ import annotations

import math

import torch

import llmpager_amd as lp
from llmpager_amd.step import AttnWeights, DecodeStep, StepShape

DEV = "cuda"

# hidden, inter, experts, top_k, group, gating, shared
QWEN30 = dict(hidden=2048, inter=768, experts=128, top_k=8, group=32, gating="softmax", shared=0)
QWEN235 = dict(hidden=4096, inter=1536, experts=128, top_k=8, group=32, gating="softmax", shared=0)
LITE = dict(hidden=2048, inter=1408, experts=64, top_k=6, group=32, gating="sigmoid", shared=2816)


def _moe(shape, tokens, layers, graph=False):
    return dict(kind="moe", tokens=tokens, layers=layers, graph=graph, **shape)


def listed():
    return [
        # one token: the latency of routing, expert and combine launches
        dict(name="moe_b1_graph", **_moe(QWEN30, 1, 12, True)),
        # small and full lockstep decode batches, launched eagerly
        dict(name="moe_b8", **_moe(QWEN30, 8, 6)),
        dict(name="moe_b32", **_moe(QWEN30, 32, 4)),
        # a short prompt or the tail of a chunk: more tokens than a decode
        # batch, few per expert
        dict(name="moe_t203", **_moe(QWEN30, 203, 2)),
        # a full prefill chunk
        dict(name="moe_prefill2048", **_moe(QWEN30, 2048, 2)),
        # sigmoid gating with a bias and an always-on shared MLP
        dict(name="moe_shared_b16", **_moe(LITE, 16, 6)),
        # rows twice as wide, an odd batch
        dict(name="moe_wide_b3", **_moe(QWEN235, 3, 3)),
        # MLA decode of a batch with ragged lengths
        dict(name="mla_b16", kind="mla", batch=16, heads=16, qk=576, c=512, capacity=4096, layers=6),
        # one sequence's attention late in a long context
        dict(name="attn_long", kind="attn", hidden=2048, heads=32, kv_heads=4, pos=13001, capacity=16384, layers=6),
        # a token through embedding, attention, experts and lm_head
        dict(name="step", kind="step", hidden=2048, heads=32, kv_heads=4, vocab=151936, capacity=4096, pos=1501,
             inter=768, experts=128, top_k=8, group=32, layers=8),
        # the launch-by-launch layer
        dict(name="launch", kind="launch", hidden=2048, heads=32, kv_heads=4, pos=1501, capacity=4096, f16=True,
             inter=768, experts=32, top_k=8, group=32, layers=4),
        # paging: 64 slots for 128 experts
        dict(name="paged", kind="paged", slots=64, tokens=12, layers=2,
             **{k: v for k, v in QWEN30.items() if k != "shared"}),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe"] * 6 + ["mla", "mla", "attn", "attn", "launch", "step", "paged"])
    if kind == "moe":
        which = rng.randrange(4)
        if which == 3:  # a generic shape: any group, any multiple of 32
            g = rng.choice([32, 32, 64, 128])
            shape = dict(hidden=g * rng.randint(768 // g, 3072 // g), inter=g * max(2, rng.randint(256 // g, 1536 // g)),
                         experts=rng.randint(16, 160), top_k=rng.randint(1, 10), group=g,
                         gating=rng.choice(["softmax", "sigmoid"]), shared=rng.choice([0, 0, g * rng.randint(4, 16)]))
        else:
            shape = (QWEN30, LITE, QWEN235)[which]
        tokens = _log(rng, 1, (2048, 2048, 512, 768)[which])
        layers = 1 if tokens > 256 else rng.randint(1, 4)
        layers = max(1, min(layers, int(1.4e9 / _moe_work(shape, tokens, 1)[0])))
        return _moe(shape, tokens, layers, tokens <= 64 and rng.random() < 0.3)
    if kind == "mla":
        return dict(kind="mla", batch=_log(rng, 1, 32), heads=rng.choice([8, 16, 16, 16]), qk=576, c=512,
                    capacity=_log(rng, 100, 6000), layers=rng.randint(2, 4))
    if kind == "paged":
        return dict(kind="paged", slots=rng.randint(24, 64), tokens=rng.randint(2, 12), layers=1,
                    **{k: v for k, v in QWEN30.items() if k != "shared"})
    heads, kv = rng.choice([(32, 4), (32, 4), (32, 8), (16, 2), (16, 16), (64 // 4, 1)])
    hidden = 128 * rng.randint(8, 32) if rng.random() < 0.5 else 2048
    if kind == "attn":
        cap = _log(rng, 64, 24000)
        return dict(kind="attn", hidden=hidden, heads=heads, kv_heads=kv, pos=rng.randrange(cap), capacity=cap,
                    layers=rng.randint(2, 5))
    cap = _log(rng, 600, 8000)
    more = dict(hidden=hidden, heads=heads, kv_heads=kv, capacity=cap, pos=rng.randrange(cap), inter=32 * rng.randint(8, 32),
                top_k=rng.randint(2, 8), group=32, layers=rng.randint(1, 4))
    if kind == "step":
        return dict(kind="step", vocab=_log(rng, 1000, 150000), experts=rng.randint(32, 128), **more)
    return dict(kind="launch", f16=rng.random() < 0.7, experts=rng.randint(8, 32), **more)


# ---- inputs (plain torch, from the seed alone) -------------------------------


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 1)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        t = torch.randn(shape, generator=self.g, device=DEV)
        return t.mul_(std).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device=DEV).mul_(hi - lo).add_(lo)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device=DEV, dtype=torch.uint8)

    def perm(self, n):
        return torch.randperm(n, generator=self.g, device=DEV)


def _regions(hidden, inter, group):
    """Offsets (scales, nibbles) of a blob's gate, up and down, and its bytes:
    a 32-byte header, then per matrix f16 scales [rows, cols / group] and
    nibbles [rows, cols / 2]."""
    at, out = 32, []
    for rows, cols in ((inter, hidden), (inter, hidden), (hidden, inter)):
        out.append((at, at + rows * (cols // group) * 2, rows, cols))
        at = out[-1][1] + rows * cols // 2
    return out, at


def _blobs(r, n, hidden, inter, group):
    """n expert blobs in slots of whole 4096-byte pages: uniform nibbles and
    scales that keep each projection's output near its input's size."""
    regions, nbytes = _regions(hidden, inter, group)
    arena = r.bytes(n, (nbytes + 4095) // 4096 * 4096)
    for so, no, rows, cols in regions:
        s = r.uniform(n, rows * (cols // group), lo=0.5, hi=1.5).mul_(0.21 / math.sqrt(cols)).to(torch.float16)
        arena[:, so:no] = s.view(torch.uint8)
    return arena


def _matrices(blob, hidden, inter, group):
    """A blob's gate, up and down in float64."""
    out = []
    for so, no, rows, cols in _regions(hidden, inter, group)[0]:
        s = blob[so:no].view(torch.float16).view(rows, cols // group).double()
        b = blob[no:no + rows * cols // 2]
        q = torch.stack((b & 15, b >> 4), dim=1).view(rows, cols // group, group).double() - 8.0
        out.append((q * s[:, :, None]).view(rows, cols))
    return out


def _tokens(r, n, hidden):
    """Normalised hidden states: a part that all tokens share (they are of
    one text), channels of different size."""
    x = 0.6 * r.normal(1, hidden) + 0.8 * r.normal(n, hidden)
    gain = torch.exp(0.4 * r.normal(1, hidden))
    x = x * gain
    return x * torch.rsqrt(x.square().mean(1, keepdim=True))


def _moe_layer(r, c, tokens):
    """One layer's weights, tokens and residual."""
    H, I, E = c["hidden"], c["inter"], c["experts"]
    d = dict(arena=_blobs(r, E, H, I, c["group"]), slots=r.perm(E).to(torch.int32),
             router=r.normal(E, H, std=2.0 / math.sqrt(H), dtype=torch.bfloat16),
             x=_tokens(r, tokens, H), h=r.normal(tokens, H, std=0.5))
    if c["gating"] == "sigmoid":
        d["bias"] = r.normal(E, std=0.05)
    if c.get("shared"):
        d["shared"] = _blobs(r, 1, H, c["shared"], c["group"])[0]
    return d


# Routed scaling of sigmoid layers (the softmax ones renormalise instead).
SCALING = 1.5


def _desc(c, d):
    H, I, g = c["hidden"], c["inter"], c["group"]
    go, uo, do = lp.blob_offsets(H, I, g)
    sig = c["gating"] == "sigmoid"
    desc = lp.LayerDesc(
        hidden=H, inter=I, experts=c["experts"], top_k=min(c["top_k"], c["experts"]), group=g,
        gating=lp.GATING_SIGMOID if sig else lp.GATING_SOFTMAX, renorm=1, routed_scaling=SCALING if sig else 1.0,
        min_weight=0.0, router_w=d["router"].data_ptr(), router_bias=d["bias"].data_ptr() if sig else 0,
        slot_table=d["slots"].data_ptr(), arena_base=d["arena"].data_ptr(), slot_span=d["arena"].shape[1],
        gate_off=go, up_off=uo, down_off=do)
    if c.get("shared"):
        desc.shared_blob, desc.shared_inter, desc.shared_group = d["shared"].data_ptr(), c["shared"], g
        desc.sh_gate_off, desc.sh_up_off, desc.sh_down_off = lp.blob_offsets(H, c["shared"], g)
    return desc


def _moe_exact(c, d, x, blobs=None):
    """The layer's addition to the residual in float64, for x [T, hidden]."""
    H, I, g, k = c["hidden"], c["inter"], c["group"], min(c["top_k"], c["experts"])
    logits = x.double() @ d["router"].double().T
    if c["gating"] == "sigmoid":
        s = torch.sigmoid(logits)
        ids = torch.topk(s + d["bias"].double(), k, dim=1).indices
        w = s.gather(1, ids)
        w = w / w.sum(1, keepdim=True) * SCALING
    else:
        w, ids = torch.topk(torch.softmax(logits, 1), k, dim=1)
        w = w / w.sum(1, keepdim=True)
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)

    def ffn(rows, blob, inter):
        gate, up, down = _matrices(blob, H, inter, g)
        a, u = rows @ gate.T, rows @ up.T
        return (a * torch.sigmoid(a) * u) @ down.T

    xd = x.double()
    for e in torch.unique(ids).tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        blob = blobs[e] if blobs is not None else d["arena"][int(d["slots"][e])]
        out.index_add_(0, t, ffn(xd[t], blob, I) * w[t, j][:, None])
    if c.get("shared"):
        out += ffn(xd, d["shared"], c["shared"])
    return out


# ---- the program's handles ----------------------------------------------------

_handles = {}


def _cuda():
    """This process's context and the stream that its calls go to."""
    if not _handles:
        torch.cuda.init()
        _handles["cuda"] = lp.Cuda(0)
        _handles["stream"] = _handles["cuda"].stream()
        _handles["K"] = lp.Kernels(_handles["cuda"])
    return _handles["cuda"], _handles["stream"], _handles["K"]


class _Step:
    """A DecodeStep that frees its buffers once nothing uses them any more."""

    def __init__(self, *args):
        self.step = DecodeStep(*args)

    def __del__(self):
        if hasattr(self, "step"):
            torch.cuda.synchronize()
            self.step.free()


class _DevArray:
    """A device buffer of `owner` as torch.as_tensor takes it."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(int(ptr), False), version=3)


def _workspace(descs, T):
    n = max(lp.ws_layout(d, T).total for d in descs)
    return torch.zeros(n + 256, dtype=torch.uint8, device=DEV), n


def _aligned(t):
    return (t.data_ptr() + 255) // 256 * 256


class _MoeState:
    def __init__(self, c, seed):
        cuda, s, _ = _cuda()
        r = _Rand(seed)
        T = c["tokens"]
        self.data = [_moe_layer(r, c, T) for _ in range(c["layers"])]
        self.x = torch.stack([d.pop("x") for d in self.data])
        self.h = torch.stack([d.pop("h") for d in self.data])
        descs = [_desc(c, d) for d in self.data]
        self.ws, self.ws_bytes = _workspace(descs, T)
        wsp, step = _aligned(self.ws), T * c["hidden"] * 4
        self.calls = [(lp.MoeLayer(cuda, d), self.x.data_ptr() + i * step, self.h.data_ptr() + i * step, T, wsp)
                      for i, d in enumerate(descs)]
        self.stream, self.graph = s, None
        if c["graph"]:
            torch.cuda.synchronize()
            cuda.capture_begin(s)
            self.launch()
            self.graph = cuda.capture_end(s)

    def launch(self):
        for layer, x, h, T, ws in self.calls:
            layer.forward(x, h, T, ws, self.stream, ws_bytes=self.ws_bytes)

    def run(self):
        if self.graph is not None:
            self.graph.launch(self.stream)
        else:
            self.launch()
        return {"h": self.h}

    def __del__(self):
        if getattr(self, "graph", None) is not None:
            self.graph.close()


def _mla_inputs(c, seed):
    r = _Rand(seed)
    B, H, qk, cap, L = c["batch"], c["heads"], c["qk"], c["capacity"], c["layers"]
    q = [r.normal(B, H, qk, std=1.0) for _ in range(L)]
    cache = [r.normal(B, cap, qk, std=1.0, dtype=torch.bfloat16) for _ in range(L)]
    lens = r.uniform(B, lo=0.25, hi=1.0).mul_(cap).to(torch.int32).clamp_(1, cap)
    return q, cache, lens


class _MlaState:
    def __init__(self, c, seed):
        _, self.stream, self.K = _cuda()
        self.c = c
        self.q, self.cache, self.lens = _mla_inputs(c, seed)
        B, H = c["batch"], c["heads"]
        self.out = torch.zeros(c["layers"], B, H, c["c"], device=DEV)
        self.ws = torch.zeros(self.K.mla_batch_ws_bytes(B, c["c"], c["capacity"]) + 256, dtype=torch.uint8, device=DEV)
        self.scale = 1.0 / math.sqrt(192.0)

    def run(self):
        c = self.c
        for l in range(c["layers"]):
            self.K.mla_attn_decode_batch(self.q[l].data_ptr(), self.cache[l].data_ptr(), c["capacity"] * c["qk"] * 2,
                                         self.lens.data_ptr(), self.out[l].data_ptr(), _aligned(self.ws), c["batch"],
                                         c["heads"], c["qk"], c["c"], c["capacity"], self.scale, self.stream)
        return {"ctx": self.out}


EPS, THETA = 1e-6, 1e6


def _attn_layer(r, c, f16=True):
    """One attention block: bf16 matrices, norms, and caches with the rows
    before pos filled (later rows too: they must not be read)."""
    H, qd, kd = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128
    bf = torch.bfloat16
    return dict(q=r.normal(qd, H, std=1 / math.sqrt(H), dtype=bf), k=r.normal(kd, H, std=1 / math.sqrt(H), dtype=bf),
                v=r.normal(kd, H, std=1 / math.sqrt(H), dtype=bf), o=r.normal(H, qd, std=1 / math.sqrt(qd), dtype=bf),
                input_ln=r.uniform(H, lo=0.5, hi=1.5), q_norm=r.uniform(128, lo=0.8, hi=1.8),
                k_norm=r.uniform(128, lo=0.8, hi=1.8), post_ln=r.uniform(H, lo=0.5, hi=1.5),
                kv=r.normal(2, c["kv_heads"], c["capacity"], 128, dtype=torch.float16 if f16 else torch.float32))


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    i = torch.arange(64, dtype=torch.float64, device=x.device)
    ang = pos * THETA ** (-2.0 * i / 128.0)
    a, b = x[:, :64], x[:, 64:]
    return torch.cat((a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()), 1)


def _attn_exact(c, w, h):
    """(h + W_o attention, rmsnorm of that, caches with the row at pos) in
    float64; the caches' own type rounds the appended row, as in earnest."""
    x = _rms(h, w["input_ln"])
    nh, nk, pos = c["heads"], c["kv_heads"], c["pos"]
    q = _rope(_rms((w["q"].double() @ x).view(nh, 128), w["q_norm"]), pos)
    k = _rope(_rms((w["k"].double() @ x).view(nk, 128), w["k_norm"]), pos)
    kv = w["kv"].clone()
    kv[0, :, pos] = k.to(kv.dtype)
    kv[1, :, pos] = (w["v"].double() @ x).view(nk, 128).to(kv.dtype)
    kk, vv = kv[0, :, :pos + 1].double(), kv[1, :, :pos + 1].double()
    s = torch.einsum("kgd,kpd->kgp", q.view(nk, nh // nk, 128), kk) / math.sqrt(128.0)
    a = torch.einsum("kgp,kpd->kgd", torch.softmax(s, -1), vv).reshape(-1)
    h = h + w["o"].double() @ a
    return h, _rms(h, w["post_ln"]), kv


def _attn_inputs(c, seed):
    r = _Rand(seed)
    return [(_attn_layer(r, c), r.normal(c["hidden"])) for _ in range(c["layers"])]


class _AttnState:
    def __init__(self, c, seed):
        _, self.stream, self.K = _cuda()
        self.c = c
        inputs = _attn_inputs(c, seed)
        self.w = [w for w, _ in inputs]
        self.h = torch.stack([h for _, h in inputs])
        self.hn = torch.zeros_like(self.h)
        qd, kd = c["heads"] * 128, c["kv_heads"] * 128
        self.q, self.k, self.v = (torch.zeros(n, device=DEV) for n in (qd, kd, kd))
        self.att = torch.zeros(qd, device=DEV)
        self.scratch = torch.zeros(c["heads"] * c["capacity"], device=DEV)

    def run(self):
        c, K, s = self.c, self.K, self.stream
        H, qd, kd = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128
        q, k, v = self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr()
        for l, w in enumerate(self.w):
            h = self.h[l].data_ptr()
            K.rmsnorm_gemv(h, w["input_ln"].data_ptr(), EPS, H,
                           [(w["q"].data_ptr(), qd, q), (w["k"].data_ptr(), kd, k), (w["v"].data_ptr(), kd, v)], s)
            K.attn_block(q, k, v, w["q_norm"].data_ptr(), w["k_norm"].data_ptr(), EPS, THETA, w["kv"][0].data_ptr(),
                         w["kv"][1].data_ptr(), self.att.data_ptr(), self.scratch.data_ptr(), c["heads"],
                         c["kv_heads"], 128, c["pos"], c["capacity"], 1.0 / math.sqrt(128.0), w["o"].data_ptr(), h,
                         w["post_ln"].data_ptr(), self.hn[l].data_ptr(), H, s)
        return {"h": self.h, "hn": self.hn, "kv": [w["kv"] for w in self.w]}


def _step_inputs(c, seed):
    """The model: routers with spread logits (a trained router's are), so
    that the last picks of a token weigh little."""
    r = _Rand(seed)
    layers = []
    for _ in range(c["layers"]):
        w = _attn_layer(r, c)
        m = dict(arena=_blobs(r, c["experts"], c["hidden"], c["inter"], c["group"]),
                 slots=r.perm(c["experts"]).to(torch.int32),
                 router=r.normal(c["experts"], c["hidden"], std=4.0 / math.sqrt(c["hidden"]), dtype=torch.bfloat16))
        layers.append((w, m))
    return dict(layers=layers, embed=r.normal(64, c["hidden"], dtype=torch.bfloat16), token=int(seed) % 64,
                final=r.uniform(c["hidden"], lo=0.5, hi=1.5),
                head=r.normal(c["vocab"], c["hidden"], std=1 / math.sqrt(c["hidden"]), dtype=torch.bfloat16))


class _StepState:
    def __init__(self, c, seed):
        cuda, self.stream, _ = _cuda()
        self.c, self.model = c, _step_inputs(c, seed)
        m, cc = self.model, dict(c, gating="softmax")
        descs = [_desc(cc, e) for _, e in m["layers"]]
        self.ws, nws = _workspace(descs, 1)
        shape = StepShape(hidden=c["hidden"], heads=c["heads"], kv_heads=c["kv_heads"], head_dim=128, vocab=c["vocab"],
                          max_seq=c["capacity"], eps=EPS, rope_theta=THETA)
        attn = [AttnWeights(**{k: w[k].data_ptr() for k in ("q", "k", "v", "o", "input_ln", "q_norm", "k_norm",
                                                            "post_ln")}) for w, _ in m["layers"]]
        own = _Step(cuda, shape, attn, [lp.MoeLayer(cuda, d) for d in descs], m["embed"].data_ptr(),
                    m["final"].data_ptr(), m["head"].data_ptr(), _aligned(self.ws), nws)
        self.step = own.step
        kv_shape = (c["kv_heads"], c["capacity"], 128)
        self.kv = []
        for i, (w, _) in enumerate(m["layers"]):
            for j, p in enumerate((self.step.kcache[i], self.step.vcache[i])):
                t = torch.as_tensor(_DevArray(own, p, kv_shape, "<f2"), device=DEV)
                t.copy_(w["kv"][j])
                self.kv.append(t)
            del w["kv"]
        self.logits = torch.as_tensor(_DevArray(own, self.step.logits, (c["vocab"],), "<f4"), device=DEV)
        torch.cuda.synchronize()

    def run(self):
        self.step.run(self.model["token"], self.c["pos"], self.stream)
        return {"logits": self.logits, "kv": self.kv}


def _launch_inputs(c, seed):
    r = _Rand(seed)
    out = []
    for _ in range(c["layers"]):
        w = _attn_layer(r, c, c["f16"])
        w["arena"] = _blobs(r, c["experts"], c["hidden"], c["inter"], c["group"])
        w["picks"] = r.perm(c["experts"])[:min(c["top_k"], c["experts"])]
        w["wts"] = torch.softmax(r.normal(len(w["picks"])), 0)
        w["router"] = r.normal(c["experts"], c["hidden"], std=2 / math.sqrt(c["hidden"]), dtype=torch.bfloat16)
        out.append((w, r.normal(c["hidden"])))
    return out


class _LaunchState:
    """The layer as decode.rs launches it, with the picks in hand (the
    engine ranks the router's logits on the host)."""

    def __init__(self, c, seed):
        _, self.stream, self.K = _cuda()
        self.c = c
        inputs = _launch_inputs(c, seed)
        self.w = [w for w, _ in inputs]
        self.h = torch.stack([h for _, h in inputs])
        H, I, E, L = c["hidden"], c["inter"], c["experts"], c["layers"]
        qd, kd, k = c["heads"] * 128, c["kv_heads"] * 128, len(self.w[0]["picks"])
        self.offs = lp.blob_offsets(H, I, c["group"])
        for w in self.w:
            w["blobs"] = w["arena"].data_ptr() + w["picks"].to(torch.int64) * w["arena"].shape[1]
        self.logits = torch.zeros(L, E, device=DEV)
        self.buf = {n: torch.zeros(m, device=DEV) for n, m in
                    dict(hn=H, q=qd, k=kd, v=kd, att=qd, proj=H, gate=k * I, up=k * I, act=k * I, y=k * H,
                         scratch=c["heads"] * c["capacity"]).items()}

    def run(self):
        c, K, s = self.c, self.K, self.stream
        H, I, E, g, nh, nk = c["hidden"], c["inter"], c["experts"], c["group"], c["heads"], c["kv_heads"]
        qd, kd, pos, cap = nh * 128, nk * 128, c["pos"], c["capacity"]
        go, uo, do = self.offs
        b = {n: t.data_ptr() for n, t in self.buf.items()}
        for l, w in enumerate(self.w):
            h, n, p = self.h[l].data_ptr(), len(w["picks"]), {m: t.data_ptr() for m, t in w.items()}
            kc, vc = w["kv"][0].data_ptr(), w["kv"][1].data_ptr()
            K.rmsnorm(h, p["input_ln"], b["hn"], 1, H, EPS, s)
            K.bf16_gemv(p["q"], b["hn"], b["q"], qd, H, s)
            K.bf16_gemv(p["k"], b["hn"], b["k"], kd, H, s)
            K.bf16_gemv(p["v"], b["hn"], b["v"], kd, H, s)
            K.rmsnorm(b["q"], p["q_norm"], b["q"], nh, 128, EPS, s)
            K.rmsnorm(b["k"], p["k_norm"], b["k"], nk, 128, EPS, s)
            K.rope(b["q"], nh, 128, pos, THETA, s)
            K.rope(b["k"], nk, 128, pos, THETA, s)
            K.kv_append(b["k"], b["v"], kc, vc, nk, 128, pos, cap, c["f16"], s)
            K.attn_decode(b["q"], kc, vc, b["att"], b["scratch"], nh, nk, 128, pos + 1, cap, 1.0 / math.sqrt(128.0),
                          c["f16"], s)
            K.bf16_gemv(p["o"], b["att"], b["proj"], H, qd, s)
            K.add(h, b["proj"], H, s)
            K.rmsnorm(h, p["post_ln"], b["hn"], 1, H, EPS, s)
            K.bf16_gemv(p["router"], b["hn"], self.logits[l].data_ptr(), E, H, s)
            K.q4g64_gemv_batch(p["blobs"], go, b["hn"], 0, b["gate"], I, H, g, n, s)
            K.q4g64_gemv_batch(p["blobs"], uo, b["hn"], 0, b["up"], I, H, g, n, s)
            K.silu_mul(b["gate"], b["up"], b["act"], n * I, s)
            K.q4g64_gemv_batch(p["blobs"], do, b["act"], I, b["y"], H, I, g, n, s)
            K.moe_reduce(b["y"], p["wts"], h, n, H, s)
        return {"h": self.h, "logits": self.logits, "kv": [w["kv"] for w in self.w]}


def _paged_inputs(c, seed):
    r = _Rand(seed)
    out = []
    for _ in range(c["layers"]):
        out.append(_moe_layer(r, c, c["tokens"]))
    return out


class _PagedState:
    def __init__(self, c, seed):
        self.cuda, self.stream, _ = _cuda()
        self.c = c
        self.data = _paged_inputs(c, seed)
        L, E, H, T = c["layers"], c["experts"], c["hidden"], c["tokens"]
        span = self.data[0]["arena"].shape[1]
        self.host = torch.empty(L, E, span, dtype=torch.uint8, pin_memory=True)
        for l, d in enumerate(self.data):
            self.host[l].copy_(d.pop("arena"))
        self.x = torch.stack([d.pop("x") for d in self.data])
        self.h = torch.stack([d.pop("h") for d in self.data])
        self.pager = lp.Pager(self.cuda, lp.PagerConfig(
            layers=L, experts_per_layer=E, slots_per_layer=c["slots"], decay_interval=256,
            blob_bytes=lp.blob_bytes(H, c["inter"], c["group"]), span=0, host_blobs=self.host.data_ptr(),
            host_stride=span, copy_streams=2, global_pool=0, source=lp.PAGER_SRC_PINNED))
        go, uo, do = lp.blob_offsets(H, c["inter"], c["group"])
        descs = [lp.LayerDesc(hidden=H, inter=c["inter"], experts=E, top_k=c["top_k"], group=c["group"],
                              gating=lp.GATING_SOFTMAX, renorm=1, routed_scaling=1.0, min_weight=0.0,
                              router_w=d["router"].data_ptr(), router_bias=0, slot_table=self.pager.slot_table(l),
                              arena_base=self.pager.arena, slot_span=self.pager.span, gate_off=go, up_off=uo,
                              down_off=do) for l, d in enumerate(self.data)]
        self.layers = [lp.MoeLayer(self.cuda, d) for d in descs]
        self.ids = lp.ws_layout(descs[0], 1).ids
        self.ws, self.ws_bytes = _workspace(descs, 1)

    def run(self):
        c, ws, s, n = self.c, _aligned(self.ws), self.stream, self.ws_bytes
        for t in range(c["tokens"]):
            for l, layer in enumerate(self.layers):
                x, h = self.x[l, t].data_ptr(), self.h[l, t].data_ptr()
                layer.route(x, 1, ws, s, ws_bytes=n)
                picks = self.cuda.download(ws + self.ids, (c["top_k"],), "int32", s)
                slots = self.pager.request(l, picks, s)
                layer.resolve(1, ws, s, ws_bytes=n)
                layer.experts(x, h, 1, ws, s, ws_bytes=n)
                self.pager.release_after(slots, s)
            self.pager.tick()
        return {"h": self.h}

    def __del__(self):
        if getattr(self, "pager", None) is not None:
            torch.cuda.synchronize()
            self.pager.close()


_STATES = dict(moe=_MoeState, mla=_MlaState, attn=_AttnState, step=_StepState, launch=_LaunchState, paged=_PagedState)


def prepare(case, seed):
    return _STATES[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without --------------------------------------------


def _expert(c, inter=None):
    return _regions(c["hidden"], inter or c["inter"], c["group"])[1] - 32


def _moe_work(c, T, passes):
    """Experts that T tokens with even picks touch, router, tokens, residual."""
    E, k, H = c["experts"], min(c["top_k"], c["experts"]), c["hidden"]
    touched = E * (1.0 - (1.0 - k / E) ** T)
    n = touched * _expert(c) + 2 * E * H + 3 * 4 * T * H
    f = 2.0 * T * H * (E + 3 * k * c["inter"])
    if c.get("shared"):
        n += _expert(c, c["shared"])
        f += 6.0 * T * H * c["shared"]
    return n * passes, f * passes


def _attn_work(c, item):
    H, qd, kd = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128
    w = H * (2 * qd + 2 * kd)
    n = 2 * w + 2 * (c["pos"] + 1) * kd * item + 4 * 6 * H
    return n, 2.0 * w + 4.0 * (c["pos"] + 1) * qd


def work(case):
    c, kind = case, case["kind"]
    if kind == "moe":
        n, f = _moe_work(c, c["tokens"], c["layers"])
    elif kind == "paged":
        n, f = _moe_work(c, 1, c["layers"] * c["tokens"])
    elif kind == "mla":
        rows = c["batch"] * c["capacity"] * 0.625
        per_row = 2 * c["qk"]
        n = c["layers"] * (rows * per_row + 4 * c["batch"] * c["heads"] * (c["qk"] + c["c"]))
        f = c["layers"] * rows * c["heads"] * 2.0 * (c["qk"] + c["c"])
    else:
        n, f = _attn_work(c, 2 if c.get("f16", True) else 4)
        if kind != "attn":
            m, g = _moe_work(c, 1, 1)
            n, f = n + m, f + g
        n, f = n * c["layers"], f * c["layers"]
        if kind == "step":
            n += 2 * c["vocab"] * c["hidden"] + 4 * c["vocab"]
            f += 2.0 * c["vocab"] * c["hidden"]
    return {"bytes": n, "flops": f}


def tolerance(case):
    """About four times what the outputs are off the float64 ones."""
    kind = case["kind"]
    if kind == "moe" and case["tokens"] * case["top_k"] >= 16 * case["experts"]:
        return {"rel": 1e-3, "max": 2e-2}  # fp16 operands
    if kind in ("moe", "paged"):
        return {"rel": 1.6e-4, "max": 4e-3}  # activations to 16 bits of each 32 columns' largest
    if kind == "mla":
        return {"rel": 2e-5, "max": 4e-4}
    if kind == "attn":
        return {"rel": 1e-5, "max": 4e-3}  # max: a cache value rounded the other way, here and below
    if kind == "launch":
        return {"rel": 6e-5, "max": 4e-3}
    return {"rel": 1e-3, "max": 2e-2}  # step: a pick may differ in the last place, where it weighs little


# ---- the same in float64 -------------------------------------------------------


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "moe":
        r = _Rand(seed)
        data = [_moe_layer(r, c, c["tokens"]) for _ in range(c["layers"])]
        return {"h": torch.stack([d["h"].double() + _moe_exact(c, d, d["x"]) for d in data])}
    if kind == "paged":
        data = _paged_inputs(c, seed)
        return {"h": torch.stack([d["h"].double() + _moe_exact(c, d, d["x"], d["arena"]) for d in data])}
    if kind == "mla":
        q, cache, lens = _mla_inputs(c, seed)
        out = torch.zeros(c["layers"], c["batch"], c["heads"], c["c"], dtype=torch.float64, device=DEV)
        for l in range(c["layers"]):
            for b, n in enumerate(lens.tolist()):
                rows = cache[l][b, :n].double()
                p = torch.softmax(q[l][b].double() @ rows.T / math.sqrt(192.0), 1)
                out[l, b] = p @ rows[:, :c["c"]]
        return {"ctx": out}
    if kind == "attn":
        got = [_attn_exact(c, w, h.double()) for w, h in _attn_inputs(c, seed)]
        return {"h": torch.stack([g[0] for g in got]), "hn": torch.stack([g[1] for g in got]),
                "kv": [g[2].double() for g in got]}
    if kind == "launch":
        hs, lg, kvs = [], [], []
        for w, h in _launch_inputs(c, seed):
            h, x, kv = _attn_exact(c, w, h.double())
            lg.append(w["router"].double() @ x)
            for e, wt in zip(w["picks"].tolist(), w["wts"].double()):
                gate, up, down = _matrices(w["arena"][e], c["hidden"], c["inter"], c["group"])
                a = gate @ x
                h = h + wt * (down @ (a * torch.sigmoid(a) * (up @ x)))
            hs.append(h)
            kvs.append(kv.double())
        return {"h": torch.stack(hs), "logits": torch.stack(lg), "kv": kvs}
    m, cc = _step_inputs(c, seed), dict(c, gating="softmax")
    h = m["embed"][m["token"]].double()
    kvs = []
    for w, e in m["layers"]:
        h, x, kv = _attn_exact(c, w, h)
        h = h + _moe_exact(cc, e, x[None])[0]
        kvs += [kv[0].double(), kv[1].double()]
    return {"logits": m["head"].double() @ _rms(h, m["final"]), "kv": kvs}
