"""The framework's main work as timed cases: what a drafting and verifying server has it do.

Every case is a dict of plain values with a ``kind``:

* ``flow``: ``FusedFlow.predict_hidden`` -- all Euler steps of both chunk experts for ``batch``
  requests (the draft of one request, or of a serving batch);
* ``latent``: the latent drafter's ``predict_hidden``: VAE encode of the context, the flow at the
  latent width, VAE decode of the drafted rows;
* ``depth``: one depth of a draft search: the path residual of every beam, then the shortlisted
  lm_head with the markov bias and the log-softmax top-k;
* ``head``: the batched bf16 head over the marginal hiddens of many requests, with its top-k;
* ``twopass``: the two-pass head: candidates from every depth's marginal hidden, their rows packed,
  one depth rescored over them;
* ``gdn``: one gated-delta-net layer of a tree verify: the tree convolution, then the state update;
* ``verify``: the end of a tree verify: the tree rows' attention merged with the prefix, then the
  greedy acceptance over the target's logits.

``exact`` restates each in float64 with plain torch.
"""
from __future__ import annotations

import math
import sys
import zlib
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "chain-flow_amd"))

from chain_flow_amd.config import TreeVAEFlowConfig, flownet  # noqa: E402
from chain_flow_amd.flow import FusedFlow  # noqa: E402
from chain_flow_amd.gdn import tree_gdn_vllm  # noqa: E402
from chain_flow_amd.head import GemmHead, PathHead, ShortlistHead  # noqa: E402
from chain_flow_amd.tree_verify import tree_attn_merge, tree_conv, tree_greedy_accept  # noqa: E402
from chain_flow_amd.vae import HiddenVAE  # noqa: E402
from chain_flow_amd.weights import param_specs  # noqa: E402

DEV = "cuda"
VOCAB, SHORTLIST, RANK, ORDER, CTX, DRAFT, CHUNK = 248320, 62642, 256, 4, 8, 8, 4


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one request's draft against a large target: the headline draft
        dict(name="flow_d5120_b1", kind="flow", d=5120, batch=1, layers=8, steps=8),
        # one request's draft at the 4B-class width without the latent drafter
        dict(name="flow_d2560_b1", kind="flow", d=2560, batch=1, layers=8, steps=8),
        # a server's batch at that width, an odd number of requests
        dict(name="flow_d2560_b13", kind="flow", d=2560, batch=13, layers=8, steps=8),
        # a full batch against a mid-size target
        dict(name="flow_d4096_b32", kind="flow", d=4096, batch=32, layers=8, steps=8),
        # the shipped latent drafter: one request, and a ragged batch
        dict(name="latent_h2560_b1", kind="latent", hidden=2560, latent=640, inter=1920, batch=1, steps=2),
        dict(name="latent_h2560_b27", kind="latent", hidden=2560, latent=640, inter=1920, batch=27, steps=2),
        # the last depth of one request's width-4 search, and of 32 requests' searches
        dict(name="depth_d5120_m4", kind="depth", d=5120, requests=1, width=4, live=4),
        dict(name="depth_d4096_m128", kind="depth", d=4096, requests=32, width=4, live=4),
        # 32 requests x 5 depths through the batched head
        dict(name="head_bf16_m160", kind="head", d=4096, rows=160, k=8),
        # one request's two-pass search: candidates, then a depth over them
        dict(name="twopass_d5120", kind="twopass", d=5120, depths=5, cands=8192, width=4),
        # a GDN layer over a 41-node draft tree, 16-bit states: the smallest calls of a verify step
        dict(name="gdn_n41", kind="gdn", nodes=41, heads=16, vheads=32, state="bf16"),
        # the tail of a verify step: four requests' trees
        dict(name="verify_s4_n40", kind="verify", seqs=4, nodes=40, heads=16, kvheads=4, dim=256, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "latent", "depth", "depth", "head", "twopass", "gdn", "verify"])
    if kind == "flow":
        d = rng.choice([1024, 2048, 2560, 4096, 5120])
        batch = _log(rng, 1, {1024: 48, 2048: 40, 2560: 32, 4096: 24, 5120: 2}[d])
        return dict(kind="flow", d=d, batch=batch, layers=rng.choice([4, 6, 8]), steps=rng.choice([2, 4, 8]))
    if kind == "latent":
        hidden, latent = rng.choice([(2560, 640), (5120, 1024)])
        return dict(kind="latent", hidden=hidden, latent=latent, inter=1920, batch=_log(rng, 1, 40),
                    steps=rng.choice([1, 2, 4]))
    if kind == "depth":
        return dict(kind="depth", d=rng.choice([1024, 2560, 4096, 5120]), requests=_log(rng, 1, 40),
                    width=rng.randint(1, 6), live=rng.randint(1, 4))
    if kind == "head":
        return dict(kind="head", d=rng.choice([1024, 2560, 4096]), rows=_log(rng, 9, 240), k=rng.randint(1, 8))
    if kind == "twopass":
        return dict(kind="twopass", d=rng.choice([2560, 4096, 5120]), depths=rng.randint(3, 7),
                    cands=_log(rng, 1000, 16000), width=rng.randint(2, 4))
    if kind == "gdn":
        heads = rng.choice([4, 8, 16])
        return dict(kind="gdn", nodes=_log(rng, 2, 64), heads=heads, vheads=heads * rng.choice([1, 2]),
                    state=rng.choice(["bf16", "fp32"]))
    return dict(kind="verify", seqs=rng.randint(1, 8), nodes=rng.randint(3, 60), heads=16, kvheads=rng.choice([2, 4, 8]),
                dim=rng.choice([128, 256]), dtype=rng.choice(["bf16", "fp16"]))


# ---------------------------------------------------------------- inputs
def _gen(name, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed((zlib.crc32(name.encode()) * 2654435761 + seed * 0x9E3779B97F4A7C15) % 2 ** 63)
    return g


def _normal(name, seed, shape, scale=1.0, dtype=torch.float16, mean=0.0):
    x = torch.randn(shape, generator=_gen(name, seed), dtype=torch.float32, device=DEV)
    return (x * scale + mean).to(dtype)


def _ints(name, seed, shape, hi, dtype=torch.int32):
    return torch.randint(0, hi, shape, generator=_gen(name, seed), device=DEV).to(dtype)


def _hidden(name, seed, shape, dtype=torch.float16):
    """Hidden states: normal rows rescaled to a root mean square of 1."""
    x = torch.randn(shape, generator=_gen(name, seed), dtype=torch.float32, device=DEV)
    return (x / x.pow(2).mean(-1, keepdim=True).sqrt()).to(dtype)


def _weights(cfg, hidden, seed, keep):
    """The drafter's parameters whose names ``keep`` accepts: matrices N(0, 1 / fan_in), biases and
    LayerNorm shifts small, LayerNorm gains near 1."""
    out = {}
    for name, (shape, kind, fan_in) in param_specs(cfg, VOCAB, target=False, hidden=hidden).items():
        if not keep(name):
            continue
        scale = {"linear": fan_in ** -0.5, "embedding": 0.5, "embedding_rank": 1.0, "bias": 0.05, "ln_w": 0.1,
                 "ln_b": 0.1}[kind]
        out[name] = _normal(name, seed, shape, scale, mean=1.0 if kind == "ln_w" else 0.0)
    return out


def _cfg(case):
    if case["kind"] == "latent":
        return TreeVAEFlowConfig(context_size=CTX, draft_length=DRAFT, chunk_size=CHUNK, expert_dim=case["hidden"],
                                 num_flow_steps=case["steps"], latent_size=case["latent"],
                                 vae_intermediate_size=case["inter"])
    return flownet(case["d"], layers=case["layers"], flow_steps=case["steps"])


def _is_flow(name):
    return name.startswith(("expert.", "extra_experts."))


def _is_path(name):
    return name.startswith("path_head.")


def _shortlist(seed):
    return torch.randperm(VOCAB, generator=_gen("shortlist", seed), device=DEV)[:SHORTLIST].sort().values.to(torch.int32)


def _head_tensors(d, seed):
    """lm_head with logits of a few units' spread, and the markov tables."""
    return (_normal("lm_head", seed, (VOCAB, d), 3.0 * d ** -0.5), _shortlist(seed),
            _normal("markov.w1", seed, (VOCAB, RANK)), _normal("markov.w2", seed, (VOCAB, RANK), RANK ** -0.5))


def _lastp(case, seed):
    """The last tokens of every beam: `live` of them, the rest absent."""
    rows = case["requests"] * case["width"]
    lastp = _ints("lastp", seed, (rows, ORDER), VOCAB)
    lastp[:, case["live"]:] = -1
    return lastp


def _tree(n, width=4):
    """A beam tree of n nodes in BFS order: `width` roots, then every level under the one before, its
    nodes spread unevenly over it."""
    return [-1 if i < width else (i // width - 1) * width + (i * 7 // 3) % width for i in range(n)]


def _gdn_inputs(case, seed):
    n, h, hv, kd = case["nodes"], case["heads"], case["vheads"], 128
    dim = 2 * h * kd + hv * kd
    bf = torch.bfloat16
    sdt = bf if case["state"] == "bf16" else torch.float32
    return dict(
        x=_normal("x", seed, (n, dim), 1.0, bf), conv=_normal("conv", seed, (n + 2, dim, 4), 1.0, bf),
        w=_normal("w", seed, (dim, 4), 0.5, bf), bias=_normal("bias", seed, (dim,), 0.1, bf),
        a=_normal("a", seed, (n, hv), 1.0, bf), b=_normal("b", seed, (n, hv), 1.0, bf),
        A_log=_normal("A_log", seed, (hv,), 0.5, torch.float32), dt=_normal("dt", seed, (hv,), 0.5, torch.float32),
        ssm=_normal("ssm", seed, (n + 2, hv, kd, kd), 0.1, sdt),
        slots=torch.arange(2, n + 2, dtype=torch.int32, device=DEV),
        parent=torch.tensor(_tree(n), dtype=torch.int32, device=DEV))


def _verify_inputs(case, seed):
    s, n, h, hk, dim = case["seqs"], case["nodes"], case["heads"], case["kvheads"], case["dim"]
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    rows, par = s * n + s, _tree(n)
    anc = torch.zeros(n, n, dtype=torch.bool)
    for i in range(n):
        m = i
        while m >= 0:
            anc[i, m] = True
            m = par[m]
    # the forward's rows: each request's committed token, then its tree nodes
    idx = torch.tensor([[q * (n + 1) + 1 + i for i in range(n)] for q in range(s)], dtype=torch.int32)
    logits = _normal("logits", seed, (rows, VOCAB), 3.0, dt)
    drafts = _ints("drafts", seed, (s, n), VOCAB)
    # along one path of each tree the draft agrees with the target
    best = logits.float().argmax(-1).view(s, n + 1).to(torch.int32)
    i = n - 1
    path = []
    while i >= 0:
        path.append(i)
        i = par[i]
    for i in path:
        drafts[:, i] = best[:, 0 if par[i] < 0 else par[i] + 1]
    return dict(
        q=_normal("q", seed, (rows, h, dim), 1.0, dt), k=_normal("k", seed, (rows, hk, dim), 1.0, dt),
        v=_normal("v", seed, (rows, hk, dim), 1.0, dt), out=_normal("out", seed, (rows, h, dim), 1.0, dt),
        pout=_normal("pout", seed, (s * n, h, dim), 0.3, dt),
        plse=_normal("plse", seed, (h, s * n), 1.0, torch.float32, mean=3.0), idx=idx.to(DEV),
        not_anc=(~anc)[None].repeat(s, 1, 1).to(DEV), logits=logits, drafts=drafts.view(-1),
        parents=torch.tensor(par * s, dtype=torch.int32, device=DEV),
        cu_draft=torch.tensor([n * (q + 1) for q in range(s)], dtype=torch.int32, device=DEV),
        cu_rows=torch.tensor([(n + 1) * (q + 1) for q in range(s)], dtype=torch.int32, device=DEV))


# ---------------------------------------------------------------- one pass
def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "flow":
        cfg = _cfg(case)
        st["flow"] = FusedFlow(cfg, _weights(cfg, None, seed, _is_flow), device=DEV)
        st["ctx"] = _hidden("ctx", seed, (case["batch"], CTX, case["d"]))
    elif kind == "latent":
        cfg = _cfg(case)
        w = _weights(cfg, case["hidden"], seed, lambda n: _is_flow(n) or n.startswith("vae."))
        st["vae"] = HiddenVAE(cfg, case["hidden"], w, device=DEV)
        st["flow"] = FusedFlow(cfg, w, device=DEV)
        st["ctx"] = _hidden("ctx", seed, (case["batch"], CTX, case["hidden"]))
    elif kind == "depth":
        d = case["d"]
        st["path"] = PathHead(_weights(flownet(d, layers=1), None, seed, _is_path), _normal("embed", seed, (VOCAB, d)),
                              ORDER, 2, DEV)
        st["head"] = ShortlistHead(*_head_tensors(d, seed))
        st["pred"] = _hidden("pred", seed, (case["requests"], DRAFT, d))
        st["lastp"] = _lastp(case, seed)
    elif kind == "head":
        st["head"] = GemmHead(_normal("lm_head", seed, (VOCAB, case["d"]), 3.0 * case["d"] ** -0.5, torch.bfloat16),
                              _shortlist(seed), packed=True)
        st["x"] = _hidden("x", seed, (case["rows"], case["d"]), torch.bfloat16)
    elif kind == "twopass":
        st["head"] = ShortlistHead(*_head_tensors(case["d"], seed))
        st["marginals"] = _hidden("marginals", seed, (1, case["depths"], case["d"]))
        st["beams"] = _hidden("beams", seed, (case["width"], case["d"]))
        st["prev"] = _ints("prev", seed, (case["width"],), VOCAB)
        st["image"] = None
    elif kind == "gdn":
        st.update(_gdn_inputs(case, seed))
    else:
        st.update(_verify_inputs(case, seed))
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "flow":
        return st["flow"].predict_hidden(st["ctx"])
    if kind == "latent":
        return st["vae"].decode(st["flow"].predict_hidden(st["vae"].encode(st["ctx"])))
    if kind == "depth":
        rows = st["path"].hidden(st["lastp"], case["live"], st["pred"][:, case["live"]])
        vals, ids, lse = st["head"].topk(rows, case["width"], prev=st["lastp"].view(-1), prev_stride=ORDER)
        return {"hidden": rows, "vals": vals, "ids": ids, "lse": lse}
    if kind == "head":
        vals, ids, lse = st["head"].topk(st["x"], case["k"])
        return {"vals": vals, "ids": ids, "lse": lse}
    if kind == "twopass":
        head = st["head"]
        _, cands = head.candidates(st["marginals"], case["cands"])
        st["image"] = head.pack_rows(cands[0], st["image"])
        vals, ids, lse = head.topk_image(st["beams"], case["width"], st["image"], case["cands"], prev=st["prev"])
        return {"vals": vals, "tokens": cands[0][ids.long()], "lse": lse}
    if kind == "gdn":
        y = tree_conv(st["x"], st["conv"], st["w"], st["bias"], st["slots"], st["parent"])
        o = tree_gdn_vllm(y, st["a"], st["b"], st["A_log"], st["dt"], st["ssm"], st["slots"], st["parent"],
                          num_q_heads=case["heads"])
        return {"conv": y, "conv_state": st["conv"], "out": o, "state": st["ssm"]}
    out = tree_attn_merge(st["q"], st["k"], st["v"], st["out"], st["pout"], st["plse"], st["idx"], st["not_anc"],
                          case["dim"] ** -0.5)
    tokens, path, length = tree_greedy_accept(st["logits"], st["cu_draft"], st["cu_rows"], st["drafts"], st["parents"],
                                              case["nodes"])
    return {"out": out, "tokens": tokens, "path": path, "length": length}


# ---------------------------------------------------------------- what a pass cannot do without
def _flow_work(d, layers, steps, batch):
    """Block matrices once per Euler step for the whole batch (QKV 3, O 1, FFN 12 d^2, output 1 / layers);
    the cross attention's four d^2 matrices once per draft; the rows' multiply-adds."""
    nch = DRAFT // CHUNK
    step = nch * (16 * layers + 1) * d * d
    once = nch * layers * 4 * d * d
    rows = sum((c + 1) * CHUNK for c in range(nch)) * batch
    flops = 2.0 * (steps * layers * 16 * d * d * rows + steps * nch * CHUNK * batch * d * d
                   + nch * layers * 4 * d * d * CTX * batch)
    return 2.0 * (steps * step + once) + 2.0 * batch * (CTX + DRAFT) * d, flops


def work(case):
    kind = case["kind"]
    if kind == "flow":
        nbytes, flops = _flow_work(case["d"], case["layers"], case["steps"], case["batch"])
    elif kind == "latent":
        h, z, i, b = case["hidden"], case["latent"], case["inter"], case["batch"]
        nbytes, flops = _flow_work(z, 8, case["steps"], b)
        vae = 2 * (h * i + 2 * 12 * i * i + i * z)          # both halves: ends and two layers each
        nbytes += 2.0 * vae + 2.0 * b * (CTX + DRAFT) * h
        flops += 2.0 * vae * CTX * b
    elif kind == "depth":
        d, m = case["d"], case["requests"] * case["width"]
        path = (case["live"] + 4) * d * d
        head = SHORTLIST * (d + RANK)
        nbytes = 2.0 * (path + head) + 2.0 * m * d * (case["live"] + 2)
        flops = 2.0 * m * (path + head)
    elif kind == "head":
        d, m = case["d"], case["rows"]
        nbytes, flops = 2.0 * d * (SHORTLIST + m) + 8.0 * m * case["k"], 2.0 * m * d * SHORTLIST
    elif kind == "twopass":
        d, m = case["d"], case["cands"]
        nbytes = 2.0 * SHORTLIST * d + 2.0 * m * (d + RANK)
        flops = 2.0 * SHORTLIST * d * case["depths"] + 2.0 * m * (d + RANK) * case["width"]
    elif kind == "gdn":
        n, hv, kd = case["nodes"], case["vheads"], 128
        dim = 2 * case["heads"] * kd + hv * kd
        state = hv * kd * kd * (2 if case["state"] == "bf16" else 4)
        nbytes = (n + 1.0) * state + 2.0 * (2 * n * dim + (n + 1) * dim * 4 + dim * 5 + n * hv * (kd + 2))
        flops = 7.0 * n * hv * kd * kd + 8.0 * n * dim
    else:
        s, n, h, hk, dim = case["seqs"], case["nodes"], case["heads"], case["kvheads"], case["dim"]
        nbytes = 2.0 * s * n * dim * (3 * h + 2 * hk) + 4.0 * s * n * h + s * n * n + 2.0 * s * (n + 1) * VOCAB
        flops = 4.0 * s * h * n * (n // 4 + 1) * dim + s * (n + 1.0) * VOCAB
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the error each path shows against float64: fp16 rounding points through every
    # block and Euler step, 16-bit logits, bf16 states
    kind = case["kind"]
    if kind in ("flow", "latent"):
        return {"rel": 4e-3, "max": 0.05}
    if kind == "depth":
        return {"rel": 5e-3, "max": 0.05, "differ": 0.01}
    if kind == "head":
        return {"rel": 0.018, "max": 0.1, "differ": 0.01}
    if kind == "twopass":
        return {"rel": 4e-3, "max": 0.05, "differ": 0.01}
    if kind == "gdn":
        return {"rel": 0.015, "max": 0.1}
    return {"rel": 7e-3, "max": 0.05}


# ---------------------------------------------------------------- float64, plain torch
def _ln(x, w, b):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w.double(), b.double(), 1e-5)


def _lin(x, w, b=None):
    y = x @ w.double().t()
    return y if b is None else y + b.double()


def _mha(q, k, v, heads, causal):
    """q [B, S, d], k / v [B, T, d]."""
    split = lambda t: t.unflatten(-1, (heads, -1)).transpose(1, 2)  # noqa: E731
    q, k, v = split(q), split(k), split(v)
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return torch.matmul(s.softmax(-1), v.contiguous()).transpose(1, 2).flatten(-2)


def _exact_flow(w, ctx, layers, steps, heads=8):
    d, nch = ctx.shape[-1], DRAFT // CHUNK
    prefixes = ["expert."] + ["extra_experts.%d." % i for i in range(nch - 1)]
    delta = ctx[:, -1:] - ctx[:, -2:-1]
    z = ctx[:, -1:] + torch.arange(1, DRAFT + 1, device=DEV, dtype=torch.float64).view(1, -1, 1) * delta
    kvs = {}
    for p in prefixes:
        for l in range(layers):
            b = "%sblocks.%d." % (p, l)
            c = _ln(ctx, w[b + "context_norm.weight"], w[b + "context_norm.bias"])
            kvs[b] = _lin(c, w[b + "cross_attn.in_proj_weight"][d:], w[b + "cross_attn.in_proj_bias"][d:]).split(d, -1)
    for s in range(steps):
        vels = []
        for ci, p in enumerate(prefixes):
            n = (ci + 1) * CHUNK
            t = torch.full((1, 1), s / steps, dtype=torch.float64, device=DEV)
            t = torch.nn.functional.silu(_lin(t, w[p + "time_mlp.0.weight"], w[p + "time_mlp.0.bias"]))
            t = _lin(t, w[p + "time_mlp.2.weight"], w[p + "time_mlp.2.bias"])
            x = z[:, :n] + w[p + "position_embedding.weight"][:n].double()
            x[:, n - CHUNK:] += t
            for l in range(layers):
                b = "%sblocks.%d." % (p, l)
                qkv = _lin(_ln(x, w[b + "self_norm.weight"], w[b + "self_norm.bias"]), w[b + "self_attn.in_proj_weight"],
                           w[b + "self_attn.in_proj_bias"])
                x = x + _lin(_mha(*qkv.split(d, -1), heads, True), w[b + "self_attn.out_proj.weight"],
                             w[b + "self_attn.out_proj.bias"])
                q = _lin(_ln(x, w[b + "cross_norm.weight"], w[b + "cross_norm.bias"]),
                         w[b + "cross_attn.in_proj_weight"][:d], w[b + "cross_attn.in_proj_bias"][:d])
                x = x + _lin(_mha(q, *kvs[b], heads, False), w[b + "cross_attn.out_proj.weight"],
                             w[b + "cross_attn.out_proj.bias"])
                g = torch.nn.functional.gelu(_lin(_ln(x, w[b + "ffn.0.weight"], w[b + "ffn.0.bias"]),
                                                  w[b + "ffn.1.weight"], w[b + "ffn.1.bias"]))
                x = x + _lin(g, w[b + "ffn.4.weight"], w[b + "ffn.4.bias"])
            x = _ln(x[:, n - CHUNK:], w[p + "out_norm.weight"], w[p + "out_norm.bias"])
            vels.append(_lin(x, w[p + "out_proj.weight"], w[p + "out_proj.bias"]))
        z = z + torch.cat(vels, 1) / steps
    return z


def _exact_vae(w, x, side, layers=2, heads=8):
    out = "vae.mu" if side == "encoder" else "vae.decoder_out"
    x = _lin(x, w["vae.%s_in.weight" % side], w["vae.%s_in.bias" % side]) \
        + w["vae.%s_pos.weight" % side][:x.shape[1]].double()
    for l in range(layers):
        b = "vae.%s.layers.%d." % (side, l)
        qkv = _lin(_ln(x, w[b + "norm1.weight"], w[b + "norm1.bias"]), w[b + "self_attn.in_proj_weight"],
                   w[b + "self_attn.in_proj_bias"])
        x = x + _lin(_mha(*qkv.chunk(3, -1), heads, False), w[b + "self_attn.out_proj.weight"],
                     w[b + "self_attn.out_proj.bias"])
        g = torch.nn.functional.gelu(_lin(_ln(x, w[b + "norm2.weight"], w[b + "norm2.bias"]), w[b + "linear1.weight"],
                                          w[b + "linear1.bias"]))
        x = x + _lin(g, w[b + "linear2.weight"], w[b + "linear2.bias"])
    return _lin(_ln(x, w["vae.%s_norm.weight" % side], w["vae.%s_norm.bias" % side]), w[out + ".weight"],
                w[out + ".bias"])


def _exact_path(w, embed, lastp, live, pred):
    h = 0
    for j in range(live):
        mask = (lastp[:, j:j + 1] >= 0).double()
        e = embed[lastp[:, j].clamp_min(0).long()].double()
        h = h + mask * _lin(e, w["path_head.offset_proj.%d.weight" % j], w["path_head.offset_proj.%d.bias" % j])
    h = _ln(h, w["path_head.norm.weight"], w["path_head.norm.bias"])
    h = torch.nn.functional.gelu(_lin(h, w["path_head.mlp.0.weight"], w["path_head.mlp.0.bias"]))
    return pred + _lin(h, w["path_head.mlp.3.weight"], w["path_head.mlp.3.bias"])


def _exact_topk(logits, k):
    return logits.log_softmax(-1).topk(k, -1).values, logits.logsumexp(-1)


def _exact_gdn(case, st):
    n, h, hv, kd = case["nodes"], case["heads"], case["vheads"], 128
    par = _tree(n)
    x, conv, w = st["x"].double(), st["conv"].double(), st["w"].double()
    y = torch.empty_like(x)
    for i in range(n):
        s = conv[1 if par[i] < 0 else 2 + par[i]].clone()
        y[i] = st["bias"].double() + (s[:, :3] * w[:, :3]).sum(-1) + x[i] * w[:, 3]
        conv[2 + i] = torch.stack([s[:, 1], s[:, 2], x[i], s[:, 3]], -1)
    y = torch.nn.functional.silu(y)
    unit = lambda t: t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt()  # noqa: E731
    rep = hv // h
    q = unit(y[:, :h * kd].view(n, h, kd)).repeat_interleave(rep, 1) * kd ** -0.5
    k = unit(y[:, h * kd:2 * h * kd].view(n, h, kd)).repeat_interleave(rep, 1)
    v = y[:, 2 * h * kd:].view(n, hv, kd)
    decay = torch.exp(-st["A_log"].double().exp() * torch.nn.functional.softplus(st["a"].double() + st["dt"].double()))
    beta = torch.sigmoid(st["b"].double())
    ssm = st["ssm"].double()
    o = torch.empty(n, hv, kd, dtype=torch.float64, device=DEV)
    for i in range(n):
        s = ssm[1 if par[i] < 0 else 2 + par[i]] * decay[i].view(hv, 1, 1)
        u = (v[i] - (s * k[i][:, None]).sum(-1)) * beta[i][:, None]
        s = s + u[:, :, None] * k[i][:, None]
        o[i] = (s * q[i][:, None]).sum(-1)
        ssm[2 + i] = s
    return {"conv": y, "conv_state": conv, "out": o, "state": ssm}


def _exact_verify(case, st):
    s, n, h, hk, dim = case["seqs"], case["nodes"], case["heads"], case["kvheads"], case["dim"]
    out = st["out"].double()
    flat = st["idx"].long().view(-1)
    take = lambda t, m: t.double()[flat].view(s, n, m, dim).repeat_interleave(h // m, 2).permute(0, 2, 1, 3).contiguous()  # noqa: E731
    q, k, v = take(st["q"], h), take(st["k"], hk), take(st["v"], hk)
    sc = torch.matmul(q, k.transpose(-1, -2).contiguous()) * dim ** -0.5
    sc = sc.masked_fill(st["not_anc"][:, None], float("-inf"))
    own = sc.logsumexp(-1)                                                     # [s, h, n]
    suffix = torch.matmul(sc.softmax(-1), v)
    pre = st["plse"].double().view(h, s, n).transpose(0, 1)
    share = torch.sigmoid(pre - own)[..., None]
    prefix = st["pout"].double().view(s, n, h, dim).permute(0, 2, 1, 3)
    out[flat] = (prefix * share + suffix * (1 - share)).permute(0, 2, 1, 3).reshape(s * n, h, dim)
    return {"out": out, "tokens": None, "path": None, "length": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "flow":
        w = _weights(_cfg(case), None, seed, _is_flow)
        return _exact_flow(w, _hidden("ctx", seed, (case["batch"], CTX, case["d"])).double(), case["layers"], case["steps"])
    if kind == "latent":
        w = _weights(_cfg(case), case["hidden"], seed, lambda n: _is_flow(n) or n.startswith("vae."))
        ctx = _hidden("ctx", seed, (case["batch"], CTX, case["hidden"])).double()
        return _exact_vae(w, _exact_flow(w, _exact_vae(w, ctx, "encoder"), 8, case["steps"]), "decoder")
    if kind == "depth":
        d, live = case["d"], case["live"]
        lastp = _lastp(case, seed)
        pred = _hidden("pred", seed, (case["requests"], DRAFT, d))[:, live].double().repeat_interleave(case["width"], 0)
        hidden = _exact_path(_weights(flownet(d, layers=1), None, seed, _is_path), _normal("embed", seed, (VOCAB, d)),
                             lastp, live, pred)
        lm, sl, w1, w2 = _head_tensors(d, seed)
        logits = _lin(hidden, lm[sl.long()]) + _lin(w1[lastp[:, 0].long()].double(), w2[sl.long()])
        vals, lse = _exact_topk(logits, case["width"])
        return {"hidden": hidden, "vals": vals, "ids": None, "lse": lse}
    if kind == "head":
        d = case["d"]
        lm = _normal("lm_head", seed, (VOCAB, d), 3.0 * d ** -0.5, torch.bfloat16)[_shortlist(seed).long()]
        vals, lse = _exact_topk(_lin(_hidden("x", seed, (case["rows"], d), torch.bfloat16).double(), lm), case["k"])
        return {"vals": vals, "ids": None, "lse": lse}
    if kind == "twopass":
        d = case["d"]
        lm, sl, w1, w2 = _head_tensors(d, seed)
        lm, w2 = lm[sl.long()], w2[sl.long()]
        best = _lin(_hidden("marginals", seed, (case["depths"], d)).double(), lm).log_softmax(-1).amax(0)
        cols = best.topk(case["cands"]).indices
        logits = _lin(_hidden("beams", seed, (case["width"], d)).double(), lm[cols]) \
            + _lin(w1[_ints("prev", seed, (case["width"],), VOCAB).long()].double(), w2[cols])
        vals, lse = _exact_topk(logits, case["width"])
        return {"vals": vals, "tokens": None, "lse": lse}
    if kind == "gdn":
        return _exact_gdn(case, _gdn_inputs(case, seed))
    return _exact_verify(case, _verify_inputs(case, seed))
