"""Performance cases of the NSA framework: the calls a user's program makes, with inputs
of the shapes and distributions it makes them with.

A case is a dict of plain values.  ``kind`` picks the public entry point:

  branch    SlidingWindowAttention / CompressionAttention / SelectionAttention .apply,
            forward alone or forward + gradients (``train``)
  core      NSACore.apply: the three branches, the gates and the mix over given
            compressed keys and selected blocks, forward or forward + gradients
  score     score_and_select: Eq. 8 -> 9 -> 10 -> top-n block indices
  compress  NSAAttention.compress_tokens, forward + gradients
  module    a whole NSAAttention layer, forward + gradients of its input and weights
  decode    NSAAttention.decode: ``steps`` tokens generated after a prompt of T tokens

``exact`` restates each in plain torch at 64 bits (dense masked attention).
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

_PKG = str(Path(__file__).resolve().parents[1] / "nsa-test_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import nsa  # noqa: E402

_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
_PAD_END = 999999  # block_ends value of a padding block (never visible)


def _case(name, kind, **kw):
    c = dict(name=name, kind=kind, dtype="bf16", B=1, train=True, n=16, w=512, l=32, d=16, lp=64)
    c.update(kw)
    return c


def listed():
    return [
        # the repository's smallest configuration: one whole layer in fp32, 512 tokens, 4 query
        # heads a group, gates from the layer's MLP; a unit test's or a toy model's training step,
        # bound by launches and latency
        _case("module_tiny", "module", dtype="fp32", H=8, G=2, T=512, dk=64, dv=64, w=256, n=4, d_model=64,
              gate="sigmoid"),
        # one layer of a small model served: a single query token at a time over a short prompt
        _case("decode_small", "decode", H=8, G=2, T=1000, dk=64, dv=64, w=256, n=16, d_model=512, steps=16,
              gate="softmax", train=False),
        # the sliding-window branch alone, the repository's benchmark of it, forward + backward
        _case("sliding_train", "branch", branch="sliding", B=2, H=8, G=2, T=4096, dk=64, dv=64),
        # a ragged evaluation batch of the selection branch (odd length, 4 heads a group)
        _case("selection_eval_ragged", "branch", branch="selection", B=3, H=16, G=4, T=1537, dk=64, dv=64,
              train=False),
        # the repository's selection stress shape: fp32, 4 query heads a group, forward + backward
        _case("selection_train_fp32", "branch", branch="selection", dtype="fp32", B=4, H=16, G=4, T=2048, dk=64,
              dv=64),
        # the compression branch, ragged length, 16 heads a group, forward + backward
        _case("compression_train_ragged", "branch", branch="compression", B=2, H=32, G=2, T=5003, dk=128, dv=128),
        # token compression (MLP pooling) of a paper-size sequence, forward + backward
        _case("compress_train", "compress", H=64, G=4, T=8192, dk=192, dv=128),
        # a whole default (paper) layer trained on a 2048-token sequence: projections, selection,
        # attention, gates, output projection, and the gradients of all weights
        _case("module_train", "module", H=64, G=4, T=2048, dk=192, dv=128, d_model=2560, gate="sigmoid"),
        # the attention core at the paper configuration, a training step
        _case("core_train_paper", "core", H=64, G=4, T=8192, dk=192, dv=128, gate="sigmoid"),
        # a long prompt evaluated: the long-context configuration's forward
        _case("core_eval_long", "core", H=32, G=2, T=32768, dk=128, dv=128, gate="sigmoid", train=False),
        # block scoring and top-n at the long-context configuration
        _case("score_long", "score", H=32, G=2, T=32768, dk=128, dv=128, train=False),
        # a batch of long sequences served: 16 requests, 16 tokens each after a 32k prompt
        _case("decode_long_batch", "decode", B=16, H=32, G=2, T=32000, dk=128, dv=128, d_model=2560, steps=16,
              gate="sigmoid", train=False),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_HEADS = [(8, 2), (16, 4), (16, 1), (32, 2), (64, 4)]
_DIMS = [(64, 64), (128, 128), (192, 128)]


def draw(rng):
    kind = rng.choice(["branch", "branch", "branch", "core", "core", "score", "compress", "module", "decode",
                       "decode"])
    c = _case("", kind)
    del c["name"]
    c["H"], c["G"] = rng.choice(_HEADS)
    c["dk"], c["dv"] = rng.choice(_DIMS)
    c["dtype"] = "fp32" if rng.random() < 0.25 else "bf16"
    c["w"] = rng.choice([128, 256, 512, 512])
    c["n"] = rng.choice([4, 8, 16, 16])
    # rows (batch x heads x tokens) of the largest listed case of the kind, in fp32 a sixteenth
    rows = 64 * 8192 // (16 if c["dtype"] == "fp32" else 1)
    if kind == "module":
        c["gate"] = rng.choice(["sigmoid", "softmax"])
        c["d_model"] = rng.choice([64, 256, 512, 1024])
        c["B"] = rng.choice([1, 1, 2, 3])
        rows = min(rows, 64 * 2048)
    elif kind == "decode":
        c["gate"] = rng.choice(["sigmoid", "softmax"])
        c["d_model"] = rng.choice([256, 512, 1024, 2560])
        c["steps"] = 16
        c["train"] = False
        c["B"] = _logint(rng, 1, 16)
        c["T"] = _logint(rng, 200, min(32000, 16 * 32000 * 2 * 128 // (c["B"] * c["G"] * c["dk"])))
        return c
    elif kind == "branch":
        c["branch"] = rng.choice(["sliding", "compression", "selection"])
        c["train"] = rng.random() < 0.6
        c["B"] = _logint(rng, 1, 4)
    elif kind == "core":
        c["gate"] = rng.choice(["sigmoid", "softmax"])
        c["train"] = rng.random() < 0.6
        c["B"] = rng.choice([1, 1, 2])
    elif kind == "score":
        c["train"] = False
        c["dv"] = c["dk"]
        c["B"] = rng.choice([1, 1, 2])
    c["T"] = _logint(rng, 200, max(256, min(16384, rows // (c["B"] * c["H"]))))
    return c


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, dt, *shape, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=g) * scale).to(dt)


def _heads(g, dt, B, T, n, d, scale):
    """[B,n,T,d] as a projection stores it: a view of [B,T,n,d]."""
    return _randn(g, dt, B, T, n, d, scale=scale).transpose(1, 2)


def _n_blocks(c):
    n = max((c["T"] - c["l"]) // c["d"] + 1, 0)
    pad = 1
    while pad < n:
        pad *= 2
    return n, pad


def _block_ends(c):
    n, pad = _n_blocks(c)
    be = torch.full((pad,), _PAD_END, dtype=torch.int32, device="cuda")
    be[:n] = torch.arange(n, dtype=torch.int32, device="cuda") * c["d"] + c["l"] - 1
    return be


def _compressed(g, dt, c):
    """K_cmp [B,G,dk,Np] and V_cmp [B,G,Np,dv] as compress_tokens lays them out (zero padding
    blocks)."""
    n, pad = _n_blocks(c)
    k = _randn(g, dt, c["B"], c["G"], pad, c["dk"])
    v = _randn(g, dt, c["B"], c["G"], pad, c["dv"])
    k[:, :, n:] = 0
    v[:, :, n:] = 0
    return k.transpose(-1, -2), v


def _indices(g, c):
    """Selected blocks [B,G,T,n] int64 as top-n gives them: the initial and the two local
    blocks, then the best of the visible ones by a score of which a block's own part (shared by
    all timesteps) and a timestep's part are of equal size; early rows run out of visible blocks
    and take later ones (masked by causality), then -1."""
    B, G, T, n, lp = c["B"], c["G"], c["T"], c["n"], c["lp"]
    nb = (T + lp - 1) // lp
    t = torch.arange(T, device="cuda")
    blk = torch.arange(nb, device="cuda")
    s = torch.randn(B, G, T, nb, device="cuda", generator=g)
    s += torch.randn(B, G, 1, nb, device="cuda", generator=g)
    s = torch.where(blk <= (t // lp).unsqueeze(-1), s, -1000.0 - blk.float())
    fixed = torch.stack([t // lp, ((t - lp) // lp).clamp(min=0), torch.zeros_like(t)], dim=-1)
    bonus = torch.zeros(T, nb, device="cuda").scatter_(1, fixed, 1000.0)
    out = torch.topk(s + bonus, min(n, nb), dim=-1).indices
    return F.pad(out, (0, n - out.shape[-1]), value=-1)


def _config(c):
    return nsa.NSAConfig(d_model=c.get("d_model", 256), head_dim_qk=c["dk"], head_dim_v=c["dv"], l=c["l"], d=c["d"],
                         l_prime=c["lp"], n=c["n"], w=c["w"], n_heads=c["H"], n_kv_groups=c["G"],
                         gate_mode=c.get("gate", "sigmoid"))


def _layer(g, c):
    """A layer with torch's usual initialisation (uniform, 1/sqrt of the input width)."""
    m = nsa.NSAAttention(_config(c)).to("cuda", _DT[c["dtype"]])
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name == "pos_embed.weight":
                b = 1.0
            else:
                lay = m.get_submodule(name.rsplit(".", 1)[0])
                b = 1.0 / math.sqrt(lay.in_features)
            p.copy_((torch.rand(p.shape, device="cuda", generator=g) * 2 - 1) * b)
    return m


def _inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    B, H, G, T, dk, dv = c["B"], c["H"], c["G"], c["T"], c["dk"], c["dv"]
    s = {"case": c, "cfg": _config(c), "scale": 1.0 / math.sqrt(dk)}
    kind = c["kind"]
    if kind == "branch":
        # contiguous [B,H,T,d], keys in the reference's [B,G,dk,T]
        s["q"] = _randn(g, dt, B, H, T, dk)
        if c["branch"] == "compression":
            s["k"], s["v"] = _compressed(g, dt, c)
            s["be"] = _block_ends(c)
        else:
            s["k"] = _randn(g, dt, B, G, dk, T)
            s["v"] = _randn(g, dt, B, G, T, dv)
        if c["branch"] == "selection":
            s["idx"] = _indices(g, c)
        s["do"] = _randn(g, dt, B, H, T, dv)
        s["leaves"] = ["q", "k", "v"]
    elif kind == "core":
        s["q"] = _heads(g, dt, B, T, H, dk, 1.0)
        s["kc"], s["vc"] = _compressed(g, dt, c)
        s["be"] = _block_ends(c)
        for br in ("s", "w"):
            s["k" + br] = _heads(g, dt, B, T, G, dk, 1.0).transpose(-1, -2)
            s["v" + br] = _heads(g, dt, B, T, G, dv, 1.0)
        s["idx"] = _indices(g, c)
        s["gates"] = _randn(g, dt, B, T, H, 3).permute(0, 2, 1, 3)
        s["do"] = _heads(g, dt, B, T, H, dv, 1.0)
        s["leaves"] = ["q", "kc", "vc", "ks", "vs", "kw", "vw", "gates"]
    elif kind == "score":
        # a component of rank 8 shared by all heads, as in the long-context configuration: peaked
        # block scores
        basis = torch.randn(B, T, 8, device="cuda", generator=g)
        pq = torch.randn(8, dk, device="cuda", generator=g)
        pk = torch.randn(8, dk, device="cuda", generator=g)
        n, pad = _n_blocks(c)
        q = torch.randn(B, T, H, dk, device="cuda", generator=g) + (basis @ pq).unsqueeze(2)
        s["q"] = q.to(dt).transpose(1, 2)
        k = torch.zeros(B, G, pad, dk, device="cuda")
        k[:, :, :n] = (torch.randn(B, G, n, dk, device="cuda", generator=g)
                       + (basis @ pk)[:, c["l"] - 1::c["d"]][:, :n].unsqueeze(1))
        s["k"] = k.to(dt).transpose(-1, -2)
        s["be"] = _block_ends(c)
    elif kind == "compress":
        s["m"] = _layer(g, c)
        s["k"] = _heads(g, dt, B, T, G, dk, 1.0)
        s["v"] = _heads(g, dt, B, T, G, dv, 1.0)
        n, pad = _n_blocks(c)
        s["dkc"] = _randn(g, dt, B, G, pad, dk).transpose(-1, -2)
        s["dvc"] = _randn(g, dt, B, G, pad, dv)
    elif kind == "module":
        s["m"] = _layer(g, c)
        s["x"] = _randn(g, dt, B, T, c["d_model"])
        s["do"] = _randn(g, dt, B, T, c["d_model"])
    else:
        s["m"] = _layer(g, c)
        s["prompt"] = _randn(g, dt, B, T, c["d_model"])
        s["x"] = _randn(g, dt, B, c["steps"], c["d_model"])
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["train"]:
        for k in s.get("leaves", []):
            s[k] = s[k].requires_grad_()
        if case["kind"] in ("compress", "module"):
            for k in ("k", "v", "x"):
                if k in s:
                    s[k] = s[k].requires_grad_()
    if case["kind"] == "decode":
        m = s["m"].eval()
        cache = nsa.NSAKVCache(s["cfg"], case["B"], case["T"] + case["steps"], "cuda", _DT[case["dtype"]])
        m.prefill(s.pop("prompt"), cache)
        s["cache"], s["n_act"] = cache, cache.n_act
    return s


_COMPRESS_WEIGHTS = ("compress_mlp.0.weight", "compress_mlp.0.bias", "compress_mlp.2.weight", "compress_mlp.2.bias",
                     "pos_embed.weight")


def _weights(m):
    """A layer's trained weights.  The compressed keys' output bias is frozen: it shifts every
    logit of a query alike, so its gradient is zero but for rounding."""
    return [(n, p) for n, p in m.named_parameters() if n != "compress_mlp.2.bias"]


def run(s):
    c = s["case"]
    kind, scale, cfg = c["kind"], s["scale"], s["cfg"]
    if kind == "branch":
        with torch.set_grad_enabled(c["train"]):
            if c["branch"] == "sliding":
                o = nsa.SlidingWindowAttention.apply(s["q"], s["k"], s["v"], scale, cfg.w, cfg)
            elif c["branch"] == "compression":
                o = nsa.CompressionAttention.apply(s["q"], s["k"], s["v"], s["be"], scale, cfg)
            else:
                o = nsa.SelectionAttention.apply(s["q"], s["k"], s["v"], s["idx"], scale, cfg)
        if not c["train"]:
            return o
        return (o.detach(), *torch.autograd.grad(o, [s[k] for k in s["leaves"]], s["do"]))
    if kind == "core":
        with torch.set_grad_enabled(c["train"]):
            o = nsa.NSACore.apply(s["q"], s["kc"], s["vc"], s["be"], s["ks"], s["vs"], s["idx"], s["kw"], s["vw"],
                                  s["gates"], scale, cfg)
        if not c["train"]:
            return o
        return (o.detach(), *torch.autograd.grad(o, [s[k] for k in s["leaves"]], s["do"]))
    if kind == "score":
        with torch.no_grad():
            return nsa.score_and_select(s["q"], s["k"], s["be"], scale, cfg)
    if kind == "compress":
        kc, vc, _, _ = s["m"].compress_tokens(s["k"], s["v"])
        ws = [s["m"].get_parameter(n) for n in _COMPRESS_WEIGHTS]
        g = torch.autograd.grad([kc, vc], [s["k"], s["v"], *ws], [s["dkc"], s["dvc"]])
        return (kc.detach(), vc.detach(), *g)
    if kind == "module":
        out, _ = s["m"](s["x"])
        g = torch.autograd.grad(out, [s["x"], *[p for _, p in _weights(s["m"])]], s["do"])
        return (out.detach(), *g)
    # the answer is generated again from the end of the prompt
    cache = s["cache"]
    cache.length, cache.n_act = c["T"], s["n_act"]
    out = torch.cat([s["m"].decode(s["x"][:, i:i + 1], cache)[0] for i in range(c["steps"])], dim=1)
    return out, cache.K_cmp, cache.V_cmp


# -------------------------------------------------------------------------------- work
def _pairs(c):
    """(sliding, compression, selection) visible (query, key) pairs per (batch, head)."""
    T, w, lp = c["T"], c["w"], c["lp"]
    t = np.arange(T, dtype=np.int64)
    n, _ = _n_blocks(c)
    sl = int(np.minimum(t + 1, w).sum())
    cm = int(np.clip((t - c["l"] + 1) // c["d"] + 1, 0, n).sum())
    full = np.minimum(c["n"] - 1, t // lp) * lp  # whole blocks before the query's own
    return sl, cm, int((full + t % lp + 1).sum())


def work(c):
    B, H, G, T, dk, dv = c["B"], c["H"], c["G"], c["T"], c["dk"], c["dv"]
    es = 2 if c["dtype"] == "bf16" else 4
    sl, cm, se = _pairs(c)
    n, pad = _n_blocks(c)
    row = B * H * T * es
    kind, train = c["kind"], c["train"]
    per_pair = 2 * (4 * dk + 3 * dv) if train else 2 * (dk + dv)

    def kv(tokens):
        return B * G * tokens * (dk + dv) * es

    def mlp(tokens, blocks):  # compression MLP, forward
        return 2 * B * G * (tokens * dk * 2 * dk + blocks * 2 * dk * dk)

    if kind == "branch":
        br = c["branch"]
        p = {"sliding": sl, "compression": cm, "selection": se}[br]
        tk = pad if br == "compression" else T
        by = row * (dk + dv) + kv(tk)
        if train:  # dO read, dq written, dk / dv written
            by += row * (dv + dk) + kv(tk)
        if br == "selection":
            by += B * G * T * c["n"] * 8
        return {"bytes": by, "flops": B * H * p * per_pair}
    if kind == "core":
        by = row * (dk + dv) + 2 * kv(T) + kv(pad) + B * G * T * c["n"] * 8 + row * 3
        if train:
            by += row * (dv + dk) + 2 * kv(T) + kv(pad) + row * 3
        return {"bytes": by, "flops": B * H * (sl + cm + se) * per_pair}
    if kind == "score":
        return {"bytes": row * dk + B * G * pad * dk * es + B * G * T * c["n"] * 8, "flops": B * H * cm * 2 * dk}
    if kind == "compress":
        return {"bytes": 2 * (kv(T) + kv(pad)) + 8 * dk * dk * es, "flops": 3 * mlp(T, n)}
    dm = c["d_model"]
    kvw = 3 * G * (dk + dv)
    weights = dm * (H * dk + kvw + dm // 2 + H * dv) + (dm // 2) * 3 * H + (dk + c["l"]) * 2 * dk + 2 * dk * dk
    if kind == "module":
        fl = 2 * B * T * weights * 3 + 3 * mlp(T, n) + B * H * (sl + cm + se) * per_pair + B * H * cm * 2 * dk
        return {"bytes": 4 * B * T * dm * es + 2 * weights * es, "flops": fl}
    seen = min(c["w"], T) + min(c["n"] * c["lp"], T)
    by = c["steps"] * (weights * es + kv(seen + n) + B * 2 * dm * es)
    fl = c["steps"] * (2 * B * weights + B * H * ((seen + n) * 2 * (dk + dv) + n * 2 * dk))
    return {"bytes": by, "flops": fl}


def tolerance(c):
    """About four times the error of the path itself against ``exact`` (the largest of its
    outputs): bf16 branches 3.2e-3; compress 2.1e-2 (a pre-activation within a rounding of zero
    switches its unit's gradient on or off, also in a layer: 5.3e-2); decoding 2.8e-2 (a rounding
    of a compressed key can change which block is chosen); fp32 1e-6, a layer 5.9e-6."""
    kind, bf = c["kind"], c["dtype"] == "bf16"
    if kind == "score":
        return "exact"  # block indices, of one fixed order of operations
    if not bf:
        return {"rel": 2.5e-5 if kind == "module" else 5e-6}
    return {"rel": {"compress": 8e-2, "module": 1e-1, "decode": 1e-1}.get(kind, 1.2e-2)}


# ------------------------------------------------------------------------------- exact
def _attend(q, k, v, vis, scale):
    """q [h,n,dk], k [S,dk], v [S,dv], vis [n,S] -> [h,n,dv]; a row that sees nothing gives 0."""
    s = (q @ k.t()) * scale
    s = s.masked_fill(~vis, -math.inf)
    m = s.amax(-1, keepdim=True).clamp(min=-1e300).detach()
    p = torch.exp(s - m)
    z = p.sum(-1, keepdim=True)
    return (p @ v) / torch.where(z > 0, z, torch.ones_like(z))


def _visible(br, c, t, S, be=None, idx=None):
    """[len(t), S] visibility of the keys 0..S-1 (compression: blocks) to the timesteps t."""
    if br == "compression":
        return be[:S] <= t.unsqueeze(1)
    j = torch.arange(S, device=t.device)
    vis = j <= t.unsqueeze(1)
    if br == "sliding":
        return vis & (j > t.unsqueeze(1) - c["w"])
    nb = (S + c["lp"] - 1) // c["lp"]
    on = torch.zeros(len(t), nb + 1, dtype=torch.bool, device=t.device)
    on.scatter_(1, torch.where((idx < 0) | (idx >= nb), nb, idx), True)
    return vis & on[:, j // c["lp"]]


def _branch_exact(c, br, q, k, v, scale, be=None, idx=None, do=None):
    """out (and dq, dk [B,G,S,dk], dv) of one branch over k, v [B,G,S,*], in float64, a group
    and a chunk of timesteps at a time; do [B,H,T,dv]."""
    B, H, T, _ = q.shape
    G, S = k.shape[1], k.shape[2]
    hp = H // G
    out = torch.empty(B, H, T, v.shape[-1], device=q.device, dtype=torch.float64)
    dq, dk, dv = (torch.zeros_like(x, dtype=torch.float64) for x in (q, k, v)) if do is not None else (None,) * 3
    step = max(16, int(2 ** 28 // (S * hp)))
    for b in range(B):
        for g in range(G):
            h = slice(g * hp, (g + 1) * hp)
            for t0 in range(0, T, step):
                t1 = min(T, t0 + step)
                s1 = S if br == "compression" else min(S, t1)
                s0 = max(0, t0 - c["w"]) if br == "sliding" else 0
                t = torch.arange(t0, t1, device=q.device)
                vis = _visible(br, c, t, s1, be, None if idx is None else idx[b, g, t0:t1])[:, s0:]
                qq, kk, vv = (x.double().detach() for x in (q[b, h, t0:t1], k[b, g, s0:s1], v[b, g, s0:s1]))
                if do is None:
                    out[b, h, t0:t1] = _attend(qq, kk, vv, vis, scale)
                    continue
                leaf = [x.requires_grad_() for x in (qq, kk, vv)]
                with torch.enable_grad():
                    o = _attend(*leaf, vis, scale)
                out[b, h, t0:t1] = o.detach()
                gq, gk, gv = torch.autograd.grad(o, leaf, do[b, h, t0:t1].double())
                dq[b, h, t0:t1] = gq
                dk[b, g, s0:s1] += gk
                dv[b, g, s0:s1] += gv
    return (out, dq, dk, dv) if do is not None else out


def _act(z, gate):
    return torch.softmax(z, -1) if gate == "softmax" else torch.sigmoid(z)


def _compress_exact(W, c, k, v, st=lambda x: x):
    """K_cmp [B,G,n,dk], V_cmp [B,G,n,dv] of k, v [B,G,T,*] (before padding), float64; st is
    applied to every intermediate that a layer stores."""
    l, d = c["l"], c["d"]
    w1, dk = W["compress_mlp.0.weight"], c["dk"]
    y = st(st(k) @ w1[:, :dk].t())
    pos = st(W["pos_embed.weight"] @ w1[:, dk:].t() + W["compress_mlp.0.bias"])
    r = st(torch.relu(y.unfold(2, l, d).transpose(-1, -2) + pos).mean(-2))
    return st(r @ W["compress_mlp.2.weight"].t() + W["compress_mlp.2.bias"]), v.unfold(2, l, d).mean(-1)


def _top_n(c, q, kc, be, scale, t):
    """Block indices [B,G,len(t),n] of the queries q [B,H,len(t),dk] at positions t (float64)."""
    B, H, n_t, _ = q.shape
    G, N = kc.shape[1], kc.shape[2]
    lp, d = c["lp"], c["d"]
    a, s = c["l"] // d, lp // d
    nsel = (N + s - 1) // s
    lg = (q.view(B, G, H // G, n_t, -1).double() @ kc.double().transpose(-1, -2).unsqueeze(2)) * scale
    vis = be[:N] <= t.unsqueeze(1)
    p = torch.softmax(lg.masked_fill(~vis, -1e300), -1) * vis
    p = F.pad(p, (0, nsel * s + s + a - N))
    agg = sum(p[..., m + i: m + i + s * nsel: s][..., :nsel] for m in range(s) for i in range(a)).sum(2)
    fixed = torch.stack([torch.zeros_like(t), ((t - lp) // lp).clamp(min=0), t // lp], -1)
    bonus = torch.zeros(n_t, max(nsel, int(t.max()) // lp + 1), device=q.device, dtype=torch.float64)
    bonus.scatter_(1, fixed, 1e6)
    agg = F.pad(agg, (0, bonus.shape[1] - nsel), value=-1.0) + bonus
    top = torch.topk(agg, min(c["n"], agg.shape[-1]), dim=-1)
    return top.indices


def _proj(W, x, name, n):
    B, T, _ = x.shape
    return (x @ W[name + ".weight"].t()).view(B, T, n, -1).transpose(1, 2)


def _gate_exact(W, x, H):
    h = torch.relu(x @ W["gate_mlp.0.weight"].t() + W["gate_mlp.0.bias"])
    z = h @ W["gate_mlp.2.weight"].t() + W["gate_mlp.2.bias"]
    return z.view(*x.shape[:2], H, 3).permute(0, 2, 1, 3)


class _BranchFn(torch.autograd.Function):
    """_branch_exact as a differentiable function of q, k, v (for the whole layer)."""

    @staticmethod
    def forward(ctx, q, k, v, c, br, scale, be, idx):
        ctx.save_for_backward(q, k, v)
        ctx.rest = (c, br, scale, be, idx)
        return _branch_exact(c, br, q, k, v, scale, be, idx)

    @staticmethod
    def backward(ctx, do):
        c, br, scale, be, idx = ctx.rest
        q, k, v = ctx.saved_tensors
        _, dq, dk, dv = _branch_exact(c, br, q, k, v, scale, be, idx, do)
        return dq, dk, dv, None, None, None, None, None


def _exact_module(s, c):
    dt, H, G, T = _DT[c["dtype"]], c["H"], c["G"], c["T"]

    def st(v):
        return v.to(dt).double()

    W = {k: p.detach().double().requires_grad_() for k, p in s["m"].named_parameters()}
    x = s["x"].double().requires_grad_()
    scale, be = s["scale"], _block_ends(c)
    q = _proj(W, x, "q_proj", H)
    k_in, v_in = _proj(W, x, "k_compress", G), _proj(W, x, "v_compress", G)
    kc, vc = _compress_exact(W, c, k_in, v_in)
    t = torch.arange(T, device="cuda")
    with torch.no_grad():  # the choice of blocks is made on the values the layer stores
        ks, _ = _compress_exact(W, c, k_in, v_in, st)
        idx = torch.cat([_top_n(c, st(q[:, :, a:a + 512]), ks, be, scale, t[a:a + 512])
                         for a in range(0, T, 512)], 2)
    o_c = _BranchFn.apply(q, kc, vc, c, "compression", scale, be, None)
    o_s = _BranchFn.apply(q, _proj(W, x, "k_select", G), _proj(W, x, "v_select", G), c, "selection", scale, None, idx)
    o_w = _BranchFn.apply(q, _proj(W, x, "k_sliding", G), _proj(W, x, "v_sliding", G), c, "sliding", scale, None, None)
    a = _act(_gate_exact(W, x, H), c["gate"])
    o = o_c * a[..., :1] + o_s * a[..., 1:2] + o_w * a[..., 2:]
    out = o.transpose(1, 2).reshape(c["B"], T, -1) @ W["o_proj.weight"].t()
    g = torch.autograd.grad(out, [x, *[W[k] for k, _ in _weights(s["m"])]], s["do"].double())
    return (out.detach(), *g)


def _exact_decode(s, c):
    dt, H, G, B, T, n_t = _DT[c["dtype"]], c["H"], c["G"], c["B"], c["T"], c["steps"]

    def st(v):
        return v.to(dt).double()

    W = {k: p.detach().double() for k, p in s["m"].named_parameters()}
    scale, outs, kcs, vcs = s["scale"], [], [], []
    cc = dict(c, T=T + n_t)
    n, pad = _n_blocks(cc)
    be = _block_ends(cc)
    for b in range(B):
        x = torch.cat([s["prompt"][b:b + 1], s["x"][b:b + 1]], 1).double()
        t = torch.arange(T, T + n_t, device="cuda")
        xq = x[:, T:]
        q = _proj(W, xq, "q_proj", H)
        kv = {m: _proj(W, x, m, G) for m in ("k_compress", "v_compress", "k_select", "v_select", "k_sliding", "v_sliding")}
        kc, vc = _compress_exact(W, c, kv["k_compress"], kv["v_compress"])
        idx = _top_n(c, st(q), _compress_exact(W, c, kv["k_compress"], kv["v_compress"], st)[0], be, scale, t)
        kcs.append(F.pad(kc, (0, 0, 0, pad - n)).transpose(-1, -2))
        vcs.append(F.pad(vc, (0, 0, 0, pad - n)))
        o = []
        for br, k, v in (("compression", kc, vc), ("selection", kv["k_select"], kv["v_select"]),
                         ("sliding", kv["k_sliding"], kv["v_sliding"])):
            r = torch.empty(1, H, n_t, c["dv"], device="cuda", dtype=torch.float64)
            for g in range(G):
                h = slice(g * (H // G), (g + 1) * (H // G))
                vis = _visible(br, c, t, k.shape[2], be, idx[0, g])
                r[0, h] = _attend(q[0, h], k[0, g], v[0, g], vis, scale)
            o.append(r)
        a = _act(_gate_exact(W, xq, H), c["gate"])
        mix = o[0] * a[..., :1] + o[1] * a[..., 1:2] + o[2] * a[..., 2:]
        outs.append(mix.transpose(1, 2).reshape(1, n_t, -1) @ W["o_proj.weight"].t())
    return torch.cat(outs), torch.cat(kcs), torch.cat(vcs)


def exact(case, seed):
    c = case
    s = _inputs(c, seed)
    kind, scale, train = c["kind"], s["scale"], c["train"]
    with torch.set_grad_enabled(train):
        if kind == "branch":
            r = _branch_exact(c, c["branch"], s["q"], s["k"].transpose(-1, -2), s["v"], scale, s.get("be"),
                              s.get("idx"), s["do"] if train else None)
            return (r[0], r[1], r[2].transpose(-1, -2), r[3]) if train else r
        if kind == "core":
            a = _act(s["gates"].double(), c["gate"])
            do = s["do"].double() if train else None
            out, dq, grads, dots = 0, 0, [], []
            for i, (br, k, v) in enumerate((("compression", "kc", "vc"), ("selection", "ks", "vs"),
                                            ("sliding", "kw", "vw"))):
                d = do * a[..., i:i + 1] if train else None
                r = _branch_exact(c, br, s["q"], s[k].transpose(-1, -2), s[v], scale, s["be"], s["idx"], d)
                o = r[0] if train else r
                out = out + o * a[..., i:i + 1]
                if train:
                    dq = dq + r[1]
                    grads += [r[2].transpose(-1, -2), r[3]]
                    dots.append((do * o).sum(-1))
            if not train:
                return out
            dots = torch.stack(dots, -1)
            da = (a * (dots - (a * dots).sum(-1, keepdim=True)) if c["gate"] == "softmax" else a * (1 - a) * dots)
            return (out, dq, *grads, da)
        if kind == "compress":
            W = {k: s["m"].get_parameter(k).detach().double().requires_grad_() for k in _COMPRESS_WEIGHTS}
            k, v = (s[x].double().requires_grad_() for x in ("k", "v"))
            kc, vc = _compress_exact(W, c, k, v)
            n, pad = _n_blocks(c)
            kc = F.pad(kc, (0, 0, 0, pad - n)).transpose(-1, -2)
            vc = F.pad(vc, (0, 0, 0, pad - n))
            g = torch.autograd.grad([kc, vc], [k, v, *W.values()], [s["dkc"].double(), s["dvc"].double()])
            return (kc.detach(), vc.detach(), *g)
        if kind == "module":
            return _exact_module(s, c)
        if kind == "decode":
            return _exact_decode(s, c)
    return None  # block indices: an order of blocks, not a computed number
