"""The work this package is timed on: calls that a program makes through its public
entry points, over the range of sizes it supports.

A case names one call: the Lighthouse layer (``lighthouse_layer``, trained or forward
only), the layer fed from the fused projection (``lighthouse_layer_rope``), dense causal
attention, the GLA and the dilated scorer modules, one Llama3 block and a small whole
model.  ``prepare`` makes its inputs on the GPU, ``run`` makes the call, ``exact`` gives
the same results in float64 with plain torch.
"""
import dataclasses
import math

import torch
import torch.nn.functional as F

import __graft_entry__

PKG = __graft_entry__.load_package()
LLAMA = PKG.llama3
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
DIL = 4         # dilation of the reference's dilated and GLA flavors
ROPE_THETA = 10000


def _layer(name, S, k, **kw):
    c = dict(name=name, kind="layer", B=1, S=S, H=8, D=128, L=3, p=4, k=k, dtype="bf16", train=True, heavy=False)
    c.update(kw)
    return c


def listed():
    return [
        # The smallest training call: one short sequence with a single selection tile.
        _layer("layer_2k", 2048, 128),
        # Two ragged sequences in fp16 whose length no pooling span divides.
        _layer("layer_11k_fp16", 11003, 512, B=2, H=6, dtype="fp16"),
        # The headline configuration: 32K tokens, k = 2048.
        _layer("layer_32k", 32768, 2048),
        # The longest row of the top-k sweep: 64K tokens, k = 6144, 5% of the keys x4.
        _layer("layer_64k", 65536, 6144, heavy=True),
        # Forward only, as in evaluation: the two-fold pooling of the lvl3 flavors.
        _layer("layer_16k_eval", 16384, 1536, p=2, train=False),
        # The head width and head count of the 2B flavor's trunk.
        _layer("layer_8k_head64", 8192, 512, H=32, D=64),
        # The 270M model's Lighthouse layer, rotary embedding folded in.
        dict(name="rope_layer_32k", kind="rope", B=1, S=32768, H=8, L=3, p=4, k=1536),
        # The full-attention layers of the 270M model.
        dict(name="dense_16k", kind="dense", B=1, S=16384, H=8, D=128, dtype="bf16"),
        # The GLA scorer at the reference's GLA configuration.
        dict(name="gla_scorer_32k", kind="gla", B=1, S=32768, H=8, D=128, L=3, p=4, dtype="bf16"),
        # The dilated scorer over the deep hierarchy.
        dict(name="dilated_scorer_16k", kind="dilated", B=1, S=16384, H=8, D=128, L=5, p=2, dtype="bf16"),
        # One Lighthouse block of the 270M trunk, forward and backward.
        dict(name="block_8k", kind="block", B=1, S=8192, L=3, p=4, k=512),
        # A whole small model of the 270M ablation flavor (dense, head width 72), one short batch.
        dict(name="model_2k_head72", kind="model", B=1, S=2048, layers=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tiles(rng, S, L, p):
    """A top-k that leaves 128 to 512 coarsest nodes per tile, as the flavors' do."""
    coarsest = S // p ** (L - 1)
    return 128 * max(1, round(coarsest / _log_int(rng, 128, 512)))


def draw(rng):
    top = _cost(next(c for c in listed() if c["name"] == "layer_64k"))
    while True:
        c = _draw(rng)
        if _cost(c) <= top:
            return c


def _draw(rng):
    kind = rng.choice(["layer"] * 6 + ["rope", "dense", "dense", "gla", "dilated", "block", "model"])
    c = dict(kind=kind, B=rng.choice([1, 1, 1, 2, 3]))
    L, p = rng.choice([(2, 2), (2, 4), (3, 2), (3, 4), (3, 4), (4, 2)])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    D = rng.choice([128, 128, 128, 64, 72])
    if kind == "layer":
        S = _log_int(rng, 2048, 65536)
        c.update(S=S, H=rng.choice([2, 4, 8, 8, 12, 16, 32]), D=D, L=L, p=p, k=_tiles(rng, S, L, p), dtype=dtype,
                 train=rng.random() < 0.7, heavy=rng.random() < 0.3)
    elif kind == "rope":
        S = _log_int(rng, 2048, 32768)
        c.update(S=S, H=rng.choice([4, 8, 16]), L=L, p=p, k=_tiles(rng, S, L, p))
    elif kind == "dense":
        c.update(S=_log_int(rng, 500, 24000), H=rng.choice([2, 8, 8, 16, 32]), D=D, dtype=dtype)
    elif kind in ("gla", "dilated"):
        S = DIL * _log_int(rng, 256, 8192 if kind == "gla" else 6000)
        c.update(S=S, H=rng.choice([4, 8, 16]), D=D, L=L, p=p, dtype=dtype)
    elif kind == "block":
        S = _log_int(rng, 2048, 16384)
        c.update(B=1, S=S, L=L, p=p, k=_tiles(rng, S, L, p))
    else:
        c.update(S=_log_int(rng, 300, 6000), layers=rng.choice([1, 2, 3]))
    return c


# ---------------------------------------------------------------------------
# sizes and work
# ---------------------------------------------------------------------------
def _selected(S, L, p, k):
    """Selected rows per (batch, head): per tile the coarsest nodes and the children of
    at most 128 selected nodes per level."""
    tiles = k // 128
    n = S // p ** (L - 1) // tiles
    total = n
    for _ in range(L - 1):
        n = p * min(n, 128)
        total += n
    return tiles * total


def _block_args(c):
    a = LLAMA.llama3_args["ablation_270m_lighthouse_topk1536_pool4_lvl3"]
    return dataclasses.replace(a, lighthouse_num_levels=c["L"], lighthouse_pooling_factor=c["p"],
                               lighthouse_topk=c["k"], lighthouse_strict=False)


def _model_args(c):
    return dataclasses.replace(LLAMA.llama3_args["ablation_270m"], n_layers=c["layers"], vocab_size=256,
                               max_seq_len=c["S"])


def _cost(c):
    w = work(c)
    return max(w["flops"] / 1e12, w["bytes"] / 3e9)


def work(case):
    c, kind = case, case["kind"]
    B, S = c["B"], c["S"]
    T = B * S
    if kind in ("layer", "rope"):
        H, D, train = c["H"], c.get("D", 128), c.get("train", True)
        n = _selected(S, c["L"], c["p"], c["k"])
        # q, k, v in, out out; trained: the upstream gradient in, three gradients out
        return {"bytes": T * H * D * 2 * (8 if train else 4) + 4 * B * H * n,
                "flops": (14 if train else 4) * D * B * H * n * (n + 1) / 2}
    if kind == "dense":
        return {"bytes": T * c["H"] * c["D"] * 2 * 8, "flops": 14 * c["D"] * B * c["H"] * S * (S + 1) / 2}
    if kind in ("gla", "dilated"):
        H, D = c["H"], c["D"]
        rows = sum(S // c["p"] ** l for l in range(c["L"]))
        io = 2 * B * H * (3 * S * D + 3 * rows * D + 2 * rows)
        if kind == "gla":  # two directions, state update and readout per token
            return {"bytes": io + 2 * T * H, "flops": 2 * T * H * 4 * D * D}
        s = S // DIL
        return {"bytes": io, "flops": 2 * 4 * D * B * H * DIL * s * (s + 1) / 2}
    if kind == "block":
        n, heads = _selected(S, c["L"], c["p"], c["k"]), 8
        params = 1024 * 1024 * 4 + 3 * 1024 * 1024
        return {"bytes": T * 1024 * 2 * 4 + 3 * params * 2,
                "flops": 6 * params * T + 14 * 128 * B * heads * n * (n + 1) / 2}
    params = c["layers"] * (4 * 576 * 576 + 3 * 576 * 1024) + 256 * 576
    return {"bytes": 3 * 2 * params + T * 256 * 2,
            "flops": 6 * params * T + c["layers"] * 14 * 72 * B * 8 * S * (S + 1) / 2}


# Relative 2-norm errors, about four times what each path shows against ``exact`` (16-bit
# rows: 3e-3 to 4e-3 in bf16, an eighth of that in fp16).  The integer outputs (selected
# indices) hang on 16-bit rounded scores, of which a few in a hundred thousand round the
# other way when a norm is summed in another order; the layer's fp16 bound allows for the
# rows that such a change moves.
def tolerance(case):
    half = case.get("dtype") == "fp16"
    return {
        "layer": {"rel": 0.008 if half else 0.016, "differ": 0.002},
        "rope": {"rel": 0.016, "differ": 0.002},
        "dense": {"rel": 0.002 if half else 0.012},
        "gla": {"rel": 0.002 if half else 0.008},
        "dilated": {"rel": 0.002 if half else 0.008},
        "block": {"rel": 0.03},
        "model": {"rel": 0.03},
    }[case["kind"]]


# ---------------------------------------------------------------------------
# inputs and the calls
# ---------------------------------------------------------------------------
def _randn(gen, *shape, dtype):
    return torch.randn(*shape, device="cuda", generator=gen).to(dtype)


def prepare(case, seed):
    c, kind = dict(case), case["kind"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": c}
    B, S = c["B"], c["S"]
    dtype = DTYPES[c.get("dtype", "bf16")]
    if kind in ("layer", "dense", "gla", "dilated"):
        H, D = c["H"], c["D"]
        xs = [torch.randn(B, S, H, D, device="cuda", generator=gen) for _ in range(3)]
        if c.get("heavy"):  # 5% of the key positions x4: heavy-tailed scores
            pos = torch.randperm(S, device="cuda", generator=gen)[:max(1, S // 20)]
            xs[1][:, pos] *= 4
        s["x"] = [x.to(dtype) for x in xs]
    if kind == "layer":
        s["dout"] = _randn(gen, B, H, S, D, dtype=dtype) if c["train"] else None
        scorer = PKG.DialatedLighthouseNormScorer(pooling_factor=c["p"], levels=c["L"])
        s["layer"] = PKG.LighthouseLocal(None, scorer, num_levels=c["L"], pooling_factor=c["p"], topk=c["k"],
                                         strict=False)
        if c["train"]:
            s["x"] = [x.requires_grad_() for x in s["x"]]
    elif kind == "dense":  # [B, H, S, D] views of the projections, as the model calls it
        s["x"] = [x.transpose(1, 2).requires_grad_() for x in s["x"]]
        s["dout"] = _randn(gen, B, S, H, D, dtype=dtype).transpose(1, 2)
        s["attention"] = PKG.dense_attention.ScaledDotProductAttention()
    elif kind == "gla":
        s["gk"] = F.logsigmoid(_randn(gen, B, S, H, dtype=dtype)) / 16
        s["scorer"] = PKG.DilatedLighthouseGLAScorer(head_dim=D, dilation=DIL, pooling_factor=c["p"], levels=c["L"])
    elif kind == "dilated":
        s["scorer"] = PKG.DilatedLighthouseScorer(head_dim=D, dilation=DIL, pooling_factor=c["p"], levels=c["L"])
    elif kind == "rope":
        W = c["H"] * 128
        s["x"] = _randn(gen, B, S, 3 * W, dtype=dtype).requires_grad_()
        s["dout"] = _randn(gen, B, S, c["H"], 128, dtype=dtype).transpose(1, 2)
        s["freqs"] = torch.view_as_real(LLAMA.precompute_freqs_cis(128, S, ROPE_THETA)).cuda()
    elif kind == "block":
        args = _block_args(c)
        torch.manual_seed(seed)
        with torch.device("cuda"):
            block = LLAMA.TransformerBlock(2, args)
            block.init_weights()
        s["block"] = LLAMA.cast_params_(block, torch.bfloat16)
        s["params"] = list(block.parameters())
        s["freqs"] = LLAMA.precompute_freqs_cis(args.dim // args.n_heads, S, args.rope_theta).cuda()
        s["x"] = _randn(gen, B, S, args.dim, dtype=dtype).requires_grad_()
        s["dout"] = _randn(gen, B, S, args.dim, dtype=dtype)
    else:
        torch.manual_seed(seed)
        with torch.device("cuda"):
            model = LLAMA.Transformer(_model_args(c))
        model.init_weights()
        s["model"] = LLAMA.cast_params_(model, torch.bfloat16)
        s["params"] = list(model.parameters())
        tokens = torch.randint(0, 256, (B, S + 1), device="cuda", generator=gen)
        s["tokens"], s["labels"] = tokens[:, :-1].contiguous(), tokens[:, 1:].contiguous()
    return s


def run(state):
    s, kind = state, state["case"]["kind"]
    if kind == "layer":
        layer = s["layer"]
        if not s["case"]["train"]:
            with torch.no_grad():
                out = layer(*s["x"])
            return {"out": out, "indices": layer.last_indices}
        out = layer(*s["x"])
        return {"out": out, "indices": layer.last_indices, "grads": torch.autograd.grad(out, s["x"], s["dout"])}
    if kind == "rope":
        c = s["case"]
        out, idx = PKG.lighthouse_layer_rope(s["x"], s["freqs"], c["H"], c["L"], c["p"], c["k"], strict=False,
                                             seq_major=True)
        return {"out": out, "indices": idx, "grads": torch.autograd.grad(out, s["x"], s["dout"])}
    if kind == "dense":
        out = s["attention"](*s["x"])
        return {"out": out, "grads": torch.autograd.grad(out, s["x"], s["dout"])}
    if kind in ("gla", "dilated"):
        with torch.no_grad():
            return s["scorer"](*s["x"], s["gk"]) if kind == "gla" else s["scorer"](*s["x"])
    if kind == "block":
        out = s["block"](s["x"], s["freqs"])
        return {"out": out, "grads": torch.autograd.grad(out, [s["x"]] + s["params"], s["dout"])}
    logits = s["model"](s["tokens"])
    loss = F.cross_entropy(logits.flatten(0, 1).float(), s["labels"].flatten(0, 1))
    return {"logits": logits, "loss": loss, "grads": torch.autograd.grad(loss, s["params"])}


# ---------------------------------------------------------------------------
# the same results in float64
# ---------------------------------------------------------------------------
def _network(s, x):
    """Descending 128-wide bitonic network on rows of s, payload x, strict exchanges."""
    i = torch.arange(128, device=s.device)
    k = 2
    while k <= 128:
        j = k // 2
        while j:
            other = i ^ j
            keep_max = ((i & j) == 0) == ((i & k) == 0)
            so, xo = s[:, other], x[:, other]
            take = torch.where(keep_max, s < so, s > so)
            s, x = torch.where(take, so, s), torch.where(take, xo, x)
            j //= 2
        k *= 2
    return s, x


def _select(sqk, skq, S, L, p, k):
    """Selected pyramid rows [R, n] in causal order, R = batch * heads, from pyramid scores
    [R, S_tot]: per tile and level the 64 best by qk, then the 64 best of the rest by kq,
    whose children are the next level's candidates (src/lighthouse_selection_cuda.py)."""
    lens = [S // p ** l for l in range(L)]
    offs = [sum(lens[:l]) for l in range(L)]
    R, tiles = sqk.shape[0], k // 128
    ncc = lens[-1] // tiles
    dev = sqk.device
    first = torch.arange(tiles, device=dev).repeat(R)[:, None] * ncc     # [R * tiles, 1]
    row = torch.arange(R, device=dev).repeat_interleave(tiles)[:, None]
    nodes, keys = [], []
    parent = None
    for level in range(L - 1, -1, -1):
        if parent is None:
            cand = first + torch.arange(ncc, device=dev)
        else:
            kids = parent[..., None] * p + torch.arange(p, device=dev)
            cand = torch.where(parent[..., None] >= 0, kids, -1).flatten(1)
        scale = p ** level << (L - 1)
        chosen = None
        if level:
            pad = -cand.shape[1] % 64
            c = F.pad(cand, (0, pad), value=-1)
            ok = c >= 0
            at = offs[level] + c.clamp_min(0)
            a = torch.where(ok, sqk[row, at], -1e6)
            b = torch.where(ok, skq[row, at], -1e6)
            slot = torch.where(ok, torch.arange(c.shape[1], device=dev).expand_as(c), -1)
            none_s = torch.full((c.shape[0], 64), -1e6, dtype=a.dtype, device=dev)
            none_x = torch.full_like(slot[:, :64], -1)
            tq, xq, tk, xk = none_s, none_x, none_s, none_x
            for o in range(0, c.shape[1], 64):
                s, x = _network(torch.cat([tq, a[:, o:o + 64]], 1), torch.cat([xq, slot[:, o:o + 64]], 1))
                tq, xq, rest = s[:, :64], x[:, :64], x[:, 64:]
                bs = torch.where(rest >= 0, b.gather(1, rest.clamp_min(0)), -1e6)
                s, x = _network(torch.cat([tk, bs], 1), torch.cat([xk, rest], 1))
                tk, xk = s[:, :64], x[:, :64]
            sel = torch.cat([xq, xk], 1)
            parent = torch.where(sel >= 0, c.gather(1, sel.clamp_min(0)), -1)
            chosen = torch.zeros(c.shape[0], c.shape[1] + 1, dtype=torch.bool, device=dev)
            chosen.scatter_(1, torch.where(sel >= 0, sel, c.shape[1]), True)
            chosen = chosen[:, :cand.shape[1]]
        key = cand * scale
        if chosen is not None:
            key = torch.where(chosen, (cand + 1) * scale - (1 << (L - 1 - level)), key)
        nodes.append(offs[level] + cand)
        keys.append(torch.where(cand >= 0, key, 1 << 62))
    nodes, keys = torch.cat(nodes, 1), torch.cat(keys, 1)
    keep = (keys < 1 << 62).sum(1).max()  # the same for every tile
    order = keys.argsort(dim=1)[:, :keep]
    return nodes.gather(1, order).view(R, -1)


def _pool(x, L, p, how):
    """Pyramid levels of x [R, S, ...] over dim 1, base first, concatenated."""
    S = x.shape[1]
    out = [x]
    for l in range(1, L):
        n, c = S // p ** l, p ** l
        y = x[:, :n * c].unflatten(1, (n, c))
        out.append(y.mean(2) if how == "mean" else y.amax(2))
    return torch.cat(out, 1)


def _fan(idx, S, L, p):
    """(level span first, last + 1) of the base rows that each selected row is added to."""
    lens = [S // p ** l for l in range(L)]
    first, span = torch.zeros_like(idx), torch.ones_like(idx)
    off = 0
    for l in range(L):
        at = (idx >= off) & (idx < off + lens[l])
        c = p ** l
        first = torch.where(at, (idx - off + 1) * c - 1, first)
        span = torch.where(at, c, span)
        off += lens[l]
    return first, (first + span).clamp_max(S)


def _attention(q, k, v, do):
    """Causal attention of one head [n, D] in float64: o, and with do its gradients."""
    n, scale = q.shape[0], q.shape[1] ** -0.5
    o = torch.empty_like(v)
    g = [torch.zeros_like(q) for _ in range(3)] if do is not None else None
    for a in range(0, n, 2048):
        b = min(n, a + 2048)
        s = (q[a:b] @ k[:b].t()) * scale
        s.masked_fill_(torch.arange(b, device=q.device) > torch.arange(a, b, device=q.device)[:, None], -math.inf)
        pr = torch.softmax(s, 1)
        o[a:b] = pr @ v[:b]
        if do is not None:
            g[2][:b] += pr.t() @ do[a:b]
            dp = do[a:b] @ v[:b].t()
            ds = pr * (dp - (do[a:b] * o[a:b]).sum(1, keepdim=True)) * scale
            g[0][a:b] = ds @ k[:b]
            g[1][:b] += ds.t() @ q[a:b]
    return o, g


def _unpool(g, S, L, p):
    """Adjoint of _pool(mean) for one head: [S_tot, D] -> [S, D]."""
    out, off = g[:S].clone(), S
    for l in range(1, L):
        n, c = S // p ** l, p ** l
        out[:n * c] += g[off:off + n].repeat_interleave(c, 0) / c
        off += n
    return out


def _exact_layer(x, norms, dout, S, L, p, topk):
    """x: q, k, v [B, S, H, D] in float64, norms: the 16-bit q and k base scores [B, S, H]."""
    B, _, H, D = x[0].shape
    heads = [t.transpose(1, 2).reshape(B * H, S, D) for t in x]
    sc = [_pool(t.transpose(1, 2).reshape(B * H, S).double(), L, p, "max") for t in norms]
    idx = _select(sc[0], sc[1], S, L, p, topk)
    out = torch.empty(B * H, S, D, dtype=torch.float64, device=x[0].device)
    grads = [torch.empty_like(out) for _ in range(3)] if dout is not None else None
    for r in range(B * H):
        cat = [_pool(t[r:r + 1], L, p, "mean")[0] for t in heads]
        first, stop = _fan(idx[r], S, L, p)
        keep = stop > first
        step = torch.zeros(S + 1, D, dtype=torch.float64, device=out.device)
        do = None
        if dout is not None:  # the adjoint of the fan-out: sums over each row's span
            run_sum = F.pad(dout.reshape(B * H, S, D)[r].double().cumsum(0), (0, 0, 1, 0))
            do = torch.where(keep[:, None], run_sum[stop.clamp_min(0)] - run_sum[first.clamp_max(S)], 0.0)
        o, g = _attention(*(c[idx[r]] for c in cat), do)
        step.index_add_(0, first[keep], o[keep])
        step.index_add_(0, stop[keep], -o[keep])
        out[r] = step.cumsum(0)[:S]
        for i in range(3 if g else 0):
            full = torch.zeros_like(cat[0]).index_add_(0, idx[r], g[i])
            grads[i][r] = _unpool(full, S, L, p)
    ret = {"out": out.view(B, H, S, D), "indices": idx.view(B, H, -1).int()}
    if grads:
        ret["grads"] = [g.view(B, H, S, D).transpose(1, 2) for g in grads]
    return ret


def _rotate(x, freqs, sign=1.0):
    """Rotation of adjacent pairs of x [B, S, H, D] by its position's angle, in float64."""
    f = freqs.double()
    f = torch.complex(f[..., 0], sign * f[..., 1])[None, :x.shape[1], None]
    return torch.view_as_real(torch.view_as_complex(x.double().unflatten(-1, (-1, 2)).contiguous()) * f).flatten(-2)


def _virtual(x):
    """[B, S, H, D] -> [B * DIL * H, S / DIL, D], the dilated view."""
    b, s, h, d = x.shape
    return x.reshape(b, s // DIL, DIL * h, d).transpose(1, 2).reshape(b * DIL * h, s // DIL, d)


def _real(scores, B, H):
    """[B * DIL * H, S / DIL] -> [B * H, S]."""
    return scores.view(B, DIL, H, -1).permute(0, 2, 3, 1).reshape(B * H, -1)


def _exact_scorer(s):
    c, kind = s["case"], s["case"]["kind"]
    B, S, H, D = s["x"][0].shape
    q, k, v = (_virtual(x.double()) for x in s["x"])
    scale = D ** -0.5
    scores = []
    if kind == "gla":
        G = _virtual(s["gk"].double()[..., None])[..., 0].cumsum(1)
    for a, b in ((q, k), (k, q)):
        norms = torch.empty(a.shape[:2], dtype=torch.float64, device=a.device)
        for r in range(a.shape[0]):
            if kind == "dilated":
                o = _attention(a[r], b[r], v[r], None)[0]
                norms[r] = o.norm(dim=1)
                continue
            for lo in range(0, a.shape[1], 2048):
                hi = min(a.shape[1], lo + 2048)
                w = (a[r, lo:hi] @ b[r, :hi].t()) * scale
                gate = G[r, lo:hi, None] - G[r, None, :hi]
                future = torch.arange(hi, device=w.device) > torch.arange(lo, hi, device=w.device)[:, None]
                w = w * gate.masked_fill(future, -math.inf).exp()
                norms[r, lo:hi] = (w @ v[r, :hi]).norm(dim=1)
        scores.append(_pool(_real(norms, B, H), c["L"], c["p"], "max").view(B, H, -1))
    cats = [_pool(x.double(), c["L"], c["p"], "mean").transpose(1, 2) for x in s["x"]]
    return (*scores, *cats)


def _exact_model(s):
    """The dense Llama3 of the model's bf16 weights in float64, with autograd."""
    m = s["model"]
    args = m.model_args
    H = args.n_heads
    w = {n: t.detach().double().requires_grad_() for n, t in m.named_parameters()}

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + args.norm_eps) * w[name]

    freqs = torch.view_as_real(m.freqs_cis)
    h = w["tok_embeddings.weight"][s["tokens"]]
    B, S, dim = h.shape
    causal = torch.ones(S, S, dtype=torch.bool, device=h.device).triu(1)
    for l in range(args.n_layers):
        pre = f"layers.{l}."
        y = norm(h, pre + "attention_norm.weight")
        q, k, v = ((y @ w[pre + f"attention.w{n}.weight"].t()).view(B, S, H, -1) for n in "qkv")
        q, k, v = (t.transpose(1, 2).contiguous() for t in (_rotate(q, freqs), _rotate(k, freqs), v))
        a = (q @ k.transpose(2, 3).contiguous()) * (dim // H) ** -0.5
        o = torch.softmax(a.masked_fill(causal, -math.inf), -1) @ v
        h = h + o.transpose(1, 2).reshape(B, S, dim) @ w[pre + "attention.wo.weight"].t()
        y = norm(h, pre + "ffn_norm.weight")
        y = F.silu(y @ w[pre + "feed_forward.w1.weight"].t()) * (y @ w[pre + "feed_forward.w3.weight"].t())
        h = h + y @ w[pre + "feed_forward.w2.weight"].t()
    logits = norm(h, "norm.weight") @ w["output.weight"].t()
    loss = F.cross_entropy(logits.flatten(0, 1), s["labels"].flatten(0, 1))
    return {"logits": logits.detach(), "loss": loss.detach(), "grads": torch.autograd.grad(loss, list(w.values()))}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "block":
        return None  # its selection hangs on activations rounded to 16 bits: no 64-bit value
    s = prepare(case, seed)
    if kind == "model":
        return _exact_model(s)
    if kind in ("gla", "dilated"):
        return _exact_scorer(s)
    if kind == "rope":
        q, k, v = (t.detach().unflatten(-1, (-1, 128)) for t in s["x"].chunk(3, -1))
        rot = [_rotate(t, s["freqs"]) for t in (q, k)]
        norms = [t.to(torch.bfloat16).double().norm(dim=-1).to(torch.bfloat16) for t in rot]
        r = _exact_layer([*rot, v.double()], norms, s["dout"], c["S"], c["L"], c["p"], c["k"])
        dq, dk, dv = r["grads"]
        r["grads"] = [torch.cat([_rotate(dq, s["freqs"], -1.0), _rotate(dk, s["freqs"], -1.0), dv], 2).flatten(2)]
        return r
    xs = [x.detach() for x in s["x"]]
    if kind == "layer":
        norms = [x.double().norm(dim=-1).to(x.dtype) for x in xs[:2]]
        return _exact_layer([x.double() for x in xs], norms, s["dout"], c["S"], c["L"], c["p"], c["k"])
    out, grads = [], [[], [], []]
    shape = xs[0].shape
    heads = [x.double().reshape(-1, *shape[2:]) for x in xs]
    for r in range(heads[0].shape[0]):
        o, g = _attention(*(h[r] for h in heads), s["dout"].double().reshape(-1, *shape[2:])[r])
        out.append(o)
        for i in range(3):
            grads[i].append(g[i])
    return {"out": torch.stack(out).view(shape), "grads": [torch.stack(g).view(shape) for g in grads]}
