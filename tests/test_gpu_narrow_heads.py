"""Head dims below 128 on their own row width (lh_attn.hip, struct Head; the row
kernels' struct Lanes): both LDS layouts at their edges and with zero tails,
against fp32 attention, and the inputs that are copied first because the kernels
cannot read them in place."""
import pytest
import torch

from conftest import assert_close
from oracle import lh_oracle as O

pytestmark = pytest.mark.gpu


# 8, 40, 56: zero tails in 64-column rows (40: half a k-slice); 64: exact; 72, 88:
# zero tails in 96 columns (72: half a k-slice); 96: exact; 104: padded to 128.
# n = 300: whole query blocks of a low-level call, half blocks of the module's
@pytest.mark.parametrize("D", [8, 40, 56, 64, 72, 88, 96, 104])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_narrow(pkg, dev, D, dtype):
    N = pkg._native
    n, H = 300, 3
    print(f"dense D={D} {dtype}", flush=True)
    g = torch.Generator().manual_seed(D)
    xs = [torch.randn(2, n, H, D, generator=g).to(dtype) for _ in range(3)]
    do = torch.randn(2, H, n, D, generator=g).to(dtype)
    xg = [x.to(dev).transpose(1, 2).requires_grad_() for x in xs]
    out = pkg.dense_attention.dense_causal_attention(*xg)
    grads = torch.autograd.grad(out, xg, do.to(dev))
    xc = [x.float().transpose(1, 2).contiguous().requires_grad_() for x in xs]
    ref = O.sdpa_causal(*xc)
    ref.backward(do.float())
    assert_close(out, ref, f"D={D} out")
    for name, a, c in zip(("dq", "dk", "dv"), grads, xc):
        assert_close(a, c.grad, f"D={D} {name}")
    if N.padded_dim(D) == D:
        xd = [x.to(dev) for x in xs]
        rows = N.Rows(*xd, xd[0].stride()[:3])
        o, lse = N.attn_fwd(rows, None, 2, H, n, D)
        delta = (do.to(dev).float() * o.float()).sum(-1)
        got = (o,) + N.attn_bwd(rows, None, 2, H, n, do.to(dev), lse, delta, D)
        for name, a, r in zip(("o", "dq", "dk", "dv"), got, [ref] + [c.grad for c in xc]):
            assert_close(a, r, f"D={D} whole blocks {name}")


# 36 heads: more blocks than CUs, from queues; 32 and 8 heads: forward and dQ by plans,
# dK/dV from queues; so workgroups run several blocks one after the other.  40, 72: the
# zero tails of both layouts have to outlast a block; 64, 96: none
@pytest.mark.parametrize("D,H,n,gathered", [(40, 36, 4607, True), (72, 36, 4607, False), (40, 32, 4608, False),
                                            (72, 32, 4608, True), (72, 8, 9001, True), (64, 36, 4607, True),
                                            (96, 36, 4607, False)])
def test_persistent_launches_narrow(pkg, dev, D, H, n, gathered):
    """Every head as when it is computed alone, with one block per workgroup, over
    repeated launches, and the first head within tolerance of fp32 attention."""
    N = pkg._native
    print(f"persistent D={D} H={H} n={n} gathered={gathered}", flush=True)
    g = torch.Generator().manual_seed(D + H)
    xs = [torch.randn(1, n, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    idx = torch.stack([torch.randperm(n, generator=g) for _ in range(H)])[None].int().to(dev) if gathered else None
    do = torch.randn(1, H, n, D, generator=g).bfloat16().to(dev)

    def run(sl):
        part = [x[:, :, sl] for x in xs]
        st = part[0].stride()[:3]
        ix = idx[:, sl].contiguous() if gathered else None
        rows = N.Rows(*part, st, *part, st, split=n) if gathered else N.Rows(*part, st)
        h = part[0].shape[2]
        d = do[:, sl].contiguous()
        o, lse = N.attn_fwd(rows, ix, 1, h, n, D)
        return (o, lse) + tuple(N.attn_bwd(rows, ix, 1, h, n, d, lse, (d.float() * o.float()).sum(-1), D))

    names = ("o", "lse", "dq", "dk", "dv")
    got = run(slice(0, H))
    for _ in range(2):
        for name, a, b in zip(names, run(slice(0, H)), got):
            assert torch.equal(a, b), f"{name} differs between launches"
    for h in range(H):
        for name, a, b in zip(names, run(slice(h, h + 1)), got):
            assert torch.equal(a[:, 0], b[:, h]), f"{name} of head {h} differs from the head alone"
    sel = idx[0, 0].long().cpu() if gathered else torch.arange(n)
    q, k, v = (x[0, :, 0].float().cpu()[sel].requires_grad_() for x in xs)
    ref = O.sdpa_causal(q[None, None], k[None, None], v[None, None])
    ref.backward(do[0, 0].float().cpu()[None, None])
    for name, a, r in zip(("o", "dq", "dk", "dv"), (got[0],) + got[2:], (ref[0, 0], q.grad, k.grad, v.grad)):
        assert_close(a[0, 0], r, f"D={D} {name}")


@pytest.mark.parametrize("D,L,p,strict", [(64, 3, 4, True), (40, 2, 2, False), (96, 3, 2, False), (72, 4, 2, False)])
def test_row_kernels_narrow(pkg, dev, D, L, p, strict):
    """Pyramid, fan-out, its adjoint and the pyramid backward give the first D columns
    of what the zero-padded 128-wide rows give, bit for bit (the sums run over the same
    values in the same order; the norms and delta add zeros)."""
    N = pkg._native
    B, S, H, k = 2, 2048 if strict else 1999, 3, 128
    print(f"row kernels D={D} L={L} p={p}", flush=True)
    g = torch.Generator().manual_seed(D + L)
    xs = [torch.randn(B, S, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    wide = [torch.nn.functional.pad(x, (0, 128 - D)) for x in xs]
    a, b = N.pyramid_fwd(*xs, L, p), N.pyramid_fwd(*wide, L, p)
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y[..., :D])
    for x, y in zip(a[3:], b[3:]):  # norms: 16 lanes' tree ends with zeros where 8 lanes' ends
        assert torch.equal(x, y)
    idx, inv = N.select_topk(b[3], b[4], S, L, p, k, strict=strict)
    n = idx.shape[-1]
    att = torch.randn(B, H, n, D, generator=g).bfloat16().to(dev)
    attw = torch.nn.functional.pad(att, (0, 128 - D))
    assert torch.equal(N.scatter_fwd(att, inv, S, S, L, p), N.scatter_fwd(attw, inv, S, S, L, p)[..., :D])
    do = torch.randn(B, H, S, D, generator=g).bfloat16().to(dev)
    dow = torch.nn.functional.pad(do, (0, 128 - D))
    (d1, e1), (d2, e2) = N.scatter_bwd(do, idx, att, S, L, p), N.scatter_bwd(dow, idx, attw, S, L, p)
    assert torch.equal(d1, d2[..., :D])
    assert torch.equal(e1, e2)
    gs = [torch.randn(B, H, n, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    got = N.pyramid_bwd(*gs, inv, B, S, H, L, p, D)
    want = N.pyramid_bwd(*[torch.nn.functional.pad(x, (0, 128 - D)) for x in gs], inv, B, S, H, L, p, 128)
    for x, y in zip(got, want):
        assert torch.equal(x, y[..., :D])


def _off(x):
    """x at an address 2 bytes past a 16-byte boundary."""
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:]
    return buf.view(x.shape).copy_(x)


def test_narrow_inputs_that_are_copied(pkg, dev):
    """Strides that differ, a strided head dim, odd strides and odd addresses: accepted
    for head dims below 128 and equal to the contiguous call."""
    n, H, D, S = 200, 2, 64, 2048
    g = torch.Generator().manual_seed(1)
    q, k, v, do = (torch.randn(1, H, n, D, generator=g).bfloat16().to(dev) for _ in range(4))
    dense = pkg.dense_attention.dense_causal_attention

    def run(q, k, v, do):
        xs = [x.detach().requires_grad_() for x in (q, k, v)]
        o = dense(*xs)
        return (o,) + torch.autograd.grad(o, xs, do)

    want = run(q, k, v, do)
    odd = torch.empty(1, H, n, D + 1, dtype=q.dtype, device=dev)[..., :D]
    forms = [(q.transpose(1, 2).contiguous().transpose(1, 2), k, v, do), (_off(q), _off(k), _off(v), _off(do)),
             (q.transpose(2, 3).contiguous().transpose(2, 3), k, v, do.transpose(2, 3).contiguous().transpose(2, 3)),
             (odd.copy_(q), odd.clone().copy_(k), v, do)]
    for i, f in enumerate(forms):
        for name, x, y in zip(("o", "dq", "dk", "dv"), run(*f), want):
            assert torch.equal(x, y), f"form {i}: {name}"

    xs = [torch.randn(1, S, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    dl = torch.randn(1, H, S, D, generator=g).bfloat16().to(dev)

    def layer(xs, dl):
        xs = [x.detach().requires_grad_() for x in xs]
        o, idx = pkg.lighthouse_layer(*xs, 3, 4, 128)
        return (o, idx) + torch.autograd.grad(o, xs, dl)

    for x, y in zip(layer([_off(x) for x in xs], _off(dl)), layer(xs, dl)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("D", [64, 72, 104])
def test_narrow_inputs_whose_single_dims_have_strides_of_their_own(pkg, dev, D):
    """One sequence or one head cut out of a larger tensor keeps that tensor's stride in
    the dimension of one element: q, k, v then differ in strides that nobody reads."""
    S = 2048
    g = torch.Generator().manual_seed(D)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).bfloat16().to(dev)

    forms = {  # [B, S, H, D] each
        "k, v a prefix of longer ones": [rnd(1, S, 2, D), rnd(1, S + 64, 2, D)[:, :S], rnd(1, S + 64, 2, D)[:, :S]],
        "v out of a fused buffer": [rnd(1, S, 2, D), rnd(1, S, 2, D), rnd(1, 3, S, 2, D)[:, 2]],
        "one head, q head-major": [rnd(1, 1, S, D).transpose(1, 2), rnd(1, S, 1, D), rnd(1, S, 1, D)],
        "one head of a prefix": [rnd(1, S, 1, D), rnd(1, S + 64, 1, D)[:, :S], rnd(1, S + 64, 1, D)[:, :S]],
        "off a 16-byte boundary": [rnd(1, S, 2, D), rnd(1, 3 * S * 2 * D + 1)[:, 1:].view(1, 3, S, 2, D)[:, 1], rnd(1, S, 2, D)],
    }
    gk = torch.nn.functional.logsigmoid(rnd(1, S, 2))

    def sums(out):
        return sum(x.float().sum() for x in out[2:])

    calls = {"layer": lambda *x: pkg.lighthouse_layer(*x, 3, 4, 128)[0],
             "dilated layer": lambda *x: pkg.lighthouse_layer(*x, 3, 4, 128, dilation=4)[0],
             "gla layer": lambda *x: pkg.lighthouse_layer(*x, 3, 4, 128, dilation=4, gk=gk[..., :x[0].shape[2]])[0],
             "scorer": lambda *x: sums(pkg.DialatedLighthouseNormScorer(4, 3)(*x)),
             "dense": lambda *x: pkg.dense_attention.dense_causal_attention(*(t.transpose(1, 2) for t in x))}
    for form, xs in forms.items():
        for name, f in calls.items():
            print(f"D={D} {form}: {name}", flush=True)
            res = []
            for ins in (xs, [x.clone(memory_format=torch.contiguous_format) for x in xs]):
                leaves = [x.detach().requires_grad_() for x in ins]
                out = f(*leaves)
                res.append((out,) + torch.autograd.grad(out, leaves, torch.ones_like(out)))
            for a, b in zip(*res):
                assert torch.equal(a, b), f"{form}: {name}"


@pytest.mark.parametrize("D", [64, 72, 104])
def test_narrow_upstream_gradients_of_any_strides(pkg, dev, D):
    """Expanded gradients (a sum's, over all or over the sequence) and a strided head dim
    give the layer, dense attention and the fan-out what a contiguous copy gives them."""
    S, H, n = 2048, 2, 300
    g = torch.Generator().manual_seed(D)
    xs = [torch.randn(1, S, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    att = torch.randn(1, H, n, D, generator=g).bfloat16().to(dev)
    idx = torch.stack([torch.randperm(S + S // 4, generator=g)[:n] for _ in range(H)])[None].int().to(dev)
    calls = [(lambda *x: pkg.lighthouse_layer(*x, 3, 4, 128)[0], xs),
             (lambda *x: pkg.dense_attention.dense_causal_attention(*(t.transpose(1, 2) for t in x)), xs),
             (lambda a: pkg.scatter_to_base_sequence(a, idx, None, S, S, 2, 4), [att])]
    one = torch.randn(1, H, 1, D, generator=g).bfloat16().to(dev)
    ups = [torch.ones(1, dtype=torch.bfloat16, device=dev).expand(1, H, S, D), one.expand(1, H, S, D),
           one[:, :1].expand(1, H, S, D), torch.randn(1, H, D, S, generator=g).bfloat16().to(dev).transpose(2, 3)]
    for c, (f, ins) in enumerate(calls):
        for u, up in enumerate(ups):
            print(f"upstream D={D} call {c} form {u}", flush=True)
            res = []
            for d in (up, up.contiguous()):
                leaves = [x.clone().requires_grad_() for x in ins]
                res.append(torch.autograd.grad(f(*leaves), leaves, d))
            for a, b in zip(*res):
                assert torch.equal(a, b), f"call {c}, form {u}"


@pytest.mark.parametrize("D", [64, 104, 128])
def test_scorers_take_any_order(pkg, dev, D):
    """Rows stored with the sequence or the heads running fastest give the scorer modules
    what contiguous rows give them."""
    B, S, H = 2, 2048, 2
    g = torch.Generator().manual_seed(D)
    xs = [torch.randn(B, S, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    gk = torch.nn.functional.logsigmoid(torch.randn(B, S, H, generator=g).to(dev)) / 16
    orders = {"sequence fastest": lambda x: x.permute(0, 2, 3, 1).contiguous().permute(0, 3, 1, 2),
              "channels last": lambda x: x.contiguous(memory_format=torch.channels_last),
              "heads fastest": lambda x: x.transpose(2, 3).contiguous().transpose(2, 3)}
    scorers = {"gla": lambda *x: pkg.DilatedLighthouseGLAScorer(D, 4, 4, 3)(*x, gk),
               "dilated": pkg.DilatedLighthouseScorer(None, 4, 4, 3), "norm": pkg.DialatedLighthouseNormScorer(4, 3)}
    for name, f in scorers.items():
        want = f(*xs)
        for order, store in orders.items():
            print(f"D={D} {name} {order}", flush=True)
            for i, (a, b) in enumerate(zip(f(*[store(x) for x in xs]), want)):
                assert torch.equal(a, b), f"{name}, {order}: output {i}"


@pytest.mark.parametrize("D", [4, 20, 36, 97, 100, 127])
def test_scorer_modules_any_width(pkg, dev, D):
    """The scorer modules and the layer composed from one take head dims that are no
    multiple of 8: the same rows as with columns of zeros, scores and attention with the
    scale of the D columns."""
    B, S, H, L, p, k = 1, 2048, 2, 3, 4, 128
    print(f"scorers D={D}", flush=True)
    g = torch.Generator().manual_seed(D)
    xs = [torch.randn(B, S, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    gk = torch.nn.functional.logsigmoid(torch.randn(B, S, H, generator=g).to(dev)) / 16

    class Scorer(pkg.DialatedLighthouseNormScorer):  # not the class itself: the composed path
        pass

    def reference(dil, gate=None):
        """Scores by the 128-wide kernels on padded rows."""
        wide = [torch.nn.functional.pad(x, (0, 128 - D)) for x in xs]
        S_tot = pkg._native.pyramid_total(S, L, p)
        if gate is not None:
            base = pkg._native.gla_scores(*wide, gate, dil, S_tot, D ** -0.5)
        else:
            base = pkg._native.dilated_scores(*wide, dil, S_tot, D ** -0.5) if dil else None
        return pkg._native.pyramid_fwd(*wide, L, p, scores=base)

    for name, out, (pq, pk, pv, sqk, skq) in (
            ("norm", Scorer(p, L)(*xs), reference(0)),
            ("dilated", pkg.DilatedLighthouseScorer(None, 4, p, L)(*xs), reference(4)),
            ("gla", pkg.DilatedLighthouseGLAScorer(D, 4, p, L)(*xs, gk), reference(4, gk))):
        for got, want in zip(out[:2], (sqk, skq)):
            assert_close(got, want, f"{name} scores", max_abs=4e-3, rel_l2=4e-3)  # bf16 scores
        for got, x, pool in zip(out[2:], xs, (pq, pk, pv)):
            assert torch.equal(got[:, :, :S], x.transpose(1, 2)) and torch.equal(got[:, :, S:],
                                                                                 pool[..., :D].transpose(1, 2)), name
    layer = pkg.LighthouseLocal(None, Scorer(p, L), L, p, k)
    leaves = [x.clone().requires_grad_() for x in xs]
    out = layer(*leaves)
    do = torch.randn(B, H, S, D, generator=g).bfloat16().to(dev)
    out.backward(do)
    xc = [x.float().cpu().requires_grad_() for x in xs]
    ref, _ = O.lighthouse_layer(*xc, L, p, k, indices=layer.last_indices.cpu().numpy())
    ref.backward(do.float().cpu())
    assert_close(out, ref, f"D={D} out")
    for name, x, c in zip("qkv", leaves, xc):
        assert_close(x.grad, c.grad, f"D={D} d{name}")


def test_fan_out_any_width(pkg, dev):
    """scatter_to_base_sequence takes row widths that are no multiple of 8."""
    S, H, L, p = 512, 2, 2, 2
    att = torch.randn(1, H, 300, 36, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev).requires_grad_()
    idx = torch.stack([torch.randperm(S + S // p)[:300] for _ in range(H)])[None].int().to(dev)
    out = pkg.scatter_to_base_sequence(att, idx, None, S, S, L, p)
    ref = O.scatter_fwd(att.detach().float().cpu(), idx.cpu().long(), S, L, p)
    assert_close(out, ref, "fan-out of 36 columns")
    out.backward(torch.ones_like(out))
    assert att.grad.shape == att.shape


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (72, torch.float16), (64, torch.bfloat16), (8, torch.bfloat16)])
def test_attn_delta(pkg, dev, D, dtype):
    """Row sums of dO * O and the contiguous dO, for contiguous, transposed, expanded
    and unaligned upstream gradients; 33 rows: two blocks, the second nearly empty."""
    N = pkg._native
    B, H, n = 2, 3, 33
    g = torch.Generator().manual_seed(D)
    o = torch.randn(B, H, n, D, generator=g).to(dtype).to(dev)
    do = torch.randn(B, n, H, D, generator=g).to(dtype).to(dev)
    forms = [do.transpose(1, 2).contiguous(), do.transpose(1, 2), do[:1, :, :1].expand(B, n, H, D).transpose(1, 2)]
    if D < 128:
        forms.append(_off(do.transpose(1, 2).contiguous()))
    for i, f in enumerate(forms):
        rows, delta = N.attn_delta(f, o)
        assert rows.is_contiguous() and torch.equal(rows, f), f"form {i}"
        ref = (f.double() * o.double()).sum(-1)
        # fp32 sums of D products of 16-bit values: D roundings at most
        bound = D * 2.0 ** -24 * (f.double() * o.double()).abs().sum(-1)
        assert bool(((delta.double() - ref).abs() <= bound).all()), f"form {i}"
        # the order of the sum: four products after each other, then pairs of neighbours
        p = torch.nn.functional.pad(f.float() * o.float(), (0, 128 - D)).unflatten(-1, (32, 4))
        p = ((p[..., 0] + p[..., 1]) + p[..., 2]) + p[..., 3]
        while p.shape[-1] > 1:
            p = p[..., 0::2] + p[..., 1::2]
        assert torch.equal(delta, p[..., 0]), f"form {i}: another order"


@pytest.mark.parametrize("D,S,L,p,dtype", [(128, 1000, 3, 4, torch.bfloat16), (72, 257, 2, 2, torch.float16),
                                           (64, 1030, 4, 2, torch.bfloat16), (128, 96, 1, 2, torch.float16)])
@pytest.mark.parametrize("given", [False, True])
def test_pyramid_cat(pkg, dev, D, S, L, p, dtype, given):
    """The one-pass scorer outputs: base rows, pooled rows and scores are those of
    pyramid_fwd, with S not a multiple of the spans or of the lanes' score runs."""
    N = pkg._native
    B, H = 2, 3
    g = torch.Generator().manual_seed(S)
    xs = [torch.randn(B, S, H, D, generator=g).to(dtype).to(dev) for _ in range(3)]
    S_tot = N.pyramid_total(S, L, p)
    base = [torch.rand(B, H, S, generator=g).to(dtype).float().to(dev) for _ in range(2)]

    def scores():
        if not given:
            return None
        buf = [torch.full((B, H, S_tot), -1.0, device=dev) for _ in range(2)]
        for x, y in zip(buf, base):
            x[..., :S] = y
        return buf

    want = N.pyramid_fwd(*xs, L, p, scores=scores())
    sqk, skq, *cats = N.pyramid_cat(*xs, L, p, scores())
    for c, x, pool in zip(cats, xs, want[:3]):
        assert torch.equal(c[:, :S], x) and torch.equal(c[:, S:], pool)
    assert torch.equal(sqk, want[3].to(dtype)) and torch.equal(skq, want[4].to(dtype))
