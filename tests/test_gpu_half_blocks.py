"""Half blocks of the query-stationary attention kernels (128 queries to a
workgroup of four waves; lh_attn.hip, half_blocks): forward, dQ and the unchanged
dK/dV against fp32 attention, at sizes around the 64-row tiles and the 128-row
blocks, for few and for many heads; and bit for bit against whole blocks, so that
a sequence has the same results alone and in a batch."""
import ctypes

import pytest
import torch

from conftest import assert_close
from oracle import lh_oracle as O

pytestmark = pytest.mark.gpu


def _inputs(n, H, dtype, dev, gathered):
    g = torch.Generator().manual_seed(n + H)
    xs = [torch.randn(1, n, H, 128, generator=g).to(dtype) for _ in range(3)]
    idx = torch.stack([torch.randperm(n, generator=g) for _ in range(H)])[None].int() if gathered else None
    do = torch.randn(1, H, n, 128, generator=g).to(dtype)
    return [x.to(dev) for x in xs], idx.to(dev) if gathered else None, do.to(dev)


# 65: two tiles; 127, 128, 129: one block and its edge; 193: a block and a half;
# 1000, 4608: the layer's short lengths
@pytest.mark.parametrize("n,H,dtype,gathered", [
    (65, 2, torch.bfloat16, True), (127, 1, torch.bfloat16, False), (128, 2, torch.float16, True),
    (129, 2, torch.bfloat16, True), (193, 3, torch.float16, False), (1000, 2, torch.bfloat16, True),
    (4608, 8, torch.bfloat16, True), (4780, 12, torch.float16, False),
    # either side of the rule's line of two blocks per CU (256): 384 and 564 half blocks
    (744, 64, torch.bfloat16, False), (6000, 12, torch.float16, True)])
def test_half_blocks(pkg, dev, n, H, dtype, gathered):
    N = pkg._native
    print(f"half blocks n={n} H={H} {dtype} gathered={gathered}", flush=True)
    xs, idx, do = _inputs(n, H, dtype, dev, gathered)
    st = xs[0].stride()[:3]
    rows = N.Rows(*xs, st, *xs, st, split=n) if gathered else N.Rows(*xs, st)
    o, lse = N.attn_fwd(rows, idx, 1, H, n, shaped=True)
    delta = (do.float() * o.float()).sum(-1)
    grads = N.attn_bwd(rows, idx, 1, H, n, do, lse, delta, shaped=True)
    o1, lse1 = N.attn_fwd(rows, idx, 1, H, n)
    assert_close(lse, lse1, "lse against whole blocks", max_abs=2e-3, rel_l2=1e-4)  # row sums of bf16 P
    heads = range(H) if n < 2000 else (0, H - 1)
    for h in heads:
        sel = idx[0, h].long().cpu() if gathered else torch.arange(n)
        q, k, v = (x[0, :, h].float().cpu()[sel].requires_grad_() for x in xs)
        ref = O.sdpa_causal(q[None, None], k[None, None], v[None, None])
        ref.backward(do[0, h].float().cpu()[None, None])
        assert_close(o[0, h], ref[0, 0], f"o head {h}")
        for name, got, r in zip(("dq", "dk", "dv"), grads, (q, k, v)):
            assert_close(got[0, h], r.grad, f"{name} head {h}")


def test_half_blocks_no_finite_score(pkg, dev):
    """Rows whose every visible score is -inf give zero and an LSE of -inf, as in whole blocks."""
    N = pkg._native
    n, H = 300, 2
    xs, _, _ = _inputs(n, H, torch.bfloat16, dev, False)
    xs[0][0, :3] = 3e38
    xs[1][0, :3] = -3e38
    rows = N.Rows(*xs, xs[0].stride()[:3])
    o, lse = N.attn_fwd(rows, None, 1, H, n, shaped=True)
    o1, lse1 = N.attn_fwd(rows, None, 1, H, n)
    assert torch.equal(lse[:, :, :3], lse1[:, :, :3]) and bool((lse[:, :, :3] == -float("inf")).all())
    assert torch.equal(o[:, :, :3], o1[:, :, :3]) and not bool(o[:, :, :3].any())


def _calls(pkg, xs, idx, do, n, H, D, shaped):
    N = pkg._native
    st = xs[0].stride()[:3]
    rows = N.Rows(*xs, st, *xs, st, split=n) if idx is not None else N.Rows(*xs, st)
    o, lse = N.attn_fwd(rows, idx, xs[0].shape[0], H, n, D, shaped=shaped)
    delta = (do.float() * o.float()).sum(-1)
    return (o, lse) + tuple(N.attn_bwd(rows, idx, xs[0].shape[0], H, n, do, lse, delta, D, shaped=shaped))


# 129 to 300: two and three half blocks, the last one nearly empty or full, beside one
# and two whole blocks; 1500 and 4780: more half blocks than CUs; 8192: exactly two to
# a CU (256); D: both narrow layouts, with zero tails (40, 72) and without
@pytest.mark.parametrize("n,H,D,dtype,gathered", [
    (129, 3, 128, torch.bfloat16, True), (200, 2, 64, torch.float16, True), (256, 2, 40, torch.bfloat16, False),
    (257, 3, 72, torch.bfloat16, True), (300, 2, 128, torch.float16, False), (1500, 36, 72, torch.bfloat16, True),
    (4780, 12, 128, torch.float16, True), (4608, 8, 40, torch.bfloat16, True), (8192, 8, 64, torch.bfloat16, False)])
@pytest.mark.parametrize("centred", [False, True])
def test_half_blocks_have_whole_blocks_bits(pkg, dev, n, H, D, dtype, gathered, centred):
    """centred: keys that share a large channel, so that dQ subtracts the key centre."""
    print(f"half blocks' bits n={n} H={H} D={D} {dtype} gathered={gathered} centred={centred}", flush=True)
    g = torch.Generator().manual_seed(n + H + D)
    xs = [torch.randn(1, n, H, D, generator=g).to(dtype).to(dev) for _ in range(3)]
    if centred:
        xs[1][..., 3] = 8.0
    idx = torch.stack([torch.randperm(n, generator=g) for _ in range(H)])[None].int().to(dev) if gathered else None
    do = torch.randn(1, H, n, D, generator=g).to(dtype).to(dev)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), _calls(pkg, xs, idx, do, n, H, D, True),
                          _calls(pkg, xs, idx, do, n, H, D, False)):
        assert torch.equal(a, b), name


class _Dim3(ctypes.Structure):
    _fields_ = [(c, ctypes.c_uint) for c in "xyz"]


class _KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def _launches(pkg, f):
    """(workgroups, threads) of every kernel that f launches, from a captured graph."""
    hip = pkg._native.lib()  # the library's handle finds the runtime that it is linked with
    f()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        f()
    raw, n = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        kind, p = ctypes.c_int(), _KernelNode()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value == 0:  # a kernel
            assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
            out.append((p.grid.x, p.block.x))
    return out


def test_which_launches_take_half_blocks(pkg, dev):
    """Four waves to a workgroup and one block of 128 rows each, up to two of them per
    CU; eight waves beyond, for one block of 128 rows, and in calls without the flag."""
    N = pkg._native
    H = 8
    most = 2 * torch.cuda.get_device_properties(dev).multi_processor_count // H  # half blocks per head
    for n, shaped, half in ((129, True, True), (most * 128, True, True), (128, True, False),
                            (most * 128 + 1, True, False), (129, False, False)):
        xs, _, do = _inputs(n, H, torch.bfloat16, dev, False)
        rows = N.Rows(*xs, xs[0].stride()[:3])
        lse = torch.zeros(1, H, n, device=dev)
        for name, f in (("forward", lambda: N.attn_fwd(rows, None, 1, H, n, shaped=shaped)),
                        ("dQ", lambda: N.attn_bwd_dq(rows, None, 1, H, n, do, lse, lse, shaped=shaped))):
            got = _launches(pkg, f)
            assert len(got) == 1 and got[0][1] == (256 if half else 512), f"{name}, n={n}, shaped={shaped}: {got}"
            if half:
                assert got[0][0] == H * -(-n // 128), f"{name}, n={n}: {got}"


@pytest.mark.parametrize("D", [128, 64])
def test_public_calls_do_not_depend_on_the_batch(pkg, dev, D):
    """A sequence's results and gradients alone (half blocks) and as one of four (whole blocks)."""
    B, H, S, k = 4, 8, 8192, 512
    print(f"batch independence D={D}", flush=True)
    g = torch.Generator().manual_seed(D)
    xs = [torch.randn(B, S, H, D, generator=g).bfloat16().to(dev) for _ in range(3)]
    dout = torch.randn(B, H, S, D, generator=g).bfloat16().to(dev)

    def run(f, ins, up):
        ins = [x.detach().requires_grad_() for x in ins]
        out = f(*ins)
        return (out,) + torch.autograd.grad(out, ins, up)

    def layer(*x):
        return pkg.lighthouse_layer(*x, 3, 4, k)[0]

    def dense(*x):
        return pkg.dense_attention.dense_causal_attention(*(t[:, :4608].transpose(1, 2) for t in x))

    freqs = torch.randn(S, 64, 2, generator=g).to(dev)

    def rope(x):
        return pkg.lighthouse_layer_rope(x, freqs, H, 3, 4, k)[0]

    calls = [(layer, xs, dout), (dense, xs, dout[:, :, :4608])]
    if D == 128:
        calls.append((rope, [torch.cat([x.flatten(2) for x in xs], -1)], dout))
    for f, ins, up in calls:
        batch = run(f, ins, up)
        for b in (0, B - 1):
            alone = run(f, [x[b:b + 1] for x in ins], up[b:b + 1])
            for i, (x, y) in enumerate(zip(alone, batch)):
                assert torch.equal(x[0], y[b]), f"{f.__name__}: result {i} of sequence {b}"
