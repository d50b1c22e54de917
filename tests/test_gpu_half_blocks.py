"""Half blocks of the query-stationary attention kernels (128 queries per
workgroup, the key tiles shared by its two halves; lh_attn.hip, fwd_half_block):
forward, dQ and the unchanged dK/dV against fp32 attention, at sizes around the
64-row tiles and the 128-row blocks, for few and for many heads."""
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


# 65: two tiles, one per half; 127, 128, 129: one block and its edge; 193: a third
# tile, so one half runs a step more; 1000, 4608: the layer's short lengths
@pytest.mark.parametrize("n,H,dtype,gathered", [
    (65, 2, torch.bfloat16, True), (127, 1, torch.bfloat16, False), (128, 2, torch.float16, True),
    (129, 2, torch.bfloat16, True), (193, 3, torch.float16, False), (1000, 2, torch.bfloat16, True),
    (4608, 8, torch.bfloat16, True), (4780, 12, torch.float16, False),
    # either side of the rule's bound by shared CUs: 64 heads take whole blocks, 12 of 6000 half blocks
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
