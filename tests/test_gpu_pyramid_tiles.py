"""The pyramid forward's two forms (lh_pyramid.hip): few spans are taken tile by
tile with a token per group, many are walked span by span.  Both sum a node's
tokens in their order, so one head alone (tiles) has the bits it has among many
(the walk), with and without the rotation, at ragged lengths."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# spans of 16 (a tile), 64 (four rounds of a tile), 4 and 2 (many per tile), no
# pooling; lengths with an incomplete last tile, span and pooled node
@pytest.mark.parametrize("S,L,p,D,dtype", [(2048, 3, 4, 128, torch.bfloat16), (1031, 3, 4, 128, torch.float16),
                                           (4099, 4, 4, 64, torch.bfloat16), (1001, 2, 4, 72, torch.bfloat16),
                                           (517, 2, 2, 128, torch.float16), (640, 1, 2, 128, torch.bfloat16)])
def test_tiles_equal_walk(pkg, dev, S, L, p, D, dtype):
    N = pkg._native
    span = p ** (L - 1)
    H = -(-2 * 256 * (16 if D > 64 else 32) // 4 // (S // span)) + 1  # more spans than a wave per CU holds
    g = torch.Generator().manual_seed(S)
    xs = [torch.randn(1, S, H, D, generator=g).to(dtype).to(dev) for _ in range(3)]
    walk = N.pyramid_fwd(*xs, L, p)
    for h in (0, H - 1):
        alone = N.pyramid_fwd(*[x[:, :, h:h + 1].contiguous() for x in xs], L, p)
        for x, y in zip(alone[:3], walk[:3]):
            assert torch.equal(x[:, :, 0], y[:, :, h])
        for x, y in zip(alone[3:], walk[3:]):
            assert torch.equal(x[:, 0], y[:, h])


@pytest.mark.parametrize("S,L,p", [(1031, 3, 4), (2050, 2, 2)])
def test_tiles_equal_walk_rope(pkg, dev, S, L, p):
    N = pkg._native
    H, D = -(-5 * 1024 * 4 // (S // p ** (L - 1))) + 1, 128
    g = torch.Generator().manual_seed(S)
    x = torch.randn(1, S, 3, H, D, generator=g).bfloat16().to(dev)
    fr = torch.randn(S, D // 2, 2, generator=g).to(dev)
    walk = N.rope_pyramid_fwd(x.view(1, S, 3 * H * D), fr, H, L, p)
    for h in (0, H - 1):
        alone = N.rope_pyramid_fwd(x[:, :, :, h].contiguous().view(1, S, 3 * D), fr, 1, L, p)
        assert torch.equal(alone[0][..., :2 * D], walk[0].view(1, S, 3, H, D)[:, :, :2, h].reshape(1, S, 2 * D))
        for a, b in zip(alone[1:4], walk[1:4]):
            assert torch.equal(a[:, :, 0], b[:, :, h])
        for a, b in zip(alone[4:], walk[4:]):
            assert torch.equal(a[:, 0], b[:, h])
