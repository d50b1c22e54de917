"""Tracing of the layer's custom ops at more than one sequence length, on the CPU: dynamo
makes the length symbolic when a compiled function meets a second one, and the fake
implementations have to take it."""
import pytest
import torch
from torch._dynamo.source import ConstantSource
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import DimDynamic, ShapeEnv, StatelessSymbolicContext

L, P, K = 3, 4, 128


def _layer(pkg, S):
    xs = [torch.empty(1, S, 2, 64, dtype=torch.bfloat16) for _ in range(3)]
    return xs, lambda *x: pkg.lighthouse_layer(*x, L, P, K, strict=False)


def _rope(pkg, S):
    xs = [torch.empty(1, S, 3 * 2 * 128, dtype=torch.bfloat16), torch.empty(S, 64, 2)]
    return xs, lambda x, f: pkg.lighthouse_layer_rope(x, f, 2, L, P, K, strict=False)


def _trace_only(seen):
    """A backend that records the traced graph's output shapes and runs nothing."""
    def backend(gm, _inputs):
        out = [n for n in gm.graph.nodes if n.op == "output"][0].args[0]
        vals = [n.meta["example_value"] for n in out]
        seen.append([tuple(int(s) for s in v.shape) for v in vals])
        return lambda *a: tuple(torch.empty(s, dtype=v.dtype) for s, v in zip(seen[-1], vals))
    return backend


@pytest.mark.parametrize("dynamic", [None, True])
@pytest.mark.parametrize("make", [_layer, _rope])
def test_compiled_at_several_lengths(pkg, make, dynamic):
    torch._dynamo.reset()
    seen = []
    call = make(pkg, 2048)[1]
    f = torch.compile(lambda *x: call(*x), backend=_trace_only(seen), fullgraph=True, dynamic=dynamic)
    for S in (2048, 4096, 3000):
        f(*make(pkg, S)[0])
        D = 64 if make is _layer else 128
        assert seen[-1][:2] == [(1, 2, S, D), (1, 2, pkg._native.geometry(S, L, P, K, False)[3])]
    torch._dynamo.reset()


@pytest.mark.parametrize("make", [_layer, _rope])
def test_fake_ops_with_a_symbolic_length(pkg, make):
    env = ShapeEnv()
    with FakeTensorMode(shape_env=env, allow_non_fake_inputs=True) as mode:
        real = make(pkg, 2048)[0]
        xs = []
        for i, x in enumerate(torch.empty(t.shape, dtype=t.dtype, device="meta") for t in real):
            dims = [DimDynamic.DYNAMIC if s == 2048 else DimDynamic.STATIC for s in x.shape]
            xs.append(mode.from_tensor(x, source=ConstantSource(f"x{i}"),
                                       symbolic_context=StatelessSymbolicContext(dynamic_sizes=dims)))
        ops = torch.ops.lighthouse_amd
        if make is _layer:
            out = ops.layer_fwd(*xs, L, P, K, "reference", False, 0, False, None, None)
        else:
            out = ops.rope_layer_fwd(*xs, 2, L, P, K, "reference", False, False)
    n = pkg._native.geometry(2048, L, P, K, False)[3]
    assert tuple(int(s) for s in out[1].shape) == (1, 2, n)


def test_cached_sizes(pkg):
    """The cache behind the sizes: plain ints hit it, and errors are raised every time."""
    N = pkg._native
    assert N.pyramid_total(1000, 3, 4) == sum(N.pyramid_lengths(1000, 3, 4)[0])
    for _ in range(2):
        with pytest.raises(AssertionError):
            N.geometry(1000, 3, 4, 128, True)
