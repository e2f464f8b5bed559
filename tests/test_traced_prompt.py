"""Calls that torch traces or transforms keep torch's own operations: a launch
by pointer would be missing from what they record."""
import pytest
import torch
from torch._subclasses import FakeTensorMode
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

import kitty  # noqa: F401


def test_recorders_and_transforms_are_seen():
    from kitty.kernels.ops import calls_followed
    seen = []

    def f(x):
        seen.append(calls_followed())
        return x * 2
    x = torch.ones(2, 3)
    f(x)
    with torch.no_grad(), torch.inference_mode(), torch.device("cpu"):      # none of these records calls
        f(x)
    assert seen == [False, False]
    seen.clear()
    torch.jit.trace(f, (x,), check_trace=False)
    make_fx(f)(x)
    torch.vmap(f)(x)
    torch.func.grad(lambda y: f(y).sum())(x)
    with FakeTensorMode():
        f(torch.ones(2))
    with forward_ad.dual_level():
        f(x)
    assert seen == [True] * 6
    compiled = torch.compile(lambda y: y * 3 if calls_followed() else y * 2, backend="eager")
    assert torch.equal(compiled(x), x * 3)


# without and with pages
@pytest.mark.gpu
@pytest.mark.parametrize("tracer", ["jit", "fx"])
@pytest.mark.parametrize("T", [40, 300])
def test_traced_prompt_replays_on_other_inputs(dev, tracer, T):
    from kitty import KittyAttentionFactory, KittyConfig
    cfg = KittyConfig(num_layers=1, num_kv_heads=2, head_dim=128, max_seq_len=1024, device="cuda:0")
    bi = torch.full((1, 2, 128), cfg.sentinel, dtype=torch.uint8)
    _, pipe, layers = KittyAttentionFactory.from_config(cfg, bi, 8)
    gen = torch.Generator().manual_seed(T)
    x, y = ([torch.randn(1, h, T, 128, generator=gen).half().to(dev) for h in (8, 2, 2)] for _ in range(2))

    def f(q, k, v):
        pipe.reset_sequence(0)
        return layers[0](q, k, v)
    with torch.no_grad():
        traced = torch.jit.trace(f, tuple(x), check_trace=False) if tracer == "jit" else make_fx(f)(*x)
        out = traced(*y).float()
        # traced attention is torch's, the eager call's the kernel: both round float32 to float16
        assert (out - f(*y).float()).abs().max() < 2e-3
