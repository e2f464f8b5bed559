"""Profiler sums without a zeroed slot buffer and scores / ranks of all layers
in one launch, against float64 and rank_channels."""
import pytest
import torch

from kitty import KittyConfig
from kitty.sensitivity import KittySensitivityProfiler, rank_channels


def _cfg(L, H, D, **kw):
    return KittyConfig(num_layers=L, num_kv_heads=H, head_dim=D, device="cuda:0", **kw)


def _off(x):
    return torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].copy_(x.reshape(-1)).view(x.shape)


# one and many chunks, more chunks in a later batch than in the first and fewer,
# reads between batches, keys off 16-byte rows in between, head_dims with and
# without slots, more layers than one launch takes
@pytest.mark.gpu
@pytest.mark.parametrize("L,H,D,batches,dtype", [
    (1, 1, 128, [(1, 1)], torch.float16),
    (3, 8, 128, [(2, 300), (1, 5), (4, 2048)], torch.bfloat16),
    (2, 2, 64, [(1, 4000), (1, 17)], torch.float16),
    (2, 3, 80, [(1, 33), (2, 10)], torch.float16),
    (2, 2, 256, [(1, 700)], torch.bfloat16),
    (70, 1, 16, [(1, 40)], torch.float16),
    (1, 2, 512, [(2, 64)], torch.float16),
])
def test_scores_and_ranks(dev, L, H, D, batches, dtype):
    gen = torch.Generator().manual_seed(D + L)
    cfg = _cfg(L, H, D)
    prof = KittySensitivityProfiler(cfg)
    # stale memory under the slot buffers must not count
    junk = [torch.full((H * D * 256,), float("nan"), device=dev) for _ in range(L)]
    del junk
    want = torch.zeros(L, H, D, dtype=torch.float64)
    tokens = 0
    for i, (B, T) in enumerate(batches):
        tokens += B * T
        for l in range(L):
            k = (torch.randn(B, T, H, D, generator=gen) * (1 + l)).to(dtype)
            want[l] += k.double().abs().sum((0, 1))
            kk = k.to(dev).permute(0, 2, 1, 3)
            prof.update(l, _off(kk) if i == 1 else kk)
            if i == 1 and l == 0:
                assert torch.allclose(prof.accumulator(0).sum_abs.cpu().double(), want[0], rtol=1e-5)
    prof.compute()
    assert torch.allclose(prof.scores_.double(), want / tokens, rtol=1e-5)
    masks, idx = rank_channels(prof.scores_, cfg.d_boost, cfg.sentinel)
    assert torch.equal(prof.boost_idx_uint8, idx) and torch.equal(prof.boost_masks, masks)
    for l in range(L):
        assert torch.allclose(prof.accumulator(l).sum_abs.cpu().double(), want[l], rtol=1e-5)
    # a second round after the read adds to the first
    k = torch.randn(1, 50, H, D, generator=gen).to(dtype)
    for l in range(L):
        prof.update(l, k.to(dev).permute(0, 2, 1, 3))
    prof.compute()
    want += k.double().abs().sum((0, 1))
    assert torch.allclose(prof.scores_.double(), want / (tokens + 50), rtol=1e-5)


@pytest.mark.gpu
def test_ties_and_nan_rank_as_on_the_host(dev):
    cfg = _cfg(2, 2, 128, boost_rate=0.25)
    prof = KittySensitivityProfiler(cfg)
    k = torch.ones(1, 2, 4, 128, dtype=torch.float16)
    k[0, 0, :, 60:70] = 3.0
    k[0, 1, 2, 100] = float("nan")
    k[0, 1, :, 7] = float("inf")
    k[0, 1, :, 64:] *= 2.0
    for l in range(2):
        prof.update(l, k.to(dev))
    prof.compute()
    masks, idx = rank_channels(prof.scores_, cfg.d_boost, cfg.sentinel)
    assert torch.equal(prof.boost_idx_uint8, idx) and torch.equal(prof.boost_masks, masks)
    assert int(idx[0, 1, 100]) == 0 and int(idx[0, 1, 7]) == 1


@pytest.mark.gpu
def test_layers_without_calibration_score_zero(dev):
    cfg = _cfg(3, 1, 128)
    prof = KittySensitivityProfiler(cfg)
    prof.update(1, torch.randn(1, 1, 64, 128).half().to(dev))
    prof.compute()
    assert int(prof.scores_[0].ne(0).sum()) == 0 and int(prof.scores_[1].eq(0).sum()) == 0
    with pytest.raises(RuntimeError, match="No tokens"):
        prof.accumulator(2)
        prof.compute()


@pytest.mark.gpu
def test_failed_scores_leave_the_sums(dev, monkeypatch):
    """A compute() whose launch is refused raises and loses nothing."""
    from kitty import _hip
    cfg = _cfg(2, 1, 128)
    prof = KittySensitivityProfiler(cfg)
    keys = [torch.randn(1, 1, 64, 128).half() for _ in range(2)]
    for l in range(2):
        prof.update(l, keys[l].to(dev))

    class Refusing:
        def __getattr__(self, name):
            return (lambda *a: _hip.KITTY_E_HIP) if name == "kitty_channel_scores" else getattr(real, name)
    real = _hip.load()
    with monkeypatch.context() as m:
        m.setattr(_hip, "_lib", Refusing())
        with pytest.raises(RuntimeError):
            prof.compute()
    for l in range(2):
        want = keys[l].double().abs().sum((0, 2))
        assert torch.allclose(prof.accumulator(l).sum_abs.cpu().double(), want, rtol=1e-5)
    prof.compute()
    assert torch.allclose(prof.scores_[1, 0].double(), keys[1].double().abs().mean((0, 1, 2)), rtol=1e-5)
