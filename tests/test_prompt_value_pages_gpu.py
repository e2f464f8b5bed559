"""Prompts of several sequences whose values fill one page each."""
import pytest
import torch


@pytest.mark.gpu
def test_prompt_batch_with_one_value_page(dev):
    """Several prompts with two key pages and one value page each: every
    sequence's values go to its own page, as when it is pushed alone."""
    from kitty import KittyAttentionFactory, KittyConfig
    T, H, D = 300, 2, 128
    gen = torch.Generator().manual_seed(8)
    k, v = (torch.randn(3, H, T, D, generator=gen).half().to(dev) for _ in range(2))
    pools = []
    for batches in ([[0, 1, 2]], [[0], [1], [2]]):
        cfg = KittyConfig(num_layers=1, num_kv_heads=H, head_dim=D, max_seq_len=512, max_batch_size=3, device="cuda:0")
        bi = torch.full((1, H, D), cfg.sentinel, dtype=torch.uint8)
        bi[0, :, :cfg.d_boost] = torch.arange(cfg.d_boost, dtype=torch.uint8)
        layout, pipe, _ = KittyAttentionFactory.from_config(cfg, bi, H)
        for ids in batches:
            pipe.push_chunk(0, k[ids[0]:ids[-1] + 1], v[ids[0]:ids[-1] + 1], ids)
        pools.append((layout.value_pool.clone(), layout.value_metadata.clone(), pipe.lens.clone()))
    for a, b in zip(*pools):
        assert torch.equal(a, b)
