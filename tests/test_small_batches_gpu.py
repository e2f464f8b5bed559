"""Decodes of few work units (the plan's short chunks and its spread over the
XCDs) and around the sizes where the plan changes its chunk."""
import numpy as np
import pytest
import torch

import oracle as O
from kvgen import random_pools

D = G = 128


# (8 pairs) units of a pair = pages + 18 (the FP16 capacity of 32 + 256 tokens):
# one page, a few, chunk 2 -> 3 -> 4 (about 238, 366, 494 pages), ragged, an empty sequence
@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,pages", [(8, 8, [1]), (4, 1, [0]), (32, 8, [7]), (8, 2, [3, 0, 9]), (16, 1, [2, 5]),
                                          (16, 2, [1, 1, 1]), (32, 8, [110]), (32, 8, [111, 109]), (8, 8, [240]),
                                          (8, 8, [366]), (8, 8, [494])])
def test_small_plans_match_oracle(dev, Hq, Hkv, pages):
    from kitty.kernels.ops import DecodePlan
    gen = torch.Generator().manual_seed(sum(pages) + Hq)
    rng = np.random.default_rng(sum(pages) + Hq)
    B, Dk, P = len(pages), 16, max(sum(pages), 1)
    bi = torch.full((Hkv, D), Dk + 1, dtype=torch.uint8)
    for h in range(Hkv):
        bi[h, torch.randperm(D, generator=gen)[:Dk]] = torch.arange(Dk, dtype=torch.uint8)
    pools = random_pools(gen, P, Hkv, D, G, Dk, bi, rng)
    bt = torch.zeros(B, max(pages + [1]), dtype=torch.int32)
    off = 0
    for b, n in enumerate(pages):
        bt[b, :n] = torch.arange(off, off + n)
        off += n
    npv = [max(0, n - 1) for n in pages]
    tails = [(17 * (b + 1)) % 128 for b in range(B)]
    tv_len = [t + (n - v) * G for t, n, v in zip(tails, pages, npv)]
    rnd = lambda *s: torch.randn(*s, generator=gen).half()
    q = rnd(B, Hq, D) * 0.25
    sk, sv, tk, tv = rnd(B, Hkv, 32, D), rnd(B, Hkv, 32, D), rnd(B, Hkv, 128, D), rnd(B, Hkv, 256, D)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    d = lambda t: t.to(dev)
    plan = DecodePlan(d(q), d(bt), i32(pages), *[d(t) for t in pools], d(bi), d(sk), d(sv), i32([32] * B), d(tk), d(tv),
                      i32(tails), num_pages_v=i32(npv), tail_len_v=i32(tv_len))
    assert plan.kernel == "mfma"
    out = plan.run().clone()
    assert torch.equal(plan.run(), out)
    n = lambda t: t.numpy()
    for b in range(B):
        pg = n(bt[b, :pages[b]])
        ref = O.paged_attention_kv(n(q[b]), pg, pg[:npv[b]], *[n(t) for t in pools], n(bi), Dk, n(sk[b]), n(sv[b]),
                                   n(tk[b, :, :tails[b]]), n(tv[b, :, :tv_len[b]]), Hq, Hkv, D)
        got, ref = out[b].float().cpu().numpy(), np.asarray(ref, np.float32)
        assert (np.abs(got - ref) <= 2e-3 + 1e-2 * np.abs(ref)).all(), (b, float(np.abs(got - ref).max()))
