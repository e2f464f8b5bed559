"""bf16 decode on the MFMA split kernel against the shape-generic kernel (which
a plan that does not promise unique boost ranks runs) and float64."""
import math
import warnings

import numpy as np
import pytest
import torch

import kitty  # noqa: F401
from kvgen import calibrate_boost_idx, outlier_keys

G = D = 128


def _case(dev, seed, Hq, H, Dk, pages_k, pages_v, tails, sinks, key_scale=1.0, val_scale=1.0, q_scale=1.0,
          bf=torch.bfloat16):
    """Pools quantised on the device from bf16 (or fp16) blocks and the decode operands;
    pages_v None: one stream."""
    from kitty.kernels.ops import pool_store, quantize_into_pools
    gen = torch.Generator().manual_seed(seed)
    B, n = len(pages_k), sum(pages_k)
    K, chans = outlier_keys(gen, (max(n, 1) * G,), H, D, max(Dk, 1), 8.0)
    K = (K.float() * key_scale).to(bf).to(dev)
    V = (torch.randn(max(n, 1) * G, H, D, generator=gen) * val_scale).to(bf).to(dev)
    bi = torch.full((H, D), Dk + 1, dtype=torch.uint8)
    if Dk:
        calib, _ = outlier_keys(gen, (64,), H, D, Dk, 8.0, channels=chans)
        bi = calibrate_boost_idx(calib, Dk, Dk + 1)
    P = n + 3
    u8 = lambda *s: torch.zeros(*s, dtype=torch.uint8, device=dev)
    pools = (u8(P, H, D, G // 4), u8(P, H, Dk, G // 4), torch.zeros(P, H, 2, D, dtype=bf, device=dev),
             u8(P, H, G, D // 4), torch.zeros(P, H, G, 2, dtype=bf, device=dev))
    perm = torch.randperm(P, generator=gen)[:max(n, 1)].to(torch.int32)
    blocks = lambda x: x.view(-1, G, H, D).permute(0, 2, 1, 3)
    quantize_into_pools(pool_store(*pools), blocks(K), blocks(V), bi.to(dev), perm.to(dev), Dk + 1)
    bt = torch.zeros(B, max(pages_k + [1]), dtype=torch.int32)
    off = 0
    for b in range(B):
        bt[b, :pages_k[b]] = perm[off:off + pages_k[b]]
        off += pages_k[b]
    rnd = lambda *s: torch.randn(*s, generator=gen).to(bf).to(dev)
    T = max(tails + [1])
    tv_len = None if pages_v is None else [t + (k - v) * G for t, k, v in zip(tails, pages_k, pages_v)]
    i32 = lambda x: None if x is None else torch.tensor(x, dtype=torch.int32, device=dev)
    q = (torch.randn(B, Hq, D, generator=gen) * q_scale).to(bf).to(dev)
    args = (q, bt.to(dev), i32(pages_k), *pools, bi.to(dev), rnd(B, H, max(sinks), D), rnd(B, H, max(sinks), D),
            i32(sinks), rnd(B, H, T, D), rnd(B, H, max(tv_len or [T]) or 1, D), i32(tails))
    return args, dict(num_pages_v=i32(pages_v), tail_len_v=i32(tv_len))


def _run(args, kw, **more):
    from kitty.kernels.ops import DecodePlan
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)
        return DecodePlan(*args, **kw, **more).run().cpu().double()


def _float64(args, kw):
    """The same decode in float64 on the CPU."""
    q, bt, npk, kb, kh, km, vp, vm, bi, sk, sv, sl, tk, tv, tl = (t.cpu() for t in args)
    B, Hq, _ = q.shape
    H, Dk = kb.shape[1], kh.shape[2]
    npv = npk if kw["num_pages_v"] is None else kw["num_pages_v"].cpu()
    out = torch.zeros(B, Hq, D, dtype=torch.float64)
    sh = torch.arange(4) * 2
    codes = lambda x: ((x.long()[..., None] >> sh) & 3).flatten(-2)
    for b in range(B):
        pk, pv = int(npk[b]), int(npv[b])
        for h in range(H):
            ids = bt[b, :pk].long()
            c = codes(kb[ids, h])                                              # (n, D, G)
            boosted = bi[h].long() < Dk
            if Dk and pk:
                c[:, boosted] += 4 * codes(kh[ids, h])[:, bi[h].long()[boosted]]
            m = km[ids, h].double()
            kp = ((c.double() - m[:, 1, :, None]) * m[:, 0, :, None]).transpose(1, 2).reshape(-1, D)
            vids = ids[:pv]
            w = vm[vids, h].double()
            vq = ((codes(vp[vids, h]).double() - w[..., 1:]) * w[..., :1]).reshape(-1, D)
            ns, nk = int(sl[b]), int(tl[b])
            nv = (pk - pv) * G + nk
            K = torch.cat([sk[b, h, :ns].double(), kp, tk[b, h, :nk].double()])
            V = torch.cat([sv[b, h, :ns].double(), vq, tv[b, h, :nv].double()])
            if len(K):
                x = q[b].double().view(H, -1, D)[h]
                out[b].view(H, -1, D)[h] = torch.softmax(x @ K.t() / math.sqrt(D), -1) @ V
    return out


# every MFMA group, padded ones, no boosted channels, empty sequences, key-only
# pages (values still in the tail), more than 64 pages of one sequence
@pytest.mark.gpu
@pytest.mark.parametrize("Hq,H,Dk,pages_k,pages_v,tails", [
    (8, 2, 16, [3, 0, 5], None, [17, 96, 0]),
    (8, 8, 16, [7], [6], [97]),
    (6, 2, 32, [1, 2], [0, 1], [1, 127]),
    (16, 2, 16, [4, 9], [3, 8], [5, 64]),
    (14, 2, 0, [2, 3], [2, 1], [0, 33]),
    (16, 1, 32, [5, 1], [4, 0], [31, 32]),
    (24, 2, 16, [3], None, [40]),
    (40, 1, 16, [2, 2], [1, 2], [3, 0]),
    (4, 1, 32, [70], [69], [12]),
    (8, 1, 16, [66, 3], [65, 2], [100, 9]),
])
def test_bf16_matches_generic_and_float64(dev, Hq, H, Dk, pages_k, pages_v, tails):
    args, kw = _case(dev, 7 * Hq + H + len(pages_k), Hq, H, Dk, pages_k, pages_v, tails, [32] * len(pages_k))
    ref = _float64(args, kw)
    fast, gen = _run(args, kw, boost_unique=True), _run(args, kw, boost_unique=False)
    e_fast, e_gen = ((x - ref).norm() / ref.norm() for x in (fast, gen))
    # both round the output to fp16 (2e-4 of it); the split operands may add nothing that shows
    assert e_fast <= 1.05 * e_gen + 1e-6, (float(e_fast), float(e_gen))
    assert ((fast - ref).abs() <= 2.0 ** -11 * ref.abs() + 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("Hq", [4, 8, 16])
@pytest.mark.parametrize("key_scale,val_scale,q_scale", [
    (1.0, 1.0, 3000.0),          # a query past what fp16 products would hold
    (2.0 ** 14, 1.0, 2.0 ** -14),   # boosted scales near fp16's largest
    (2.0 ** -12, 2.0 ** -12, 2.0 ** 12),
    (1.0, 200.0, 1.0),
])
def test_bf16_ranges(dev, Hq, key_scale, val_scale, q_scale):
    args, kw = _case(dev, 91, Hq, 1, 16, [4], [3], [20], [32], key_scale, val_scale, q_scale)
    ref = _float64(args, kw)
    fast, gen = _run(args, kw, boost_unique=True), _run(args, kw, boost_unique=False)
    assert torch.isfinite(fast).all()
    e_fast, e_gen = ((x - ref).norm() / ref.norm() for x in (fast, gen))
    # scores up to ~1e5 at q_scale 3000: fp32 itself moves them by 1e-2, so the
    # two fp32 paths are compared with each other's error, not with a rounding
    assert e_fast <= 1.5 * e_gen + 1e-5, (float(e_fast), float(e_gen))


@pytest.mark.gpu
@pytest.mark.parametrize("Hq", [4, 8, 16])
def test_bf16_pools_with_scales_past_fp16(dev, Hq):
    """Metadata that bf16 holds and fp16 does not (a pool written by a program
    of its own): scales of 2^16 .. 2^20 and 2^-30 decode as in the fp32 kernel."""
    args, kw = _case(dev, 17, Hq, 1, 16, [5], None, [9], [32], q_scale=2.0 ** -17)
    km, vm = args[5], args[7]
    km[:, :, 0, ::3] *= 2.0 ** 17
    km[2, :, 0] *= 2.0 ** -30
    vm[:, :, ::2, 0] *= 0.25
    vm[1, :, 5, 0] = 3.0e4
    ref = _float64(args, kw)
    assert ref.abs().max() < 6e4
    fast, gen = _run(args, kw, boost_unique=True), _run(args, kw, boost_unique=False)
    e_fast, e_gen = ((x - ref).norm() / ref.norm() for x in (fast, gen))
    assert e_fast <= 1.5 * e_gen + 1e-5, (float(e_fast), float(e_gen))


@pytest.mark.gpu
def test_bf16_invalid_pages_poison_one_sequence(dev):
    args, kw = _case(dev, 23, 8, 2, 16, [3, 4], [2, 3], [5, 6], [32, 32])
    clean = _run(args, kw, boost_unique=True)
    args[1][1, 3] = 1 << 20                      # a key-only page of sequence 1 outside the pool
    out = _run(args, kw, boost_unique=True)
    assert torch.equal(out[0], clean[0]) and out[1].isnan().all()


@pytest.mark.gpu
def test_bf16_small_workspace_runs_the_generic_kernel(dev):
    """A caller's workspace that holds only the generic kernel's partials
    (many short sequences) still decodes."""
    from kitty.kernels.ops import DecodePlan
    B = 40
    args, kw = _case(dev, 29, 8, 8, 16, [1] * B, None, [3] * B, [32] * B)
    gen = _run(args, kw, boost_unique=False)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)
        plan = DecodePlan(*args, **kw, boost_unique=True)
    full = plan.run().cpu().double()
    assert plan.args.workspace_bytes > 1 << 20
    plan.args.workspace_bytes = 1 << 20             # the generic partials: 40 x 8 x 2 rows of 520 bytes
    assert torch.equal(plan.run().cpu().double(), gen)
    assert ((full - gen).abs() <= 2.0 ** -10 * gen.abs() + 1e-4).all()
    plan.args.workspace_bytes = 1 << 10
    with pytest.raises(ValueError, match="workspace too small"):
        plan.run()


@pytest.mark.gpu
def test_bf16_plans_name_the_kernel_that_runs(dev):
    """split_kernel tells the bfloat16 instance from the shape-generic kernel, and
    the notice about the one does not swallow the warning about the other."""
    import kitty.kernels.ops as ops
    args, kw = _case(dev, 31, 8, 2, 16, [2], None, [3], [32])
    ops._warned_generic = ()
    with pytest.warns(RuntimeWarning, match="bfloat16 instance"):
        plan = ops.DecodePlan(*args, **kw, boost_unique=True)
    assert (plan.kernel, plan.split_kernel) == ("generic", "mfma_bf16")
    off = list(args)
    off[9] = torch.empty(args[9].numel() + 1, dtype=args[9].dtype, device=dev)[1:].view(args[9].shape)   # sink_k
    with pytest.warns(RuntimeWarning, match="shape-generic kernel because .* aligned"):
        plan = ops.DecodePlan(*off, **kw, boost_unique=True)
    assert (plan.kernel, plan.split_kernel) == ("generic", "generic")
    with pytest.warns(RuntimeWarning, match="repeats a rank"):
        assert ops.DecodePlan(*args, **kw, boost_unique=False).split_kernel == "generic"
    with warnings.catch_warnings():
        warnings.simplefilter("error")          # each once
        ops.DecodePlan(*args, **kw, boost_unique=True)
        ops.DecodePlan(*off, **kw, boost_unique=True)
