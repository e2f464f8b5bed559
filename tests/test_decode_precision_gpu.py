"""The matrix-core decodes are no further from float64 than the fp32
shape-generic kernel, whatever the chunks that a plan cuts pages into."""
import pytest
import torch

import kitty  # noqa: F401
from test_bf16_decode_gpu import _case, _float64, _run


# groups of 4 (and 1, padded to 4): P' in fp8 terms.  Split plans with chunks of
# one, two and many pages, and the pair kernel (0: 7 and 2 pages)
@pytest.mark.gpu
@pytest.mark.parametrize("Hq,H,Dk,pages,tails", [(32, 8, 16, [60], [20]), (8, 8, 16, [7], [96]), (16, 4, 32, [2], [5]),
                                                 (12, 4, 0, [30, 3], [0, 64])])
@pytest.mark.parametrize("per_split", [0, 1, 2, 16])
def test_fp16_decode_error(dev, Hq, H, Dk, pages, tails, per_split):
    args, kw = _case(dev, 5 * Hq + len(pages), Hq, H, Dk, pages, None, tails, [32] * len(pages), bf=torch.float16)
    ref = _float64(args, kw)
    fast, gen = _run(args, kw, boost_unique=True, pages_per_split=per_split), _run(args, kw, boost_unique=False)
    e_fast, e_gen = (float((x - ref).norm() / ref.norm()) for x in (fast, gen))
    # both round the output to fp16, about 2.1e-4 of it; what the fp8 terms
    # add (12 bits each, 1e-5 of the output over a page) is not to show in it
    assert e_fast <= 1.05 * e_gen + 1e-6, (e_fast, e_gen)


# sharp to flat softmax rows: the flatter, the more the zero points cancel
@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 0.5, 0.2])
@pytest.mark.parametrize("Hq,H,Dk,pages", [(32, 8, 16, [200]), (16, 4, 32, [90, 3]), (64, 8, 16, [160]), (32, 2, 0, [120])])
def test_bf16_decode_error(dev, Hq, H, Dk, pages, scale):
    args, kw = _case(dev, 3 * Hq + len(pages), Hq, H, Dk, pages, None, [20] * len(pages), [32] * len(pages), q_scale=scale)
    ref = _float64(args, kw)
    fast, gen = _run(args, kw, boost_unique=True), _run(args, kw, boost_unique=False)
    e_fast, e_gen = (float((x - ref).norm() / ref.norm()) for x in (fast, gen))
    # an error of up to 1e-5 of the output, in quadrature with its fp16 rounding of 2.1e-4
    assert e_fast <= 1.001 * e_gen + 1e-7, (e_fast, e_gen)


# key scales that fp16 holds in few bits or not at all, with queries that make
# their scores count; value scales down to 2^-114
@pytest.mark.gpu
@pytest.mark.parametrize("Hq", [4, 8, 16])
@pytest.mark.parametrize("key_exp,val_exp", [(-20, 0), (-34, -20), (-60, 0), (-100, 0), (0, -114)])
def test_bf16_tiny_scales(dev, Hq, key_exp, val_exp):
    args, kw = _case(dev, 37, Hq, 1, 16, [5], [4], [9], [32], q_scale=2.0 ** min(-key_exp, 100))
    q, sk, tk, km, vm = args[0], args[9], args[12], args[5], args[7]
    km[:, :, 0] *= 2.0 ** key_exp
    vm[:, :, :, 0] *= 2.0 ** val_exp
    sk *= 2.0 ** key_exp
    tk *= 2.0 ** key_exp
    ref = _float64(args, kw)
    fast, gen = _run(args, kw, boost_unique=True), _run(args, kw, boost_unique=False)
    e_fast, e_gen = (float((x - ref).norm() / ref.norm()) for x in (fast, gen))
    assert e_fast <= 1.05 * e_gen + 1e-6, (e_fast, e_gen)
