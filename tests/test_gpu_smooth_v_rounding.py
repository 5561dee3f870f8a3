"""fp16 outputs of smooth_v are rounded once (GPU).

O = T(acc * inv + mean) is formed by one mixed-precision fma per output, rounded to fp16 from the
exact sum. Zero queries on three keys make every term known: all probabilities are 1, so acc is the
sum of three products of the quantized V and the keys' e4m3 weights, and inv = RN(S / (3 * 448)).
A sum that is rounded to fp32 first gives another fp16 value for about 3 in 1000 of them; the
planes are enough to hold some of those.
"""
import numpy as np
import oracle
import pytest
import torch

from sage_testutil import have_gfx950

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not have_gfx950(), reason="needs a gfx950 GPU")]


@pytest.mark.parametrize("D,kernel", [(128, 1), (128, 2), (128, 3), (64, 1), (64, 3), (64, 4)])
def test_one_rounding(D, kernel):
    from sageattention.sk1_backend import sk1_forward
    from sageattention.sk1_backend.sk1_loader import SageLib
    print("case", D, kernel, flush=True)
    H = 4000 * 128 // D
    g = torch.Generator().manual_seed(D)
    k, v = (torch.randn(1, H, 3, D, generator=g).half() for _ in range(2))
    v = v + torch.randn(1, H, 1, D, generator=g).half() * 3
    q = torch.zeros(1, H, 1, D, dtype=torch.float16)
    o = sk1_forward(SageLib.get(), q.cuda(), k.cuda(), v.cuda(), smooth_v=True, kernel=kernel)
    o = o.cpu().view(H, D).numpy()

    vr = v.view(H, 3, D)
    vmean = oracle.kseq_mean(vr)
    v8t, sv = oracle.quant_v(vr, 64, mean=vmean)
    s, svp = oracle.fold_v_scale(sv)
    w8 = (svp[:, :3] * 448.0).to(torch.float8_e4m3fn).double()
    terms = w8[:, None, :] * v8t[:, :, :3].double()            # (H, D, 3), exact
    acc = terms.sum(2)
    inv = (s / np.float32(3 * 448)).double()
    exact = (acc * inv[:, None] + vmean.double()).numpy()
    # the matrix core keeps fewer than 14 bits below the largest product of a sum (terms of
    # -0.3164, -96 and 96 lose the first one's last bits): compared where every term is a multiple
    # of 2^-10 of the largest one's power of two
    unit = torch.exp2(torch.floor(torch.log2(terms.abs().amax(2).clamp(min=2.0 ** -20))) - 10)
    safe = (torch.remainder(terms, unit[:, :, None]) == 0).all(2).numpy()
    once = exact.astype(np.float16)
    twice = exact.astype(np.float32).astype(np.float16)
    assert ((once != twice) & safe).sum() >= 1000
    assert safe.mean() > 0.9
    assert np.array_equal(o[safe], once[safe]), int((o != once)[safe].sum())
