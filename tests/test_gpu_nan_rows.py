"""Rows that hold a NaN: the row's scale comes from its other values, whatever kind of NaN it is and
wherever it stands (GPU).

The quantizers take a row's absmax over the values that are no NaN. A bf16 row is widened by a shift,
so a signalling NaN reaches the maxima as one, and the hardware's maximum then returns a NaN instead
of the other operand. Every column of a row, both signs, quiet and signalling, in V, K and Q rows.
"""
import pytest
import torch

from sage_testutil import bytes_equal, have_gfx950

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not have_gfx950(), reason="needs a gfx950 GPU")]

#: quiet, signalling with the lowest and the highest payload
NANS = {torch.bfloat16: (0x7fc0, 0x7f81, 0x7fbf), torch.float16: (0x7e00, 0x7c01, 0x7dff)}


def _rows(dtype, D, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(1, 2, 2 * D, D, generator=g).to(dtype)


def _with_nans(x, pattern):
    """Row n gets the pattern in column n % D, its sign bit set in the second half of the rows."""
    n, d = x.shape[2], x.shape[3]
    y = x.clone()
    rows = torch.arange(n)
    p = torch.where(rows < n // 2, pattern, pattern | 0x8000)
    y.view(torch.int16)[:, :, rows, rows % d] = p.to(torch.int16)
    return y


def _zeroed(x):
    y = x.clone()
    rows = torch.arange(x.shape[2])
    y[:, :, rows, rows % x.shape[3]] = 0
    return y


def _others(t, D):
    """The bytes of a (planes, rows, D) tensor without those of the NaNs."""
    t = t.clone().view(torch.uint8)
    rows = torch.arange(t.shape[1])
    t[:, rows, rows % D] = 0
    return t


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("dtype,int8", [(torch.bfloat16, False), (torch.float16, True),
                                        (torch.float16, False)])
def test_a_nan_does_not_touch_the_rest_of_its_row(dtype, int8, D):
    from sageattention.sk1_backend.hip_prologue import HipPrologue
    from sageattention.sk1_backend.sk1_loader import SageLib
    print("case", dtype, int8, D, flush=True)
    lib = SageLib.get()
    x = _rows(dtype, D, D)

    def quantized(t):
        k8, sk, v8t, sv = HipPrologue().quant_kv(t.cuda(), t.cuda(), int8=int8)
        q8, sq, cq = lib.quant_q(t.cuda(), D ** -0.5, qk_int8=int8)
        torch.cuda.synchronize()
        planes = lambda y: y.reshape(2, -1, D).cpu()
        return ([_others(planes(k8), D), _others(planes(v8t.view(torch.uint8).transpose(1, 2).contiguous()), D),
                 _others(planes(q8), D)], [y.cpu() for y in (sk, sv, sq, cq)])

    want_bytes, want_scales = quantized(_zeroed(x))
    for pattern in NANS[dtype]:
        got_bytes, got_scales = quantized(_with_nans(x, pattern))
        for name, g, w in zip(("K8", "V8T", "Q8"), got_bytes, want_bytes):
            assert torch.equal(g, w), (hex(pattern), name)
        for name, g, w in zip(("SK", "SV", "sq", "c_q"), got_scales, want_scales):
            assert bytes_equal(g, w), (hex(pattern), name)
