"""The prologue's steps and row groups against the oracle, bit for bit (GPU).

Both passes work in steps of 128 rows (head_dim 128) or 256 (64), 8 consecutive rows to a thread,
whose maxima the 16 (8) lanes of a row group exchange so that lane i holds row i's scale. Lengths
around a row group (8), a 64-key block and a step, planes of one and of several steps per block,
rows whose largest value sits in any column (every lane of the exchange), zero rows, and rows beyond
448 (S > 1).
"""
import pytest
import torch

from sage_testutil import have_gfx950, make_qkv, quantized_bit_exact

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not have_gfx950(), reason="needs a gfx950 GPU")]


def _spread_maxima(x):
    """Row n's largest magnitude in column n (mod D), by a factor that leaves it the maximum."""
    n, d = x.shape[2], x.shape[3]
    rows = torch.arange(n)
    x[:, :, rows, rows % d] = 9.0 + (rows % 7).to(x.dtype) * 0.5
    return x


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("layout", ["HND", "NHD"])
@pytest.mark.parametrize("dtype,k_int8", [(torch.float16, True), (torch.float16, False),
                                          (torch.bfloat16, False)])
@pytest.mark.parametrize("N", [1, 7, 8, 9, 63, 65, 127, 128, 129, 191, 255, 256, 257, 513, 1337])
def test_steps_bit_exact(N, dtype, k_int8, layout, D):
    print("case", N, dtype, k_int8, layout, D, flush=True)
    q, k, v = make_qkv(1, 3, N, seed=N + D, dtype=dtype, k_offset_std=2.0, d=D)
    _spread_maxima(k)
    _spread_maxima(v)
    k[0, 1, N // 2] = 0.0
    v[0, 1, N // 2] = 0.0
    v[0, 2, N - 1, :] = 900.0            # S > 1 in this plane
    if layout == "NHD":
        k, v = (t.transpose(1, 2).contiguous() for t in (k, v))
    assert quantized_bit_exact(k, v, layout, k_int8)


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("BH,N", [(1, 40000), (500, 300), (1025, 200), (300, 1030)],
                         ids=["one_plane", "two_parts", "one_part", "several_steps"])
def test_parts_bit_exact(BH, N, D):
    # one plane over all the blocks (up to 313 mean partials), two blocks per plane, one block per
    # plane, and blocks of several steps
    g = torch.Generator().manual_seed(BH)
    k, v = (torch.randn(1, BH, N, D, generator=g).half() for _ in range(2))
    k += 1.5
    assert quantized_bit_exact(k, v, "HND", True)
