"""Query and output tiles at their edges, and causal grids in every order branch, through every
main-loop kernel; the two forms of the head_dim 64 per-key constants (GPU).

A wave quantizes 32 query rows together (16 or 8 lanes to a row, 4 or 8 rows to a load) and writes
its output tile in whole row pieces, through LDS; a causal grid starts its tiles longest first, per
XCD where the planes share out over the 8 XCDs, else over all planes. Row counts around 32 and the
query tiles, row strides that are no multiple of a row, rows with one large value in any column,
zero rows; planes below, at and beyond a multiple of 8, with one to many tiles per compute unit. A head_dim 64 launch takes its
per-key constants from LDS once it has more than 1 (key split), 2 or 3 (causal) blocks for each of
256 compute units. Bars: the emulation's; kernels 1-3 bit for bit.
"""
import oracle
import pytest
import torch

from sage_testutil import COS_MIN, cosine, have_gfx950, make_qkv, rel_l1, rel_l1_bar

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not have_gfx950(), reason="needs a gfx950 GPU")]


def _forward(q, k, v, **kw):
    from sageattention.sk1_backend import sk1_forward
    from sageattention.sk1_backend.sk1_loader import SageLib
    r = sk1_forward(SageLib.get(), q, k, v, **kw)
    torch.cuda.synchronize()
    return r


def _kernels(D, causal):
    return [1, 3] + ([2] if D == 128 else []) + ([4] if D == 64 and not causal else [])


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N", [1, 7, 8, 31, 32, 33, 63, 97, 129, 255, 257])
def test_query_and_output_tile_edges(N, dtype, causal, D):
    print("case", N, dtype, causal, D, flush=True)
    q, k, v = make_qkv(1, 3, N, seed=N + 3 * D, dtype=dtype, k_offset_std=2.0, d=D,
                       v_offset_std=1.0)
    rows = torch.arange(N)
    q[:, :, rows, (5 * rows) % D] = 6.0          # the row maximum in any column
    q[0, 1, N // 2] = 0.0
    r = oracle.emulate_sageattn(q, k, v, is_causal=causal, smooth_v=True)
    # rows D + 8 elements apart, the heads' rows interleaved
    wide = torch.zeros(1, N, 3, D + 8, dtype=dtype, device="cuda")
    wide[..., :D] = q.cuda().transpose(1, 2)
    qv = wide[..., :D].transpose(1, 2)
    first = None
    for kern in _kernels(D, causal):
        o, lse = _forward(qv, k.cuda(), v.cuda(), is_causal=causal, kernel=kern, smooth_v=True,
                          return_lse=True)
        o, lse = o.cpu(), lse.cpu()
        assert cosine(o, r["o"]) >= COS_MIN
        assert rel_l1(o, r["o"]) <= rel_l1_bar(dtype == torch.float16), (kern, rel_l1(o, r["o"]))
        if kern != 4:
            first = first or (o, lse)
            assert torch.equal(o, first[0]) and torch.equal(lse, first[1]), kern


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("B,H,N", [(1, 3, 700), (1, 9, 1100), (1, 17, 2100), (1, 24, 2000),
                                   (2, 8, 2600), (1, 16, 4200), (1, 48, 1500), (1, 40, 1000)])
def test_causal_orders_same_bits(B, H, N, D):
    # kernel 1 keeps planes together; 2 and 3 reorder (planes per XCD whole or not, two or three
    # blocks per compute unit, several rounds)
    print("case", B, H, N, D, flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    q, k, v = (torch.randn(B, H, N, D, generator=g, device="cuda").half() for _ in range(3))
    outs = {kern: _forward(q, k, v, is_causal=True, kernel=kern) for kern in _kernels(D, True)}
    assert torch.isfinite(outs[1]).all()
    for kern, o in outs.items():
        assert torch.equal(o, outs[1]), kern


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,N,causal,kern", [
    (256, 128, False, 3), (257, 128, False, 3), (512, 1, False, 3), (513, 129, False, 3),
    (171, 300, False, 3), (768, 100, True, 3), (769, 77, True, 3), (257, 321, True, 3),
    (64, 256, False, 4), (65, 256, False, 4), (257, 33, False, 4), (43, 400, False, 4)])
def test_d64_constants_same_bits_in_small_and_large_grids(H, N, causal, kern, dtype):
    # each plane's result is the one it has in a grid of 20 planes, on either side of the line
    print("case", H, N, causal, kern, dtype, flush=True)
    q, k, v = (t.cuda() for t in make_qkv(1, H, N, seed=H + N, dtype=dtype, d=64,
                                          k_offset_std=2.0, v_offset_std=1.0))
    kw = dict(is_causal=causal, kernel=kern, smooth_v=True, return_lse=True)
    o, lse = _forward(q, k, v, **kw)
    assert torch.isfinite(o).all()
    for h in (0, H - 20):
        ps = slice(h, h + 20)
        op, lp = _forward(q[:, ps].contiguous(), k[:, ps].contiguous(), v[:, ps].contiguous(), **kw)
        assert torch.equal(op, o[:, ps]) and torch.equal(lp, lse[:, ps])
