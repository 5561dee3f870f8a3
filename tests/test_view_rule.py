"""`strided_view_reason`'s early answers are the rule's: every view of small sizes and of strides around
their extents, against the rule written out (CPU)."""
import itertools

import torch


def _rule(t):
    st = t.stride()
    if st[3] != 1:
        return "stride_last"
    if min(st) <= 0:
        return "stride_nonpos"
    if any(s % 8 for s in st[:3]):
        return "stride_align"
    if t.data_ptr() % 16:
        return "ptr_align"
    dims = sorted((s, n) for s, n in zip(st, t.shape) if n > 1)
    if any(s1 < s0 * n0 for (s0, n0), (s1, _) in zip(dims, dims[1:])):
        return "stride_overlap"
    return None


def test_every_small_view():
    from sageattention.sk1_backend.sk1_loader import strided_view_reason
    buf = torch.empty(1 << 14, dtype=torch.float16)
    base = (-buf.data_ptr() // 2) % 8          # 16-byte aligned
    seen = set()
    for n in itertools.product((1, 2, 3), repeat=3):
        for st in itertools.product((0, 8, 56, 60, 64, 72, 128, 192, 384), repeat=3):
            for off in (0, 4):
                t = buf.as_strided((*n, 64), (*st, 1), base + off)
                want = _rule(t)
                assert strided_view_reason(t) == want, (n, st, off)
                seen.add(want)
    assert seen == {None, "stride_nonpos", "stride_align", "ptr_align", "stride_overlap"}
