"""The dK/dV kernel reads its Q and dO tiles from the caller's tensors where
their rows allow it and from padded copies otherwise; both give the same bits
for every layout, and rows past the end are never read into the result."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _bwd(do, q, k, v, out, lse, staged):
    from avgen_amd import ops

    return ops._bwd_impl(do, q, k, v, out, lse, None, 1.0 / math.sqrt(q.shape[-1]), stage_ds=staged)


@pytest.mark.parametrize("staged", [True, False])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [1, 63, 64, 65, 193])
def test_query_layouts_give_the_same_bits(Lq, D, staged):
    from avgen_amd import ops

    B, H, Hkv, Lk = 2, 4, 2, 150
    g = torch.Generator(device="cuda").manual_seed(Lq * D)

    def rnd(*shape):
        return torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)

    q, k, v = rnd(B, H, Lq, D), rnd(B, Hkv, Lk, D), rnd(B, Hkv, Lk, D)
    row = rnd(B, H, 1, D)
    do = row.expand(B, H, Lq, D).contiguous()
    out, lse = ops.flash_fwd(q, k, v, None, None, None, 1.0 / math.sqrt(D))
    want = _bwd(do, q, k, v, out, lse, staged)

    def poisoned(x):  # the rows after x's last one hold NaN
        buf = torch.full((B, H, Lq + 70, D), float("nan"), device="cuda", dtype=torch.bfloat16)
        buf[:, :, :Lq] = x
        return buf[:, :, :Lq]

    def blhd(x):  # (B, L, H, D) memory
        return x.transpose(1, 2).contiguous().transpose(1, 2)

    layouts = {
        "rows followed by NaN": (poisoned(do), poisoned(q)),
        "(B, L, H, D) memory": (blhd(do), blhd(q)),
        "dO rows sharing memory (copied)": (row.expand(B, H, Lq, D), q),
    }
    for name, (d2, q2) in layouts.items():
        got = _bwd(d2, q2, k, v, out, lse, staged)
        for label, a, b in zip(("dq", "dk", "dv"), got, want):
            assert torch.isfinite(a.float()).all(), (name, label)
            assert torch.equal(a, b), (name, label)
