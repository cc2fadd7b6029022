"""dK/dV with every key block split over ranges of queries (short grids)
against the unsplit kernel: equal up to fp32 summation order and one bf16
rounding, masked keys exactly zero, dq the same bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,lens", [
    (1, 4, 4, 4097, 129, None),          # few blocks, a last tile of one row
    (1, 3, 3, 1600, 70, (50,)),
    (2, 8, 4, 2200, 300, (300, 0)),      # grouped heads, 8 pairs, a row without keys
    (2, 6, 6, 4500, 520, (20, 500)),     # 12 pairs: the plain XCD map
    (4, 20, 20, 12031, 512, (512, 1, 0, 256)),  # more blocks than CUs: not split
])
def test_split_equals_unsplit(B, Hq, Hkv, Lq, Lk, lens, D):
    from avgen_amd import _lib, ops

    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(Lq)

    def rnd(*shape):
        return torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)

    q, do, k, v = rnd(B, Hq, Lq, D), rnd(B, Hq, Lq, D), rnd(B, Hkv, Lk, D), rnd(B, Hkv, Lk, D)
    mask = None if lens is None else torch.arange(Lk, device="cuda")[None] < torch.tensor(lens, device="cuda")[:, None]
    s = 1 / math.sqrt(D)
    out, lse = ops.flash_fwd(q, k, v, mask, None, None, s)
    staged = lib.avattn_bwd_staged_workspace_size(B, Hq, Hkv, Lq, Lk, D, B * Hkv)
    split = lib.avattn_bwd_split_workspace_size(B, Hq, Hkv, Lq, Lk, D)
    assert (split > staged) == (B * Hkv * ((Lk + 127) // 128) <= 256)
    got, ref = (ops._bwd_impl(do, q, k, v, out, lse, mask, s,
                              workspace=torch.full((n,), 255, dtype=torch.uint8, device="cuda"))
                for n in (split, staged))
    assert torch.equal(got[0], ref[0])
    for label, a, b in zip(("dk", "dv"), got[1:], ref[1:]):
        assert torch.isfinite(a.float()).all(), label
        # the fp32 sums differ by reassociation only: at most one bf16 step
        assert (a.float() - b.float()).abs().max() <= 2.0**-7 * b.float().abs().max(), label
        assert ((a.float() - b.float()).abs() <= 2.0**-7 * b.float().abs() + 1e-4 * b.float().abs().max()).all(), label
        if mask is not None:
            assert (a.transpose(1, 2)[~mask] == 0).all(), label
    again = ops._bwd_impl(do, q, k, v, out, lse, mask, s,
                          workspace=torch.zeros(split, dtype=torch.uint8, device="cuda"))
    for a, b in zip(got, again):
        assert torch.equal(a, b)
