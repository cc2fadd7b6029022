"""Key tiles without an attended key are left out of the forward and of the
staged backward: the bits are those of the same call without these keys, and
a value that would reach the result through such a tile (a NaN or infinite
masked key, value or query row) still does."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def _rnd(*shape, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, device="cuda", generator=g) * scale).to(torch.bfloat16)


def _run(q, k, v, do, mask):
    from avgen_amd import ops

    scale = 1.0 / math.sqrt(q.shape[-1])
    out, lse = ops.flash_fwd(q, k, v, mask, None, None, scale)
    return (out, lse, *ops._bwd_impl(do, q, k, v, out, lse, mask, scale, stage_ds=True))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lead,valid,tail", [(0, 64, 1), (0, 100, 412), (64, 64, 64), (128, 45, 200), (256, 130, 0)])
def test_masked_ends_equal_a_shorter_key_sequence(lead, valid, tail, D):
    B, H, Hkv, Lq = 2, 4, 2, 150
    L = lead + valid + tail
    q, do = _rnd(B, H, Lq, D, seed=1), _rnd(B, H, Lq, D, seed=2)
    # Masked keys of small norm: the head's largest key norm, which the
    # forward's score bound uses, is an attended key's.
    k, v = _rnd(B, Hkv, L, D, seed=3, scale=0.05), _rnd(B, Hkv, L, D, seed=4)
    sl = slice(lead, lead + valid)
    k[:, :, sl] = _rnd(B, Hkv, valid, D, seed=5)
    mask = torch.zeros(B, L, dtype=torch.bool, device="cuda")
    mask[:, sl] = True
    out, lse, dq, dk, dv = _run(q, k, v, do, mask)
    ref = _run(q, k[:, :, sl].contiguous(), v[:, :, sl].contiguous(), do, None)
    for label, a, b in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, dq, dk[:, :, sl], dv[:, :, sl]), ref):
        assert torch.equal(a, b), label
    for label, g in (("dk", dk), ("dv", dv)):
        assert (g[:, :, :lead] == 0).all() and (g[:, :, lead + valid:] == 0).all(), label


@pytest.mark.parametrize("D", [64, 128])
def test_masked_tile_in_the_middle_and_a_row_without_keys(D):
    B, H, Lq, L = 2, 2, 70, 384
    q, do = _rnd(B, H, Lq, D, seed=1), _rnd(B, H, Lq, D, seed=2)
    k, v = _rnd(B, H, L, D, seed=3), _rnd(B, H, L, D, seed=4)
    mask = torch.zeros(B, L, dtype=torch.bool, device="cuda")
    mask[0, 70:128] = True
    mask[0, 256:300] = True
    out, lse, dq, dk, dv = _run(q, k, v, do, mask)
    s = (q[0].float() @ k[0].float().transpose(-1, -2)) / math.sqrt(D)
    p = s.masked_fill(~mask[0], -INF).softmax(-1)
    # 2^-8 per rounding of P and of the output, sums of 102 terms of size <= 4
    assert (out[0].float() - p @ v[0].float()).abs().max() <= 2e-2
    for t in (out[1], dq[1], dk[1], dv[1], dk[0, :, ~mask[0]], dv[0, :, ~mask[0]]):
        assert (t == 0).all()
    assert (lse[1] == -INF).all()
    assert torch.isfinite(dq.float()).all() and torch.isfinite(dk.float()).all()


@pytest.mark.parametrize("where,value", [("k", NAN), ("k", INF), ("v", NAN), ("v", INF)])
def test_value_of_a_masked_tile_still_reaches_the_output(where, value):
    B, H, Lq, D, L = 1, 2, 70, 128, 320
    q, do = _rnd(B, H, Lq, D, seed=1), _rnd(B, H, Lq, D, seed=2)
    k, v = _rnd(B, H, L, D, seed=3), _rnd(B, H, L, D, seed=4)
    (k if where == "k" else v)[0, 0, 300, 5] = value
    mask = torch.arange(L, device="cuda")[None] < 100
    out, lse, dq, _, _ = _run(q, k, v, do, mask)
    if where == "k":
        # an infinite score is NaN once masked where it is +inf, -inf else
        rows = torch.ones(Lq, dtype=torch.bool, device="cuda") if value != value else q[0, 0, :, 5] > 0
        assert out[0, 0, rows].isnan().all() and lse[0, 0, rows].isnan().all() and dq[0, 0, rows].isnan().any()
        assert torch.isfinite(lse[0, 0, ~rows]).all()
    else:
        assert out[0, 0, :, 5].isnan().all() and torch.isfinite(lse).all()
    assert torch.isfinite(out[0, 1].float()).all() and torch.isfinite(dq[0, 1].float()).all()


def test_nan_query_row_without_keys_stays_nan():
    B, H, Lq, D, L = 1, 1, 300, 128, 128
    q, do = _rnd(B, H, Lq, D, seed=1), _rnd(B, H, Lq, D, seed=2)
    k, v = _rnd(B, H, L, D, seed=3), _rnd(B, H, L, D, seed=4)
    q[0, 0, 7, 3] = NAN
    mask = torch.zeros(B, L, dtype=torch.bool, device="cuda")
    out, lse, _, _, _ = _run(q, k, v, do, mask)
    assert out[0, 0, 7].isnan().all() and lse[0, 0, 7].isnan()
    keep = torch.arange(Lq, device="cuda") != 7
    assert (out[0, 0, keep] == 0).all() and (lse[0, 0, keep] == -INF).all()


@pytest.mark.parametrize("D", [64, 128])
def test_masked_ends_in_several_passes(D):
    """One (batch, kv head) pair of dS per pass: every pass leaves out its own
    pair's tiles."""
    from avgen_amd import _lib, ops

    B, H, Hkv, Lq, L = 2, 4, 2, 150, 400
    q, do = _rnd(B, H, Lq, D, seed=1), _rnd(B, H, Lq, D, seed=2)
    k, v = _rnd(B, Hkv, L, D, seed=3), _rnd(B, Hkv, L, D, seed=4)
    k[1, 1, 390, 7] = NAN  # this pair's last tile cannot be left out
    key = torch.arange(L, device="cuda")
    mask = torch.stack([(key >= 130) & (key < 200), key < 70])
    s = 1.0 / math.sqrt(D)
    out, lse = ops.flash_fwd(q, k, v, mask, None, None, s)
    lib = _lib.load()
    one, every = (ops._bwd_impl(do, q, k, v, out, lse, mask, s, stage_ds=True, workspace=torch.full(
        (lib.avattn_bwd_staged_workspace_size(B, H, Hkv, Lq, L, D, n),), 255, dtype=torch.uint8, device="cuda"))
        for n in (1, B * Hkv))
    for label, a, b in zip(("dq", "dk", "dv"), one, every):
        assert torch.equal(a.isnan(), b.isnan()), label
        assert torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0)), label
    assert torch.isfinite(one[0][0].float()).all() and one[0][1, 2:].isnan().any()
    for g in one[1:]:
        assert (g.transpose(1, 2)[~mask] == 0).all()
