"""The float32 kernels with a split last round (forward over keys, dK/dV over
queries) against the unsplit ones: equal up to the order of fp32 sums, with
NaN and infinite keys in the rows where the softmax has them; and dQ from
staged dS at row counts around its workgroups' 128 and 256."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rnd(*shape, seed=0):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed))


def _forward(q, k, v, mask, lo, hi, nbytes):
    from avgen_amd import _lib, ops

    B, H, Lq, D = q.shape
    Lk = k.shape[2]
    out, lse = torch.empty_like(q), torch.empty((B, H, Lq), device="cuda")
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")
    st = _lib.load().avattn_fwd_f32_split(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), ops._strides3(q), ops._strides3(k), ops._strides3(v), B, H, H,
        Lq, Lk, D, ops._ptr(mask), 0 if mask is None else Lk, ops._ptr(lo), ops._ptr(hi), 0, 1 / math.sqrt(D),
        out.data_ptr(), ops._strides3(out), lse.data_ptr(), ws.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream)
    assert st == 0
    return out, lse


@pytest.mark.parametrize("variant", ["plain", "mask", "window"])
@pytest.mark.parametrize("B,H,Lq,Lk,D", [(1, 4, 1024, 1024, 64), (2, 2, 129, 517, 128), (1, 33, 2049, 1001, 128),
                                         (1, 24, 4097, 700, 64)])
def test_forward_split_equals_unsplit(B, H, Lq, Lk, D, variant):
    from avgen_amd import _lib, ops

    lib = _lib.load()
    need = lib.avattn_fwd_f32_split_workspace_size(B, H, Lq, Lk, D)
    assert need > 0
    q, k, v = _rnd(B, H, Lq, D, seed=1), _rnd(B, H, Lk, D, seed=2), _rnd(B, H, Lk, D, seed=3)
    mask = lo = hi = None
    if variant == "mask":
        mask = torch.rand(B, Lk, device="cuda", generator=torch.Generator(device="cuda").manual_seed(4)) > 0.3
        mask[:, : Lk // 2] = False  # parts without an attended key
        mask[-1, :] = B == 1
        mask = mask.view(torch.uint8)
    if variant == "window":
        row = torch.arange(Lq, device="cuda")
        lo = (row * Lk // (2 * Lq)).int()
        hi = (lo + row % 97).clamp(max=Lk).int()  # some empty
    (o1, l1), (o2, l2) = (_forward(q, k, v, mask, lo, hi, nbytes) for nbytes in (need, 0))
    # sums of up to Lk terms in another order: sqrt(Lk) * 2^-24 of |v| <= 6, with margin
    assert (o1 - o2).abs().max() <= 2e-5
    assert torch.equal(l1 == float("-inf"), l2 == float("-inf"))
    f = torch.isfinite(l2)
    assert (l1[f] - l2[f]).abs().max() <= 1e-5


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("variant", ["plain", "mask", "window"])
@pytest.mark.parametrize("keys", ["part", "first tile", "last key", "every key"])
@pytest.mark.parametrize("H,Lq,Lk,D", [(4, 1024, 1024, 64), (2, 129, 517, 128)])
def test_not_finite_keys_reach_their_rows(H, Lq, Lk, D, keys, variant, value, split):
    """A NaN or infinite key, alone in its part (or tile) or beside finite
    ones, gives exactly the rows that the softmax of the scores makes NaN."""
    from avgen_amd import _lib

    need = _lib.load().avattn_fwd_f32_split_workspace_size(1, H, Lq, Lk, D)
    assert need > 0
    q, k, v = _rnd(1, H, Lq, D, seed=1), _rnd(1, H, Lk, D, seed=2), _rnd(1, H, Lk, D, seed=3)
    sl = {"part": slice(256, 384), "first tile": slice(0, 32), "last key": slice(Lk - 1, Lk),
          "every key": slice(0, Lk)}[keys]
    k[0, H - 1, sl, 5] = value
    mask = lo = hi = None
    allowed = torch.ones(Lq, Lk, dtype=torch.bool, device="cuda")
    if variant == "mask":  # the keys in question and one more tile masked
        mask = torch.ones(1, Lk, dtype=torch.uint8, device="cuda")
        mask[:, sl] = 0
        mask[:, 64:96] = 0
    if variant == "window":
        row = torch.arange(Lq, device="cuda")
        lo = (row * Lk // (2 * Lq)).int()
        hi = (lo + row % 397).clamp(max=Lk).int()
        key = torch.arange(Lk, device="cuda")
        allowed = (key >= lo[:, None]) & (key < hi[:, None])
    out, lse = _forward(q, k, v, mask, lo, hi, need if split else 0)
    s = q.double() @ k.double().transpose(-1, -2) / math.sqrt(D)
    if mask is not None:  # added to the scores: a NaN or +inf one stays or becomes NaN
        s = s + torch.where(mask[0] != 0, 0.0, float("-inf"))
    s = s.masked_fill(~allowed, float("-inf"))
    nan = s.isnan().any(-1) | (s == float("inf")).any(-1)
    empty = (s == float("-inf")).all(-1)
    assert torch.equal(out.isnan().any(-1), nan) and torch.equal(out.isnan().all(-1), nan)
    assert torch.equal(lse.isnan(), nan)
    assert (out[empty] == 0).all() and torch.equal(lse == float("-inf"), empty)
    ok = ~nan & ~empty
    if not ok.any():
        return
    # sums of up to Lk terms of size |v| <= 6 in fp32
    assert (out.double() - s.softmax(-1) @ v.double())[ok].abs().max() <= 2e-5
    assert (lse.double() - s.logsumexp(-1))[ok].abs().max() <= 1e-5


@pytest.mark.parametrize("variant", ["plain", "mask", "window"])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lk,D", [(45, 45, 200, 700, 64), (66, 33, 97, 1100, 128)])
def test_backward_split_equals_unsplit(Hq, Hkv, Lq, Lk, D, variant):
    from avgen_amd import _lib, ops

    lib = _lib.load()
    q, do = _rnd(1, Hq, Lq, D, seed=1), _rnd(1, Hq, Lq, D, seed=2)
    k, v = _rnd(1, Hkv, Lk, D, seed=3), _rnd(1, Hkv, Lk, D, seed=4)
    mask = windows = None
    if variant == "mask":
        mask = torch.arange(Lk, device="cuda")[None] % 5 != 2
    if variant == "window":
        row = torch.arange(Lq, device="cuda")
        lo = (row * Lk // (2 * Lq)).int()
        windows = (lo, (lo + Lk // 3).clamp(max=Lk).int(), 0)
    s = 1 / math.sqrt(D)
    out, lse = ops._fwd_f32_launch("t", q, k, v, *(windows or (None, None, 0)), mask, s)
    staged = lib.avattn_bwd_f32_staged_workspace_size(1, Hq, Hkv, Lq, Lk, Hkv)
    split = lib.avattn_bwd_f32_split_workspace_size(1, Hq, Hkv, Lq, Lk, D)
    assert split > staged
    got = ops._bwd_f32_impl("t", do, q, k, v, out, lse, mask, s, windows=windows)
    real = ops._alloc_bwd_f32_workspace
    ops._alloc_bwd_f32_workspace = lambda *a: torch.empty(staged, dtype=torch.uint8, device="cuda")
    try:
        ref = ops._bwd_f32_impl("t", do, q, k, v, out, lse, mask, s, windows=windows)
    finally:
        ops._alloc_bwd_f32_workspace = real
    assert torch.equal(got[0], ref[0])  # dq does not depend on the split
    for a, b in zip(got[1:], ref[1:]):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    if mask is not None:
        assert (got[1][:, :, ~mask[0]] == 0).all() and (got[2][:, :, ~mask[0]] == 0).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,Lq", [(4, 1), (4, 31), (4, 33), (4, 127), (4, 128), (4, 129), (4, 257),
                                  (200, 129), (200, 256), (100, 257), (66, 515)])  # 256-row workgroups
def test_dq_rows(H, Lq, D):
    from avgen_amd import ops

    q, do = _rnd(1, H, Lq, D, seed=1), _rnd(1, H, Lq, D, seed=2)
    k, v = _rnd(1, H // 2, 75, D, seed=3), _rnd(1, H // 2, 75, D, seed=4)
    s = 1 / math.sqrt(D)
    out, lse = ops.flash_fwd(q, k, v, None, None, None, s)
    dq = ops.flash_bwd(do, q, k, v, out, lse, None, s)[0]
    qd, kd, vd = q.double(), k.double().repeat_interleave(2, 1), v.double().repeat_interleave(2, 1)
    p = (qd @ kd.transpose(-1, -2) * s).softmax(-1)
    dp = do.double() @ vd.transpose(-1, -2)
    ref = (p * (dp - (p * dp).sum(-1, keepdim=True)) * s) @ kd
    assert (dq - ref).abs().max() <= 1e-5 * ref.abs().max() + 1e-6
    lo, hi = torch.zeros(Lq, dtype=torch.int32, device="cuda"), torch.full((Lq,), 75, dtype=torch.int32, device="cuda")
    windowed = ops.flash_bwd_windowed(do, q, k, v, out, lse, lo, hi, None, s, monotone=True)[0]
    assert torch.equal(windowed, dq)
