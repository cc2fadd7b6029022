"""The forward at both workgroup sizes (128 and 256 query rows): last rows and
last key tiles of either, on each side of the limits that choose between them,
with key masks, key windows and the rotation of q, against float32."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["plain", "mask", "window", "rope"])
@pytest.mark.parametrize("H,Lq,Lk,D", [
    (300, 1, 513, 128),      # 300 workgroups of 256 rows, one row each
    (52, 1281, 577, 128),    # six per head, the last of one row; last key tile of one
    (52, 1281, 512, 128),    # few keys: 128 rows
    (256, 256, 640, 128),    # one workgroup of 256 rows per CU
    (257, 256, 640, 128),
    (128, 255, 640, 128),    # at most one workgroup of 128 rows per CU: 128 rows
    (129, 255, 640, 128),
    (4, 300, 1024, 128),     # ... and up to 1,024 keys
    (4, 300, 1025, 128),
    (3, 129, 1, 128),
    (40, 385, 130, 64),
])
def test_forward_against_float32(H, Lq, Lk, D, variant):
    from avgen_amd import ops

    g = torch.Generator(device="cuda").manual_seed(H + Lq)

    def rnd(*shape):
        return torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)

    q, k, v = rnd(1, H, Lq, D), rnd(1, H, Lk, D), rnd(1, H, Lk, D)
    scale = 1.0 / math.sqrt(D)
    allowed = torch.ones(Lq, Lk, dtype=torch.bool, device="cuda")
    qf = q.float()
    if variant == "mask":
        mask = torch.arange(Lk, device="cuda") % 7 != 3
        allowed &= mask
        out, lse = ops.flash_fwd(q, k, v, mask[None], None, None, scale)
    elif variant == "window":
        row = torch.arange(Lq, device="cuda")
        lo = (row * Lk // (2 * Lq)).int()
        hi = (lo + 1 + row * Lk // (3 * Lq)).clamp(max=Lk).int()
        key = torch.arange(Lk, device="cuda")
        allowed &= (key >= lo[:, None]) & (key < hi[:, None])
        out, lse = ops.flash_fwd_windowed(q, k, v, lo, hi, None, scale)
    elif variant == "rope":
        ang = torch.randn(1, 1, Lq, D // 2, device="cuda", generator=g)
        out, lse = ops.flash_fwd(q, k, v, None, ang.cos(), ang.sin(), scale)
        qf = ops.rope_apply(q, ang.cos(), ang.sin(), False).float()
    else:
        out, lse = ops.flash_fwd(q, k, v, None, None, None, scale)
    s = (qf @ k.float().transpose(-1, -2) * scale).masked_fill(~allowed, float("-inf"))
    # bf16 P and output: 2^-9 relative each, |out| <= max|v| < 6
    assert (out.float() - s.softmax(-1) @ v.float()).abs().max() <= 2e-2
    assert (lse - s.logsumexp(-1)).abs().max() <= 1e-3
