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


@pytest.mark.parametrize("staged", [True, False])
@pytest.mark.parametrize("shared", ["q", "dO", "both"])
@pytest.mark.parametrize("first", ["dense", "shared"])
def test_kept_query_side_serves_another_layout(first, shared, staged):
    """A call that reuses the query side may pass the same values in another
    layout, rows sharing memory among them."""
    from avgen_amd import _lib, ops

    B, H, Lq, Lk, D = 1, 2, 130, 150, 64
    g = torch.Generator(device="cuda").manual_seed(5)

    def rnd(*shape):
        return torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)

    q, do, k, v = rnd(B, H, 1, D), rnd(B, H, 1, D), rnd(B, H, Lk, D), rnd(B, H, Lk, D)
    layouts = {"dense": [t.expand(B, H, Lq, D).contiguous() for t in (do, q)]}
    layouts["shared"] = [t.expand(B, H, Lq, D) if shared in (n, "both") else d
                         for n, t, d in zip(("dO", "q"), (do, q), layouts["dense"])]
    second = "shared" if first == "dense" else "dense"
    s = 1.0 / math.sqrt(D)
    out, lse = ops.flash_fwd(layouts["dense"][1], k, v, None, None, None, s)
    want = _bwd(*layouts["dense"], k, v, out, lse, staged)
    lib = _lib.load()
    need = (lib.avattn_bwd_staged_workspace_size(B, H, H, Lq, Lk, D, B * H) if staged
            else lib.avattn_bwd_workspace_size(B, H, H, Lq, Lk, D))
    ws = torch.full((need,), 255, dtype=torch.uint8, device="cuda")
    for name, reuse in ((first, False), (second, True)):
        got = ops._bwd_impl(*layouts[name], k, v, out, lse, None, s, workspace=ws, reuse_query_side=reuse,
                            stage_ds=staged)
        for label, a, b in zip(("dq", "dk", "dv"), got, want):
            assert torch.equal(a, b), (name, label)
