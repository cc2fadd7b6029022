"""The forward with its last round split over ranges of keys against the
unsplit one, at every entry point that splits: the same result up to the
rounding of the merge, and the row states (no attended key, NaN) merged
exactly."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(lib, q, k, v, mask, nbytes):
    from avgen_amd import ops

    B, H, Lq, D = q.shape
    out, lse = torch.empty_like(q), torch.empty((B, H, Lq), device="cuda")
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    st = lib.avattn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), ops._strides3(q), ops._strides3(k), ops._strides3(v),
                        B, H, k.shape[1], Lq, k.shape[2], D, None if mask is None else mask.data_ptr(),
                        0 if mask is None else mask.stride(0), None, None, 0, 1.0 / math.sqrt(D), out.data_ptr(),
                        ops._strides3(out), lse.data_ptr(), ws.data_ptr(), ws.numel(),
                        torch.cuda.current_stream().cuda_stream)
    assert st == 0
    return out, lse


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,H,Lq,Lk,D", [
    (1, 4, 1024, 4096, 64),     # every block split
    (2, 2, 1000, 4097, 128),    # ragged rows and keys
    (1, 16, 4725, 5000, 128),   # full rounds of 256-row blocks, then a split one
    (1, 31, 3201, 2049, 64),
])
def test_split_equals_unsplit(B, H, Lq, Lk, D, masked):
    from avgen_amd import _lib

    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(Lq)
    q, k, v = (torch.randn(B, H, n, D, device="cuda", generator=g).to(torch.bfloat16) for n in (Lq, Lk, Lk))
    k[:, :, -1] *= 4  # a late key raises the reference max of the last part only
    mask = None
    if masked:
        mask = torch.rand(B, Lk, device="cuda", generator=g) > 0.3
        mask[:, : Lk // 2] = False  # parts without an attended key
        if B > 1:
            mask[1] = False
        mask = mask.view(torch.uint8)
    if not masked:
        q[0, 0, 5, 3] = float("nan")
    base = lib.avattn_fwd_workspace_size(B, H, Lk, D)
    split = lib.avattn_fwd_split_workspace_size(B, H, H, Lq, Lk, D, 0)
    assert split > base
    (o1, l1), (o2, l2) = _call(lib, q, k, v, mask, split), _call(lib, q, k, v, mask, base)
    assert torch.equal(o1.isnan(), o2.isnan()) and torch.equal(l1.isnan(), l2.isnan())
    assert torch.equal(l1 == float("-inf"), l2 == float("-inf"))
    # one bf16 rounding of P (2^-9 of each term) and of the output apart
    d = (o1.float() - o2.float()).nan_to_num(0.0).abs()
    assert (d <= 2.0**-7 * o2.float().nan_to_num(0.0).abs() + 2.0**-8).all()
    f = torch.isfinite(l2)
    assert (l1[f] - l2[f]).abs().max() <= 1e-5 * l2[f].abs().max() if f.any() else True
    if masked and B > 1:
        assert (o1[1] == 0).all()
    assert torch.equal(_call(lib, q, k, v, mask, split)[0].view(torch.int16), o1.view(torch.int16))


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kind", ["rotated", "fp8", "ring first", "ring merge"])
def test_entry_points_split_equals_unsplit(kind, D, masked):
    """Grouped heads, q rotated, e4m3 scores (their own merge constants) and the
    ring's fp32 accumulator, with parts that hold no attended key."""
    from avgen_amd import _lib, ops

    lib = _lib.load()
    B, Hq, Hkv, Lq, Lk = 2, 4, 2, 700, 4097
    g = torch.Generator(device="cuda").manual_seed(D)

    def rnd(*shape):
        return torch.randn(shape, device="cuda", generator=g)

    q, k, v = rnd(B, Hq, Lq, D).bfloat16(), rnd(B, Hkv, Lk, D).bfloat16(), rnd(B, Hkv, Lk, D).bfloat16()
    if kind == "fp8":
        k[:, :, -1] *= 2  # the last part's reference is the largest
    else:
        q[0, 0, 5, 3] = float("nan")
    mask = None
    if masked:
        mask = rnd(B, Lk) > -0.5
        mask[:, : Lk // 2] = False
        mask[1] = False
        mask = mask.view(torch.uint8)
    ang, angk = rnd(1, 1, Lq, D // 2), rnd(1, 1, Lk, D // 2)
    tables = [t.contiguous() for t in (ang.cos(), ang.sin(), angk.cos(), angk.sin())]
    qs, ks = (ops.fp8_absmax_scales(q), ops.fp8_absmax_scales(k)) if kind == "fp8" else (None, None)
    acc0, lse0 = rnd(B, Hq, Lq, D), rnd(B, Hq, Lq)
    lse0[:, :, ::3] = float("-inf")  # rows nothing was merged into yet
    stream = torch.cuda.current_stream().cuda_stream
    fp8 = int(kind == "fp8")
    base = (lib.avattn_fwd_fp8_workspace_size if fp8 else lib.avattn_fwd_workspace_size)(B, Hkv, Lk, D)
    split = lib.avattn_fwd_split_workspace_size(B, Hq, Hkv, Lq, Lk, D, fp8)
    assert split > base

    def call(nbytes):
        out, lse = torch.empty_like(q), torch.empty((B, Hq, Lq), device="cuda")
        acc, lacc = acc0.clone(), lse0.clone()
        ws = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")
        head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), ops._strides3(q), ops._strides3(k), ops._strides3(v), B, Hq,
                Hkv, Lq, Lk, D, ops._ptr(mask), 0 if mask is None else Lk)
        s = 1.0 / math.sqrt(D)
        cq, sq, ck, sk = (t.data_ptr() for t in tables)
        if kind == "rotated":
            st = lib.avattn_fwd_rotary(*head, cq, sq, 0, ck, sk, 0, s, out.data_ptr(), ops._strides3(out),
                                       lse.data_ptr(), ws.data_ptr(), nbytes, stream)
        elif kind == "fp8":
            st = lib.avattn_fwd_fp8(*head, qs.data_ptr(), ks.data_ptr(), s, out.data_ptr(), ops._strides3(out),
                                    lse.data_ptr(), ws.data_ptr(), nbytes, stream)
        else:
            flags = _lib.RING_LAST | (_lib.RING_FIRST if kind == "ring first" else 0)
            st = lib.avattn_ring_fwd_step(*head, cq, sq, 0, ck, sk, 0, s, acc.data_ptr(), lacc.data_ptr(),
                                          out.data_ptr(), ops._strides3(out), flags, ws.data_ptr(), nbytes, stream)
            lse = lacc
        assert st == 0
        return out, lse, acc

    (o1, l1, a1), (o2, l2, a2) = call(split), call(base)
    assert torch.equal(o1.isnan(), o2.isnan()) and torch.equal(l1.isnan(), l2.isnan())
    assert torch.equal(l1 == float("-inf"), l2 == float("-inf"))
    # as test_split_equals_unsplit; the ring adds the running output, exactly
    d = (o1.float() - o2.float()).nan_to_num(0.0).abs()
    assert (d <= 2.0**-7 * o2.float().nan_to_num(0.0).abs() + 2.0**-8).all()
    if kind.startswith("ring"):
        d = (a1 - a2).nan_to_num(0.0).abs()
        assert (d <= 2.0**-7 * a2.nan_to_num(0.0).abs() + 2.0**-8).all()
    f = torch.isfinite(l2)
    assert (l1[f] - l2[f]).abs().max() <= 1e-5 * l2[f].abs().max()
    if masked and kind != "ring merge":
        rows = ~o1[1].isnan().any(-1)
        assert (o1[1][rows] == 0).all() and (l1[1][rows] == float("-inf")).all()


@pytest.mark.parametrize("kind", ["bf16", "fp8", "ring", "f32"])
def test_runs_unsplit_where_the_parts_do_not_fit(kind, monkeypatch):
    """The parts' room is optional: an allocator that has the base workspace
    only gives the unsplit call's bits."""
    from avgen_amd import _lib, ops, ring
    from avgen_amd.rope import RotaryTables

    lib = _lib.load()
    B, H, L, D = 1, 4, 2048, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(B, H, L, D, device="cuda", generator=g) for _ in range(3))
    if kind != "f32":
        q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    s = 1.0 / math.sqrt(D)
    ang = torch.randn(1, 1, L, D // 2, device="cuda", generator=g)
    tables = RotaryTables(ang.cos(), ang.sin())

    def call():
        with torch.no_grad():
            if kind == "fp8":
                qs, ks = ops.fp8_absmax_scales(q), ops.fp8_absmax_scales(k)
                return ops.flash_fwd_fp8(q, k, v, None, qs, ks, s)
            if kind == "ring":
                return ring.ring_attention(q, k, v, cp=1, tables_q=tables, tables_k=tables)
            return ops.flash_fwd(q, k, v, None, None, None, s)

    base = {"bf16": lib.avattn_fwd_workspace_size(B, H, L, D), "ring": lib.avattn_fwd_workspace_size(B, H, L, D),
            "fp8": lib.avattn_fwd_fp8_workspace_size(B, H, L, D), "f32": 256}[kind]
    real, sizes = ops._workspace, []

    def small(nbytes, device):
        sizes.append(nbytes)
        if nbytes > base:
            raise torch.OutOfMemoryError("no room for the parts")
        return real(nbytes, device)

    monkeypatch.setattr(ops, "_workspace", small)
    got = call()
    assert len(sizes) == 2 and sizes[0] > base >= sizes[1]
    monkeypatch.setattr(ops, "_workspace", real)
    name = "avattn_fwd_f32_split_workspace_size" if kind == "f32" else "avattn_fwd_split_workspace_size"
    monkeypatch.setattr(lib, name, lambda *a: 0 if kind == "f32" else base)
    for a, b in zip(got, call()):
        assert torch.equal(a, b)
