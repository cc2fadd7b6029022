"""A call without grad rotates k inside the forward's copy of it: the bits of
rotating k first, over layouts, tails, masks and per-sample tables; the errors
stay those of the composition."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(B, H, Hkv, Lq, Lk, D, layout, table_batch):
    g = torch.Generator(device="cuda").manual_seed(Lq * 1000 + Lk)

    def rnd(n, length):
        if layout == "blhd":
            return torch.randn(B, length, n, D, device="cuda", generator=g).bfloat16().transpose(1, 2)
        if layout == "shared":  # one sample's rows under batch stride 0
            return torch.randn(1, n, length, D, device="cuda", generator=g).bfloat16().expand(B, -1, -1, -1)
        if layout == "offset":  # rows not 16-byte aligned
            return torch.randn(B, n, length, D + 4, device="cuda", generator=g).bfloat16()[..., 4:]
        return torch.randn(B, n, length, D, device="cuda", generator=g).bfloat16()

    def tables(length):
        from avgen_amd.rope import RotaryTables

        ang = torch.randn(table_batch, 1, length, D // 2, device="cuda", generator=g)
        return RotaryTables(ang.cos(), ang.sin())

    return rnd(H, Lq), rnd(Hkv, Lk), rnd(Hkv, Lk), tables(Lq), tables(Lk)


@pytest.mark.parametrize("layout", ["bhld", "blhd", "shared", "offset"])
@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,D,tb", [
    (1, 1, 1, 2, 3, 64, 1), (2, 4, 2, 63, 65, 64, 2), (2, 4, 4, 257, 64, 128, 1), (1, 8, 2, 130, 700, 128, 1),
])
@pytest.mark.parametrize("masked", [False, True])
def test_same_bits_as_rotating_k_first(B, H, Hkv, Lq, Lk, D, tb, layout, masked):
    from avgen_amd import attention as A
    from avgen_amd import ops

    q, k, v, tq, tk = _case(B, H, Hkv, Lq, Lk, D, layout, tb)
    mask = (torch.arange(Lk, device="cuda")[None] < max(1, Lk // 3)).expand(B, -1) if masked else None
    with torch.no_grad():
        out = A.rotary_attention(q, k, v, tq, key_tables=tk, enable_gqa=True,
                                 attn_mask=None if mask is None else mask[:, None, None, :])
        k_rot = ops.rope_apply(k, tk.cos, tk.sin, False)
        ref, _ = ops.flash_fwd(q, k_rot, v, mask, tq.cos, tq.sin, ops.default_scale(D))
    assert torch.equal(out, ref)
    with torch.enable_grad():  # the composition, which autograd sees
        grad = A.rotary_attention(q, k.clone().requires_grad_(True), v, tq, key_tables=tk, enable_gqa=True,
                                  attn_mask=None if mask is None else mask[:, None, None, :])
    assert grad.requires_grad and torch.equal(grad.detach(), ref)


@pytest.mark.parametrize("layout", ["bhld", "blhd", "shared", "offset"])
@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,D,tb", [(1, 1, 1, 1, 2, 64, 1), (2, 4, 2, 63, 165, 64, 2),
                                                (1, 3, 1, 257, 31, 128, 1)])
def test_float32_pair_has_the_bits_of_two_rotations(B, H, Hkv, Lq, Lk, D, tb, layout):
    from avgen_amd import attention as A
    from avgen_amd import ops

    q, k, v, tq, tk = _case(B, H, Hkv, Lq, Lk, D, layout, tb)
    q, k, v = q.float(), k.float(), v.float()
    mask = torch.arange(Lk, device="cuda")[None] < max(1, Lk // 2)
    with torch.no_grad():
        out = A.rotary_attention(q, k, v, tq, key_tables=tk, enable_gqa=True, attn_mask=mask[:, None, None, :])
        qr, kr = ops.rope_apply(q, tq.cos, tq.sin, False), ops.rope_apply(k, tk.cos, tk.sin, False)
        ref, _ = ops.flash_fwd(qr, kr, v, mask, None, None, ops.default_scale(D))
    assert torch.equal(out, ref)


def test_errors_are_those_of_the_composition():
    from avgen_amd import attention as A
    from avgen_amd.rope import RotaryTables

    q, k, v, tq, tk = _case(1, 2, 2, 64, 96, 64, "bhld", 1)
    with torch.no_grad():
        with pytest.raises(ValueError, match="rope_apply: sequence length 96 does not match"):
            A.rotary_attention(q, k, v, tq)
        with pytest.raises(TypeError, match="rope_apply: rotary tables must be float32"):
            A.rotary_attention(q, k, v, tq, key_tables=RotaryTables(tk.cos.double(), tk.sin.double()))
        with pytest.raises(TypeError):
            A.rotary_attention(q.float(), k, v, tq, key_tables=tk)
        with pytest.raises(TypeError):
            A.rotary_attention(q, k.float(), v.float(), tq, key_tables=tk)
        with pytest.raises(ValueError, match="rope_apply: sequence length 64 does not match"):
            A.rotary_attention(q.float(), k.float(), v.float(), tk, key_tables=tk)


def test_key_tables_are_checked_at_the_c_entry():
    from avgen_amd import _lib, ops

    q, k, v, tq, tk = _case(1, 2, 2, 64, 96, 64, "bhld", 1)
    out, lse = torch.empty_like(q), torch.empty(1, 2, 64, device="cuda")
    lib = _lib.load()
    ws = ops._workspace(lib.avattn_fwd_workspace_size(1, 2, 96, 64), q.device)

    def call(cos_k, sin_k, stride):
        return lib.avattn_fwd_rotary(q.data_ptr(), k.data_ptr(), v.data_ptr(), ops._strides3(q), ops._strides3(k),
                                     ops._strides3(v), 1, 2, 2, 64, 96, 64, None, 0, tq.cos.data_ptr(),
                                     tq.sin.data_ptr(), 0, cos_k, sin_k, stride, 0.125, out.data_ptr(),
                                     ops._strides3(out), lse.data_ptr(), ws.data_ptr(), ws.numel(),
                                     torch.cuda.current_stream().cuda_stream)

    c, s = tk.cos.data_ptr(), tk.sin.data_ptr()
    assert call(c, None, 0) != _lib.OK and call(c + 4, s, 0) != _lib.OK and call(c, s, 2) != _lib.OK
    assert call(c, s, 0) == _lib.OK
    torch.cuda.synchronize()
