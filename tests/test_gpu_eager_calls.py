"""Plain eager calls skip the dispatcher's op layers; everything those layers
serve still sees the ops, and both ways give the same bits."""

import math

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.namespace == "avgen_amd":
            self.names.append(func.name().split("::")[1])
        return func(*args, **(kwargs or {}))


def _inputs(dtype):
    g = torch.Generator(device="cuda").manual_seed(0)

    def rnd(*shape):
        return torch.randn(shape, device="cuda", generator=g).to(dtype)

    ang = rnd(1, 1, 96, 32).float()
    return dict(q=rnd(1, 4, 96, 64), k=rnd(1, 2, 96, 64), v=rnd(1, 2, 96, 64), w=rnd(64), cos=ang.cos(),
                sin=ang.sin(), do=rnd(1, 4, 96, 64), lo=torch.zeros(96, dtype=torch.int32, device="cuda"),
                hi=torch.full((96,), 70, dtype=torch.int32, device="cuda"))


def _calls():
    from avgen_amd import ops, ring
    from avgen_amd.rope import RotaryTables

    s = 1.0 / math.sqrt(64)
    return {
        "flash_fwd": lambda x: ops.flash_fwd(x["q"], x["k"], x["v"], None, x["cos"], x["sin"], s)[0],
        "flash_fwd_windowed": lambda x: ops.flash_fwd_windowed(x["q"], x["k"], x["v"], x["lo"], x["hi"], None, s)[0],
        "qk_norm_rope": lambda x: ops.qk_norm_rope(x["q"], x["w"], 1e-6, x["cos"], x["sin"]),
        "rope_apply": lambda x: ops.rope_apply(x["q"], x["cos"], x["sin"], False),
        "ring_attention_rope": lambda x: ring.ring_attention(
            x["q"], x["k"], x["v"], cp=2, tables_q=RotaryTables(x["cos"], x["sin"]),
            tables_k=RotaryTables(x["cos"], x["sin"]))[0],
    }


NAMES = ["flash_fwd", "flash_fwd_windowed", "qk_norm_rope", "rope_apply", "ring_attention_rope"]


def _run(name, x):
    leaves = {n: x[n].detach().clone().requires_grad_(True) for n in ("q", "k", "v", "w")}
    out = _calls()[name]({**x, **leaves})
    grads = torch.autograd.grad(out, list(leaves.values()), x["do"], allow_unused=True)
    return [out.detach()] + [g for g in grads if g is not None]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", NAMES)
def test_both_ways_give_the_same_bits(name, dtype):
    if name == "ring_attention_rope" and dtype is torch.float32:
        pytest.skip("float32 rings run per chunk")
    x = _inputs(dtype)
    eager = _run(name, x)
    with Seen() as seen:
        through_ops = _run(name, x)
    assert name in seen.names  # a dispatch mode sees the op, in the forward
    assert len(seen.names) >= 2  # ... and in the backward
    assert len(eager) == len(through_ops)
    for a, b in zip(eager, through_ops):
        assert torch.equal(a, b)
    with torch.no_grad():
        assert torch.equal(_calls()[name](x), eager[0])
    with torch.inference_mode():
        assert torch.equal(_calls()[name](x), eager[0])


@pytest.mark.parametrize("name", NAMES)
def test_saved_tensor_hooks_and_no_second_order(name):
    x = _inputs(torch.bfloat16)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.cuda()):
        got = _run(name, x)
    assert packed
    for a, b in zip(got, _run(name, x)):
        assert torch.equal(a, b)
    if name == "rope_apply":
        return  # its backward is itself differentiable
    q = x["q"].clone().requires_grad_(True)
    out = _calls()[name]({**x, "q": q})
    with pytest.raises(RuntimeError):
        (g,) = torch.autograd.grad(out, q, x["do"].clone().requires_grad_(True), create_graph=True)
        torch.autograd.grad(g.float().sum(), q)


@pytest.mark.parametrize("name", NAMES)
def test_batched_gradients_use_the_ops(name, monkeypatch):
    from avgen_amd import ops

    x = _inputs(torch.bfloat16)
    q = x["q"].clone().requires_grad_(True)
    out = _calls()[name]({**x, "q": q})
    ref = [torch.autograd.grad(out, q, d, retain_graph=True)[0] for d in (x["do"], 2 * x["do"])]
    real, batched = ops._plain_eager, []

    def spy(*tensors):
        plain = real(*tensors)
        if any(t is not None and "Batched" in str(torch._C._dispatch_keys(t)) for t in tensors):
            batched.append(plain)
        return plain

    monkeypatch.setattr(ops, "_plain_eager", spy)
    got = torch.autograd.grad(out, q, torch.stack([x["do"], 2 * x["do"]]), is_grads_batched=True)[0]
    assert batched and not any(batched)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])


def test_profiled_calls_use_the_ops():
    x = _inputs(torch.bfloat16)
    with torch.autograd.profiler.profile() as prof:
        _run("flash_fwd", x)
    assert any("avgen_amd::flash_fwd" in e.name for e in prof.function_events)


def test_a_profile_of_the_ring_names_its_steps():
    x = _inputs(torch.bfloat16)
    want = _run("ring_attention_rope", x)
    with torch.autograd.profiler.profile() as prof:
        got = _run("ring_attention_rope", x)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    names = [e.name for e in prof.function_events]
    for name, count in (("ring_fwd_step", 2), ("ring_bwd_step", 2), ("ring_dq_finish", 1)):
        assert names.count(f"avgen_amd::{name}") == count, name
