"""Performance cases of the video-DiT attention path.

Each case is one call (forward, or forward and backward) that a training or
sampling program makes through the package's public entry points, with the
inputs, rotation tables, masks and plans it holds beforehand.  ``listed()``
names a fixed set, ``draw(rng)`` gives further cases of the same ranges;
``prepare`` / ``run`` / ``exact`` make a case's inputs, run it and compute the
same outputs in float64 with plain torch operations.

Kinds (``case["kind"]``):

* ``rotary``  rotary_attention, forward only (sampling), bf16 or float32;
* ``block``   self_attention_core: head split, q/k RMSNorm + rotation,
  attention, flatten; forward and backward (a DiT block in training);
* ``ring``    ring_attention with rotation over ``cp`` KV chunks, forward and
  backward; with ``text`` slots at its end and a key-padding mask it is the
  joint text+video attention;
* ``cross``   attention over text keys with a key-padding mask, forward and
  backward;
* ``window``  temporal_neighbour_attention, forward and backward;
* ``varlen``  varlen_attention over packed clips, forward and backward;
* ``fp8``     attention_fp8, forward only (sampling).
"""

from __future__ import annotations

import math

import torch

from avgen_amd import attention as A
from avgen_amd import layers, ring
from avgen_amd.rope import RotaryTables

FPS = 8.0  # latent frames per second of the coordinate grids


def listed():
    """The fixed cases, smallest first."""
    return [
        # The smoke configuration: one float32 forward over a 4x16x16 latent.
        dict(name="smoke_f32", kind="rotary", dtype="float32", B=1, H=4, Hkv=4, D=64, F=4, Y=16, X=16),
        # A block of a small model in training: 4x16x16 latent, 4 heads of 64.
        dict(name="block_small", kind="block", dtype="bfloat16", B=1, H=4, Hkv=4, D=64, F=4, Y=16, X=16),
        # One latent frame (an image) sampled with a guidance pair.
        dict(name="image_sample", kind="rotary", dtype="bfloat16", B=2, H=20, Hkv=20, D=128, F=1, Y=45, X=80),
        # A short low-resolution clip in training; 13x15x27 tokens fill no tile.
        dict(name="block_clip", kind="block", dtype="bfloat16", B=1, H=20, Hkv=20, D=128, F=13, Y=15, X=27),
        # A full DiT block in training: 16x32x32 latent, 2 samples, 20 heads.
        dict(name="block_full", kind="block", dtype="bfloat16", B=2, H=20, Hkv=20, D=128, F=16, Y=32, X=32),
        # One rank's share of a 21x45x80 latent split over 4 ranks.
        dict(name="ring_share", kind="ring", dtype="bfloat16", B=1, H=40, Hkv=40, D=128, F=21, Y=45, X=80, cp=4,
             shard=18900, text=0, text_lens=""),
        # Joint text+video attention over 6 latent frames and 512 text slots.
        dict(name="joint", kind="ring", dtype="bfloat16", B=1, H=40, Hkv=40, D=128, F=6, Y=45, X=80, cp=1,
             shard=22112, text=512, text_lens="301"),
        # Cross-attention of a 21x45x80 latent into its text; the second row
        # is the unconditional sample (no text).
        dict(name="cross", kind="cross", dtype="bfloat16", B=2, H=40, Hkv=40, D=128, Lq=75600, Lk=512,
             text_lens="388,0"),
        # Temporal neighbourhoods: keys within 0.25 s over 12 latent frames.
        dict(name="window", kind="window", dtype="bfloat16", B=1, H=20, Hkv=20, D=128, F=12, P=1800, seconds=0.25),
        # Clips of 8/6/4/2.5 frames of 45x40 packed with some padding.
        dict(name="varlen", kind="varlen", dtype="bfloat16", B=1, H=20, Hkv=20, D=128, L=37800,
             segments="14400,10800,7200,4500"),
        # Sampling with fp8 q k^T, a guidance pair over 5 latent frames.
        dict(name="sample_fp8", kind="fp8", dtype="bfloat16", B=2, H=40, Hkv=40, D=128, Lq=18000, Lk=18000),
        # A float32 block's attention in training (its own fp32 kernels).
        dict(name="train_f32", kind="ring", dtype="float32", B=1, H=20, Hkv=20, D=128, F=4, Y=32, X=32, cp=1,
             shard=4096, text=0, text_lens=""),
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _fit_heads(rng, pairs_flops, cap, choices=(4, 8, 12, 16, 20, 24, 32, 40)):
    """A head count whose work stays under ``cap`` (``pairs_flops`` per head)."""
    ok = [h for h in choices if h * pairs_flops <= cap] or [choices[0]]
    return rng.choice(ok)


def _heads(rng, per_head, cap):
    h = _fit_heads(rng, per_head, cap)
    return h, h // rng.choice([1, 1, 1, 2, 4])


def draw(rng):
    """One more case of the ranges ``listed()`` stands for."""
    kind = rng.choice(["rotary", "rotary_f32", "block", "block", "ring", "joint", "cross", "window", "varlen", "fp8",
                       "ring_f32"])
    D = rng.choice([64, 128, 128])
    if kind in ("rotary", "rotary_f32", "block"):
        f32 = kind == "rotary_f32"
        F = rng.choice([1, 1, 2, 4, 7, 13, 16])
        yx = _log(rng, 64, 2048) if f32 else _log(rng, 64, 3600)
        Y = max(4, int(math.sqrt(yx * rng.uniform(0.5, 1.0))))
        X = max(4, yx // Y)
        F = max(1, min(F, (6000 if f32 else 18900) // (X * Y)))
        L = F * Y * X
        B = rng.choice([1, 2])
        H, Hkv = _heads(rng, 12.0 * B * L * L * D, 1.0e12 if f32 else 1.7e13)
        return dict(kind="block" if kind == "block" else "rotary", dtype="float32" if f32 else "bfloat16", B=B, H=H,
                    Hkv=Hkv, D=D, F=F, Y=Y, X=X)
    if kind in ("ring", "ring_f32"):
        f32 = kind == "ring_f32"
        cp = rng.choice([1, 2, 4]) if not f32 else 1
        Y = rng.randint(6, 45)
        X = rng.randint(8, 80)
        F = max(cp, min(24, _log(rng, 1024, 5000 if f32 else 18900) // (Y * X)))
        F -= F % cp
        shard = F * Y * X // cp
        H, Hkv = _heads(rng, 12.0 * shard * shard * cp * D, 4.0e12 if f32 else 4.0e13)
        return dict(kind="ring", dtype="float32" if f32 else "bfloat16", B=1, H=H, Hkv=Hkv, D=D, F=F, Y=Y, X=X, cp=cp,
                    shard=shard, text=0, text_lens="")
    if kind == "joint":
        B = rng.choice([1, 2])
        Y = rng.randint(6, 45)
        X = rng.randint(8, 80)
        F = max(1, min(24, _log(rng, 1024, 18900) // (Y * X)))
        text = _log(rng, 77, 512)
        L = F * Y * X + text
        H, Hkv = _heads(rng, 12.0 * B * L * L * D, 3.0e13)
        return dict(kind="ring", dtype="bfloat16", B=B, H=H, Hkv=Hkv, D=D, F=F, Y=Y, X=X, cp=1, shard=L, text=text,
                    text_lens=",".join(str(rng.randint(16, text)) for _ in range(B)))
    if kind == "cross":
        B = rng.choice([1, 2])
        Lq, Lk = _log(rng, 1024, 75600), _log(rng, 77, 512)
        H, Hkv = _heads(rng, 12.0 * B * Lq * Lk * D, 1.0e13)
        return dict(kind="cross", dtype="bfloat16", B=B, H=H, Hkv=Hkv, D=D, Lq=Lq, Lk=Lk,
                    text_lens=",".join(str(0 if b and rng.random() < 0.5 else rng.randint(16, Lk)) for b in range(B)))
    if kind == "window":
        F, P = rng.randint(4, 21), _log(rng, 120, 1800)
        seconds = rng.choice([0.25, 0.25, 0.375, 0.5])
        H, Hkv = _heads(rng, 12.0 * (F * P) ** 2 * D, 6.0e13)
        return dict(kind="window", dtype="bfloat16", B=1, H=H, Hkv=Hkv, D=D, F=F, P=P, seconds=seconds)
    if kind == "varlen":
        n = rng.randint(2, 6)
        seg = [_log(rng, 200, 9000) for _ in range(n)]
        L = sum(seg) + rng.choice([0, rng.randint(1, 900)])
        H, Hkv = _heads(rng, 12.0 * sum(s * s for s in seg) * D, 3.0e13)
        return dict(kind="varlen", dtype="bfloat16", B=1, H=H, Hkv=Hkv, D=D, L=L,
                    segments=",".join(str(s) for s in seg))
    L = _log(rng, 1024, 18900)
    H, Hkv = _heads(rng, 4.0 * 2 * L * L * D, 1.4e13)
    return dict(kind="fp8", dtype="bfloat16", B=2, H=H, Hkv=Hkv, D=D, Lq=L, Lk=L)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _ints(text):
    return [int(t) for t in text.split(",")] if text else []


def _tables(case, device):
    """cos/sin ``(B, 1, length, D/2)`` float32 of the video grid (seconds,
    2*row, 2*column), text slots at zero coordinates: interleaved pairs, a
    third of them each for rows and columns, the rest for time."""
    t = torch.arange(case["F"], dtype=torch.float32, device=device) / FPS
    r = torch.arange(case["Y"], dtype=torch.float32, device=device) * 2.0
    c = torch.arange(case["X"], dtype=torch.float32, device=device) * 2.0
    coords = torch.stack(torch.meshgrid(t, r, c, indexing="ij"), dim=-1).reshape(-1, 3)
    if case.get("text"):
        coords = torch.cat([coords, torch.zeros(case["text"], 3, device=device)])
    pairs = case["D"] // 2
    third = pairs // 3
    angles = []
    for axis, n in enumerate((pairs - 2 * third, third, third)):
        freq = torch.pow(10000.0, -torch.arange(n, dtype=torch.float32, device=device) / n)
        angles.append(coords[:, axis:axis + 1] * freq)
    ang = torch.cat(angles, 1)[None, None].expand(case["B"], -1, -1, -1)
    return ang.cos().contiguous(), ang.sin().contiguous()


def _key_mask(lengths, slots, lead, device):
    """(B, lead + slots) bool: ``lead`` valid keys, then each row's text."""
    n = torch.tensor(lengths, device=device)[:, None]
    text = torch.arange(slots, device=device)[None] < n
    return torch.cat([torch.ones(len(lengths), lead, dtype=torch.bool, device=device), text], 1)


def _inputs(case, seed):
    """The case's tensors from the seed alone: projections of unit-variance
    activations (q, k, v ~ N(0, 1/2)), output gradients ~ N(0, 1), norm gains
    around 1."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    dtype = getattr(torch, case["dtype"])

    def rnd(*shape, scale=math.sqrt(0.5), mean=0.0):
        return (torch.randn(shape, device=dev, generator=gen) * scale + mean).to(dtype)

    B, H, Hkv, D = case["B"], case["H"], case["Hkv"], case["D"]
    kind = case["kind"]
    x = dict(case=case)
    if kind == "block":
        L = case["F"] * case["Y"] * case["X"]
        x.update(q=rnd(B, L, H * D), k=rnd(B, L, Hkv * D), v=rnd(B, L, Hkv * D), do=rnd(B, L, H * D, scale=1.0),
                 wq=rnd(D, scale=0.1, mean=1.0), wk=rnd(D, scale=0.1, mean=1.0))
        x["cos"], x["sin"] = _tables(case, dev)
        return x
    if kind == "rotary":
        Lq = Lk = case["F"] * case["Y"] * case["X"]
    elif kind == "ring":
        Lq, Lk = case["shard"], case["F"] * case["Y"] * case["X"] + case["text"]
    elif kind == "window":
        Lq = Lk = case["F"] * case["P"]
    elif kind == "varlen":
        Lq = Lk = case["L"]
    else:
        Lq, Lk = case["Lq"], case["Lk"]
    x.update(q=rnd(B, H, Lq, D), k=rnd(B, Hkv, Lk, D), v=rnd(B, Hkv, Lk, D))
    if kind not in ("rotary", "fp8"):
        x["do"] = rnd(B, H, Lq, D, scale=1.0)
    if kind in ("rotary", "ring"):
        x["cos"], x["sin"] = _tables(case, dev)
    if kind == "ring" and case["text"]:
        x["mask"] = _key_mask(_ints(case["text_lens"]), case["text"], Lk - case["text"], dev)
    if kind == "cross":
        x["mask"] = _key_mask(_ints(case["text_lens"]), Lk, 0, dev)
    if kind == "window":
        x["seconds"] = (torch.arange(case["F"], dtype=torch.float32, device=dev) / FPS).repeat_interleave(
            case["P"])[None].expand(B, -1).contiguous()
    if kind == "varlen":
        seg = [0] + _ints(case["segments"])
        x["cu"] = torch.tensor(seg, device=dev).cumsum(0).to(torch.int32)
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    for name in ("q", "k", "v", "wq", "wk"):
        if name in x and kind not in ("rotary", "fp8"):
            x[name].requires_grad_(True)
    if "cos" in x:
        x["tables"] = RotaryTables(cos=x["cos"], sin=x["sin"])
        if kind == "ring":
            x["tables_q"] = x["tables"].slice(0, case["shard"])
    if kind == "window":
        # Built once per model forward and used by every block.
        x["neighbourhood"] = A.temporal_neighbourhood(x["seconds"], x["seconds"], window_seconds=case["seconds"])
    return x


def run(x):
    case = x["case"]
    kind, gqa = case["kind"], case["H"] != case["Hkv"]
    q, k, v = x["q"], x["k"], x["v"]
    if kind == "rotary":
        with torch.no_grad():
            return A.rotary_attention(q, k, v, x["tables"], enable_gqa=gqa)
    if kind == "fp8":
        with torch.no_grad():
            return A.attention_fp8(q, k, v, enable_gqa=gqa)
    if kind == "block":
        out = layers.self_attention_core(q, k, v, head_dim=case["D"], q_norm_weight=x["wq"], k_norm_weight=x["wk"],
                                         rope=x["tables"])
        return (out.detach(), *torch.autograd.grad(out, (q, k, v, x["wq"], x["wk"]), x["do"]))
    if kind == "ring":
        out, lse = ring.ring_attention(q, k, v, cp=case["cp"], key_mask=x.get("mask"), tables_q=x["tables_q"],
                                       tables_k=x["tables"])
        return (out.detach(), lse.detach(), *torch.autograd.grad(out, (q, k, v), x["do"]))
    if kind == "cross":
        out = A.attention(q, k, v, attn_mask=x["mask"][:, None, None, :], enable_gqa=gqa)
    elif kind == "window":
        out = A.temporal_neighbour_attention(q, k, v, neighbourhood=x["neighbourhood"], enable_gqa=gqa)
    else:
        out = A.varlen_attention(q, k, v, x["cu"], enable_gqa=gqa)
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), x["do"]))


# ---------------------------------------------------------------------------
# Work and tolerances
# ---------------------------------------------------------------------------


def work(case):
    B, H, Hkv, D, kind = case["B"], case["H"], case["Hkv"], case["D"], case["kind"]
    size = 4 if case["dtype"] == "float32" else 2
    if kind in ("block", "rotary"):
        Lq = Lk = case["F"] * case["Y"] * case["X"]
        pairs = B * Lq * Lk
    elif kind == "ring":
        Lq, Lk = case["shard"], case["F"] * case["Y"] * case["X"] + case["text"]
        keys = sum(Lk - case["text"] + n for n in _ints(case["text_lens"])) if case["text"] else B * Lk
        pairs = Lq * keys
    elif kind == "cross":
        Lq, Lk = case["Lq"], case["Lk"]
        pairs = Lq * sum(_ints(case["text_lens"]))
    elif kind == "window":
        F, P = case["F"], case["P"]
        Lq = Lk = F * P
        near = int(math.floor(case["seconds"] * FPS + 1e-6))
        pairs = B * P * P * sum(1 for i in range(F) for j in range(F) if abs(i - j) <= near)
    elif kind == "varlen":
        Lq = Lk = case["L"]
        pairs = B * sum(s * s for s in _ints(case["segments"]))
    else:
        Lq, Lk = case["Lq"], case["Lk"]
        pairs = B * Lq * Lk
    qb, kb = B * H * Lq * D * size, B * Hkv * Lk * D * size
    if kind in ("rotary", "fp8"):
        nbytes, products = 2 * qb + 2 * kb, 2
    else:
        # read q, k, v and the output's gradient, write the output and the
        # gradients of q, k, v
        nbytes, products = 4 * qb + 4 * kb, 6
    if "F" in case and "Y" in case:
        nbytes += 2 * B * Lk * (D // 2) * 4  # rotation tables
    return {"bytes": nbytes, "flops": 2.0 * products * H * pairs * D}


def tolerance(case):
    # About four times the largest distance from the float64 result measured
    # on an MI355X over the listed and some drawn cases: float32 1.4e-6 (order
    # of sums); bf16 3.9e-3, with the block's norm and rotation 6.5e-3 (q, k,
    # P, dS and the results rounded to 8 bits); fp8 1.9e-2 (q and k to 4 bits).
    if case["dtype"] == "float32":
        return {"rel": 6e-6}
    if case["kind"] == "fp8":
        return {"rel": 8e-2}
    return {"rel": 2.5e-2 if case["kind"] == "block" else 1.5e-2}


# ---------------------------------------------------------------------------
# float64 results
# ---------------------------------------------------------------------------


def _rotate(x, cos, sin):
    """Interleaved-pair rotation of x (..., L, D)."""
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack((e * cos - o * sin, e * sin + o * cos), -1).flatten(-2)


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w


def _head(q, k, v, do, allowed):
    """out, lse (and dq, dk, dv) of one head in float64, in blocks of query
    rows.  ``allowed(a, b)``: None or a bool mask for rows [a, b)."""
    Lq, D = q.shape
    Lk = k.shape[0]
    scale = 1.0 / math.sqrt(D)
    rows = max(1, min(Lq, int(4e8 // max(Lk, 1))))
    out, lse = torch.empty_like(q), q.new_empty(Lq)
    grads = None if do is None else (torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v))
    for a in range(0, Lq, rows):
        b = min(Lq, a + rows)
        s = (q[a:b] @ k.T).mul_(scale)
        m = allowed(a, b)
        if m is not None:
            s.masked_fill_(~m, float("-inf"))
        z = torch.logsumexp(s, -1)
        lse[a:b] = z
        p = s.sub_(z.masked_fill(z == float("-inf"), 0.0)[:, None]).exp_()
        out[a:b] = p @ v
        if do is not None:
            dq, dk, dv = grads
            dv += p.T @ do[a:b]
            delta = (do[a:b] * out[a:b]).sum(-1, keepdim=True)
            ds = (do[a:b] @ v.T).sub_(delta).mul_(p).mul_(scale)
            dq[a:b] = ds @ k
            dk += ds.T @ q[a:b]
    return (out, lse) if do is None else (out, lse, *grads)


def exact(case, seed):
    x = _inputs(case, seed)
    kind, B, H, Hkv, D = case["kind"], case["B"], case["H"], case["Hkv"], case["D"]
    group = H // Hkv
    Lk_all = x["k"].shape[1 if kind == "block" else 2]
    cos = x["cos"].double() if "cos" in x else None
    sin = x["sin"].double() if "cos" in x else None

    def heads(t, n):  # (B, n, L, D) view of a block's projection
        return t.unflatten(-1, (n, D)).transpose(1, 2) if kind == "block" else t

    q, k, v = heads(x["q"], H), heads(x["k"], Hkv), heads(x["v"], Hkv)
    do = heads(x["do"], H) if "do" in x else None
    mask, sec = x.get("mask"), x.get("seconds")
    seg = torch.searchsorted(x["cu"][1:].long(), torch.arange(case["L"], device="cuda"), right=True) \
        if kind == "varlen" else None
    nseg = len(_ints(case["segments"])) if kind == "varlen" else 0

    def allowed(b):
        if mask is not None:
            return lambda r0, r1: mask[b][None].expand(r1 - r0, -1)
        if kind == "window":
            return lambda r0, r1: (sec[b, r0:r1, None] - sec[b][None]).abs() <= case["seconds"]
        if kind == "varlen":
            return lambda r0, r1: (seg[r0:r1, None] == seg[None]) & (seg[None] < nseg)
        return lambda r0, r1: None

    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.empty(q.shape[:3], dtype=torch.float64, device="cuda")
    if do is not None:
        dq = torch.empty_like(out)
        dk = torch.zeros(k.shape, dtype=torch.float64, device="cuda")
        dv = torch.zeros_like(dk)
    dwq, dwk = (torch.zeros(D, dtype=torch.float64, device="cuda") for _ in range(2))
    Lq = q.shape[2]

    def prologue(t, w, b, length):
        """Norm and rotation of one head's rows (a leaf and the result)."""
        leaf = t.double().requires_grad_(do is not None)
        gain = None if w is None else w.double().requires_grad_(True)
        y = leaf if w is None else _rms(leaf, gain)
        if cos is not None:
            y = _rotate(y, cos[b, 0, :length], sin[b, 0, :length])
        return leaf, gain, y

    for b in range(B):
        for hk in range(Hkv):
            kl, kg, ky = prologue(k[b, hk], x.get("wk"), b, Lk_all)
            dky = torch.zeros_like(ky, requires_grad=False)
            for h in range(hk * group, (hk + 1) * group):
                ql, qg, qy = prologue(q[b, h], x.get("wq"), b, Lq)
                r = _head(qy.detach(), ky.detach(), v[b, hk].double(), None if do is None else do[b, h].double(),
                          allowed(b))
                out[b, h], lse[b, h] = r[0], r[1]
                if do is None:
                    continue
                g = torch.autograd.grad(qy, [ql] + ([qg] if qg is not None else []), r[2]) if qy is not ql else (r[2],)
                dq[b, h] = g[0]
                if qg is not None:
                    dwq += g[1]
                dky += r[3]
                dv[b, hk] += r[4]
            if do is not None:
                g = torch.autograd.grad(ky, [kl] + ([kg] if kg is not None else []), dky) if ky is not kl else (dky,)
                dk[b, hk] = g[0]
                if kg is not None:
                    dwk += g[1]

    if kind in ("rotary", "fp8"):
        return out

    def flat(t):
        return t.transpose(1, 2).flatten(2) if kind == "block" else t

    if kind == "block":
        return flat(out), flat(dq), flat(dk), flat(dv), dwq, dwk
    if kind == "ring":
        return out, lse, dq, dk, dv
    return out, dq, dk, dv
