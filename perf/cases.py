"""Workloads of the SageAttention2 forward path, as its callers run it.

Every case is one call through the package's public entry points on tensors
already on the GPU: `forward` (prepare, then attend), `forward_noalloc` (the
same without a workspace), `forward_qkv` (fed from the fused QKV projection)
and `QkvPrologue.run` (the projection's own prologue). They span a 256-token
call of two heads up to 17776 tokens of 48 heads, both head dims, bf16 and
fp16, dense, causal, grouped-query and KV-merged keys, the fused QK
LayerNorm, and the caller's layouts.

A case is a dict: entry, batch, heads, kv_heads, tokens, head_dim, dtype
("bf16" / "f16"), causal, layout ("bthd", "bhtd", "packed"), merge (1, 2, 4;
`frames` frames of 17 special tokens and a 21 x 32 grid), qk_norm (the sage
options' LayerNorm), norm and rope (the QKV prologue's), pv16 and k_off (the
spread of K's per-channel offset).
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT / "sota-papers-lab_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "sota-papers-lab_amd"))

import spl_sage as S  # noqa: E402
from spl_sage import qkv as Q  # noqa: E402

SPECIAL, GRID_H, GRID_W = 17, 21, 32  # a VGGT frame at 512 x 336
FRAME = SPECIAL + GRID_H * GRID_W     # 689 tokens
MOST_FLOPS = 4.0 * 48 * 17776 * 17776 * 64  # the largest listed case
MOST_BYTES = 1.0e9
LOG2E = 1.4426950408889634


def _case(entry="forward", batch=1, heads=16, kv_heads=0, tokens=0, head_dim=64, dtype="bf16", causal=False,
          layout="bthd", frames=0, merge=1, qk_norm=False, norm="", rope="", pv16=False, k_off=2.0, name=None):
    c = dict(entry=entry, batch=batch, heads=heads, kv_heads=kv_heads or heads, tokens=tokens or frames * FRAME,
             head_dim=head_dim, dtype=dtype, causal=causal, layout=layout, frames=frames, merge=merge,
             qk_norm=qk_norm, norm=norm, rope=rope, pv16=pv16, k_off=k_off)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest call: two heads of 256 tokens (the CPU-checkable configuration).
        _case(name="c1_h2_n256_d64", heads=2, tokens=256, dtype="f16"),
        # One VGGT frame, head-major as the trunk hands it over: too few query
        # tiles to fill the chip.
        _case(name="frame1_h16_d64", frames=1, layout="bhtd"),
        # A serving prefill of two ragged prompts, grouped heads, causal, no workspace.
        _case(name="prefill_gqa_n1000_d128", entry="noalloc", batch=2, heads=32, kv_heads=8, tokens=1000, head_dim=128,
              dtype="f16", causal=True),
        # Global attention over a few frames fed from the QKV projection (LayerNorm and 2D RoPE fused).
        _case(name="frames4_qkv_d64", entry="qkv", frames=4, norm="layer", rope="vggt"),
        # Frame attention: a batch of frames in the packed projection layout, with the sage QK LayerNorm.
        _case(name="frame_batch8_qknorm_d64", batch=8, tokens=FRAME, layout="packed", qk_norm=True),
        # The QKV prologue on its own: eight frames, V in fp16.
        _case(name="qkv_prologue_frames8", entry="prologue", frames=8, norm="layer", rope="vggt"),
        # Global attention over KV-merged keys.
        _case(name="merge4_frames40_d64", frames=40, merge=4, layout="bhtd"),
        # The same from the QKV projection at head dim 128: a larger model's layer.
        _case(name="qkv_n2048_d128", entry="qkv", heads=24, tokens=2048, head_dim=128, norm="rms", rope="dinov3"),
        # The headline configuration.
        _case(name="c2_b2_h32_n4096_d128", batch=2, heads=32, tokens=4096, head_dim=128),
        # Long-context causal prefill, and the same with grouped heads.
        _case(name="c3_causal_n16384_d128", heads=32, tokens=16384, head_dim=128, dtype="f16", causal=True),
        _case(name="c4_gqa_n8192_d128", heads=32, kv_heads=8, tokens=8192, head_dim=128, causal=True),
        # The longest: video-length tokens with a ragged tail.
        _case(name="c5_h48_n17776_d64", heads=48, tokens=17776, dtype="f16", k_off=3.0),
    ]


def _keys(c):
    """(keys after merging, query-key pairs of one head)."""
    n = c["tokens"]
    if c["merge"] > 1:
        m = c["merge"]
        tk = c["frames"] * (SPECIAL + -(-GRID_H // m) * -(-GRID_W // m))
        return tk, n * tk
    return n, n * (n + 1) // 2 if c["causal"] else n * n


def work(case):
    """Inputs read once, outputs written once; 4 D operations per visible
    (query, key) pair, or the QKV prologue's few per element (norm, rotation)."""
    b, h, g, n, d = (case[k] for k in ("batch", "heads", "kv_heads", "tokens", "head_dim"))
    qkv = 2.0 * b * n * (h + 2 * g) * d
    if case["entry"] == "prologue":
        return {"bytes": 2 * qkv, "flops": 10.0 * b * n * (h + 2 * g) * d}
    return {"bytes": qkv + 2.0 * b * n * h * d, "flops": 4.0 * b * h * d * _keys(case)[1]}


def draw(rng):
    while True:
        entry = rng.choice(["forward", "forward", "forward", "noalloc", "qkv", "qkv", "prologue"])
        d = rng.choice([64, 128])
        kv = rng.choice([1, 2, 4, 8, 12, 16, 24, 32])
        group = rng.choice([1, 1, 1, 2, 4, 8])
        batch = rng.choice([1, 1, 1, 2, 3, 8])
        tokens = int(round(math.exp(rng.uniform(math.log(200), math.log(17776)))))
        fused = entry in ("qkv", "prologue")
        c = _case(entry=entry, batch=batch, heads=kv * group, kv_heads=kv, tokens=tokens, head_dim=d,
                  dtype="bf16" if fused else rng.choice(["bf16", "f16"]), k_off=rng.choice([0.0, 1.0, 2.0, 3.0]))
        c["causal"] = entry != "prologue" and rng.random() < 0.35
        if fused:
            c["norm"] = rng.choice(["", "layer", "rms"])
            c["rope"] = rng.choice(["vggt", "vggt", "dinov3"])
        else:
            c["layout"] = rng.choice(["bthd", "bhtd", "packed"]) if group == 1 else rng.choice(["bthd", "bhtd"])
            c["qk_norm"] = rng.random() < 0.25
            c["pv16"] = rng.random() < 0.15
            if entry == "forward" and rng.random() < 0.3:
                c["frames"] = max(1, min(48, int(round(math.exp(rng.uniform(0, math.log(48)))))))
                c["tokens"] = c["frames"] * FRAME
                c["merge"] = rng.choice([2, 4])
                c["causal"] = False
        w = work(c)
        # Within the largest listed case's work, and the no-workspace entry's 128 MiB.
        if w["flops"] > MOST_FLOPS or w["bytes"] > MOST_BYTES:
            continue
        if entry == "noalloc" and batch * (c["tokens"] + 128) * (c["heads"] + 2 * c["kv_heads"]) * d * 1.2 > 100e6:
            continue
        return c


def _dtype(c):
    return torch.bfloat16 if c["dtype"] == "bf16" else torch.float16


def _qkv_data(c, gen):
    """Q, V ~ N(0, 1) and K ~ N(0, 1) plus an offset per (head, channel), as
    [batch][token][head][dim] views of the case's layout."""
    b, h, g, n, d = (c[k] for k in ("batch", "heads", "kv_heads", "tokens", "head_dim"))
    t = _dtype(c)
    off = c["k_off"] * torch.randn((g, d), generator=gen, device="cuda")

    def rows(heads, add=None):
        x = torch.randn((b, n, heads, d), generator=gen, device="cuda")
        return x if add is None else x + add

    if c["layout"] == "packed":
        y = torch.empty((b, n, 3, h, d), dtype=t, device="cuda")
        y[:, :, 0], y[:, :, 1], y[:, :, 2] = rows(h), rows(g, off), rows(g)
        return y[:, :, 0], y[:, :, 1], y[:, :, 2]
    xs = [rows(h).to(t), rows(g, off).to(t), rows(g).to(t)]
    if c["layout"] == "bhtd":
        xs = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in xs]
    return tuple(xs)


def _projection(c, gen):
    """The fused projection and the prologue's parameters."""
    b, h, g, n, d = (c[k] for k in ("batch", "heads", "kv_heads", "tokens", "head_dim"))
    width = (h + 2 * g) * d
    p = {}
    y = torch.randn((b, n, width), generator=gen, device="cuda")
    p["y"] = (y + 0.5 * torch.randn((width,), generator=gen, device="cuda")).to(torch.bfloat16)
    p["bias"] = (0.2 * torch.randn((width,), generator=gen, device="cuda")).to(torch.bfloat16)
    p["nw"] = [(s + w * torch.randn((d,), generator=gen, device="cuda")).float()
               for s, w in ((1, 0.2), (0, 0.1), (1, 0.2), (0, 0.1))]  # q weight, q bias, k weight, k bias
    if c["frames"]:
        gh, gw, special = GRID_H, GRID_W, SPECIAL
    else:
        gh, gw, special = -(-n // 64), 64, 0
    make = Q.RopeTable.vggt if c["rope"] == "vggt" else Q.RopeTable.dinov3
    table = make(gh, gw, special, 100.0, d)
    p["table"], p["frame_len"] = table.upload(), table.frame_len
    return p


def _ln_params(c, gen):
    d = c["head_dim"]
    r = lambda: torch.randn((d,), generator=gen, device="cuda")  # noqa: E731
    return torch.cat([1 + 0.2 * r(), 0.1 * r(), 1 + 0.2 * r(), 0.1 * r()]).float().contiguous()


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    b, h, g, n, d = (c[k] for k in ("batch", "heads", "kv_heads", "tokens", "head_dim"))
    pv = S.PvAccum.F16 if c["pv16"] else S.PvAccum.F32
    sa = S.SageAttention(torch.cuda.current_stream(), d, S.Config(S.Tile.for_head_dim(d), pv))
    shape = S.Shape(b, h, n, g)
    merge = S.KvMerge.Dense
    if c["merge"] > 1:
        merge = S.KvMerge.Pool(c["merge"], S.FrameLayout(c["frames"], SPECIAL, GRID_H, GRID_W, 0))
    s = {"case": c, "sa": sa, "shape": shape}
    if c["entry"] in ("qkv", "prologue"):
        p = _projection(c, gen)
        nw = p["nw"]
        kind = {"layer": Q.NormKind.LayerNorm, "rms": Q.NormKind.Rms}.get(c["norm"])
        s["norm"] = None if kind is None else Q.QkNorm(kind, nw[0], nw[2], nw[1], nw[3], 1e-6)
        layout = Q.RopeLayout.Vggt if c["rope"] == "vggt" else Q.RopeLayout.Dinov3
        s["rope"] = Q.Rope(p["table"], layout, p["frame_len"])
        s["in"] = Q.QkvIn(p["y"], (h + 2 * g) * d, bias=p["bias"])
        if c["entry"] == "prologue":
            q, k, v = (torch.empty((b, m, n, d), dtype=t, device="cuda").transpose(1, 2)
                       for m, t in ((h, torch.bfloat16), (g, torch.bfloat16), (g, torch.float16)))
            s["outs"] = (q, k, v)
            s["out"] = Q.QkvOut(S.TensorMut(q), S.TensorMut(k), S.TensorMut(v))
            s["prologue"] = Q.QkvPrologue(sa)
            return s
        o = torch.empty((b, n, h, d), dtype=torch.bfloat16, device="cuda")
    else:
        q, k, v = _qkv_data(c, gen)
        s["qkv"] = tuple(S.Tensor(x) for x in (q, k, v))
        if c["layout"] == "bhtd":
            o = torch.empty((b, h, n, d), dtype=_dtype(c), device="cuda").transpose(1, 2)
        else:
            o = torch.empty((b, n, h, d), dtype=_dtype(c), device="cuda")
    s["opts"] = S.Options(causal=c["causal"], qk_norm=S.QkNorm(_ln_params(c, gen)) if c["qk_norm"] else None)
    s["o"], s["out"] = o, S.TensorMut(o)
    if c["entry"] != "noalloc":
        s["ws"] = sa.workspace(shape, merge)
    return s


def run(state):
    s = state
    entry = s["case"]["entry"]
    if entry == "prologue":
        c = s["case"]
        s["prologue"].run(s["in"], c["tokens"], c["heads"], s["norm"], s["rope"], s["out"], batch=c["batch"],
                          kv_heads=c["kv_heads"])
        return s["outs"]
    if entry == "qkv":
        s["sa"].forward_qkv(s["ws"], s["in"], s["out"], s["norm"], s["rope"], s["opts"])
    elif entry == "noalloc":
        s["sa"].forward_noalloc(s["shape"], *s["qkv"], s["out"], s["opts"])
    else:
        s["sa"].forward(s["ws"], *s["qkv"], s["out"], s["opts"])
    return s["o"]


def tolerance(case):
    """Outputs are 16-bit. With the keys of every 64-key block in another order
    (the same codes, scales and running maxima, other sums) attention outputs
    move by a relative 2-norm of 1.0e-4 (256 tokens) to 8.2e-4 (the normed
    frames), and at most 0.043 of the larger of a value and the result's root
    mean square: about four times that is allowed. The blocks themselves keep
    their order: sweeping them in another moves the online softmax's running
    maximum and with it the E4M3 grid of the probabilities (2.3e-2 to 3.0e-2).
    The QKV prologue rounds each fp32 row once: half a step of its 16-bit
    outputs here and there."""
    return {"rel": 1e-3} if case["entry"] == "prologue" else {"rel": 4e-3, "max": 0.17}


# ---------------------------------------------------------------- float64


def _norm64(x, w, b, eps, rms=False):
    mean = 0.0 if rms else x.mean(-1, keepdim=True)
    y = x - mean
    return y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps) * w.double() + (0.0 if b is None else b.double())


def _rope64(x, layout, gh, gw, special, n):
    """2D RoPE of [.., token, dim] rows: VGGT rotates pairs (i, i + D/4) inside
    each half by (row + 1, column + 1), DINOv3 pairs (i, i + D/2) by
    2 pi times centred coordinates in [-1, 1]; special tokens stay."""
    d = x.shape[-1]
    axis = d // 4
    t = torch.arange(n, device=x.device) % (special + gh * gw)
    cell = (t - special).clamp(min=0)
    row, col = (cell // gw).double(), (cell % gw).double()
    p = torch.arange(d // 2, device=x.device)
    freq = torch.pow(torch.tensor(100.0, dtype=torch.float64, device=x.device), -(p % axis).double() / axis)
    if layout == "vggt":
        pos = torch.where(p < axis, row[:, None] + 1, col[:, None] + 1)
    else:
        pos = 2 * math.pi * torch.where(p < axis, (row[:, None] + 0.5) / gh * 2 - 1, (col[:, None] + 0.5) / gw * 2 - 1)
    ang = torch.where((t >= special)[:, None], pos * freq, torch.zeros((), dtype=torch.float64, device=x.device))
    half = d // 4 if layout == "vggt" else d // 2
    first = (p // half) * (2 * half) + p % half
    a, b = x[..., first], x[..., first + half]
    out = torch.empty_like(x)
    out[..., first] = a * ang.cos() - b * ang.sin()
    out[..., first + half] = b * ang.cos() + a * ang.sin()
    return out


def _pooled64(x, c):
    """Keys of [heads, token, dim] averaged over merge x merge patch cells of
    every frame (special tokens stay single), and each key's member count."""
    m, f = c["merge"], c["frames"]
    h, _, d = x.shape
    x = x.reshape(h, f, FRAME, d)
    sp, grid = x[:, :, :SPECIAL], x[:, :, SPECIAL:].reshape(h, f, GRID_H, GRID_W, d)
    cells, counts = [], []
    for y0 in range(0, GRID_H, m):
        for x0 in range(0, GRID_W, m):
            block = grid[:, :, y0:y0 + m, x0:x0 + m]
            cells.append(block.mean((2, 3)))
            counts.append(block.shape[2] * block.shape[3])
    keys = torch.cat([sp, torch.stack(cells, 2)], 2)
    count = torch.tensor([1] * SPECIAL + counts, dtype=torch.float64, device=x.device).repeat(f)
    return keys.reshape(h, -1, d), count


def exact(case, seed):
    """The same in float64 from the 16-bit inputs: no quantisation, and no
    rounding between the projection and the attention."""
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    b, h, g, n, d = (c[k] for k in ("batch", "heads", "kv_heads", "tokens", "head_dim"))
    fused = c["entry"] in ("qkv", "prologue")
    if fused:
        p = _projection(c, gen)
        gh, gw, special = (GRID_H, GRID_W, SPECIAL) if c["frames"] else (-(-n // 64), 64, 0)

        def heads_of(part, i, j):  # [token, dim] rows of head j of batch item i
            s = (0, h, h + g)[part] + j
            x = p["y"][i, :, s * d:(s + 1) * d].double() + p["bias"][s * d:(s + 1) * d].double()
            if part < 2:
                if c["norm"]:
                    rms = c["norm"] == "rms"
                    x = _norm64(x, p["nw"][2 * part], None if rms else p["nw"][2 * part + 1], 1e-6, rms)
                x = _rope64(x, c["rope"], gh, gw, special, n)
            return x

        if c["entry"] == "prologue":
            return tuple(torch.stack([torch.stack([heads_of(part, i, j) for j in range(m)], 1) for i in range(b)])
                         for part, m in ((0, h), (1, g), (2, g)))
    else:
        qkv = _qkv_data(c, gen)
        ln = _ln_params(c, gen) if c["qk_norm"] else None

        def heads_of(part, i, j):
            x = qkv[part][i, :, j].double()
            if ln is not None and part < 2:
                x = _norm64(x, ln[2 * part * d:(2 * part + 1) * d], ln[(2 * part + 1) * d:(2 * part + 2) * d], 1e-5)
            return x

    out = torch.empty((b, n, h, d), dtype=torch.float64, device="cuda")
    for i in range(b):
        for j in range(g):
            k, v = heads_of(1, i, j), heads_of(2, i, j)
            bias = None
            if c["merge"] > 1:
                k, count = _pooled64(k[None], c)
                v, _ = _pooled64(v[None], c)
                k, v, bias = k[0], v[0], count.log()
            for e in range(h // g):
                q = heads_of(0, i, j * (h // g) + e)
                for r in range(0, n, 4096):
                    s = (q[r:r + 4096] @ k.T).mul_(1.0 / math.sqrt(d))
                    if bias is not None:
                        s += bias
                    if c["causal"]:
                        rows = torch.arange(r, r + s.shape[0], device="cuda")
                        s.masked_fill_(torch.arange(n, device="cuda") > rows[:, None], -math.inf)
                    out[i, r:r + s.shape[0], :, :][:, j * (h // g) + e] = torch.softmax(s, -1) @ v
    return out
