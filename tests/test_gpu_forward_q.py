"""forward quantises Q in the attention kernel where the whole-key kernel runs
(its workgroup owns the query rows); prepare followed by attend does it in the
prologue. Both must leave the same codes and scales in the workspace and the
same output bit for bit, over ragged last tiles, strides, both input types,
grouped, causal and merged plans, and an output written over Q itself or over
rows that other workgroups still read."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import from_device16, to_device16
from sage_gpu_helpers import split_of

pytestmark = pytest.mark.gpu

# batch, heads, tokens, head_dim, extra Problem arguments, layout: grids of
# more tiles than the keys-split kernels take.
CASES = [
    (1, 58, 1000, 64, {}, "bthd"),
    (1, 450, 17, 64, dict(dtype=1), "bhtd"),
    (2, 11, 1025, 128, dict(dtype=1), "packed"),
    (1, 164, 1, 128, {}, "bthd"),
    (1, 72, 1001, 64, dict(kv_heads=9, causal=True), "bhtd"),
    (2, 20, 1050, 128, dict(causal=True), "packed"),
    (1, 19, 16 * 95, 64, dict(merge=2, layout=(16, 5, 9, 10, 0)), "bhtd"),
    (1, 11, 16 * 95, 128, dict(merge=4, layout=(16, 5, 9, 10, 2), dtype=1), "bthd"),
]
NAMES = ("q8", "q_scale", "k8", "k_scale", "v8", "stats")


def _setup(torch, oracle, b, h, n, d, kw, layout):
    import spl_sage as S

    p = oracle.Problem(b, h, n, d, **kw)
    q, k, v = oracle.generate(p, oracle.GenSpec(k_off_std=2.0, seed=n + d))
    q[:, n // 3] = 0  # an all-zero row, and (below) an all-zero group
    if n > 64:
        q[:, 32:48] = 0
    if layout == "packed":
        y = to_device16(torch, np.stack([q, k, v], axis=2), p.dtype)
        ts = [y[:, :, i] for i in range(3)]
    elif layout == "bhtd":
        ts = [to_device16(torch, np.ascontiguousarray(x.transpose(0, 2, 1, 3)), p.dtype).transpose(1, 2) for x in (q, k, v)]
    else:
        ts = [to_device16(torch, x, p.dtype) for x in (q, k, v)]
    assert split_of(p)[0] == 0, "a grid of the keys-split kernels: Q stays with the prologue"
    sa = S.SageAttention(None, d)
    merge = S.KvMerge.Dense if p.merge == 1 else S.KvMerge.Pool(p.merge, S.FrameLayout(*p.layout))
    ws = sa.workspace(S.Shape(b, h, n, p.kv_heads), merge)
    return S, p, sa, ws, ts, S.Options(causal=p.causal)


@pytest.mark.parametrize("b,h,n,d,kw,layout", CASES, ids=[f"b{c[0]}h{c[1]}n{c[2]}d{c[3]}" for c in CASES])
def test_forward_equals_prepare_and_attend(oracle, torch_gpu, b, h, n, d, kw, layout):
    torch = torch_gpu
    S, p, sa, ws, ts, opts = _setup(torch, oracle, b, h, n, d, kw, layout)
    tens = [S.Tensor(t) for t in ts]
    o1, o2, o3 = (torch.zeros(ts[0].shape, dtype=ts[0].dtype, device="cuda") for _ in range(3))
    sa.prepare(ws, *tens, opts)
    sa.attend(ws, S.TensorMut(o1))
    want = {m: ws.tensor(m).clone() for m in NAMES}
    ws2 = sa.workspace(ws.plan().shape, ws.plan().merge)
    sa.forward(ws2, *tens, S.TensorMut(o2), opts)
    sa.attend(ws2, S.TensorMut(o3))  # from the codes that forward left
    torch.cuda.synchronize()
    for m in NAMES:
        assert torch.equal(ws2.tensor(m).view(torch.uint8), want[m].view(torch.uint8)), m
    assert np.array_equal(from_device16(o2), from_device16(o1))
    assert np.array_equal(from_device16(o3), from_device16(o1))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("where", ["over q", "shifted over q"])
def test_output_over_q(oracle, torch_gpu, d, where):
    """out = Q in place, and out one head away from Q in one buffer (its rows
    are other heads' queries, still to be read): the same result as apart."""
    torch = torch_gpu
    h = 475 if d == 64 else 240
    S, p, sa, ws, ts, opts = _setup(torch, oracle, 1, h, 130, d, {}, "bthd")
    o = torch.empty_like(ts[0])
    sa.prepare(ws, *(S.Tensor(t) for t in ts), opts)
    sa.attend(ws, S.TensorMut(o))
    buf = torch.zeros(ts[0].numel() + d, dtype=ts[0].dtype, device="cuda")
    q = buf[: ts[0].numel()].view(ts[0].shape)
    q.copy_(ts[0])
    out = q if where == "over q" else buf[d:].view(ts[0].shape)
    sa.forward(ws, S.Tensor(q), S.Tensor(ts[1]), S.Tensor(ts[2]), S.TensorMut(out), opts)
    torch.cuda.synchronize()
    assert np.array_equal(from_device16(out), from_device16(o))


@pytest.mark.parametrize("d", [64, 128])
def test_output_over_a_broadcast_q(oracle, torch_gpu, d):
    """One query row a token, broadcast over the heads of one KV head, and the
    output over it: every head's result is the same row, from the Q of before
    the call."""
    torch = torch_gpu
    h = 475 if d == 64 else 240
    S, p, sa, ws, ts, opts = _setup(torch, oracle, 1, h, 130, d, dict(kv_heads=1), "bthd")
    q = ts[0][:, :, :1].contiguous()
    want = torch.empty_like(ts[0])
    st = S.Strides(130 * d, d, 0)
    sa.prepare(ws, S.Tensor(q, st), S.Tensor(ts[1]), S.Tensor(ts[2]), opts)
    sa.attend(ws, S.TensorMut(want))
    sa.forward(ws, S.Tensor(q, st), S.Tensor(ts[1]), S.Tensor(ts[2]), S.TensorMut(q, st), opts)
    torch.cuda.synchronize()
    assert np.array_equal(from_device16(q)[:, :, 0], from_device16(want)[:, :, 0])
    assert np.array_equal(from_device16(want)[:, :, -1], from_device16(want)[:, :, 0])


def test_refused_output_leaves_a_prepared_workspace(oracle, torch_gpu):
    """An output that attend refuses: forward reports attend's text, and the
    workspace holds prepare's codes, as after the two calls."""
    torch = torch_gpu
    S, p, sa, ws, ts, opts = _setup(torch, oracle, 1, 58, 1000, 64, {}, "bthd")
    tens = [S.Tensor(t) for t in ts]
    short = torch.empty(64, dtype=ts[0].dtype, device="cuda")
    with pytest.raises(S.SageError, match="output holds 64 elements"):
        sa.forward(ws, *tens, S.TensorMut(short, S.Strides.bthd(1000, 58, 64)), opts)
    _check_left_prepared(S, torch, sa, ws, ts, tens, opts)


def test_output_of_another_type_leaves_a_prepared_workspace(oracle, torch_gpu):
    """The same for an output that the Python layer refuses; a bad Q is still
    the first refusal."""
    torch = torch_gpu
    S, p, sa, ws, ts, opts = _setup(torch, oracle, 1, 58, 1000, 64, {}, "bthd")
    tens = [S.Tensor(t) for t in ts]
    f32 = torch.empty(ts[0].shape, dtype=torch.float32, device="cuda")
    with pytest.raises(S.SageError, match="Q holds 64 elements"):
        sa.forward(ws, S.Tensor(f32.to(ts[0].dtype)[0, 0, 0].clone(), S.Strides.bthd(1000, 58, 64)), *tens[1:],
                   S.TensorMut(f32), opts)
    with pytest.raises(S.SageError, match="sage tensors are bf16 or fp16"):
        sa.forward(ws, *tens, S.TensorMut(f32), opts)
    _check_left_prepared(S, torch, sa, ws, ts, tens, opts)


def _check_left_prepared(S, torch, sa, ws, ts, tens, opts):
    o1, o2 = torch.empty_like(ts[0]), torch.empty_like(ts[0])
    sa.attend(ws, S.TensorMut(o1))
    sa.forward(ws, *tens, S.TensorMut(o2), opts)
    torch.cuda.synchronize()
    assert np.array_equal(from_device16(o1), from_device16(o2))


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("d", [64, 128])
def test_special_queries(oracle, torch_gpu, d, dtype):
    """16-row groups holding a NaN, an infinity, only NaNs, the smallest
    subnormals (127 / amax overflows in bf16), the largest finite value, and
    ties of the rounding: the codes and scales equal the prologue's."""
    torch = torch_gpu
    h = 475 if d == 64 else 240
    S, p, sa, ws, ts, opts = _setup(torch, oracle, 1, h, 200, d, dict(dtype=dtype), "bthd")
    q = ts[0].view(torch.int16)
    bits = lambda x: int(np.uint16(x).view(np.int16))  # noqa: E731
    nan, inf, big = (0x7FC0, 0x7F80, 0x7F7F) if dtype == 0 else (0x7E00, 0x7C00, 0x7BFF)
    q[:, 5, :, 3] = bits(nan)
    q[:, 6, :, 4] = bits(nan | 0x8000)
    q[:, 20, :, 7] = bits(inf | 0x8000)
    q[:, 52:68] = bits(nan)
    q[:, 80:96] = 0
    q[:, 80:96, :, ::5] = bits(1)
    q[:, 97, :, 0] = bits(big)
    ties = torch.zeros(d, device="cuda")
    ties[0] = 127.0
    ties[1:] = torch.arange(1, d, device="cuda") - 31.5
    q[:, 112:128] = ties.to(ts[0].dtype).view(torch.int16)
    tens = [S.Tensor(t) for t in ts]
    o = torch.empty_like(ts[0])
    sa.prepare(ws, *tens, opts)
    want = [ws.tensor(m).clone() for m in ("q8", "q_scale")]
    ws2 = sa.workspace(ws.plan().shape)  # zero-filled
    sa.forward(ws2, *tens, S.TensorMut(o), opts)
    torch.cuda.synchronize()
    for m, w in zip(("q8", "q_scale"), want):
        assert torch.equal(ws2.tensor(m).view(torch.uint8), w.view(torch.uint8)), m
