"""The attention kernels on both sides of the line between split and whole keys.

Grids of few query tiles run the kernel that splits a query group's keys over
two or four waves; larger ones the whole-key kernels, with a remainder of tiles
over a whole number a CU split beside whole ones. Each case sits at a place
where the split can go wrong: fewer key blocks than shares, a ragged last
block, blocks past the 64 whose scales a wave holds at a time, causal groups
whose last share is the diagonal alone, grouped heads, merged biases, and a
running maximum that moves in the last share (token 0.9 N scaled up). The cases
over the line keep the whole-key kernels' own masks and tails covered, the
eight-wave layout among them. The gate is the fuzz test's: 2e-2 plus half an
output step of the emulated reference arithmetic, and no further from f64.

The softmax block is written out in sage_attn, in the eight-wave layout and in
the keys-split kernels, and the probabilities must be the same E4M3 codes in all
of them: the same heads are run in grids on either side of the line and compared
far more tightly than any gate against the reference arithmetic.
"""
from __future__ import annotations

import numpy as np
import pytest

from sage_gpu_helpers import run, sample_rows, split_of
from test_gpu_fuzz import _check

pytestmark = pytest.mark.gpu

SPLIT = [
    # batch, heads, tokens, head_dim, extra Problem arguments
    (1, 1, 63, 64, {}),                                  # one ragged block, three empty shares
    (1, 3, 129, 128, {}),                                # three blocks on four shares
    (2, 5, 257, 64, dict(kv_heads=1, dtype=1)),
    (1, 1, 4500, 64, {}),                                # 71 blocks: two chunks of K scales
    (1, 1, 8200, 128, dict(dtype=1)),                    # 129 blocks, the last one of 8 keys
    (1, 34, 1000, 64, {}),                               # 256 tiles whole, 16 split
    (1, 5, 7000, 64, dict(dtype=1)),                     # 275 tiles: uneven XCD ranges
    (2, 33, 1003, 64, dict(kv_heads=11)),                # 512 whole, 16 split
    (1, 5, 6700, 128, {}),                               # 265: one buffer a wave
    (2, 34, 1003, 128, dict(dtype=1)),                   # 512 whole, 32 split
    (1, 2, 4170, 128, dict(causal=True)),
    (3, 4, 700, 64, dict(kv_heads=2, causal=True)),
    (1, 8, 1000, 64, dict(causal=True)),                 # dealt longest first
    (1, 48, 700, 64, dict(causal=True)),                 # two shares (288 tiles of short keys)
    (1, 48, 1100, 64, dict(causal=True, dtype=1)),       # 432 tiles
    (1, 32, 1050, 128, dict(kv_heads=4, causal=True)),   # two shares (288 tiles)
    (1, 3, 3 * 95, 64, dict(merge=2, layout=(3, 5, 9, 10, 1))),
    (1, 2, 50 * 95, 128, dict(merge=4, layout=(50, 5, 9, 10, 0))),
]
WHOLE = [
    (1, 58, 1000, 64, {}),
    (1, 21, 1000, 128, dict(dtype=1)),
    (1, 72, 1001, 64, dict(kv_heads=9, causal=True)),
    (2, 20, 1050, 128, dict(causal=True)),
    (1, 19, 16 * 95, 64, dict(merge=2, layout=(16, 5, 9, 10, 0))),
    (1, 11, 16 * 95, 128, dict(merge=2, layout=(16, 5, 9, 10, 2))),
]


def _problem(oracle, b, h, n, d, kw, seed):
    p = oracle.Problem(b, h, n, d, **kw)
    q, k, v = oracle.generate(p, oracle.GenSpec(k_off_std=2.0, seed=seed))
    # A late key that outgrows every row's maximum so far.
    t = int(0.9 * n)
    k[:, t] = oracle.encode16(2.0 * oracle.decode16(k[:, t], p.dtype), p.dtype)
    return p, q, k, v


@pytest.mark.parametrize("b,h,n,d,kw", SPLIT + WHOLE, ids=[f"b{c[0]}h{c[1]}n{c[2]}d{c[3]}" for c in SPLIT + WHOLE])
def test_against_reference_arithmetic(oracle, torch_gpu, b, h, n, d, kw):
    p, q, k, v = _problem(oracle, b, h, n, d, kw, 100 + n + d)
    assert (split_of(p)[0] > 0) == ((b, h, n, d, kw) in SPLIT)
    _, o = run(torch_gpu, p, q, k, v, want_ws=False)
    rows = sample_rows(n, max(8, 4096 // (b * h)), seed=n)
    _check(oracle, p, oracle.prologue(p, q, k, v), o, rows, q, k, v, p.dtype, f"b{b} h{h} n{n} d{d} {kw}")


@pytest.mark.parametrize("b,h,n,d,kw", [c for c in WHOLE if "merge" not in c[4]],
                         ids=[f"h{c[1]}d{c[3]}" for c in WHOLE if "merge" not in c[4]])
def test_eight_waves_equal_four_over_the_line(oracle, torch_gpu, b, h, n, d, kw):
    import spl_sage as S

    p, q, k, v = _problem(oracle, b, h, n, d, kw, 200 + n)
    assert split_of(p)[0] == 0
    _, base = run(torch_gpu, p, q, k, v, want_ws=False)
    _, o = run(torch_gpu, p, q, k, v, want_ws=False, tile=S.Tile(8, 1, 3))
    assert np.array_equal(o, base)


# tokens, head dim, heads (split, whole), Problem arguments
SAME = [
    (1000, 64, 4, 58, {}),
    (1000, 64, 34, 58, {}),                     # most tiles whole beside split ones
    (1000, 128, 4, 21, dict(dtype=1)),
    (1003, 128, 34, 43, {}),
    (700, 64, 16, 72, dict(causal=True)),
    (700, 64, 48, 72, dict(causal=True, dtype=1)),   # two shares
    (1050, 128, 8, 40, dict(causal=True)),
    (1050, 128, 30, 40, dict(causal=True)),     # two shares
    (12 * 95, 64, 4, 26, dict(merge=2, layout=(12, 5, 9, 10, 1))),
    (12 * 95, 128, 4, 15, dict(merge=4, layout=(12, 5, 9, 10, 0))),
]


@pytest.mark.parametrize("n,d,few,many,kw", SAME, ids=[f"n{c[0]}d{c[1]}h{c[2]}_{c[3]}" for c in SAME])
def test_the_same_heads_split_and_whole(oracle, torch_gpu, n, d, few, many, kw):
    """The two sides differ by the order of fp32 sums of up to N terms alone: l and
    O move by some tens of roundings (64 * 2^-24 of the largest output, taken as
    4e-6), so an output moves by that and, where it lies that close to a rounding
    edge of the 16-bit type (4e-6 against steps of 2^-8 or 2^-9: 2e-3 of all),
    one step more. Probabilities of another E4M3 grid (a share's own maximum
    instead of the running one) move outputs by 2e-2 in the 2-norm and most of
    them by a step; what is let through here is sqrt(2e-3) * 2^-8 = 2e-4."""
    p, q, k, v = _problem(oracle, 1, many, n, d, kw, 300 + n + d)
    f = oracle.Problem(1, few, n, d, **kw)
    assert split_of(p)[0] == 0 and split_of(f)[0] > 0
    _, whole = run(torch_gpu, p, q, k, v, want_ws=False)
    _, split = run(torch_gpu, f, *(np.ascontiguousarray(x[:, :, :few]) for x in (q, k, v)), want_ws=False)
    a, b = (oracle.decode16(x, p.dtype).astype(np.float64) for x in (whole[:, :, :few], split))
    step = 2.0 ** (-7 if p.dtype == 0 else -10)  # the widest step of the type at 1
    moved = np.abs(a - b)
    print(f"{(moved > 0).mean():.2e} of outputs moved, at most {moved.max() / np.abs(a).max():.2e} of the largest")
    assert np.all(moved <= 4e-6 * np.abs(a).max() + step * np.abs(a))
    assert (moved > 0).mean() <= 2e-3
    assert np.linalg.norm(a - b) <= 2e-4 * np.linalg.norm(a)
