"""The channel statistics on both sides of the fold's line: sequences of up to
16 (head dim 64) or 12 (128) 128-token tiles fold the partials inside the code
pass, longer ones in a launch of their own. Codes, scales and statistics equal
the oracle's bit for bit at one tile, at odd and even counts, at the line and
one tile past it, with K or V smoothing off, grouped heads, merged keys and the
QK LayerNorm."""
from __future__ import annotations

import numpy as np
import pytest

from sage_gpu_helpers import assert_prologue_equal, run

pytestmark = pytest.mark.gpu

CASES = [
    (64, 1, dict(tokens=5)), (64, 2, dict(tokens=256, dtype=1)), (64, 3, dict(tokens=300, smooth_k=False)),
    (64, 16, dict(tokens=2048, kv_heads=1)), (64, 16, dict(tokens=1921)), (64, 17, dict(tokens=2049)),
    (128, 1, dict(tokens=128)), (128, 11, dict(tokens=1300, dtype=1)), (128, 12, dict(tokens=1536)),
    (128, 13, dict(tokens=1537, kv_heads=1)), (128, 5, dict(tokens=513, smooth_v=False)),
    (64, 3, dict(tokens=3 * 95, merge=2, layout=(3, 5, 9, 10, 1))),
    (128, 3, dict(tokens=3 * 95, merge=4, layout=(3, 5, 9, 10, 0), ln=True)),
    (64, 6, dict(tokens=689, ln=True, dtype=1)),
]


@pytest.mark.parametrize("d,tiles,kw", CASES, ids=[f"d{c[0]}t{c[1]}_{i}" for i, c in enumerate(CASES)])
def test_statistics(oracle, torch_gpu, d, tiles, kw):
    kw = dict(kw)
    n = kw.pop("tokens")
    assert -(-n // 128) == tiles
    if kw.pop("ln", False):
        rng = np.random.default_rng(n)
        kw["ln"] = np.concatenate([s + 0.3 * rng.standard_normal(d) for s in (1, 0, 1, 0)]).astype(np.float32)
    p = oracle.Problem(2, 3, n, d, **kw)
    q, k, v = oracle.generate(p, oracle.GenSpec(k_off_std=2.0, seed=n + d))
    pro, _ = run(torch_gpu, p, q, k, v)
    assert_prologue_equal(pro, oracle.prologue(p, q, k, v))
