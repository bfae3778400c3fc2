"""Host side of the C ABI on the CPU (no GPU compute): the library loads and
exports every function include/sage_hip.h declares, the ctypes mirror has
the C struct layouts, and the plan / stride / tile / flops logic passes the
reference's own known-answer tests (tests.rs:135-283) and error texts."""
from __future__ import annotations

import ctypes as C
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "sage_hip.h"


@pytest.fixture(scope="module")
def S():
    import spl_sage

    return spl_sage


def _header_functions() -> list[str]:
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    names = re.findall(r"^\s*[A-Za-z_][\w \*]*?\b(sage_\w+)\s*\(", text, flags=re.M)
    return sorted(set(names))


def test_library_exports_every_declared_function(S):
    from spl_sage import _abi

    names = _header_functions()
    assert len(names) >= 20, names
    lib = C.CDLL(str(_abi.LIB_PATH))
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing
    # and the Python mirror binds each of them with a signature
    assert sorted(_abi.SIGNATURES) == names


def test_ctypes_structs_match_the_c_layout(S, tmp_path):
    """sizeof / offsetof of every ABI struct, compiled from the header with gcc,
    equal the ctypes mirror's (the role of geom_matches_the_cuda_struct,
    tests.rs:234-243, at this boundary)."""
    from spl_sage import _abi

    structs = {
        "sage_tile": ["warps", "m_tiles", "stages"],
        "sage_config": ["tile", "pv_accum"],
        "sage_shape": ["batch", "heads", "tokens", "kv_heads"],
        "sage_frame_layout": ["frames", "special", "grid_h", "grid_w", "dense_frames"],
        "sage_kv_merge": ["stride", "layout"],
        "sage_plan": ["shape", "merge", "tq_pad", "tk", "tk_pad"],
        "sage_strides": ["batch", "token", "head"],
        "sage_tensor": ["data", "len", "strides", "dtype"],
        "sage_tensor_mut": ["data", "len", "strides", "dtype"],
        "sage_options": ["softmax_scale", "has_softmax_scale", "smooth_k", "smooth_v", "qk_norm_params",
                         "qk_norm_len", "qk_norm_eps", "causal"],
        "sage_ws_buffers": ["q8", "q_scale", "k8", "k_scale", "v8", "stats", "kbias", "q8_len", "q_scale_len",
                            "k8_len", "k_scale_len", "v8_len", "stats_len", "kbias_len"],
    }
    lines = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{HEADER}"', "int main(void) {"]
    for s, fields in structs.items():
        lines.append(f'printf("{s} %zu\\n", sizeof({s}));')
        for f in fields:
            lines.append(f'printf("{s}.{f} %zu\\n", offsetof({s}, {f}));')
    lines.append("return 0; }")
    src = tmp_path / "layout.c"
    src.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-std=c11", "-Wall", "-o", str(exe), str(src)], check=True)
    got = dict(l.split() for l in subprocess.run([str(exe)], check=True, capture_output=True,
                                                 text=True).stdout.splitlines())
    for s, fields in structs.items():
        cls = getattr(_abi, s)
        assert int(got[s]) == C.sizeof(cls), s
        for f in fields:
            assert int(got[f"{s}.{f}"]) == getattr(cls, f).offset, f"{s}.{f}"


def test_vggt_dense_geometry(S):
    """tests.rs:137-148: 200 frames x 689 tokens."""
    plan = S.Plan.new(S.Shape(1, 16, 200 * 689))
    assert (plan.tq_pad, plan.tk, plan.tk_pad) == (137856, 137800, 137856)


def _vggt_layout(S, frames: int, dense_frames: int = 0):
    return S.FrameLayout(frames, 17, 21, 32, dense_frames)


def test_vggt_merge_key_counts(S):
    """tests.rs:149-152 and :96-110: merged key counts of the pooled layouts."""
    layout = _vggt_layout(S, 200)
    assert layout.tokens_per_frame() == 689
    shape = S.Shape(1, 16, 200 * 689)
    assert S.Plan.new(shape, S.KvMerge.Pool(2, layout)).tk == 200 * (17 + 11 * 16)
    assert S.Plan.new(shape, S.KvMerge.Pool(4, layout)).tk == 200 * (17 + 6 * 8)
    dense1 = _vggt_layout(S, 3, dense_frames=1)
    assert S.Plan.new(S.Shape(1, 1, 3 * 689), S.KvMerge.Pool(4, dense1)).tk == 689 + 2 * 65


def test_plan_rejects_bad_layouts(S):
    """tests.rs:175-190, with the reference's error texts."""
    layout = _vggt_layout(S, 2)
    with pytest.raises(S.SageError, match="frame layout"):
        S.Plan.new(S.Shape(1, 2, 1000), S.KvMerge.Pool(2, layout))
    shape = S.Shape(1, 2, 2 * 689)
    with pytest.raises(S.SageError, match="KV merge stride must be 2 or 4, got 3"):
        S.Plan.new(shape, S.KvMerge.Pool(3, layout))
    S.Plan.new(shape, S.KvMerge.Pool(4, layout))
    with pytest.raises(S.SageError, match="empty attention shape"):
        S.Plan.new(S.Shape(1, 2, 0))


def test_plan_range_checks(S):
    """mod.rs:406-439: an empty patch grid, and every count the kernels index
    with i32 (padded queries, padded keys, batch x heads) refused with the
    reference's texts."""
    with pytest.raises(S.SageError, match="KV merge needs a patch grid"):
        S.Plan.new(S.Shape(1, 1, 10), S.KvMerge.Pool(2, S.FrameLayout(2, 5, 0, 4, 0)))
    with pytest.raises(S.SageError, match="padded queries = 2147483648 does not fit in i32"):
        S.Plan.new(S.Shape(1, 1, 2**31 - 5))
    with pytest.raises(S.SageError, match="batch .* heads = 2147483648 does not fit in i32"):
        S.Plan.new(S.Shape(2**16, 2**15, 128))
    # Sizes whose padding or product would wrap 64 bits are refused, not wrapped.
    with pytest.raises(S.SageError, match="padded queries"):
        S.Plan.new(S.Shape(1, 1, 2**64 - 1))
    with pytest.raises(S.SageError, match="batch .* heads"):
        S.Plan.new(S.Shape(2**40, 2**30, 128))
    # A frame layout whose token count wraps 64 bits is refused: 2 frames of
    # 2^63 + 1 tokens would otherwise wrap to the sequence's 2 tokens.
    with pytest.raises(S.SageError, match="covers more than 2\\^64 tokens, the sequence has 2"):
        S.Plan.new(S.Shape(1, 1, 2), S.KvMerge.Pool(2, S.FrameLayout(2, 1, 1, 2**63, 0)))
    with pytest.raises(S.SageError, match="covers more than 2\\^64 tokens"):
        S.Plan.new(S.Shape(1, 1, 2), S.KvMerge.Pool(2, S.FrameLayout(1, 0, 2**32, 2**32, 0)))
    # The largest sizes that fit are accepted.
    p = S.Plan.new(S.Shape(1, 1, 2**31 - 128))
    assert p.tq_pad == 2**31 - 128 and p.tk_pad == 2**31 - 128
    S.Plan.new(S.Shape(2**16, 2**15 - 1, 128))


def test_extent_does_not_wrap(S):
    """Strides whose extent would wrap 64 bits report the largest extent, so a
    view with them can never pass the length check."""
    shape = S.Shape(1, 1, 5)
    assert S.Strides(8, 2**62, 8).extent(shape, 64) == 2**64 - 1
    assert S.Strides(8, 2**61, 8).extent(shape, 64) == 4 * 2**61 + 64


def test_plan_padding_and_tails(S):
    """mod.rs:431-434: tq_pad to 128, tk_pad to 64; the C5 tail shape."""
    p = S.Plan.new(S.Shape(1, 48, 17776))
    assert (p.tq_pad, p.tk, p.tk_pad) == (17792, 17776, 17792)
    assert p.q_tiles() == 139 and p.kblocks() == 278
    p = S.Plan.new(S.Shape(2, 32, 4096))
    assert (p.tq_pad, p.tk_pad) == (4096, 4096)


def test_plan_rejects_bad_grouped_heads(S):
    with pytest.raises(S.SageError):
        S.Plan.new(S.Shape(1, 32, 128, kv_heads=5))
    assert S.Plan.new(S.Shape(1, 32, 128, kv_heads=8)).kv_heads() == 8


def test_strides_cover_the_tensor(S):
    """tests.rs:245-261."""
    shape = S.Shape(2, 3, 5)
    d = 64
    assert S.Strides.bthd(5, 3, d).extent(shape, d) == 2 * 5 * 3 * d
    assert S.Strides.bhtd(5, 3, d).extent(shape, d) == 2 * 3 * 5 * d
    assert S.Strides.packed_qkv(5, 3, d).extent(shape, d) + 2 * 3 * d == 2 * 5 * 3 * 3 * d
    with pytest.raises(S.SageError, match="x strides must be multiples of 8 elements"):
        S.Strides.bthd(5, 3, 60).check("x")


def test_flops_counts_the_metric(S):
    """mod.rs:905-910 (4 B H Tq Tk D); causal counts the visible half, 2 B H D N (N + 1)."""
    c2 = S.Plan.new(S.Shape(2, 32, 4096))
    assert S.flops(c2, 128) == 4.0 * 2 * 32 * 4096 * 4096 * 128
    assert abs(S.flops(c2, 128) - 5.498e11) / 5.498e11 < 1e-3
    c3 = S.Plan.new(S.Shape(1, 32, 16384))
    assert S.flops(c3, 128, causal=True) == 2.0 * 32 * 128 * 16384 * 16385
    c1 = S.Plan.new(S.Shape(1, 2, 256))
    assert S.flops(c1, 64) == 4.0 * 2 * 256 * 256 * 64  # 3.36e7


def test_v8_position_is_the_operand_permutation(S):
    """Every key of a 64-key block has one byte in its V^T row, and key k sits
    where lane-half g = (k >> 2) & 1, register (k >> 5) * 4 + ((k >> 3) & 3),
    byte k & 3 of the FP8 B operand puts it."""
    pos = [S.v8_position(k) for k in range(64)]
    assert sorted(pos) == list(range(64))
    for k in range(64):
        g, reg, byte = (k >> 2) & 1, (k >> 5) * 4 + ((k >> 3) & 3), k & 3
        assert pos[k] == 32 * g + 4 * reg + byte


def _reference_tile_ok(w: int, m: int, st: int) -> bool:
    """Tile::validate (mod.rs:158-167), restated."""
    return w in (2, 4, 8) and m in (1, 2, 4) and 2 <= st <= 6 and 128 % (16 * m * w) == 0


def test_tile_menu_and_errors(S):
    """mod.rs:116-168: exactly the tiles the reference accepts validate; every
    other tile is refused with the reference's message, which names it."""
    accepted = 0
    for w in range(0, 10):
        for m in range(0, 6):
            for st in range(0, 8):
                t = S.Tile(w, m, st)
                if _reference_tile_ok(w, m, st):
                    t.validate()
                    accepted += 1
                else:
                    with pytest.raises(S.SageError, match=r"unsupported sage tile Tile \{ warps: %d, m_tiles: %d, "
                                       r"stages: %d \}" % (w, m, st)):
                        t.validate()
    # (2,1), (2,2), (2,4), (4,1), (4,2), (8,1) with stages 2..6
    assert accepted == 6 * 5
    for t in (S.Tile(4, 4, 3), S.Tile(8, 2, 3), S.Tile(8, 1, 7), S.Tile(4, 1, 1), S.Tile(3, 1, 2)):
        with pytest.raises(S.SageError, match="unsupported sage tile"):
            t.validate()


def test_default_tiles_are_the_references(S):
    """Tile::DEFAULT {4,2,3} and Tile::D128 {4,1,3} (mod.rs:128-147); Config::for_head_dim
    picks D128 above head dim 64 (mod.rs:141-147, 194-200) with PvAccum::F32."""
    assert S.Tile.DEFAULT == S.Tile(4, 2, 3) and S.Tile.D128 == S.Tile(4, 1, 3)
    assert S.Config.for_head_dim(64) == S.Config(S.Tile(4, 2, 3), S.PvAccum.F32)
    assert S.Config.for_head_dim(128) == S.Config(S.Tile(4, 1, 3), S.PvAccum.F32)
    assert S.Tile.for_head_dim(64) == S.Tile.DEFAULT and S.Tile.for_head_dim(128) == S.Tile.D128
    assert S.Tile.DEFAULT.rows() == 128 and S.Tile.D128.rows() == 64


def test_device_gate_without_a_gpu(S):
    """check_device reports, without a GPU, a device error rather than crashing."""
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    with pytest.raises(S.SageError):
        S.check_device(0)


@pytest.mark.parametrize("d", [64, 128])
def test_rope_tables_match_the_oracle(S, oracle, d):
    """RopeTable::vggt / ::dinov3 (qkv.rs:87-136) built by the library equal the
    oracle's restatement, which the reference's own table tests pin; too small
    an output buffer is refused with the reference's buffer message."""
    import numpy as np

    from spl_sage import qkv as Q

    for layout in (Q.RopeLayout.Vggt, Q.RopeLayout.Dinov3):
        t = Q.RopeTable._build(layout, 21, 32, 17, 100.0, d)
        assert t.frame_len == 17 + 21 * 32
        assert np.array_equal(t.cos_sin, oracle.rope_table(int(layout), d, 21, 32, 17, 100.0))
    out = np.empty(10, np.float32)
    with pytest.raises(S.SageError, match="RoPE table: buffer holds 10 elements, needs"):
        _check = S._check
        _check(S.lib().sage_rope_table(0, d, 2, 2, 1, 100.0, out.ctypes.data, out.size))


# (shape, Q strides, output strides, output's offset in elements), head dim 64
Q_BESIDE = [
    ((2, 3, 5), (960, 192, 64), (960, 192, 64), 0),          # in place
    ((2, 3, 5), (960, 64, 320), (960, 64, 320), 0),          # in place, head-major
    ((2, 3, 5), (2880, 576, 64), (2880, 576, 64), 0),        # in place in a packed projection
    ((2, 3, 5), (960, 192, 64), (960, 192, 64), 1920),       # apart
    ((2, 3, 5), (960, 192, 64), (960, 192, 64), 64),         # one head on
    ((2, 3, 5), (960, 192, 64), (960, 64, 320), 0),          # other strides over the same memory
    ((1, 3, 5), (0, 192, 64), (0, 192, 64), 0),              # a stride that is never taken
    ((2, 3, 5), (320, 64, 0), (320, 64, 0), 0),              # Q and output broadcast over heads
    ((2, 3, 5), (0, 192, 64), (0, 192, 64), 0),              # over batch items
    ((2, 3, 5), (960, 128, 64), (960, 128, 64), 0),          # heads of one token in the next one's
    ((2, 3, 5), (960, 192, 32), (960, 192, 32), 0),          # rows half in each other
    ((2, 2, 2), (64, 256, 128), (64, 256, 128), 0),          # batch items between the heads
]


@pytest.mark.parametrize("shape,qs,os_,off", Q_BESIDE)
def test_queries_read_beside_the_output(S, shape, qs, os_, off):
    """The attention kernel reads a workgroup's query rows, writes the same
    rows of the output and runs beside workgroups that do the same, so a forward
    call leaves Q to it only where no output row touches another query's row
    (here by every pair of rows)."""
    from spl_sage import _abi

    b, h, n = shape
    f = _abi.lib()._ZN4sage17q_readable_besideEmRK10sage_shapePK11sage_tensorPK15sage_tensor_mut
    f.restype = C.c_bool
    base, d = 1 << 20, 64
    q = _abi.sage_tensor(base, 1 << 30, qs, 0)
    o = _abi.sage_tensor_mut(base + 2 * off, 1 << 30, os_, 0)
    got = f(C.c_uint64(d), C.byref(_abi.sage_shape(b, h, n, h)), C.byref(q), C.byref(o))
    rows = [(i, t, j) for i in range(b) for t in range(n) for j in range(h)]
    at = lambda r, s, o: o + sum(x * y for x, y in zip(r, s))  # noqa: E731
    safe = all(abs(at(r, qs, 0) - at(w, os_, off)) >= d for r in rows for w in rows if r != w)
    assert safe or not got  # never where a row is overwritten before its reader
    if qs == os_ and off == 0:
        assert got == safe
    elif off >= 1920:
        assert got


@pytest.mark.parametrize("script,says", [("kill -9 $$", "killed by signal 9"), ("echo why >&2; exit 3", "exit status 3")])
def test_a_failed_build_step_says_how(tmp_path, monkeypatch, script, says):
    """A compiler that is killed writes nothing: the step and its status are
    named all the same."""
    import build as hip_build

    cc = tmp_path / "hipcc"
    cc.write_text(f"#!/bin/sh\n{script}\n")
    cc.chmod(0o755)
    monkeypatch.setattr(hip_build, "HIPCC", str(cc))
    monkeypatch.setattr(hip_build, "OBJ", tmp_path)
    with pytest.raises(RuntimeError, match=rf"compiling sage_api.cpp.o failed \({says}\)"):
        hip_build._compile(("sage_api.cpp", "sage_api.cpp.o", []))


# (head dim, tiles, heads, key blocks, merge stride, causal) -> (shares, whole):
# both sides of lines where the other kernel took longer.
SPLITS = [
    ((128, 278, 2, 278, 1, True), (0, 0)),     # few heads of long keys: two shares 379 us, whole keys 297
    ((128, 252, 4, 126, 1, True), (2, 0)),
    ((128, 288, 18, 32, 1, True), (2, 0)),
    ((128, 288, 72, 8, 1, True), (0, 0)),      # short keys: 40.9, 36.7
    ((64, 460, 2, 460, 1, True), (0, 0)),      # 457, 415
    ((64, 480, 15, 64, 1, True), (4, 0)),
    ((64, 200, 100, 3, 1, True), (4, 0)),      # 15.0, 16.1 (two shares)
    ((64, 288, 48, 12, 1, True), (2, 0)),
    ((128, 144, 144, 2, 1, False), (0, 0)),    # 28.0, 24.3
    ((128, 160, 5, 64, 1, False), (4, 0)),
    ((128, 584, 73, 16, 1, False), (0, 0)),    # 73.3, 69.1: over three workgroups a CU
    ((128, 576, 72, 16, 1, False), (4, 512)),
    ((128, 834, 6, 278, 1, False), (4, 768)),  # 645, 700
    ((128, 848, 53, 32, 1, False), (0, 0)),    # 130.8, 128.9
    ((128, 576, 288, 4, 1, False), (0, 0)),    # 51.5, 48.9
    ((64, 1060, 530, 4, 1, False), (0, 0)),
    ((64, 352, 16, 44, 1, False), (4, 256)),
    ((64, 640, 80, 16, 1, False), (4, 512)),   # 47.8, 45.6
    ((64, 880, 220, 8, 1, False), (0, 0)),     # 46.9, 46.1
    ((64, 876, 73, 24, 1, False), (4, 768)),   # 72.0, 73.2
    ((64, 648, 81, 16, 1, False), (0, 0)),     # 136 over 512: a second round of workgroups
    ((128, 344, 43, 16, 1, False), (0, 0)),    # 51.0, 50.6
    ((128, 336, 4, 168, 1, False), (4, 256)),  # 231, 217
    ((128, 120, 20, 4, 4, False), (0, 0)),     # merged, stride 4: 49.2, 45.3
    ((64, 222, 37, 2, 4, False), (0, 0)),      # 35.2, 32.4
    ((128, 132, 22, 12, 1, True), (2, 0)),     # 31.6, 33.0
    ((64, 222, 37, 4, 2, False), (2, 0)),
]


@pytest.mark.parametrize("args,want", SPLITS)
def test_key_split_lines(S, args, want):
    from sage_gpu_helpers import key_split

    d, tiles, heads, *rest = args
    assert key_split(d, tiles // heads * 128, heads, *rest) == want


def test_ragged_tiles_count_by_their_quarters(S):
    """Split kernels have no workgroup for 32-query groups past the sequence."""
    from sage_gpu_helpers import key_split

    assert key_split(128, 308, 50, 5, 1, True) == (4, 0)   # ten groups a head, 125 tiles of them
    assert key_split(128, 384, 50, 6, 1, True) == (0, 0)   # twelve: 150
    assert key_split(64, 17, 450, 1, 1, False) == (0, 0)   # one key block: nothing to share


def test_key_split_gives_what_the_kernels_are_built_for(S):
    """Merged plans two shares, dense ones four (alone or beside a whole number
    of tiles a CU with a remainder), causal ones four or two."""
    from sage_gpu_helpers import key_split

    for d in (64, 128):
        for heads in [*range(1, 2100, 7), 1 << 20]:
            for tokens in (1, 33, 128, 200, 1000, 2040, 17776, 1 << 24):
                kb, tiles = -(-tokens // 64), -(-tokens // 128) * heads
                s, w = key_split(d, tokens, heads, kb, 1, False)
                assert (s, w) == (0, 0) or (s == 4 and w % 256 == 0 and w < tiles), (d, tokens, heads)
                assert not w or tiles - w < 256
                s, w = key_split(d, tokens, heads, kb, 1, True)
                assert s in (0, 2, 4) and w == 0
                for m in (2, 4):
                    assert key_split(d, tokens, heads, kb, m, False) in ((0, 0), (2, 0))
