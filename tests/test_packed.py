"""The runners of stride_amd.harness pass packed parameter blocks (no GPU): the library
they call is the one that was loaded, and every field of every block arrives where the
C structs have it."""
import ctypes as C
import os
import shutil
import subprocess
import sys

import pytest
import torch

from stride_amd import _lib, harness, tc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_packed_is_the_loaded_library(tmp_path):
    """load() of another path (relative, and the folder left afterwards): the packed entry
    points are that library's, not the default one's."""
    shutil.copy(_lib.LIB_PATH, tmp_path / "other.so")
    code = """
import os, sys
sys.path.insert(0, sys.argv[1])
from stride_amd import _lib
lib = _lib.load("./other.so")
os.chdir("/")
packed = _lib.packed()
print(packed._name, packed._handle == lib._handle)
print(sum("other.so" in line for line in open("/proc/self/maps")) > 0, _lib.LIB_PATH in open("/proc/self/maps").read())
"""
    res = subprocess.run([sys.executable, "-c", code, ROOT], cwd=tmp_path, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    assert res.stdout.split() == ["./other.so", "True", "True", "False"]


class Recorder:
    """Stands for the library: keeps the block and the other arguments of the last call."""

    def __getattr__(self, name):
        def call(*args):
            self.last = (name, *args)
            return 0
        return call


@pytest.fixture
def recorder(monkeypatch):
    rec = Recorder()
    monkeypatch.setattr(_lib, "packed", lambda: rec)
    tc.set_kernel_stream(77)
    yield rec
    tc.set_kernel_stream(None)


def fields(struct):
    """{name: value} of a ctypes structure, nested ones as tuples, pointers as ints."""
    out = {}
    for name, kind in struct._fields_:
        v = getattr(struct, name)
        out[name] = tuple(fields(v).values()) if isinstance(v, C.Structure) else (0 if v is None else v)
    return out


def received(rec, name, struct, *others):
    assert rec.last[0] == name and rec.last[2:] == (*others, 77)
    assert len(rec.last[1]) == C.sizeof(struct)
    return fields(struct.from_buffer_copy(rec.last[1]))


def tiles(rt, ct):
    return torch.zeros((rt, ct, 16, 16), dtype=torch.int16)


def test_gemm_blocks(recorder):
    w, w3, x, o = tiles(3, 5), tiles(4, 6), tiles(2, 5), tiles(2, 3)
    P = lambda t: t.data_ptr()  # noqa: E731
    l = (19, 2, 0, 0)
    harness.gemm_residual(w, x, o, 19, 2, 4)
    assert received(recorder, "stride_tc_gemm_residual", _lib.TcGemmResidualParams, 2, 4) == {
        "l": l, "x": P(x), "m": (P(w), 3, 80), "h": P(o)}
    harness.lm_full(w, x, 19, o)
    assert received(recorder, "stride_tc_lm_full", _lib.TcLmFullParams, 1) == {
        "l": l, "x": P(x), "m": (P(w), 3, 80), "logits": P(o)}
    harness.mlp13(w, w3, x, 19, o, 2, 1)
    assert received(recorder, "stride_tc_mlp13", _lib.TcMlp13Params, 2, 1) == {
        "l": l, "x": P(x), "w1": (P(w), 3, 80), "w3": (P(w3), 4, 96), "z": P(o)}
    harness.lm_greedy(w, x, 19, 47, o, 1, 2)
    assert received(recorder, "stride_tc_lm_greedy", _lib.TcLmGreedyParams, 1, 2) == {
        "l": l, "x": P(x), "m": (P(w), 3, 80), "vocab": 47, "best": P(o)}


def test_embed_and_norm_blocks(recorder):
    e, t, h, w = tiles(3, 5), torch.zeros(33, dtype=torch.int32), torch.zeros((3, 5, 16, 16)), torch.zeros(80)
    x = tiles(3, 5)
    P = lambda t: t.data_ptr()  # noqa: E731
    harness.embed(e, t, 33, 80, h)
    assert received(recorder, "stride_tc_embed", _lib.TcEmbedParams) == {
        "l": (33, 3, 0, 0), "embed": P(e), "tokens": P(t), "h": P(h), "dim": 80}
    harness.norm(h, 33, w, 0.25, False, x)
    assert received(recorder, "stride_tc_norm", _lib.TcNormParams, 0) == {
        "l": (33, 3, 0, 0), "h": P(h), "x": P(x), "weight": P(w), "dim": 80, "eps": 0.25}


@pytest.mark.parametrize("listed", [False, True])
def test_attention_and_qkv_blocks(recorder, listed):
    P = lambda t: t.data_ptr()  # noqa: E731
    kv = harness.PagedKv.create(2, 100, 3, 64, 2, 32, "cpu")
    kvf = tuple(fields(kv.ref).values())
    q, slot, pos = torch.zeros(5, 768), torch.zeros(5, dtype=torch.int32), torch.zeros(5, dtype=torch.int32)
    out, scratch = tiles(1, 48), torch.zeros(9)
    items = torch.zeros(14, dtype=torch.int32) if listed else None
    harness.attention(q, kv, slot, pos, 3, 64, 0.125, layer=1, max_pages=4, items=items, scratch=scratch if listed else None,
                      out_tiles=out, one_kernel=not listed)
    assert received(recorder, "stride_tc_attention", _lib.AttentionParams) == {
        "l": (5, 1, 0, 0), "q": P(q), "q_stride": 768, "out": P(out), "out_cols": 768, "kv": kvf, "row_slot": P(slot),
        "row_pos": P(pos), "items": P(items) if listed else 0, "item_count": 7 if listed else -1,
        "scratch": P(scratch) if listed else 0, "max_pages": 4, "rec_floats": 264, "layer": 1, "n_kv": 3, "n_q": 4,
        "head_dim": 64, "scale": 0.125}
    wq, wk, wv, x, rope = tiles(48, 2), tiles(12, 2), tiles(12, 2), tiles(1, 2), torch.zeros(4)
    harness.qkv(wq, wk, wv, x, 5, 64, rope, slot, pos, kv, 1, q)
    assert received(recorder, "stride_tc_qkv", _lib.TcQkvParams) == {
        "l": (5, 1, 0, 0), "x": P(x), "q": (P(wq), 48, 32), "k": (P(wk), 12, 32), "v": (P(wv), 12, 32), "q_out": P(q),
        "q_stride": 768, "kv": kvf, "rope": P(rope), "row_slot": P(slot), "row_pos": P(pos), "layer": 1, "head_dim": 64}
