"""Attention over more than 512 rows: tiles of sixteen rows that share their pages run
as fp32 MFMAs, the rest item by item (stride_amd/csrc/tc_aux.hip). Bit for bit against
the oracle at the edges of the tile form: sequences that end inside a tile, positions
around page ends, tiles of one row, rows that share nothing, rows of two sequences in
turn; then lists other than the engine's, whose unlisted pages come from scratch, and
values (infinities, NaN, -0) that must not reach rows that do not see them."""
import numpy as np
import pytest
import torch

from stride_amd import harness, layout

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bf16_bits(a):
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)


def prompts(*spans):
    """(slots, positions) of consecutive rows: one (first, last + 1) span per sequence."""
    slots = [s for s, (a, b) in enumerate(spans) for _ in range(a, b)]
    return np.array(slots, np.int32), np.array([p for a, b in spans for p in range(a, b)], np.int32)


def make(seed, slots, pos, n_kv, hd, page, k=None, v=None):
    rng = np.random.default_rng(seed)
    m, cap, ns = len(slots), int(pos.max()) + 1, int(slots.max()) + 1
    q = rng.standard_normal((m, n_kv * 4, hd)).astype(np.float32)
    k = bf16_bits(rng.standard_normal((ns, n_kv, cap, hd))) if k is None else k
    v = bf16_bits(rng.standard_normal((ns, n_kv, cap, hd))) if v is None else v
    kv = harness.PagedKv.create(ns, cap, n_kv, hd, 1, page, DEV, shuffle_seed=seed + 1)
    kv.fill_dense(0, 0, torch.from_numpy(k.view(np.int16)))
    kv.fill_dense(0, 1, torch.from_numpy(v.view(np.int16)))
    return q, k, v, kv, -(-cap // 64)


def run(q, kv, slots, pos, n_kv, hd, pages, **kw):
    out = harness.attention(torch.from_numpy(q.reshape(len(slots), -1)).to(DEV), kv, torch.from_numpy(slots).to(DEV),
                            torch.from_numpy(pos).to(DEV), n_kv, hd, hd ** -0.5, max_pages=pages, **kw)
    torch.cuda.synchronize()
    return layout.untile_lanes(out.cpu(), len(slots)).numpy().view(np.uint16)


def interleaved(a, b):
    s, p = prompts(a, b)
    order = np.argsort(p, kind="stable")
    return s[order], p[order]


CASES = [prompts((0, 513)), prompts((0, 250), (3, 210), (190, 300)),                # sequences ending inside tiles
         prompts(*[(40 + i, 90 + i) for i in range(11)]),                           # 50 rows each: three in a tile
         interleaved((0, 300), (1, 290)),                                           # two sequences in turn
         (np.arange(530, dtype=np.int32) % 37, (np.arange(530) * 7 % 200).astype(np.int32)),  # nothing shared
         prompts((100, 612), (0, 1))]                                               # a tile of one row


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("n_kv,hd,page", [(2, 64, 16), (1, 128, 64), (1, 32, 32)])
def test_tiles(exact, case, n_kv, hd, page):
    print("attention tiles", case, n_kv, hd, page, flush=True)
    slots, pos = CASES[case]
    q, k, v, kv, pages = make(case + hd, slots, pos, n_kv, hd, page)
    got = run(q, kv, slots, pos, n_kv, hd, pages)
    assert np.array_equal(got, exact.tc_attention(q, k, v, slots, pos, hd ** -0.5))


def test_partial_lists(exact):
    """Listed pages are summed and stored, the others combined from scratch: two calls
    that list a page each in turn give the whole list's bits, for tiles that share."""
    print("attention tiles, partial lists", flush=True)
    slots, pos = prompts((60, 610))
    q, k, v, kv, pages = make(5, slots, pos, 1, 64, 16)
    items = [(j, c) for j in range(len(pos)) for c in range((pos[j] >> 6) + 1)]
    scratch = torch.zeros(len(pos) * pages * 264, dtype=torch.float32, device=DEV)
    for half in (0, 1):
        part = torch.tensor([it for n, it in enumerate(items) if n % 2 == half], dtype=torch.int32, device=DEV).reshape(-1)
        got = run(q, kv, slots, pos, 1, 64, pages, items=part, scratch=scratch)
    assert np.array_equal(got, exact.tc_attention(q, k, v, slots, pos, 0.125))


def test_unseen_positions_stay_out(exact):
    """A row's result does not depend on later positions, whatever they hold, nor on
    the sign of zeros: rows before a non-finite position equal the same rows without it."""
    print("attention tiles, unseen values", flush=True)
    slots, pos = prompts((0, 520))
    q, k, v, kv, pages = make(6, slots, pos, 1, 64, 16)
    v[0, 0, ::3] = 0x8000  # -0
    k2, v2 = k.copy(), v.copy()
    for at, bits in ((70, 0x7F80), (201, 0xFF80), (333, 0x7FC0), (450, 0x7F80)):
        v2[0, 0, at, ::5] = bits
        k2[0, 0, at, 1::7] = bits
    want = run(q, make(6, slots, pos, 1, 64, 16, k, v)[3], slots, pos, 1, 64, pages)
    assert np.array_equal(want, exact.tc_attention(q, k, v, slots, pos, 0.125))
    got = run(q, make(6, slots, pos, 1, 64, 16, k2, v2)[3], slots, pos, 1, 64, pages)
    assert np.array_equal(got[:70], want[:70])
    assert not np.array_equal(got[70], want[70])
