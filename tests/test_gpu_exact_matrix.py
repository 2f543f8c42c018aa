"""The exact path's batched GEMMs (four batch lanes, stride_amd/csrc/exact.hip) against
the oracle's restatement of the CPU exact path, bit for bit, at the edges of their
tiles: rows around multiples of 16 and 64, weight groups that leave part of a
workgroup's rows dead, K of less than one line per chain up to partial last batches,
and a shape for every form that the dispatch picks."""
import numpy as np
import pytest
import torch

from stride_amd import exact as E
from stride_amd import tc
from stride_amd._lib import GemmResidualParams, KvRef, LmFullParams, LmGreedyParams, Mlp13Params, NormParams, QkvParams

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bf16(rng, *shape, std=0.05):
    return (np.ascontiguousarray(rng.standard_normal(shape) * std, np.float32).view(np.uint32) >> 16).astype(np.uint16)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def groups(w, order=None):
    return dev(E.pack_groups(w.view(np.int16), order))


def same(got, want):
    return np.array_equal(np.ascontiguousarray(got).view(np.uint32), np.ascontiguousarray(want).view(np.uint32))


# (rows, n, k): the 16 x 16 tiles they make pick the tile and waves of the launch.
SHAPES = [(2, 64, 8), (5, 100, 264), (16, 4096, 256), (17, 64, 2064),        # up to 256 tiles
          (9, 4104, 520),                                                    # one lane tile, more rows
          (4, 32772, 72),                                                    # one lane tile, a vocabulary
          (33, 2064, 1544),                                                  # up to 512 tiles, partial batches
          (49, 3076, 40), (64, 4096, 768),                                   # up to 1024
          (130, 2600, 96),                                                   # up to 1536
          (127, 3200, 288), (113, 3588, 24),                                 # up to 2048, four and odd lane tiles
          (250, 3000, 64)]                                                   # more


# Up to eight rows of many weights: the vector form (whole slices of 256 columns), its
# last workgroup partly dead; then the forms either side of its lines.
FEW_ROWS = [(2, 8196, 4096), (5, 14340, 1024), (8, 13320, 1280), (7, 35204, 2048), (3, 8228, 4352),
            (8, 8192, 4096), (5, 13316, 1032), (9, 8196, 4096), (8, 12292, 264), (6, 35204, 64), (4, 28676, 256),
            (2, 13316, 3072)]
# A line or two for every chain at most, more than one lane tile.
FEW_COLS = [(35, 3076, 512), (17, 4100, 64), (33, 3076, 256), (50, 2052, 8), (250, 4100, 136)]


@pytest.mark.parametrize("m,n,k", SHAPES + FEW_ROWS + FEW_COLS)
def test_matrix_gemms(exact, m, n, k):
    print("exact matrix gemm", m, n, k, flush=True)
    rng = np.random.default_rng(m + n + k)
    w, w3 = bf16(rng, n, k), bf16(rng, n, k)
    x, h = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    J, _, stride = E.lane_shape(m)
    xd, wd, w3d = dev(E.dim_major(x, stride)), groups(w), groups(w3)
    n4 = wd.shape[0] * 4
    logits = torch.zeros((n4, stride), device=DEV)
    E.k_lm_full(LmFullParams(E.lanes(m), tc.ptr(xd), E.mat(wd, k), tc.ptr(logits)), J)
    hd = dev(E.dim_major(h, stride))
    hd = torch.cat([hd, torch.zeros((n4 - n, stride), device=DEV)])
    E.k_gemm_residual(GemmResidualParams(E.lanes(m), tc.ptr(xd), E.mat(wd, k), tc.ptr(hd)), J)
    z = torch.zeros((n4, stride), device=DEV)
    E.k_mlp13(Mlp13Params(E.lanes(m), tc.ptr(xd), E.mat(wd, k), E.mat(w3d, k), tc.ptr(z)), J)
    best = torch.zeros((m, 2), dtype=torch.int32, device=DEV)
    best[:, 0], best[:, 1] = -8388608, -1
    E.k_lm_greedy(LmGreedyParams(E.lanes(m), tc.ptr(xd), E.mat(wd, k), n - 3, tc.ptr(best)), J)
    torch.cuda.synchronize()
    back = lambda t: t.cpu().numpy()[:n, :m].T  # noqa: E731
    assert same(back(logits), exact.gemm(w, x))
    assert same(back(hd), exact.gemm_residual(w, x, h))
    assert same(back(z), exact.mlp13(w, w3, x))
    rv, ri = exact.lm_greedy(w, n - 3, x)
    b = best.cpu().numpy()
    assert np.array_equal(b[:, 1], ri) and np.array_equal(b[:, 0].view(np.uint32), rv.view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(3, 64, 264), (18, 4096, 256), (37, 2064, 40), (70, 4096, 48), (130, 3200, 24)])
def test_lanes_inside_a_wider_buffer(exact, m, n, k):
    """x as the last lane groups of a wider buffer (it ends with the last live lane):
    lane, row and stride differ, the bits do not."""
    print("exact matrix gemm, a run of lanes", m, n, k, flush=True)
    rng = np.random.default_rng(m + n + k)
    w, x = bf16(rng, n, k), rng.standard_normal((m, k)).astype(np.float32)
    J, lane_groups, run = E.lane_shape(m)
    stride = run + 64
    wide = dev(np.full((k, stride), np.float32(np.nan)))
    wide[:, 64:64 + m] = dev(np.ascontiguousarray(x.T))
    wd = groups(w)
    out = torch.zeros((wd.shape[0] * 4, stride), device=DEV)
    l = tc.Lanes(m, lane_groups, stride, 0)
    E.k_lm_full(LmFullParams(l, tc.ptr(wide) + 4 * 64, E.mat(wd, k), tc.ptr(out) + 4 * 64), J)
    torch.cuda.synchronize()
    out = out.cpu().numpy()
    assert same(out[:n, 64:64 + m].T, exact.gemm(w, x))
    assert not out[:, :64].any()


@pytest.mark.parametrize("m,hd,kvh", [(3, 32, 1), (18, 64, 3), (70, 128, 2)])
def test_matrix_qkv(exact, m, hd, kvh):
    """q, k and v in one launch: row blocks that straddle the three matrices."""
    print("exact matrix qkv", m, hd, kvh, flush=True)
    rng = np.random.default_rng(m + hd)
    k, nkv, page, max_blocks = 328, kvh * hd, 64, 3
    nq = 4 * nkv
    wq, wk, wv = bf16(rng, nq, k), bf16(rng, nkv, k), bf16(rng, nkv, k)
    x, pos = rng.standard_normal((m, k)).astype(np.float32), rng.integers(0, max_blocks * page, m).astype(np.int32)
    rope = rng.standard_normal((max_blocks * page, hd // 2, 2)).astype(np.float32)
    rq, rk, rv = exact.qkv(wq, wk, wv, x, hd, rope, pos)
    J, _, stride = E.lane_shape(m)
    order = rng.permutation(m * max_blocks).astype(np.int32).reshape(m, max_blocks)
    arena = torch.zeros((m * max_blocks, 2, kvh, page, hd), device=DEV)
    table, posd, slot, roped, xd = dev(order), dev(pos), dev(np.arange(m, dtype=np.int32)), dev(rope), dev(E.dim_major(x, stride))
    kv = KvRef(tc.ptr(arena), tc.ptr(table), arena[0].numel(), arena[0].numel(), arena[0, 0].numel(), page * hd, max_blocks, hd)
    q = torch.zeros((m, nq), device=DEV)
    g = [groups(w, E.rope_group_rows(w.shape[0], hd)) for w in (wq, wk, wv)]
    E.k_qkv(QkvParams(E.lanes(m), tc.ptr(xd), E.mat(g[0], k), E.mat(g[1], k), E.mat(g[2], k), tc.ptr(q), nq, kv,
                      tc.ptr(roped), tc.ptr(slot), tc.ptr(posd), 0, hd), J)
    torch.cuda.synchronize()
    assert same(q.cpu().numpy(), rq)
    a = arena.cpu().numpy()
    rows = a[order[np.arange(m), pos // page], :, :, pos % page]  # [m][K|V][head][hd]
    assert same(rows[:, 0].reshape(m, -1), rk)
    # V keeps the plain row order of its packed groups: (d0, d0 + 1, d0 + D/2, ...) like K
    assert same(rows[:, 1].reshape(m, -1), rv)


@pytest.mark.parametrize("m", [2, 8])
def test_lanes_inside_a_wider_buffer_vector_form(exact, m):
    """As above for the vector form, which up to eight rows of many weights take."""
    test_lanes_inside_a_wider_buffer(exact, m, 8196, 4096)


@pytest.mark.parametrize("m,dim", [(4, 4), (7, 132), (33, 2048), (2, 4096)])
def test_norm_rows_equal_single_rows(m, dim):
    """Four-lane RMSNorm against the same rows one at a time (one lane, whose chains
    read their LDS items whole), at dims of less than a unit per chain upward."""
    print("exact norm", m, dim, flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + dim)
    h, w = torch.randn(m, dim, generator=g, device=DEV) * 3, torch.randn(dim, generator=g, device=DEV)
    J, _, stride = E.lane_shape(m)
    hd = E.dim_major(h, stride)
    out, one = torch.zeros_like(hd), torch.zeros(m, dim, device=DEV)
    E.k_norm(NormParams(E.lanes(m), tc.ptr(hd), tc.ptr(out), tc.ptr(w), dim, 1e-5), J)
    for r in range(m):
        E.k_norm(NormParams(E.lanes(1), tc.ptr(h[r]), tc.ptr(one[r]), tc.ptr(w), dim, 1e-5), 1)
    torch.cuda.synchronize()
    assert torch.equal(out[:, :m].T.contiguous().view(torch.int32), one.view(torch.int32))
    want = w.double() * (h.double() / torch.sqrt((h.double() ** 2).mean(1, keepdim=True) + 1e-5))
    assert torch.allclose(one.double(), want, rtol=2e-6, atol=0)
