"""GPU: W8A16 products of more than 64 rows, in the prompt-sized kernel at the
edges of its tiles, K halves and scale groups and in the split-K kernel beside
it, against the product in 64 bits.  Bar: 1e-3
normwise per row, the W8A16 bar (fp16 rounding of an output leaves 2^-11)."""
import numpy as np
import pytest

from devutil import empty_dev, stream, to_dev, to_dev_raw, to_host
from test_gpu_w8a16 import TOL, _cache, operands, packed_dev, rows_close

pytestmark = pytest.mark.gpu


def both(tl, dx, w, ds, M, N, K, gs):
    """fp16(x @ W) from the row-major weights and from the packed ones."""
    out, dw = empty_dev((M, N)), to_dev_raw(w)
    tl.w8a16_matmul(dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), out.data_ptr(), M, N, K, gs, stream())
    dh, dp = to_dev(np.zeros((M, N), np.uint16)), packed_dev(tl, w)
    tl.w8a16_matmul_residual(dx.data_ptr(), dp.data_ptr(), ds.data_ptr(), dh.data_ptr(), M, N, K, gs, stream(),
                             packed=True)
    return to_host(out), to_host(dh)


def product(x, w, s, K, gs):
    """x @ dequant(w, s) in 64 bits (the outputs here are too many for the oracle)."""
    sc = np.repeat(s.view(np.float16).astype(np.float64).reshape(-1, w.shape[1]), gs, axis=0)[:K]
    return x.view(np.float16).astype(np.float64) @ (w.astype(np.float64) * sc)


# Shapes at the edges of both kernels' tiles; which runs each is the planner's
# choice (TILE_SHAPES states it).
@pytest.mark.parametrize("M,N,K,gs", [
    (65, 36304, 32, 32),     # one row over, one k step: no chunk at all, a column tail
    (127, 18608, 64, 64),    # one chunk of two steps: the second K half is empty
    (128, 18432, 96, 32),    # full tiles, an unpaired last step
    (129, 18304, 160, 128),  # one row over, a partial last scale group
    (257, 9232, 128, 32),    # two groups per chunk, a column tail
    (320, 8208, 288, 64),    # several row tiles, K % 64 == 32 inside a group
    (200, 6560, 2080, 512),  # few rows with a long K; groups across chunks and the K halves' boundary
    (2390, 1008, 192, 256),  # more row tiles than a panel, a group longer than K
    (9250, 256, 64, 32),     # one column tile
    (600, 8192, 1056, 128),  # 128 x 192 tiles
])
def test_w8a16_tile_edges(tl, orc, M, N, K, gs):
    rng = np.random.default_rng(M + 3 * N + 7 * K + gs)
    x, w, s = operands(orc, rng, M, N, K, gs)
    ref = product(x, w, s, K, gs)
    got, got_p = both(tl, to_dev(x), w, to_dev(s), M, N, K, gs)
    assert rows_close(got, ref) <= TOL
    # zero residual: fp16(0 + v) drops only the sign of a -0
    assert np.array_equal(np.where(got == 0x8000, 0, got), got_p)


# Every tile of the kernel in both layouts, at the edges of its rows, columns, K
# chunks, K halves and scale groups: (M, N, K, group size), the tile with
# row-major weights and with packed ones.
TILE_SHAPES = [
    ((641, 9232, 32, 64), (128, 256), (128, 256)),     # one row over; one k step: no chunk at all
    ((257, 16400, 64, 64), (128, 256), (64, 128)),     # one chunk: the second K half is empty; several rounds
    ((2048, 4096, 96, 256), (128, 256), (128, 256)),   # full tiles, an unpaired last step, a group longer than K
    ((641, 9232, 160, 128), (128, 256), (128, 256)),   # a partial last group
    ((2047, 4080, 1056, 128), (128, 256), (128, 256)), # rows and columns short of the last tile, groups over chunks
    ((585, 8208, 160, 128), (128, 192), (128, 192)),
    ((65, 24592, 96, 128), (128, 128), (128, 128)),    # 63 rows of padding
    ((129, 16400, 288, 64), (64, 256), (64, 256)),     # K % 64 == 32 inside a group
    ((65, 16400, 2080, 512), (64, 192), (64, 192)),    # a group over the boundary of the K halves
    ((65, 12304, 1056, 512), (64, 128), (64, 128)),
    ((9250, 1008, 192, 256), (128, 192), (64, 128)),   # more row tiles than a panel
    ((200, 16400, 1056, 32), (128, 192), (128, 192)),  # two groups per chunk, from here
    ((65, 24592, 1120, 32), (128, 128), (128, 128)),
    ((129, 16400, 1056, 32), (64, 256), (64, 256)),
    ((65, 18608, 1056, 32), (64, 192), (64, 192)),
    ((129, 9232, 1056, 32), (64, 128), (64, 128)),
]


@pytest.mark.parametrize("shape,tile,tile_packed", TILE_SHAPES)
def test_w8a16_every_tile(tl, orc, shape, tile, tile_packed):
    M, N, K, gs = shape
    assert tl.w8a16_plan(*shape) == ("tile", *tile) and tl.w8a16_plan(*shape, packed=True) == ("tile", *tile_packed)
    rng = np.random.default_rng(M + 3 * N + 7 * K + gs)
    x, w, s = operands(orc, rng, M, N, K, gs)
    ref = product(x, w, s, K, gs)
    got, got_p = both(tl, to_dev(x), w, to_dev(s), M, N, K, gs)
    assert rows_close(got, ref) <= TOL
    assert np.array_equal(np.where(got == 0x8000, 0, got), got_p)


def test_w8a16_tile_scales(tl, orc):
    """Zero scales (whole columns, first, middle and last groups), negative and
    subnormal ones, and scales far apart."""
    M, N, K, gs = 96, 24592, 512, 64
    rng = np.random.default_rng(8)
    x, w, s = operands(orc, rng, M, N, K, gs)
    f = s.view(np.float16).reshape(K // gs, N)
    f[:, 3] = 0
    f[0, 5] = f[1, 5] = f[4, 6] = f[-1, 7] = f[3, 17:40] = 0
    f[2, 8] = -f[2, 8]
    f[1, 9], f[5, 10] = 6e-8, 3e-6   # subnormal
    # (64 products of |x| < 5, |w| <= 128, x of unit variance: |sum| < 6 * 128 * 8, times 5 below 65504)
    f[2, 11], f[3, 11] = 5.0, 1e-5
    f[6, 12] = -0.0
    ref = product(x, w, s, K, gs)
    got, got_p = both(tl, to_dev(x), w, to_dev(s), M, N, K, gs)
    g = got.view(np.float16).astype(np.float64)
    cols = np.abs(g - ref).max(axis=0) / np.maximum(np.abs(ref).max(axis=0), 1e-30)
    assert np.all(g[:, 3] == 0) and cols.max() <= TOL  # per column: small columns count as much
    assert np.array_equal(np.where(got == 0x8000, 0, got), got_p)


def test_w8a16_tile_infinite_scales(tl, orc):
    """Infinite and NaN scales: what folding each group's product gives, +-inf
    by the product's sign (two infinite groups in a row, or one before a zero
    scale, included), NaN where it is zero."""
    M, N, K, gs = 2047, 4080, 512, 64
    rng = np.random.default_rng(9)
    x, w, s = operands(orc, rng, M, N, K, gs)
    f = s.view(np.float16).reshape(K // gs, N)
    inf = np.inf
    for col, groups in {20: {2: inf}, 21: {2: inf, 3: inf}, 22: {2: inf, 3: 0}, 23: {0: inf}, 24: {7: inf},
                        25: {1: inf, 3: inf}, 26: {2: -inf}, 27: {2: inf, 3: -inf}, 28: {2: np.nan}, 29: {2: inf},
                        30: {2: 0, 3: inf}, 31: {1: inf, 6: inf}}.items():
        for g, v in groups.items():
            f[g, col] = v
    w[128:192, 29] = 0
    cols = np.arange(20, 32)
    # K halves of four groups each: (half, group, row, column)
    p = np.einsum("mgk,gkc->gmc", x.view(np.float16).astype(np.float64).reshape(M, 8, 64),
                  w[:, cols].astype(np.float64).reshape(8, 64, -1)).reshape(2, 4, M, -1)
    with np.errstate(invalid="ignore"):
        ref = (p * f[:, None, cols].astype(np.float64).reshape(2, 4, 1, -1)).sum(axis=1).sum(axis=0)
    got, got_p = both(tl, to_dev(x), w, to_dev(s), M, N, K, gs)
    g = got.view(np.float16).astype(np.float64)
    # (opposite infinities within a half: not a number in the fold, not finite here)
    same = (g[:, cols] == ref) | (np.isnan(g[:, cols]) & np.isnan(ref))
    clash = np.isin(cols, (21, 25, 27)) & np.isnan(ref) & np.isinf(g[:, cols])
    assert np.all(same | clash)
    assert np.isinf(ref[:, [0, 2, 3, 4, 6, 10]]).all() and np.isinf(ref[:, 1]).sum() > M // 4
    other = np.ones(N, bool)
    other[cols] = False
    sc = np.repeat(f[:, other].astype(np.float64), gs, axis=0)
    assert rows_close(got[:, other], x.view(np.float16).astype(np.float64) @ (w[:, other] * sc)) <= TOL
    h = got_p.view(np.float16).astype(np.float64)
    assert np.all((g == h) | (np.isnan(g) & np.isnan(h)))


def test_w8a16_tile_unaligned_output(tl, orc):
    """An output base two bytes past a 16-byte boundary: element stores, and
    nothing outside the matrix is written."""
    M, N, K, gs = 300, 8208, 128, 128
    rng = np.random.default_rng(4)
    x, w, s = operands(orc, rng, M, N, K, gs)
    dx, dw, ds = to_dev(x), to_dev_raw(w), to_dev(s)
    out, off = empty_dev((M, N)), to_dev(np.full(M * N + 2, 0x3555, np.uint16))
    tl.w8a16_matmul(dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), out.data_ptr(), M, N, K, gs, stream())
    tl.w8a16_matmul(dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), off.data_ptr() + 2, M, N, K, gs, stream())
    got = to_host(off)
    assert np.array_equal(got[1:-1], to_host(out).reshape(-1)) and got[0] == got[-1] == 0x3555


def test_w8a16_tile_element_stores(tl, orc):
    """The same in the tile kernel."""
    M, N, K, gs = 585, 8208, 160, 128
    assert tl.w8a16_plan(M, N, K, gs)[0] == "tile"
    rng = np.random.default_rng(14)
    x, w, s = operands(orc, rng, M, N, K, gs)
    dx, dw, ds = to_dev(x), to_dev_raw(w), to_dev(s)
    out, off = empty_dev((M, N)), to_dev(np.full(M * N + 2, 0x3555, np.uint16))
    tl.w8a16_matmul(dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), out.data_ptr(), M, N, K, gs, stream())
    tl.w8a16_matmul(dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), off.data_ptr() + 2, M, N, K, gs, stream())
    got = to_host(off)
    assert np.array_equal(got[1:-1], to_host(out).reshape(-1)) and got[0] == got[-1] == 0x3555


@pytest.mark.parametrize("paged,B,Hkv,kernels", [
    (False, 650, 16, ("tile", "split-k")),  # q, and k and v
    (True, 650, 16, ("tile", "split-k")),
    (False, 1200, 32, ("tile", "tile")),
    (True, 1200, 32, ("tile", "tile")),
])
def test_project_tiles_equal_products(tl, orc, paged, B, Hkv, kernels):
    """The projections whose q part, or all parts, run in the tile kernel."""
    assert tuple(tl.w8a16_plan(B, n * 128, 320, 64)[0] for n in (4 * Hkv, Hkv)) == kernels
    test_project_large_batch_equals_products(tl, orc, paged, B, Hkv, 128)


@pytest.mark.parametrize("paged,B,Hkv,D", [
    (False, 130, 2, 64),    # all columns to the split-K kernel
    (True, 650, 8, 128),    # as the first, with more columns
    (False, 1200, 8, 256),  # q to the tile kernel, k and v to the split-K one
    (True, 1200, 8, 256),
])
def test_project_large_batch_equals_products(tl, orc, paged, B, Hkv, D):
    """The fused projection's cache bytes and q_out are those of the separate
    products, whatever columns share the call."""
    from devutil import read_dev
    rng = np.random.default_rng(31 + paged)
    G, hidden, gs = 4, 320, 64
    row, Hq = Hkv * D, Hkv * G
    lens = [int(v) for v in rng.integers(1, 12, size=B)]
    g, _, ids, _k = _cache(tl, orc, np.random.default_rng(6), 1, Hkv, D, 16, lens, paged)
    g2, _, ids2, _k2 = _cache(tl, orc, np.random.default_rng(6), 1, Hkv, D, 16, lens, paged)
    x = orc.f2h(rng.standard_normal((B, hidden)).astype(np.float32))
    ws = [operands(orc, rng, 1, n, hidden, gs)[1:] for n in (row, row, Hq * D)]
    dx = to_dev(x)
    dev = [(to_dev_raw(w), to_dev(s)) for w, s in ws]
    (dwk, dsk), (dwv, dsv), (dwq, dsq) = dev
    batch, q_out = tl.DecodeBatch(g, B, Hq), empty_dev((B, Hq * D))
    batch.prepare(ids, stream())
    batch.project(0, dx.data_ptr(), hidden, gs, dwk.data_ptr(), dsk.data_ptr(), dwv.data_ptr(), dsv.data_ptr(),
                  dwq.data_ptr(), dsq.data_ptr(), q_out.data_ptr(), stream())
    outs = [empty_dev((B, n)) for n in (row, row, Hq * D)]
    for (dw, ds), o in zip(dev, outs):
        tl.w8a16_matmul(dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), o.data_ptr(), B, o.shape[1], hidden, gs, stream())
    batch2 = tl.DecodeBatch(g2, B, Hq)
    batch2.prepare(ids2, stream())
    batch2.append(0, 1, outs[0].data_ptr(), outs[1].data_ptr(), stream())
    n = g.slot_bytes() // 2 * (B + 1)
    assert np.array_equal(read_dev(g.pool(), n), read_dev(g2.pool(), n))
    assert np.array_equal(to_host(q_out), to_host(outs[2]))
    assert rows_close(to_host(q_out), product(x, *ws[2], hidden, gs)) <= TOL
