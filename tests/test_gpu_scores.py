"""GPU: get_attention_weights and softmax at the edges of their tiles, against
the oracle.  The weights keep the reference's sequential fmaf order, so every
output is bit-exact; softmax outputs are within one fp16 step of the oracle's
fp32 value (rounding 2^-11 relative, doubled for the order of the sum)."""
import numpy as np
import pytest

from devutil import empty_dev, stream, to_dev, to_host

pytestmark = pytest.mark.gpu


def bits(rng, shape, std=1.0):
    return (rng.standard_normal(shape) * std).astype(np.float16).view(np.uint16)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,Lq,Lk,D", [
    (1, 1, 1, 1),          # one product
    (2, 1, 8, 32),         # the smallest vector shape
    (3, 64, 256, 64),      # full 64 x 64 tiles
    (2, 65, 264, 64),      # ... with one query and eight keys over
    (2, 33, 129, 40),      # element stores (odd row pitch), a tile of one key
    (1, 130, 31, 128),     # three query tiles, half of a key tile
    (2, 200, 320, 136),    # two stages of dimensions, the second of one piece
    (1, 70, 96, 257),      # three stages, odd dimensions
])
def test_attention_weights_tiles_bit_exact(tl, orc, heads, Lq, Lk, D, causal):
    rng = np.random.default_rng(Lq * 7 + Lk + D)
    q, k = bits(rng, (1, heads, Lq, D)), bits(rng, (1, heads, Lk, D))
    dq, dk, w = to_dev(q), to_dev(k), to_dev(np.full((heads, Lq, Lk), 0x7E00, np.uint16))
    scale = D ** -0.5
    tl.get_attention_weights(dq.data_ptr(), dk.data_ptr(), w.data_ptr(), scale, 1, heads, Lq, Lk, D,
                             causal, stream())
    _, ref = orc.get_attention_weights(q, k, scale, 1, heads, Lq, Lk, D, causal)
    assert np.array_equal(to_host(w).reshape(ref.shape), ref)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,Lq,Lk,D", [
    (128, 200, 200, 64),   # exactly 512 tiles of 128 x 128, two on each of 256 CUs
    (128, 129, 264, 8),    # one query and eight keys over; one piece of dimensions
    (128, 129, 264, 72),   # ... two stages of dimensions, the second of one piece
    (128, 129, 257, 40),   # element stores
    (128, 129, 264, 33),   # element loads
    (128, 160, 257, 129),  # both; three stages, the last of one dimension
    (176, 257, 100, 16),   # the upper half of a wave's keys four wide, and empty in the next
])
def test_attention_weights_large_tiles_bit_exact(tl, orc, heads, Lq, Lk, D, causal):
    """Launches of 128 x 128 tiles: at least two for every CU."""
    assert -(-Lq // 128) * -(-Lk // 128) * heads >= 512 and Lq > 64
    test_attention_weights_tiles_bit_exact(tl, orc, heads, Lq, Lk, D, causal)


@pytest.mark.parametrize("off", [0, 1, 2])
def test_attention_weights_large_tiles_unaligned_bases(tl, orc, off):
    """Large tiles with q and k, or the output, two bytes past a 16-byte
    boundary: element loads with vector stores, and the reverse."""
    rng = np.random.default_rng(6)
    heads, Lq, Lk, D = 128, 130, 136, 24
    q, k = bits(rng, (heads, Lq, D)), bits(rng, (heads, Lk, D))
    i, o = int(off == 1), int(off == 2)
    dq, dk = (to_dev(np.concatenate([np.zeros(i, np.uint16), t.reshape(-1)])) for t in (q, k))
    w = to_dev(np.full(heads * Lq * Lk + 2, 0x7E00, np.uint16))
    tl.get_attention_weights(dq.data_ptr() + 2 * i, dk.data_ptr() + 2 * i, w.data_ptr() + 2 * o, 0.2, 1, heads, Lq, Lk, D,
                             True, stream())
    _, ref = orc.get_attention_weights(q, k, 0.2, 1, heads, Lq, Lk, D, True)
    got = to_host(w)
    assert np.array_equal(got[o:o + ref.size], ref.reshape(-1)) and np.all(got[o + ref.size:] == 0x7E00)


def test_attention_weights_unaligned_bases_bit_exact(tl, orc):
    """Bases two bytes past a 16-byte boundary take the element path."""
    rng = np.random.default_rng(5)
    heads, Lq, Lk, D = 2, 40, 72, 64
    q, k = bits(rng, (heads, Lq, D)), bits(rng, (heads, Lk, D))
    dq = to_dev(np.concatenate([[0], q.reshape(-1)]).astype(np.uint16))
    dk = to_dev(np.concatenate([[0], k.reshape(-1)]).astype(np.uint16))
    w = empty_dev(heads * Lq * Lk + 1)
    tl.get_attention_weights(dq.data_ptr() + 2, dk.data_ptr() + 2, w.data_ptr() + 2, 0.125, 1, heads, Lq, Lk, D,
                             False, stream())
    _, ref = orc.get_attention_weights(q, k, 0.125, 1, heads, Lq, Lk, D, False)
    assert np.array_equal(to_host(w)[1:], ref.reshape(-1))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rows,S", [(1, 1), (5, 8), (3, 511), (4, 512), (9, 520), (2, 1024), (3, 1025),
                                    (2, 2048), (3, 2056), (2, 4096), (2, 4101), (1, 8192), (2, 8200)])
def test_softmax_row_lengths(tl, orc, rows, S, offset):
    rng = np.random.default_rng(rows + S)
    x = bits(rng, (rows, S), 2.0)
    x.reshape(-1)[0] = 0xFC00 if S > 1 else x.reshape(-1)[0]  # -inf: weight zero
    dx = to_dev(np.concatenate([np.zeros(offset, np.uint16), x.reshape(-1)]))
    y = empty_dev(rows * S + offset)
    tl.softmax(dx.data_ptr() + 2 * offset, y.data_ptr() + 2 * offset, rows, S, stream())
    got = to_host(y)[offset:].view(np.float16).astype(np.float64).reshape(rows, S)
    ref32, _ = orc.softmax(x, rows, S)
    ref32 = ref32.reshape(rows, S)
    assert np.all(np.abs(got - ref32) <= np.abs(ref32) * 2.0 ** -10 + 2.0 ** -24)


@pytest.mark.parametrize("rows,S", [(33001, 512), (17001, 1000), (8193, 2048), (8193, 2056), (4099, 4104)])
def test_softmax_streaming_stores(tl, orc, rows, S):
    """Outputs of more than 32 MB, whose stores bypass the caches, are those of
    the same rows in two calls of less, and the oracle's."""
    assert rows * S * 2 > 32 << 20 and rows * S < 32 << 20
    rng = np.random.default_rng(S)
    x = bits(rng, (rows, S), 2.0)
    dx, y, halves = to_dev(x), empty_dev((rows, S)), empty_dev((rows, S))
    tl.softmax(dx.data_ptr(), y.data_ptr(), rows, S, stream())
    h = rows // 2
    for a, n in ((0, h), (h, rows - h)):
        tl.softmax(dx.data_ptr() + 2 * a * S, halves.data_ptr() + 2 * a * S, n, S, stream())
    got = to_host(y)
    assert np.array_equal(got, to_host(halves))
    pick = np.concatenate([[0, 1, rows - 3, rows - 2, rows - 1], rng.integers(0, rows, size=60)])
    ref32, _ = orc.softmax(np.ascontiguousarray(x[pick]), len(pick), S)
    ref32 = ref32.reshape(len(pick), S)
    assert np.all(np.abs(got[pick].view(np.float16).astype(np.float64) - ref32) <= np.abs(ref32) * 2.0 ** -10 + 2.0 ** -24)


def test_softmax_masked_rows(tl):
    """A row of lowest values, one of -inf only, one with +inf, one with NaN:
    uniform, zero, NaN, NaN."""
    x = np.zeros((4, 40), np.float16)
    x[0], x[1], x[2, 3], x[3, 5] = -65504.0, -np.inf, np.inf, np.nan
    dx, y = to_dev(x.view(np.uint16)), empty_dev((4, 40))
    tl.softmax(dx.data_ptr(), y.data_ptr(), 4, 40, stream())
    got = to_host(y).view(np.float16)
    assert np.all(got[0] == np.float16(1 / 40)) and np.all(got[1] == 0)
    assert np.all(np.isnan(got[2])) and np.all(np.isnan(got[3]))
