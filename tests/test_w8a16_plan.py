"""CPU: the kernel and tile that a W8A16 product runs (tl_w8a16_plan), on the 256
CUs of an MI355X.  The measured times (us, split-K against tile) are of K rows
of int8 weights in groups of 128 on one card."""
import pytest

CUS = 256


@pytest.fixture(scope="module")
def tl():
    import tinyllm_kv
    tinyllm_kv.load()
    return tinyllm_kv


def plan(tl, M, N, K, gs=128, packed=False):
    return tl.w8a16_plan(M, N, K, gs, packed=packed, num_cus=CUS)


@pytest.mark.parametrize("M,N,K,gs", [
    (1152, 8192, 512, 128),   # row-major 33 against 46
    (1536, 6144, 512, 128),   # 33 against 38
    (641, 11264, 512, 128),   # 26 against 30
    (1152, 2048, 512, 128),   # 11.8 against 12.8
    (192, 14336, 512, 128),   # 12.3 against 13.2
    (768, 4096, 4096, 32),    # 54 against 62
    (1536, 2048, 4096, 32),   # 53 against 62
    (641, 8192, 4096, 32),    # 98 against 118
    (257, 28672, 4096, 32),   # packed 134 against 149
    (80, 11264, 4096, 32),    # 42 against 44.5
    (641, 4096, 4096, 128),   # the q part of a projection of 641 x (4096 + 2 x 1024): 63 against 67 packed
    (641, 4096, 2048, 128),   # ... (4096 + 2 x 512): 33 against 43 row-major
    (1152, 2048, 2048, 128),  # ... (2048 + 2 x 256): 31 against 43 row-major
])
def test_split_k_where_the_tiles_are_slower(tl, M, N, K, gs):
    for packed in (False, True):
        assert plan(tl, M, N, K, gs, packed)[0] == "split-k"


@pytest.mark.parametrize("M,N,K", [
    (2048, 4096, 4096),    # 118 against 78
    (585, 8192, 8192),
    (1024, 4096, 4096),
    (400, 14336, 1024),    # 48 against 28
    (320, 14336, 14336),   # 330 against 187
    (4096, 1024, 1024),    # 29 against 17
    (192, 8192, 2048),     # 29 against 19
    (256, 5120, 5120),
])
def test_tiles_where_they_are_faster(tl, M, N, K):
    for packed in (False, True):
        assert plan(tl, M, N, K, 128, packed)[0] == "tile"


def test_tile_shape_by_the_time_of_its_rounds(tl):
    """Row-major 1536 x 4096 x 4096: one round of the largest tile (75 us), not
    three of the smallest (97).  Packed, where two of the smallest share a CU,
    three rounds of it (68 against 70)."""
    assert plan(tl, 1536, 4096, 4096) == ("tile", 128, 256)
    assert plan(tl, 1536, 4096, 4096, packed=True) == ("tile", 64, 128)
    # groups of 32 leave no room for two: 155 us, 197 in sixteen rounds of the smallest
    assert plan(tl, 4096, 8192, 1024, 32, packed=True) == ("tile", 128, 192)


def test_kernel_by_size_alone(tl):
    """The kernel, and with it the order of the sums, is the same for both
    layouts, whatever the tile."""
    for M in (1, 64, 65, 100, 256, 257, 500, 640, 641, 1000, 2048, 8192):
        for N in (16, 256, 1024, 4096, 8192, 8208, 14336):
            for K in (32, 96, 512, 2048, 4096, 4128, 14336):
                for gs in (32, 64, 128, 512):
                    a, b = plan(tl, M, N, K, gs), plan(tl, M, N, K, gs, True)
                    assert a[0] == b[0]
                    assert (a[0] == "decode") == (M <= 64 and K % 128 == 0 and K <= 4096)
                    assert M > 64 or a[0] != "tile"
                    assert a[0] != "tile" or (a[1] in (64, 128) and a[2] in (128, 192, 256))
                    assert gs > 32 or a[1:] != (128, 256)


def test_plan_rejects_and_falls_back(tl):
    assert plan(tl, 100, 100, 4096)[0] == "reference" and plan(tl, 100, 128, 100)[0] == "reference"
    assert plan(tl, 100, 128, 4096, 16)[0] == "reference"
    for bad in ((0, 16, 32, 32), (1, 0, 32, 32), (1, 16, 0, 32), (1, 16, 32, 0)):
        with pytest.raises(tl.TinyLLMError):
            tl.w8a16_plan(*bad)
