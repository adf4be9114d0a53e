"""Dense products of 257 - 288 rows against many weight rows (the head of a wide tree): one tile of 288 rows, whose ring has two slots."""
import pytest
import test_tile_kinds as tiles


# stages of 64 k: the ring's two, four and six; a last block of 16 weight rows, of 240 and of 256; the first and the last row count
@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [(257, 130064, 256), (288, 131056, 128), (273, 131072, 128), (288, 130064, 384)])
def test_one_tile_of_288_rows(T, N, K):
    tiles.test_every_tile_of_packed_weights(T, N, K, 1)


# several tiles of 288 tokens, the last of them in part, against fewer weight rows; K in slabs: of five stages, the fewest, six and seven, and a shorter last slab
MORE = [(545, 28688, 384, 1), (576, 28672, 128, 1), (1150, 16384, 256, 1), (2250, 8176, 128, 1), (280, 28688, 640, 2), (560, 14352, 768, 2), (288, 18448, 896, 3), (280, 20496, 1280, 3)]


def test_shapes_get_the_tile_of_288_rows():
    from umbrella_amd import _lib
    kind = _lib.load().umb_gemm_tile_kind
    assert all(kind(*s, 1) == 7 for s in [(257, 130064, 256), (288, 131056, 128), (273, 131072, 128), (288, 130064, 384)])
    assert all(kind(*s) == 7 for s in MORE) and kind(289, 130064, 256, 1) != 7 and kind(256, 130064, 256, 1) != 7
    assert all(kind(*s) != 7 for s in [(280, 28688, 512, 2), (288, 16400, 256, 2), (280, 65552, 384, 2), (280, 20496, 256, 3)])      # slabs of fewer than five stages
    assert kind(128, 130064, 256, 1) < 0 and kind(300, 256, 0, 1) < 0


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K,S", MORE)
def test_several_tiles_of_288_rows(T, N, K, S):
    tiles.test_every_tile_of_packed_weights(T, N, K, S)
