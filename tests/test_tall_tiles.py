"""Dense products of 257 - 288 rows against many weight rows (the head of a wide tree): one tile of 288 rows, whose ring has two slots."""
import pytest
import test_tile_kinds as tiles


# stages of 64 k: the ring's two, four and six; a last block of 16 weight rows, of 240 and of 256; the first and the last row count
@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [(257, 130064, 256), (288, 131056, 128), (273, 131072, 128), (288, 130064, 384)])
def test_one_tile_of_288_rows(T, N, K):
    tiles.test_every_tile_of_packed_weights(T, N, K, 1)
