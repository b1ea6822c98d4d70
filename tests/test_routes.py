"""CPU checks of the rules that pick a route by size, on both sides of their lines."""
import ctypes

import pytest


@pytest.mark.parametrize("rows,columns,batch,one", [
    (512, 2048, 1, 1), (512, 2048, 64, 1), (16, 32, 1, 1), (16384, 128, 64, 1),
    (65536, 256, 64, 1), (4096, 2048, 17, 1), (4096, 2048, 32, 0), (6144, 2048, 8, 1),
    (8192, 1024, 17, 1), (8192, 1024, 32, 0), (16384, 1024, 1, 1), (16384, 1024, 64, 0),
    (4096, 4096, 8, 1), (4096, 4096, 16, 0), (512, 4096, 64, 1), (16, 4128, 1, 0),
    (512, 8192, 8, 0), (32768, 2048, 1, 0)])
def test_q8_products_split_their_rows_where_that_is_faster(pkg, rows, columns, batch, one):
    """A large product whose every row tile splits its input again took up to 2.7
    times as long as with the rows split once."""
    fn = pkg.load().ph_q8_one_launch
    assert fn(*(ctypes.c_size_t(n) for n in (rows, columns, batch))) == one
