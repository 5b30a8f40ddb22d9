"""pa_transform_len (host only): the length of the transform that serves a block."""
import pytest

import privacyamplification_amd as P


@pytest.mark.parametrize("n,m,length", [
    (64, 32, 64), (96, 32, 128), (16384, 6144, 16384), (131072 + 32, 4096, 1 << 18), (3 << 16, 1 << 16, 1 << 18),
    ((1 << 18) + 32, 1 << 17, 3 << 17), (3 << 17, 1 << 17, 3 << 17), ((3 << 17) + 32, 1 << 17, 1 << 19),
    (3000032, 750016, 3 << 20), (1 << 22, 3 << 19, 1 << 22), (3 << 23, 9 << 20, 3 << 23),
    ((3 << 23) + 32, 9 << 20, 1 << 25), ((1 << 25) + 32, 1 << 20, 1 << 26), (1 << 29, 3 << 26, 1 << 29)])
def test_transform_len(n, m, length):
    assert P.transform_len(n, m) == length
    holds, touched, _ = P.block_extents(n, m)
    assert holds in (length, length // 3 * 4)
    assert touched["spec_key"] in (0, 4 * length)  # a complex value per two bits


@pytest.mark.parametrize("n,m,flags", [(1000, 96, 3), (1024, 1024, 3), (3 << 20, 3 << 18, P.XOR_KEY_REST), (1 << 30, 3 << 27, 3)])
def test_transform_len_of_unsupported_shapes(n, m, flags):
    assert P.transform_len(n, m, flags) == 0
