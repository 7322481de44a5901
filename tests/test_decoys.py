"""The random orientations of the chance calibration: any whole number names a draw (its product modulo
2^32 enters the hash), one draw or several at a time give the same ones."""
import numpy as np
import pytest

from zebsdsolve_amd import _hash_u32, _unit_rand, decoys


def _one(n, draw):
    s = _hash_u32(np.arange(n, dtype=np.uint64) + 1) ^ np.uint64((draw * 0x9E3779B9) & 0xFFFFFFFF)
    u1, a2, a3 = _unit_rand(s), _unit_rand(s + np.uint64(1)) * 2 * np.pi, _unit_rand(s + np.uint64(2)) * 2 * np.pi
    ra, rb = np.sqrt(1 - u1), np.sqrt(u1)
    return np.stack([ra * np.sin(a2), ra * np.cos(a2), rb * np.sin(a3), rb * np.cos(a3)], -1).astype(np.float32)


@pytest.mark.parametrize("draw", [0, 1, 7, -1, -12345, 2 ** 31, 2 ** 40 + 3, 2 ** 70 + 5])
def test_any_whole_number_names_a_draw(draw):
    assert np.array_equal(decoys(9, draw), _one(9, draw))


@pytest.mark.parametrize("draws", [range(8), [3, -2], []])
def test_several_draws_are_the_single_ones(draws):
    got = decoys(5, np.array(list(draws), np.int64))
    assert got.shape == (len(draws), 5, 4)
    assert all(np.array_equal(g, decoys(5, d)) for g, d in zip(got, draws))


def test_a_fraction_names_none():
    with pytest.raises(TypeError):
        decoys(5, 1.5)
