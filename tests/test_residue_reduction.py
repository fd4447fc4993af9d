"""The reduction of the int8 products' int32 sums to residues (the epilogue of
k_gemm_i8 in uvatrmm_amd/csrc/uvt_split.hip), modelled in FP32 and checked
against exact integers over the whole int32 range: for every modulus up to 255
the result is congruent to the sum and fits a byte, with the quotient's
product off by one unit in the last place either way too (a fused multiply-add
is correctly rounded; the model allows for less)."""
import numpy as np
import pytest

MODS = [255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199]


@pytest.mark.parametrize("m", MODS)
def test_residue_is_congruent_and_fits_a_byte(m):
    c16 = 65536 % m
    c16 -= m if c16 > m // 2 else 0
    inv = np.float32(1.0) / np.float32(m)
    quarter = np.float32(0.25) * inv
    rng = np.random.default_rng(m)
    edges = [v + d for v in (-2**31, 0, 2**31 - 1, 128**2 * 130816, -127**2 * 130816) for d in range(-4 * m, 4 * m)]
    low = [(h << 16) + v for h in range(-32768, 32768, 331) for v in (0, 1, m - 1, m, 65535 - m, 65534, 65535)]
    x = np.concatenate([rng.integers(-2**31, 2**31, 400000), np.array(edges + low, dtype=np.int64)])
    x = x[(x >= -2**31) & (x < 2**31)]
    h, lo = x >> 16, x & 0xFFFF
    y = h * c16 + lo
    assert np.abs(y).max() < 2**23  # exact in FP32, factors within 24 bits
    assert np.array_equal(y.astype(np.float32).astype(np.int64), y)
    t = (y.astype(np.float64) * np.float64(inv) + np.float64(quarter)).astype(np.float32)
    for q in (np.floor(t), np.floor(np.nextafter(t, np.float32(-np.inf))), np.floor(np.nextafter(t, np.float32(np.inf)))):
        r = y - q.astype(np.int64) * m
        assert ((x - r) % m == 0).all()
        assert r.min() >= 0 and r.max() <= 255
