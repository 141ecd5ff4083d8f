"""Ancestor search of the exact resampling on weights that reach every way a window is decided: keys that decide, keys
that tie (exact resolution), totals small enough for exact keys, and weights beyond the keys' range."""
import numpy as np
import pytest

from dogm_ctypes import DOGM, tuning_override
from oracle_ctypes import OracleDOGM
from parity_util import assert_bits_equal, assert_int_equal, small_params, small_scene

pytestmark = pytest.mark.gpu

SEED = 17


def _weights(kind, n, rng):
    if kind == "uniform":
        return np.full(n, 3e-7)
    if kind == "dominant":  # one weight per 256 dwarfs the others: draws on the small ones share keys
        w = np.full(n, 2.0 ** -24)
        w[rng.integers(0, 256):: 256] = 1.0
        return w
    if kind == "decades":
        return 10.0 ** (-30.0 * rng.random(n))
    if kind == "raw_units":  # totals of a few fixed-point units (2^-88): integer keys
        return rng.integers(0, 3, n) * 2.0 ** -88
    if kind == "below_units":  # truncated to 0 in fixed point, but for a few
        w = np.full(n, 2.0 ** -90)
        w[:: 97] = 2.0 ** -85
        return w
    if kind == "zero":
        return np.zeros(n)
    if kind == "sparse":
        return np.where(rng.random(n) < 2e-3, 1e-3, 0.0)
    if kind == "mixed_scales":  # windows far below the CDF before them
        w = np.full(n, 2.0 ** -80)
        w[: n // 2] = 2.0 ** 20
        return w
    if kind == "large":
        return np.where(rng.random(n) < 0.01, 2.0 ** 27, 1.0)
    assert kind == "infinite"
    w = rng.random(n)
    w[n // 3] = np.inf
    return w


@pytest.mark.parametrize("wide", [1, 2])
@pytest.mark.parametrize("kind", ["uniform", "dominant", "decades", "raw_units", "below_units", "zero", "sparse",
                                  "mixed_scales", "large", "infinite"])
@pytest.mark.parametrize("n,b", [(1, 0), (1023, 1), (1025, 300), (200_003, 20_001)])
def test_ancestors(kind, n, b, wide):
    rng = np.random.default_rng(n)
    w = _weights(kind, n + b, rng).astype(np.float32)
    p = small_params(gs=16, res=0.5, n=n, b=b)
    m = small_scene(gs=16, res=0.5).measurement(0)
    tuning_override({"merge_slice": wide})
    try:
        with DOGM(p, seed=SEED) as gpu:
            orc = OracleDOGM(p, seed=SEED)
            for o in (gpu, orc):
                o.update_measurement_grid(m)
            for draws in ("multinomial", "systematic"):
                gpu.set_resampling_mode(draws)
                orc.set_draw_mode(draws)
                for o in (gpu, orc):
                    o.set_weight_array(w[:n])
                    if b:
                        o.set_birth_particles(weight=w[n:])
                    o.resampling()
                assert_int_equal(f"{kind} {draws}", gpu.get_resampled_indices(), orc.get_resampled_indices())
                assert_bits_equal(f"{kind} {draws}", gpu.get_particles()["weight"], orc.get_particles()["weight"])
            orc.close()
    finally:
        tuning_override(None)
