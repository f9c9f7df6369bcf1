"""The full-vocabulary passes scale a logit by the temperature as
float(double(x) * (1 / T in double)) (f_scaled in csrc/gs_full.hpp).  That is
the float quotient x / T the reference computes (src/sampler.rs:41) wherever
the quotient is a normal float, zero, infinite or NaN; below 2^-126 it may be
one step of 2^-149 off.  The bound is exact: the product is within 2^-52 of
the quotient, which lies 2^-49 or more from the nearest midpoint of two
floats.  Restated here in numpy, whose float and double arithmetic is IEEE's.
"""
import numpy as np
import pytest


def _draw(kind, rng, T, n):
    if kind == "logits":
        return (rng.standard_normal(n) * 6).astype(np.float32)
    if kind == "bits":      # every float: subnormal, huge, infinite, NaN
        x = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32).view(np.float32)
        x[:6] = [0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45]
        return x
    # quotients as close to a midpoint of two floats as a float x gets
    q = rng.integers(1 << 23, 1 << 24, n).astype(np.float64) + 0.5
    return (q * 2.0 ** rng.integers(-30, -15) * np.float64(T)).astype(np.float32)


@pytest.mark.parametrize("kind", ["logits", "bits", "midpoints"])
def test_scaled_quotient(kind):
    rng = np.random.default_rng(len(kind))
    Ts = [0.7, 0.8, 0.9, 1.3, 2.0, 1e-6, 1e6, np.inf, np.nan, 1e-45, 3e38]
    Ts += list(rng.uniform(0.05, 3.0, 40)) + list(2.0 ** rng.uniform(-126, 127, 40))
    with np.errstate(all="ignore"):
        for T in np.asarray(Ts, np.float32):
            x = _draw(kind, rng, T, 100000)
            want = x / T
            got = (x.astype(np.float64) * (1.0 / np.float64(T))).astype(np.float32)
            nan = np.isnan(want)
            assert (np.isnan(got) == nan).all(), T
            off = (want.view(np.uint32) != got.view(np.uint32)) & ~nan
            tiny = np.abs(want) < 2.0 ** -126
            assert not (off & ~tiny).any(), (T, x[off & ~tiny][:4])
            assert (np.abs(want[off].astype(np.float64) - got[off]) <= 2.0 ** -149).all(), T
