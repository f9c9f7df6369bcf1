"""The full-vocabulary passes scale a logit by the temperature as
float(double(x) * (1 / T in double)) (f_scaled in csrc/gs_full.hpp).  That is
the float quotient x / T the reference computes (src/sampler.rs:41) wherever
the quotient is a normal float, zero, infinite or NaN; below 2^-126 it may be
one step of 2^-149 off for a few even T (f_may_tie), and a row with such
elements and such a T is sorted whole.  The bound is exact: the product is within 2^-52 of
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


def _may_tie(T):
    """f_may_tie: only an even T has quotients that are midpoints of subnormal
    floats, and only where 1 / T is off by more than 2^-54 may the product lie
    beside the midpoint."""
    if not np.isfinite(T) or T < 2 or np.trunc(T / 2) != T / 2:
        return False
    n = int(T)      # |T iT - 1| > 2^-54, exactly
    num, den = (1.0 / np.float64(T)).as_integer_ratio()
    return abs(n * num - den) << 54 > den


def test_scaled_quotient_ties():
    """Products that are not the quotient: none without f_may_tie, and only
    below 2^-126 (where the rows with such elements are sorted whole)."""
    k = np.arange(1, 1 << 16, dtype=np.float64)
    rng = np.random.default_rng(3)
    Ts = list(range(1, 600)) + [0.25 * n for n in range(1, 200)] + list(rng.uniform(0.05, 300.0, 200))
    found = 0
    for T in np.asarray(Ts, np.float32):
        x = (k * 2.0 ** -149).astype(np.float32)
        off = x / T != (x.astype(np.float64) * (1.0 / np.float64(T))).astype(np.float32)
        assert not off.any() or _may_tie(T), T
        assert (x[off] < T * np.float32(2.0 ** -126)).all()
        found += off.any()
    assert found and not any(_may_tie(np.float32(T)) for T in (0.7, 0.75, 0.9, 1.5, 2.0, 4.0, 6.0, 10.0))


@pytest.mark.gpu
@pytest.mark.parametrize("penalized", [False, True])
def test_tied_quotients(gpu, torch, oracle, penalized):
    """T = 98: 147 steps of 2^-149 over T is 1.5 steps, a midpoint that rounds
    to 2; the product would round to 1, and the order among the logits of one
    step would be lost.  A draw for every part of the row, with the tied
    logits in the row itself or left behind by the penalty."""
    import workloads
    B, V = 256, 2001
    rng = np.random.default_rng(8)
    lg = (rng.standard_normal(V) * 150).astype(np.float32)
    at = rng.choice(V, 100, replace=False)
    lg[at] = (rng.choice([98, 147], 100) * 2.0 ** -149).astype(np.float32)
    rec = None
    if penalized:
        lg[at] = (lg[at].astype(np.float64) * 2).astype(np.float32)
        rec = np.tile(at.astype(np.uint32), (B, 1))
    lg = np.tile(lg, (B, 1))
    u = ((np.arange(B) + 0.5) / B).astype(np.float32)
    params = workloads.params_rows(zip([98.0] * B, [0] * B, [0.97] * B, [2.0 if penalized else 1.0] * B))
    tok = torch.zeros(B, dtype=torch.int32, device="cuda")
    st = torch.full((B,), 99, dtype=torch.int32, device="cuda")
    s = gpu.Sampler(1.0, 0, 0.95, 1.0, seed=1)
    print("tied quotients", penalized, flush=True)
    s.sample_batch(torch.from_numpy(lg).cuda(), tok,
                   params=torch.from_numpy(np.ascontiguousarray(params).view(np.uint8)).cuda(),
                   recent=None if rec is None else torch.from_numpy(rec.view(np.int32)).cuda(),
                   u=torch.from_numpy(u).cuda(), status=st)
    torch.cuda.synchronize()
    want = oracle.sample_batch(lg, params, u, recent=rec, nthreads=8)
    assert (st.cpu().numpy() == 0).all()
    assert np.array_equal(tok.cpu().numpy().astype(np.int64), want)
