"""Full-vocabulary rows at the edges of the plans: rows whose largest logits
are penalized, rows whose softmax sum lies a little above a power of two (the
normalized sums then need the finest grids; half of them with a nucleus that
ends at the end of the row or not at all), and rows that the top logit
dominates.  Tokens must equal the oracle's, and the rows must stay on the
increment-histogram path (a fallback is exact too, but several times slower).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

B = 24


def _case(shape, V, rng):
    lg = (rng.standard_normal((B, V)) * rng.uniform(1.5, 3.0, (B, 1))).astype(np.float32)
    T = rng.uniform(0.5, 1.3, B).astype(np.float32)
    p = rng.choice([0.85, 0.9, 0.95, 1.0], B).astype(np.float32)
    rep = np.ones(B, np.float32)
    rec = rng.integers(0, V, (B, 256)).astype(np.uint32)
    u = rng.random(B, dtype=np.float32) * np.float32(0.99)
    for b in range(B):
        if shape == "penalized":
            top = np.argsort(-lg[b])[:40]
            lg[b, top] += rng.uniform(0, 8, 40).astype(np.float32)
            rec[b, :120] = np.repeat(top, 3)
            rep[b] = rng.uniform(1.05, 1.3)
        else:
            # the top logit raised until the others add `rest` to the sum
            rest = rng.uniform(0.02, 0.33) if shape == "low" else 10.0 ** rng.uniform(-7, -3)
            i = int(np.argmax(lg[b]))
            y = lg[b].astype(np.float64) / T[b]
            y[i] = -np.inf
            R = np.log(np.exp(y - y.max()).sum()) + y.max()
            lg[b, i] = np.float32((R - np.log(rest)) * T[b])
            if shape == "low" and b % 2:
                p[b] = rng.uniform(0.98, 0.9999)        # a cut at the end of the row, or none
            if shape == "dominated" and p[b] < 1.0:     # (at 1 such a draw may miss the sum: not planned)
                u[b] = rng.choice([u[b], np.float32(1.0 - 1e-4)])
    return lg, T, p, rep, rec, u


@pytest.mark.parametrize("V", [4099, 50257, 200000])
@pytest.mark.parametrize("shape", ["penalized", "low", "dominated"])
def test_full_plan_edges(gpu, torch, oracle, shape, V):
    import workloads
    rng = np.random.default_rng(V + len(shape))
    lg, T, p, rep, rec, u = _case(shape, V, rng)
    print("full plans", shape, V, flush=True)
    params = workloads.params_rows(zip(T, np.zeros(B, np.uint32), p, rep))
    tok = torch.zeros(B, dtype=torch.int32, device="cuda")
    st = torch.full((B,), 99, dtype=torch.int32, device="cuda")
    s = gpu.Sampler(1.0, 0, 0.95, 1.0, seed=1)
    s.sample_batch(torch.from_numpy(lg).cuda(), tok,
                   params=torch.from_numpy(np.ascontiguousarray(params).view(np.uint8)).cuda(),
                   recent=torch.from_numpy(rec.view(np.int32)).cuda(), u=torch.from_numpy(u).cuda(), status=st)
    torch.cuda.synchronize()
    want = oracle.sample_batch(lg, params, u, recent=rec, nthreads=8)
    assert (st.cpu().numpy() == 0).all()
    assert np.array_equal(tok.cpu().numpy().astype(np.int64), want)
    n = s.fallback_rows()
    print("fallback rows", n, flush=True)
    assert n <= 1, "%d of %d rows fell back" % (n, B)
