"""Decisions on the edge of their rounding: draws whose u lies within a few units of 2^-53 of a cumulative
weight of the reference's own folds (the RNG state is chosen for it), and top-p cuts whose cumulative lies
within 1e-12 of top_p (one tail logit is tuned for it), past the candidates and among them, with and without
penalties, in batches that share their deep passes (at most 16 rows) and in larger ones."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MASK = (1 << 64) - 1


def state_for(m):
    """A xoshiro256** state whose next unit() is m / 2^53."""
    out = (m << 11) & MASK
    x = out * pow(9, -1, 1 << 64) & MASK
    x = ((x >> 7) | (x << 57)) & MASK
    return [0x1234567, x * pow(5, -1, 1 << 64) & MASK, 0x9876543, 0x5555]


def folds(row, temp):
    """(the index-order total, ids in rank order, the rank-order cumulatives) at T = temp, in f64 folds."""
    order = np.lexsort((np.arange(len(row)), -row))
    v = row.astype(np.float64)
    w = O.exp_array((v - v[order[0]]) / np.float64(np.float32(temp)))
    return np.add.accumulate(w)[-1], order, np.add.accumulate(w[order])


def penalised(row, hist):
    out = row.copy()
    ids = np.unique(hist)
    out[ids] -= np.float32(0.5)
    return out


def run_rows(x, params, hist, states, small):
    """Tokens of the rows that share x, in one call, or in calls of at most 16 rows."""
    from artemis_amd import Context, Sampling
    dev = torch.device("cuda")
    d = torch.from_numpy(x).to(dev).view(1, -1)
    rows = len(states)
    ctx = Context(max_rows=rows, max_vocab=len(x))
    got = []
    for at in range(0, rows, 16 if small else rows):
        st = states[at:at + (16 if small else rows)]
        rng = torch.from_numpy(np.array(st, np.uint64).view(np.int64)).to(dev)
        off = ids = None
        if len(hist):
            off = torch.arange(len(st) + 1, dtype=torch.int32, device=dev) * len(hist)
            ids = torch.from_numpy(np.tile(hist, len(st)).astype(np.int32)).to(dev)
        s = [Sampling(p["temp"], p.get("top_k", 0), p.get("top_p", 1.0), p.get("min_p", 0.0), p.get("presence", 0.0))
             for p in [params] * len(st)]
        tok, status, *_ = ctx.sample_batch(d, s, rng, off, ids, row_stride=0, n_vocab=len(x))
        got += tok.cpu().numpy().astype(np.uint32).tolist()
        assert (status.cpu().numpy() & 0xFF == 0).all()
    ctx.close()
    return got


def oracle_tokens(x, params, hist, states):
    out = []
    for st in states:
        s = O.Sampler(0, **params)
        if len(hist):
            s.add_history(hist)
        s.set_rng_state(st)
        out.append(s.sample(x))
    return out


@pytest.mark.parametrize("n", [4097, 50_001, 248_320])
@pytest.mark.parametrize("kind", ["plain", "cold", "hot", "penalised", "nucleus", "topk"])
@pytest.mark.parametrize("small", [True, False])
def test_draws_beside_a_cumulative(n, kind, small):
    gen = np.random.default_rng(n)
    x = (gen.standard_normal(n) * 2.5).astype(np.float32)
    params = {"plain": dict(temp=1.0), "cold": dict(temp=0.7), "hot": dict(temp=1.5),
              "penalised": dict(temp=1.0, presence=0.5), "nucleus": dict(temp=0.8, top_p=0.97),
              "topk": dict(temp=1.0, top_k=min(1000, n // 2))}[kind]
    hist = gen.integers(0, n, 300).astype(np.uint32) if kind == "penalised" else np.zeros(0, np.uint32)
    row = penalised(x, hist) if len(hist) else x
    total, order, cum = folds(row, params["temp"])
    if kind == "nucleus":
        t1, _, c1 = folds(row, 1.0)
        keep = int(np.searchsorted(c1 / t1, np.float64(np.float32(0.97)))) + 1
        total = cum[keep - 1]
    elif kind == "topk":
        keep = params["top_k"]
        total = cum[keep - 1]
    else:
        keep = n
    states = []
    ranks = [0, 1, 30] + [int(keep * f) for f in (0.02, 0.1, 0.3, 0.6, 0.9, 0.98)] + [keep - 2, keep - 1]
    for j in ranks:
        at = min(int(cum[j] / total * 2.0 ** 53), (1 << 53) - 1)
        for d in (-200, -3, -1, 0, 1, 2, 5, 300):
            states.append(state_for(min(max(at + d, 0), (1 << 53) - 1)))
    assert run_rows(x, params, hist, states, small) == oracle_tokens(x, params, hist, states)


@pytest.mark.parametrize("n", [50_001, 248_320])
@pytest.mark.parametrize("small", [True, False])
def test_cuts_beside_top_p(n, small):
    gen = np.random.default_rng(n + 1)
    for frac in (0.002, 0.05, 0.3):
        x = (gen.standard_normal(n) * 2.5).astype(np.float32)
        t1, order, c1 = folds(x, 1.0)
        j = int(n * frac)
        p = np.float32(c1[j] / t1)
        # One tail value tuned so that c1[j] / total is p: rank 2j's weight takes the difference.
        top, at = np.float64(x[order[0]]), order[2 * j]
        w = np.exp(np.float64(x[at]) - top) + (c1[j] / np.float64(p) - t1)
        if w <= 0.0 or np.log(w) + top >= x[order[j + 1]]:
            continue
        x[at] = np.float32(np.log(w) + top)
        params = dict(temp=0.9, top_p=float(p))
        states = [state_for(m) for m in [0, 1 << 51, (1 << 53) - 1, (1 << 53) - 2]] + [O_state(s) for s in range(16)]
        assert run_rows(x, params, np.zeros(0, np.uint32), states, small) == \
            oracle_tokens(x, params, np.zeros(0, np.uint32), states)


def O_state(seed):
    s = O.Sampler(seed)
    return [int(v) for v in s.rng_state()]
