"""Decisions on the edge of their rounding: draws whose u lies within a few units of 2^-53 of a cumulative
weight of the reference's own folds (the RNG state is chosen for it), and top-p cuts whose cumulative lies
within 1e-12 of top_p (one tail logit is tuned for it), past the candidates and among them, with and without
penalties, in batches that share their deep passes (at most 16 rows) and in larger ones. And the same at a
distance that the deep passes' bounds straddle until the row's total is folded exactly: these rows' status
must show the deep passes and not the exact-order path, which the closest ones must take.

The distances, in units U = 2^-53 of the value that the decision compares with: the bins' sums lie within
E = 2e-12 / U plus their fullest bin's values of the exact ones, a total in index order within n, a cumulative
at rank r within r (top-p's quotients: 2 r). The first pass decides beyond 2 E + n + r, with the folded total
beyond E + r: halfway between lies 1.5 E + n / 2 + r."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MASK = (1 << 64) - 1
EXACT, DEEP = 0x100, 0x400  # the status' path bits
U = 2.0 ** -53
E = 2e-12 / U + 1500  # in units; 1,500: about the fullest bin's values


def halfway(n, r):
    return 1.5 * E + 0.5 * n + r


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
    """Tokens and status words of the rows that share x, in one call, or in calls of at most 16 rows."""
    from artemis_amd import Context, Sampling
    dev = torch.device("cuda")
    d = torch.from_numpy(x).to(dev).view(1, -1)
    rows = len(states)
    ctx = Context(max_rows=rows, max_vocab=len(x))
    got, words = [], []
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
        words += status.cpu().tolist()
    ctx.close()
    assert all(w & 0xFF == 0 for w in words)
    return got, words


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
    states, near, beside = [], [], []
    ranks = [0, 1, 30] + [int(keep * f) for f in (0.02, 0.1, 0.3, 0.6, 0.9, 0.98)] + [keep - 2, keep - 1]
    for j in ranks:
        f = cum[j] / total
        at = min(int(f * 2.0 ** 53), (1 << 53) - 1)
        past = n > 5000 and j >= 0.1 * n and j < keep - 2  # past any row's candidates
        for d in (-200, -3, -1, 0, 1, 2, 5, 300):
            near += [len(states)] if past and abs(d) <= 5 else []
            states.append(state_for(min(max(at + d, 0), (1 << 53) - 1)))
        # The next cumulatives on both sides must lie beyond the widest bounds themselves.
        alone = past and min(cum[j + 1] - cum[j], cum[j] - cum[j - 1]) > 2.0 * (2.0 * E + n + j) * U * cum[j]
        for d in (-1, 1):
            beside += [len(states)] if alone else []
            states.append(state_for(min(max(at + d * int(f * halfway(n, j)), 0), (1 << 53) - 1)))
    got, words = run_rows(x, params, hist, states, small)
    assert got == oracle_tokens(x, params, hist, states)
    assert all(words[i] & EXACT for i in near)
    if kind in ("plain", "cold", "hot", "penalised"):  # no filter: the draw compares with the row's total
        assert (len(near) >= 15 and len(beside) >= 6) or n < 5000
        assert all(words[i] & DEEP and not words[i] & EXACT for i in beside)


def tune(x, j, p, off):
    """x with one tail logit changed so that the reference's cumulative at rank j is p (1 + off) of total1, and
    how far from that it came."""
    t1, order, c1 = folds(x, 1.0)
    need = c1[j] / (float(p) * (1.0 + off)) - t1
    w = np.diff(c1, prepend=0.0)
    at = int(np.argmax(w <= max(4e-7 * t1, 4.0 * abs(need))))  # the weight steps by about 1e-7 of itself
    assert at > j + 1
    y = x.copy()
    y[order[at]] = np.float32(np.log(w[at] + need) + np.float64(x[order[0]]))
    t1, order2, c2 = folds(y, 1.0)
    assert (order2[:j + 2] == order[:j + 2]).all()
    return y, abs(c2[j] / t1 / (float(p) * (1.0 + off)) - 1.0)


@pytest.mark.parametrize("n", [50_001, 248_320])
@pytest.mark.parametrize("small", [True, False])
def test_cuts_beside_top_p(n, small):
    gen = np.random.default_rng(n + 1)
    for frac in (0.002, 0.1, 0.3):
        x = (gen.standard_normal(n) * 2.5).astype(np.float32)
        t1, order, c1 = folds(x, 1.0)
        j = int(n * frac)
        p = np.float32(c1[j] / t1)
        for off in (0.0, -halfway(n, 2 * j) * U, halfway(n, 2 * j) * U):
            y, miss = tune(x, j, p, off)
            assert miss < 1e-12 if off == 0.0 else miss < 0.1 * abs(off)
            params = dict(temp=0.9, top_p=float(p))
            # Draws of rank j - 5 decide nothing by themselves; the others fall anywhere, the last kept among them.
            total, _, cum = folds(y, 0.9)
            mid = state_for(int((cum[j - 6] + cum[j - 5]) / 2 / cum[j] * 2.0 ** 53))
            states = [mid] + [state_for(m) for m in [0, 1 << 51, (1 << 53) - 1, (1 << 53) - 2]] + [O_state(s) for s in range(16)]
            got, words = run_rows(y, params, np.zeros(0, np.uint32), states, small)
            assert got == oracle_tokens(y, params, np.zeros(0, np.uint32), states)
            if frac >= 0.1:  # past any row's candidates
                assert words[0] & EXACT if off == 0.0 else words[0] & DEEP and not words[0] & EXACT


def O_state(seed):
    s = O.Sampler(seed)
    return [int(v) for v in s.rng_state()]
