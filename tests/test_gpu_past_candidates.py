"""Rows whose kept set runs past the sorted candidates and whose draw the candidates cannot settle, beside rows
that they do settle: top-p with and without min-p, T below, at and above 1, rows of one slice and of many, in
batches with shared deep passes (at most 16 rows) and without, and calls that ask for kept lists."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

KINDS = [dict(temp=0.6, top_p=0.95), dict(temp=1.0, top_p=0.999), dict(temp=1.4, top_p=0.9),
         dict(temp=0.8, top_p=0.98, min_p=1e-4), dict(temp=1.0, min_p=1e-5), dict(temp=0.05, top_p=0.9)]


@pytest.mark.parametrize("n", [1025, 20_000, 100_003])
@pytest.mark.parametrize("rows", [3, 16, 17, 40])
@pytest.mark.parametrize("kept", [0, 64])
def test_tokens_match_the_oracle(n, rows, kept):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from artemis_amd import Context, Sampling, states_tensor
    gen = np.random.default_rng(n + rows)
    x = (gen.standard_normal((rows, n)) * 2.5).astype(np.float32)
    x[1::3] *= np.float32(0.3)  # flat rows: nearly every draw past the candidates
    x[2::3] *= np.float32(2.0)  # peaked ones: nearly none
    params = [KINDS[r % len(KINDS)] for r in range(rows)]
    seeds = [int(s) for s in gen.integers(0, 1 << 31, rows)]
    dev = torch.device("cuda")
    ctx = Context(max_rows=rows, max_vocab=n)
    s = [Sampling(p["temp"], 0, p.get("top_p", 1.0), p.get("min_p", 0.0)) for p in params]
    rng = states_tensor(seeds, dev)
    got = []
    for _ in range(2):  # a second draw: the streams advance alike on every path
        tok, status, *_ = ctx.sample_batch(torch.from_numpy(x).to(dev), s, rng, kept_cap=kept)
        assert (status.cpu().numpy() & 0xFF == 0).all()
        got.append(tok.cpu().numpy().astype(np.uint32).tolist())
    ctx.close()
    samplers = [O.Sampler(seed, **p) for seed, p in zip(seeds, params)]
    assert got == [[sm.sample(x[r]) for r, sm in enumerate(samplers)] for _ in range(2)]
