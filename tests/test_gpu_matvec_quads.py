"""The K-quants' matvec kernel at the edges of its layouts: row lengths around each thread count's quads
(128 values each), row counts around a workgroup's rows, tables that start mid-word, and inputs whose
products or sums are subnormal, infinite or NaN. Bit for bit with the reference's order."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_matvec import random_table

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from artemis_amd import Context
    c = Context(max_rows=4, max_vocab=16)
    yield c
    c.close()


@pytest.mark.parametrize("name", ["Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("k", [256, 512, 768, 1024, 1280, 2048, 2304, 4096, 8192])
@pytest.mark.parametrize("skew", [0, 2])
def test_every_layout_bit_for_bit(ctx, name, k, skew):
    gen = np.random.default_rng(k + skew)
    for rows, kind in [(1, "plain"), (15, "tiny"), (17, "zeros"), (65, "plain"), (33, "special"), (257, "plain")]:
        table = random_table(gen, name, rows, k)
        x = gen.standard_normal(k).astype(np.float32)
        if kind == "tiny":
            x *= np.float32(1e-39)  # subnormal inputs and products
        elif kind == "zeros":
            x[gen.random(k) < 0.5] = -0.0
        elif kind == "special":
            x[gen.integers(0, k, 2)] = [np.inf, np.nan]
            x[gen.integers(0, k, 4)] = 3e38
        buf = torch.zeros(table.size + 16, dtype=torch.uint8, device="cuda")
        w = buf[skew:skew + table.size]
        w.copy_(torch.from_numpy(table.reshape(-1)))
        got = ctx.matvec(w, O.WTYPES[name], rows, k, torch.from_numpy(x).cuda()).cpu().numpy()
        want = O.matvec(O.WTYPES[name], table.tobytes(), rows, k, x)
        nan = np.isnan(want)
        assert (np.isnan(got) == nan).all() and (got.view(np.uint32)[~nan] == want.view(np.uint32)[~nan]).all(), (rows, kind)
