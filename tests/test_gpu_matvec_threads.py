"""The K-quants' threads per row: row lengths of 5 to 24 quads (128 values each) and row counts on both sides of
each line that the choice has (16,384 and 32,768 rows), logits and head_argmax's pick, bit for bit with the
reference's order. Tables that start mid-word take the other Q6_K loads."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_matvec import random_table

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("name", ["Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("k", [768, 1024, 1280, 2048, 2304, 3072])
def test_every_choice_bit_for_bit(name, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from artemis_amd import Context
    gen = np.random.default_rng(k)
    most = 32_769 if name == "Q6_K" and k > 2048 else 16_385
    table = random_table(gen, name, most, k)
    x = gen.standard_normal(k).astype(np.float32)
    want = O.matvec(O.WTYPES[name], table.tobytes(), most, k, x)
    dev = torch.device("cuda")
    dx = torch.from_numpy(x).to(dev)
    ctx = Context(max_rows=1, max_vocab=16)
    for skew in (0, 2):
        buf = torch.zeros(table.size + 16, dtype=torch.uint8, device=dev)
        w = buf[skew:skew + table.size]
        w.copy_(torch.from_numpy(table.reshape(-1)))
        for rows in {1, 2, 31, 16_383, 16_384, most - 2, most - 1, most}:
            y = torch.full((rows + 1,), 7.0, device=dev)
            ids = torch.full((1,), 7, dtype=torch.int32, device=dev)
            out = torch.zeros(1, dtype=torch.int64, device=dev)
            ctx.head_argmax(w, O.WTYPES[name], rows, k, dx, ids, out, 0, 8, logits=y)
            plain = ctx.matvec(w, O.WTYPES[name], rows, k, dx).cpu().numpy()
            got, pick = y.cpu().numpy(), O.argmax_row(want[:rows])
            nan = np.isnan(want[:rows])
            for v in (plain, got[:rows]):
                assert (np.isnan(v) == nan).all(), rows
                assert (v.view(np.uint32)[~nan] == want[:rows].view(np.uint32)[~nan]).all(), rows
            assert got[rows] == 7.0
            assert int(ids.item()) & 0xFFFFFFFF == (0xFFFFFFFF if pick is None else pick)
    ctx.close()
