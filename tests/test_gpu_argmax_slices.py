"""argmax_rows over rows cut into slices: widths at the slices' edges, row counts on both sides of the
one-slice rule, unaligned rows, picks planted in every slice, and repeated calls (a row's count of
ended slices must be back at zero)."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,rows,pad", [(1, 1, 0), (3, 2, 1), (4095, 1, 1), (4096, 5, 0), (8191, 1, 1), (8192, 1, 0), (8193, 3, 3),
                                        (12289, 767, 3), (12288, 768, 0), (12288, 800, 4), (100_003, 1, 1),
                                        (248_317, 2, 3), (248_320, 1, 0), (248_320, 16, 0)])
def test_slices_give_the_twins_pick(n, rows, pad):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from artemis_amd import Context
    gen = np.random.default_rng(n + rows)
    x = (gen.random((rows, n + pad), dtype=np.float32) * 16 - 8)
    for r in range(rows):
        at = gen.integers(0, n, 3)
        kind = r % 5
        if kind == 1:
            x[r, at] = 9.0  # ties across slices
        elif kind == 2:
            x[r, at] = [np.nan, np.inf, -np.inf]
        elif kind == 3:
            x[r, :n] = -1.0
            x[r, at] = [-0.0, 0.0, -0.0]  # a tie of signed zeros
        elif kind == 4:
            x[r, :n] = np.inf if r % 2 else np.nan  # no finite value
    dev = torch.device("cuda")
    d = torch.from_numpy(x).to(dev)[:, :n]  # row stride n + pad
    ctx = Context(max_rows=1, max_vocab=16)
    ids = torch.empty(rows, dtype=torch.int32, device=dev)
    out = torch.empty(rows, dtype=torch.int64, device=dev)
    want = [O.argmax_row(x[r, :n]) for r in range(rows)]
    for _ in range(3):
        ids.fill_(7)
        out.fill_(7)
        ctx.argmax_rows(d, ids, out, 1 << 33, 210)
        got, addr = ids.cpu().numpy().astype(np.uint32), out.cpu().numpy()
        assert got.tolist() == [0xFFFFFFFF if w is None else w for w in want]
        assert addr.tolist() == [(1 << 33) + (0 if w is None else w) * 210 for w in want]
    ctx.close()


@pytest.mark.parametrize("skew", [0, 1])
def test_a_row_that_ends_within_a_step_of_2_to_the_32(skew):
    # 1,500 short of 2^32: a thread's next index past the row's end does not fit 32 bits. skew 1: the row is
    # not 16-byte aligned and takes the scalar loads.
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from artemis_amd import Context
    n = (1 << 32) - 1500
    if torch.cuda.mem_get_info()[0] < 6 * n:
        pytest.skip("less than 24 GiB of memory free")
    dev = torch.device("cuda")
    x = torch.full((n + 4,), -1.0, dtype=torch.float32, device=dev)[skew:skew + n]
    ids = torch.empty(1, dtype=torch.int32, device=dev)
    out = torch.empty(1, dtype=torch.int64, device=dev)
    ctx = Context(max_rows=1, max_vocab=16)
    for at, v in ((0, 0.0), (n - 1, 2.0), (n // 2, 2.0)):  # each the row's largest, the last one by a tie
        x[at] = v
        ctx.argmax_rows(x, ids, out, 0, 4)
        assert (int(ids.item()) & 0xFFFFFFFF, int(out.item())) == (at, 4 * at)
    ctx.close()
