"""argmax_rows calls that overlap: graphs captured from one context and replayed on two streams beside its eager
calls, and replayed after the context is gone. Each call's picks are its own rows'."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,rows", [(12_289, 3), (248_320, 1), (248_320, 6)])
def test_replays_beside_other_calls(n, rows):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from artemis_amd import Context
    gen = np.random.default_rng(n + rows)
    dev = torch.device("cuda")
    home = torch.cuda.Stream()
    ctx = Context(max_rows=1, max_vocab=16, stream=home)
    xs = [torch.empty((rows, n), dtype=torch.float32, device=dev) for _ in range(3)]
    ids = [torch.empty(rows, dtype=torch.int32, device=dev) for _ in range(3)]
    out = [torch.empty(rows, dtype=torch.int64, device=dev) for _ in range(3)]
    for x in xs:
        x.fill_(0.0)
    torch.cuda.synchronize()
    graphs = []
    for i in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=home):
            ctx.argmax_rows(xs[i], ids[i], out[i], 0, 210)
        graphs.append(g)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def fresh():
        want = []
        for x in xs:
            h = gen.standard_normal((rows, n)).astype(np.float32)
            x.copy_(torch.from_numpy(h))
            want.append([O.argmax_row(r) for r in h])
        torch.cuda.synchronize()
        return want

    def check(i, want):
        assert ids[i].cpu().tolist() == want and out[i].cpu().tolist() == [w * 210 for w in want]

    for _ in range(4):
        want = fresh()
        for _ in range(20):
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
            ctx.argmax_rows(xs[2], ids[2], out[2], 0, 210)
        torch.cuda.synchronize()
        for i in range(3):
            check(i, want[i])
    ctx.close()
    want = fresh()
    for g in graphs:
        g.replay()
    torch.cuda.synchronize()
    for i in range(2):
        check(i, want[i])
