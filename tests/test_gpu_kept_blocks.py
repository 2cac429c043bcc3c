"""Device blocks kept between trees: results must not depend on what an
earlier tree left in them, on trees living side by side, or on threads with
streams of their own building and destroying trees; and a captured search
replays with its own memory."""
import threading

import numpy as np
import pytest

from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


def _pos(n, seed):
    import torch

    return torch.tensor(datagen.clustered(n, 100.0, nhalo=max(4, n // 2000), seed=seed)[0].T.copy(), device="cuda")


def _answers(pos, form):
    """Build, search, label, destroy, on the current stream."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    n = pos.shape[1]
    t = DeviceTree(pos, kerntype=nb.KSPH, period=100.0, form=form)
    nn = torch.empty((n, 16), dtype=torch.int32, device="cuda")
    d2 = torch.empty((n, 16), dtype=torch.float64, device="cuda")
    lab = torch.empty(n, dtype=torch.int32, device="cuda")
    t.knn(16, nn, d2, layout=nb.LAYOUT_BY_ID)
    ng = t.fof(0.2 * datagen.mean_spacing(n, 100.0), 8, lab)
    out = nn.cpu().numpy(), d2.cpu().numpy(), lab.cpu().numpy(), ng
    del t
    return out


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a[:3], b[:3])) and a[3] == b[3]


@pytest.mark.parametrize("form", [0, 1])
def test_trees_in_turn(gpu, form):
    sizes = (40000, 9000, 40000, 60, 41000, 9000)
    pos = {n: _pos(n, n) for n in set(sizes)}
    first = {}
    for rep in range(2):
        for n in sizes:
            print(f"kept blocks form={form} n={n}", flush=True)
            got = _answers(pos[n], form)
            assert _same(first.setdefault(n, got), got)


def test_threads_and_streams(gpu):
    import torch

    pos = [_pos(30000 + 500 * i, i) for i in range(3)]
    ref = [_answers(p, i % 2) for i, p in enumerate(pos)]
    torch.cuda.synchronize()
    bad, errs = [], []

    def work(i):
        try:
            torch.cuda.set_device(0)
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for rep in range(4):
                    if not _same(ref[i], _answers(pos[i], i % 2)):
                        bad.append((i, rep))
        except Exception as e:  # reported below, on the main thread
            errs.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for x in th:
        x.start()
    for x in th:
        x.join(timeout=100)
    assert not any(x.is_alive() for x in th), "a caller did not return"
    assert not errs and not bad, (errs, bad)


def test_captured_search(gpu):
    """The FP64 search under graph capture: replays, with eager searches on
    the tree between them, equal the eager answer."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    n, k = 20000, 12
    print("captured search", flush=True)
    t = DeviceTree(_pos(n, 5), kerntype=nb.KSPH)
    nn = torch.empty((n, k), dtype=torch.int32, device="cuda")
    d2 = torch.empty((n, k), dtype=torch.float64, device="cuda")
    t.knn(k, nn, d2, layout=nb.LAYOUT_BY_ID)
    torch.cuda.synchronize()
    want = nn.clone(), d2.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        t.knn(k, nn, d2, layout=nb.LAYOUT_BY_ID)
    other = torch.empty((n, 30), dtype=torch.int32, device="cuda")
    for _ in range(3):
        nn.fill_(-5)
        d2.fill_(-1.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(nn, want[0]) and torch.equal(d2, want[1])
        t.knn(30, other)
        torch.cuda.synchronize()
