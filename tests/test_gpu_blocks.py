"""Device blocks that matrices free are handed out again: matrices built and
closed in turn by two threads with contexts and streams of their own, and after
every context was closed, are the ones a single thread builds.  Equal bits."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _build(stream, lists, out):
    from epetreco_amd import geometry as G
    from epetreco_amd.api import Context
    s, g, nrays = G.workload("small")
    with torch.cuda.stream(stream):
        ctx = Context(0, stream)
        ctx.set_geometry(s, g, nrays=nrays, seed=1)
        for lst in lists:
            A = ctx.sm_build(lst)
            rp, col, val, _ = A.to_torch()
            A.attach_transpose()
            A.close()
            out.append((rp.cpu(), col.cpu(), val.cpu()))
        ctx.close()


def test_threads_and_contexts():
    lists = [[np.arange(k, 11250, 3 + k % 4, dtype=np.int32) for k in range(a, 16, 2)] for a in (0, 1)]
    outs = [[], []]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    th = [threading.Thread(target=_build, args=(streams[i], lists[i], outs[i])) for i in (0, 1)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for i in (0, 1):
        alone = []
        _build(streams[i], lists[i], alone)
        assert len(outs[i]) == len(alone) == len(lists[i])
        for got, want in zip(outs[i], alone):
            assert all(torch.equal(a, b) for a, b in zip(got, want))
