"""UnifiedSampling rows above 16384 logits (cut into pieces over several
workgroups) against the oracle, token for token: vocabularies at the edges of a
4096-logit piece, every way the kept prefix can end (significant terms in LDS,
whole bins, inside one bin of a large prefix, in a bin too large to sort,
nothing cut), rows that fall back to the row form, more rows than scratch
slots, and two streams and graph replays in flight at once."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_sampling import _run

pytestmark = pytest.mark.gpu
F32, BF16 = H.F32, H.BF16
OPTS = [None, dict(), dict(temperature=0.6, top_k=20, top_p=0.9), dict(top_k=5000), dict(top_p=0.97),
        dict(temperature=2.0, top_p=0.9, min_p=0.01), dict(temperature=3.0, top_p=0.99, top_k=9000)]


def _check(qmm, oracle, x, dt, vocab, batch, opts, mask=None):
    seeds = np.random.default_rng(vocab).integers(0, 2 ** 63, batch, dtype=np.uint64)
    kw = {} if opts is None else dict(opts, seeds=seeds)
    want = oracle.unified_sampling(x, batch, vocab, t_dt=dt, bitmask=mask, **kw)
    method = qmm.SamplingMethod(stochastic=opts is not None, **(opts or {}))
    got = _run(qmm, x, dt, vocab, batch, method, None if opts is None else seeds, mask)
    assert np.array_equal(got, want), (opts, np.flatnonzero(got != want)[:8])


@pytest.mark.parametrize("opts", OPTS, ids=str)
@pytest.mark.parametrize("vocab,batch,dt,sd", [(16385, 3, F32, 2.0), (20480, 2, BF16, 0.5), (32769, 2, F32, 8.0)])
def test_edges(qmm, oracle, opts, vocab, batch, dt, sd):
    rng = np.random.default_rng(vocab)
    x = H.store(oracle, rng.normal(0, sd, batch * vocab).astype(np.float32), dt)
    mask = rng.integers(0, 2 ** 32, batch * ((vocab + 31) // 32), dtype=np.uint64).astype(np.uint32)
    _check(qmm, oracle, x, dt, vocab, batch, opts, mask if vocab == 32769 else None)


@pytest.mark.parametrize("opts", [dict(top_k=700), dict(top_k=4500), dict(top_p=0.3), dict(top_p=0.99, temperature=3.0),
                                  dict(min_p=0.2), dict(min_p=1.0)], ids=str)
def test_ties(qmm, oracle, opts):
    """Whole-number logits: bins of thousands of equal values, which the index order cuts."""
    x = np.round(np.random.default_rng(6).normal(0, 2, (2, 20000))).astype(np.float32)
    _check(qmm, oracle, x.ravel(), F32, 20000, 2, opts)


@pytest.mark.parametrize("opts", [None, dict(temperature=0.5), dict(temperature=0.5, top_k=8), dict(temperature=0.5, top_p=0.5)],
                         ids=str)
def test_fallback_rows(qmm, oracle, opts):
    """A NaN, an overflowing temperature, a row with every logit masked, and an ordinary row in one call."""
    vocab, batch = 17000, 4
    x = np.random.default_rng(7).normal(0, 3, (batch, vocab)).astype(np.float32)
    x[0, 16999] = np.nan
    x[1, 5] = 3.0e38
    mask = np.full((batch, (vocab + 31) // 32), 0xFFFFFFFF, np.uint32)
    mask[2] = 0
    _check(qmm, oracle, x.ravel(), F32, vocab, batch, opts, mask.ravel())


def test_more_rows_than_slots(qmm, oracle):
    vocab, batch = 16400, 300
    x = np.random.default_rng(8).normal(0, 2, batch * vocab).astype(np.float32)
    for opts in (None, dict(temperature=0.8, top_k=30, top_p=0.9)):
        _check(qmm, oracle, x, F32, vocab, batch, opts)


def test_more_greedy_rows_than_slots(qmm, oracle):
    x = np.random.default_rng(18).normal(0, 2, 300 * 81000).astype(np.float32)
    _check(qmm, oracle, x, F32, 81000, 300, None)


@pytest.mark.parametrize("vocab", [2, 33, 600])
def test_many_short_rows(qmm, oracle, vocab):
    """Past 256 rows, short filtered rows take the row form; top-k of all logits filters nothing."""
    x = np.random.default_rng(vocab).normal(0, 2, 300 * vocab).astype(np.float32)
    for opts in (None, dict(temperature=0.8), dict(temperature=0.8, top_k=vocab), dict(top_k=vocab, top_p=0.9),
                 dict(top_k=max(1, vocab // 2)), dict(temperature=2.0, top_p=0.7, min_p=0.1)):
        _check(qmm, oracle, x, F32, vocab, 300, opts)


@pytest.mark.parametrize("vocab,top_k", [(4096, 1024), (4096, 1025), (8192, 4096), (20000, 3000)])
def test_large_top_k(qmm, oracle, vocab, top_k):
    """Both sides of the size up to which the sorting stage ends every row."""
    x = np.random.default_rng(top_k).normal(0, 2, 3 * vocab).astype(np.float32)
    for opts in (dict(top_k=top_k), dict(top_k=top_k, top_p=0.999, temperature=3.0), dict(top_k=top_k, min_p=1e-4)):
        _check(qmm, oracle, x, F32, vocab, 3, opts)


def test_streams_and_replays(qmm, oracle):
    """Calls on two streams and replays of a captured call in flight together give the tokens of single calls."""
    vocab, batch = 40000, 5
    rng = np.random.default_rng(9)
    xs = [torch.from_numpy(rng.normal(0, 3, batch * vocab).astype(np.float32)).cuda() for _ in range(3)]
    seeds = torch.from_numpy(rng.integers(0, 2 ** 62, batch)).cuda()
    method = qmm.SamplingMethod(stochastic=True, temperature=0.9, top_p=0.9)
    want = [qmm.unified_sampling(x, F32, vocab, batch, method, seeds=seeds) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(streams[2]):
        with torch.cuda.graph(graph, stream=streams[2]):
            captured = qmm.unified_sampling(xs[2], F32, vocab, batch, method, seeds=seeds)
    for _ in range(8):
        got = []
        for i in (0, 1):
            with torch.cuda.stream(streams[i]):
                got.append(qmm.unified_sampling(xs[i], F32, vocab, batch, method, seeds=seeds))
        with torch.cuda.stream(streams[2]):
            graph.replay()
        torch.cuda.synchronize()
        for g, w in zip(got + [captured], want):
            assert torch.equal(g, w)
