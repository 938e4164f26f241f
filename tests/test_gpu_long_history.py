"""Histories past one id per thread on the fused full-vocabulary kernel (its long-history instances up to 4,096 ids
where the grid is resident at once, the pre-pass beyond): every id distinct and in one slice, ids repeated thousands
of times, rows at and over max_history, masks and the soft-cap, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from diskllm_amd import workloads as W
from test_gpu_edges import make, mask_rows

pytestmark = pytest.mark.gpu


def check(w, max_history, path=0, flagged=()):
    from diskllm_amd import _lib, api
    print(f"[case] {w.name} rows={w.rows} V={w.vocab} max_history={max_history} path={path}", flush=True)
    db = api.to_device(w)
    api.sample(db, api.params_of(w, max_history=max_history, path=path))
    res = api.results(db)
    assert res["status"] == (_lib.DLK_STATUS_HISTORY_TOO_LONG if flagged else 0)
    for r in range(w.rows):
        if r in flagged:
            assert res["ids"][r] == -1 and int(res["states"][r]) == int(w.seeds[r])
            continue
        o = O.sample_row(O.prepared_row(w, r), int(w.seeds[r]), w.temperature, w.top_k, w.top_p, w.min_p)
        assert int(res["ids"][r]) == o["token"] and int(res["states"][r]) == o["state"], (w.name, r)


@pytest.mark.parametrize("n", [513, 1024, 1025, 3000, 4096, 4097])
@pytest.mark.parametrize("rows,V", [(5, 50257), (64, 60000)])
def test_long_histories(cuda, n, rows, V):
    rng = np.random.default_rng(n + rows)
    kinds = [rng.integers(0, V, n), 100 + rng.permutation(8000)[:n], np.full(n, 7), rng.integers(V - 9, V + 3, n),
             np.concatenate([rng.integers(0, 40, n - n // 3), rng.integers(-1, V, n // 3)])]
    hist = [kinds[r % 5] for r in range(rows)]
    lg = rng.normal(0, 2, size=(rows, V)).astype(np.float32)
    lg[:, 100:8100] += np.float32(2)
    # (a factor per occurrence: few repeats keep the penalised logits finite)
    w = make(f"long-{n}-{rows}-{V}", rows, V, seed=n, logits=lg, hist=hist, rep=1.0005, freq=0.001, pres=0.3,
             order=W.ORDER_NORTH_STAR, top_p=0.95, temperature=0.9)
    check(w, n)
    if rows == 5:
        check(w, n, path=2)
        w.min_p = 1e-4
        w.mask = mask_rows(rows, V, [np.arange(r, V, 3) for r in range(rows)])
        check(w, n)
        w.softcap = 25.0
        check(w, n)


@pytest.mark.parametrize("limit", [2000, 4096])
def test_history_past_the_limit(cuda, limit):
    """Rows over the caller's own bound are flagged, rows at it are not."""
    V, rows = 40000, 6
    rng = np.random.default_rng(limit)
    sizes = [limit, limit + 1, 10, 0, limit - 1, limit + 700]
    w = make(f"limit-{limit}", rows, V, seed=1, hist=[rng.integers(0, V, s) for s in sizes], rep=1.3, top_p=0.9)
    check(w, limit, flagged=(1, 5))
