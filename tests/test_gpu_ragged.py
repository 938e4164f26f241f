"""Rows of any length and alignment on the fused full-vocabulary and top-k kernels: vocabularies that are no
multiple of four (a last group of 1, 2 or 3 entries; a last slice of one entry), rows that start at any float,
with the history, the mask and the draw reaching the last entries, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from diskllm_amd import workloads as W
from test_gpu_edges import make, mask_rows

pytestmark = pytest.mark.gpu


def run(w, path, shift):
    """The workload through dlk_sample, its rows starting `shift` floats into an allocation."""
    import torch
    from diskllm_amd import api
    print(f"[case] {w.name} rows={w.rows} V={w.vocab} k={w.top_k} T={w.temperature} path={path} shift={shift}", flush=True)
    db = api.to_device(w)
    buf = torch.full((w.rows * w.vocab + shift,), 1e30, dtype=torch.float32, device="cuda")
    moved = buf[shift:].view(w.rows, w.vocab)
    moved.copy_(db.logits)
    db.logits = moved
    api.sample(db, api.params_of(w, path=path))
    res = api.results(db)
    assert res["status"] == 0
    ids = res["ids"]
    for r in range(w.rows):
        o = O.sample_row(O.prepared_row(w, r), int(w.seeds[r]), w.temperature, w.top_k, w.top_p, w.min_p)
        assert int(ids[r]) == o["token"], (w.name, r, int(ids[r]), o["token"])
        assert int(res["states"][r]) == o["state"], (w.name, r)
    return res


def batch(V, rows, seed, **kw):
    """Rows with weight on the last entries, a history that names them (and ids past the row)."""
    rng = np.random.default_rng(seed)
    lg = rng.normal(0, 2, size=(rows, V)).astype(np.float32)
    lg[:, V - 6:] += np.float32(9.0)
    lg[::2, V - 1] += np.float32(3.0)
    hist = [np.concatenate([rng.integers(0, V, 40), [V - 1, V - 1, V - 3, V, V + 1, V + 2, -1, V - 5]])
            for _ in range(rows)]
    return make(f"ragged-{V}-{seed}", rows, V, seed=seed, logits=lg, hist=hist, rep=1.2, freq=0.2, pres=0.3,
                order=W.ORDER_NORTH_STAR, **kw)


@pytest.mark.parametrize("V,rows", [(8193, 3), (8194, 40), (8195, 300), (16385, 5), (50257, 8), (98305, 7), (151935, 64)])
@pytest.mark.parametrize("path", [0, 2])
def test_full_vocab_ragged(cuda, V, rows, path):
    for i, kw in enumerate([dict(top_p=0.95), dict(temperature=0.7), dict(top_p=0.9, min_p=1e-4), dict(top_p=0.999)]):
        run(batch(V, rows, V + i, **kw), path, (i + 1) % 4)


@pytest.mark.parametrize("V", [50257, 32770])
def test_full_vocab_ragged_masked_and_capped(cuda, V):
    rng = np.random.default_rng(V)
    w = batch(V, 6, 3, top_p=0.95)
    w.mask = mask_rows(6, V, [[V - 1], [V - 2, 5], [V - 3], rng.choice(V, 1000, replace=False), np.arange(V - 7, V),
                              np.arange(0, V, 2)])
    run(w, 0, 1)
    w.softcap = 30.0
    run(w, 0, 3)
    w = batch(V, 4, 4, top_p=0.9)
    w.logits[0, V - 1] = np.nan
    w.logits[1, V - 2] = np.inf
    w.logits[2, :] = -np.inf
    run(w, 0, 2)


@pytest.mark.parametrize("V,rows,hist", [(50257, 3, 512), (50257, 3, 1024), (50257, 3, 1500), (50257, 3, 4097),
                                         (50257, 40, 1500)])
def test_full_vocab_ragged_history_sizes(cuda, V, rows, hist):
    """Histories of one id per thread, of the long-history instances (whose table shares LDS up to 1,024 ids), past
    those and past the grids they take (the pre-pass), the last entries among them."""
    rng = np.random.default_rng(hist)
    w = batch(V, rows, hist, top_p=0.95)
    lists = [np.concatenate([rng.integers(0, V, hist - 3), [V - 1, V - 2, V - 1]]) for _ in range(rows)]
    w.hist_ids = np.concatenate(lists).astype(np.int32)
    w.hist_off = (np.arange(rows + 1) * hist).astype(np.int32)
    run(w, 0, 1)


@pytest.mark.parametrize("V,rows", [(8193, 3), (50257, 8), (131071, 300), (65537, 9)])
def test_topk_ragged(cuda, V, rows):
    for i, kw in enumerate([dict(top_k=40, top_p=0.95, temperature=0.8), dict(top_k=200), dict(temperature=0.0),
                            dict(top_k=7, top_p=0.9)]):
        w = batch(V, rows, V + i, **kw)
        if i == 3:
            w.softcap = 20.0
        run(w, 0, (i + 1) % 4)


@pytest.mark.parametrize("rows,V", [(203, 65536), (516, 20480), (129, 40961), (96, 151936)])
@pytest.mark.parametrize("path", [0, 2])
def test_full_vocab_grids_past_the_resident_workgroups(cuda, rows, V, path):
    """Grids of more workgroups than the device holds at once, of whole groups of eight rows and not, with and
    without every row's exact fallbacks."""
    rng = np.random.default_rng(rows)
    lg = rng.normal(0, 2, size=(rows, V)).astype(np.float32)
    hist = [rng.integers(0, V, 33) for _ in range(rows)]
    run(make(f"grid-{rows}-{V}", rows, V, seed=rows, logits=lg, top_p=0.92, temperature=0.9, hist=hist, rep=1.2), path, 0)
