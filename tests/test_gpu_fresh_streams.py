"""First calls on streams that hold no workspace yet, beside work on other streams: ids, states and status of every
row, through dlk_sample and the drop-in sampler."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_edges import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_k=40, temperature=0.8), dict(temperature=0.0)])
def test_first_call_on_fresh_streams(cuda, kw):
    import torch
    from diskllm_amd import _lib, api
    rows, V = 8, 151936
    rng = np.random.default_rng(5)
    w = make("fresh", rows, V, seed=5, logits=rng.normal(0, 2, (rows, V)).astype(np.float32), **kw)
    want = [O.sample_row(O.prepared_row(w, r), int(w.seeds[r]), w.temperature, w.top_k, w.top_p, w.min_p)
            for r in range(rows)]
    batches = [api.to_device(w) for _ in range(12)]
    busy = torch.empty(1 << 26, device="cuda")
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in batches]
    for i, (db, st) in enumerate(zip(batches, streams)):
        print(f"[case] fresh stream {i} {kw}", flush=True)
        busy.fill_(i)                                        # work of the null stream, which these do not wait for
        api.sample(db, stream=st.cuda_stream)
        st.synchronize()
    for db, st in zip(batches, streams):
        res = api.results(db)
        assert res["status"] == 0
        assert [int(x) for x in res["ids"]] == [o["token"] for o in want]
        if w.temperature:
            assert [int(x) for x in res["states"]] == [o["state"] for o in want]
        _lib.check(_lib.lib().dlk_release_stream(st.cuda_stream), "dlk_release_stream")


def test_first_tokens_of_fresh_samplers(cuda):
    """(A first call whose barriers time out is run again on the row kernel: right, but half a second late.)"""
    import time
    from diskllm_amd import _lib
    L = _lib.lib()
    V = 151936
    row = np.random.default_rng(6).normal(0, 3, V).astype(np.float32)
    objects, slow = [], []
    for i in range(12):
        cfg = _lib.SamplerConfig(1.0, 0, 0.9, 0.0, 100 + i)
        s = L.sampler_create(C.byref(cfg))
        print(f"[case] fresh sampler {i}", flush=True)
        t0 = time.perf_counter()
        token = L.sampler_sample(s, row.ctypes.data, V)
        slow.append(time.perf_counter() - t0)
        objects.append(s)
        assert token == O.sample_row(row, 100 + i, 1.0, 0, 0.9, 0.0)["token"]
    for s in objects:
        L.sampler_free(s)
    assert max(slow[2:]) < 0.25, slow                        # (the first two load code objects)


@pytest.mark.parametrize("shapes", [((96, 151936), (203, 65536)), ((129, 40961), (516, 20480))])
def test_two_streams_past_the_resident_workgroups(cuda, shapes):
    """Two grids of more workgroups than the device holds, let go together on two streams: each row's workgroups wait
    for one another while both grids' take places by turns."""
    import torch
    from diskllm_amd import _lib, api
    work = []
    for rows, V in shapes:
        rng = np.random.default_rng(rows)
        w = make(f"two-{rows}", rows, V, seed=rows, logits=rng.normal(0, 2, (rows, V)).astype(np.float32), top_p=0.92)
        db = api.to_device(w)
        st = torch.cuda.Stream()
        api.sample(db, stream=st.cuda_stream)                # its workspace
        st.synchronize()
        db.reset_rng()
        work.append((w, db, st))
    busy = torch.empty(1 << 28, device="cuda")
    torch.cuda.synchronize()
    for i in range(3):
        print(f"[case] two streams {shapes} {i}", flush=True)
        gate = torch.cuda.Stream()
        with torch.cuda.stream(gate):
            for k in range(4):
                busy.fill_(k)
            go = torch.cuda.Event()
            go.record()
        for w, db, st in work:
            db.reset_rng()
        torch.cuda.current_stream().synchronize()
        for w, db, st in work:
            st.wait_event(go)
            api.sample(db, stream=st.cuda_stream)
        torch.cuda.synchronize()
        for w, db, st in work:
            res = api.results(db)
            assert res["status"] == 0
            for r in range(w.rows):
                o = O.sample_row(O.prepared_row(w, r), int(w.seeds[r]), w.temperature, w.top_k, w.top_p, w.min_p)
                assert int(res["ids"][r]) == o["token"] and int(res["states"][r]) == o["state"], (w.name, r)
    for _, _, st in work:
        _lib.check(_lib.lib().dlk_release_stream(st.cuda_stream), "dlk_release_stream")


def test_three_streams_of_resident_grids(cuda):
    """Three streams that each keep a batch of 64 rows going, every grid as large as the device."""
    import torch
    from diskllm_amd import _lib, api
    rng = np.random.default_rng(12)
    rows, V = 64, 151936
    w = make("three", rows, V, seed=12, logits=rng.normal(0, 2, (rows, V)).astype(np.float32), top_p=0.9)
    want = []
    for r in range(rows):
        state, tokens = int(w.seeds[r]), []
        row = O.prepared_row(w, r)
        for _ in range(2):
            o = O.sample_row(row, state, w.temperature, w.top_k, w.top_p, w.min_p)
            tokens.append(o["token"])
            state = o["state"]
        want.append(tokens)
    work = []
    for i in range(3):
        db, st = api.to_device(w), torch.cuda.Stream()
        torch.cuda.synchronize()
        api.sample(db, stream=st.cuda_stream)
        st.synchronize()
        assert db.out_ids.cpu().tolist() == [t[0] for t in want]
        work.append((db, st))
    for step in range(20):
        print(f"[case] three streams {step}", flush=True)
        for db, st in work:
            with torch.cuda.stream(st):
                db.reset_rng()
                for _ in range(2):
                    api.sample(db, stream=st.cuda_stream)
        torch.cuda.synchronize()
        for db, _ in work:
            assert int(db.status.item()) == 0
            assert db.out_ids.cpu().tolist() == [t[1] for t in want]
    for _, st in work:
        _lib.check(_lib.lib().dlk_release_stream(st.cuda_stream), "dlk_release_stream")
