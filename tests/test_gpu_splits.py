"""Calls whose rows take several launches: batches past the workspace of one launch, and the no-allocation call over
rows of odd length, whose fixed array holds fewer."""
import ctypes as C

import numpy as np
import pytest

from diskllm_amd import _lib
from oracle import oracle as O
from test_gpu_edges import make

pytestmark = pytest.mark.gpu


def test_batch_past_the_workspace_of_one_launch(cuda):
    """820 rows of 151,936 (some 680 KB of workspace a row, 512 MB a launch): rows at the ends and around the split."""
    import torch
    from diskllm_amd import api
    rows, V, hist = 820, 151936, 32
    g = torch.Generator(device="cuda")
    g.manual_seed(8)
    lg = torch.randn((rows, V), device="cuda", generator=g) * 2
    ids = torch.randint(0, V, (rows, hist), device="cuda", generator=g, dtype=torch.int32)
    look = [0, 1, 7, 8, 400] + list(range(740, 800, 3)) + [rows - 9, rows - 8, rows - 1]
    w = make("split", len(look), V, seed=1, logits=lg[look].cpu().numpy(), top_p=0.9, rep=1.1,
             hist=list(ids[look].cpu().numpy()))
    off = torch.arange(rows + 1, dtype=torch.int32, device="cuda") * hist
    seeds = torch.randint(1, 2 ** 62, (rows,), device="cuda", generator=g, dtype=torch.int64)
    db = api.DeviceBatch(w=w, logits=lg, seeds=seeds, rng=seeds.clone(), hist_off=off, hist_ids=ids.reshape(-1), mask=None,
                         mask_row=None, out_ids=torch.full((rows,), -7, dtype=torch.int32, device="cuda"), cand_ids=None,
                         cand_probs=None, cand_logprobs=None, status=torch.zeros(1, dtype=torch.int32, device="cuda"))
    print("[case] 820 x 151936", flush=True)
    api.sample(db, api.params_of(w))
    res = api.results(db)
    assert res["status"] == 0 and (res["ids"] >= 0).all()
    states = seeds.cpu().numpy().view(np.uint64)
    for i, r in enumerate(look):
        o = O.sample_row(O.prepared_row(w, i), int(states[r]), w.temperature, w.top_k, w.top_p, w.min_p)
        assert int(res["ids"][r]) == o["token"] and int(res["states"][r]) == o["state"], r
    _lib.check(_lib.lib().dlk_release_stream(api.stream_handle()), "dlk_release_stream")


@pytest.mark.parametrize("rows", [8, 300])
@pytest.mark.parametrize("kw", [dict(top_p=0.9, rep=1.2), dict(top_k=40), dict(temperature=0.0)])
def test_noalloc_rows_of_odd_length(cuda, rows, kw):
    """dlk_sample_noalloc over packed rows of 50,257: what dlk_sample gives, the oracle's on some rows."""
    from diskllm_amd import api
    rng = np.random.default_rng(rows)
    V = 50257
    w = make(f"odd-{rows}", rows, V, seed=rows, logits=rng.normal(0, 2, (rows, V)).astype(np.float32),
             hist=[rng.integers(0, V, 20) for _ in range(rows)], **kw)
    got = []
    for fn in ("dlk_sample_noalloc", "dlk_sample"):
        print(f"[case] {fn} {rows} x {V} {kw}", flush=True)
        db = api.to_device(w)
        b, prm = api.batch_struct(db), api.params_of(w)
        assert getattr(_lib.lib(), fn)(C.byref(b), rows, V, C.byref(prm), api.stream_handle()) == _lib.DLK_OK
        got.append(api.results(db))
        assert got[-1]["status"] == 0
    np.testing.assert_array_equal(got[0]["ids"], got[1]["ids"])
    np.testing.assert_array_equal(got[0]["states"], got[1]["states"])
    for r in range(0, rows, max(1, rows // 8)):
        o = O.sample_row(O.prepared_row(w, r), int(w.seeds[r]), w.temperature, w.top_k, w.top_p, w.min_p)
        assert int(got[0]["ids"][r]) == o["token"]
