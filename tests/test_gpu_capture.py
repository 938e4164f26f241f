"""dlk_sample captured into HIP graphs: on streams with and without a workspace, for rows of every layout, and replayed
after a later call has needed a larger workspace."""
import numpy as np
import pytest

from test_gpu_edges import make, run_and_check

pytestmark = pytest.mark.gpu


def captured(torch, w, stream):
    from diskllm_amd import api
    db = api.to_device(w)
    prm = api.params_of(w)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=stream):
        api.sample(db, prm)
    return db, g


def replays(torch, db, g, want, n=3):
    for _ in range(n):
        db.reset_rng()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(db.out_ids.cpu().numpy(), want)


@pytest.mark.parametrize("V", [9000, 16384])
@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_k=20)])
def test_whole_groups_without_workspace_under_capture(cuda, V, kw):
    """Captured on a stream that holds no workspace yet, rows of whole 16-byte groups run on the row kernel, as odd
    ones do."""
    import torch
    rng = np.random.default_rng(9)
    w = make("capture", 3, V, seed=4, logits=rng.normal(0, 2, (3, V)).astype(np.float32), **kw)
    want = run_and_check(w, 1)["ids"]
    db, g = captured(torch, w, torch.cuda.Stream())
    replays(torch, db, g, want)


@pytest.mark.parametrize("V", [50257, 50256])
@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_k=20)])
def test_replay_after_a_larger_call(cuda, V, kw):
    """The graph's workspace outlives a call on its stream that takes a larger one."""
    import torch
    from diskllm_amd import _lib, api
    rng = np.random.default_rng(V)
    st = torch.cuda.Stream()
    w = make("graph", 4, V, seed=2, logits=rng.normal(0, 2, (4, V)).astype(np.float32), **kw)
    want = run_and_check(w, 0)["ids"]
    warm = api.to_device(w)
    api.sample(warm, stream=st.cuda_stream)                  # the stream's workspace
    db, g = captured(torch, w, st)
    replays(torch, db, g, want)
    big = make("larger", 300, V, seed=3, logits=rng.normal(0, 2, (300, V)).astype(np.float32), **kw)
    dbig = api.to_device(big)
    torch.cuda.synchronize()
    api.sample(dbig, stream=st.cuda_stream)
    st.synchronize()
    fill = torch.full((1 << 26,), 0x5a5a5a5a, dtype=torch.int32, device="cuda")   # (what was freed would be here)
    replays(torch, db, g, want)
    del fill, g
    torch.cuda.synchronize()
    _lib.check(_lib.lib().dlk_release_stream(st.cuda_stream), "dlk_release_stream")
