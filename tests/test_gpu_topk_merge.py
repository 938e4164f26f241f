"""The top-k kernel's merge of its slices' lists where its bounds and sorts can go wrong: a short last slice, one
list, few and many lists, a top k that lies in one slice or in runs of equal logits, lists shorter than the bound
takes from them, and survivors around the sizes at which the sort shares a key among threads."""
import numpy as np
import pytest

from diskllm_amd import workloads as W
from test_gpu_edges import make, mask_rows, run_and_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,rows", [(128256, 1), (131072, 2), (4100, 3), (69632, 40), (65537, 700)])
@pytest.mark.parametrize("k", [1, 8, 40, 64, 100, 250])
def test_topk_lists(cuda, V, rows, k):
    rng = np.random.default_rng(V + k)
    lg = rng.normal(0, 2.5, size=(rows, V)).astype(np.float32)
    for r in range(rows):
        kind = r % 5
        if kind == 1:                                  # the top k in consecutive entries of one slice
            at = int(rng.integers(0, V - 2 * k))
            lg[r, at:at + 2 * k] += np.float32(30)
        elif kind == 2:                                # and in the row's last entries
            lg[r, V - k - 3:] += np.float32(30)
        elif kind == 3:                                # runs of equal logits
            lg[r] = np.round(lg[r] * 2) / 2
        elif kind == 4:                                # sorted rows: the lists hold very unlike values
            lg[r] = np.sort(lg[r])[::(-1) ** (r // 5)]
    hist = [rng.integers(0, V, 30) for _ in range(rows)]
    w = make(f"lists-{V}-{k}", rows, V, seed=k, logits=lg, temperature=0.8, top_k=k, top_p=0.97, rep=1.3, hist=hist,
             n_out=min(k, 16))
    run_and_check(w, 0)


@pytest.mark.parametrize("allowed", [3, 60, 400, 3000])
def test_topk_short_lists(cuda, allowed):
    """Masks that leave most lists shorter than the bound's c, some empty, in all fewer than k or a little more."""
    V, rows = 128256, 4
    rng = np.random.default_rng(allowed)
    mask = mask_rows(rows, V, [rng.choice(V if r % 2 else V // 3, allowed, replace=False) for r in range(rows)])
    w = make(f"short-{allowed}", rows, V, seed=allowed, temperature=0.7, top_k=50, top_p=0.95, mask=mask, n_out=8,
             order=W.ORDER_REFERENCE)
    run_and_check(w, 0)


@pytest.mark.parametrize("rows,V", [(64, 128256), (1, 4097), (3, 70001), (300, 32768)])
def test_greedy_first_of_equal_maxima(cuda, rows, V):
    """The lowest index of the maximum, wherever in a group and slice it lies, the maximum penalised or masked too."""
    rng = np.random.default_rng(rows)
    lg = rng.normal(0, 2, size=(rows, V)).astype(np.float32)
    hist = []
    for r in range(rows):
        at = rng.choice(V, 4, replace=False)
        lg[r, at] = np.float32(20)
        hist.append([int(at.min())] if r % 3 == 0 else [int(rng.integers(0, V))])
    run_and_check(make(f"greedy-{rows}", rows, V, seed=rows, logits=lg, temperature=0.0, rep=1.5, hist=hist), 0)


@pytest.mark.parametrize("n", [255, 257, 642, 1024])
@pytest.mark.parametrize("kw", [dict(top_k=31, temperature=0.8, top_p=0.9), dict(temperature=0.0), dict(top_k=9)])
def test_topk_many_patches(cuda, n, kw):
    """Hundreds of penalised ids in a slice, among them its best entries (the exact pass over its groups), ids that
    share a group or a hash chain, and ids repeated through the history."""
    rows, V = 24, 48896
    rng = np.random.default_rng(n)
    lg = rng.normal(0, 2.5, size=(rows, V)).astype(np.float32)
    hist = []
    for r in range(rows):
        kind = r % 4
        h = rng.integers(0, V, n)
        if kind == 1:
            h = np.argsort(-lg[r])[:n]                 # the row's best entries
        elif kind == 2:
            h = 4096 + np.arange(n)                    # neighbours, whole groups
        elif kind == 3:
            h = rng.integers(0, 50, n) * 256           # repeats
        hist.append(h)
    w = make(f"patches-{n}", rows, V, seed=n, logits=lg, hist=hist, rep=1.29, pres=0.2, **kw)
    run_and_check(w, 0)
    if kw.get("top_k") == 9:
        w.softcap = 30.0
        run_and_check(w, 0)


@pytest.mark.parametrize("V,k", [(131776, 60), (131761, 87), (66240, 40), (8192 * 3 + 513, 100), (65536 + 870, 112)])
def test_topk_small_last_slice(cuda, V, k):
    """A last slice with too few entries for a threshold from every wave and more than the candidate buffer holds,
    and the same from a mask whose allowed ids lie in a cluster."""
    rows = 3
    rng = np.random.default_rng(V)
    lg = rng.normal(0, 3, size=(rows, V)).astype(np.float32)
    lg[1, V - 700:] += np.float32(6)
    w = make(f"last-{V}", rows, V, seed=k, logits=lg, temperature=1.05, top_k=k, top_p=0.94, n_out=8, rep=1.2,
             hist=[np.arange(V - 20, V), [], rng.integers(0, V, 50)])
    run_and_check(w, 0)
    w.mask = mask_rows(rows, V, [np.arange(5000, 5700), np.arange(9000, 9900), np.arange(V - 800, V)])
    run_and_check(w, 0)


@pytest.mark.parametrize("rows,V,k", [(3, 131776, 113), (2, 66240, 300), (5, 50257, 200), (2, 131072 + 600, 211),
                                      (3, 8192 * 3 + 513, 112), (300, 20481, 130)])
@pytest.mark.parametrize("cap", [0.0, 30.0])
def test_topk_more_candidates_than_the_buffer_holds(cuda, rows, V, k, cap):
    """Slices that leave too many candidates whatever their threshold: large k, short last slices, allowed ids in a
    cluster, sorted rows, equal logits (one value, two, quantised), the best ids penalised, with and without a cap."""
    rng = np.random.default_rng(V + k)
    lg = rng.normal(0, 3, size=(rows, V)).astype(np.float32)
    for r in range(rows):
        kind = r % 6
        if kind == 1:
            lg[r] = np.round(lg[r] * 4) / 4                  # (as logits rounded to fewer bits are)
        elif kind == 2:
            lg[r] = np.sort(lg[r])[::(-1) ** (r // 6)]
        elif kind == 3:
            lg[r] = np.float32(r % 2)                        # all equal
        elif kind == 4:
            lg[r] = np.where(rng.random(V) < 0.3, np.float32(2.5), np.float32(-1))
    hist = [np.argsort(-lg[r], kind="stable")[:40] if r % 2 else [] for r in range(rows)]
    w = make(f"over-{V}-{k}-{cap}", rows, V, seed=k, logits=lg, temperature=1.1, top_k=k, top_p=0.97, n_out=8, rep=1.2,
             hist=hist)
    w.softcap = cap
    run_and_check(w, 0)
    allowed = [np.arange(5000, 5000 + k + 900), np.arange(V - 1200, V), np.arange(0, V, 3)]
    w.mask = mask_rows(rows, V, [allowed[r % 3] for r in range(rows)])
    run_and_check(w, 0)


def call_us(torch, w, path):
    from diskllm_amd import api
    db = api.to_device(w)
    f = api.sampler(db, api.params_of(w, path=path))
    best = np.inf
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / 5)
    return best


@pytest.mark.parametrize("rows,V,k,flat", [(300, 50257, 200, False), (64, 50257, 150, False), (64, 50257, 40, True),
                                           (8, 151937, 150, False)])
def test_topk_is_not_behind_the_row_kernel(cuda, rows, V, k, flat):
    """Rows of odd length took the row kernel before the fused one did: large k and equal logits must not cost more
    there (383 us against 229, 213 against 85, 570 against 186, while such slices fell back to one workgroup's
    selection over the whole row)."""
    rng = np.random.default_rng(k)
    lg = np.zeros((rows, V), np.float32) if flat else rng.normal(0, 2.5, size=(rows, V)).astype(np.float32)
    w = make(f"time-{rows}-{V}-{k}", rows, V, seed=k, logits=lg, top_k=k, temperature=0.8)
    auto, row = call_us(cuda, w, 0), call_us(cuda, w, 1)
    print(f"[case] {rows} x {V} k {k}: {auto:.1f} us, row kernel {row:.1f}", flush=True)
    assert auto < 1.1 * row


def test_rows_without_workspace_under_capture(cuda):
    """Rows of odd length captured on a stream that holds no workspace yet run on the row kernel."""
    import torch
    from diskllm_amd import api
    rng = np.random.default_rng(9)
    V = 9001
    for kw in (dict(top_p=0.9), dict(top_k=20)):
        w = make("capture", 3, V, seed=4, logits=rng.normal(0, 2, (3, V)).astype(np.float32), **kw)
        want = run_and_check(w, 1)["ids"]
        db = api.to_device(w)
        prm = api.params_of(w)
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=torch.cuda.Stream()):
            api.sample(db, prm)
        for _ in range(3):
            db.reset_rng()
            g.replay()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(db.out_ids.cpu().numpy(), want)
