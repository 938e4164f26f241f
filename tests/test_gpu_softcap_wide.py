"""The soft-cap where a wave holds values past the common range: every kind of them, in every place of a group of four,
alone and many, in place and inside the sampling kernels; and its time, which must not hang on one such value."""
import numpy as np
import pytest

from diskllm_amd import _lib
from oracle import oracle as O
from test_gpu_edges import make, run_and_check

pytestmark = pytest.mark.gpu

KINDS = dict(inf=np.inf, ninf=-np.inf, nan=np.nan, zero=0.0, nzero=-0.0, tiny=1e-30, denormal=1e-42, big=3e38)


def rows_of(cap, n=4096):
    """Rows of ordinary logits with other values put in: quotients around each edge of the forms, each kind alone in
    a wave's group of 256 and many of them."""
    rng = np.random.default_rng(3)
    rows = [rng.normal(0, 0.1 * cap, n), rng.normal(0, 2 * cap, n), rng.normal(0, 8 * cap, n)]
    edges = np.array([0.5198, 0.52, 0.9999, 1.0, 1.0001, 7.7499, 7.75, 9.0, 15.99, 16.0, 22.0, 100.0]) * cap
    for v in list(KINDS.values()) + list(edges) + list(-edges):
        one, many = rng.normal(0, 0.1 * cap, n), rng.normal(0, cap, n)
        one[rng.integers(0, 256, 3) + 256 * rng.integers(0, n // 256, 3)] = v
        many[rng.random(n) < 0.4] = v
        rows += [one, many]
    return np.array(rows, np.float32)


@pytest.mark.parametrize("cap", [30.0, 0.75, 1.99999988, 1e-7])
def test_softcap_values_past_the_common_range(cuda, cap):
    import torch
    x = rows_of(cap)
    d = torch.from_numpy(x).cuda()
    rows, V = x.shape
    _lib.check(_lib.lib().dlk_softcap(d.data_ptr(), V, rows, V, cap, torch.cuda.current_stream().cuda_stream), "dlk_softcap")
    want = x.copy()
    for r in range(rows):
        O.lib().orc_softcap(want[r], want[r], V, np.float32(cap))
    got = d.cpu().numpy()
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all()
    np.testing.assert_array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


def test_capped_sampling_of_wide_logits(cuda):
    rng = np.random.default_rng(4)
    rows, V = 6, 40000
    lg = rng.normal(0, 1, (rows, V)).astype(np.float32) * np.array([[3], [15], [60], [300], [2], [2]], np.float32)
    lg[4, rng.integers(0, V, 50)] = 0.0
    lg[5, rng.random(V) < 0.5] = -np.inf
    for kw in (dict(top_p=0.95), dict(temperature=0.7, min_p=1e-4), dict(top_k=40)):
        w = make("wide", rows, V, seed=4, logits=lg, **kw)
        w.softcap = 30.0
        run_and_check(w, 0)


@pytest.mark.parametrize("cap,sd", [(15.0, 5.0), (30.0, 10.0), (50.0, 10.0)])
def test_softcap_time_of_wide_logits(cuda, cap, sd):
    """Logits of which some lie past the common range cost little more than those of which none do (1.65 to 2.2 times
    while one such value sent its wave's group through the general form)."""
    import torch
    rows, V = 256, 262144
    L = _lib.lib()
    st = torch.cuda.current_stream().cuda_stream
    x = torch.empty((rows, V), device="cuda")

    def us(sd):
        base = torch.randn((rows, V), device="cuda").mul_(sd).clamp_(-8 * sd, 8 * sd)
        t = []
        for _ in range(12):
            x.copy_(base)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            L.dlk_softcap(x.data_ptr(), V, rows, V, cap, st)
            b.record()
            b.synchronize()
            t.append(a.elapsed_time(b) * 1e3)
        return float(np.median(t[2:]))
    narrow, wide = us(cap / 20), us(sd)
    print(f"[case] cap {cap}: {narrow:.1f} us, wide logits {wide:.1f}", flush=True)
    assert wide < 1.5 * narrow
