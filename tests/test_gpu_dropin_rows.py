"""The drop-in sampler and penalty calls against the oracle: rows of every length on one sampler object (its
staging grows, a row's last group of four is cut), penalties with repeated and out-of-range ids, long histories,
and a caller that changes its row between calls."""
import ctypes as C

import numpy as np
import pytest

from diskllm_amd import _lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,p,mp", [(1.0, 0, 0.9, 0.0), (0.8, 40, 0.95, 0.0), (0.0, 0, 1.0, 0.0), (0.7, 0, 1.0, 0.02),
                                      (0.9, 900, 0.97, 0.0)])
def test_sampler_rows_vs_oracle(cuda, T, k, p, mp):
    L = _lib.lib()
    rng = np.random.default_rng(int(T * 10) + k)
    state = int(rng.integers(1, 2 ** 63))
    cfg = _lib.SamplerConfig(T, k, p, mp, state)
    s = L.sampler_create(C.byref(cfg))
    assert s
    try:
        for V in (5, 1, 4097, 151936, 3, 50257, 151939, 2, 262144, 4, 7):
            row = rng.normal(0, 3, V).astype(np.float32)
            keep = row.copy()
            o = O.sample_row(row, state, T, k, p, mp)
            assert L.sampler_sample(s, row.ctypes.data, V) == o["token"], (V, T, k)
            state = o["state"]
            np.testing.assert_array_equal(row, keep)          # the row is read only
    finally:
        L.sampler_free(s)


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 256, 5000])
@pytest.mark.parametrize("V", [1, 300, 151936])
def test_penalties_rows_vs_oracle(cuda, n, V):
    L = _lib.lib()
    rng = np.random.default_rng(n + V)
    seen = rng.integers(-2, V + 2, n).astype(np.int32)
    seen[n // 2:] = rng.choice(seen, n - n // 2)              # repeats
    row = rng.normal(0, 3, V).astype(np.float32)
    row[rng.integers(0, V, min(V, 20))] = np.array([0.0, -0.0, np.inf, -np.inf], np.float32)[rng.integers(0, 4, min(V, 20))]
    for op, value, call in ((_lib.OP_PRESENCE, 0.7, L.sampler_apply_presence_penalty),
                            (_lib.OP_REPETITION, 1.3, L.sampler_apply_repetition_penalty),
                            (_lib.OP_PRESENCE, -0.4, L.sampler_apply_presence_penalty)):
        got = row.copy()
        call(got.ctypes.data, V, seen.ctypes.data, n, value)
        want = O.penalties(row, seen, op, value if op == _lib.OP_REPETITION else 1.0, 0.0,
                           value if op == _lib.OP_PRESENCE else 0.0)
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
        row = got
