"""dlk_grammar_mask where its blocks and its per-token summary can go wrong: vocabularies that end inside a
block or a mask word, more rows than a block takes, token strings longer than a block stages, strings with a
NUL inside, and rows whose next byte is escaped, against the oracle (src/core/grammar.c:275-308)."""
import ctypes as C

import numpy as np
import pytest

from diskllm_amd import _lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BUFFERS = [b"", b" \n", b"{", b'{"a', b'{"a\\', b'["x\\\\', b'{"k": [[1, 2], {"b": ', b"[[[", b'{"a": 1}', b"}",
           b'{"bbox_2d": [1', b'{"bbox_2d": [1,2,3,4], "text_content": "a\\', b'{"bbox_2d":[1,2,3,4]', b"x" * 8185]
TEXTS = [b"object", b"bbox_2d", b"plain"]
ALPHABET = np.frombuffer(b'{}[]{}[]"""\\\\:, \t0123456789bxotex_dn' + bytes([0, 0x80, 0xa0]), np.uint8)


def token_table(rng, V, longest):
    lens = np.minimum(rng.geometric(0.25, V) - 1, 20)
    lens[rng.integers(0, V, max(1, V // 200))] = longest          # (an empty token where the draw gave 0)
    off = np.zeros(V + 1, np.uint32)
    off[1:] = np.cumsum(lens)
    data = ALPHABET[rng.integers(0, ALPHABET.size, int(off[-1]) + 1)]
    return off, np.ascontiguousarray(data)


@pytest.mark.parametrize("V,rows,longest", [(1, 1, 5), (31, 3, 30), (512, 64, 40), (513, 65, 700), (5003, 130, 3000),
                                            (2049, 7, 9000)])
def test_grammar_mask_shapes(cuda, V, rows, longest):
    import torch
    L = _lib.lib()
    rng = np.random.default_rng(V + rows)
    off, data = token_table(rng, V, longest)
    picks = [(TEXTS[i % 3], BUFFERS[(i // 3) % len(BUFFERS)]) for i in range(rows)]
    states = (_lib.GrammarRow * rows)()
    for s, (text, buf) in zip(states, picks):
        L.dlk_grammar_row_init(C.byref(s), L.dlk_grammar_mode_of(text))
        L.dlk_grammar_row_feed(C.byref(s), buf, len(buf))
    dev = torch.device("cuda:0")
    W, ld = (V + 31) // 32, V + 3
    d_off = torch.from_numpy(off.view(np.int32)).to(dev)
    d_data = torch.from_numpy(data).to(dev)
    d_states = torch.frombuffer(bytearray(bytes(states)), dtype=torch.uint8).to(dev)
    d_mask = torch.full((rows, W + 1), -1, dtype=torch.int32, device=dev)
    logits = rng.normal(0, 1, (rows, ld)).astype(np.float32)
    d_logits = torch.from_numpy(logits).to(dev)
    d_valid = torch.full((rows,), -5, dtype=torch.int32, device=dev)
    eos = V // 2
    rc = L.dlk_grammar_mask(d_off.data_ptr(), d_data.data_ptr(), V, d_states.data_ptr(), rows, eos, d_mask.data_ptr(),
                            W + 1, d_logits.data_ptr(), ld, d_valid.data_ptr(), None)
    assert rc == 0
    torch.cuda.synchronize()
    mask, valid = d_mask.cpu().numpy().view(np.uint32), d_valid.cpu().numpy()
    got = d_logits.cpu().numpy()
    assert (mask[:, W] == 0xFFFFFFFF).all()                       # the word past a row's mask is not written
    ids = np.arange(V)
    seen = {}
    for r, pick in enumerate(picks):
        if pick not in seen:
            g = O.grammar(pick[0])
            O.lib().orc_grammar_advance(C.byref(g), pick[1])
            row, n = O.grammar_mask(g, off, data, eos, np.zeros(V, np.float32))
            seen[pick] = (np.isfinite(row), n)
        want, n = seen[pick]
        bits = (mask[r][ids >> 5] >> (ids & 31).astype(np.uint32)) & 1
        np.testing.assert_array_equal(bits.astype(bool), want, err_msg=str(pick))
        assert valid[r] == n, pick
        np.testing.assert_array_equal(got[r, :V], np.where(want, logits[r, :V], -np.inf))
        np.testing.assert_array_equal(got[r, V:], logits[r, V:])
