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


RECEIPT = b'{"bbox_2d":[1, 2,3,4], "text_content": "a\\b"}'


def step_us(torch, L, V, mode, bufs, calls=20):
    """Microseconds of one mask call, the shortest of five runs of `calls`."""
    off, data = token_table(np.random.default_rng(V), V, 16)
    states = (_lib.GrammarRow * len(bufs))()
    for s, buf in zip(states, bufs):
        L.dlk_grammar_row_init(C.byref(s), mode)
        L.dlk_grammar_row_feed(C.byref(s), buf, len(buf))
    d = [torch.from_numpy(x).cuda() for x in (off.view(np.int32), data, np.frombuffer(bytes(states), np.uint8).copy())]
    W = (V + 31) // 32
    mask = torch.zeros((len(bufs), W), dtype=torch.int32, device="cuda")
    best = np.inf
    for _ in range(6):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(calls):
            L.dlk_grammar_mask(d[0].data_ptr(), d[1].data_ptr(), V, d[2].data_ptr(), len(bufs), V - 1, mask.data_ptr(), W,
                               None, 0, None, torch.cuda.current_stream().cuda_stream)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / calls)
    return best


def test_rows_are_not_taken_one_after_another(cuda):
    """Receipt rows cost about what JSON rows do, whether they share a state or not, and 65 rows of a small vocabulary
    about what one does (a block that took them in turn made them 15 and 2.3 times as long)."""
    L = _lib.lib()
    one = step_us(cuda, L, 1000, 1, [b"{"])
    many = step_us(cuda, L, 1000, 1, [b"{"] * 65)
    same = step_us(cuda, L, 1000, 2, [b""] * 65)
    unlike = step_us(cuda, L, 1000, 2, [RECEIPT[:i % len(RECEIPT)] for i in range(65)])
    print(f"[case] 1000 tokens: one row {one:.1f} us, 65 {many:.1f}, 65 receipt rows {same:.1f} and {unlike:.1f}", flush=True)
    assert many < 1.6 * one and max(same, unlike) < 2.5 * many


@pytest.mark.parametrize("V,rows", [(700, 70), (1536, 9)])
def test_receipt_states(cuda, V, rows):
    """Every position of a receipt, several to a block, states that no buffer leads to (they are scanned byte by
    byte), and a validator that has rejected."""
    import torch
    L = _lib.lib()
    rng = np.random.default_rng(V)
    off, data = token_table(rng, V, 60)
    states = (_lib.GrammarRow * rows)()
    for i, s in enumerate(states):
        L.dlk_grammar_row_init(C.byref(s), 2)
        buf = RECEIPT[:i % (len(RECEIPT) + 1)] + (b"}" if i % 19 == 18 else b"")
        L.dlk_grammar_row_feed(C.byref(s), buf, len(buf))
        if i % 7 == 6:
            s.scan.flag ^= 1                                     # (a digit or none, where no position has it so)
        if i % 11 == 10:
            s.scan.m = 3
            s.scan.n = 9 if s.scan.pc == 2 else s.scan.n
    d = [torch.from_numpy(x).cuda() for x in (off.view(np.int32), data, np.frombuffer(bytes(states), np.uint8).copy())]
    W = (V + 31) // 32
    mask = torch.zeros((rows, W), dtype=torch.int32, device="cuda")
    assert L.dlk_grammar_mask(d[0].data_ptr(), d[1].data_ptr(), V, d[2].data_ptr(), rows, -1, mask.data_ptr(), W, None, 0,
                              None, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    bits = mask.cpu().numpy().view(np.uint32)
    for r in range(rows):
        for t in range(V):
            tok = bytes(data[off[t]:off[t + 1]]).split(b"\0")[0]
            s = _lib.GrammarRow()
            C.memmove(C.byref(s), C.byref(states[r]), C.sizeof(s))
            L.dlk_grammar_row_feed(C.byref(s), tok, len(tok))    # (the scanner, on the host)
            assert ((bits[r, t >> 5] >> (t & 31)) & 1) == (len(tok) > 0 and s.scan.pc != 255), (r, t, tok)
