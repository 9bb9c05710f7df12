"""Words of a step that travel as launch arguments and come back through pinned memory."""
import ctypes

import numpy as np
import pytest
import torch

from doppler_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 16])
def test_words_there_and_back(n):
    """In order with the work around them, next to words that stay, and again with other values."""
    L = capi.init(torch.cuda.current_device())
    d = torch.full((24,), 7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for seed in (1, 2):
        words = np.random.default_rng(seed).integers(0, 1 << 32, n, dtype=np.uint32)
        capi.check(L.dh_fill_zero(d.data_ptr(), 8, 4 * n))
        capi.check(L.dh_set_words(d.data_ptr(), 8, words.ctypes.data, n))
        kept = words.copy()
        words[:] = 0                                # the launch has them already
        got = np.zeros(n, np.uint32)
        capi.check(L.dh_read_words(got.ctypes.data, d.data_ptr(), 8, n))
        assert np.array_equal(got, kept)
        assert np.array_equal(d.cpu().numpy().view(np.uint32), np.concatenate([[7, 7], kept, [7] * (22 - n)]).astype(np.uint32))


def test_words_refusals():
    L = capi.init(torch.cuda.current_device())
    d = torch.zeros(24, dtype=torch.int32, device="cuda")
    w = np.zeros(17, np.uint32)
    for n, p, off, message in ((0, d.data_ptr(), 0, "words"), (17, d.data_ptr(), 0, "words"), (1, None, 0, "null"), (1, d.data_ptr(), 2, "aligned")):
        assert L.dh_set_words(p, off, w.ctypes.data, n) == 1 and message in L.dh_last_error().decode()
        assert L.dh_read_words(w.ctypes.data, p, off, n) == 1 and message in L.dh_last_error().decode()


@pytest.mark.parametrize("hidden,buckets,pos", [(8, 0, 0), (13, 11, 0), (2056, 11, 5), (64, 1 << 40, 3)])
def test_words_and_embedding_in_one_launch(hidden, buckets, pos):
    """The words and rows that two launches leave, aligned and not, in one and two slices of columns, with the row the token before it picks."""
    L = capi.init(torch.cuda.current_device())
    vocab, positions, g = 50, 9, torch.Generator(device="cuda").manual_seed(hidden)
    table = lambda rows, t: torch.randn(rows, hidden, generator=g, device="cuda").to(t)
    embed, bigram, places, half = table(vocab, torch.bfloat16), table(12, torch.bfloat16), table(positions, torch.bfloat16), table(vocab, torch.float16)
    mul = (3, 5) if buckets < 100 else (0, 1 << 39)                                  # (row 0 or half of the buckets: only the first exists here)
    ld = (hidden + 63) // 64 * 64
    for token in (0, 49, 50, 4) if buckets < 100 else (4, 48):
        words = np.array([token, 0, 7], np.uint32)
        args = (embed.data_ptr(), vocab, bigram.data_ptr() if buckets else None, buckets, *mul, places.data_ptr(), positions)
        ids, got = (torch.full((4,), 9, dtype=torch.int32, device="cuda") for _ in range(2))
        outs = [torch.full((ld,), 3.0, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        capi.check(L.dh_set_words(ids.data_ptr(), 0, words.ctypes.data, 3))
        capi.check(L.dh_embed_sum(ids.data_ptr(), 0, ids.data_ptr() + 8, *args, outs[0].data_ptr(), ld, 1, hidden, pos, None))
        capi.check(L.dh_embed_sum_words(got.data_ptr(), token, 0, 7, *args, outs[1].data_ptr(), ld, hidden, pos))
        capi.check(L.dh_sync())
        assert torch.equal(outs[0], outs[1]) and torch.equal(ids, got)
        got.fill_(9)
        torch.cuda.synchronize()
        capi.check(L.dh_gather_f16(ids.data_ptr(), half.data_ptr(), outs[2].data_ptr(), 1, hidden, vocab, 0))
        capi.check(L.dh_gather_f16_words(got.data_ptr(), token, 0, 7, half.data_ptr(), outs[3].data_ptr(), hidden, vocab))
        capi.check(L.dh_sync())
        assert torch.equal(outs[2], outs[3]) and torch.equal(ids, got)


@pytest.mark.parametrize("hidden", [4, 250, 252, 256, 257, 260, 1024, 1028])
def test_embedding_rows_of_any_length(hidden):
    """A table's rows and zeros for ids outside it, element by element and in pieces, on tables and outputs that allow pieces and that do not."""
    L = capi.init(torch.cuda.current_device())
    table = torch.randn(9 * hidden + 1, device="cuda").half()
    ids = torch.tensor([3, 0, 8, 9, 1 << 30, 8, 2], dtype=torch.int32, device="cuda")
    for shift in (0, 1):
        rows, out = table[shift:shift + 9 * hidden].view(9, hidden), torch.full((5 * hidden + 1,), 7.0, device="cuda")
        torch.cuda.synchronize()
        capi.check(L.dh_gather_f16(ids.data_ptr(), rows.data_ptr(), out.data_ptr() + 4 * shift, 5, hidden, 9, 2))
        capi.check(L.dh_sync())
        want = torch.cat([rows.float(), torch.zeros(1, hidden, device="cuda")])[[8, 9, 9, 8, 2]]
        assert torch.equal(out[shift:shift + 5 * hidden].view(5, hidden), want) and out[-1 if not shift else 0] == 7.0


def test_more_rows_than_a_grid_has_workgroups_of():
    """At 2^24 rows a workgroup each is more threads than a launch can have, at one less it is not."""
    L = capi.init(torch.cuda.current_device())
    T = 1 << 24
    ids = (torch.arange(T, device="cuda") % 11).to(torch.int32)
    for rows, hidden in ((T, 4), (T - 1, 256)):
        table, out = torch.arange(8 * hidden, device="cuda").to(torch.float16).reshape(8, hidden), torch.zeros(rows, hidden, device="cuda")
        torch.cuda.synchronize()
        capi.check(L.dh_gather_f16(ids.data_ptr(), table.data_ptr(), out.data_ptr(), rows, hidden, 8, 0))
        capi.check(L.dh_sync())
        want = torch.cat([table.float(), torch.zeros(3, hidden, device="cuda")])
        assert all(torch.equal(out[a:a + (1 << 20)], want[ids[a:min(a + (1 << 20), rows)].long()]) for a in range(0, rows, 1 << 20))


def test_words_of_a_token_are_refused_while_a_graph_is_captured():
    """A replay would set the same words: the refusal of dh_set_words, in front of anything that would go into the graph."""
    L = capi.init(torch.cuda.current_device())
    half, out, ids = torch.ones(8, 8, dtype=torch.float16, device="cuda"), torch.full((64,), 3.0, device="cuda"), torch.full((4,), 9, dtype=torch.int32, device="cuda")
    cleared, g = torch.ones(64, device="cuda"), ctypes.c_void_p()
    torch.cuda.synchronize()
    capi.check(L.dh_graph_begin())
    refused = [(L.dh_gather_f16_words(ids.data_ptr(), 1, 0, 0, half.data_ptr(), out.data_ptr(), 8, 8), L.dh_last_error().decode()),
               (L.dh_embed_sum_words(ids.data_ptr(), 1, 0, 0, half.data_ptr(), 8, None, 0, 0, 0, None, 0, out.data_ptr(), 64, 8, 0), L.dh_last_error().decode())]
    capi.check(L.dh_fill_zero(cleared.data_ptr(), 0, 256))
    capi.check(L.dh_graph_end(0, ctypes.byref(g)))
    assert all(rc == 1 and "captured" in message for rc, message in refused)
    capi.check(L.dh_graph_launch(g, 0))
    capi.check(L.dh_sync())
    assert not cleared.any() and (out == 3).all() and (ids == 9).all()
    capi.check(L.dh_graph_destroy(g))


@pytest.mark.parametrize("vocab", [1, 7, 2048, 2049, 32000, 70001])
def test_token_of_a_head_on_the_host(vocab):
    """The token both heads leave on the device and bring to the host is their logits' first maximum, with one to all of the candidates a final
    reduction takes, among equal ones in other waves and threads, and 0 where no logit is a number."""
    L = capi.init(torch.cuda.current_device())
    K, g = 64, torch.Generator(device="cuda").manual_seed(vocab)
    row, ones, eps = torch.randn(K, generator=g, device="cuda"), torch.ones(K, device="cuda"), 1e-6
    ws = torch.zeros(int(L.dh_lmhead_argmax_workspace_bytes(vocab)), dtype=torch.uint8, device="cuda")
    token, logits, host = torch.zeros(2, dtype=torch.int32, device="cuda"), torch.zeros(vocab, device="cuda"), np.zeros(1, np.uint32)
    for case in range(4):
        W = torch.randn(vocab, K, generator=g, device="cuda")
        if case in (1, 2) and vocab > 1:                                       # equal rows, the largest by far
            at = torch.randint(0, vocab, (5,), generator=g, device="cuda") if case == 1 else torch.tensor([vocab - 1, vocab // 2], device="cuda")
            W[at] = 20.0 * row
        if case == 3:
            W[:] = float("nan")
        for dtype in (torch.float16, torch.bfloat16):
            E = W.to(dtype)
            token.fill_(-1)
            torch.cuda.synchronize()
            if dtype == torch.float16:
                capi.check(L.dh_lmhead_argmax_f16_rmsnorm_read(row.data_ptr(), ones.data_ptr(), eps, 0, E.data_ptr(), vocab, K, -1, 0.0, ws.data_ptr(),
                                                               token.data_ptr(), 1, logits.data_ptr(), host.ctypes.data))
            else:
                capi.check(L.dh_dense_lmhead_argmax_read(row.data_ptr(), ones.data_ptr(), K, eps, E.data_ptr(), K, vocab, K, 1.0, ws.data_ptr(),
                                                         token.data_ptr(), 1, logits.data_ptr(), host.ctypes.data))
            want = 0 if case == 3 else int((logits == logits.max()).nonzero()[0])
            assert token.tolist() == [-1, want] and host[0] == want, (case, dtype)


def test_logits_that_are_not_numbers():
    """One of the candidates a head leaves is neither more nor less than another: its place decides, as it does inside a candidate's workgroup.  256 candidates of
    which a few are no numbers, against the pairwise reduction by halves: lanes, then waves."""
    L = capi.init(torch.cuda.current_device())

    def beats(a, b):
        return a[0] > b[0] or (not a[0] < b[0] and a[1] < b[1])

    def fold(c):                                             # 64 lanes, the first one's view: the other half's best against its own half's
        lanes = list(c)
        for off in (32, 16, 8, 4, 2, 1):
            lanes = [lanes[i ^ off] if beats(lanes[i ^ off], lanes[i]) else lanes[i] for i in range(64)]
        return lanes[0]
    g = np.random.default_rng(5)
    ws = torch.zeros(int(L.dh_argmax_workspace_bytes()), dtype=torch.uint8, device="cuda")
    token = torch.zeros(1, dtype=torch.int32, device="cuda")
    for trial in range(24):
        # a stretch of 256 logits a candidate; one logit of a stretch stands out, so that what a workgroup leaves does not depend on its own order
        big = g.choice(np.array([np.nan, np.inf, 3.0, 4.0, 5.0], np.float32), 256, p=[(0.02, 0.3)[trial % 2], 0.02, 0.2, 0.2, (0.56, 0.28)[trial % 2]])
        logits = np.full(65536, -np.inf, np.float32)
        logits[np.arange(256) * 256] = big                  # (the first of a stretch: an infinity below it is less, and a number's place before it)
        want = [(float(big[i]), 256 * i) for i in range(256)]
        waves = [fold(want[64 * w:64 * w + 64]) for w in range(4)]
        best = waves[0]
        for w in waves[1:]:
            best = w if beats(w, best) else best
        d = torch.from_numpy(logits).cuda()
        torch.cuda.synchronize()
        capi.check(L.dh_argmax(d.data_ptr(), 65536, -1, 0.0, ws.data_ptr(), token.data_ptr(), 0))
        capi.check(L.dh_sync())
        assert token.item() == best[1], trial
