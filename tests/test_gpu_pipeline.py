"""dtl_forward_ranges: the codec window's forwards and symbol ranges with several
chunks in flight on separate streams.  Every range must equal the oracle's
(det-coder logits_to_symbol_range over det-model logits) and the
chunk-at-a-time path's, whatever the chunk split, the final chunk's size
(the decode-attention path below five positions) or the start position.

A session whose max_chunk is below 256 runs chunks of 256 on wide lanes of
its own; DETLLM_NO_WIDE_LANES keeps it on lanes of max_chunk, so that a short
text has many chunks, and DETLLM_LANE_MEMORY bounds what lanes may take, as
a card without room would.
"""
import ctypes as C
import dataclasses
import gc

import numpy as np
import pytest

import detref

pytestmark = pytest.mark.gpu


def _rows_symbols(n, vocab, tail, seed):
    """Rows 0..n-1 in order, some repeated (byte escapes share the logits of
    the last token) and some skipped; symbols over the whole alphabet."""
    rng = np.random.default_rng(seed)
    rows = []
    for r in range(n):
        k = int(rng.integers(0, 3))  # 0, 1 or 2 symbols coded against row r
        rows += [r] * k
    rows = np.array(rows, np.uint32)
    syms = rng.integers(0, vocab + tail, rows.size).astype(np.uint32)
    return rows, syms


def _oracle_ranges(data, tokens, pos0, rows, syms, tail):
    logits = detref.Model(data).logits(tokens)
    return [detref.symbol_range(logits[pos0 + int(r)], int(s), tail) for r, s in zip(rows, syms)]


@pytest.mark.parametrize("n,chunk,pos0", [(17, 3, 0), (17, 4, 5), (9, 8, 0), (3, 1, 2)])
@pytest.mark.parametrize("tail", [0, 256])
@pytest.mark.parametrize("wide", [True, False])  # one chunk on a wide lane; several on the session's own
def test_forward_ranges_matches_oracle(monkeypatch, n, chunk, pos0, tail, wide):
    from detllm_amd import synth
    from detllm_amd.model import F32Llama

    if not wide:
        monkeypatch.setenv("DETLLM_NO_WIDE_LANES", "1")  # read when the session is created

    # the tiny all-F32 shape with room for 22 positions
    w = dataclasses.replace(synth.WORKLOADS["tiny"], ctx=32)
    data = synth.build_model(w)
    toks = synth.tokens(w, pos0 + n)
    m = F32Llama.from_gguf(data)
    rows, syms = _rows_symbols(n, m.vocab, tail, seed=n * 31 + chunk)
    print(f"forward_ranges tiny n={n} chunk={chunk} pos0={pos0} tail={tail}", flush=True)
    with m.forward_workspace(pos0 + n, chunk) as s:
        for p in range(0, pos0, chunk):
            s.forward_chunk(toks[p:min(p + chunk, pos0)], p)
        cum, freq, total = s.forward_ranges(toks[pos0:], pos0, rows, syms, tail)
    got = [(int(c), int(f), int(t)) for c, f, t in zip(cum, freq, total)]
    assert got == _oracle_ranges(data, toks, pos0, rows, syms, tail)


@pytest.mark.parametrize("name,layers,n,chunk,lanes", [
    ("tinyllama", 2, 194, 64, None),  # final chunk of 2: decode attention with its own K/V store
    ("tinyllama", 1, 197, 64, None),  # final chunk of 5: chunked attention
    ("qwen05", 2, 70, 16, None),      # Q8_0 with bias
    ("qwen05", 1, 90, 16, "4"),       # six chunks, four in flight whatever the queue count
    ("qwen05", 1, 90, 16, "1"),       # several chunks on one lane
])
def test_forward_ranges_equals_chunk_at_a_time(monkeypatch, name, layers, n, chunk, lanes):
    from detllm_amd import synth
    from detllm_amd.model import F32Llama

    monkeypatch.setenv("DETLLM_NO_WIDE_LANES", "1")
    if lanes:
        monkeypatch.setenv("DETLLM_LANES", lanes)  # read when the session is created

    w = synth.WORKLOADS[name]
    data = synth.build_model(w, layers=layers)
    toks = synth.tokens(w, n)
    m = F32Llama.from_gguf(data)
    tail = 256
    rows, syms = _rows_symbols(n, m.vocab, tail, seed=n)
    print(f"forward_ranges {name} layers={layers} n={n} chunk={chunk} lanes={lanes}", flush=True)
    with m.forward_workspace(n, chunk) as s:
        cum, freq, total = s.forward_ranges(toks, 0, rows, syms, tail)
        again = s.forward_ranges(toks, 0, rows, syms, tail)
        want = [], [], []
        for p in range(0, n, chunk):
            T = min(chunk, n - p)
            s.forward_chunk(toks[p:p + T], p)
            sel = (rows >= p) & (rows < p + T)
            if sel.any():
                for dst, src in zip(want, s.symbol_ranges_rows(rows[sel] - p, syms[sel], tail)):
                    dst.append(src)
    for got, rep, ref in zip((cum, freq, total), again, want):
        ref = np.concatenate(ref)
        assert np.array_equal(got, ref)
        assert np.array_equal(rep, got)
    # spot-check a few rows against the oracle at full width
    if name == "qwen05":
        pick = [0, rows.size // 2, rows.size - 1]
        ref = _oracle_ranges(data, toks, 0, rows[pick], syms[pick], tail)
        assert [(int(cum[i]), int(freq[i]), int(total[i])) for i in pick] == ref


@pytest.mark.parametrize("name,n,chunk,lanes", [
    ("tinyllama", 515, 64, None),   # two wide lanes, the first reused, a last chunk of three
    ("smollm2", 1030, 1, None),     # both reused, from a single-position session
    ("smollm2", 770, 64, "1"),      # four wide chunks on one lane, a last chunk of two
    ("smollm2", 700, 300, None),    # the session's own lanes (max_chunk past 256)
    ("smollm2", 1282, 256, "4"),    # its own four, two of them reused, a last chunk of two
    ("smollm2", 1285, 256, "3"),    # three, each used twice, a last chunk of five
    ("smollm2", 1285, 256, "1"),
    ("smollm2", 257, 255, None),
])
def test_forward_ranges_over_several_wide_chunks(monkeypatch, name, n, chunk, lanes):
    from detllm_amd import synth
    from detllm_amd.model import F32Llama

    if lanes:
        monkeypatch.setenv("DETLLM_LANES", lanes)
    w = dataclasses.replace(synth.WORKLOADS[name], vocab=1001)
    m = F32Llama.from_gguf(synth.build_model(w, layers=2))
    toks = synth.tokens(w, n)
    rows, syms = _rows_symbols(n, m.vocab, 256, seed=n)
    with m.forward_workspace(n, 128) as s:
        want = [], [], []
        for p in range(0, n, 128):
            T = min(128, n - p)
            s.forward_chunk(toks[p:p + T], p)
            sel = (rows >= p) & (rows < p + T)
            if sel.any():
                for dst, src in zip(want, s.symbol_ranges_rows(rows[sel] - p, syms[sel], 256)):
                    dst.append(src)
    with m.forward_workspace(n, chunk) as s:
        for _ in range(3):
            for got, ref in zip(s.forward_ranges(toks, 0, rows, syms, 256), want):
                assert np.array_equal(got, np.concatenate(ref))
            # the session's own lanes afterwards, on the cache the wide lanes wrote
            s.forward_chunk(toks[n - 1:], n - 1)
            cum, freq, total = s.symbol_ranges([7], 0, 256)
            with m.forward_workspace(n, 64) as t:
                for p in range(0, n, 64):
                    t.forward_chunk(toks[p:min(n, p + 64)], p)
                last = t.symbol_ranges([7], (n - 1) % 64, 256)
            assert (cum[0], freq[0], total[0]) == (last[0][0], last[1][0], last[2][0])


@pytest.mark.parametrize("rows", [0, 40, 330])
def test_forward_ranges_without_room_for_lanes(monkeypatch, rows):
    # Room for `rows` positions of lanes beside the session's first, which
    # takes 16: none (every chunk on that lane); two more of its kind and no
    # wide one; one wide lane and not the second.
    from detllm_amd import synth
    from detllm_amd.model import F32Llama

    n = 600
    w = dataclasses.replace(synth.WORKLOADS["smollm2"], vocab=1001)
    # a lane's bytes per position: logits and CDF exps, scores, activations
    row = 8 * w.vocab + 4 * w.heads * n + 12 * w.ff + 16 * w.d + 8 * (w.d // w.heads) * w.kv_heads + 6 * w.ff
    m = F32Llama.from_gguf(synth.build_model(w, layers=2))
    toks = synth.tokens(w, n)
    syms = [(int(t) * 7 + 1) % w.vocab for t in toks]
    with m.forward_workspace(n, 16) as s:
        want = s.forward_ranges(toks, 0, range(n), syms, 256)
    monkeypatch.setenv("DETLLM_LANE_MEMORY", str(rows * row))
    with m.forward_workspace(n, 16) as s:
        for _ in range(2):
            for got, ref in zip(s.forward_ranges(toks, 0, range(n), syms, 256), want):
                assert np.array_equal(got, ref)


@pytest.mark.parametrize("env,lanes", [({}, [1, 2]), ({"DETLLM_LANES": "1"}, [1, 1]),
                                       ({"DETLLM_LANE_MEMORY": "0"}, [0, 0])])
def test_wide_lanes_are_set_up_as_calls_need_them(monkeypatch, env, lanes):
    # A call of one chunk takes one wide lane's memory, a longer one the
    # second's; one lane per session stays at one.
    from detllm_amd import synth
    from detllm_amd.model import F32Llama

    hip = C.CDLL("libamdhip64.so.7")  # the runtime the library is linked with

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    for k, v in env.items():
        monkeypatch.setenv(k, v)
    w = synth.WORKLOADS["smollm2"]
    m = F32Llama.from_gguf(synth.build_model(w, layers=1))
    toks = synth.tokens(w, 300)
    lane = 256 * 8 * w.vocab  # logits and CDF exps, nearly all of a lane of this vocabulary
    gc.collect()
    with m.forward_workspace(300, 16) as warm:  # what a first launch of each kernel takes
        warm.forward_ranges(toks, 0, range(300), toks, 256)
    with m.forward_workspace(300, 16) as s:
        free = free_bytes()
        for n, count in zip((70, 300), lanes):
            s.forward_ranges(toks[:n], 0, range(n), toks[:n], 256)
            took = (free - free_bytes()) / lane
            assert count - 0.2 <= took <= 1.2 * count + 0.1, (n, took)


def test_two_lanes_run_side_by_side_whatever_other_sessions_there_are(monkeypatch):
    # The lanes' streams run side by side (0.7 of one lane's time), however many
    # streams the process has: on one hardware queue two lanes take 0.96 of it, on
    # two queues of one pipe 1.4.
    import time

    from detllm_amd import synth
    from detllm_amd.model import F32Llama

    w = dataclasses.replace(synth.WORKLOADS["qwen05"], vocab=4000)
    m = F32Llama.from_gguf(synth.build_model(w, layers=6))
    tiny = F32Llama.from_gguf(synth.build_model(synth.WORKLOADS["tiny"]))
    n = 1000
    toks = synth.tokens(w, n)

    def ms():
        with m.forward_workspace(2048, 64) as s:
            s.forward_ranges(toks, 0, range(n), toks, 256)
            best = 1e9
            for _ in range(5):
                t = time.perf_counter()
                s.forward_ranges(toks, 0, range(n), toks, 256)
                best = min(best, time.perf_counter() - t)
        return best * 1e3

    monkeypatch.setenv("DETLLM_LANES", "1")
    one = ms()
    monkeypatch.delenv("DETLLM_LANES")
    others = []
    for k in range(10):
        two = ms()
        print(f"{k} other sessions: one lane {one:.2f} ms, two {two:.2f} ms", flush=True)
        assert two < 0.85 * one, k
        others.append(tiny.forward_workspace(8, 3))
        if k == 5:
            del others[::2]  # queues used unevenly


def test_forward_ranges_errors():
    from detllm_amd import synth
    from detllm_amd._lib import DetllmError
    from detllm_amd.model import F32Llama

    w = synth.WORKLOADS["tiny"]
    m = F32Llama.from_gguf(synth.build_model(w))
    toks = synth.tokens(w, 6)
    with m.forward_workspace(8, 3) as s:
        with pytest.raises(DetllmError) as e:       # rows must not decrease
            s.forward_ranges(toks, 0, [2, 1], [0, 0], 0)
        assert e.value.status == 1
        with pytest.raises(DetllmError) as e:       # row past the tokens
            s.forward_ranges(toks, 0, [6], [0], 0)
        assert e.value.status == 1
        with pytest.raises(DetllmError) as e:       # symbol outside vocab + tail
            s.forward_ranges(toks, 0, [0], [m.vocab], 0)
        assert e.value.status == 23
        with pytest.raises(DetllmError) as e:       # past n_ctx
            s.forward_ranges(toks, 4, [0], [0], 0)
        assert e.value.status == 1
        # the session still works afterwards, on its first lane
        cum, freq, total = s.forward_ranges(toks, 0, [0, 5], [1, 2], 0)
        logits = s.forward_chunk(toks[:3], 0, want_logits=True)
        assert logits.shape == (3, m.vocab)
