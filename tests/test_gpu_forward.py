"""Full decoder forward on the GPU: logits bit-identical to the reference.

The tiny-f32 / tiny-qmix fixtures are checked against the reference's own
committed SHA-256 values; the SmolLM2-, Qwen2.5- and TinyLlama-shaped synthetic models against the
oracle at full width (a few positions, truncated depth where noted) and
through size-independent properties (chunk invariance, repeatability).
"""
import numpy as np
import pytest

import detref
from conftest import GOLDEN

pytestmark = pytest.mark.gpu


def _model(data):
    from detllm_amd.model import F32Llama

    return F32Llama.from_gguf(data)


def _fixture_tokens():
    return [int(t) for t in (GOLDEN / "tiny.tokens.txt").read_text().strip().split(",")]


@pytest.mark.parametrize("name", ["tiny-f32", "tiny-qmix"])
@pytest.mark.parametrize("chunk", [1, 2, 3, 6])
def test_fixture_hash_matches_reference_golden(name, chunk):
    m = _model((GOLDEN / f"{name}.gguf").read_bytes())
    want = (GOLDEN / f"{name}.logits.sha256").read_text().strip()
    assert m.logits_hash_for_tokens_chunked(_fixture_tokens(), chunk).hex() == want


def _compare_with_oracle(data, tokens, chunk):
    m = _model(data)
    ref = detref.Model(data).logits(tokens)
    got = []
    m.visit_logits_for_tokens_chunked(tokens, chunk, lambda row: got.append(row.copy()))
    got = np.stack(got)
    assert got.shape == ref.shape
    bad = np.nonzero(got.view(np.uint32) != ref.view(np.uint32))
    assert bad[0].size == 0, f"first mismatch at position {bad[0][:1]}, index {bad[1][:1]}"
    return m, got


def test_tiny_workload_matches_oracle_all_chunks():
    from detllm_amd import synth

    w = synth.WORKLOADS["tiny"]
    data = synth.build_model(w)
    toks = synth.tokens(w)
    m, got = _compare_with_oracle(data, toks, w.chunk)
    ref_hash = detref.Model(data).logits_hash(toks)
    for chunk in (1, 2, 3, 8):
        assert m.logits_hash_for_tokens_chunked(toks, chunk) == ref_hash


@pytest.mark.parametrize("name,layers,n_tok,chunk", [
    ("smollm2", 4, 5, 2),
    ("qwen05", 3, 5, 3),
    ("tinyllama", 2, 4, 4),
    # chunks of >= 16 positions run the token-parallel kernels (and the fused
    # gate/up/SwiGLU pass for Q4_K), including a partial final chunk
    ("smollm2", 2, 40, 32),
    ("qwen05", 1, 21, 21),
    ("tinyllama", 1, 70, 64),
    ("tinyllama", 1, 37, 37),   # Q4_K GEMM tiles with positions past the chunk
])
def test_baseline_shapes_match_oracle(name, layers, n_tok, chunk):
    from detllm_amd import synth

    w = synth.WORKLOADS[name]
    data = synth.build_model(w, layers=layers)
    _compare_with_oracle(data, synth.tokens(w, n_tok), chunk)


@pytest.mark.parametrize("name,heads,kv_heads", [
    ("smollm2", 9, 3),   # 64-wide heads
    ("qwen05", 14, 2),   # biases on the concatenated q/k/v launch
    ("smollm2", 18, 6),  # 32-wide heads
])
@pytest.mark.parametrize("chunk", [1, 3, 4, 8, 13, 34])
def test_f32_model_matches_oracle(name, heads, kv_heads, chunk):
    # F32 weights: q/k/v and gate/up/SwiGLU in one launch each, by GEMV up to
    # four positions and on the matrix cores beyond.
    import dataclasses

    from detllm_amd import synth

    w = dataclasses.replace(synth.WORKLOADS[name], weight="f32", vocab=515, heads=heads, kv_heads=kv_heads)
    _compare_with_oracle(synth.build_model(w, layers=2), synth.tokens(w, min(36, 3 * chunk)), chunk)


@pytest.mark.parametrize("name,layers,n_tok,chunk", [
    ("smollm2", 2, 9, 9), ("qwen05", 1, 13, 13), ("tinyllama", 2, 11, 11), ("tinyllama", 1, 15, 15),
])
def test_chunks_past_the_decode_gemvs_match_oracle(name, layers, n_tok, chunk):
    # Nine to fifteen positions: one partial position tile of the chunk GEMMs.
    from detllm_amd import synth

    w = synth.WORKLOADS[name]
    _compare_with_oracle(synth.build_model(w, layers=layers), synth.tokens(w, n_tok), chunk)


@pytest.mark.parametrize("d,chunk", [(576, 5), (576, 6), (512, 7), (1024, 5), (1024, 6), (1024, 8)])
def test_int8_few_positions_match_oracle(d, chunk):
    # Q8_0 chunks at the edge between the GEMVs and the chunk GEMMs,
    # block counts of a row that are and are not multiples of four, a gate and
    # up pair of few rows (K split over the waves).
    import dataclasses

    from detllm_amd import synth

    w = dataclasses.replace(synth.WORKLOADS["smollm2"], d=d, heads=d // 64, kv_heads=1, ff=736, vocab=300)
    _compare_with_oracle(synth.build_model(w, layers=2), synth.tokens(w, 2 * chunk), chunk)


@pytest.mark.parametrize("mirror", [True, False])
@pytest.mark.parametrize("chunk", [3, 4, 8])
def test_q4k_few_positions_match_oracle(monkeypatch, mirror, chunk):
    # Q4_K chunks at the edge between the GEMV and the chunk GEMMs, and past
    # it without the f32 copies (the GEMV then serves up to eight positions).
    from detllm_amd import synth

    if not mirror:
        monkeypatch.setenv("DETLLM_NO_F32_MIRROR", "1")
    w = synth.WORKLOADS["tinyllama"]
    _compare_with_oracle(synth.build_model(w, layers=2), synth.tokens(w, chunk), chunk)


@pytest.mark.parametrize("name,d,heads,kv_heads", [
    ("smollm2", 576, 36, 12),  # 16-wide heads
    ("qwen05", 448, 14, 2),    # 32, split-half RoPE, biases
    ("smollm2", 640, 8, 4),    # 80
    ("smollm2", 576, 6, 6),    # 96, one query head per key head
    ("qwen05", 896, 7, 1),     # 128
    ("smollm2", 128, 2, 1),    # 64
])
@pytest.mark.parametrize("prefix", [0, 250, 2045])
@pytest.mark.parametrize("graph", [True, False])
def test_decode_attention_head_widths_match_oracle(monkeypatch, name, d, heads, kv_heads, prefix, graph):
    # Decode attention of one to four positions at the edges of its key tiles
    # (256 keys), of the score blocks (128) and of the 2048-key limit of the
    # 64-wide kernels, by graph replay and by eager launches.
    import dataclasses

    from detllm_amd import synth

    if not graph:
        monkeypatch.setenv("DETLLM_NO_GRAPH", "1")
    if prefix > 1000:  # a narrow model of the same head width keeps the oracle quick
        hd = d // heads
        d, heads, kv_heads = 2 * hd + (-2 * hd) % 32, 2, 1
        if d != 2 * hd:
            pytest.skip("no narrow model of this head width has whole 32-element blocks")
    w = dataclasses.replace(synth.WORKLOADS[name], d=d, heads=heads, kv_heads=kv_heads, ff=64, vocab=300, ctx=2100)
    data = synth.build_model(w, layers=1)
    toks = [int(t) for t in synth.tokens(w, prefix + 14)]
    ref = detref.Model(data).logits(toks)
    m = _model(data)
    with m.forward_workspace(2100, 64) as s:
        for p in range(0, prefix, 64):
            s.forward_chunk(toks[p:min(prefix, p + 64)], p)
        p = prefix
        for n in (1, 1, 2, 1, 4, 1, 3, 1):
            got = s.forward_chunk(toks[p:p + n], p, want_logits=True)
            assert np.array_equal(got.view(np.uint32), ref[p:p + n].view(np.uint32)), (p, n)
            p += n


@pytest.mark.parametrize("name,d,heads,kv_heads", [
    ("smollm2", 576, 36, 12),  # 16-wide heads, three query heads per key head
    ("qwen05", 448, 14, 2),    # 32, seven
    ("smollm2", 640, 8, 4),    # 80
    ("smollm2", 576, 6, 6),    # 96, one
    ("qwen05", 896, 7, 1),     # 128, seven
])
@pytest.mark.parametrize("chunks", [(5, 11), (33, 64, 31), (130, 7)])
def test_chunk_attention_head_widths_match_oracle(name, d, heads, kv_heads, chunks):
    # Chunk attention on the matrix cores: tiles of 16 or 32 query rows that
    # start and end inside a position, partial key tiles, position 0 (which
    # copies its value row), rows past one 64-key slice.
    import dataclasses

    from detllm_amd import synth

    w = dataclasses.replace(synth.WORKLOADS[name], d=d, heads=heads, kv_heads=kv_heads, ff=64, vocab=300, ctx=301)
    data = synth.build_model(w, layers=2)
    toks = [int(t) for t in synth.tokens(w, sum(chunks))]
    ref = detref.Model(data).logits(toks)
    with _model(data).forward_workspace(301, 130) as s:
        p = 0
        for n in chunks:
            got = s.forward_chunk(toks[p:p + n], p, want_logits=True)
            bad = np.nonzero(got.view(np.uint32) != ref[p:p + n].view(np.uint32))
            assert bad[0].size == 0, (p, bad[0][:1], bad[1][:1])
            p += n


@pytest.mark.parametrize("name,d,heads,kv_heads,ctx", [
    ("smollm2", 64, 8, 4, 200),     # widths that only the general kernels take: 8
    ("qwen05", 192, 8, 2, 200),     # 24, split-half RoPE, biases
    ("smollm2", 384, 8, 2, 200),    # 48, one workgroup per group of heads
    ("smollm2", 384, 8, 2, 9000),   # 48, a score row per wave in memory (no room in LDS)
    ("smollm2", 864, 18, 1, 200),   # 48, more than sixteen heads per group
    ("smollm2", 448, 4, 2, 200),    # 112
    ("qwen05", 512, 2, 1, 200),     # 256
    ("smollm2", 576, 2, 1, 200),    # 288, past the one-workgroup kernel's width
    ("smollm2", 832, 13, 1, 200),   # 64, nine to sixteen heads per group
    ("smollm2", 1152, 18, 1, 200),  # 64, more: the matrix-core launches
])
def test_attention_of_other_head_shapes_matches_oracle(name, d, heads, kv_heads, ctx):
    import dataclasses

    from detllm_amd import synth

    w = dataclasses.replace(synth.WORKLOADS[name], d=d, heads=heads, kv_heads=kv_heads, ff=64, vocab=300, ctx=ctx)
    data = synth.build_model(w, layers=2)
    steps = (1, 5, 1, 33, 4, 70, 1, 3)
    toks = [int(t) for t in synth.tokens(w, sum(steps))]
    ref = detref.Model(data).logits(toks)
    with _model(data).forward_workspace(ctx, 70) as s:
        p = 0
        for n in steps:
            got = s.forward_chunk(toks[p:p + n], p, want_logits=True)
            bad = np.nonzero(got.view(np.uint32) != ref[p:p + n].view(np.uint32))
            assert bad[0].size == 0, (p, n, bad[0][:1], bad[1][:1])
            p += n


@pytest.mark.parametrize("d,heads,layers,prefix,chunks", [
    (256, 2, 2, 1485, (33, 70)),    # 128-wide heads
    (192, 2, 2, 700, (5, 130)),     # 96
    (160, 2, 2, 700, (64, 17)),     # 80
    (32, 2, 2, 2045, (6, 100)),     # 16
    (1024, 16, 1, 1760, (20, 13, 30)),  # 64, sixteen heads per group: to and past the one-launch kernel's LDS
])
def test_chunk_attention_long_rows_match_oracle(d, heads, layers, prefix, chunks):
    # Chunk attention far into a window: every position of the chunks is
    # compared, and with two layers the prefix's own attention reaches them.
    import dataclasses

    from detllm_amd import synth

    n = prefix + sum(chunks)
    w = dataclasses.replace(synth.WORKLOADS["smollm2"], d=d, heads=heads, kv_heads=1, ff=64, vocab=300, ctx=n)
    data = synth.build_model(w, layers=layers)
    toks = [int(t) for t in synth.tokens(w, n)]
    ref = detref.Model(data).logits(toks)
    with _model(data).forward_workspace(n, 256) as s:
        for p in range(0, prefix, 256):
            s.forward_chunk(toks[p:min(prefix, p + 256)], p)
        p = prefix
        for c in chunks:
            got = s.forward_chunk(toks[p:p + c], p, want_logits=True)
            bad = np.nonzero(got.view(np.uint32) != ref[p:p + c].view(np.uint32))
            assert bad[0].size == 0, (p, c, bad[0][:1], bad[1][:1])
            p += c


@pytest.mark.parametrize("d,heads,prefix,chunks", [
    (512, 8, 4205, (8, 13, 30)),   # 64-wide heads, eight per group: to and past the one-launch kernel's LDS
    (32, 2, 19100, (55, 25, 40)),  # 16-wide: past the softmax launch's LDS (about 19170 keys)
])
def test_chunk_attention_of_very_long_rows_equals_decode(d, heads, prefix, chunks):
    # Rows too long for the oracle: the chunks' logits against those of single
    # positions, whose attention the tests above compare with the oracle.
    import dataclasses

    from detllm_amd import synth

    n = prefix + sum(chunks)
    w = dataclasses.replace(synth.WORKLOADS["smollm2"], d=d, heads=heads, kv_heads=1, ff=64, vocab=300, ctx=n)
    toks = [int(t) for t in synth.tokens(w, n)]
    with _model(synth.build_model(w, layers=2)).forward_workspace(n, 512) as s:
        for p in range(0, prefix, 512):
            s.forward_chunk(toks[p:min(prefix, p + 512)], p)
        p = prefix
        for c in chunks:
            got = s.forward_chunk(toks[p:p + c], p, want_logits=True)
            for i in range(c):
                one = s.forward_one(toks[p + i], p + i)
                assert np.array_equal(got[i].view(np.uint32), one.view(np.uint32)), p + i
            p += c


def test_decode_attention_long_row_matches_oracle():
    # The Z chains run in segments of 8192 exps: rows just below, at and past one.
    import dataclasses

    from detllm_amd import synth

    w = dataclasses.replace(synth.WORKLOADS["smollm2"], d=32, heads=2, kv_heads=1, ff=32, vocab=257, ctx=8300)
    data = synth.build_model(w, layers=1)
    toks = [int(t) for t in synth.tokens(w, 8300)]
    ref = detref.Model(data).logits(toks)
    with _model(data).forward_workspace(8300, 512) as s:
        for p in range(0, 8190, 512):
            s.forward_chunk(toks[p:min(8190, p + 512)], p)
        for p, n in ((8190, 1), (8191, 1), (8192, 1), (8193, 4), (8299, 1)):
            if p == 8299:
                s.forward_chunk(toks[8197:8299], 8197)
            got = s.forward_chunk(toks[p:p + n], p, want_logits=True)
            assert np.array_equal(got.view(np.uint32), ref[p:p + n].view(np.uint32)), (p, n)


@pytest.mark.parametrize("name,chunk", [("qwen05", 1), ("qwen05", 4), ("smollm2", 5)])
@pytest.mark.parametrize("fused", [True, False])
def test_decode_gemv_fusion_matches_oracle(monkeypatch, name, chunk, fused):
    # Up to five positions the Q8_0 layers run the fused decode GEMVs
    # (rmsnorm / quantisation in the GEMV prologue, q/k/v in one launch,
    # gate/up finishing as swiglu); both that and the separate launches must
    # give the reference bits.
    from detllm_amd import synth

    if not fused:
        monkeypatch.setenv("DETLLM_NO_FUSED_DECODE", "1")
    monkeypatch.setenv("DETLLM_NO_GRAPH", "1")
    w = synth.WORKLOADS[name]
    _compare_with_oracle(synth.build_model(w, layers=2), synth.tokens(w, 10), chunk)


def test_fused_decode_mixed_q8_0_q4_0_fixture():
    # tiny-qmix mixes Q8_0 and Q4_0 within q/k/v and gate/up: each matrix
    # gets its own fused launch; the reference's golden hash must hold.
    m = _model((GOLDEN / "tiny-qmix.gguf").read_bytes())
    want = (GOLDEN / "tiny-qmix.logits.sha256").read_text().strip()
    assert m.logits_hash_for_tokens_chunked(_fixture_tokens(), 1).hex() == want


@pytest.mark.parametrize("env", ["DETLLM_NO_F32_MIRROR", "DETLLM_NO_Q6K_PLANES"])
def test_packed_chunk_paths_match_oracle(monkeypatch, env):
    # Without the encode copies (Q4_K f32 weights, Q6_K matrix-core planes)
    # the chunked GEMMs decode the packed superblocks themselves; every path
    # must give the reference bits.
    from detllm_amd import synth

    monkeypatch.setenv(env, "1")
    w = synth.WORKLOADS["tinyllama"]
    _compare_with_oracle(synth.build_model(w, layers=1), synth.tokens(w, 40), 40)


@pytest.mark.parametrize("name", ["qwen05", "tinyllama"])
def test_single_position_graph_replay_matches_oracle(monkeypatch, name):
    # One-position forwards replay a captured graph (the position reaches the
    # kernels through device memory); every replay, a reset session and the
    # eager launches must give the reference bits.
    from detllm_amd import synth

    w = synth.WORKLOADS[name]
    data = synth.build_model(w, layers=1)
    toks = [int(t) for t in synth.tokens(w, 12)]
    ref = detref.Model(data).logits(toks)
    m = _model(data)
    with m.forward_workspace(16, 1) as s:
        for rep in range(2):
            for p, tok in enumerate(toks):
                got = s.forward_one(tok, p)
                assert np.array_equal(got.view(np.uint32), ref[p].view(np.uint32)), (rep, p)
            s.reset()
    monkeypatch.setenv("DETLLM_NO_GRAPH", "1")
    with m.forward_workspace(16, 1) as s:
        for p, tok in enumerate(toks[:4]):
            assert np.array_equal(s.forward_one(tok, p).view(np.uint32), ref[p].view(np.uint32))


@pytest.mark.parametrize("cores", [1, 2, 99])
def test_large_logits_reach_the_host_whatever_the_cores(cores):
    # Results of 2 MB and more by as many threads as the caller has cores; one
    # core takes the single copy.  Rows on both sides of a slice's end.
    import os

    from detllm_amd import synth

    w = synth.WORKLOADS["smollm2"]
    m = _model(synth.build_model(w, layers=1))
    toks = synth.tokens(w, 45)
    mine = os.sched_getaffinity(0)
    with m.forward_workspace(45, 45) as s:
        s.forward_chunk(toks, 0)
        want = np.concatenate([s.logits(i, 1) for i in range(45)])  # 197 KB each: one copy
        try:
            os.sched_setaffinity(0, set(sorted(mine)[:cores]))
            for n in (11, 16, 17, 45):  # two slices and a part, three, three and a part, eight and a part
                assert np.array_equal(s.logits(0, n).view(np.uint32), want[:n].view(np.uint32))
        finally:
            os.sched_setaffinity(0, mine)


def test_repeat_runs_are_bitwise_identical():
    from detllm_amd import synth

    w = synth.WORKLOADS["smollm2"]
    m = _model(synth.build_model(w, layers=2))
    toks = synth.tokens(w, 16)
    hashes = {m.logits_hash_for_tokens_chunked(toks, c) for c in (1, 5, 16, 16)}
    assert len(hashes) == 1


def test_session_errors_mirror_reference_shape_checks():
    from detllm_amd._lib import DetllmError

    m = _model((GOLDEN / "tiny-f32.gguf").read_bytes())
    with m.forward_workspace(4, 2) as s:
        with pytest.raises(DetllmError) as e:
            s.forward_chunk([0, 1, 2], 0)  # more positions than max_chunk
        assert e.value.status == 1
        with pytest.raises(DetllmError) as e:
            s.forward_one(10_000, 0)      # token outside the vocabulary
        assert e.value.status == 1
        with pytest.raises(DetllmError) as e:
            s.forward_one(0, 4)           # position outside the window
        assert e.value.status == 1


def test_cdf_on_device_logits_matches_oracle():
    from detllm_amd import synth

    w = synth.WORKLOADS["smollm2"]
    data = synth.build_model(w, layers=2)
    m = _model(data)
    toks = synth.tokens(w, 6)
    with m.forward_workspace(8, 6) as s:
        logits = s.forward_chunk(toks, 0, want_logits=True)
        syms = [int(t) for t in synth.tokens(w, 7)[1:7]]
        for tail in (0, 256):
            cum, freq, total = s.symbol_ranges(syms, 0, tail)
            for i in range(6):
                assert (int(cum[i]), int(freq[i]), int(total[i])) == detref.symbol_range(logits[i], syms[i], tail)
            f, c, t = s.cdf(2, tail)
            rf, rc, rt = detref.logits_to_cdf(logits[2], tail)
            assert np.array_equal(f, rf) and np.array_equal(c, rc) and t == rt
            # values inside, at the start and at the end of symbols, including the
            # 4096-symbol work-block edges, the last vocab symbol and the escapes
            values = {0, rt - 1, int(rc[100]), int(rc[100]) + int(rf[100]) - 1}
            for sym in (4095, 4096, 4097, 8191, 8192, len(rf) - tail - 1):
                values |= {int(rc[sym]), int(rc[sym]) + int(rf[sym]) - 1}
            if tail:
                values |= {int(rc[len(rf) - tail]), int(rc[len(rf) - 1])}
            for value in sorted(values):
                assert s.decoder_lookup(value, 2, tail) == detref.decoder_lookup(logits[2], value, tail), value
            assert s.decoder_total(2, tail) == rt


@pytest.mark.parametrize("tail", [0, 256])
def test_fused_decode_steps_match_oracle_ranges(tail):
    """dtl_forward_decode / dtl_decoder_decode against a payload coded with
    the oracle's symbol ranges: the symbols and, after every step, the range
    decoder's state equal a host decoder fed the oracle's ranges.  The
    symbols sit on the 4096-symbol work-block edges, at the vocabulary's end,
    on the most likely token and (tail 256) on byte escapes, which are not
    forwarded, so the next decode reads the same row again."""
    from detllm_amd import coder, synth
    from detllm_amd._lib import DetllmError

    w = synth.WORKLOADS["smollm2"]
    data = synth.build_model(w, layers=2)
    m = _model(data)
    V = w.vocab
    t0 = int(synth.tokens(w, 1)[0])
    esc = (V + 3, V + 255) if tail else (17, 30000)
    with m.forward_workspace(16, 1) as s:
        lg = s.forward_one(t0, 0)
        syms = [4095, 4096, V - 1, esc[0], None, 8192, 0, esc[1], 12345, 4097]  # None: the argmax
        enc, ranges, pos = coder.RangeEncoder(), [], 1
        for i, want in enumerate(syms):
            if want is None:
                want = syms[i] = int(np.argmax(lg))
            r = detref.symbol_range(lg, want, tail)
            enc.encode(*r)
            ranges.append(r)
            if want < V:
                lg = s.forward_one(want, pos)
                pos += 1
        payload = enc.finish()

    def state(d):
        st = d.snapshot()
        return st.low, st.range, st.code, st.pos

    with m.forward_workspace(16, 1) as s:
        dec, host = coder.RangeDecoder(payload), coder.RangeDecoder(payload)
        s.forward_one(t0, 0, want_logits=False)
        pos, pend = 1, None
        for want, (cum, freq, total) in zip(syms, ranges):
            if pend is None:
                got = s.decode_symbol(dec, 0, tail)
            else:
                got = s.forward_decode(pend, pos, dec, tail)
                pos += 1
            v = host.decode_freq(total)
            assert cum <= v < cum + freq
            host.advance(cum, freq, total)
            assert got == want
            assert state(dec) == state(host)
            pend = got if got < V else None
        # a decoder between decode_freq and advance, a token outside the vocabulary
        host.decode_freq(ranges[0][2])
        with pytest.raises(DetllmError) as e:
            s.decode_symbol(host, 0, tail)
        assert e.value.status == 30
        with pytest.raises(DetllmError) as e:
            s.forward_decode(V, pos, dec, tail)
        assert e.value.status == 1


@pytest.mark.parametrize("V", [4, 256, 32000, 151936])
def test_standalone_cdf_kernel_matches_oracle(V):
    from detllm_amd import coder

    rng = np.random.default_rng(V)
    lg = rng.normal(0, 4, V).astype(np.float32)
    if V == 4:
        lg[:] = 0.0
    else:
        lg[:11] = [0.0, -1.0, 3.25, 3.25, -88.5, np.float32(2 ** -149), -12.0, 0.5, -0.25, 2.0, -1000.0]
    for tail in (0, 256):
        got = coder._cdf(lg, tail)
        rf, rc, rt = detref.logits_to_cdf(lg, tail)
        assert np.array_equal(got.freq, rf) and np.array_equal(got.cum, rc) and got.total == rt
        for s in (0, V // 2, V - 1, V + tail - 1):
            r = coder._range(lg, s, tail)
            assert (r.cum, r.freq, r.total) == detref.symbol_range(lg, s, tail)


@pytest.mark.parametrize("V", [32767, 32768, 40003, 151936, 261888])
@pytest.mark.parametrize("pattern", ["equal", "halves", "spread", "peaked", "growing", "tiny chains", "ulps", "random"])
def test_cdf_normaliser_by_many_threads_matches_oracle(V, pattern):
    # From 32768 logits a few rows' Z chains are summed by many threads (maps
    # of rounded increments, composed): terms that are ties of the running
    # sum's grid in both directions, sums that cross many binades, late or in
    # one block, one dominant term, terms far below the grid, chains whose
    # sums stay subnormal, and (f sensitive to Z's last bits) large
    # probabilities in each.
    from detllm_amd import coder

    rng = np.random.default_rng(V)
    ln2 = np.log(2.0)
    if pattern == "equal":
        lg = np.zeros(V)
    elif pattern == "halves":  # e near powers of two: bits just below the grid
        lg = -ln2 * rng.integers(0, 24, V)
    elif pattern == "spread":
        lg = np.linspace(-80, 0, V)[rng.permutation(V)]
    elif pattern == "peaked":
        lg = rng.normal(-20, 3, V)
        lg[V // 3], lg[V // 2], lg[7] = 0.0, -0.7, -3.0
    elif pattern == "growing":  # the largest terms last
        lg = np.linspace(-60, 0, V)
    elif pattern == "tiny chains":  # only chain 3 holds terms that are not subnormal
        lg = np.full(V, -200.0)
        lg[3::8] = rng.normal(-1, 1, lg[3::8].size)
    elif pattern == "ulps":
        lg = rng.normal(0, 1e-6, V)
        lg[: V // 2] -= 9.0
    else:
        lg = rng.normal(0, 3, V)
    lg = lg.astype(np.float32)
    rf, rc, rt = detref.logits_to_cdf(lg, 256)
    got = coder.logits_to_cdf_with_byte_escapes(lg)
    assert np.array_equal(got.freq, rf) and np.array_equal(got.cum, rc) and got.total == rt
    for sym in (0, V // 3, V - 1):
        r = coder.logits_to_symbol_range_with_byte_escapes(lg, sym)
        assert (r.cum, r.freq, r.total) == (int(rc[sym]), int(rf[sym]), rt)


@pytest.mark.parametrize("graph", [True, False])
def test_decode_attention_regimes_match_oracle(monkeypatch, graph):
    """Single-position forwards in a 4096-position window (1-layer SmolLM2
    shape) through every decode attention they can take, bit for bit against
    the oracle.

    graph: positions below 512 replay the graph whose attention is one launch
    (k_attn_fused); from 512 on, the graph sized for the whole window, whose
    attention takes its tiled P.V launch (k_attn_tiles_pv).
    eager (DETLLM_NO_GRAPH=1, the path under profiling or after a failed
    capture): the launch is sized by the row: k_attn_fused up to 512 keys,
    the split pair (k_attn_split_scores + k_attn_split_pv) up to 2048,
    k_attn_tiles_pv beyond; the positions between are forwarded in chunks of
    64 (chunk attention)."""
    import dataclasses

    from detllm_amd import synth

    if not graph:
        monkeypatch.setenv("DETLLM_NO_GRAPH", "1")
    w = dataclasses.replace(synth.WORKLOADS["smollm2"], ctx=4096)
    data = synth.build_model(w, layers=1)
    if graph:
        singles = list(range(524))
        n = 524
    else:
        singles = [0, 1, 2, 3, 600, 601, 602, 603, 2048, 2049, 2050, 2051, 2052, 2053]
        n = 2054
    toks = [int(t) for t in synth.tokens(w, n)]
    print(f"oracle logits of {n} positions", flush=True)
    ref = detref.Model(data).logits(toks)
    m = _model(data)
    with m.forward_workspace(4096, 64) as s:
        p = 0
        while p < n:
            if p in singles:
                if p in (0, 512, 600, 2048):
                    print(f"{'graph' if graph else 'eager'} single-position forwards from {p}", flush=True)
                got = s.forward_one(toks[p], p)
                assert np.array_equal(got.view(np.uint32), ref[p].view(np.uint32)), p
                p += 1
            else:
                end = min(n, p + 64, min((q for q in singles if q > p), default=n))
                lg = s.forward_chunk(toks[p:end], p, want_logits=True)
                assert np.array_equal(lg[-1].view(np.uint32), ref[end - 1].view(np.uint32)), end - 1
                p = end
