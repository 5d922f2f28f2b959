"""What a token does not see has no part in its attention: keys behind its position - rows of its last block that nobody has
written, rows of an earlier sequence, later tokens of its prompt - may hold anything, numbers that are not finite too."""
import threading
from types import SimpleNamespace

import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from nerva_amd.runtime import attention_workspace
from test_gpu_any_width import walked
from test_gpu_ops import _attention_case, _attention_oracle, dev
from test_gpu_session import BF16, E2E_REL_L2, F16, REL_L2, oracle_follow, random_model, rel_l2, started

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,hd,dtype", [(32, 8, 128, BF16), (28, 4, 128, BF16), (10, 2, 128, F16), (14, 2, 64, F16),
                                                     (16, 2, 64, BF16), (4, 2, 80, BF16)])
def test_rows_behind_the_position_may_hold_anything(heads, kv_heads, hd, dtype):
    """Every cache element but those of keys 0 .. position is a NaN or an infinity; positions at both ends of a group of four
    rows of a block, in the first block, and where several splits merge."""
    nan, inf = (0x7fc0, 0x7f80) if dtype == BF16 else (0x7e00, 0x7c00)
    for tokens in (0, 3, 4, 5, 14, 15, 16, 129, 1001, 1007):
        c = _attention_case(dtype, heads, kv_heads, hd, tokens, 1e4, False, heads * 3 + tokens)
        ref, _, _ = _attention_oracle(c)
        cache = N.PagedKvCache(c["layers"], c["n_blocks"], kv_heads, hd, c["table"])
        written = cache.host_layout(c["layer"], np.ones_like(c["k_rows"]), np.ones_like(c["v_rows"]))
        images = cache.host_layout(c["layer"], c["k_rows"], c["v_rows"])
        for image, mark, buf in zip(images, written, (cache.k, cache.v)):
            rest = np.where(np.arange(image.size) % 3 == 0, nan, np.where(np.arange(image.size) % 3 == 1, inf, inf | 0x8000))
            buf.upload(np.where(mark != 0, image, rest).astype(np.uint16))
        out16, out32 = N.DeviceBuffer(heads * hd * 2), N.DeviceBuffer(heads * hd * 4)
        N.paged_attention(dtype, heads, kv_heads, hd, cache, c["layer"], tokens, dev(c["qkv"]), attention_workspace(heads, hd), out16,
                          out_f32=out32, append=True, rope_theta=1e4)
        assert rel_l2(out32.numpy(np.float32), ref) <= REL_L2, tokens


# hidden, heads, kv, hd, inter, vocab, layers; half precision, whose largest number is in reach
OVERFLOWING = [(192, 10, 2, 64, 320, 301, 2), (896, 14, 2, 64, 1728, 300, 2), (768, 6, 2, 128, 1536, 300, 2), (2048, 16, 4, 128, 4096, 300, 2)]


def overflowing_model(geom):
    """A model one of whose tokens (0) has a value past the largest number in dims 5 and 40 of its first layer's key head 1:
    its embedding is constant, the other tokens' have no constant part, and those dims sum the embedding up."""
    hidden, heads, kv, hd, inter, vocab, layers = geom
    weights, _ = random_model(F16, hidden, heads, kv, hd, inter, vocab, layers, hidden, 1e4, False, False)
    rng = np.random.default_rng(hidden)
    table = rng.normal(0, 1, (vocab, hidden))
    table -= table.mean(axis=1, keepdims=True)
    table[0] = 1.0
    weights.embeddings[:] = O.encode16(F16, table).reshape(weights.embeddings.shape)
    weights.layers[0]["rms_attn"][:] = O.encode16(F16, np.ones(hidden))
    w_v = weights.layers[0]["w_v"].reshape(kv * hd, hidden)
    w_v[[hd + 5, hd + 40]] = O.encode16(F16, np.full(hidden, 1e5 / hidden))
    return weights


@pytest.mark.parametrize("geom", OVERFLOWING, ids=str)
def test_a_later_tokens_infinity_does_not_reach_earlier_tokens(geom):
    """A prompt with the overflowing token in it: at its start, inside and at the edges of a step of 64 keys, and behind a
    prefix long enough for splits. The tokens before it have the logits that a walk token by token gives them; those that see
    it have none that are finite, as there."""
    weights = overflowing_model(geom)
    s, walk = N.DecodeSession.create(weights, 900), walked(weights, 900)
    assert s.create_result.prefill_chunk_tokens > 1 and walk.create_result.prefill_chunk_tokens == 1
    rng = np.random.default_rng(7)
    for prefix, tokens, at in ((0, 3, 1), (0, 70, 9), (0, 70, 63), (0, 130, 64), (650, 40, 20), (650, 150, 149)):
        prompt = rng.integers(1, weights.vocab, prefix + tokens).astype(np.uint32)
        prompt[prefix + at] = 0
        places = sorted({0, at // 2, max(0, at - 3), at - 1, min(at + 2, tokens - 1)})
        rows = []
        for session in (s, walk):
            assert session.release_sequence() == 0
            if prefix:
                rc, _, _, _ = session.extend(prompt[:prefix])
                assert rc == 0
            rows.append(session.extend(prompt[prefix:], places)[2])
        for place, got, want in zip(places, *rows):
            assert np.all(np.isfinite(want)) == (place < at), (prefix, at, place)
            if place < at:
                assert rel_l2(got, want) <= E2E_REL_L2, (prefix, at, place)
            else:
                assert not np.any(np.isfinite(got)), (prefix, at, place)
    for session in (s, walk):
        session.destroy()


@pytest.mark.parametrize("geom", OVERFLOWING, ids=str)
def test_an_earlier_sequences_rows_do_not_reach_the_next(geom):
    """A session whose cache holds infinities of the sequence before, up to behind the next one's end: prompt, steps and
    logits are those of a session that has held nothing else."""
    weights = overflowing_model(geom)
    used, fresh = N.DecodeSession.create(weights, 128), N.DecodeSession.create(weights, 128)
    used.extend(np.zeros(100, np.uint32))
    assert used.release_sequence() == 0
    for length in (1, 2, 21, 64, 70):
        prompt = np.random.default_rng(length).integers(1, weights.vocab, length).astype(np.uint32)
        results = []
        for session in (used, fresh):
            rc, _ = session.start(prompt)
            assert rc == 0
            rc, _, tokens = session.advance(4)
            assert rc == 0
            results.append((tokens.tolist(), session.logits().copy()))
            assert session.release_sequence() == 0
        assert np.all(np.isfinite(results[1][1])) and rel_l2(results[0][1], results[1][1]) <= E2E_REL_L2, length
        top = np.sort(results[1][1])
        assert results[0][0][:1] == results[1][0][:1] or top[-1] - top[-2] <= E2E_REL_L2 * np.max(np.abs(top)), length
    for session in (used, fresh):
        session.destroy()


@pytest.mark.parametrize("scale", [1.0, 1e-4, 3e3])
@pytest.mark.parametrize("heads,kv_heads,hd", [(28, 4, 128), (5, 1, 128), (6, 2, 128), (48, 8, 128), (14, 2, 64), (8, 8, 64), (32, 4, 64)])
@pytest.mark.parametrize("dtype", [BF16, F16])
def test_step_attention_keeps_the_bits_of_f32(dtype, heads, kv_heads, hd, scale):
    """Heads of 64, and of 128 with 3, 5, 6 or 7 query heads a key head, against 64 bits: queries and probabilities that had
    16 bits (bf16) or fell below half precision's smallest numbers were 3e-6 off, whatever the number of keys. 24 bits of each
    and sums in f32 leave 2^-23 from the query and the probability and less than that again from sums in pieces of 16 and 64
    (bound: four times 2^-23). Queries of 1e-4 and keys of as many times more, and the other way round: the size of either alone does not matter."""
    for n in (75, 600):
        rng = np.random.default_rng(heads * n)
        table = rng.permutation(n // 16 + 2).astype(np.uint32)
        k = O.encode16(dtype, rng.normal(0, 1 / scale, (n, kv_heads * hd)))
        v = O.encode16(dtype, rng.normal(0, 1, (n, kv_heads * hd)))
        q = rng.normal(0, scale, (heads + 2 * kv_heads) * hd).astype(np.float32)
        cache = N.PagedKvCache(1, table.size, kv_heads, hd, table)
        cache.fill(0, k, v)
        out16, out32 = N.DeviceBuffer(heads * hd * 2), N.DeviceBuffer(heads * hd * 4)
        N.paged_attention(dtype, heads, kv_heads, hd, cache, 0, n - 1, dev(q), attention_workspace(heads, hd), out16, out_f32=out32,
                          append=False)
        keys, values = (O.decode16(dtype, a).astype(np.float64).reshape(n, kv_heads, 1, hd) for a in (k, v))
        score = (keys * q[:heads * hd].astype(np.float64).reshape(1, kv_heads, -1, hd)).sum(3) / np.sqrt(hd)
        weight = np.exp(score - score.max(0))
        want = (weight[..., None] * values).sum(0) / weight.sum(0)[..., None]
        assert rel_l2(out32.numpy(np.float32), want.reshape(-1)) <= 4 * 2.0 ** -23, n


@pytest.mark.parametrize("geom", [(896, 14, 2, 64, 1728, 300, 2), (1536, 12, 2, 128, 2944, 301, 2)], ids=str)
def test_queries_below_half_precisions_smallest(geom):
    """Query weights of 1e-4 and key weights of 1e4: scores as large as any, of query elements that half precision rounds to
    some 1e-3 in their own units. Prompt blocks and batch steps against the oracle, in a model whose second layer sees little
    but the first one's attention. Rounding to 16 bits is 2^-12 of an element, in three stages up to there (embedding and
    normalised row, attention, row of the second layer): a bound of 8e-4 (scores off by 3e-3 had left up to 9.6e-4)."""
    hidden, heads, kv, hd, inter, vocab, layers = geom
    weights, _ = random_model(F16, hidden, heads, kv, hd, inter, vocab, layers, hidden, 1e4, True, False)
    weights.embeddings[:] = O.encode16(F16, 0.01 * O.decode16(F16, weights.embeddings))
    for layer in weights.layers:
        layer["q_norm"][:] = O.encode16(F16, np.full(hd, 1e-4))
        layer["k_norm"][:] = O.encode16(F16, np.full(hd, 1e4))
    weights.layers[0]["w_down"][:] = 0
    omodel = O.Model(F16, hidden, heads, kv, hd, inter, vocab, 1e-6, 1e4, weights.embeddings, weights.layers, weights.final_norm,
                     weights.lm_head)
    parent = N.DecodeSession.create(weights, 256, plan=N.WeightPlan.from_weights(weights))
    sessions = [parent, parent.fork_shared_weights(), parent.fork_shared_weights()]
    assert parent.shares_weight_stream()
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, vocab, n).astype(np.uint32) for n in (5, 70, 200)]
    streams = [[started(s, p)] for s, p in zip(sessions, prompts)]
    for _ in range(3):
        rc, _, tokens = N.DecodeSession.batch_advance_one(sessions, 3, 2)
        assert rc == 0
        for stream, token in zip(streams, tokens):
            stream.append(int(token))
    for session, prompt, stream in zip(sessions, prompts, streams):
        ctx, _ = oracle_follow(omodel, 256, prompt, stream[:-1])
        for token in (*range(2, prompt.size, 7), *range(prompt.size, prompt.size + 3)):
            for got, want in zip(session.kv_row(1, token), ctx.read_kv16(1, token)):
                assert rel_l2(O.decode16(F16, got), O.decode16(F16, want)) <= 8e-4, (prompt.size, token)
        ctx.close()
    for s in sessions[::-1]:
        s.destroy()


@pytest.mark.parametrize("geom", [(1280, 40, 8, 128, 1280, 301, 2), (896, 28, 4, 128, 896, 301, 2), (1024, 48, 8, 64, 1024, 301, 2)], ids=str)
def test_sessions_on_streams_of_their_own_do_not_hold_each_other_up(geom):
    """Four sessions decode at once, a thread and a stream each, at contexts whose splits merge inside the launch: every step
    ends without a merge that gave up, and the tokens are those of the sessions one after the other."""
    hidden, heads, kv, hd, inter, vocab, layers = geom
    weights, _ = random_model(BF16, hidden, heads, kv, hd, inter, vocab, layers, hidden, 1e4, False, False)
    sessions = [N.DecodeSession.create(weights, 1400) for _ in range(4)]
    prompts = [np.random.default_rng(i).integers(0, vocab, 1000 + 50 * i).astype(np.uint32) for i in range(4)]

    def advance(session, results, at):
        results[at] = [session.advance(25) for _ in range(6)]

    results = {}
    for how in ("alone", "together"):
        results[how] = [None] * 4
        for session, prompt in zip(sessions, prompts):
            assert session.start(prompt)[0] == 0
        threads = [threading.Thread(target=advance, args=(s, results[how], i)) for i, s in enumerate(sessions)]
        for thread in threads:
            thread.start()
            if how == "alone":
                thread.join()
        for thread in threads:
            thread.join()
    for alone, together in zip(results["alone"], results["together"]):
        for (rc, res, tokens), (rc2, res2, tokens2) in zip(alone, together):
            assert rc == rc2 == 0 and res2.hip_error == 0
            assert tokens.tolist() == tokens2.tolist()
    for session in sessions:
        session.destroy()


@pytest.mark.parametrize("heads,kv_heads,hd", [(60, 60, 64), (65, 65, 64), (171, 57, 128), (56, 56, 64), (40, 8, 128), (5, 1, 128), (96, 16, 64)])
def test_merges_by_few_workgroups(heads, kv_heads, hd):
    """Numbers of kv heads around the one from which no split may wait, and where a workgroup merges several parts."""
    c = _attention_case(BF16, heads, kv_heads, hd, 1500, 1e4, False, heads)
    ref, _, _ = _attention_oracle(c)
    cache = N.PagedKvCache(c["layers"], c["n_blocks"], kv_heads, hd, c["table"])
    cache.fill(c["layer"], c["k_rows"], c["v_rows"])
    out16, out32, ws = N.DeviceBuffer(heads * hd * 2), N.DeviceBuffer(heads * hd * 4), attention_workspace(heads, hd)
    qkv = dev(c["qkv"])
    for splits in (0, 0, 2, 4, 64):
        N.paged_attention(BF16, heads, kv_heads, hd, cache, c["layer"], 1500, qkv, ws, out16, out_f32=out32, append=True, rope_theta=1e4,
                          splits=splits)
        assert rel_l2(out32.numpy(np.float32), ref) <= REL_L2, splits
    assert N.paged_attention_status(ws, heads, hd) == (0, 0)


@pytest.mark.parametrize("heads,kv_heads,hd,dtype", [(28, 4, 128, BF16), (14, 2, 64, F16), (4, 2, 80, BF16)])
def test_caches_and_workspaces_at_any_address_of_their_elements(heads, kv_heads, hd, dtype):
    """Caches from an odd 16-bit element on, a workspace from an odd 32-bit one on, where element by element always did."""
    for tokens, shift, ws_shift in ((70, 2, 0), (1000, 14, 0), (1000, 0, 4), (1000, 6, 12)):
        c = _attention_case(dtype, heads, kv_heads, hd, tokens, 1e4, False, heads + tokens)
        ref, _, _ = _attention_oracle(c)
        cache = N.PagedKvCache(c["layers"], c["n_blocks"], kv_heads, hd, c["table"])
        images = cache.host_layout(c["layer"], c["k_rows"], c["v_rows"])
        buffers = [N.DeviceBuffer(image.nbytes + 16) for image in images]
        for buf, image in zip(buffers, images):
            buf.upload(image, shift)
        views = [SimpleNamespace(ptr=buf.ptr + shift) for buf in buffers]
        shifted = SimpleNamespace(k=views[0], v=views[1], table=cache.table, block_count=cache.block_count)
        room = N.DeviceBuffer.zeros(N.abi.load().nerva_hip_paged_attention_workspace_bytes(heads, hd) + 16)
        out16, out32 = N.DeviceBuffer(heads * hd * 2), N.DeviceBuffer(heads * hd * 4)
        N.paged_attention(dtype, heads, kv_heads, hd, shifted, c["layer"], tokens, dev(c["qkv"]), room.ptr + ws_shift, out16,
                          out_f32=out32, append=True, rope_theta=1e4)
        assert rel_l2(out32.numpy(np.float32), ref) <= REL_L2, (tokens, shift, ws_shift)


def test_a_workspace_at_an_odd_word_at_the_shapes_of_the_step_kernel():
    c = _attention_case(BF16, 32, 8, 128, 1000, 1e4, False, 5)
    ref, _, _ = _attention_oracle(c)
    cache = N.PagedKvCache(c["layers"], c["n_blocks"], 8, 128, c["table"])
    cache.fill(c["layer"], c["k_rows"], c["v_rows"])
    room = N.DeviceBuffer.zeros(N.abi.load().nerva_hip_paged_attention_workspace_bytes(32, 128) + 16)
    out16, out32 = N.DeviceBuffer(32 * 128 * 2), N.DeviceBuffer(32 * 128 * 4)
    N.paged_attention(BF16, 32, 8, 128, cache, c["layer"], 1000, dev(c["qkv"]), room.ptr + 4, out16, out_f32=out32, append=True, rope_theta=1e4)
    assert rel_l2(out32.numpy(np.float32), ref) <= REL_L2


@pytest.mark.parametrize("heads,kv_heads,hd", [(28, 4, 128), (14, 2, 64), (32, 8, 128)])
def test_a_captured_call_replayed_on_other_inputs(heads, kv_heads, hd):
    """One call on its workspace in a graph, replayed with new projections (and so a new key and value) each time, with eager
    calls on the same workspace and synchronizations between: no partial of the replay before is taken for this one's."""
    import ctypes as C
    c = _attention_case(BF16, heads, kv_heads, hd, 1500, 1e4, False, heads)
    cache = N.PagedKvCache(c["layers"], c["n_blocks"], kv_heads, hd, c["table"])
    cache.fill(c["layer"], c["k_rows"], c["v_rows"])
    qkv, ws = dev(c["qkv"]), attention_workspace(heads, hd)
    out16, out32 = N.DeviceBuffer(heads * hd * 2), N.DeviceBuffer(heads * hd * 4)
    req = N.abi.NervaHipPagedAttentionRequest()
    req.dtype, req.heads, req.kv_heads, req.head_dim = BF16, heads, kv_heads, hd
    req.layer, req.block_count, req.position, req.append = c["layer"], c["n_blocks"], 1500, 1
    req.rms_eps, req.rope_theta = 1e-6, 1e4
    req.qkv_f32, req.k_cache, req.v_cache, req.block_table = qkv.ptr, cache.k.ptr, cache.v.ptr, cache.table.ptr
    req.workspace, req.output_f32, req.output16 = ws.ptr, out32.ptr, out16.ptr
    lib = N.abi.load()
    call, err = lib.nerva_hip_paged_gqa_decode, C.c_int32(0)
    assert call(C.byref(req), None, C.byref(err)) == 0     # (the rotation table is made by a first call)
    N.Device.synchronize()
    hip = C.CDLL(lib._name)                                # (the runtime that the library is linked with)
    stream, graph, replayable = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    captured = call(C.byref(req), stream, C.byref(err))
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and captured == 0
    assert hip.hipGraphInstantiate(C.byref(replayable), graph, None, None, C.c_size_t(0)) == 0
    rng = np.random.default_rng(heads)
    for replay in range(12):
        c["qkv"] = (rng.normal(0, 1, c["qkv"].size) * (1 + replay)).astype(np.float32)
        ref, _, _ = _attention_oracle(c)
        qkv.upload(c["qkv"])
        if replay % 4 == 3:
            assert call(C.byref(req), None, C.byref(err)) == 0
            N.Device.synchronize()
        assert hip.hipGraphLaunch(replayable, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
        assert rel_l2(out32.numpy(np.float32), ref) <= REL_L2, replay
    assert N.paged_attention_status(ws, heads, hd) == (0, 0)
    assert hip.hipGraphExecDestroy(replayable) == 0 and hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
