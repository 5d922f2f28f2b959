"""Prompt blocks, batch steps and the decode attention at widths, head sizes and numbers of query heads a key head outside
the power-of-two ones: against the oracle where an operator can be called alone, else against the same session walking
token by token (whose kernels the other files hold to the oracle)."""
import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from nerva_amd.runtime import attention_workspace
from test_gpu_ops import _attention_case, _attention_device, _attention_oracle, dev
from test_gpu_session import BF16, E2E_REL_L2, F16, REL_L2, random_model, rel_l2, started

pytestmark = pytest.mark.gpu

# dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias
WIDTHS = [
    (BF16, 416, 6, 2, 128, 608, 517, 2, 1e6, True, False),     # K an odd multiple of 32: blocks of 128 rows only; 3 heads a key head
    (F16, 192, 10, 2, 64, 320, 301, 3, 1e4, False, True),      # heads of 64, 5 a key head; K of 3 and 5 blocks of 64
    (BF16, 1344, 14, 2, 64, 2112, 1003, 2, 1e6, True, True),   # heads of 64, 7 a key head; 21 and 33 blocks of 64, ragged row groups
    (BF16, 1536, 12, 2, 128, 2944, 801, 2, 1e6, False, True),  # 6 heads a key head; a gate/up pair that is no multiple of 128
    (F16, 640, 5, 5, 128, 1728, 402, 2, 1e4, True, False),     # a key head each
]


@pytest.mark.parametrize("heads,kv_heads,hd,dtype,theta,qk_norm,bias", [
    (6, 2, 128, BF16, 1e6, True, False), (20, 4, 128, F16, 1e4, False, True), (12, 2, 128, BF16, 0, True, True),
    (28, 4, 128, BF16, 1e6, False, True), (8, 8, 64, F16, 1e4, True, False), (32, 8, 64, BF16, 5e5, False, False),
    (14, 2, 64, BF16, 1e6, True, True), (16, 2, 64, F16, 0, False, False)])
def test_step_attention_of_any_group_and_head(heads, kv_heads, hd, dtype, theta, qk_norm, bias):
    """Edges of the 16-token tiles, one split and many, more tiles a wave than it requests ahead (few forced splits)."""
    for tokens, splits in ((0, 0), (15, 0), (16, 0), (70, 0), (1000, 0), (2500, 2)):
        c = _attention_case(dtype, heads, kv_heads, hd, tokens, theta, qk_norm, heads * 7 + tokens, bias=bias)
        ref, k16, v16 = _attention_oracle(c)
        if splits == 0:
            got32, got16, k_new, v_new, _, _ = _attention_device(c)
            assert np.max(np.abs(k_new.astype(np.int32) - k16.astype(np.int32))) <= 1
            assert np.array_equal(v_new, v16)
            assert np.array_equal(got16, O.encode16(dtype, got32))
        else:
            cache = N.PagedKvCache(c["layers"], c["n_blocks"], kv_heads, hd, c["table"])
            cache.fill(c["layer"], c["k_rows"], c["v_rows"])
            out16, out32 = N.DeviceBuffer(heads * hd * 2), N.DeviceBuffer(heads * hd * 4)
            opt = lambda a: dev(a) if a is not None else None   # noqa: E731
            qb, kb, vb = (opt(b) for b in c["biases"])
            N.paged_attention(dtype, heads, kv_heads, hd, cache, c["layer"], tokens, dev(c["qkv"]), attention_workspace(heads, hd), out16,
                              out_f32=out32, append=True, rope_theta=theta, q_norm=opt(c["qn"]), k_norm=opt(c["kn"]), q_bias=qb,
                              k_bias=kb, v_bias=vb, splits=splits)
            got32 = out32.numpy(np.float32)
        assert rel_l2(got32, ref) <= REL_L2, (tokens, splits)


def test_more_splits_than_stay_resident_still_run_where_they_did():
    """Heads of 64 took any split factor (their kernel had no splits); they still do."""
    c = _attention_case(BF16, 16, 8, 64, 1100, 1e6, True, 3)
    ref, _, _ = _attention_oracle(c)
    cache = N.PagedKvCache(c["layers"], c["n_blocks"], 8, 64, c["table"])
    cache.fill(c["layer"], c["k_rows"], c["v_rows"])
    out16, out32 = N.DeviceBuffer(16 * 64 * 2), N.DeviceBuffer(16 * 64 * 4)
    N.paged_attention(BF16, 16, 8, 64, cache, c["layer"], 1100, dev(c["qkv"]), attention_workspace(16, 64), out16, out_f32=out32,
                      append=True, rope_theta=1e6, q_norm=dev(c["qn"]), k_norm=dev(c["kn"]), splits=64)
    assert rel_l2(out32.numpy(np.float32), ref) <= REL_L2


def walked(weights, max_ctx):
    N.Device.set_tuning("prefill_walk", 1)
    try:
        return N.DecodeSession.create(weights, max_ctx)
    finally:
        N.Device.set_tuning("prefill_walk", 0)


@pytest.mark.parametrize("geom", WIDTHS)
def test_prompt_blocks_match_the_token_walk(geom):
    """Prompts that end in a block of 1 token, just past 32, 64, 128 and 256 rows, and in the second block of 512."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = geom
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, hidden, theta, qk_norm, bias)
    s, walk = N.DecodeSession.create(weights, 704), walked(weights, 704)
    assert s.create_result.prefill_chunk_tokens == (512 if hidden % 64 == 0 and inter % 64 == 0 else 128)
    assert walk.create_result.prefill_chunk_tokens == 1
    rng = np.random.default_rng(hidden)
    for n in (2, 3, 34, 66, 130, 258, 300, 515, 640):
        prompt = rng.integers(0, vocab, n).astype(np.uint32)
        for session in (s, walk):
            rc, res = session.start(prompt)
            assert rc == 0 and res.hot_path_allocations == 0
        assert rel_l2(s.logits(), walk.logits()) <= E2E_REL_L2, n
        for layer in range(layers):
            for got, want in zip(s.kv_range(layer, 0, n), walk.kv_range(layer, 0, n)):
                tol = 2e-3 if layer == 0 else E2E_REL_L2
                assert rel_l2(O.decode16(dtype, got), O.decode16(dtype, want)) <= tol, (n, layer)
    for session in (s, walk):
        session.destroy()


@pytest.mark.parametrize("geom", [WIDTHS[2], WIDTHS[3], (F16, 2048, 16, 4, 128, 4096, 1000, 2, 1e6, True, False)])
def test_passes_of_several_blocks_match_single_blocks(geom):
    """A pass takes the projections of several blocks of 512 together: one row into the second, an edge of 256, the largest
    pass (4096) and one row, and a block, past it; in a prompt that starts behind another (not at a block's edge)."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = geom
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, hidden, theta, qk_norm, bias)
    s = N.DecodeSession.create(weights, 4800)
    N.Device.set_tuning("prefill_block_tokens", 512)
    try:
        single = N.DecodeSession.create(weights, 4800)
    finally:
        N.Device.set_tuning("prefill_block_tokens", 0)
    assert s.create_result.prefill_chunk_tokens == single.create_result.prefill_chunk_tokens == 512
    rng = np.random.default_rng(hidden)
    for n in (513, 769, 1024, 1500, 4097, 4650):
        prompt = rng.integers(0, vocab, n).astype(np.uint32)
        for session in (s, single):
            rc, res = session.start(prompt)
            assert rc == 0 and res.hot_path_allocations == 0
        assert rel_l2(s.logits(), single.logits()) <= E2E_REL_L2, n
        for layer in range(layers):
            for got, want in zip(s.kv_range(layer, 0, n), single.kv_range(layer, 0, n)):
                tol = 2e-3 if layer == 0 else E2E_REL_L2
                assert rel_l2(O.decode16(dtype, got), O.decode16(dtype, want)) <= tol, (n, layer)
    places = [0, 511, 600, 601, 602, 1088]
    head, more = rng.integers(0, vocab, 77).astype(np.uint32), rng.integers(0, vocab, 1089).astype(np.uint32)
    rows = []
    for session in (s, single):
        session.start(head)
        rc, _, logits, _ = session.extend(more, places)
        assert rc == 0
        rows.append(logits)
    assert rel_l2(rows[0], rows[1]) <= E2E_REL_L2
    for session in (s, single):
        session.destroy()


@pytest.mark.parametrize("geom,count", [(WIDTHS[2], 2), (WIDTHS[2], 17), (WIDTHS[3], 5), (WIDTHS[3], 32), (WIDTHS[4], 3)])
def test_batch_steps_match_sequences_alone(geom, count):
    """The rows every sequence appends in batch steps are those it appends alone on the same history."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = geom
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, count, theta, qk_norm, bias)
    parent = N.DecodeSession.create(weights, 96, plan=N.WeightPlan.from_weights(weights))
    sessions = [parent] + [parent.fork_shared_weights() for _ in range(count - 1)]
    assert parent.shares_weight_stream()
    rng = np.random.default_rng(count)
    prompts = [rng.integers(0, vocab, 1 + (11 * i) % 50).astype(np.uint32) for i in range(count)]
    streams = [[started(s, p)] for s, p in zip(sessions, prompts)]
    for _ in range(3):
        rc, res, tokens = N.DecodeSession.batch_advance_one(sessions, 32, 2)
        assert rc == 0 and res.block_tokens == count and res.hot_path_allocations == 0
        for stream, token in zip(streams, tokens):
            stream.append(int(token))
    solo = parent.fork_shared_weights()
    for i in sorted({0, 1, count // 2, count - 1}):
        assert solo.release_sequence() == 0
        rc, _, _, _ = solo.extend(prompts[i])
        assert rc == 0
        for token in streams[i][:-1]:       # the same history, one step at a time
            rc, _, logits, _ = solo.extend([token], [0])
            assert rc == 0
        top = np.sort(logits[0])
        assert streams[i][-1] == int(np.argmax(logits[0])) or top[-1] - top[-2] <= E2E_REL_L2 * np.max(np.abs(logits))
        at = len(prompts[i])
        for layer in range(layers):
            for got, want in zip(sessions[i].kv_range(layer, at, 3), solo.kv_range(layer, at, 3)):
                tol = 2e-3 if layer == 0 else E2E_REL_L2
                assert rel_l2(O.decode16(dtype, got), O.decode16(dtype, want)) <= tol, (i, layer)
    solo.destroy()
    for s in sessions[::-1]:
        s.destroy()


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("rows,cols", [(3073, 1088),     # one cache line into the second batch
                                       (2050, 1984), (5003, 3584), (1027, 9728),
                                       (50000, 64),      # rows shorter than one request
                                       (700, 12224),     # the widest an f32 input is kept for
                                       (133, 30656)])    # the widest a 16-bit one is
def test_lean_gemv_of_ragged_rows(dtype, rows, cols):
    """Rows that are no whole number of batches, in all forms: what lies behind a row's end is the next row (or, behind the
    last, nothing), so a lane too many shows. The activations of the general kernel, whose oracle is the same."""
    rng = np.random.default_rng(rows + cols)
    seed = rows * 131 + cols
    w = O.synth_16(dtype, seed, 1, rows * cols, 0.0, 0.02).reshape(rows, cols)
    dw = dev(w)
    x16 = O.encode16(dtype, rng.normal(0, 1, cols).astype(np.float32))
    res = rng.normal(0, 1, rows).astype(np.float32)
    bias = O.encode16(dtype, rng.normal(0, 1, rows).astype(np.float32))
    y, y16 = N.DeviceBuffer(rows * 4), N.DeviceBuffer(rows * 2 + 16)
    kernel = lambda prologue, epilogue, n: N.gemv_launch_shape(prologue, epilogue, n, cols)[0]   # noqa: E731
    assert kernel(0, 1, rows) == 3
    N.gemv(dtype, dw, rows, cols, input16=dev(x16), residual=dev(res), out_f32=y, epilogue=1)
    assert rel_l2(y.numpy(np.float32), O.gemv_x16(dtype, w, x16) + res) <= REL_L2
    if cols > 12288:
        return
    h = rng.normal(0, 1, cols).astype(np.float32)
    gamma = O.encode16(dtype, rng.normal(1, 0.02, cols))
    n16 = O.encode16(dtype, O.rms_norm(dtype, h, gamma, 1e-6))
    ref = O.gemv_x16(dtype, w, n16)
    N.gemv(dtype, dw, rows, cols, input_f32=dev(h), gamma=dev(gamma), eps=1e-6, bias=dev(bias), out_f32=y)
    got = y.numpy(np.float32).copy()
    assert rel_l2(got, ref + O.decode16(dtype, bias)) <= REL_L2
    N.gemv(dtype, dw, rows, cols, input_f32=dev(h), gamma=dev(gamma), eps=1e-6, bias=dev(bias), out16=y16, epilogue=3)
    assert np.array_equal(y16.numpy(np.uint16, rows), O.encode16(dtype, got))
    pairs = rows // 2
    if 2 * pairs * cols >= 3 << 20:
        assert kernel(1, 2, pairs) == 3
    g, u = ref[:pairs], ref[pairs:2 * pairs]
    ff = (g / (1.0 + np.exp(-g.astype(np.float64)))).astype(np.float32) * u
    N.gemv(dtype, dw, pairs, cols, input_f32=dev(h), gamma=dev(gamma), eps=1e-6, out16=y16, epilogue=2)
    assert rel_l2(O.decode16(dtype, y16.numpy(np.uint16, pairs)), O.decode16(dtype, O.encode16(dtype, ff))) <= 4e-3   # one 16-bit rounding


@pytest.mark.parametrize("hidden,vocab", [(576, 20011), (1344, 40001), (704, 517)])
def test_ragged_head_takes_the_largest(hidden, vocab):
    """The head of a width off the 1024 grid, in workgroups of 4 and of 16 waves: every logit is the oracle's (one layer, one
    token: one bf16 flip, as in the single-layer test), the token is the first of the largest."""
    weights, omodel = random_model(BF16, hidden, hidden // 64, hidden // 64, 64, 320, vocab, 1, hidden, 1e4, False, False)
    s = N.DecodeSession.create(weights, 32)
    ctx = O.Context(omodel, 32, staging=1)
    ctx.forward_token(3, prompt_token=True, want_logits=True)
    rc, _ = s.start([3])
    assert rc == 0
    logits = s.logits()
    assert np.max(np.abs(logits - ctx.logits())) <= 6e-3 * np.max(np.abs(logits)) and rel_l2(logits, ctx.logits()) <= 6e-3
    rc, _, tokens = s.advance(1)
    assert rc == 0 and tokens[0] == np.argmax(logits)


@pytest.mark.parametrize("sizes", [[1400], [513, 300, 1, 586]], ids=str)
def test_stack_blocks_of_widths_off_the_power_of_two_grid(sizes):
    """Projections of a mixed stack in operand order at K of 3, 5 and 32 blocks of 64, in blocks past 512 token rows (with a
    scan in several launches), whole and in portions, as the oracle has them."""
    import stack_models as M
    import test_gpu_mixed_stack as T
    cfg = M.config([M.attention(16, 4, 128, 128, rot=32, chunk=700, ff=320), M.mingru(width=320, ff=448), M.mingru(width=64, ff=0)],
                   width=192, vocab=300)
    T.check(cfg, M.weights(cfg, seed=31), T.tokens_of(cfg, 1400, seed=9), sizes, 0)


@pytest.mark.parametrize("n,kind", [(151937, "sorted"), (65601, "one run"), (40000, "equal"), (2112, "lowest"), (151936, "spread")])
def test_top_k_collects_from_the_runs_that_hold_candidates(n, kind):
    """Logits placed so that all candidates share a chunk, a run of 64, the end of the vocabulary, or tie (more of them than
    are collected: the general selection), and with the type's lowest number as a logit like any other."""
    from nerva_amd import abi
    rng = np.random.default_rng(n)
    l = rng.standard_normal(n).astype(np.float32)
    if kind == "sorted":
        l.sort()
    elif kind == "one run":
        l[n - 70:] += 50.0
    elif kind == "equal":
        l[:] = 1.5
    elif kind == "lowest":
        l[:] = -np.finfo(np.float32).max
        l[[3, 64, n - 1]] = [1.0, 2.0, 3.0]
    buf, ws = dev(l), N.DeviceBuffer.zeros(abi.load().nerva_hip_sample_workspace_bytes(n))
    close = 0
    for top_k in (1, 2, 40, 127, 128, 0):
        for position in range(4):
            want, margin = O.sample(l, 0.9, 0.97, top_k, 11, position)
            got = N.sample(buf, n, 0.9, 0.97, top_k, 11, position, ws)
            if got != want:   # (a draw within rounding of a boundary, as in the rule's own test)
                assert margin < 1e-5, (top_k, position, got, want, margin)
                close += 1
    assert close <= 1


@pytest.mark.parametrize("geom,lengths", [
    ((BF16, 512, 40, 8, 64, 512, 301, 2), (1601, 3333)),    # 272 and 560 workgroups
    ((F16, 512, 48, 16, 64, 512, 301, 2), (1600, 2903)),    # 320 and 592
    ((F16, 512, 32, 8, 128, 512, 301, 2), (2501, 4096)),    # 320 and 512
    ((BF16, 512, 28, 4, 128, 512, 301, 2), (1999, 3001)),   # 252 and 376
])
def test_passes_through_one_attention_launch(geom, lengths):
    """Passes whose attention takes all its blocks in one launch without splits - in each branch of the rule that says so - with
    a ragged last group of tokens, from the start and behind 77 tokens, against passes of one block. That the launch is taken
    shows in their number: the same as for a prompt of one block."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers = geom
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, hidden, 1e5, True, False)
    s = N.DecodeSession.create(weights, 4200)
    N.Device.set_tuning("prefill_block_tokens", 512)
    try:
        single = N.DecodeSession.create(weights, 4200)
    finally:
        N.Device.set_tuning("prefill_block_tokens", 0)
    rng = np.random.default_rng(hidden)
    for prefix in (0, 77):
        for n in lengths:
            tokens = rng.integers(0, vocab, prefix + n).astype(np.uint32)

            def prompt(session, count):
                assert session.release_sequence() == 0
                if prefix:
                    assert session.extend(tokens[:prefix])[0] == 0
                rc, res, _, _ = session.extend(tokens[prefix:prefix + count])
                assert rc == 0
                return res.kernel_launches

            assert prompt(s, n) == prompt(s, 500) < prompt(single, n)
            prompt(s, n)
            assert rel_l2(s.logits(), single.logits()) <= E2E_REL_L2, (prefix, n)
            for layer in range(layers):
                for got, want in zip(s.kv_range(layer, 0, prefix + n), single.kv_range(layer, 0, prefix + n)):
                    tol = 2e-3 if layer == 0 else E2E_REL_L2
                    assert rel_l2(O.decode16(dtype, got), O.decode16(dtype, want)) <= tol, (prefix, n, layer)
    for session in (s, single):
        session.destroy()


@pytest.mark.parametrize("vocab", [98305, 98306, 100003])
def test_wanted_logits_of_a_large_vocabulary_of_any_size(vocab):
    """From 98304 rows on a head takes two row tiles a wave; a vocabulary that is no multiple of 4 stores its logits one by
    one. Rows side by side against each of them alone, through the head of a step."""
    weights, _ = random_model(BF16, 192, 6, 2, 64, 320, vocab, 1, 5, 1e4, False, False)
    s = N.DecodeSession.create(weights, 64)
    tokens = np.random.default_rng(vocab).integers(0, vocab, 40).astype(np.uint32)
    rc, _, rows, _ = s.extend(tokens, range(40))
    assert rc == 0
    for place in (0, 1, 31, 32, 38, 39):
        assert s.release_sequence() == 0
        rc, _, alone, _ = s.extend(tokens[:place + 1], [place])
        assert rc == 0
        assert rel_l2(rows[place], alone[0]) <= E2E_REL_L2 and np.max(np.abs(rows[place] - alone[0])) <= E2E_REL_L2 * np.max(np.abs(alone[0]))
    s.destroy()


def test_a_merge_that_gives_up_behind_a_prompt_in_blocks():
    """The step-fault hook set once the prompt is in: its last token came with its block, so the first step that fails is the
    one behind it - of heads of 64, five a key head, where few workgroups merge."""
    weights, _ = random_model(F16, 640, 10, 2, 64, 1280, 301, 2, 9, 1e4, False, False)
    s = N.DecodeSession.create(weights, 720)
    prompt = np.random.default_rng(9).integers(0, 301, 700).astype(np.uint32)
    assert s.start(prompt)[0] == 0
    N.Device.set_tuning("attn_merge_spin_limit", 4)
    N.Device.set_tuning("attn_withhold_split", 1 + 3)
    try:
        rc, res, tokens = s.advance(6)
    finally:
        N.Device.set_tuning("attn_merge_spin_limit", 0)
        N.Device.set_tuning("attn_withhold_split", 0)
    from nerva_amd import abi
    assert rc == -1 and res.hip_error == abi.NERVA_HIP_ERROR_STEP_FAULT
    slots = s.slots(len(prompt) - 1, 2).view(np.uint32).reshape(2, -1)
    assert slots[0, 8] != abi.NERVA_HIP_SLOT_DEVICE_FAULT and slots[1, 8] == abi.NERVA_HIP_SLOT_DEVICE_FAULT
    s.destroy()


def test_stack_passes_past_4096_tokens():
    """The largest pass of a mixed stack and some tokens behind it, through chunks of keys that start inside the pass and a
    layer that sees everything, against the same tokens in portions of a block (which the tests of stacks hold to the oracle)."""
    import stack_models as M
    cfg = M.config([M.attention(16, 4, 128, 128, rot=32, chunk=700, ff=320), M.mingru(width=320, ff=448), M.attention(8, 2, 64, 64, rot=16, chunk=5000, ff=0)],
                   width=192, vocab=300)
    tensors, tokens = M.weights(cfg, seed=33), np.random.default_rng(4).integers(0, 300, 4500).astype(np.uint32)
    rows = []
    for sizes in ([4500], [512]):
        s = M.session(cfg, tensors, 4600)
        rows.append(M.feed(s, tokens, sizes))
        s.destroy()
    worst = M.errors(rows[0], rows[1])
    assert worst.max() < 0.05, "position %d: %.2e" % (int(worst.argmax()), worst.max())   # (the bound of 16-bit stacks)
