"""Decode steps of wider models whose layers run in one launch of a workgroup a CU, against the oracle and against the launches they stand in for."""
import threading
import time

import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from nerva_amd import abi
from oracle.links import chain_budget, run_traced_stream
from test_gpu_session import BF16, F16, random_model, rel_l2

pytestmark = pytest.mark.gpu

# dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias: rows of whole and of part requests, rows in one, two, four and eight parts, shares
# that do not go round, one to eight query heads a key head of both sizes, rows of one to eight pairs a thread, inputs smaller and larger than the attention's place
SHAPES = [
    (BF16, 1024, 16, 8, 128, 2816, 301, 4, 1e6, True, False),
    (F16, 1000, 9, 3, 128, 3608, 301, 4, 1e4, False, True),
    (BF16, 264, 4, 4, 64, 7704, 301, 4, 1e6, True, True),
    (F16, 2568, 7, 1, 64, 1032, 301, 4, 0, True, False),
    (BF16, 512, 64, 8, 128, 520, 301, 4, 1e6, False, False),
    (BF16, 2048, 16, 2, 64, 1800, 301, 5, 5e5, True, False),
    (F16, 5128, 2, 2, 128, 520, 301, 4, 1e6, False, True),       # (in bf16 its launches are 2.7e-2 from the oracle after ten steps, too)
    (F16, 256, 10, 2, 64, 12288, 301, 4, 1e4, True, False),
    (F16, 5120, 5, 1, 128, 520, 301, 4, 1e6, True, False),       # (five pairs a thread; five and seven query heads a key head of 128)
    (F16, 3584, 7, 1, 128, 1032, 301, 4, 1e6, False, True),
]


@pytest.mark.parametrize("shape", SHAPES)
def test_every_link_of_a_step_in_one_launch_matches_the_oracle(shape):
    """Each vector that a layer hands on, at 1e-3 of the oracle's operator on the device's own input, and the stream's logits within the
    budget of the chain; the same stream from one call. Positions cross a cache block."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, model = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, hidden, theta, qk_norm, bias)
    prompt = np.random.default_rng(1).integers(0, vocab, 11).astype(np.uint32)
    s = N.DecodeSession.create(weights, 64)
    tokens, worst, e2e = run_traced_stream(s, model, prompt, 10, 64)
    assert s.start(prompt)[0] == 0
    rc, res, again = s.advance(10)
    assert rc == 0 and res.graph_nodes == 3 and res.graph_replays == 9 and again.tolist() == tokens
    s.destroy()
    print(sorted(worst.items()), e2e, flush=True)


@pytest.mark.parametrize("shape", SHAPES[:6] + [(dtype,) + shape[1:] for shape in SHAPES[8:] for dtype in (BF16, F16)])
def test_longer_contexts_in_one_launch_give_what_launches_give(shape):
    """Contexts of one split, of the first several, of as many as there are and of several blocks a wave, behind prompts that both kinds of session
    have read alike: logits and cache rows of the steps. Only roundings of 16-bit values that lie on a boundary may fall differently."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 7, theta, qk_norm, bias)
    rng = np.random.default_rng(3)
    results = []
    lengths = (30, 125, 130, 255, 1100, 4500)
    prompts = [rng.integers(0, vocab, n).astype(np.uint32) for n in lengths]
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create(weights, 4600)
            out = []
            for prompt in prompts:
                assert s.start(prompt)[0] == 0
                assert s.advance(1)[0] == 0
                for step in range(3):
                    rc, res = s.extend(prompt[step:step + 1])[:2]     # the same tokens whatever the logits say
                    assert rc == 0 and res.kernel_launches == (3 if mode == 0 else 3 + 5 * layers)
                out.append((s.logits(), s.kv_range(layers - 1, len(prompt), 3)))
            results.append(out)
            s.destroy()
    finally:
        N.Device.reset_tuning()
    for n, (want, want_rows), (got, got_rows) in zip(lengths, *results):
        assert np.all(np.isfinite(got)) and rel_l2(got, want) <= chain_budget(layers), (n, rel_l2(got, want))
        for a, b in zip(want_rows, got_rows):
            assert rel_l2(O.decode16(dtype, b), O.decode16(dtype, a)) <= chain_budget(layers), n


@pytest.mark.parametrize("dtype,hidden,heads,kv,hd,inter,context", [(BF16, 1024, 16, 8, 128, 4096, 32768), (F16, 1024, 16, 8, 64, 4096, 32768), (BF16, 1024, 8, 1, 128, 4096, 8192),
                                                                    (F16, 1280, 20, 4, 64, 5120, 8192)])
def test_the_longest_contexts_in_one_launch_and_the_first_behind_them(dtype, hidden, heads, kv, hd, inter, context):
    """As many blocks a wave as there can be: the logits of the steps of the last positions that one launch takes, against launches; and one call across the line, in sixes, singly and launch by
    launch, against calls of one step."""
    layers, vocab = 4, 301
    cfg = dict(dtype=dtype, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, intermediate=inter, vocab=vocab, layers=layers, rms_eps=1e-6, rope_theta=1e6)
    prompt = np.random.default_rng(3).integers(0, vocab, context - 40).astype(np.uint32)
    rows = []
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create_synthetic(cfg, context + 64)
            assert s.start(prompt[:-2])[0] == 0
            for token in prompt[-2:]:
                rc, res, logits, _ = s.extend([token], [0])
                assert rc == 0 and res.graph_nodes == (3 if mode == 0 else 3 + 5 * layers)
            rows.append(logits[0])
            if mode == 2:
                s.destroy()
    finally:
        N.Device.reset_tuning()
    assert np.all(np.isfinite(rows[1])) and rel_l2(rows[1], rows[0]) <= chain_budget(layers)
    assert s.start(prompt)[0] == 0
    single = [s.advance(1) for _ in range(61)]
    assert [res.graph_nodes for _, res, _ in single[1:]] == [3] * 40 + [3 + 5 * layers] * 20
    want, logits = [int(tokens[0]) for _, _, tokens in single], s.logits()
    assert s.start(prompt)[0] == 0
    rc, res, tokens = s.advance(61)
    assert rc == 0 and res.graph_replays == 60 and res.graph_launches == 6 + 4 + 20
    assert tokens.tolist() == want and np.array_equal(s.logits(), logits)
    s.destroy()


def test_wide_steps_that_give_up_are_taken_again():
    """A workgroup that stays away twice at every position: the other waits end, the step is void and taken again, and the tokens are those of a session
    where nobody does; one that stays away for good is a step fault."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[0]
    cfg = dict(dtype=dtype, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, intermediate=inter, vocab=vocab, layers=layers, rms_eps=1e-6, rope_theta=theta)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).astype(np.uint32)
    s = N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7, weight_std=0.05)
    assert s.start(prompt)[0] == 0
    rc, res, want = s.advance(8)
    assert rc == 0 and res.graph_replays == 7
    s.destroy()
    try:
        N.Device.set_tuning("attn_merge_spin_limit", 1000)
        N.Device.set_tuning("step_chain_withhold", 2)
        s = N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7, weight_std=0.05)
        assert s.start(prompt)[0] == 0
        rc, res, got = s.advance(8)
        assert rc == 0 and res.graph_replays == 3 * 7 and got.tolist() == want.tolist()
        s.destroy()
        N.Device.set_tuning("attn_merge_spin_limit", 20)
        N.Device.set_tuning("step_chain_withhold", 100000)
        s = N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7, weight_std=0.05)
        assert s.start(prompt)[0] == 0
        rc, res, got = s.advance(3)
        assert rc == -1 and res.hip_error == abi.NERVA_HIP_ERROR_STEP_FAULT
        s.destroy()
    finally:
        N.Device.reset_tuning()


@pytest.mark.parametrize("shape", [SHAPES[0], (BF16, 256, 2, 2, 128, 512, 301, 4, 1e6, True, True)], ids=["wide", "narrow"])
def test_steps_that_never_find_their_places_go_launch_by_launch(shape):
    """Waits that run out at once, as where somebody else keeps the places for good: after some of them a call goes on in launches, whichever call it is, and gives what launches give."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).astype(np.uint32)
    sampler = abi.NervaHipHfDecodeSamplerConfig()
    sampler.temperature, sampler.top_p, sampler.top_k, sampler.seed = 0.9, 0.95, 0, 11

    def calls(s, mode):
        out = []
        assert s.start(prompt)[0] == 0
        for n in (1, 2, 40):
            rc, res, tokens = s.advance(n)
            assert rc == 0 and (n == 1 or res.graph_nodes == 3 + 5 * layers)
            out.append(tokens)
        out.append(s.logits())
        s.destroy()
        s = fresh(mode)
        assert s.start(prompt, eos=vocab - 1, sampler=sampler)[0] == 0
        rc, res, tokens = s.advance(20)
        assert rc == 0
        out.append(tokens)
        s.destroy()
        s = fresh(mode)
        rc, res, tokens = s.run(prompt, 30)
        assert rc == 0
        out.append(tokens)
        s.destroy()
        s = fresh(mode)
        assert s.extend(prompt)[0] == 0
        rc, res, rows, _ = s.extend([3], [0])
        assert rc == 0
        out.append(rows)
        s.destroy()
        s = fresh(mode)
        assert s.start(prompt)[0] == 0 and s.advance(1)[0] == 0
        rc, res, token, trace = s.traced_advance()
        assert rc == 0
        out += [token, trace["logits"]]
        s.destroy()
        return out

    def fresh(mode):
        N.Device.set_tuning("step_chain", mode)
        N.Device.set_tuning("attn_merge_spin_limit", 1)       # (contexts of one split: the attention launches wait for nothing)
        return N.DecodeSession.create(weights, 64)
    try:
        got, want = (calls(fresh(mode), mode) for mode in (1, 2))
    finally:
        N.Device.reset_tuning()
    for i, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a, b), i


def test_sessions_of_wide_and_narrow_models_take_turns():
    """Six sessions of a wide model and two of a narrow one, more than there are hardware queues, from threads of their own: each gives what it gives alone, in the same
    launches, and all of them together take no longer than one after the other (a step in front of the one that it waits for would stand still for as long as the waits' limits)."""
    wide = (BF16, 1024, 16, 8, 128, 2816, 301, 4, 1e6, True, False)
    narrow = (BF16, 512, 4, 2, 128, 1024, 301, 6, 1e6, True, False)
    rng = np.random.default_rng(8)
    prompts = [rng.integers(0, 301, n).astype(np.uint32) for n in (20, 300, 900, 150, 9, 40, 500, 70)]
    weights = [random_model(*g[:8], 3, *g[8:])[0] for g in (wide, narrow)]
    first = N.DecodeSession.create(weights[0], 1300)

    def all_steps(s, prompt, out):
        rc = s.start(prompt)[0]
        for _ in range(15):
            if rc == 0:
                rc, res, tokens = s.advance(10)
                out.append((rc, tokens.tolist()))
                out.append(res.graph_nodes)
        out.append(rc)

    lone = []
    all_steps(first, prompts[0], lone)
    assert lone[-1] == 0 and lone[1] == 3
    thin = N.DecodeSession.create(weights[1], 1300)
    sessions = [first] + [first.fork_shared_weights() for _ in range(5)] + [thin, thin.fork_shared_weights()]
    alone = [[] for _ in sessions]
    for s, prompt, out in zip(sessions, prompts, alone):
        all_steps(s, prompt, [])                                          # (its graphs are there)
    begin = time.perf_counter()
    for s, prompt, out in zip(sessions, prompts, alone):
        all_steps(s, prompt, out)
    in_turn = time.perf_counter() - begin
    together = [[] for _ in sessions]
    begin = time.perf_counter()
    threads = [threading.Thread(target=all_steps, args=a) for a in zip(sessions, prompts, together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    taken = time.perf_counter() - begin
    print("one after the other %.1f ms, together %.1f" % (in_turn * 1e3, taken * 1e3), flush=True)
    assert all(out[-1] == 0 for out in alone + together)
    assert together == alone
    assert all(nodes == 3 for out in alone for nodes in out[1:-1:2])
    assert alone[0] == lone
    assert taken < 3 * in_turn
    for s in sessions[:0:-1]:
        s.destroy()
    again = []
    all_steps(first, prompts[0], again)
    assert again == lone
    first.destroy()


@pytest.mark.parametrize("layers,hidden,heads,kv,hd,inter", [(1, 4096, 32, 8, 128, 10008), (2, 2048, 16, 8, 128, 4360), (3, 2056, 6, 2, 64, 5608)])
def test_models_of_few_layers(layers, hidden, heads, kv, hd, inter):
    """One to three layers, the first and the last of a launch among them: the logits of a step behind a prompt that both kinds of session have read alike, at contexts of one split and
    of several, within the budget of the chain."""
    cfg = dict(dtype=BF16, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, intermediate=inter, vocab=301, layers=layers, rms_eps=1e-6, rope_theta=1e6)
    results = []
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create_synthetic(cfg, 400)
            out = []
            for n in (9, 300):
                assert s.start(np.arange(n, dtype=np.uint32) % 301)[0] == 0
                rc, res, _ = s.advance(2)
                assert rc == 0 and res.graph_nodes == (3 if mode == 0 else 3 + 5 * layers)
                out.append(s.logits())
            results.append(out)
            s.destroy()
    finally:
        N.Device.reset_tuning()
    for launches, one in zip(*results):
        assert rel_l2(one, launches) <= chain_budget(layers)
