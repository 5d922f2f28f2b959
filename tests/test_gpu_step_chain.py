"""Decode steps of narrow models whose layers run in one launch, against the oracle and against the launches they stand in for."""
import threading

import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from nerva_amd import abi
from oracle.links import chain_budget, run_traced_stream
from test_gpu_session import BF16, F16, random_model, rel_l2

pytestmark = pytest.mark.gpu

# dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias: widths of whole and of part columns a request, one to
# eight query heads a key head (three, five and seven among them) of both sizes, units that do not go round evenly, the largest of everything
SHAPES = [
    (F16, 512, 8, 4, 64, 1376, 803, 4, 1e4, False, False),
    (BF16, 256, 2, 2, 128, 512, 301, 4, 1e6, True, True),
    (BF16, 520, 3, 1, 128, 1000, 301, 4, 0, True, False),
    (F16, 640, 10, 2, 64, 2056, 301, 5, 1e4, False, True),
    (BF16, 1024, 4, 2, 128, 1024, 511, 4, 1e6, True, False),
    (F16, 1016, 7, 1, 128, 776, 301, 4, 1e6, False, False),
    (BF16, 256, 32, 4, 128, 3000, 301, 4, 1e6, True, True),
    (F16, 264, 20, 20, 64, 4096, 301, 4, 1e4, True, False),
    (BF16, 1024, 1, 1, 64, 776, 301, 4, 1e4, False, True),      # (fewer heads' rows than workgroups)
]


@pytest.mark.parametrize("shape", SHAPES)
def test_every_link_of_a_chained_step_matches_the_oracle(shape):
    """Each vector that a layer hands on, at 1e-3 of the oracle's operator on the device's own input, and the stream's logits within the
    budget of the chain; the same stream from one call. Positions cross a cache block."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, model = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, hidden, theta, qk_norm, bias)
    prompt = np.random.default_rng(1).integers(0, vocab, 11).astype(np.uint32)
    s = N.DecodeSession.create(weights, 64)
    tokens, worst, e2e = run_traced_stream(s, model, prompt, 12, 64)
    assert s.start(prompt)[0] == 0
    rc, res, again = s.advance(12)
    assert rc == 0 and res.graph_nodes == 3 and res.graph_replays == 11 and again.tolist() == tokens
    s.destroy()
    print(sorted(worst.items()), e2e, flush=True)


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[4], SHAPES[5], SHAPES[6], SHAPES[7]])
def test_a_chain_over_longer_contexts_gives_what_launches_give(shape):
    """Contexts of one split, of the first several and of as many as there are, behind prompts that both kinds of session have
    read alike: logits and cache rows of the steps. Only roundings of 16-bit values that lie on a boundary may fall differently."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 7, theta, qk_norm, bias)
    rng = np.random.default_rng(3)
    results = []
    lengths = (30, 125, 130, 255, 700, 1100)
    prompts = [rng.integers(0, vocab, n).astype(np.uint32) for n in lengths]
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create(weights, 1200)
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


def test_sampled_and_stopped_chains_and_forks():
    """The sampler behind a chain, a stop token, a fork of a running sequence and a second sequence on the same words."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[0]
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).astype(np.uint32)
    sampler = abi.NervaHipHfDecodeSamplerConfig()
    sampler.temperature, sampler.top_p, sampler.top_k, sampler.seed = 0.9, 0.95, 0, 11
    s = N.DecodeSession.create(weights, 64)
    assert s.start(prompt, sampler=sampler)[0] == 0
    rc, res, drawn = s.advance(16)
    assert rc == 0 and res.graph_nodes == 4
    assert s.start(prompt)[0] == 0
    rc, res, greedy = s.advance(6)
    assert rc == 0 and res.graph_nodes == 3
    fork = s.fork_shared_weights()
    rest = s.advance(8)[2].tolist()
    assert fork.advance(8)[2].tolist() == rest
    assert s.start(prompt, sampler=sampler)[0] == 0
    assert s.advance(16)[2].tolist() == drawn.tolist()
    stop = greedy.tolist() + rest
    last = next(i for i in range(2, 14) if stop[i] not in stop[:i])
    assert s.start(prompt, eos=stop[last])[0] == 0
    rc, res, stopped = s.advance(14)
    assert rc == 0 and stopped.tolist() == stop[:last + 1]
    fork.destroy()
    s.destroy()


def test_a_prompt_walked_by_chains_is_the_one_that_launches_walk():
    """run() takes a prompt's tokens step by step: the logits behind it, the tokens from them, the rows in the cache."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[0]
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.random.default_rng(2).integers(0, vocab, 37).astype(np.uint32)
    results = []
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create(weights, 64)
            rc, res, tokens = s.run(prompt, 1)
            logits = s.logits()
            assert rc == 0 and res.graph_replays == 37 and tokens.tolist() == [O.greedy_argmax(logits, skip_nonfinite=True)]
            results.append((logits, s.kv_range(layers - 1, 0, 37)))
            rc, res, more = s.run(prompt, 14)
            assert rc == 0 and len(more) == 14 and more[0] == tokens[0]
            s.destroy()
    finally:
        N.Device.reset_tuning()
    (want, want_rows), (got, got_rows) = results
    assert np.all(np.isfinite(got)) and rel_l2(got, want) <= chain_budget(layers)
    for a, b in zip(want_rows, got_rows):
        assert rel_l2(O.decode16(dtype, b), O.decode16(dtype, a)) <= chain_budget(layers)


@pytest.mark.parametrize("shape,line", [(SHAPES[0], 4096), (SHAPES[4], 2048)])
def test_a_sequence_that_leaves_the_chain_goes_on_with_launches(shape, line):
    """From some number of keys on a step is its launches again: one call across that line, the steps on either side of it against a session
    that has the launches throughout - the logits, the launches counted, the rows that the chain left in the cache - and a fork behind it."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 7, theta, qk_norm, bias)
    prompt = np.random.default_rng(3).integers(0, vocab, line - 5).astype(np.uint32)
    results = []
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create(weights, line + 32)
            assert s.start(prompt)[0] == 0
            rc, res, tokens = s.advance(12)     # the prompt's token and eleven steps, five of them in one launch
            assert rc == 0 and res.graph_replays == 11 and res.kernel_launches == (11 * (3 + 5 * layers) if mode == 2 else 5 * 3 + 6 * (3 + 5 * layers))
            fork = s.fork_shared_weights()
            assert fork.advance(4)[2].tolist() == s.advance(4)[2].tolist()
            fork.destroy()
            s.release_sequence()
            assert s.extend(prompt)[0] == 0
            rows = []
            for i, t in enumerate(prompt[:10]):               # the same tokens whatever the logits say
                rc, res, logits, _ = s.extend([t], [0])
                assert rc == 0 and res.kernel_launches == (3 if mode == 0 and i < 5 else 3 + 5 * layers)
                rows.append(logits[0])
            results.append((np.array(rows), s.kv_range(layers - 1, len(prompt), 10)))
            s.destroy()
    finally:
        N.Device.reset_tuning()
    (want, want_rows), (got, got_rows) = results
    assert np.all(np.isfinite(got))
    for i in range(10):
        assert rel_l2(got[i], want[i]) <= chain_budget(layers), i
    for a, b in zip(want_rows, got_rows):
        assert rel_l2(O.decode16(dtype, b), O.decode16(dtype, a)) <= chain_budget(layers)


def test_a_wait_that_runs_out_ends_the_sequence():
    """With a limit of one poll a chain's waits run out: every wait ends, the slot says so, advance returns the step fault; a
    sequence started afterwards is the healthy one."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[4]
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).astype(np.uint32)
    s = N.DecodeSession.create(weights, 64)
    assert s.start(prompt)[0] == 0
    want = s.advance(12)[2].tolist()
    fork = s.fork_shared_weights()
    N.Device.set_tuning("attn_merge_spin_limit", 1)
    try:
        assert fork.start(prompt)[0] == 0
        rc, res, tokens = fork.advance(3)         # (captured with the limit)
    finally:
        N.Device.reset_tuning()
    assert rc == -1 and res.hip_error == abi.NERVA_HIP_ERROR_STEP_FAULT
    fork.destroy()
    assert s.start(prompt)[0] == 0
    assert s.advance(12)[2].tolist() == want
    s.destroy()


@pytest.mark.parametrize("mode", [0, 2])
def test_a_batch_counts_the_launches_of_its_sequences_own_steps(mode):
    """Sequences of a narrow model step one by one: two projections each where the layers are one launch (that one and the head), else all there are."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[1]
    cfg = dict(dtype=dtype, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, intermediate=inter, vocab=vocab, layers=layers, rms_eps=1e-6, rope_theta=theta)
    try:
        N.Device.set_tuning("step_chain", mode)
        s = N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7, weight_std=0.05)
        sessions = [s] + [s.fork_shared_weights() for _ in range(2)]
    finally:
        N.Device.reset_tuning()
    for i, q in enumerate(sessions):
        assert q.start(np.arange(5 + i, dtype=np.uint32))[0] == 0 and q.advance(1)[0] == 0
    rc, res, tokens = N.DecodeSession.batch_advance_one(sessions, 3, 3)
    got = (res.pack_kernel_launches, res.projection_kernel_launches, res.dependency_kernel_launches, res.sampling_kernel_launches)
    assert rc == 0 and got == tuple(3 * n for n in ((0, 2, 0, 1) if mode == 0 else (1, 4 * layers + 1, layers, 1)))
    for q in sessions[::-1]:
        q.destroy()


# Polls that a wait is given where a test has many run out: an eighth of what it has, and far more than a healthy one takes
SHORT_WAIT = 2000


def test_steps_that_give_up_are_taken_again():
    """A workgroup that stays away twice at every position, as one that finds no place on a shared chip: the other waits end, the step is void and
    taken again, and every call gives what it gives without - advance, with a stop token too, run, extend with its logits, a traced step, a batch of
    sequences that step one by one, and the sampler."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[1]
    cfg = dict(dtype=dtype, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, intermediate=inter, vocab=vocab, layers=layers, rms_eps=1e-6, rope_theta=theta)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).astype(np.uint32)
    sampler = abi.NervaHipHfDecodeSamplerConfig()
    sampler.temperature, sampler.top_p, sampler.top_k, sampler.seed = 0.9, 0.95, 0, 11
    s = N.DecodeSession.create_synthetic(cfg, 64, weight_hash=7, weight_std=0.05)

    def calls(s):
        out = []
        assert s.start(prompt)[0] == 0
        rc, res, tokens = s.advance(6)
        assert rc == 0
        out += [tokens, s.logits()]
        replays = res.graph_replays
        assert s.start(prompt, eos=int(tokens[3]))[0] == 0
        rc, res, stopped = s.advance(12)
        assert rc == 0 and len(stopped) <= 4
        out.append(stopped)
        rc, res, walked = s.run(prompt, 5)
        assert rc == 0
        out.append(walked)
        s.release_sequence()
        assert s.extend(prompt)[0] == 0
        for t in prompt[:3]:
            rc, res, rows, _ = s.extend([t], [0])
            assert rc == 0
            out.append(rows)
        assert s.start(prompt)[0] == 0
        assert s.advance(2)[0] == 0
        rc, res, token, trace = s.traced_advance()
        assert rc == 0
        out += [token, trace["x0"], trace["logits"]] + [layer[k] for layer in trace["layers"] for k in sorted(layer)]
        assert s.start(prompt, sampler=sampler)[0] == 0
        rc, res, drawn = s.advance(8)
        assert rc == 0
        out.append(drawn)
        others = [s.fork_shared_weights() for _ in range(2)]
        for i, q in enumerate([s] + others):
            assert q.start(prompt[:5 + i])[0] == 0 and q.advance(1)[0] == 0
        for _ in range(3):
            rc, res, tokens = N.DecodeSession.batch_advance_one([s] + others, 3, 3)
            assert rc == 0
            out.append(tokens)
        for q in others:
            q.destroy()
        return out, replays

    want, replays = calls(s)
    assert replays == 5 and not s.shares_weight_stream()
    fork = s.fork_shared_weights()
    N.Device.set_tuning("attn_merge_spin_limit", SHORT_WAIT)
    N.Device.set_tuning("step_chain_withhold", 2)
    try:
        got, replays = calls(fork)
    finally:
        N.Device.reset_tuning()
    assert replays == 3 * 5
    for i, (a, b) in enumerate(zip(want, got)):
        assert np.array_equal(a, b), i
    fork.destroy()
    s.destroy()


def test_a_chain_that_never_runs_is_a_step_fault():
    """Steps that give up again and again end the sequence: advance says so in the slot, a one-token extend in its result."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = SHAPES[1]
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.arange(9, dtype=np.uint32)
    N.Device.set_tuning("attn_merge_spin_limit", 50)
    N.Device.set_tuning("step_chain_withhold", 100000)
    try:
        s = N.DecodeSession.create(weights, 64)
        assert s.start(prompt)[0] == 0
        rc, res, tokens = s.advance(3)
        assert rc == -1 and res.hip_error == abi.NERVA_HIP_ERROR_STEP_FAULT
        s.release_sequence()
        assert s.extend(prompt)[0] == 0
        rc, res = s.extend([3], [0])[:2]
        assert rc == -1 and res.hip_error == abi.NERVA_HIP_ERROR_STEP_FAULT
        s.destroy()
    finally:
        N.Device.reset_tuning()


def test_many_chains_and_a_wide_attention_at_once():
    """Six sessions of the largest chains, and one whose attention wants every CU, from threads of their own: whatever of it is resident at a
    time, each gives what it gives alone."""
    narrow = (BF16, 1024, 4, 2, 128, 1024, 301, 6, 1e6, True, False)
    wide = (BF16, 2048, 16, 8, 128, 2048, 301, 2, 1e6, True, False)
    rng = np.random.default_rng(8)
    prompts = [rng.integers(0, 301, n).astype(np.uint32) for n in (1800, 20, 150, 300, 40, 700, 9)]
    weights = [random_model(*g[:8], 3, *g[8:])[0] for g in (narrow, wide)]
    first, broad = N.DecodeSession.create(weights[0], 1024), N.DecodeSession.create(weights[1], 2048)
    sessions = [broad, first] + [first.fork_shared_weights() for _ in range(5)]

    def all_steps(i, out):
        s = sessions[i]
        rc = s.start(prompts[i])[0]
        for _ in range(20):
            if rc == 0:
                rc, res, tokens = s.advance(10)
                out.append((rc, res.graph_nodes, tokens.tolist()))
        out.append(rc)

    alone = [[] for _ in sessions]
    for i in range(len(sessions)):
        all_steps(i, alone[i])
    together = [[] for _ in sessions]
    threads = [threading.Thread(target=all_steps, args=(i, together[i])) for i in range(len(sessions))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(out[-1] == 0 for out in alone + together)
    assert together == alone
    assert all(nodes == (3 if i else 3 + 5 * 2) for i, out in enumerate(alone) for rc, nodes, tokens in out[:-1])
    for s in sessions[::-1]:
        s.destroy()


@pytest.mark.parametrize("scale,eps", [(1e20, 1e-6), (1e-20, 0.0), (2e-19, 0.0), (1e15, 1e-6)])
def test_norms_of_rows_at_the_ends_of_f32(scale, eps):
    """Rows whose sum of squares overflows (their norm is zero), whose mean square is a denormal or just not: what the launches give."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers = BF16, 256, 4, 2, 64, 512, 64, 4
    rng = np.random.default_rng(4)

    def matrix(shape, mean=0.0, std=0.05):
        return O.encode16(dtype, rng.normal(mean, std, shape).astype(np.float32))
    A, KV = heads * hd, kv * hd
    blocks = [dict(rms_attn=matrix(hidden, 1.0), rms_mlp=matrix(hidden, 1.0), w_q=matrix((A, hidden)), w_k=matrix((KV, hidden)), w_v=matrix((KV, hidden)),
                   w_o=O.encode16(dtype, rng.normal(0, 0.05 * min(scale, 1.0), (hidden, A)).astype(np.float32)), w_gate=matrix((inter, hidden)),
                   w_up=matrix((inter, hidden)), w_down=O.encode16(dtype, rng.normal(0, 0.05 * min(scale, 1.0), (hidden, inter)).astype(np.float32)))
              for _ in range(layers)]
    weights = N.ModelWeights(dtype, hidden, heads, kv, hd, inter, vocab, eps, 1e4, matrix((vocab, hidden), 0.0, scale), blocks, matrix(hidden, 1.0), matrix((vocab, hidden)))
    out = []
    try:
        for mode in (2, 0):
            N.Device.set_tuning("step_chain", mode)
            s = N.DecodeSession.create(weights, 32)
            for t in (3, 9, 27):
                rc, res, rows, _ = s.extend([t], [0])
                assert rc == 0 and res.graph_nodes == (3 if mode == 0 else 3 + 5 * layers)
            out.append(rows[0])
            s.destroy()
    finally:
        N.Device.reset_tuning()
    assert np.all(np.isfinite(out[0])) and np.all(np.isfinite(out[1]))
    assert np.linalg.norm(out[1] - out[0]) <= chain_budget(layers) * np.linalg.norm(out[0])


@pytest.mark.parametrize("wide", [False, True])
def test_steps_that_go_out_together_give_what_single_ones_give(wide):
    """Greedy and sampled, one session and a second beside it: a call of 100 steps against calls of one."""
    shape = (BF16, 1024, 16, 8, 128, 2816, 301, 4, 1e6, True, False) if wide else SHAPES[0]
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).astype(np.uint32)
    sampler = abi.NervaHipHfDecodeSamplerConfig()
    sampler.temperature, sampler.top_p, sampler.top_k, sampler.seed = 0.9, 0.95, 0, 11
    s = N.DecodeSession.create(weights, 160)
    for beside in (False, True):
        other = s.fork_shared_weights() if beside else None
        for config in (None, sampler):
            assert s.start(prompt, sampler=config)[0] == 0
            single = np.concatenate([s.advance(1)[2] for _ in range(101)])
            logits = s.logits()
            assert s.start(prompt, sampler=config)[0] == 0
            rc, res, tokens = s.advance(101)
            assert rc == 0 and res.graph_replays == 100 and res.graph_launches == 16 + 4
            assert tokens.tolist() == single.tolist() and np.array_equal(s.logits(), logits)
        if other is not None:
            other.destroy()
    s.destroy()


@pytest.mark.parametrize("shape,context", [(SHAPES[0], 4096), (SHAPES[7], 1536)])
def test_one_call_across_the_context_where_steps_become_launches(shape, context):
    """From sixes to single steps to launches: one call against calls of one step."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers, theta, qk_norm, bias = shape
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 5, theta, qk_norm, bias)
    prompt = np.random.default_rng(2).integers(0, vocab, context - 70).astype(np.uint32)
    s = N.DecodeSession.create(weights, context + 64)
    assert s.start(prompt)[0] == 0
    single = [s.advance(1) for _ in range(91)]
    assert [res.graph_nodes for _, res, _ in single[1:]] == [3] * 70 + [3 + 5 * layers] * 20
    want, logits = [int(tokens[0]) for _, _, tokens in single], s.logits()
    assert s.start(prompt)[0] == 0
    rc, res, tokens = s.advance(91)
    assert rc == 0 and res.graph_replays == 90 and res.graph_launches == 11 + 4 + 20 and res.graph_nodes == 3 + 5 * layers
    assert tokens.tolist() == want and np.array_equal(s.logits(), logits)
    s.destroy()
