"""Rows of long prompts: there once for all sessions on the same weights, which take turns on them."""
import threading

import numpy as np
import pytest

import nerva_amd as N
import stack_models as M
from nerva_amd import abi
from test_gpu_any_width import walked
from test_gpu_session import BF16, E2E_REL_L2, F16, random_model, rel_l2

pytestmark = pytest.mark.gpu

# dtype, hidden, heads, kv, hd, inter, vocab, layers
DENSE = (BF16, 1536, 12, 2, 128, 2944, 801, 2)


def dense(geom=DENSE):
    dtype, hidden, heads, kv, hd, inter, vocab, layers = geom
    return random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, hidden, 1e6, False, False)[0]


def decoder_session(max_context):
    return N.DecodeSession.create(dense(), max_context)


def stack_session(max_context):
    cfg = M.config([M.attention(16, 4, 128, 128, rot=32, chunk=700, ff=320), M.mingru(width=320, ff=448), M.mingru(width=64, ff=0)],
                   width=192, vocab=300)
    return M.session(cfg, M.weights(cfg, seed=31), max_context)


def without_cache(session):
    return session.create_result.device_arena_bytes - session.create_result.resident_kv_bytes


def test_only_the_weights_hold_rows_for_passes():
    """A fork has rows for a block of 512, the creating session those for passes of 4096 besides; sessions that take no
    passes (128-row blocks, a walk token by token, a head size without blocks) have neither, whatever their context."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers = DENSE
    row = 10 * hidden + 4 * (heads + 2 * kv) * hd + 2 * heads * hd + 2 * inter
    parent = decoder_session(4800)
    fork = parent.fork_shared_weights()
    assert without_cache(parent) - without_cache(fork) >= 4096 * row
    for s in (fork, parent):
        s.destroy()
    odd, eighty = dense((BF16, 416, 6, 2, 128, 608, 517, 2)), dense((F16, 320, 4, 2, 80, 640, 301, 2))
    for create in (lambda ctx: walked(dense(), ctx), lambda ctx: N.DecodeSession.create(odd, ctx), lambda ctx: N.DecodeSession.create(eighty, ctx)):
        small, large = create(512), create(4800)
        assert without_cache(large) - without_cache(small) <= (4800 - 512) * 64
        for s in (small, large):
            s.destroy()
    parent = stack_session(4800)
    fork = parent.fork_shared_weights()
    assert without_cache(parent) - without_cache(fork) >= 4096 * 192 * 10
    for s in (fork, parent):
        s.destroy()


@pytest.mark.parametrize("create", [decoder_session, stack_session])
def test_long_prompts_of_sessions_on_the_same_weights(create):
    """Three sessions on one set of weights, a thread each: long prompts, short ones and steps between them, twice over, as
    each has them alone; and the forks go on when the creating session is gone."""
    parent = create(2600)
    sessions = [parent, parent.fork_shared_weights(), parent.fork_shared_weights()]
    prompts = [[np.random.default_rng(10 * i + k).integers(0, parent.vocab, n).astype(np.uint32) for k, n in enumerate(lengths)]
               for i, lengths in enumerate(((1700, 40, 900), (513, 2100, 300), (600, 601, 1025)))]

    def work(session, own, results, at):
        out = []
        for prompt in own + own:
            rc, _, logits, _ = session.extend(prompt, [0, prompt.size - 1])
            assert rc == 0
            rc, _, tokens = session.advance(3)
            assert rc == 0 and session.release_sequence() == 0
            out.append((logits, tokens.tolist()))
        results[at] = out

    def run(who, together):
        results = [None] * 3
        threads = [threading.Thread(target=work, args=(sessions[i], prompts[i], results, i)) for i in who]
        for thread in threads:
            thread.start()
            if not together:
                thread.join()
        for thread in threads:
            thread.join()
        return results

    alone, together = run((0, 1, 2), False), run((0, 1, 2), True)
    parent.destroy()
    orphaned = run((1, 2), True)
    for i in range(3):
        for got in (together, orphaned):
            if got is orphaned and i == 0:
                continue
            for (logits, tokens), (want, want_tokens) in zip(got[i], alone[i]):
                assert np.array_equal(logits, want) and tokens == want_tokens, i      # the same launches on the same rows
    for s in sessions[1:]:
        s.destroy()


def test_a_fork_made_under_other_overrides():
    """A fork that takes passes where the creating session did not has no rows for them; one that does not, where it did,
    takes none: both have the prompt's logits."""
    prompt = np.random.default_rng(5).integers(0, DENSE[6], 1500).astype(np.uint32)
    logits = []
    for first, second in ((0, 512), (512, 0), (1024, 0), (0, 1024)):
        sessions = []
        for cap in (first, second):
            N.Device.set_tuning("prefill_block_tokens", cap)
            try:
                sessions.append(sessions[0].fork_shared_weights() if sessions else N.DecodeSession.create(dense(), 1600))
            finally:
                N.Device.set_tuning("prefill_block_tokens", 0)
        for s in sessions:
            assert s.start(prompt)[0] == 0
            logits.append(s.logits().copy())
        for s in sessions[::-1]:
            s.destroy()
    for got in logits[1:]:
        assert rel_l2(got, logits[0]) <= E2E_REL_L2


@pytest.mark.parametrize("geom", [(BF16, 512, 8, 2, 64, 1024, 301, 3), (BF16, 1024, 16, 8, 128, 2816, 301, 4)])   # (steps of launches, of one for the whole device)
def test_sequences_begun_one_behind_the_other(geom):
    """Starts and extensions whose callers wait for nothing in between, on sessions of one set of weights and on one session that begins again, the callers' memory written over as soon as
    a call returns: tokens, logits and cache rows of each as when it is alone."""
    dtype, hidden, heads, kv, hd, inter, vocab, layers = geom
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, vocab, layers, 4, 1e6, True, False)
    rng = np.random.default_rng(6)
    prompts = [rng.integers(0, 301, n).astype(np.uint32) for n in (5, 300, 1, 17, 130, 64)]
    sampler = abi.NervaHipHfDecodeSamplerConfig()
    sampler.temperature, sampler.top_p, sampler.top_k, sampler.seed = 0.8, 0.9, 0, 3
    first = N.DecodeSession.create(weights, 400)
    sessions = [first] + [first.fork_shared_weights() for _ in prompts[1:]]

    def result(s, n):
        rc, res, tokens = s.advance(6)
        assert rc == 0
        return tokens.tolist(), s.logits().tolist(), [rows.tolist() for rows in s.kv_range(2, 0, n + 5)]
    alone = []
    for i, prompt in enumerate(prompts):
        assert first.start(prompt, sampler=sampler if i % 2 else None)[0] == 0
        alone.append(result(first, len(prompt)))
    for round_ in range(3):
        for i, (s, prompt) in enumerate(zip(sessions, prompts)):
            buffer = prompts[(i + 1) % len(prompts)].copy()
            assert s.start(buffer, sampler=None if i % 2 else sampler)[0] == 0      # (begun again at once, with another prompt and sampler)
            buffer = prompt.copy()
            assert s.start(buffer, sampler=sampler if i % 2 else None)[0] == 0
            buffer[:] = 7
        for i in (range(len(prompts)) if round_ % 2 == 0 else reversed(range(len(prompts)))):
            assert result(sessions[i], len(prompts[i])) == alone[i], (round_, i)
    parts = [rng.integers(0, 301, n).astype(np.uint32) for n in (40, 3, 1, 20)]

    def extended(s):
        s.release_sequence()
        out = []
        for part in parts:
            buffer = part.copy()
            rc, _, rows, _ = s.extend(buffer, [len(part) - 1])
            buffer[:] = 7
            assert rc == 0
            out.append(rows.tolist())
        return out
    want = extended(first)
    assert all(extended(s) == want for s in sessions[1:])
    for s in sessions[::-1]:
        s.destroy()


def test_walked_prompts_begun_one_behind_the_other():
    """Prompts walked step by step, whose attention launches wait within themselves: begun on five sessions of two models without a wait in between."""
    geoms = [(BF16, 2048, 16, 8, 128, 2048, 301, 2), (BF16, 512, 8, 2, 64, 1024, 301, 2)]
    rng = np.random.default_rng(8)
    prompts = [rng.integers(0, 301, n).astype(np.uint32) for n in (300, 260, 310, 290, 280)]
    try:
        N.Device.set_tuning("prefill_walk", 1)
        models = [N.DecodeSession.create(random_model(*g, 4, 1e6, True, False)[0], 400) for g in geoms]
        sessions = [models[0], models[1], models[0].fork_shared_weights(), models[1].fork_shared_weights(), models[0].fork_shared_weights()]

        def result(s):
            rc, _, tokens = s.advance(4)
            assert rc == 0
            return tokens.tolist(), s.logits().tolist()
        alone = []
        for s, prompt in zip(sessions, prompts):
            assert s.start(prompt)[0] == 0
            alone.append(result(s))
        for s, prompt in zip(sessions, prompts):
            assert s.start(prompt)[0] == 0
        for s in sessions:
            assert s.logits().shape == (301,)      # (waits for the session's own work, so that no step meets another's prompt)
        assert [result(s) for s in sessions] == alone
        for s in sessions[::-1]:
            s.destroy()
    finally:
        N.Device.reset_tuning()


def test_calls_behind_walked_prompts_under_way():
    """A start of a walked prompt, and of one whose last token takes a step, returns while its attention launches are under way. What the next call brings on another session - tokens walked or alone,
    steps in launches, in one launch of the whole device, of a narrow model - comes behind them: every result as when nothing is under way."""
    geoms = [(BF16, 2048, 16, 8, 128, 2048, 301, 2), (BF16, 1024, 16, 8, 128, 2816, 301, 4), (BF16, 512, 4, 2, 128, 1024, 301, 4)]
    rng = np.random.default_rng(9)
    prompt = rng.integers(0, 301, 700).astype(np.uint32)
    sessions = []
    try:
        for walk in (1, 0):
            N.Device.set_tuning("prefill_walk", walk)
            sessions += [N.DecodeSession.create(random_model(*g, 4, 1e6, True, False)[0], 1100) for g in geoms]
    finally:
        N.Device.reset_tuning()
    walked, blocks = sessions[:3], sessions[3:]

    def begun(s):
        assert s.start(prompt[:90])[0] == 0 and s.advance(2)[0] == 0

    def stepped(s):
        rc, _, tokens = s.advance(5)
        return rc, tokens.tolist()

    def extended(s):
        return [(rc, rows.tolist()) for rc, _, rows, _ in (s.extend(prompt[:n], [n - 1]) for n in (30, 1))]

    def ran(s):
        rc, _, tokens = s.run(prompt[:40], 4)
        return rc, tokens.tolist()
    want = {}
    for s in sessions:
        for call in (stepped, extended, ran):
            begun(s)
            want[s, call] = call(s)
    for first, start in [(s, prompt) for s in walked] + [(s, prompt[:1]) for s in blocks] + [(blocks[0], prompt[:513])]:
        for s in sessions:
            if s is first:
                continue
            for call in (stepped, extended, ran):
                begun(s)
                assert first.start(start)[0] == 0
                assert call(s) == want[s, call]
    for s in sessions[::-1]:
        s.destroy()


def test_starts_behind_sessions_that_are_gone():
    """What the last starts have left to wait for may have been on sessions that have ended since: walked prompts, single tokens, prompts in blocks, on the same weights and on others."""
    prompts = [np.arange(n, dtype=np.uint32) for n in (1, 40, 300)]
    tokens = []
    for walk in (0, 1, 0):
        N.Device.set_tuning("prefill_walk", walk)
        try:
            s = decoder_session(400)
        finally:
            N.Device.reset_tuning()
        for _ in range(4):
            for prompt in prompts:
                fork = s.fork_shared_weights()
                assert fork.start(prompt)[0] == 0
                fork.destroy()
                assert s.start(prompt)[0] == 0
                rc, _, out = s.advance(3)
                assert rc == 0
                tokens.append((walk, len(prompt), out.tolist()))
        s.destroy()
    assert all(a[2] == b[2] for a in tokens for b in tokens if a[:2] == b[:2])
