"""Kernels of short prompts, of few token rows and of batch steps, against the oracle and against the kernels they stand in for."""
import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from test_gpu_ops import dev
from test_gpu_session import BF16, E2E_REL_L2, F16, random_model, rel_l2, started

pytestmark = pytest.mark.gpu


# 1 to 8 query heads a key head, both head sizes; with q/k norms, biases, no rotation
@pytest.mark.parametrize("dtype,heads,kv,hd,theta,qk_norm,bias", [
    (BF16, 4, 4, 128, 1e6, True, False), (F16, 8, 4, 64, 1e4, False, True), (BF16, 6, 2, 64, 1e6, True, True),
    (BF16, 16, 4, 128, 0, True, False), (F16, 10, 2, 128, 1e4, False, True), (F16, 12, 2, 64, 1e6, True, False),
    (BF16, 14, 2, 128, 1e6, False, True), (F16, 16, 2, 128, 1e6, True, False)])
def test_narrow_and_wide_prompt_attention_give_the_same_bits(dtype, heads, kv, hd, theta, qk_norm, bias):
    """Prompts at the edges of a wave's and a workgroup's tokens (16 / G and 64 / G in the narrow workgroups, 256 / G in the wide
    ones) and of steps of 64 keys, from the start and behind a prefix. Both add a token's keys up in the same order, one split
    each: the same logits and cache rows to the last bit."""
    group, vocab = heads // kv, 301
    weights, _ = random_model(dtype, 512, heads, kv, hd, 512, vocab, 2, heads, theta, qk_norm, bias)
    s = N.DecodeSession.create(weights, 700)
    rng = np.random.default_rng(heads)
    few, wave = 16 // group, 4 * (16 // group)
    for prefix, n in ((0, 2), (0, few + 1), (0, wave), (0, wave + 1), (0, 64), (0, 65), (0, 16 * (16 // group) + 1), (0, 320), (63, 2),
                      (63, wave + 1), (130, 129), (200, 333)):
        tokens = rng.integers(0, vocab, prefix + n).astype(np.uint32)
        results = []
        try:
            N.Device.set_tuning("prompt_splits", 1)
            for waves in (4, 8):
                N.Device.set_tuning("prompt_waves", waves)
                assert s.release_sequence() == 0
                if prefix:
                    assert s.extend(tokens[:prefix])[0] == 0
                rc, _, rows, _ = s.extend(tokens[prefix:], sorted({0, n // 2, n - 1}))
                assert rc == 0
                results.append((rows.copy(), s.kv_range(1, 0, prefix + n)))
        finally:
            N.Device.reset_tuning()
        assert np.all(np.isfinite(results[0][0])) and np.array_equal(results[0][0], results[1][0]), (prefix, n)
        for got, want in zip(results[0][1], results[1][1]):
            assert np.array_equal(got, want), (prefix, n)
    s.destroy()


@pytest.fixture
def tuned():
    yield N.Device.set_tuning
    N.Device.reset_tuning()


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("rows,cols,tokens", [(16, 2048, 1), (20, 2048, 5), (48, 4096, 16), (4100, 2048, 17), (36, 6144, 32), (64, 10240, 15),
                                              (32, 14336, 31)])
def test_few_rows_without_slices_match_the_oracle(tuned, dtype, rows, cols, tokens):
    """Row counts off the grid of 16, 4 to 28 blocks a wave in whole rounds of four (the operator takes no other widths: those are in
    the next test), one and two token tiles: plain, with bias, residual and rounding, and gate/up pairs in rows and in operand order."""
    tuned("gemm_few", 1)
    rng = np.random.default_rng(rows + cols + tokens)
    w = O.encode16(dtype, rng.normal(0, 0.02, (2 * rows, cols)))
    x = O.encode16(dtype, rng.normal(0, 1, (tokens, cols)))
    bias, res = O.encode16(dtype, rng.normal(0, 0.1, rows)), rng.normal(0, 1, (tokens, rows)).astype(np.float32)
    packed, _ = N.gemm_operand_order(x)
    exact = O.decode16(dtype, x).astype(np.float64) @ O.decode16(dtype, w).astype(np.float64).T
    y, dw, dx = N.DeviceBuffer(tokens * rows * 4), dev(w), dev(packed)
    N.gemm_rows(dtype, dw, rows, cols, tokens, dx, epilogue=0, out_f32=y, input_operand_order=True)
    got = y.numpy(np.float32).reshape(tokens, rows)
    assert max(rel_l2(g, e) for g, e in zip(got, exact[:, :rows])) <= 2e-6      # sums of f32 over at most 14336 columns
    N.gemm_rows(dtype, dw, rows, cols, tokens, dx, epilogue=1, bias=dev(bias), residual=dev(res), out_f32=y, round_output=True,
                input_operand_order=True)
    got = y.numpy(np.float32).reshape(tokens, rows)
    assert rel_l2(got, O.decode16(dtype, O.encode16(dtype, (exact[:, :rows] + O.decode16(dtype, bias) + res).astype(np.float32)))) <= 4e-3
    gate, up = exact[:, :rows], exact[:, rows:]
    pairs = O.decode16(dtype, O.encode16(dtype, (gate / (1 + np.exp(-gate)) * up).astype(np.float32)))
    out = N.DeviceBuffer(tokens * rows * 2)
    N.gemm_rows(dtype, dw, rows, cols, tokens, dx, epilogue=2, out16=out, input_operand_order=True)
    assert rel_l2(O.decode16(dtype, out.numpy(np.uint16, tokens * rows)).reshape(tokens, rows), pairs) <= 4e-3
    if rows % 32 == 0:
        out = N.DeviceBuffer(32 * rows * 2)
        N.gemm_rows(dtype, dw, rows, cols, tokens, dx, epilogue=2, out16=out, input_operand_order=True, output16_operand_order=True)
        _, at = N.gemm_operand_order(np.zeros((tokens, rows), np.uint16))
        gate, up = exact[:, :rows], exact[:, rows:]
        got = O.decode16(dtype, out.numpy(np.uint16, 32 * rows)[at])
        assert rel_l2(got, O.decode16(dtype, O.encode16(dtype, (gate / (1 + np.exp(-gate)) * up).astype(np.float32)))) <= 4e-3


# dtype, hidden, heads, kv, hd, inter: the first normed projection reads fewer blocks of 64 columns than it has waves, an odd number, all
NORMED = [(BF16, 512, 4, 2, 128, 1024), (F16, 960, 10, 2, 64, 2560), (BF16, 1024, 8, 4, 128, 3072)]


@pytest.mark.parametrize("geom", NORMED, ids=str)
def test_projections_that_norm_their_input(tuned, geom):
    """2 to 16 tokens of a sequence, and 17, whose projections have a norm in front, with the kernel and without it."""
    dtype, hidden, heads, kv, hd, inter = geom
    weights, _ = random_model(dtype, hidden, heads, kv, hd, inter, 301, 3, hidden, 1e6, True, False)
    s = N.DecodeSession.create(weights, 64)
    rng = np.random.default_rng(hidden)
    for n in (2, 3, 15, 16, 17):
        tokens, rows = rng.integers(0, 301, 20 + n).astype(np.uint32), []
        for mode in (0, 2):
            tuned("gemm_few", mode)
            assert s.release_sequence() == 0
            assert s.extend(tokens[:20])[0] == 0
            rc, _, logits, _ = s.extend(tokens[20:], range(n))
            assert rc == 0
            rows.append((logits.copy(), s.kv_range(0, 20, n)))
        assert rel_l2(rows[0][0], rows[1][0]) <= E2E_REL_L2, n
        for got, want in zip(rows[0][1], rows[1][1]):    # of the first layer: the sums' order alone
            assert rel_l2(O.decode16(dtype, got), O.decode16(dtype, want)) <= 2e-3, n
    s.destroy()


# dtype, hidden, heads, kv, hd, inter: eight waves, four blocks of 64 columns of each in flight - of inter's 1 a wave or none, 6, 5 or 6, 6 or 7,
# 10 or 11 (whole rounds of four and a remainder, unequal waves); of hidden's 1 or none, 2, 1 or 2, 1 or none, 2 or 3
FEW = [(F16, 64, 2, 1, 64, 448), (BF16, 1024, 8, 4, 128, 3072), (BF16, 704, 6, 2, 64, 2624), (F16, 320, 4, 4, 64, 3520), (BF16, 1088, 6, 2, 128, 5248)]


@pytest.mark.parametrize("geom", FEW, ids=str)
def test_few_rows_of_any_width_match_the_oracle(tuned, geom):
    """2 to 16 tokens of a sequence, 17 and 31, behind 20 others, through the kernel without K slices wherever it can run and as the
    estimate has it: logits, and every layer's keys and values, against the oracle's token by token."""
    dtype, hidden, heads, kv, hd, inter = geom
    weights, model = random_model(dtype, hidden, heads, kv, hd, inter, 301, 2, hidden, 1e6, True, False)
    tokens = np.random.default_rng(hidden).integers(0, 301, 51).astype(np.uint32)
    oracle, want, rows = O.Context(model, 64), [], []
    for i, token in enumerate(tokens):
        oracle.forward_token(int(token), prompt_token=True)
        want.append(oracle.logits())
        rows.append([oracle.read_kv16(layer, i) for layer in range(2)])
    s = N.DecodeSession.create(weights, 64)
    for mode in (1, 0):
        tuned("gemm_few", mode)
        for n in (2, 3, 15, 16, 17, 31):
            assert s.release_sequence() == 0
            assert s.extend(tokens[:20])[0] == 0
            rc, _, logits, _ = s.extend(tokens[20:20 + n], range(n))
            assert rc == 0
            assert max(rel_l2(g, w) for g, w in zip(logits, want[20:20 + n])) <= E2E_REL_L2, (mode, n)
            for layer in range(2):
                for which, got in enumerate(s.kv_range(layer, 0, 20 + n)):
                    ref = np.stack([r[layer][which] for r in rows[:20 + n]])
                    got = O.decode16(dtype, got).reshape(ref.shape)
                    assert rel_l2(got, O.decode16(dtype, ref)) <= (2e-3 if layer == 0 else E2E_REL_L2), (mode, n, layer)
    s.destroy()


# the batch step's attention: partial sums of q, k, v as they come (2048 wide, many sequences) or added; 1 to 8 query heads a key head
@pytest.mark.parametrize("dtype,hidden,heads,kv,hd,count,length", [
    (BF16, 1024, 16, 8, 128, 6, 764),    # from one split a sequence to several
    (F16, 1024, 16, 8, 128, 4, 573),     # the same where splits come earlier
    (BF16, 1024, 16, 8, 128, 32, 2046),  # a workgroup a CU and up to 16 tiles a wave in the step kernel, then the block kernel
    (F16, 1024, 16, 8, 64, 32, 1100),    # the same in one split, heads of 64
    (BF16, 2048, 16, 8, 128, 32, 30), (F16, 512, 8, 4, 64, 9, 250), (BF16, 512, 14, 2, 64, 3, 129), (F16, 768, 10, 2, 128, 2, 513),
    (BF16, 512, 16, 2, 128, 5, 63), (BF16, 512, 16, 16, 64, 20, 15)])    # (the last: more workgroups than CUs)
def test_batch_attention_matches_sequences_alone(dtype, hidden, heads, kv, hd, count, length):
    """Contexts of a key, around a wave's four requested tiles, and across the lengths where the split factor or the kernel changes."""
    vocab, layers, steps = 301, 2, 6
    weights, _ = random_model(dtype, hidden, heads, kv, hd, 1024, vocab, layers, count, 1e6, True, True)
    parent = N.DecodeSession.create(weights, length + 16, plan=N.WeightPlan.from_weights(weights))
    sessions = [parent] + [parent.fork_shared_weights() for _ in range(count - 1)]
    assert parent.shares_weight_stream() or hidden < 1024
    rng = np.random.default_rng(count)
    prompts = [rng.integers(0, vocab, length if i % 3 == 0 else 1 + (length * i) // count).astype(np.uint32) for i in range(count)]
    streams = [[started(s, p)] for s, p in zip(sessions, prompts)]
    for _ in range(steps):
        rc, _, tokens = N.DecodeSession.batch_advance_one(sessions, 32, 2)
        assert rc == 0
        for stream, token in zip(streams, tokens):
            stream.append(int(token))
    solo = parent.fork_shared_weights()
    for i in sorted({0, 1, count - 1}):
        assert solo.release_sequence() == 0
        assert solo.extend(prompts[i])[0] == 0
        for token in streams[i][:-1]:
            assert solo.extend([token], [0])[0] == 0
        for layer in range(layers):
            for got, want in zip(sessions[i].kv_range(layer, len(prompts[i]), steps), solo.kv_range(layer, len(prompts[i]), steps)):
                tol = 2e-3 if layer == 0 else E2E_REL_L2
                assert rel_l2(O.decode16(dtype, got), O.decode16(dtype, want)) <= tol, (i, layer)
    solo.destroy()
    for s in sessions[::-1]:
        s.destroy()


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("tokens", [65, 80, 81, 96, 97, 112, 113, 129, 160, 161, 192, 193, 224, 225])
def test_blocks_of_fewer_tiles_than_their_layout(dtype, tokens):
    """Both ends of every number of token tiles between 5 and 16, in workgroups of three and of four wave pairs and of one and two
    row tiles; token slots without a token hold NaN, which must not get anywhere."""
    rng = np.random.default_rng(tokens)
    for rows, cols in ((192, 2048), (256, 2048), (12288, 2048)):
        pairs = rows == 256
        w = O.encode16(dtype, rng.normal(0, 0.02, ((2 if pairs else 1) * rows, cols)))
        x = O.encode16(dtype, rng.normal(0, 1, (tokens, cols)))
        packed, at = N.gemm_operand_order(x)
        packed[:] = 0x7fff
        packed[at] = x
        exact = O.decode16(dtype, x).astype(np.float32) @ O.decode16(dtype, w).astype(np.float32).T
        ws, y = N.DeviceBuffer(N.gemm_rows_workspace_bytes(2 * rows)), N.DeviceBuffer(tokens * rows * 4)
        N.gemm_rows(dtype, dev(w[:rows]), rows, cols, tokens, dev(packed), out_f32=y, input_operand_order=True, workspace=ws)
        assert rel_l2(y.numpy(np.float32).reshape(tokens, rows), exact[:, :rows]) <= 4e-6     # f32 sums of 2048 on both sides
        if pairs:
            out = N.DeviceBuffer(tokens * rows * 2)
            N.gemm_rows(dtype, dev(w), rows, cols, tokens, dev(packed), epilogue=2, out16=out, input_operand_order=True, workspace=ws)
            gate, up = exact[:, :rows], exact[:, rows:]
            got = O.decode16(dtype, out.numpy(np.uint16, tokens * rows)).reshape(tokens, rows)
            assert rel_l2(got, O.decode16(dtype, O.encode16(dtype, gate / (1 + np.exp(-gate)) * up))) <= 4e-3


@pytest.mark.parametrize("tokens", [3, 70, 130, 300])
def test_gates_of_any_size(tokens):
    """A gate/up pair whose gates are small, large, with a divisor that has no normal reciprocal in 32 bits (-87.5 to -88.5), past
    where e^-g is finite in 32 bits, infinite and NaN."""
    rows, cols = 128, 2048
    values = np.array([0.0, -0.0, 1e-20, -1e-20, 0.5, -0.5, 9.0, -9.0, 80.0, -80.0, 87.0, -87.0, -87.5, -88.0, -88.5, 90.0, -90.0, -104.0, 300.0,
                       -300.0, 3e38, -3e38, np.inf, -np.inf, np.nan], np.float32)
    gates = O.decode16(BF16, O.encode16(BF16, np.resize(values, rows)))
    w = np.zeros((2 * rows, cols), np.float32)
    w[:rows, 0], w[rows:, 0] = gates, 1.5
    x = np.zeros((tokens, cols), np.float32)
    x[:, 0] = 1.0
    packed, _ = N.gemm_operand_order(O.encode16(BF16, x))
    out, ws = N.DeviceBuffer(tokens * rows * 2), N.DeviceBuffer(N.gemm_rows_workspace_bytes(2 * rows))
    N.gemm_rows(BF16, dev(O.encode16(BF16, w)), rows, cols, tokens, dev(packed), epilogue=2, out16=out, input_operand_order=True, workspace=ws)
    got = O.decode16(BF16, out.numpy(np.uint16, tokens * rows)).reshape(tokens, rows)
    with np.errstate(all="ignore"):
        g = gates.astype(np.float64)
        want = np.where(np.isfinite(g), g / (1 + np.exp(-np.clip(g, -700, 700))) * 1.5, np.where(g > 0, np.inf, np.nan))
        want[(g < -88.73) & np.isfinite(g)] = 0.0    # (the exponential is infinite in 32 bits)
    for row in got:
        assert np.array_equal(np.isnan(row), np.isnan(want)) and np.array_equal(np.isinf(row), np.abs(want) > 3.39e38)
        fine = np.isfinite(want) & (np.abs(want) <= 3.39e38)
        assert np.all(np.abs(row[fine] - want[fine]) <= 2.0 ** -8 * np.abs(want[fine]))    # a rounding to 16 bits


@pytest.mark.parametrize("experts", [1, 3, 48, 64, 65, 129, 255, 256, 257])
def test_routes_of_any_number_of_experts(experts):
    """Both kernels of the route: ties, experts without a share, logits that are not finite, all experts chosen."""
    rng = np.random.default_rng(experts)
    for kind in range(5):
        logits = rng.normal(0, 2, experts).astype(np.float32)
        if kind == 1:
            logits = np.round(logits)                     # ties
        if kind == 2:
            logits[:] = 0.5
        if kind == 3:
            logits[rng.random(experts) < 0.5] = -200.0    # probabilities of 0, the rest ahead of them
        if kind == 4:
            logits[rng.random(experts) < 0.3] = -np.inf
            logits[0] = 1.0
        for top in sorted({1, min(8, experts), min(64, experts)}):
            for norm in (True, False):
                ids, weights, _, _ = N.moe_route_softmax(logits, top, norm)
                want_ids, want = O.moe_route_softmax(np.maximum(logits, -1e30), top, norm)    # (the oracle takes finite logits: e^-1e30 is 0 too)
                assert ids.tolist() == want_ids.tolist(), (kind, top)
                assert np.allclose(weights, want, rtol=2e-6, atol=1e-38), (kind, top)
    logits = rng.normal(0, 2, experts).astype(np.float32)
    logits[experts // 2] = np.nan     # no expert with a NaN has a share; places that nobody takes hold expert 0 with weight 0
    ids, weights, _, _ = N.moe_route_softmax(logits, min(4, experts), False)
    assert np.all(np.isfinite(weights)) and not np.any((ids == experts // 2) & (weights > 0))
