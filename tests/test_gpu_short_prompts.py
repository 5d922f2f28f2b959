"""Kernels of short prompts, against the kernels of long ones and the token walk."""
import numpy as np
import pytest

import nerva_amd as N
from test_gpu_session import BF16, F16, random_model

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
