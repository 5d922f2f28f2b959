"""What a token does not see has no part in its attention: keys behind its position - rows of its last block that nobody has
written, rows of an earlier sequence, later tokens of its prompt - may hold anything, numbers that are not finite too."""
import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from nerva_amd.runtime import attention_workspace
from test_gpu_ops import _attention_case, _attention_oracle, dev
from test_gpu_session import BF16, F16, REL_L2, rel_l2

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

