"""Which kernel, schedule and parts an attention call takes, as the library describes its own choice (host
only; 256 CUs)."""
import pytest
import torch

import kyro_amd
from kyro_amd.attention import describe_attention

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def describe(H, Hkv, D, batch, max_q, blocks, dtype="bf16", total_q=None, **kw):
    return describe_attention(kyro_amd.PagedAttention(16, H, D, Hkv), batch=batch, total_q=total_q or batch * max_q,
                              max_q_len=max_q, max_blocks_per_seq=blocks, num_blocks=batch * blocks, dtype=DTYPES[dtype],
                              **kw)


@pytest.mark.parametrize("H,Hkv,D,batch,max_q,blocks,dtype", [
    (32, 8, 128, 2, 4, 63, "bf16"), (8, 2, 128, 1, 1, 19, "bf16"), (32, 8, 64, 4, 1, 19, "bf16"),
    (32, 8, 128, 2, 8, 256, "f32"), (28, 4, 80, 4, 1, 256, "f32"),
])
def test_padding_rows_do_not_choose_the_kernel(H, Hkv, D, batch, max_q, blocks, dtype):
    """q may have rows that belong to no sequence (a batch padded to a captured size): the call takes the
    kernel of the rows its sequences can bring, not the one for many rows."""
    text = describe(H, Hkv, D, batch, max_q, blocks, dtype, total_q=512)
    assert text == describe(H, Hkv, D, batch, max_q, blocks, dtype)
    assert "attn_mfma" in text, text
