"""The host-side length check on the GPU: a length past the page table's capacity is
refused wherever it stands, for vectors that are copied to the host whole (up to 4096
bytes) and longer ones, and nothing is written by the refused call."""

import pytest
import torch

from cpu_attention import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 5, 1024, 1025])
def test_a_length_past_the_table_is_refused(cuda, n):
    h, d, page, width = 1, 32, 16, 2
    kc = torch.zeros(2, h, page, d, device=cuda)
    vc = torch.zeros_like(kc)
    q, k, v = (torch.ones(n, 1, h, d, device=cuda) for _ in range(3))
    table = torch.zeros(n, width, dtype=torch.int32, device=cuda)
    for at in sorted({0, n // 2, n - 1}):
        lens = torch.full((n,), 3, dtype=torch.int32, device=cuda)
        lens[at] = width * page  # one more does not fit
        with pytest.raises(ValueError, match="exceed the page table"):
            flash_attn_with_kvcache(q, kc, vc, k=k, v=v, cache_seqlens=lens, page_table=table)
        assert not kc.any() and not vc.any()
        lens[at] = width * page - 1
        flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens, page_table=table)
