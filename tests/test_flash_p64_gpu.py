"""flash_bf16_p64_kernel on the GPU, on the E = 128 calls that duo_plan leaves to it
(test_duo_geometry.py asserts that they are): causal pairs of 256-row query blocks, one
query block per block, and split keys, with and without waves that take the safe pass,
against the float64 oracle on sampled rows."""

import random

import numpy as np
import pytest
import torch

from cpu_attention import flash_attn_func
from helpers import assert_close, values
from oracle.attention import attention
from test_duo_geometry import P64

pytestmark = pytest.mark.gpu
D = 128

# A key some 180 log2 units above every row's first-tile max, past the fast walk's
# headroom, for the rows that see it and have q > 0: (key, first row with q < 0) as
# parts of the keys and rows.  Of the pairs (nqb - 1 - j, j) that leaves pass 0 alone
# (the key lies past the low blocks' rows), pass 1 alone, or both.
FAILING = {"none": None, "pass 0": (0.66, 1.0), "pass 1": (0.03, 0.5), "both": (0.02, 1.0)}


@pytest.mark.parametrize("failing", list(FAILING))
@pytest.mark.parametrize("shape,causal", [(s, c) for s, c, _, _ in P64])
def test_against_the_oracle(cuda, shape, causal, failing):
    b, sq, sk, h = shape
    print(f"64-row kernel {shape} causal={causal} failing={failing}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(sq + sk)
    q, k, v = (0.5 * torch.randn(b, n, h, D, generator=g, device=cuda) for n in (sq, sk, sk))
    q, v = q + 1.0, 2 * v
    if FAILING[failing]:
        key, neg = FAILING[failing]
        k[:, int(key * sk)] = 184 / (1.4427 * D ** 0.5)
        q[:, int(neg * sq):] *= -1.0
    q, k, v = (x.bfloat16() for x in (q, k, v))
    out = flash_attn_func(q, k, v, causal=causal)
    r = random.Random(sq)
    rows = sorted({0, 63, 64, sq - 1, *(min(sq - 1, i + r.randrange(256)) for i in range(0, sq, 256)),
                   *(r.randrange(sq) for _ in range(8))})
    for hh in (0, h // 2, h - 1):
        qv, kv, vv = (values(x[:, :, hh:hh + 1]) for x in (q, k, v))
        ref = [attention(qv[:, i:i + 1], kv[:, :n], vv[:, :n], D ** -0.5)[0, 0, 0]
               for i in rows for n in (min(sk, i + 1 + sk - sq) if causal else sk,)]
        assert_close(out[0, rows, hh], np.stack(ref), torch.bfloat16, paged=False)
