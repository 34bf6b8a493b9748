"""flash_duo_kernel on the GPU at the edges of its tiles and of duo_plan's rules, with
and without rows that take the safe walk, against the float64 oracle on sampled rows."""

import math
import random

import numpy as np
import pytest
import torch

from cpu_attention import flash_attn_func
from helpers import assert_close, values
from oracle.attention import attention
from test_duo_geometry import EDGES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gap", [0, 180])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("shape", EDGES)
def test_edges(cuda, shape, d, causal, gap):
    """gap: a key past the first tiles whose logits exceed theirs by about that many
    log2 units in every other head, past the fixed max's headroom, so that some blocks
    walk twice (both key groups, both passes of a pair, every split)."""
    b, sq, sk, h = shape
    print(f"duo edges {shape} d={d} causal={causal} gap={gap}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(sq + sk + d)
    q, k, v = (torch.randn(b, h, n, d, generator=g, device=cuda).transpose(1, 2) for n in (sq, sk, sk))
    if gap:
        q = q + 1.0
        k[:, sk * 2 // 3, ::2] = (gap + 4) / (1.4427 * d ** 0.5)
    q, k, v = (x.bfloat16() for x in (q, k, v))
    out = flash_attn_func(q, k, v, causal=causal)
    r = random.Random(sq * sk + d)
    rows = sorted({0, sq - 1, min(sq - 1, 127), *(r.randrange(sq) for _ in range(12))})
    pairs = {(0, 0), (b - 1, h - 1), *((r.randrange(b), r.randrange(h)) for _ in range(3))}
    for bi, hi in sorted(pairs):
        qv, kv, vv, ov = (values(t[bi:bi + 1, :, hi:hi + 1]) for t in (q, k, v, out))
        ref = []
        for i in rows:
            ke = min(sk, max(0, i + 1 + sk - sq)) if causal else sk
            ref.append(attention(qv[:, i:i + 1], kv[:, :ke], vv[:, :ke], d ** -0.5)[0, 0, 0] if ke else np.zeros(d))
        assert_close(torch.from_numpy(ov[0, rows, 0]), np.stack(ref), torch.bfloat16, paged=False)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("shape", [(1, 256, 900, 2), (1, 128, 2048, 2)])  # two key groups, split keys
def test_first_tile_without_a_finite_logit(cuda, shape, d, causal):
    """Every key of a group's or split's first tile has a logit of -inf, the others lie
    near -200 log2 units: the row max is not fixed at 0, where their p would flush."""
    b, sq, sk, h = shape
    print(f"duo first tile -inf {shape} d={d} causal={causal}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(sk + d)
    q, k, v = (torch.randn(b, h, n, d, generator=g, device=cuda).transpose(1, 2) for n in (sq, sk, sk))
    q[..., :2], k[..., 0], k[..., 1] = 1.0, 0.0, -200 / 1.4427 * d ** 0.5
    gone = [i for i in range(sk) if i // 64 in (1, 4)]
    keep = [i for i in range(sk) if i // 64 not in (1, 4)]
    k[:, gone, :, 0] = float("-inf")
    q, k, v = (x.bfloat16() for x in (q, k, v))
    out = values(flash_attn_func(q, k, v, causal=causal))
    qv, kv, vv = values(q), values(k[:, keep]), values(v[:, keep])
    rows = [0, 1, 63, 64, sq - 1]
    ref = []
    for i in rows:
        n = sum(x <= i + sk - sq for x in keep) if causal else len(keep)
        ref.append(attention(qv[:, i:i + 1], kv[:, :n], vv[:, :n], d ** -0.5)[0, 0])
    assert_close(torch.from_numpy(out[0, rows]), np.stack(ref), torch.bfloat16, paged=False)


# (shape, first tiles of its passes or splits, causal): two key groups, split keys, and at
# d = 128 the 64-row kernel's unsplit blocks, its split keys and its causal pairs
FIRSTS = [((1, 256, 900, 2), (0,), True), ((1, 128, 2048, 2), (0, 4), True), ((1, 256, 2560, 240), (0,), False),
          ((1, 512, 6144, 17), (0, 14), False), ((1, 6144, 6144, 11), (0,), True)]


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("shape,tiles,causal", FIRSTS)
def test_first_tile_of_a_walk_without_a_finite_logit(cuda, shape, tiles, causal, d):
    """As above, of the tile that fixes the max of every walk."""
    b, sq, sk, h = shape
    print(f"first tile -inf {shape} d={d} causal={causal}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(sk + d)
    q, k, v = (torch.randn(b, h, n, d, generator=g, device=cuda).transpose(1, 2) for n in (sq, sk, sk))
    q[..., :2], k[..., 0], k[..., 1] = 1.0, 0.0, -200 / 1.4427 * d ** 0.5
    for t in tiles:
        k[:, 64 * t:64 * t + 64, :, 0] = float("-inf")
    q, k, v = (x.bfloat16() for x in (q, k, v))
    out = flash_attn_func(q, k, v, causal=causal)
    keep = [i for i in range(sk) if i // 64 not in tiles]
    rows = [i for i in (0, 31, 64, 100, 255, 256, 3000, sq - 1) if i < sq and (not causal or i + sk - sq >= 64)]
    for hh in (0, h - 1):
        qv, kv, vv = values(q[:, rows, hh:hh + 1]), values(k[:, keep, hh:hh + 1]), values(v[:, keep, hh:hh + 1])
        ref = []
        for j, i in enumerate(rows):
            n = sum(x <= i + sk - sq for x in keep) if causal else len(keep)
            ref.append(attention(qv[:, j:j + 1], kv[:, :n], vv[:, :n], d ** -0.5)[0, 0, 0])
        assert_close(out[0, rows, hh], np.stack(ref), torch.bfloat16, paged=False)


# log2 units above the first tile's logits: a later key of the first tile's group (or
# split) and a key in the first tile of the other one
PEAKS = [(127.75, 126.25), (125, 127), (127.5, 127), (120, 118), (116, 128)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("peaks", PEAKS)
@pytest.mark.parametrize("d", [32, 64, 128])
def test_groups_of_far_apart_maxima(cuda, d, peaks, causal):
    """Key 160 (tile 2, of key group 0) carries as much weight as key 70 (tile 1, group
    1's first), both about 2^120 times the rest.  A max that each group fixed at its own
    first tile would leave group 0's share a merge weight below the smallest fp32."""
    far_apart(cuda, (1, 256, 900, 2), d, causal, {160: peaks[0], 70: peaks[1]})


# (1, 128, 2048): 8 splits of 256 keys; (1, 512, 6144): 7 of 896, at d = 128 on the 64-row kernel
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("peaks", PEAKS)
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("shape,key", [((1, 128, 2048, 2), 262), ((1, 512, 6144, 17), 902)])
def test_splits_of_far_apart_maxima(cuda, shape, key, d, peaks, causal):
    """As above, of two splits' partials: key 160 lies in tile 2 of split 0, `key` in the
    first tile of split 1."""
    far_apart(cuda, shape, d, causal, {160: peaks[0], key: peaks[1]})


def far_apart(device, shape, d, causal, keys):
    """Logits (log2 units) of 0 or a little more, and of keys[i] at key i."""
    b, sq, sk, h = shape
    print(f"duo far apart {shape} d={d} causal={causal} {keys}", flush=True)
    g = torch.Generator(device=device).manual_seed(sk + d)
    q, k, v = (0.1 * torch.randn(b, h, n, d, generator=g, device=device).transpose(1, 2) for n in (sq, sk, sk))
    v = 10 * v
    q[..., :2], k[..., :2] = 1.0, 0.0
    for i, x in keys.items():
        k[:, i, :, 0], k[:, i, :, 1] = int(x), x - int(x)
    q, k, v = (x.bfloat16() for x in (q, k, v))
    out = flash_attn_func(q, k, v, softmax_scale=math.log(2), causal=causal)
    q, k, v, out = (values(x[:, :, [0, h - 1]]) for x in (q, k, v, out))
    ref = attention(q, k, v, math.log(2), causal)
    assert_close(torch.from_numpy(out), ref, torch.bfloat16, paged=False)
