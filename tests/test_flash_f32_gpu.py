"""The fp32 prefill's split operands (flash_f32_kernel) on the GPU: the edges of its
tiles and of f32_exact, every schedule, values that leave the split's range or that
large neighbours would hide, and the error against 64 bits."""

import math

import numpy as np
import pytest
import torch

from cpu_attention import flash_attn_func
from helpers import values
from oracle.attention import attention

pytestmark = pytest.mark.gpu

# (batch, seq_q, seq_k, heads): one block, partial tiles and query blocks, both sides of
# f32_exact and of the two key groups' line, split keys (few blocks), one query block
# per block, causal pairs with two key groups and with one
SHAPES = [(1, 17, 32, 2), (1, 40, 33, 2), (2, 20, 64, 3), (1, 129, 65, 3), (1, 30, 192, 2), (1, 64, 193, 2),
          (1, 70, 191, 2), (3, 330, 350, 20), (1, 100, 1000, 3), (1, 200, 1500, 5), (2, 300, 300, 60),
          (1, 700, 700, 100), (1, 2048, 2048, 32), (1, 2100, 2100, 33)]


def tensors(shape, d, seed, device):
    b, sq, sk, h = shape
    g = torch.Generator(device=device).manual_seed(seed)
    return [torch.randn(b, h, n, d, generator=g, device=device).transpose(1, 2) for n in (sq, sk, sk)]


def some_heads(h):
    return sorted({0, h // 2, h - 1})


def reference(q, k, v, causal, heads, scale=None):
    d = q.shape[-1]
    return attention(*(values(x[:, :, heads]) for x in (q, k, v)), d ** -0.5 if scale is None else scale, causal)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("shape", SHAPES)
def test_error_against_64_bits(cuda, shape, d, causal):
    """A logit is a sum of d products, each off by at most 2^-23 + 2^-23 + 2^-22 of its
    size (the two splits and the dropped low.low term, for values within 2^12 of the
    largest, as nearly all of these are), and of fp32 additions; p and v are split alike.
    With sums of random signs the 2-norm error stays a few 2^-24: 2e-6 bounds it at these
    sizes (4e-7 or less is seen).  Values of very different size are below."""
    print(f"f32 split {shape} d={d} causal={causal}", flush=True)
    q, k, v = tensors(shape, d, sum(shape) + d, cuda)
    heads = some_heads(shape[3])
    out = values(flash_attn_func(q, k, v, causal=causal)[:, :, heads])
    ref = reference(q, k, v, causal, heads)
    assert np.linalg.norm(out - ref) <= 2e-6 * np.linalg.norm(ref)


RANGES = {"large": lambda q, k, v: (q * 2.0 ** 30, k * 2.0 ** -30, v * 2.0 ** 39),
          "past the range": lambda q, k, v: (q * 2.0 ** 60, k * 2.0 ** -60, v * 2.0 ** 80),
          "tiny": lambda q, k, v: (q, k, v * 2.0 ** -100),
          "late large key": lambda q, k, v: (q * 0.1, _scaled(k, -3, 100.0), _scaled(v, -3, 1e5)),
          "late small keys": lambda q, k, v: (q, _scaled(k, slice(96, None), 1e-6), _scaled(v, slice(96, None), 1e-7)),
          "first tile zero": lambda q, k, v: (q, _scaled(k, slice(0, 32), 0.0), _scaled(v, slice(0, 32), 0.0)),
          "all zero": lambda q, k, v: (q * 0, k * 0, v * 0)}


def _scaled(x, rows, f):
    x = x.clone()
    x[:, rows] *= f
    return x


@pytest.mark.parametrize("shape", [(1, 150, 300, 3), (1, 64, 1500, 3), (1, 600, 600, 110)])
@pytest.mark.parametrize("what", list(RANGES))
@pytest.mark.parametrize("d", [32, 64, 128])
def test_values_out_of_the_splits_range(cuda, d, what, shape):
    print(f"f32 range {what} {shape} d={d}", flush=True)
    q, k, v = RANGES[what](*tensors(shape, d, d, cuda))
    heads = some_heads(shape[3])
    out = values(flash_attn_func(q, k, v, causal=True)[:, :, heads])
    ref = reference(q, k, v, True, heads)
    # 2e-6 as above, of the largest values: a dominant key carries its error into all of a row
    assert np.isfinite(out).all()
    assert np.linalg.norm(out - ref) <= 2e-6 * max(np.linalg.norm(ref), 1e-300)


@pytest.mark.parametrize("first", [2.0 ** 10, 0.0])
@pytest.mark.parametrize("shape", [(1, 150, 300, 3), (1, 64, 1500, 3), (1, 600, 600, 110)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_values_far_below_the_first_tiles(cuda, d, shape, first):
    """The first tile's keys get no weight, and the values behind them lie below the
    smallest fp16 at that tile's scale (or at the scale of a tile of zeros): they are
    what the rows consist of, not zeros."""
    print(f"f32 below the first tile's {first} {shape} d={d}", flush=True)
    q, k, v = tensors(shape, d, d + 3, cuda)
    q[..., 0], k[..., 0] = 40.0, 0.0
    k[:, :32, :, 0] = -100.0  # a logit of -4000 d^-0.5: e^-353 of the others at most
    v[:, :32] *= first
    v[:, 32:] *= 2.0 ** -38
    heads = some_heads(shape[3])
    out = values(flash_attn_func(q, k, v)[:, :, heads])
    ref = reference(q, k, v, False, heads)
    assert np.linalg.norm(out - ref) <= 2e-6 * np.linalg.norm(ref)


def _channel(x, c, f):
    x = x.clone()
    x[..., c] *= f
    return x


def _logit(q, k, keys, x):
    """Logits of x on top for those keys, 0 for the others."""
    q, k = q.clone(), k.clone()
    q[..., 0], k[..., 0] = 4.0, 0.0
    k[:, keys, :, 0] = x / 4 * q.shape[-1] ** 0.5
    return q, k


def _sink(q, k, v, r):
    return *_logit(q * 0.3, k, 40, math.log(k.shape[1] / r)), _scaled(v, 40, 0.0)


def _one_hot(q, k, v, r):
    d = v.shape[-1]
    one = torch.eye(d, device=v.device)[torch.arange(v.shape[1], device=v.device) % d]
    return *_logit(q * 0.3, k, slice(3, None, d), math.log(r)), one[None, :, None].expand_as(v)


# what lies r below the rest, and how large a logit that takes
SPREADS = {"a channel of v": (lambda q, k, v, r: (q, k, _channel(v, 5, r)), 0),
           "the other channels of v": (lambda q, k, v, r: (q, k, _channel(v, 5, 1 / r)), 0),
           "every other key of v": (lambda q, k, v, r: (q, k, _scaled(v, slice(0, None, 2), r)), 0),
           "the keys of v that weigh": (lambda q, k, v, r: (*_logit(q, k, slice(1, None, 2), -60),
                                                            _scaled(v, slice(0, None, 2), r)), 60),
           "the first row of v": (lambda q, k, v, r: (q, k, _scaled(v, 0, r)), 0),
           "a channel of k": (lambda q, k, v, r: (_channel(q, 3, 1 / r), _channel(k, 3, r), v), 0),
           "a channel of q": (lambda q, k, v, r: (_channel(q, 3, r), _channel(k, 3, 1 / r), v), 0),
           "every other key": (lambda q, k, v, r: (q, _scaled(k, slice(0, None, 2), r), v), 0),
           "the weight of all but a key of zeros": (_sink, math.log),
           "the weight of one channel's keys": (_one_hot, math.log)}


@pytest.mark.parametrize("r", [1e-3, 1e-5, 1e-7, 1e-11])
@pytest.mark.parametrize("shape", [(1, 150, 300, 2), (1, 64, 1500, 3), (1, 600, 600, 110)])
@pytest.mark.parametrize("what", list(SPREADS))
@pytest.mark.parametrize("d", [32, 64, 128])
def test_values_of_very_different_size(cuda, d, what, shape, r):
    """Small values beside large ones, r apart, that the large ones do not hide: every
    row's and every channel's error in its own norm.  A row or channel alone sees less
    averaging than the whole output, so 3e-6 (the 32-bit MFMAs: up to 1.8e-6); a logit x
    is a sum of d products, whose roundings, of 2^-24 x each, reach p as they are."""
    make, size = SPREADS[what]
    print(f"f32 spread {what} {r} {shape} d={d}", flush=True)
    heads = some_heads(shape[3])
    q, k, v = make(*tensors(shape, d, d + 4, cuda), r)
    x = size if isinstance(size, int) else abs(size(r / shape[2]))
    tol = 3e-6 + x * d ** 0.5 * 2.0 ** -23
    for causal in (False, True):
        out = values(flash_attn_func(q, k, v, causal=causal)[:, :, heads])
        ref = reference(q, k, v, causal, heads)
        rows = (what != "the other channels of v") * np.linalg.norm(out - ref, axis=3) / np.linalg.norm(ref, axis=3)
        channels = np.linalg.norm(out - ref, axis=1) / np.linalg.norm(ref, axis=1)
        assert rows.max() <= tol and channels.max() <= tol, (rows.max(), channels.max(), tol)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("shape", [(1, 40, 31, 3), (1, 40, 16, 3), (1, 40, 15, 3), (1, 40, 5, 3), (1, 17, 32, 2),
                                   (2, 33, 60, 3), (1, 40, 2049, 3), (1, 40, 2064, 3), (1, 300, 260, 30)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_a_channel_in_few_keys(cuda, d, shape, causal):
    """No whole key tile, one and a part of one, splits that hold a part alone (too few
    keys to judge a channel by, and just enough), and more rows than keys."""
    q, k, v = tensors(shape, d, d + 6, cuda)
    v = _channel(v, 5, 1e-7)
    heads = some_heads(shape[3])
    out, ref = values(flash_attn_func(q, k, v, causal=causal)[:, :, heads]), reference(q, k, v, causal, heads)
    channels = np.linalg.norm(out - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert channels.max() <= 3e-6, channels.max()


@pytest.mark.parametrize("shape", [(1, 150, 300, 2), (1, 64, 1500, 3), (1, 600, 600, 110)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_infinite_and_nan_values(cuda, d, shape):
    """A key whose logit is -inf for every query drops out; a NaN query row is NaN and
    the others of its block keep their values; a NaN value reaches only rows that see
    its key, in its dims."""
    q, k, v = tensors(shape, d, d + 1, cuda)
    q = q.abs() + 0.1
    heads = [0]
    k[:, 70, :, 3] = float("-inf")
    q[:, 5] = float("nan")
    out = values(flash_attn_func(q, k, v)[:, :, heads])
    keep = [i for i in range(shape[2]) if i != 70]
    ref = reference(q, k[:, keep], v[:, keep], False, heads)
    rows = [i for i in range(shape[1]) if i != 5]
    if shape[1] != 64:  # split keys: the combine takes a row of no comparable logit as one without keys
        assert np.isnan(out[:, 5]).all()
    assert np.linalg.norm(out[:, rows] - ref[:, rows]) <= 2e-6 * np.linalg.norm(ref[:, rows])
    q, k, v = tensors(shape, d, d + 2, cuda)
    v[:, 100, :, 1] = float("nan")
    out = values(flash_attn_func(q, k, v)[:, :, heads])
    assert np.isnan(out[..., 1]).all() and np.isfinite(np.delete(out, 1, -1)).all()


@pytest.mark.parametrize("scale", [-0.3, 0.0, 4.0])
def test_softmax_scales(cuda, scale):
    q, k, v = tensors((1, 150, 300, 2), 64, 9, cuda)
    for causal in (False, True):
        out = values(flash_attn_func(q, k, v, softmax_scale=scale, causal=causal))
        ref = reference(q, k, v, causal, [0, 1], scale)
        # logits of size |scale| * 64^0.5 * few: their rounding reaches p times as large
        assert np.linalg.norm(out - ref) <= (2e-6 + 2e-6 * abs(scale) * 8) * np.linalg.norm(ref)
