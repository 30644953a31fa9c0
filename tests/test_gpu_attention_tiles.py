"""The by-name attention's tiled kernel (kernels_abi.hip), taken for the whole
grid of 512 tokens or more, against a float64 softmax at the reference
operator test's tolerance (tests/kernels.cpp:114-137): the first size that
takes it and the last that does not, a partial last tile, sequences of one
token and of more key blocks than waves, tiles that straddle sequences,
tokens with no key, ranges unlike their neighbours', and windows."""
import numpy as np
import pytest

from test_gpu_operators import attention_reference, dev, host

pytestmark = pytest.mark.gpu
OPS = {"eg2_attention256": (4, 256, 512, 2), "eg2_attention512": (4, 512, 512, 4), "eg2_attention256x3": (3, 256, 256, 3)}


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("lens,window,odd", [([511], 0, False), ([512], 0, False), ([1, 300, 17, 211, 1], 0, True),
                                             ([1, 300, 17, 211, 1], 50, True), ([16] * 33, 3, False)],
                         ids=["511", "512", "ragged", "ragged-w50", "33x16-w3"])
def test_tiled_attention_against_float64(eg2, gpu, op, lens, window, odd):
    import torch

    heads, d, kvs, group = OPS[op]
    n = sum(lens)
    rng = np.random.default_rng(n + window + d)
    starts = np.concatenate([[0], np.cumsum(lens)])
    bounds = np.array([(starts[s], starts[s + 1]) for s in range(len(lens)) for _ in range(lens[s])], np.uint32)
    if odd:
        bounds[40] = (7, 7)       # no key
        bounds[41] = (9, 3)       # none either
        bounds[300] = (2, 450)    # a range of its own
        bounds[n - 1] = (0, n)
    q = (rng.standard_normal(n * heads * d) / np.sqrt(d)).astype(np.float32)
    k = rng.standard_normal(n * kvs).astype(np.float32)
    v = rng.standard_normal(n * kvs).astype(np.float32)
    y = torch.full((n * heads * d,), float("nan"), device=gpu)
    qd, kd, vd, bd = dev(q, gpu), dev(k, gpu), dev(v, gpu), dev(bounds.reshape(-1).view(np.int32), gpu)
    rec = eg2.EgAttention(y.data_ptr(), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), bd.data_ptr(), n, window)
    eg2.ops.op(op, rec, heads * n, 64)
    got = host(y).reshape(n, heads, d)
    empty = []
    full = bounds.copy()
    for t in range(n):
        lo, hi = int(bounds[t, 0]), int(bounds[t, 1])
        if window:
            lo, hi = max(lo, t - window), min(hi, t + window + 1)
        if hi <= lo:
            empty.append(t)
            full[t] = (t, t + 1)  # the reference needs a key; compared with zero below
    want = attention_reference(q, k, v, full.reshape(-1), n, heads, d, kvs, lambda h: h // group, window)
    want = want.reshape(n, heads, d)
    want[empty] = 0.0
    assert np.abs(got - want).max() <= 2e-5
    assert (got[empty] == 0).all()


@pytest.mark.parametrize("op", list(OPS))
def test_non_finite_values_stay_in_their_sequence(eg2, gpu, op):
    """An infinite and a NaN value row: the sequence that holds them is not
    finite, and the others are what they are without them. (A tile that meets
    such values in a partial block is computed in the per-row form, so its rows
    may differ by both forms' tolerance, 2 x 2e-5.)"""
    import torch

    heads, d, kvs, _ = OPS[op]
    lens = [250, 21, 9, 300]
    n = sum(lens)
    rng = np.random.default_rng(d)
    starts = np.concatenate([[0], np.cumsum(lens)])
    bounds = np.array([(starts[s], starts[s + 1]) for s in range(len(lens)) for _ in range(lens[s])], np.uint32)
    q, k, v = ((rng.standard_normal(n * w) * 0.1).astype(np.float32) for w in (heads * d, kvs, kvs))
    bad = v.reshape(n, kvs).copy()
    bad[252, 5] = np.inf
    bad[270, 300 % kvs] = np.nan
    out = []
    for values in (v, bad):
        y = torch.full((n * heads * d,), float("nan"), device=gpu)
        t = [dev(a, gpu) for a in (q, k, values.reshape(-1), bounds.reshape(-1).view(np.int32))]
        rec = eg2.EgAttention(y.data_ptr(), *(a.data_ptr() for a in t), n, 0)
        eg2.ops.op(op, rec, heads * n, 64)
        out.append(host(y).reshape(n, heads * d))
    rows = np.r_[0:250, 271:n]
    assert np.abs(out[0][rows] - out[1][rows]).max() <= 4e-5
    assert not np.isfinite(out[1][250:271]).all(axis=1).any()


def softmax_reference(q, k, v, bounds, n, heads, d, kvs, group, window):
    """float64 attention where a score of -inf weighs nothing, and a NaN or
    +inf score, or no score above -inf, makes the row NaN."""
    out = np.zeros((n, heads, d))
    q, k, v = q.reshape(n, heads, d).astype(np.float64), k.reshape(n, kvs), v.reshape(n, kvs).astype(np.float64)
    for t in range(n):
        lo, hi = int(bounds[t, 0]), int(bounds[t, 1])
        if window:
            lo, hi = max(lo, t - window), min(hi, t + window + 1)
        for h in range(heads):
            cols = slice(h // group * d, (h // group + 1) * d)
            with np.errstate(all="ignore"):
                s = (k[lo:hi, cols].astype(np.float64) * q[t, h]).sum(1)
                s[s < -3.5e38] = -np.inf  # past the range of 32 bits
                w = np.exp(s - s.max())
                out[t, h] = (w / w.sum()) @ v[lo:hi, cols]
    return out


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("n", [511, 512, 640])
@pytest.mark.parametrize("window", [0, 20])
def test_scores_of_minus_infinity_weigh_nothing(eg2, gpu, op, n, window):
    """Keys whose score is -inf, by an infinite element or by a dot product
    past the range of 32 bits: alone in a 16-key block of their text (its 17th
    and 33rd key), as a text's only key, and 70 in a row at a text's start, so
    that whole blocks and chunks of a row score -inf before a finite one; and
    keys that score +inf or NaN, which make their text's rows NaN."""
    import torch

    heads, d, kvs, group = OPS[op]
    lens = [17, 33, 60, 1, n - 111]
    starts = np.concatenate([[0], np.cumsum(lens)])
    bounds = np.array([(starts[s], starts[s + 1]) for s in range(len(lens)) for _ in range(lens[s])], np.uint32)
    rng = np.random.default_rng(n + d + window)
    q = (rng.standard_normal((n, heads, d)) / np.sqrt(d)).astype(np.float32)
    q[:, :, 3] = 2.0
    k, v = (rng.standard_normal((n, kvs)).astype(np.float32) for _ in range(2))
    k[16, 3::d] = -np.inf
    k[49, 3::d] = -3e38
    k[80, 3::d] = np.inf
    k[110, 3::d] = -np.inf
    k[111:181, 3::d] = -np.inf
    if window:
        k[300, 3::d] = np.nan
    y = torch.full((n * heads * d,), 7.0, device=gpu)
    t = [dev(a, gpu) for a in (q, k, v, bounds.reshape(-1).view(np.int32))]
    rec = eg2.EgAttention(y.data_ptr(), *(a.data_ptr() for a in t), n, window)
    eg2.ops.op(op, rec, heads * n, 64)
    got = host(y).reshape(n, heads, d)
    want = softmax_reference(q, k, v, bounds, n, heads, d, kvs, group, window)
    assert np.isnan(want[110]).all() and np.isfinite(want[:50]).all() and np.isfinite(want[400:]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.nanmax(np.abs(got - want)) <= 2e-5


def short_lens(seed, total, top):
    rng, out = np.random.default_rng(seed), []
    while sum(out) < total:
        out.append(int(rng.integers(1, top + 1)))
    return out


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("lens,window", [([1] * 513, 0), ([3] * 200, 0), ([8] * 70, 2), (short_lens(1, 600, 15), 0),
                                         (short_lens(2, 600, 15), 4), ([16] * 32, 0), ([17] * 31, 0), ([24, 40] * 9, 0),
                                         ([32] * 17, 0), ([33] * 16, 0), ([64] * 9, 0), ([65] * 8, 0), ([600], 1),
                                         ([600], 24), ([600], 25), (short_lens(3, 700, 40), 0)],
                         ids=lambda v: f"{len(v)}x{v[0]}" if isinstance(v, list) else f"w{v}")
def test_short_texts_and_narrow_windows(eg2, gpu, op, lens, window):
    """Tiles that reach few keys: texts shorter than a tile and up to a few
    blocks, aligned with the tiles and not, and windows that leave as few."""
    import torch

    heads, d, kvs, group = OPS[op]
    n = sum(lens)
    starts = np.concatenate([[0], np.cumsum(lens)])
    bounds = np.array([(starts[s], starts[s + 1]) for s in range(len(lens)) for _ in range(lens[s])], np.uint32)
    rng = np.random.default_rng(n + d + window)
    q = (rng.standard_normal((n, heads, d)) / np.sqrt(d)).astype(np.float32)
    k, v = (rng.standard_normal((n, kvs)).astype(np.float32) for _ in range(2))
    y = torch.full((n * heads * d + 64,), 7.0, device=gpu)
    t = [dev(a, gpu) for a in (q, k, v, bounds.reshape(-1).view(np.int32))]
    rec = eg2.EgAttention(y.data_ptr(), *(a.data_ptr() for a in t), n, window)
    eg2.ops.op(op, rec, heads * n, 64)
    got = host(y)
    want = softmax_reference(q, k, v, bounds, n, heads, d, kvs, group, window)
    assert np.abs(got[:-64].reshape(n, heads, d) - want).max() <= 2e-5
    assert (got[-64:] == 7.0).all()


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("n,width", [(512, 1), (528, 8), (1100, 8), (1100, 100)])
def test_scattered_ranges(eg2, gpu, op, n, width):
    """Neighbouring tokens with key ranges far apart."""
    import torch

    heads, d, kvs, group = OPS[op]
    rng = np.random.default_rng(n + width)
    lo = rng.integers(0, n - width + 1, n)
    bounds = np.stack([lo, lo + width], 1).astype(np.uint32)
    q = (rng.standard_normal((n, heads, d)) / np.sqrt(d)).astype(np.float32)
    k, v = (rng.standard_normal((n, kvs)).astype(np.float32) for _ in range(2))
    y = torch.full((n * heads * d,), 7.0, device=gpu)
    t = [dev(a, gpu) for a in (q, k, v, bounds.reshape(-1).view(np.int32))]
    rec = eg2.EgAttention(y.data_ptr(), *(a.data_ptr() for a in t), n, 0)
    eg2.ops.op(op, rec, heads * n, 64)
    want = softmax_reference(q, k, v, bounds, n, heads, d, kvs, group, 0)
    assert np.abs(host(y).reshape(n, heads, d) - want).max() <= 2e-5


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("length", [7, 40, 130])
def test_packing_moves_rounding_only(eg2, gpu, op, length):
    """A text alone (the per-row form) and inside a packing of 512 tokens and
    more, at several places in it: equal but for rounding (each is within 2e-5
    of the exact result)."""
    import torch

    heads, d, kvs, _ = OPS[op]
    rng = np.random.default_rng(length + d)
    text = [(rng.standard_normal((length, w)) * s).astype(np.float32)
            for w, s in ((heads * d, d ** -0.5), (kvs, 1), (kvs, 1))]
    out = []
    for before, after in ((0, 0), (0, 600), (3, 600), (300, 250), (509, 0)):
        n = before + length + after
        q, k, v = (np.concatenate([rng.standard_normal((before, t.shape[1])).astype(np.float32), t,
                                   rng.standard_normal((after, t.shape[1])).astype(np.float32)]) for t in text)
        b = np.array([(0, before)] * before + [(before, before + length)] * length +
                     [(before + length, n)] * after, np.uint32)
        y = torch.full((n * heads * d,), 7.0, device=gpu)
        t = [dev(a, gpu) for a in (q, k, v, b.reshape(-1).view(np.int32))]
        rec = eg2.EgAttention(y.data_ptr(), *(a.data_ptr() for a in t), n, 0)
        eg2.ops.op(op, rec, heads * n, 64)
        out.append(host(y).reshape(n, heads * d)[before:before + length])
    for o in out[1:]:
        assert np.abs(o - out[0]).max() <= 4e-5
