"""The by-name projections' two forms (kernels_abi.hip): the bf16-part form of
aligned operands with k a multiple of 32, against a float64 product and
against the general form (reached by moving an operand off its alignment), at
the sizes where it can go wrong: partial tiles both ways, odd block counts
(Q8_0 blocks then start on both halves of a word), one step and a step count
that leaves waves idle; and infinities, NaN and a Q8_0 dot that overflows
before its scale, which the general form must decide, bit for bit."""
import numpy as np
import pytest

from test_gpu_operators import MM_VARIANTS, dev, encode_weights, host

pytestmark = pytest.mark.gpu
TYPES = [0, 1, 8, 30]


def run(eg2, gpu, variant, x, raw, wtype, m, x_shift=0, w_shift=0):
    """x_shift floats and w_shift bytes put before the operands."""
    import torch

    name, width, height, _ = variant
    n, k = x.shape
    xd = dev(np.concatenate([np.zeros(x_shift, np.float32), x.reshape(-1)]), gpu)
    wd = dev(np.concatenate([np.zeros(w_shift, np.uint8), raw.reshape(-1).view(np.uint8)]), gpu)
    yd = torch.full((n, m), float("nan"), dtype=torch.float32, device=gpu)
    rec = eg2.EgMM(yd.data_ptr(), xd.data_ptr() + 4 * x_shift, wd.data_ptr() + w_shift, n, k, m, wtype)
    eg2.ops.op(name, rec, ((m + width - 1) // width, (n + height - 1) // height), 256)
    return host(yd)


@pytest.mark.parametrize("variant", MM_VARIANTS[:3], ids=[v[0] for v in MM_VARIANTS[:3]])
@pytest.mark.parametrize("wtype", TYPES)
@pytest.mark.parametrize("shape", [(1, 32, 1), (17, 96, 35), (65, 160, 130), (130, 768, 67)])
def test_aligned_form_against_float64_and_general(eg2, gpu, variant, wtype, shape):
    n, k, m = shape
    rng = np.random.default_rng(n + k + wtype)
    x = (rng.standard_normal((n, k)) * 10.0 ** rng.uniform(-3, 3, (n, 1))).astype(np.float32)
    raw, dec = encode_weights((rng.standard_normal((m, k)) * 0.05).astype(np.float32), wtype)
    x64, w64 = x.astype(np.float64), dec.astype(np.float64)
    want, mag = x64 @ w64.T, np.abs(x64) @ np.abs(w64).T
    got = run(eg2, gpu, variant, x, raw, wtype, m)
    general = run(eg2, gpu, variant, x, raw, wtype, m, x_shift=1)
    # A 32-bit sum of k products: at most k roundings of 2^-24 each.
    assert np.all(np.abs(got - want) <= k * 2.0 ** -24 * mag)
    # Precision is not lost against the general form: the rms of the errors in
    # units of sum |x w| (over enough outputs to be steady).
    if n * m >= 500:
        rms = lambda y: np.sqrt((((y - want) / mag) ** 2).mean())
        assert rms(got) <= 1.1 * rms(general)
    if wtype == 8:  # blocks at the other parity, and at odd addresses (the general form)
        assert np.array_equal(run(eg2, gpu, variant, x, raw, wtype, m, w_shift=2), got)
        assert np.array_equal(run(eg2, gpu, variant, x, raw, wtype, m, w_shift=1), general)


@pytest.mark.parametrize("variant", MM_VARIANTS[:3], ids=[v[0] for v in MM_VARIANTS[:3]])
@pytest.mark.parametrize("wtype", TYPES)
def test_non_finite_sums_take_the_general_form(eg2, gpu, variant, wtype):
    n, k, m = 70, 128, 70
    rng = np.random.default_rng(wtype)
    w = (rng.standard_normal((m, k)) * 0.05).astype(np.float32)
    w[3, :32] = 0.0
    raw, _ = encode_weights(w, wtype)
    for bad in (np.inf, -np.inf, np.nan, np.uint32(0x7F800001).view(np.float32), np.float32(3e38)):
        x = rng.standard_normal((n, k)).astype(np.float32)
        x[5, 7] = bad
        got = run(eg2, gpu, variant, x, raw, wtype, m)
        general = run(eg2, gpu, variant, x, raw, wtype, m, x_shift=1)
        assert np.array_equal(np.isnan(got), np.isnan(general))
        assert np.array_equal(got[5], general[5], equal_nan=True) or bad == np.float32(3e38)
        ok = np.isfinite(general)
        assert np.array_equal(ok, np.isfinite(got)) and np.allclose(got[ok], general[ok], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("wtype", TYPES)
@pytest.mark.parametrize("k", [32, 64, 96, 160, 288])
def test_few_steps_keep_the_general_form_s_precision(eg2, gpu, wtype, k):
    """A 16 x 16 tile over a few 32-deep steps, where the split of the chains
    over the waves is uneven: 64k outputs, so the rms errors of two equally
    good orders agree within a few parts in a thousand."""
    n = m = 256
    rng = np.random.default_rng(k + wtype)
    x = rng.standard_normal((n, k)).astype(np.float32)
    raw, dec = encode_weights((rng.standard_normal((m, k)) * 0.05).astype(np.float32), wtype)
    want = x.astype(np.float64) @ dec.astype(np.float64).T
    rms = lambda y: np.sqrt(((y - want) ** 2).mean())
    got, general = (run(eg2, gpu, MM_VARIANTS[0], x, raw, wtype, m, x_shift=s) for s in (0, 1))
    assert rms(got) <= 1.01 * rms(general)


@pytest.mark.parametrize("variant", MM_VARIANTS[:3], ids=[v[0] for v in MM_VARIANTS[:3]])
@pytest.mark.parametrize("wtype", TYPES)
def test_small_activations_keep_their_bits(eg2, gpu, variant, wtype):
    """Rows of 2^-100 to 2^-126: the lowest part of such a value is below what
    bf16 holds. Weights of 2^12, so that the sums are normal numbers."""
    n, k, m = 70, 256, 70
    rng = np.random.default_rng(wtype)
    x = rng.standard_normal((n, k)) * 2.0 ** -np.linspace(100, 126, n)[:, None]
    x[::7] = rng.standard_normal((len(x[::7]), k))  # ordinary rows between them
    x = x.astype(np.float32)
    w = rng.standard_normal((m, k)) * 2.0 ** 12
    raw, dec = encode_weights(w.astype(np.float32), wtype)
    x64, w64 = x.astype(np.float64), dec.astype(np.float64)
    want, mag = x64 @ w64.T, np.abs(x64) @ np.abs(w64).T
    got, general = (run(eg2, gpu, variant, x, raw, wtype, m, x_shift=s) for s in (0, 1))
    rms = lambda y: np.sqrt((((y - want) / mag) ** 2).mean())
    assert np.all(np.abs(got - want) <= k * 2.0 ** -24 * mag)
    assert rms(got) <= 1.1 * rms(general)


@pytest.mark.parametrize("variant", MM_VARIANTS[:3], ids=[v[0] for v in MM_VARIANTS[:3]])
@pytest.mark.parametrize("wtype", TYPES)
def test_rows_do_not_depend_on_their_neighbours(eg2, gpu, variant, wtype):
    """NaN, infinite, overflowing and tiny rows: the others keep their bits."""
    n, k, m = 70, 128, 70
    rng = np.random.default_rng(wtype)
    raw, _ = encode_weights((rng.standard_normal((m, k)) * 0.05).astype(np.float32), wtype)
    x = rng.standard_normal((n, k)).astype(np.float32)
    clean = run(eg2, gpu, variant, x, raw, wtype, m)
    bad = x.copy()
    bad[3, 5], bad[20, 31], bad[41, 100] = np.nan, -np.inf, 3e38
    bad[64] *= np.float32(2.0 ** -118)
    got = run(eg2, gpu, variant, bad, raw, wtype, m)
    rest = np.setdiff1d(np.arange(n), [3, 20, 41, 64])
    assert np.array_equal(got[rest].view(np.uint32), clean[rest].view(np.uint32))


@pytest.mark.parametrize("variant", MM_VARIANTS[:3], ids=[v[0] for v in MM_VARIANTS[:3]])
@pytest.mark.parametrize("wtype", TYPES)
def test_non_finite_weights_take_the_general_form(eg2, gpu, variant, wtype):
    """An infinity or a NaN among the weights (of Q8_0: a block's scale): its
    column is the general form's, bit for bit, and no other column changes."""
    n, k, m = 70, 128, 70
    rng = np.random.default_rng(wtype)
    w = (rng.standard_normal((m, k)) * 0.05).astype(np.float32)
    x = rng.standard_normal((n, k)).astype(np.float32)
    x[9] = 0.0
    raw, _ = encode_weights(w, wtype)
    clean = run(eg2, gpu, variant, x, raw, wtype, m)
    codes = {0: (0x7F800000, 0xFF800000, 0x7FC00000), 30: (0x7F80, 0xFF80, 0x7FC0)}.get(wtype, (0x7C00, 0xFC00, 0x7E00))
    for code in codes:
        bad = raw.reshape(-1).view(np.uint8).copy()
        if wtype == 8:
            bad.reshape(m, k // 32, 34)[17, 2, :2].view(np.uint16)[0] = code
        else:
            bad.view(np.uint32 if wtype == 0 else np.uint16).reshape(m, k)[17, 70] = code
        got = run(eg2, gpu, variant, x, bad, wtype, m)
        general = run(eg2, gpu, variant, x, bad, wtype, m, x_shift=1)
        assert not np.isfinite(general[:, 17]).any()
        assert np.array_equal(got[:, 17], general[:, 17], equal_nan=True)
        other = np.arange(m) != 17
        assert np.array_equal(got[:, other], clean[:, other])
