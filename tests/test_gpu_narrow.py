"""The projections around the lines where the launchers change kernels: the
16-row-tile kernels of small waves (gemm_narrow.hpp) and the 32 x 32-tile
kernels, each against the oracle bit for bit. Sizes are the edges: one row, a
row tile's remainder, one past it, the last size of the narrow kernels and
the first of the wide ones, block counts that fill a chunk, overrun it or
leave a part of one, and widths that leave a part of a column tile."""
import numpy as np
import pytest

import gguf_py
import oracle_lib as OL
from oracle_lib import HEAD_DIM, N_EMBD, N_FF, quantize_q8_0
from test_gpu_ops import (bits, dev, device_q8, device_weights, empty, host, oracle_gelu_q8, oracle_qk_norm_rope,
                          run_geglu)

pytestmark = pytest.mark.gpu


def operands(n, m, k, seed, std=0.02):
    rng = np.random.default_rng(seed)
    return (quantize_q8_0((rng.standard_normal((m, k)) * std).astype(np.float32)),
            quantize_q8_0(rng.standard_normal((n, k)).astype(np.float32)))


@pytest.mark.parametrize("n,m,k", [
    (1, 768, 768), (15, 33, 32), (16, 768, 1152), (17, 40, 800), (31, 100, 1184), (48, 70, 1600),
    (512, 896, 768),    # 32 x 56 tiles: the last narrow size
    (512, 912, 224), (513, 896, 192), (700, 768, 320),  # wide ones; 7 and 10 blocks take the loop's tail
    # both sides of the line at one block, a third and two thirds of a chunk, one block in the second and third chunk
    (64, 288, 32), (80, 288, 32), (192, 768, 256), (208, 768, 256), (512, 768, 512), (513, 768, 512),
    (304, 768, 1568), (305, 768, 1568), (304, 768, 3104), (321, 768, 3104)])
def test_gemm_edges(eg2, gpu, n, m, k):
    import torch

    w, xb = operands(n, m, k, n + m + k)
    y = empty((n, m + 3), torch.float32, gpu)
    eg2.ops.gemm_q8(*device_q8(eg2, xb, k, gpu), *device_weights(eg2, w, k, gpu), y, m)
    got = host(y)
    assert np.array_equal(bits(got[:, :m]), bits(OL.gemm_q8_0(w, xb)))
    assert (got[:, m:] == 0).all()


@pytest.mark.parametrize("n,ff,k,tied", [(1, N_FF, N_EMBD, False), (15, 64, 416, False), (33, 96, 832, True),
                                         (192, N_FF, N_EMBD, True), (193, N_FF, N_EMBD, True), (224, 64, 160, False),
                                         # one round of other widths and block counts, and what is past it or has
                                         # too few blocks
                                         (224, N_FF, N_EMBD, False), (225, N_FF, N_EMBD, False), (2048, 64, 256, True),
                                         (2049, 64, 256, False), (17, 64, 224, False), (112, N_FF, 1024, False),
                                         (113, N_FF, 1024, False), (40, 2304, 992, False),
                                         # the wide kernel up to a workgroup per CU and past it
                                         (448, N_FF, N_EMBD, True), (449, N_FF, N_EMBD, True), (450, N_FF, 160, False)])
def test_geglu_edges(eg2, gpu, n, ff, k, tied):
    """tied: repeated weight rows, so blocks with equal maxima."""
    rng = np.random.default_rng(n + ff)
    wg, wu = ((rng.standard_normal((ff, k)) * 0.04).astype(np.float32) for _ in range(2))
    if tied:
        for w in (wg, wu):
            w[1:32] = w[0]
            w[33:64:2] = w[32:64:2]
    wg, wu = quantize_q8_0(wg), quantize_q8_0(wu)
    xb = quantize_q8_0(rng.standard_normal((n, k)).astype(np.float32))
    q, d = run_geglu(eg2, gpu, xb, wg, wu, k, ff, n + 2)
    wq, wd = oracle_gelu_q8(OL.gemm_q8_0(wg, xb), OL.gemm_q8_0(wu, xb))
    assert np.array_equal(q, wq)
    assert np.array_equal(bits(d[:, :n].T), bits(wd))
    assert (d[:, n:] == -3.0).all()


@pytest.mark.parametrize("n,k", [(1, 768), (17, 224), (256, 768), (257, 768), (260, 224)])
def test_qkv_rope_edges(eg2, gpu, n, k):
    """The operator, which is one kernel at every size (a recorded wave's
    projection changes kernels at 256 rows: test_wave_edges)."""
    import torch

    rng = np.random.default_rng(n + k)
    w, xb = operands(n, eg2.QKV_COLS, k, n + k, 0.05)
    qw, kw = ((1 + 0.1 * rng.standard_normal(HEAD_DIM)).astype(np.float32) for _ in range(2))
    pos = rng.integers(0, 2048, n).astype(np.int32)
    out = torch.full((n + 1, eg2.QKV_COLS), 7.0, device=gpu)
    eg2.ops.gemm_q8_qkv_rope(*device_q8(eg2, xb, k, gpu), *device_weights(eg2, w, k, gpu), n, dev(qw, gpu),
                             dev(kw, gpu), dev(eg2.rope_table(1e4), gpu), dev(pos, gpu), 1e-6, out)
    got = host(out)
    assert np.array_equal(bits(got[:n]), bits(oracle_qk_norm_rope(OL.gemm_q8_0(w, xb), qw, kw, pos, 1e4)))
    assert (got[n] == 7.0).all()


@pytest.fixture(scope="module")
def encoder(eg2, gpu, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("narrow") / "model.gguf")
    eg2.synth_gguf(path, seed=9, n_layer=2, dense_head=True, sliding_window=64, sliding_window_pattern=2,
                   rope_base_full=1e6, rope_base_swa=1e4, threads=8)
    enc = eg2.Encoder(path)
    yield enc, gguf_py.oracle_model(path)
    enc.close()


@pytest.mark.parametrize("tokens", [50, 64, 65, 192, 193, 224, 225, 256, 257])
@pytest.mark.parametrize("texts", [1, 7])
def test_wave_edges(encoder, tokens, texts):
    """Waves on both sides of the lines where the recorded layers change
    kernels: the smallest that is not a short wave (64 rows), gate|up (up to
    192 rows the narrow kernel) and Q|K|V (up to 256 rows two kernels)."""
    enc, model = encoder
    rng = np.random.default_rng(tokens + texts)
    cuts = np.sort(rng.choice(np.arange(1, tokens), texts - 1, replace=False))
    offsets = np.concatenate([[0], cuts, [tokens]])
    ids = rng.integers(0, OL.VOCAB, tokens).astype(np.int32)
    want = OL.forward(model, ids, offsets.astype(np.uint64), threads=8)
    for _ in range(2):  # the second call replays the graph
        assert np.array_equal(enc.batch(ids, offsets), want)
