"""Waves of up to 48 tokens take fused kernels of their own (short_wave.hpp:
the residual with the next projection, attention in one kernel, rows padded
to a multiple of 16); their embeddings against the oracle bit for bit at the edges:
one token, a full 16-, 32- and 48-row wave and one past each, packings with and
without a padding sequence, sequences of one token, and a window that cuts
into the sequences on two layers of three."""
import json
import os

import numpy as np
import pytest

import gguf_py
import oracle_lib as OL

pytestmark = pytest.mark.gpu

LENS = [[1], [11], [16], [17], [31], [32], [33], [1] * 16, [1] * 17, [3, 9, 4], [20, 12], [5, 8, 2, 9, 1], [16, 1],
        [47], [48], [49], [33, 15], [30, 1, 10], [1] * 48, [7] * 6]


@pytest.fixture(scope="module", params=[0, 8])
def windowed(request, eg2, gpu, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("short") / f"w{request.param}.gguf")
    eg2.synth_gguf(path, seed=5, n_layer=3, dense_head=True, sliding_window=request.param, sliding_window_pattern=2,
                   rope_base_full=1e6, rope_base_swa=1e4, threads=8)
    enc = eg2.Encoder(path)
    yield enc, gguf_py.oracle_model(path)
    enc.close()


@pytest.mark.parametrize("lens", LENS, ids=lambda v: "-".join(map(str, v)) if len(v) < 8 else f"{len(v)}x1")
def test_short_wave_equals_oracle(windowed, lens):
    enc, model = windowed
    ids = np.random.default_rng(sum(lens) + len(lens)).integers(0, OL.VOCAB, sum(lens)).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(lens)])
    want = OL.forward(model, ids, offsets.astype(np.uint64), threads=8)
    for _ in range(2):  # the second call replays the graph
        assert np.array_equal(enc.batch(ids, offsets), want)


def test_profile_names_of_a_short_wave(eg2, gpu, tmp_path, capfd):
    """EG2_HIP_PROFILE=1 on a wave of up to 48 tokens: the fused launches under
    names of their own, each with a positive time; the embeddings unchanged."""
    path = str(tmp_path / "m.gguf")
    eg2.synth_gguf(path, seed=5, n_layer=3, dense_head=True, rope_base_full=1e6, rope_base_swa=1e4, threads=8)
    ids = np.random.default_rng(0).integers(0, OL.VOCAB, 30).astype(np.int32)
    enc = eg2.Encoder(path)
    want = enc.batch(ids, [0, 11, 30])
    enc.close()
    os.environ["EG2_HIP_PROFILE"] = "1"
    try:
        enc = eg2.Encoder(path)
        capfd.readouterr()
        got = enc.batch(ids, [0, 11, 30])
        enc.close()
    finally:
        del os.environ["EG2_HIP_PROFILE"]
    assert np.array_equal(got, want)
    line, = [x for x in capfd.readouterr().err.splitlines() if x.startswith("HIP_PROFILE ")]
    ms = json.loads(line[len("HIP_PROFILE "):])["command_ms"]
    assert set(ms) == {"embed", "gemm_qkv", "residual_gemm_qkv", "attention", "gemm_o", "residual_gemm_gate_up_geglu",
                       "gemm_down", "residual", "output_norm", "pool", "dense_quant", "dense_2", "dense_3", "dense_l2"}
    assert all(v > 0 for v in ms.values())
