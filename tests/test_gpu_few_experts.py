"""Batches on few experts: passes of four tokens up to as many as 64 tokens per expert, tiles beyond."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import assert_layer_close, build_layer, oracle_layer

pytestmark = pytest.mark.gpu

PASSES, TILES = "expert_stream_kernel", "expert_stream_kernel_tiles"
# the layers' kernels (tests/test_host_transfers.py holds them to it), E, k, H, F, T, weight in front of the FFN
LAYERS = [(PASSES, 1, 1, 2880, 2880, 34, 0), (PASSES, 1, 1, 2880, 2880, 34, 1), (PASSES, 1, 1, 1152, 7392, 36, 0),
          (PASSES, 1, 1, 4096, 6144, 8, 0), (PASSES, 1, 1, 3808, 8096, 12, 0), (PASSES, 1, 1, 2464, 672, 57, 0),
          (PASSES, 2, 2, 4512, 640, 39, 0), (PASSES, 2, 1, 5312, 5472, 7, 0), (PASSES, 4, 1, 1088, 7328, 29, 1),
          (TILES, 1, 1, 2880, 2880, 24, 0), (TILES, 1, 1, 2880, 2880, 31, 1), (TILES, 2, 2, 1312, 2464, 25, 0),
          (TILES, 4, 4, 2688, 1504, 30, 0)]


@pytest.mark.parametrize("kernel,E,k,H,F,T,wbf", LAYERS)
def test_few_experts(lib, oracle, kernel, E, k, H, F, T, wbf):
    L = synth.LayerInputs(E, k, H, F, seed=T)
    hidden = synth.hidden_states(T, H, seed=E + T)
    with build_layer(lib, L, weight_before_ffn=bool(wbf)) as layer:
        got, pairs = layer.forward(hidden, want_pairs=True)
    want, wpairs = oracle_layer(oracle, L, hidden, weight_before_ffn=bool(wbf))
    assert np.array_equal(pairs[..., 0], wpairs[..., 0])
    assert_layer_close(got, want)


# calls of a single expert that takes every eighth token: k, H, F, T, weight in front
CALLS = [(PASSES, 4, 2880, 2880, 20, 0), (PASSES, 4, 2880, 2880, 28, 1), (PASSES, 4, 2048, 768, 60, 0), (PASSES, 2, 1024, 4096, 33, 1)]


@pytest.mark.parametrize("kernel,k,H,F,T,wbf", CALLS)
def test_an_eighth_of_the_tokens(lib, oracle, kernel, k, H, F, T, wbf):
    rng = np.random.default_rng(T)
    hidden = rng.normal(0, 1, (T, H)).astype(np.float32)
    pairs = np.empty((T, k, 2), np.float32)
    pairs[..., 0], pairs[..., 1] = np.arange(10, 10 + k), rng.uniform(0.1, 0.9, (T, k))
    pairs[::8, k - 1, 0] = 5
    b = [rng.normal(0, 0.01, n).astype(np.float32) for n in (F, F, H)]
    w = [synth.mxfp4_blocks(3, 0, 5, i, F if i < 2 else H, H if i < 2 else F) for i in range(3)]
    hs = [lib.mxfp4_upload(m, H if i == 2 else F, F if i == 2 else H) for i, m in enumerate(w)]
    try:
        got = lib.expert_mlp(5, hidden, F, *hs, *b, pairs, weight_before_ffn=bool(wbf))
    finally:
        for h in hs:
            lib.mxfp4_free(h)
    want = oracle.expert_mlp(5, hidden, F, *w, *b, pairs, weight_before_ffn=bool(wbf))
    assert np.all(got[np.arange(T) % 8 != 0] == 0)
    assert_layer_close(got, want)
