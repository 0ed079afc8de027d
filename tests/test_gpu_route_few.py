"""A few tokens: every workgroup of the gate/up kernel routes the batch itself.  What the kernels behind it and
csk_layer_last_dispatch read has to be the dispatch that the selection asks for, and the rows those of the experts' tokens."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import assert_layer_close, build_layer, oracle_layer

pytestmark = pytest.mark.gpu


# rows of two to sixteen steps per wave; 64 assignments; one expert that takes every token; as many experts as there can be
@pytest.mark.parametrize("E,k,H,F,hot", [(8, 2, 96, 64, 0), (256, 16, 2880, 96, 0), (16, 4, 1056, 256, 1), (4, 4, 1568, 96, 0),
                                         (5, 1, 2080, 2880, 0), (128, 4, 4128, 32, 8), (3, 3, 5632, 64, 0), (6, 2, 8192, 96, 0)])
@pytest.mark.parametrize("T", [2, 3, 4])
def test_few_tokens(lib, oracle, E, k, H, F, hot, T):
    check(lib, oracle, E, k, H, F, hot, T)


# two selections per wave, experts with more tokens than a group holds; the last of each is routed by a launch of its own
@pytest.mark.parametrize("E,k,H,F,hot", [(4, 3, 1056, 96, 0), (16, 4, 2880, 64, 1), (2, 1, 96, 64, 0), (128, 4, 96, 96, 8)])
@pytest.mark.parametrize("T", [5, 6, 7, 8, 9])
def test_more_tokens_than_waves(lib, oracle, E, k, H, F, hot, T):
    check(lib, oracle, E, k, H, F, hot, T)


def check(lib, oracle, E, k, H, F, hot, T):
    L = synth.LayerInputs(E, k, H, F, seed=T, hot_experts=hot)
    hidden = synth.hidden_states(T, H, seed=H)
    with build_layer(lib, L) as layer:
        got, pairs = layer.forward(hidden, want_pairs=True)
        counts, tokens = layer.last_dispatch(T)
    want, wpairs = oracle_layer(oracle, L, hidden)
    assert np.array_equal(pairs[..., 0], wpairs[..., 0])
    assert_layer_close(got, want)
    ids = pairs[..., 0].astype(int)
    assert np.array_equal(counts, np.bincount(ids.ravel(), minlength=E))
    assert np.array_equal(tokens, np.concatenate([np.flatnonzero((ids == e).any(axis=1)) for e in range(E)]))
