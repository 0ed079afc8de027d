"""The dispatch kernel reads the expert ids four at a time in rounds of 8192 and places them in chunks of 1024: counts and lists
have to be those that the selection asks for, whatever is left over."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import build_layer

pytestmark = pytest.mark.gpu


# assignments short of and past a load of four, a chunk, the first half of a round and a round; one expert, experts with no
# token, as many experts as there can be
@pytest.mark.parametrize("E,k,T", [(4, 3, 65), (256, 1, 1025), (1, 1, 1023), (8, 3, 1365), (5, 1, 4097), (64, 16, 257),
                                   (32, 4, 2048), (7, 3, 2731), (256, 16, 1025)])
def test_dispatch(lib, E, k, T):
    L = synth.LayerInputs(E, k, 64, 32, seed=T, hot_experts=E // 3)
    with build_layer(lib, L) as layer:
        for _ in range(2):
            _, pairs = layer.forward(synth.hidden_states(T, 64, seed=E), want_pairs=True)
        counts, tokens = layer.last_dispatch(T)
    ids = pairs[..., 0].astype(int)
    assert np.array_equal(counts, np.bincount(ids.ravel(), minlength=E))
    assert np.array_equal(tokens, np.concatenate([np.flatnonzero((ids == e).any(axis=1)) for e in range(E)]))
