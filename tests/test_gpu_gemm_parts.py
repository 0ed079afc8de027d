"""From 1536 work units on, a die of the grouped GEMM takes two parts of the unit sequence instead of one.  The batch in
passes too short for that (tokens are independent, and the kernels' sums the same) has to give the same bits."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import build_layer, nbits_differ

pytestmark = pytest.mark.gpu


# about 1450, 1540 and 2000 gate/up units (12 per M tile); 1560 down units (top-1, whose routing weight is 1 whatever the
# number of splits of H that the logits are summed in); an expert with most of the tokens
@pytest.mark.parametrize("E,k,H,F,T,hot", [(8, 4, 64, 2880, 1880, 0), (8, 4, 64, 2880, 2000, 0), (7, 3, 96, 2880, 3500, 0),
                                           (4, 1, 2880, 64, 16500, 0), (64, 2, 64, 5760, 2100, 1)])
def test_two_parts_equal_short_passes(lib, E, k, H, F, T, hot):
    L = synth.LayerInputs(E, k, H, F, seed=19, hot_experts=hot)
    hidden = synth.hidden_states(T, H, seed=8)
    with build_layer(lib, L, device_weights=True) as layer:
        whole, pairs = layer.forward(hidden, want_pairs=True)
        try:
            lib.set_pass_tokens((T + 2) // 3)
            short, spairs = layer.forward(hidden, want_pairs=True)
        finally:
            lib.set_pass_tokens(32768)
    assert np.all(np.isfinite(whole))
    assert nbits_differ(pairs, spairs) == 0
    assert nbits_differ(whole, short) == 0
