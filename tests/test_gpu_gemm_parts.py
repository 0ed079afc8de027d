"""From three work units per place on (1536 on 256 compute units), a die of the grouped GEMM takes two parts of the unit
sequence instead of one.  The batch in passes too short for that (tokens are independent, and the kernels' sums the same) has
to give the same bits."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import build_layer, nbits_differ

pytestmark = pytest.mark.gpu


def units(pairs, E, N):
    """Work units of 256 gate and up rows each (512 rows of the down projection: N / 2) that these routing decisions give."""
    tokens = np.bincount(pairs[..., 0].astype(int).ravel(), minlength=E)
    return int(np.sum(-(-tokens // 64))) * int(np.ceil(N / 256))


# about 1450, 1550 and 2000 gate/up units (12 per M tile); 1560 down units (top-1, whose routing weight is 1 whatever the
# number of splits of H that the logits are summed in); 1656 units with an expert that every token selects
@pytest.mark.parametrize("E,k,H,F,T,hot,two", [(8, 4, 64, 2880, 1880, 0, ""), (8, 4, 64, 2880, 2000, 0, "up"),
                                               (7, 3, 96, 2880, 3500, 0, "up"), (4, 1, 2880, 64, 16500, 0, "down"),
                                               (16, 2, 64, 5760, 2100, 1, "up")])
def test_two_parts_equal_short_passes(lib, E, k, H, F, T, hot, two):
    L = synth.LayerInputs(E, k, H, F, seed=19, hot_experts=hot)
    hidden = synth.hidden_states(T, H, seed=8)
    each = (T + 2) // 3
    with build_layer(lib, L, device_weights=True) as layer:
        whole, pairs = layer.forward(hidden, want_pairs=True)
        try:
            lib.set_pass_tokens(each)
            short, spairs = layer.forward(hidden, want_pairs=True)
        finally:
            lib.set_pass_tokens(32768)
    line = 3 * 2 * lib.device_info()[1]
    assert (units(pairs, E, F) >= line, units(pairs, E, H / 2) >= line) == (two == "up", two == "down")
    for t in range(0, T, each):
        assert max(units(spairs[t:t + each], E, F), units(spairs[t:t + each], E, H / 2)) < line
    assert np.all(np.isfinite(whole))
    assert nbits_differ(pairs, spairs) == 0
    assert nbits_differ(whole, short) == 0
