"""One token whose largest logits are closer than the order of their additions decides: the gate/up kernel recomputes them in the
reference's order, eight side by side, in the LDS that its pointer table and rows take afterwards."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import assert_layer_close, build_layer, oracle_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("close,k", [(5, 4), (8, 4), (9, 4), (17, 16), (2, 1)])
@pytest.mark.parametrize("H", [96, 2880, 8192])
@pytest.mark.parametrize("opts", [dict(), dict(weight_before_ffn=True)])  # rows that arrive as FP6 terms, and fp32 rows
def test_one_token(lib, oracle, close, k, H, opts):
    E, F, T = 128, 32, 12
    L = synth.LayerInputs(E, k, H, F, seed=close)
    rng = np.random.default_rng([close, H])
    them = rng.choice(E, close, replace=False)
    L.gate_w[them] = L.gate_w[them[0]] + rng.normal(0, 5e-6 / np.sqrt(H), (close, H)).astype(np.float32)
    L.gate_b[them] = 6.0  # above all others
    hidden = synth.hidden_states(T, H, seed=H)
    logits = -np.sort(-oracle.router_logits(hidden, L.gate_w, L.gate_b), axis=1)[:, :k + 1]
    differ = logits[:, :-1] != logits[:, 1:]  # slot from the one below it
    differ[:, 1:] &= differ[:, :-1].copy()  # (the order of equal ones is that of the reference's sort)
    close_by = logits[:, :1] - logits[:, k:k + 1] < 8 * 2.0 ** -24 * np.sqrt(H) * logits[:, :1]
    assert differ.mean() > 0.3 and close_by.sum() > T // 2
    with build_layer(lib, L, **opts) as layer:
        got, pairs = map(np.concatenate, zip(*(layer.forward(hidden[t:t + 1], want_pairs=True) for t in range(T))))
    want, wpairs = oracle_layer(oracle, L, hidden, **opts)
    assert np.array_equal(pairs[differ][:, 0], wpairs[differ][:, 0])
    same = np.all(pairs[..., 0] == wpairs[..., 0], axis=1)
    assert_layer_close(got[same], want[same])
