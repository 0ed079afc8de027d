"""Close calls among a few logits: their chains of additions are cut into segments that begin with a guess of what lies in front of
them.  The order of the experts is that of the reference's sequential sums, at row lengths around what is staged at once
(3072 products of two rows, 1536 of four, 768 of eight), for sums that stay small and for sums that grow and fall again,
where the guesses miss; from the selection kernel of large batches and from those of small ones."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import build_layer

pytestmark = pytest.mark.gpu


def _close_rows(rng, E, H, close, swing):
    """Gate rows of which `close` give nearly the same logit, above all others."""
    g = rng.normal(0, 1 / np.sqrt(H), (E, H)).astype(np.float32)
    them = rng.choice(E, close, replace=False)
    base = g[them[0]].copy()
    if swing:  # the rows' first half adds up to about `swing`, the second takes it away again
        base[:H // 2] += swing / H
        base[H // 2:] -= swing / H
    g[them] = base + rng.normal(0, 3e-6 / np.sqrt(H), (close, H)).astype(np.float32)
    b = rng.normal(0, 0.01, E).astype(np.float32)
    b[them] = 6.0
    return g, b


def _same_order(got, logits, idx, k):
    """Slots that no equal logit is next to hold the oracle's experts; most slots are such."""
    top = -np.sort(-logits, axis=1)[:, :k + 1]
    differ = top[:, :k] != top[:, 1:k + 1]
    differ[:, 1:] &= differ[:, :-1].copy()  # (the order of equal ones is that of the reference's sort)
    assert differ.mean() > 0.4
    assert np.array_equal(got[..., 0][differ], idx[..., 0][differ])


@pytest.mark.parametrize("close", [2, 3, 4, 5, 9])
@pytest.mark.parametrize("H", [4, 36, 772, 2880, 3072, 3076, 6148])
@pytest.mark.parametrize("swing", [0.0, 8.0])
def test_selection_kernel(lib, oracle, close, H, swing):
    E, T = 40, 96
    k = max(2, close - 1)
    rng = np.random.default_rng([close, H, int(swing)])
    g, b = _close_rows(rng, E, H, close, swing)
    x = (rng.normal(0, 1, (T, H)) + (1.0 if swing else 0.0)).astype(np.float32)
    _same_order(lib.moe_router(x, g, b, k), oracle.router_logits(x, g, b), oracle.router(x, g, b, k), k)


@pytest.mark.parametrize("T", [3, 4, 16, 31])
@pytest.mark.parametrize("close,H", [(2, 2880), (2, 3104), (4, 1568), (8, 800), (2, 32)])
@pytest.mark.parametrize("swing", [0.0, 8.0])
def test_small_batches(lib, oracle, T, close, H, swing):
    E = 16
    k = max(2, close - 1)
    rng = np.random.default_rng([T, close, H])
    L = synth.LayerInputs(E, k, H, 32, seed=3)
    L.gate_w, L.gate_b = _close_rows(rng, E, H, close, swing)
    got, want, logits = [], [], []
    with build_layer(lib, L) as layer:
        for _ in range(64 // T + 1):
            x = (rng.normal(0, 1, (T, H)) + (1.0 if swing else 0.0)).astype(np.float32)
            got.append(layer.forward(x, want_pairs=True)[1])
            want.append(oracle.router(x, L.gate_w, L.gate_b, k))
            logits.append(oracle.router_logits(x, L.gate_w, L.gate_b))
    _same_order(np.concatenate(got), np.concatenate(logits), np.concatenate(want), k)
