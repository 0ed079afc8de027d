"""Router logits of many tokens from gate rows shorter than the 64 columns of the matrix-core router's step: nothing of another
expert's row, nor of what lies behind the last one, takes part."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [16, 32, 48, 64, 80])
@pytest.mark.parametrize("E", [3, 32, 64])
def test_neighbours_take_no_part(lib, oracle, H, E):
    T = 100
    rng = np.random.default_rng(H + E)
    x = rng.normal(0, 1, (T, H)).astype(np.float32)
    g = rng.normal(0, 0.3, (E, H)).astype(np.float32)
    b = rng.normal(0, 0.1, E).astype(np.float32)
    want = oracle.router_logits(x, g, b)
    assert np.allclose(lib.moe_router_logits(x, g, b), want, rtol=1e-5, atol=3 * 2.0 ** -24 * np.sqrt(H))
    g[1::2] = np.nan  # every row's neighbour, and the last row's too if their number is even
    got = lib.moe_router_logits(x, g, b)
    assert np.allclose(got[:, ::2], want[:, ::2], rtol=1e-5, atol=3 * 2.0 ** -24 * np.sqrt(H))
