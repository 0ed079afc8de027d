"""An expert's three matrices travel as one transfer, and the cells that take a refused block are cleared only after one was refused:
matrices of every size arrive whole, a refused block is named with its place in its own matrix, and what is uploaded next is
not taken for refused."""
import numpy as np
import pytest

from coalsack_amd import capi

pytestmark = pytest.mark.gpu


def _blocks(rng, rows, cols):
    b = rng.integers(0, 256, (rows * cols // 32, 17), dtype=np.uint8)
    b[:, 0] = 117 + b[:, 0] % 5
    return b


# through the pinned area, through the ring in pieces of 64 KiB (one matrix a whole number of them), once round the ring
@pytest.mark.parametrize("H,F", [(64, 96), (1024, 1024), (2048, 2048), (2880, 2880), (4096, 8192)])
def test_refused_block_and_after(lib, H, F):
    rng = np.random.default_rng([H, F])
    shapes = {capi.W_UP: (F, H), capi.W_GATE: (F, H), capi.W_DOWN: (H, F)}
    w = {k: _blocks(rng, *s) for k, s in shapes.items()}
    with lib.layer(1, 1, H, F) as layer:
        for which, at in ((capi.W_UP, 3), (capi.W_DOWN, len(w[capi.W_DOWN]) - 1)):
            kept = w[which][at].copy()
            w[which][at] = 255  # codes of 6 under scale byte 255: infinities
            with pytest.raises(Exception, match=f"block {at}, "):
                layer.set_expert(0, *(w[k].reshape(-1) for k in (capi.W_UP, capi.W_GATE, capi.W_DOWN)))
            w[which][at] = kept
            lib.f16_free(lib.f16_upload_f32(np.ones((2, 32), np.float32)))  # (uses one of the cells for something else)
            layer.set_expert(0, *(w[k].reshape(-1) for k in (capi.W_UP, capi.W_GATE, capi.W_DOWN)))
            for k in shapes:
                assert np.array_equal(layer.export(0, k), w[k].reshape(-1))
