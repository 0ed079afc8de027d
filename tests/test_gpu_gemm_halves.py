"""Where the last round of a die's work units would occupy at most half of its compute units, the grouped GEMM takes those units in
halves of 32 tokens.  The batch in short passes, whose last rounds lie elsewhere, has to give the same bits."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import build_layer, nbits_differ

pytestmark = pytest.mark.gpu

DIES = 8


def halved(pairs, E, N, per, cus):
    """Units of `per` rows that a die takes in halves under these routing decisions (fewer than three per place: one part per die)."""
    tokens = np.bincount(pairs[..., 0].astype(int).ravel(), minlength=E)
    units = int(np.sum(-(-tokens // 64))) * -(-N // per)
    assert units < 3 * 2 * cus
    last = -(-units // DIES) % (cus // DIES)
    return last if 2 * last <= cus // DIES else 0


# rows of one and of several units; few tokens per last tile and many; one expert that takes most of them
@pytest.mark.parametrize("E,k,H,F,hot,tokens", [(8, 2, 1536, 4096, 0, (980, 1010, 1040, 1100)), (4, 2, 4096, 2880, 0, (1400, 1461, 2080, 2133)),
                                                (16, 4, 3072, 4512, 1, (700, 741, 800, 860))])
def test_halves_equal_short_passes(lib, E, k, H, F, hot, tokens):
    L = synth.LayerInputs(E, k, H, F, seed=23, hot_experts=hot)
    cus = lib.device_info()[1]
    seen = [0, 0]
    with build_layer(lib, L, device_weights=True) as layer:
        for T in tokens:
            assert T * k > 16 * E and (T * k // 64 + E) * -(-F // 256) > 2 * cus  # units of 512 rows
            hidden = synth.hidden_states(T, H, seed=T)
            whole, pairs = layer.forward(hidden, want_pairs=True)
            try:
                lib.set_pass_tokens(T // 2 + 7)
                short, spairs = layer.forward(hidden, want_pairs=True)
            finally:
                lib.set_pass_tokens(32768)
            here = halved(pairs, E, F, 256, cus), halved(pairs, E, H, 512, cus)
            seen = [s + (h > 0) for s, h in zip(seen, here)]
            same = np.all(pairs[..., 0] == spairs[..., 0], axis=1)
            assert same.mean() > 0.99 and np.all(np.isfinite(whole))
            assert np.max(np.abs(whole[same] - short[same])) <= 2e-6 * np.max(np.abs(whole))  # (the routing weights' last bits)
    assert min(seen) > 0, seen
