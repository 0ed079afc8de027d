"""A few tokens: the down projection and the weighted merge are one launch.  The rows have to be those that the two launches
give, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from coalsack_amd import synth
from coalsack_amd.capi import FWD_RESIDUAL, Layer
from tests.helpers import assert_layer_close, build_layer, nbits_differ, oracle_layer

pytestmark = pytest.mark.gpu


# rows of the down projection of every count of steps per wave; one and two tiles of outputs per workgroup, a last tile that
# is half empty; fewer groups than teams, more than one round of them, one group for all tokens, one expert
@pytest.mark.parametrize("E,H,F,hot,batches", [
    (8, 96, 32, 0, [(1, 1), (1, 8), (2, 4), (8, 1), (3, 2)]), (16, 1056, 1536, 0, [(1, 2), (1, 8), (4, 2)]),
    (9, 8192, 256, 0, [(1, 1), (1, 6), (3, 2)]), (4, 4128, 1504, 2, [(1, 4), (5, 1)]),
    (8, 2880, 2048, 0, [(1, 3), (4, 1)]), (8, 96, 2496, 1, [(1, 4), (2, 2)]), (8, 2080, 2880, 0, [(1, 4), (3, 1)]),
    (6, 4160, 2912, 0, [(2, 2)]), (4, 64, 3584, 0, [(1, 4)]), (4, 4352, 4096, 0, [(1, 4)]), (4, 1024, 6144, 0, [(1, 2), (2, 1)]),
    (4, 96, 8192, 0, [(1, 1), (1, 2)]), (4, 4128, 8160, 0, [(2, 1)]), (1, 2080, 96, 0, [(1, 1), (3, 1), (8, 1)])])
@pytest.mark.parametrize("wbf", [False, True])
def test_one_launch(lib, oracle, E, H, F, hot, batches, wbf):
    for T, k in batches:
        L = synth.LayerInputs(E, k, H, F, seed=T * 16 + k, hot_experts=hot)
        hidden = synth.hidden_states(T, H, seed=H)
        with build_layer(lib, L, weight_before_ffn=wbf) as layer:
            got, pairs = layer.forward(hidden, FWD_RESIDUAL, want_pairs=True)
        want, wpairs = oracle_layer(oracle, L, hidden, residual=True, weight_before_ffn=wbf)
        assert np.array_equal(pairs[..., 0], wpairs[..., 0])
        assert_layer_close(got, want)
        two, tpairs = frame(lib, L, hidden, wbf)
        assert nbits_differ(pairs, tpairs) == 0
        assert nbits_differ(got, two) == 0, (T, k)


def frame(lib, L, hidden, wbf):
    """The layer as a frame, whose experts' rows stay there to be asked for: two launches."""
    T, h, hs, n = len(hidden), C.c_void_p(), [], C.c_int()
    lib.check(lib.dll.csk_layer_create_view(L.E, L.k, L.H, L.F, C.byref(h)))
    out, pairs = np.empty((T, L.H), np.float32), np.empty((T, L.k, 2), np.float32)
    try:
        with Layer.adopt(lib, h, L.E, L.k, L.H, L.F) as view:
            view.set_router(L.gate_w, L.gate_b)
            view.set_options(weight_before_ffn=wbf)
            for e in range(L.E):
                m = [lib.mxfp4_upload(L.blocks(e, i), *((L.H, L.F) if i == 2 else (L.F, L.H))) for i in range(3)]
                hs += m
                lib.check(lib.dll.csk_layer_attach_expert(h, e, *m, *[b[e].ctypes.data for b in (L.b_up, L.b_gate, L.b_down)]))
            lib.check(lib.dll.csk_moe_frame_begin(h, hidden.ctypes.data, T, pairs.ctypes.data, FWD_RESIDUAL, C.byref(n)))
            assert n.value == 1
            lib.check(lib.dll.csk_moe_frame_merged(h, out.ctypes.data, C.byref(n)))
            assert n.value == 1
    finally:
        for m in hs:
            lib.mxfp4_free(m)
    return out, pairs
