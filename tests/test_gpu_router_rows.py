"""Routing of small batches holds rows of up to 4096, and of up to 8192, values in registers and reads longer ones
again: the rows at both lines, with and without RMSNorm, one expert and four per workgroup."""
import numpy as np
import pytest

from coalsack_amd import capi, synth
from tests.helpers import assert_layer_close, build_layer, classify_index_mismatches, nbits_differ, oracle_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [4096, 4128, 8160, 8192, 8224])
@pytest.mark.parametrize("E,k,T,norm", [(4, 2, 1, True), (5, 2, 6, False), (130, 2, 33, True)])
def test_rows_at_the_lines(lib, oracle, H, E, k, T, norm):
    L = synth.LayerInputs(E, k, H, 32, seed=3, with_norm=norm)
    hidden = synth.hidden_states(T, H, seed=H + T)
    with build_layer(lib, L, norm=norm) as layer:
        got, pairs = layer.forward(hidden, capi.FWD_RMSNORM if norm else 0, want_pairs=True)
    want, wpairs = oracle_layer(oracle, L, hidden, norm=norm)
    x = oracle.rmsnorm(hidden, L.norm_w, 1e-5) if norm else hidden
    real, near = classify_index_mismatches(oracle, x, L, pairs, wpairs)
    assert real == 0, (real, near)
    same = np.all(pairs[..., 0] == wpairs[..., 0], axis=1)
    assert np.max(np.abs(pairs[same] - wpairs[same])) < 1.7e-5  # 1e-5 at 2880 values, growing with sqrt(H)
    assert_layer_close(got[same], want[same])


@pytest.mark.parametrize("H,want", [(4096, 1.0), (4128, 0.0), (8192, 0.0), (8224, 0.0)])
@pytest.mark.parametrize("E,T", [(4, 2), (130, 33)])
@pytest.mark.parametrize("last", [False, True])
def test_order_of_a_quads_sum(lib, H, want, E, T, last):
    """A logit of one quad, 4097 * 4097 - (2^24 + 8192): 4097^2 = 2^24 + 8193 is a tie that fp32 rounds to 2^24 + 8192, so
    the sum is 0 where the first product is rounded and 1 where the second is.  The latter is the order of rows of up to
    4096 values; longer ones round the first, whether they are held in registers or read again."""
    L = synth.LayerInputs(E, 1, H, 32, seed=3)
    c = H - 4 if last else 0
    hidden = np.zeros((T, H), np.float32)
    hidden[:, c], hidden[:, c + 1] = 4097.0, 1.0
    L.gate_w[:] = 0.0
    L.gate_w[0, c], L.gate_w[0, c + 1] = 4097.0, -(2.0 ** 24 + 8192.0)
    L.gate_b[:] = -1000.0  # no close call
    L.gate_b[0] = 0.0
    with build_layer(lib, L, device_weights=True, sigmoid=True) as layer:
        _, pairs = layer.forward(hidden, want_pairs=True)
    assert np.all(pairs[:, 0, 0] == 0)
    assert np.all(np.abs(pairs[:, 0, 1] - 1.0 / (1.0 + np.exp(-want))) < 1e-6)


@pytest.mark.parametrize("E,H,T,short,norm", [(128, 4096, 33, 12, True), (124, 8192, 17, 10, True), (128, 5120, 13, 8, False)])
def test_four_experts_per_workgroup_give_the_bits_of_one(lib, E, H, T, short, norm):
    """The shortest batches on 256 compute units that take four experts per workgroup, and the same tokens in passes that
    take one: routing weights of the same bits."""
    L = synth.LayerInputs(E, 4, H, 32, seed=6, with_norm=norm)
    hidden = synth.hidden_states(T, H, seed=2)
    with build_layer(lib, L, device_weights=True, norm=norm) as layer:
        _, four = layer.forward(hidden, capi.FWD_RMSNORM if norm else 0, want_pairs=True)
        try:
            lib.set_pass_tokens(short)
            _, one = layer.forward(hidden, capi.FWD_RMSNORM if norm else 0, want_pairs=True)
        finally:
            lib.set_pass_tokens(32768)
    assert nbits_differ(four, one) == 0
