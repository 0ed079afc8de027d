"""Pairs that name an expert in several slots of a token: the expert takes the token once, with the first slot's weight."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import assert_layer_close

pytestmark = pytest.mark.gpu

# call, its kernels with and without the weight in front (tests/test_host_transfers.py holds them to it), k, H, F, T
BATCHES = [("expert", "expert_stream_kernel", 3, 256, 224, 10),
           ("expert", "expert_stream_kernel_tiles", 4, 2880, 2880, 32),
           ("expert", "expert_gemm_mx_kernel", 4, 96, 160, 150),
           ("expert_f16", "expert_f16_kernel", 4, 96, 160, 33),
           ("expert_f16", "expert_f16_gemm_kernel", 4, 96, 160, 130)]


def batch(T, k, H, seed):
    """More slots that name expert 5 than there are tokens."""
    rng = np.random.default_rng(seed)
    pairs = np.empty((T, k, 2), np.float32)
    pairs[..., 0] = rng.choice([5, 2, 8], (T, k), p=[0.7, 0.2, 0.1])
    pairs[..., 1] = rng.uniform(0.1, 0.9, (T, k))
    pairs[T // 2, :, 0] = 2
    return rng.normal(0, 1, (T, H)).astype(np.float32), pairs


@pytest.mark.parametrize("what,kernel,k,H,F,T", BATCHES)
@pytest.mark.parametrize("wbf", [False, True])
def test_expert_in_several_slots(lib, oracle, what, kernel, k, H, F, T, wbf):
    rng = np.random.default_rng(T)
    b = [rng.normal(0, 0.01, n).astype(np.float32) for n in (F, F, H)]
    hidden, pairs = batch(T, k, H, seed=1)
    others, opairs = batch(4 * T, k, H, seed=2)  # leaves rows of its own in the buffers
    assert (pairs[..., 0] == 5).sum() > T
    if what == "expert_f16":
        w = [(rng.normal(0, 1, s) / np.sqrt(s[1])).astype(np.float16) for s in ((F, H), (F, H), (H, F))]
        lib.expert_mlp_f16(5, others, *w, *b, opairs, weight_before_ffn=wbf)
        got = lib.expert_mlp_f16(5, hidden, *w, *b, pairs, weight_before_ffn=wbf)
        want = oracle.expert_mlp_f16(5, hidden, *w, *b, pairs, weight_before_ffn=wbf)
    else:
        w = [synth.mxfp4_blocks(3, 0, 5, i, F if i < 2 else H, H if i < 2 else F) for i in range(3)]
        hs = [lib.mxfp4_upload(m, H if i == 2 else F, F if i == 2 else H) for i, m in enumerate(w)]
        try:
            lib.expert_mlp(5, others, F, *hs, *b, opairs, weight_before_ffn=wbf)
            got = lib.expert_mlp(5, hidden, F, *hs, *b, pairs, weight_before_ffn=wbf)
        finally:
            for h in hs:
                lib.mxfp4_free(h)
        want = oracle.expert_mlp(5, hidden, F, *w, *b, pairs, weight_before_ffn=wbf)
    assert np.all(got[T // 2] == 0)
    assert_layer_close(got, want)
