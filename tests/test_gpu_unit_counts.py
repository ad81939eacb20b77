"""GPU parity of the Q2_0 decode kernels at rows of three, five and seven units per lane (1536, 384, 2560, 640, 896
values), in the fused small batch and in the batched launches, with the oracle's device order bit for bit."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_native import bits, dev, host, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 3, 9])
@pytest.mark.parametrize("H, F", [(1536, 384), (2560, 640), (896, 128)])
def test_forward_odd_unit_counts(torch, H, F, T):  # noqa: F811
    say(f"case: odd unit counts H={H} F={F} T={T}")
    g = O.Geom(n_embd=H, n_ff=F, n_ff_shared=F, n_expert=16, top_k=4)
    w_host = O.make_weights(g, 31)
    x = O.gen_normal(31, 100, T * H).reshape(T, H)
    ml = S.MoELayer(S.Geom(**vars(g)), S.synth_layer(S.Geom(**vars(g)), 31), max_tokens=T)
    want = O.moe_decode_dev(g, w_host, x, n_threads=8)
    assert np.array_equal(bits(host(torch, ml.forward(dev(torch, x)))), bits(want))
