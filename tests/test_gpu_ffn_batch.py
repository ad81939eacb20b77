"""The whole layer call (smoe_ffn_run) of batches whose hyper-connection read runs on the matrix cores: bit for bit the
read, the block and the write called one after the other (each held to the oracle by its own tests), with a native and a
fused shared expert, in place, and on the same layer again with fewer tokens, where the read's rows are the oracle's."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_hc import GUARD, bits, dev, hc_dev, host, say, streams, torch  # noqa: F401
from test_gpu_native import native_layer

pytestmark = pytest.mark.gpu

CASES = [
    # n_embd, hc, hc_lr, the first batch on the matrix cores, shared types (gate/up, down), tokens in turn on one layer
    (2048, 4, 320, 17, (0, 0), (160, 17, 100, 1, 16)),
    (2048, 4, 320, 17, (O.Q3_K, O.IQ4_NL), (200, 17, 3, 130)),
    (512, 2, 960, 41, (O.Q8_0, O.Q8_0), (130, 41, 40)),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_ffn_batches(torch, case):  # noqa: F811
    n, hc, hc_lr, first, (gu, down), tokens = CASES[case]
    g = O.Geom(n_embd=n, n_ff=128, n_ff_shared=256, n_expert=16, top_k=3, **(dict(sh_type=gu, sh_down_type=down) if gu else {}))
    sg = S.Geom(**vars(g))
    w_dev = native_layer(torch, g, 930 + case)[1] if gu else S.synth_layer(sg, 930 + case)
    w = O.make_hc(n, hc, hc_lr, 930 + case)
    H, H2 = hc_dev(torch, w, n), hc_dev(torch, w, n)
    ffn, moe = S.FfnLayer(sg, w_dev, H, max(tokens)), S.MoELayer(sg, w_dev, max(tokens))
    for T in tokens:
        say(f"case: layer call n={n} hc={hc} hc_lr={hc_lr} shared {gu} {down} T={T}")
        R = streams(940 + T, T, hc, n)
        for add_shared in (True, False):
            m, i = H2.read(dev(torch, R))
            want = host(torch, H2.write(dev(torch, R), moe.forward(m, add_shared=add_shared), i))
            og = torch.full((T * hc * n + GUARD,), 7.0, dtype=torch.float32, device="cuda")
            ffn.run(dev(torch, R), out=og[:T * hc * n].view(T, hc, n), add_shared=add_shared)
            got = host(torch, og)
            assert (got[T * hc * n:] == 7.0).all(), "guard words written"
            assert np.array_equal(bits(got[:T * hc * n].reshape(T, hc, n)), bits(want))
            Rd = dev(torch, R)
            ffn.run(Rd, out=Rd, add_shared=add_shared)
            assert np.array_equal(bits(host(torch, Rd)), bits(want))
        want_m, _ = O.hc_read_dev(R, n, w)
        assert np.array_equal(bits(host(torch, m)), bits(want_m)) == (T < first)
