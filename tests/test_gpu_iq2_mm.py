"""GPU parity of IQ2_S batches of six and more pairs per expert with the oracle's device order, bit for bit: every row length
on both sides, columns with remainders, one or no column, the shared expert, and the same call traced (which runs the row
kernels). With so few experts only the batch of 140 pairs per expert is on the matrix cores (smoe_iq2_mm.hip); the lines
between the two and the other matrix-core batches are test_gpu_iq2_mm_rule.py's."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_iq2 import GUARD, bits, dev, host, torch  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # geometry, T, add_shared
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=16, top_k=4, sh_type=22), 23, True),
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=16, top_k=4, sh_type=22), 24, True),
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=16, top_k=4, sh_type=22), 33, False),
    (dict(n_embd=1024, n_ff=512, n_expert=8, top_k=2, sh_type=-1), 37, True),
    (dict(n_embd=2048, n_ff=512, n_ff_shared=512, n_expert=24, top_k=4, sh_type=22), 50, True),
    (dict(n_embd=512, n_ff=2048, n_ff_shared=2048, n_expert=6, top_k=2, sh_type=22), 33, True),
    (dict(n_embd=2048, n_ff=1024, n_expert=5, top_k=3, sh_type=-1), 23, True),
    (dict(n_embd=1024, n_ff=1024, n_ff_shared=1024, n_expert=3, top_k=2, sh_type=22), 210, True),  # the matrix cores: chunks of 64 columns
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=16, top_k=4, sh_type=O.Q8_0), 80, True),  # a native shared expert
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_forward_iq2_s_batches(torch, case):  # noqa: F811
    gkw, T, add_shared = CASES[case]
    print(f"case: IQ2_S batch {gkw} T={T}", flush=True)
    g = O.Geom(w_type=22, **gkw)
    w_host = O.make_weights(g, 90 + case)
    base = S.Geom(**vars(g))
    if g.sh_type not in (-1, 22):
        base.sh_type = 22
    w_dev = S.synth_layer(base, 90 + case)
    if g.sh_type not in (-1, 22):
        for n in ("gate_sh", "up_sh", "down_sh"):
            w_dev[n] = dev(torch, getattr(w_host, n))
    x = O.gen_normal(90 + case, 100, T * g.n_embd).reshape(T, g.n_embd)
    x[1] = 0.0  # every product zero
    x[2] *= np.float32(1e4)
    ml = S.MoELayer(S.Geom(**vars(g)), w_dev, max_tokens=T)
    yg = torch.full((T * g.n_embd + GUARD,), 7.0, dtype=torch.float32, device="cuda")
    ml.forward(dev(torch, x), y=yg[:T * g.n_embd].view(T, g.n_embd), add_shared=add_shared)
    got = host(torch, yg)
    assert (got[T * g.n_embd:] == 7.0).all(), "guard words past y were written"
    got = got[:T * g.n_embd].reshape(T, g.n_embd)
    want = O.moe_decode_dev(g, w_host, x, add_shared=add_shared, n_threads=16)
    assert np.array_equal(bits(got), bits(want)), f"max rel {O.rel_l1_rows(got, want).max()}"
    y2, _ = ml.forward(dev(torch, x), add_shared=add_shared, trace=True, stages=True)
    assert np.array_equal(bits(host(torch, y2)), bits(want))


@pytest.mark.parametrize("n_embd, n_ff", [(2048, 512), (2048, 1024)])
def test_iq2_s_down_passes(torch, n_embd, n_ff):  # noqa: F811
    """Six pairs per expert of 512: the traced call's bits (the down kernel's two passes are test_gpu_iq2_mm_rule.py's)."""
    g = S.Geom(w_type=22, sh_type=22, n_embd=n_embd, n_ff=n_ff, n_ff_shared=n_ff, n_expert=512, top_k=10)
    T = 311
    print(f"case: IQ2_S down passes H={n_embd} F={n_ff} T={T}", flush=True)
    ml = S.MoELayer(g, S.synth_layer(g, 7), max_tokens=T)
    x = dev(torch, O.gen_normal(7, 100, T * n_embd).reshape(T, n_embd))
    y = ml.forward(x)
    y2, _ = ml.forward(x, trace=True, stages=True)
    assert np.array_equal(bits(host(torch, y)), bits(host(torch, y2)))
