"""GPU parity of the IQ2_S products at the batches where they change to the matrix cores (iq2_mm_gains), bit for bit the
oracle's device order on both sides of the line: every row length on both sides, experts of several chunks and of none,
a native shared expert; the down kernel's two passes; and a token of infinities or NaN beside the others."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_iq2 import GUARD, bits, dev, host, torch  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # geometry, T, add_shared, the logit added to the first top_k experts
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=64, top_k=4, sh_type=22), 127, True, 0.0),  # the row kernels
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=64, top_k=4, sh_type=22), 128, True, 0.0),
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=64, top_k=4, sh_type=22), 130, False, 3.0),  # 130 columns, many empty
    (dict(n_embd=2048, n_ff=512, n_expert=64, top_k=8, sh_type=-1), 66, True, 0.0),
    (dict(n_embd=1024, n_ff=1024, n_ff_shared=1024, n_expert=64, top_k=8, sh_type=22), 65, True, 0.0),
    (dict(n_embd=512, n_ff=2048, n_ff_shared=2048, n_expert=3, top_k=2, sh_type=22), 193, True, 0.0),
    (dict(n_embd=2048, n_ff=1024, n_expert=2, top_k=2, sh_type=-1), 127, True, 0.0),  # the row kernels
    (dict(n_embd=2048, n_ff=1024, n_expert=2, top_k=2, sh_type=-1), 129, True, 0.0),
    (dict(n_embd=512, n_ff=512, n_ff_shared=512, n_expert=64, top_k=8, sh_type=O.Q8_0), 80, True, 0.0),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_forward_iq2_s_line(torch, case):  # noqa: F811
    gkw, T, add_shared, hot = CASES[case]
    print(f"case: IQ2_S line {gkw} T={T}", flush=True)
    g = O.Geom(w_type=22, **gkw)
    bias = None if not hot else np.where(np.arange(g.n_expert) < g.top_k, hot, 0.0).astype(np.float32)
    w_host = O.make_weights(g, 190 + case, zipf_bias=bias)
    base = S.Geom(**vars(g))
    if g.sh_type not in (-1, 22):
        base.sh_type = 22
    w_dev = S.synth_layer(base, 190 + case, logit_bias=None if bias is None else dev(torch, bias))
    if g.sh_type not in (-1, 22):
        for n in ("gate_sh", "up_sh", "down_sh"):
            w_dev[n] = dev(torch, getattr(w_host, n))
    x = O.gen_normal(190 + case, 100, T * g.n_embd).reshape(T, g.n_embd)
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
def test_iq2_s_two_passes(torch, n_embd, n_ff):  # noqa: F811
    """Enough items for the down kernel's two passes of 256 rows: the row kernels' bits (those of a traced call)."""
    g = S.Geom(w_type=22, sh_type=22, n_embd=n_embd, n_ff=n_ff, n_ff_shared=n_ff, n_expert=512, top_k=10)
    T = 361
    print(f"case: IQ2_S down passes H={n_embd} F={n_ff} T={T}", flush=True)
    ml = S.MoELayer(g, S.synth_layer(g, 7), max_tokens=T)
    x = dev(torch, O.gen_normal(7, 100, T * n_embd).reshape(T, n_embd))
    y = ml.forward(x)
    y2, _ = ml.forward(x, trace=True, stages=True)
    assert np.array_equal(bits(host(torch, y)), bits(host(torch, y2)))


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_iq2_s_other_tokens(torch, value):  # noqa: F811
    """A token of infinities or NaN changes no bit of the other tokens' rows."""
    g = S.Geom(w_type=22, sh_type=22, n_embd=512, n_ff=512, n_ff_shared=512, n_expert=64, top_k=4)
    T = 140
    print(f"case: IQ2_S batch with a token of {value}", flush=True)
    ml = S.MoELayer(g, S.synth_layer(g, 8), max_tokens=T)
    x = O.gen_normal(8, 100, T * g.n_embd).reshape(T, g.n_embd)
    y0 = host(torch, ml.forward(dev(torch, x)))
    x[70, ::5] = value
    y = host(torch, ml.forward(dev(torch, x)))
    keep = np.arange(T) != 70
    assert np.array_equal(bits(y[keep]), bits(y0[keep])) and np.isfinite(y[keep]).all()
