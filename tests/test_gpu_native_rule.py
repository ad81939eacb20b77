"""GPU parity of the native shared expert at the token counts where it changes kernels: two launches or the stage kernels
for a few tokens (native_few_gains), the row kernels or the matrix cores for a prompt (native_mm_gains).  Where a call
runs the row kernels' order it is theirs bit for bit (smoe_mmvq's chain, the oracle's), traced or not; on the matrix cores
within the bounds that test_gpu_native_mm.py derives; and a token of infinities or NaN leaves the others' rows."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_native import bits, dev, host, native_layer, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def layer(torch, H, F, tg, tu, td, T, seed):  # noqa: F811
    g = O.Geom(n_embd=H, n_ff=128, n_ff_shared=F, n_expert=16, top_k=2, sh_type=tg, sh_up_type=tu, sh_down_type=td)
    w_host, w = native_layer(torch, g, seed)
    return g, w_host, w, S.MoELayer(S.Geom(**vars(g)), w, max_tokens=T)


def shared_rows(torch, w, x, tr, H, F, tg, tu, td):  # noqa: F811
    T = x.shape[0]
    xq = S.quantize_q8_1(x)
    hq = S.swiglu_q8(S.mmvq(tg, w["gate_sh"], xq, H, F, T), S.mmvq(tu, w["up_sh"], xq, H, F, T))
    return (S.mmvq(td, w["down_sh"], hq, F, H, T) * torch.sigmoid(tr["sgate"].view(T, 1))).double()


@pytest.mark.parametrize("T", [1, 2, 4, 5, 127])
@pytest.mark.parametrize("types", [(O.Q8_0, O.Q8_0, O.IQ4_NL), (O.Q8_0, O.Q4_0, O.Q8_0)])
def test_prefill_contract_traced_and_not(torch, types, T):  # noqa: F811
    """The prefill contract on few tokens: the same bits with the stages traced and without."""
    H, F = 512, 256
    say(f"case: native shared, prefill contract traced and not, types {types} T={T}")
    _, _, _, ml = layer(torch, H, F, *types, T, 800 + T)
    x = dev(torch, O.gen_normal(800 + T, 100, T * H).reshape(T, H))
    y = host(torch, ml.forward(x, path=S.PATH_MFMA))
    y2, _ = ml.forward(x, path=S.PATH_MFMA, trace=True, stages=True)
    assert np.array_equal(bits(y), bits(host(torch, y2)))


@pytest.mark.parametrize("H, F, T", [(2048, 2048, 2), (2048, 2048, 3), (4096, 1024, 3), (4096, 2048, 1), (4096, 4096, 1)])
def test_few_tokens(torch, H, F, T):  # noqa: F811
    """The decode contract at both sides of the two-launch line, the oracle's bits."""
    say(f"case: native shared, few tokens H={H} F={F} T={T}")
    g, w_host, _, ml = layer(torch, H, F, O.Q3_K, O.Q3_K, O.IQ4_NL, T, 830 + T)
    x = O.gen_normal(830 + T, 100, T * H).reshape(T, H)
    want = O.moe_decode_dev(g, w_host, x, n_threads=16)
    assert np.array_equal(bits(host(torch, ml.forward(dev(torch, x)))), bits(want))


MM = [
    # H, F, gate, up, down, T: row tiles of 32 and 64 with remainders, column remainders, odd and short chunks
    (2048, 512, O.Q3_K, O.Q3_K, O.IQ4_NL, 128),
    (2560, 640, O.Q3_K, O.Q3_K, O.IQ4_NL, 129),     # down: two chunks and a half
    (1024, 384, O.Q8_0, O.Q8_0, O.Q8_0, 200),       # down: a chunk and a half
    (1280, 512, O.Q4_0, O.Q4_0, O.Q5_0, 131),       # gate/up: five chunks
    (640, 128, O.Q5_0, O.IQ4_NL, O.Q4_0, 1010),     # gate and up apart; down: half a chunk
    (512, 160, O.Q8_0, O.Q8_0, O.Q4_0, 1370),       # row tiles of 64, the last half dead
    (1536, 768, O.Q4_K, O.Q8_0, O.Q3_K, 177),       # one projection keeps the row kernels
]


@pytest.mark.parametrize("case", range(len(MM)))
def test_prompt(torch, case):  # noqa: F811
    H, F, tg, tu, td, T = MM[case]
    say(f"case: native shared, matrix cores H={H} F={F} types {tg} {tu} {td} T={T}")
    _, _, w, ml = layer(torch, H, F, tg, tu, td, T, 860 + case)
    x = dev(torch, O.gen_normal(860 + case, 100, T * H).reshape(T, H))
    y, tr = ml.forward(x, trace=True, path=S.PATH_MFMA)
    got = y.double() - ml.forward(x, add_shared=False, path=S.PATH_MFMA).double()
    want = shared_rows(torch, w, x, tr, H, F, tg, tu, td)
    rel = (got - want).norm(dim=1) / want.norm(dim=1)
    noise = float((2.0 ** -23 * y.double().norm(dim=1) / want.norm(dim=1)).max())
    say(f"  rel median {float(rel.median()):.2e} max {float(rel.max()):.2e} noise {noise:.2e}")
    assert float(rel.median()) <= 5e-6 + noise
    assert float(rel.max()) <= 3 * 3 / 127 / F ** 0.5 + noise


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("T", [3, 200])
def test_other_tokens(torch, T, value):  # noqa: F811
    """A token of infinities or NaN changes no bit of the other tokens' rows."""
    H, F = 1024, 384
    say(f"case: native shared, a token of {value} among {T}")
    _, _, _, ml = layer(torch, H, F, O.Q8_0, O.Q8_0, O.Q8_0, T, 890)
    x = O.gen_normal(890, 100, T * H).reshape(T, H)
    y0 = host(torch, ml.forward(dev(torch, x)))
    x[1, ::5] = value
    y = host(torch, ml.forward(dev(torch, x)))
    keep = np.arange(T) != 1
    assert np.array_equal(bits(y[keep]), bits(y0[keep])) and np.isfinite(y[keep]).all()
