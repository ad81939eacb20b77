"""GPU parity of the prefill contract's native shared expert against the row kernels' chain (smoe_mmvq, bitwise the
oracle's): the shared rows are what add_shared adds to the block's output. From 128 columns on the products run on the
matrix cores (k_native_mm), fewer on the row kernels; more matrix-core cases are test_gpu_native_rule.py's.

Both form every 32-value dot exactly and differ in the order and number of f32 roundings, a few 2^-24 of a sum, and where
such a difference moves one of h's q8_1 values a step: 1/127 of its block's largest, in a row of n_ff values about
3 / 127 / sqrt(n_ff) of the row's norm (1.2e-3 at 384), for about one value in 10^4.  So a row is within three such
steps, and half of the rows, which have none, within 5e-6 (the rounding of the difference of two outputs included)."""
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_native import dev, native_layer, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # H, F, gate, up, down, T
    (2048, 512, O.Q3_K, O.Q3_K, O.IQ4_NL, 160),
    (2560, 640, O.Q3_K, O.Q3_K, O.IQ4_NL, 129),  # down: two chunks and a half
    (1024, 384, O.Q8_0, O.Q8_0, O.Q8_0, 33),     # the row kernels
    (1280, 512, O.Q4_0, O.Q4_0, O.Q5_0, 31),     # the row kernels
    (640, 128, O.Q5_0, O.IQ4_NL, O.Q4_0, 1),     # the row kernels, gate and up apart
    (2048, 512, O.Q8_0, O.Q8_0, O.Q4_0, 545),    # row tiles of 64: more than 256 work-groups
    (1536, 768, O.Q4_K, O.Q8_0, O.Q3_K, 64),     # the row kernels
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_native_shared_mm(torch, case):  # noqa: F811
    H, F, tg, tu, td, T = CASES[case]
    say(f"case: native shared matrix cores H={H} F={F} types {tg} {tu} {td} T={T}")
    g = O.Geom(n_embd=H, n_ff=F, n_ff_shared=F, n_expert=16, top_k=2, sh_type=tg, sh_up_type=tu, sh_down_type=td)
    _, w = native_layer(torch, g, 400 + case)
    x = dev(torch, O.gen_normal(400 + case, 100, T * H).reshape(T, H))
    ml = S.MoELayer(S.Geom(**vars(g)), w, max_tokens=T)
    y, tr = ml.forward(x, trace=True, path=S.PATH_MFMA)
    got = y.double() - ml.forward(x, add_shared=False, path=S.PATH_MFMA).double()
    xq = S.quantize_q8_1(x)
    hq = S.swiglu_q8(S.mmvq(tg, w["gate_sh"], xq, H, F, T), S.mmvq(tu, w["up_sh"], xq, H, F, T))
    want = (S.mmvq(td, w["down_sh"], hq, F, H, T) * torch.sigmoid(tr["sgate"].view(T, 1))).double()
    # (a row's difference carries the rounding of the two outputs it is taken from)
    rel = (got - want).norm(dim=1) / want.norm(dim=1)
    noise = float((2.0 ** -23 * y.double().norm(dim=1) / want.norm(dim=1)).max())
    say(f"  rel median {float(rel.median()):.2e} max {float(rel.max()):.2e} noise {noise:.2e}")
    assert float(rel.median()) <= 5e-6 + noise
    assert float(rel.max()) <= 3 * 3 / 127 / F ** 0.5 + noise
