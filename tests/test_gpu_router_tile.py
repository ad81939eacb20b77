"""GPU parity of the tiled router (k_router_tile: router_tiles) with the oracle's device order, bit for bit,
at the edges of its tiles: rows past the last row group, tokens past the last token tile, rows shorter than a stage of 512
values and no multiple of it, both tile shapes, bf16 and f32 rows, the shared gate and the x images behind the tiles."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_decode import bits, dev, host, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,T", [(8, 1, 5), (520, 17, 6), (2048, 513, 16), (1544, 64, 111), (2048, 49, 112), (8192, 31, 117),
                                   (512, 700, 203)])
def test_bf16_rows(torch, H, E, T):  # noqa: F811
    print(f"case: bf16 rows H={H} E={E} T={T}", flush=True)
    xb, W = O.gen_bf16(5, 1, T * H, 1.0), O.gen_bf16(5, 2, E * H, 0.02)
    got = host(torch, S.bf16_gemv(dev(torch, xb.view(np.int16)), dev(torch, W.view(np.int16)), H, E))
    for t in range(T):
        assert np.array_equal(bits(got[t]), bits(O.bf16_gemv_dev(xb[t * H:(t + 1) * H], W, H, E))), t


@pytest.mark.parametrize("router", [S.ROUTER_BF16, S.ROUTER_F32])
@pytest.mark.parametrize("H,E,T", [(384, 33, 7), (1280, 40, 21), (384, 65, 115)])
def test_block(torch, H, E, T, router):  # noqa: F811
    """The whole decode-contract block on those logits, with rows of very small and very large x among the tokens."""
    print(f"case: block H={H} E={E} T={T} router {router}", flush=True)
    g = O.Geom(n_embd=H, n_ff=128, n_ff_shared=128, n_expert=E, top_k=3, router_dtype=router)
    w_host = O.make_weights(g, 77)
    x = O.gen_normal(77, 100, T * H).reshape(T, H)
    x[1] *= np.float32(1e-30)
    x[3] *= np.float32(1e4)
    ml = S.MoELayer(S.Geom(**vars(g)), S.synth_layer(S.Geom(**vars(g)), 77), max_tokens=T)
    y, tr = ml.forward(dev(torch, x), trace=True, path=S.PATH_GEMV)
    want, wtr = O.moe_decode_dev(g, w_host, x, trace=True, n_threads=8)
    for k in ("logits", "sgate", "ids", "weights"):
        a, b = host(torch, tr[k]), np.asarray(wtr[k])
        bad = np.argwhere(bits(a).reshape(b.shape) != bits(b))
        assert not len(bad), (k, bad[:8].tolist(), a.reshape(b.shape)[tuple(bad[0])], b[tuple(bad[0])])
    assert np.array_equal(bits(host(torch, y)), bits(want))
