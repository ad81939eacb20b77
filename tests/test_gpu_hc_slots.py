"""GPU parity of the hyper-connection read of few tokens (k_hc_proj) at every count of streams, values per thread and
pieces of a gate row that has registers of its own, and with the norm loaded after the scales, with the oracle's device
order bit for bit."""
import numpy as np
import pytest

import oracle as O
from test_gpu_hc import GUARD, bits, dev, hc_dev, host, say, streams, torch  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # n_embd, hc, hc_lr, T
    (512, 1, 64, 2), (1016, 2, 8, 3), (1032, 1, 16, 2), (1536, 2, 24, 2), (2560, 2, 40, 1), (3072, 1, 8, 2), (4096, 2, 16, 1),
    (264, 3, 8, 3), (768, 4, 64, 2), (1288, 4, 16, 2), (2304, 3, 24, 1), (2560, 4, 64, 16), (3000, 4, 8, 2), (4096, 3, 16, 2),
    (256, 7, 8, 2), (1024, 5, 32, 2), (1536, 6, 64, 16), (2048, 5, 8, 2), (2560, 6, 16, 2), (3072, 5, 16, 1),
    (2048, 6, 64, 16), (4096, 3, 64, 16), (2048, 8, 64, 15),  # the norm after the scales
    (64, 2, 72, 3), (64, 3, 128, 2), (64, 1, 184, 2), (64, 4, 256, 1), (64, 2, 520, 2), (64, 5, 1016, 2), (64, 2, 1032, 1),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_hc_read_slots(torch, case):  # noqa: F811
    n, hc, hc_lr, T = CASES[case]
    say(f"case: hc_read slots n={n} hc={hc} hc_lr={hc_lr} T={T}")
    w = O.make_hc(n, hc, hc_lr, 500 + case)
    R = streams(500 + case, T, hc, n)
    mg = torch.full((T * n + GUARD,), 7.0, dtype=torch.float32, device="cuda")
    ig = torch.full((T * hc + GUARD,), 7.0, dtype=torch.float32, device="cuda")
    hc_dev(torch, w, n).read(dev(torch, R), mixed=mg[:T * n], inject=ig[:T * hc])
    m, i = host(torch, mg), host(torch, ig)
    assert (m[T * n:] == 7.0).all() and (i[T * hc:] == 7.0).all(), "guard words written"
    want_m, want_i = O.hc_read_dev(R, n, w)
    assert np.array_equal(bits(m[:T * n].reshape(T, n)), bits(want_m))
    assert np.array_equal(bits(i[:T * hc].reshape(T, hc)), bits(want_i))


@pytest.mark.parametrize("n,hc,T", [(60, 8, 30), (64, 8, 1919), (64, 8, 1920), (252, 3, 5), (256, 8, 3), (260, 5, 757), (512, 8, 64),
                                    (1028, 2, 66), (1028, 2, 3061), (3000, 5, 769), (2048, 4, 3)])
def test_hc_write_kinds(torch, n, hc, T):  # noqa: F811
    """The write by values, by stream and through all streams, at the first batches of each and at rows whose last piece
    is not full; and at streams that are not 16-byte aligned, by values."""
    say(f"case: hc_write kinds n={n} hc={hc} T={T}")
    R = streams(n, T, hc, n)
    y = O.gen_normal(n, 51, T * n).reshape(T, n)
    inj = (O.gen_normal(n, 52, T * hc) * 4.0).reshape(T, hc).astype(np.float32)
    want = bits(O.hc_write_dev(R, y, inj, n, hc))
    H = hc_dev(torch, O.make_hc(n, hc, 8, n), n)
    og = torch.full((T * hc * n + GUARD,), 7.0, dtype=torch.float32, device="cuda")
    for at in (0, 1):
        og.fill_(7.0)
        H.write(dev(torch, R), dev(torch, y), dev(torch, inj), out=og[at:at + T * hc * n])
        got = host(torch, og)
        assert (got[at + T * hc * n:] == 7.0).all() and (got[:at] == 7.0).all()
        assert np.array_equal(bits(got[at:at + T * hc * n].reshape(T, hc, n)), want)
