"""The hyper-connection read at the batch sizes where it changes kernels (hc_mm_gains): on the matrix cores against the
oracle's row order within the bounds that test_gpu_hc_batch.py derives, one token below and at unaligned streams on the
row-per-wave kernels, the oracle's bits; and what one token's infinities and NaN leave of the others."""
import numpy as np
import pytest

import oracle as O
from test_gpu_hc import bits, dev, hc_dev, host, rel_l1, say, streams, torch  # noqa: F401

pytestmark = pytest.mark.gpu

FIRST = [
    # n_embd, hc, hc_lr, the first batch on the matrix cores
    (2048, 4, 320, 17),
    (2048, 2, 64, 42),
    (512, 2, 960, 41),   # the widest low-rank tile
    (3264, 5, 72, 22),   # five streams of more than 2048 values
    (192, 3, 200, 245),  # three streams, hc_lr no multiple of 64, an odd chunk count
    (256, 8, 64, 279),   # eight streams, a ragged last token tile
]


def close(n, hc, hc_lr, R, w, m, i):
    want_m, want_i = O.hc_read_dev(R, n, w)
    T = R.shape[0]
    worst = max(rel_l1(m[t], want_m[t]) for t in range(T))
    say(f"  mixed rel_l1 {worst:.2e}, inject {np.abs(i - want_i).max():.2e}")
    assert worst <= 2.0 ** -8 / hc_lr ** 0.5
    xn = R / np.sqrt((R.astype(np.float64) ** 2).mean(axis=2, keepdims=True)) * w.norm.reshape(1, hc, n)
    inj = np.abs((w.inject.astype(np.uint32) << 16).view(np.float32)).astype(np.float64).reshape(hc, hc * n)
    assert (np.abs(i - want_i) <= 1e-5 * (np.abs(xn).reshape(T, -1) @ inj.T)).all()
    return np.array_equal(bits(m), bits(want_m)) and np.array_equal(bits(i), bits(want_i))


@pytest.mark.parametrize("case", range(len(FIRST)))
def test_hc_read_first_batch(torch, case):  # noqa: F811
    n, hc, hc_lr, T = FIRST[case]
    say(f"case: hc_read first matrix-core batch n={n} hc={hc} hc_lr={hc_lr} T={T}")
    w = O.make_hc(n, hc, hc_lr, 700 + case)
    R = streams(700 + case, T, hc, n)
    H = hc_dev(torch, w, n)
    Rd = dev(torch, R)
    m, i = (host(torch, t) for t in H.read(Rd))
    assert not close(n, hc, hc_lr, R, w, m, i)  # (the matrix cores' order: not every bit the rows')
    m, i = (host(torch, t) for t in H.read(Rd[:T - 1]))  # the workspace of the larger call
    assert close(n, hc, hc_lr, R[:T - 1], w, m, i)


def test_hc_read_unaligned_batch(torch):  # noqa: F811
    n, hc, hc_lr, T = 2048, 4, 64, 40
    say("case: hc_read of a batch, streams 4-byte aligned")
    w = O.make_hc(n, hc, hc_lr, 9)
    R = streams(9, T, hc, n)
    buf = torch.empty(T * hc * n + 1, dtype=torch.float32, device="cuda")
    Rd = buf[1:].view(T, hc, n)
    Rd.copy_(torch.from_numpy(R))
    m, i = (host(torch, t) for t in hc_dev(torch, w, n).read(Rd))
    assert close(n, hc, hc_lr, R, w, m, i)


@pytest.mark.parametrize("value", [np.inf, np.nan, 3e38])
def test_hc_read_batch_other_tokens(torch, value):  # noqa: F811
    """A token of infinities, NaN or squares past f32 changes no bit of the others' rows."""
    n, hc, hc_lr, T = 512, 4, 320, 130
    say(f"case: hc_read batch with a token of {value}")
    H = hc_dev(torch, O.make_hc(n, hc, hc_lr, 11), n)
    R = streams(11, T, hc, n)
    m0, i0 = (host(torch, t) for t in H.read(dev(torch, R)))
    R[70, :, ::7] = value
    m, i = (host(torch, t) for t in H.read(dev(torch, R)))
    keep = np.arange(T) != 70
    assert np.array_equal(bits(m[keep]), bits(m0[keep])) and np.array_equal(bits(i[keep]), bits(i0[keep]))
    assert np.isfinite(m[keep]).all()
