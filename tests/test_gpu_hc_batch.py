"""GPU parity of the hyper-connection read of batches, on the matrix cores (k_hc_proj_mm and k_hc_mix_mm) or the
row-per-wave kernels by hc_mm_gains, against the oracle's row order on the same inputs.  Both sum exact bf16 products in
f32 in different orders, so inject differs by the f32 sums' rounding (hc * n products: below 1e-5 of the products'
magnitude), and mixed where a low-rank value's bf16 rounding falls to the other side: one of hc_lr values moves by up to
2^-8 of itself, so a gate by about 2^-8 / sqrt(hc_lr) of its argument, and a row's mean by less (sigmoid's slope is at
most 1/4)."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_hc import GUARD, dev, hc_dev, host, rel_l1, streams, torch  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # n_embd, hc, hc_lr, T: token tiles of 32 and 64 with remainders, row tiles of 128, K slices, chunk tails (the first
    # batches of other shapes: test_gpu_hc_mm.py)
    (2048, 4, 320, 17),
    (2048, 4, 320, 130),
    (64, 1, 8, 16400),   # one chunk of K, one row tile mostly empty, the last token tile ragged
    (192, 3, 200, 75),   # the row-per-wave kernels, as the next three
    (256, 8, 64, 64),
    (512, 2, 960, 31),
    (3264, 5, 72, 20),
    (4096, 4, 512, 95),  # the largest activation row, an lq tile too wide for 64 tokens
    (320, 4, 128, 700),  # many token tiles
    (2048, 2, 64, 31),   # the row-per-wave kernels, as the next
    (2048, 2, 64, 32),
    (1088, 1, 1000, 40),  # hc_lr past the matrix-core tile: the row-per-wave kernels
    (72, 3, 24, 40),      # no whole 64-value chunks: the row-per-wave kernels
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_hc_read_batch(torch, case):  # noqa: F811
    n, hc, hc_lr, T = CASES[case]
    print(f"case: hc_read batch n={n} hc={hc} hc_lr={hc_lr} T={T}", flush=True)
    w = O.make_hc(n, hc, hc_lr, 300 + case)
    R = streams(300 + case, T, hc, n)
    H = hc_dev(torch, w, n)
    mg = torch.full((T * n + GUARD,), 7.0, dtype=torch.float32, device="cuda")
    ig = torch.full((T * hc + GUARD,), 7.0, dtype=torch.float32, device="cuda")
    H.read(dev(torch, R), mixed=mg[:T * n], inject=ig[:T * hc])
    m, i = host(torch, mg), host(torch, ig)
    assert (m[T * n:] == 7.0).all() and (i[T * hc:] == 7.0).all(), "guard words written"
    m, i = m[:T * n].reshape(T, n), i[:T * hc].reshape(T, hc)
    want_m, want_i = O.hc_read_dev(R, n, w)
    worst = max(rel_l1(m[t], want_m[t]) for t in range(T))
    print(f"  mixed rel_l1 {worst:.2e}, inject {np.abs(i - want_i).max():.2e}", flush=True)
    assert worst <= 2.0 ** -8 / hc_lr ** 0.5
    # the products' magnitude: |act| . |inj| per stream, act = (R / rms) * norm
    xn = R / np.sqrt((R.astype(np.float64) ** 2).mean(axis=2, keepdims=True)) * w.norm.reshape(1, hc, n)
    inj = np.abs((w.inject.astype(np.uint32) << 16).view(np.float32)).astype(np.float64).reshape(hc, hc * n)
    mag = np.abs(xn).reshape(T, -1) @ inj.T
    assert (np.abs(i - want_i) <= 1e-5 * mag).all()


def test_hc_read_batch_unaligned(torch):  # noqa: F811
    """Streams at a 4-byte aligned address take the row-per-wave kernels: the oracle's bits."""
    n, hc, hc_lr, T = 2048, 4, 64, 24
    w = O.make_hc(n, hc, hc_lr, 9)
    R = streams(9, T, hc, n)
    H = hc_dev(torch, w, n)
    buf = torch.empty(T * hc * n + 1, dtype=torch.float32, device="cuda")
    Rd = buf[1:].view(T, hc, n)
    Rd.copy_(torch.from_numpy(R))
    m, i = H.read(Rd)
    want_m, want_i = O.hc_read_dev(R, n, w)
    assert np.array_equal(host(torch, m).view(np.uint32), want_m.view(np.uint32))
    assert np.array_equal(host(torch, i).view(np.uint32), want_i.view(np.uint32))
