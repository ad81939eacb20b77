"""GPU parity of the native types' GEMV at the column counts where it changes between a work-group per column and column
tiles (native_cols), bit for bit the oracle's; and a column of infinite or NaN scale beside the others of its tile."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_native import TYPES, bits, dev, host, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def run(torch, t, w, xq, n_in, n_out, n_col):  # noqa: F811
    y = torch.full((n_col * n_out + 16,), 7.0, dtype=torch.float32, device="cuda")
    wd, xd = dev(torch, w), dev(torch, xq)
    S._check(S.lib().smoe_mmvq(t, wd.data_ptr(), 0, xd.data_ptr(), n_in, n_out, n_col, y.data_ptr(), S._stream()))
    got = host(torch, y)
    assert (got[n_col * n_out:] == 7.0).all(), "guard words written"
    return got[:n_col * n_out].reshape(n_col, n_out)


@pytest.mark.parametrize("t", TYPES)
def test_mmvq_native_columns(torch, t):  # noqa: F811
    # columns and rows on both sides of the rule: by columns, tiles of 4, 8 and 16 with live and dead columns and rows
    for n_in, n_out, n_col in [(256, 8195, 3), (256, 8195, 4), (256, 8195, 5), (256, 8195, 6), (256, 8195, 9), (256, 2047, 7),
                               (256, 2047, 12), (256, 1759, 12), (4352, 1031, 27), (4352, 1031, 31), (768, 33, 300)]:
        say(f"case: mmvq columns type {t} n_in={n_in} n_out={n_out} n_col={n_col}")
        w = O.gen_native_blocks(t, 8, n_in + n_out, n_in * n_out)
        xq = O.quant_q8_1(O.gen_normal(t, n_in + 1, n_col * n_in).reshape(n_col, n_in))
        want = O.native_gemv(t, w, xq, n_in, n_out, n_col)
        assert np.array_equal(bits(run(torch, t, w, xq, n_in, n_out, n_col)), bits(want)), (n_in, n_out, n_col)


@pytest.mark.parametrize("t", TYPES)
def test_mmvq_native_other_columns(torch, t):  # noqa: F811
    n_in, n_out, n_col = 512, 2047, 16
    say(f"case: mmvq columns beside one of infinite and NaN scales, type {t}")
    w = O.gen_native_blocks(t, 8, 3, n_in * n_out)
    xq = np.ascontiguousarray(O.quant_q8_1(O.gen_normal(t, 9, n_col * n_in).reshape(n_col, n_in))).reshape(n_col, -1, 36)
    want = run(torch, t, w, xq, n_in, n_out, n_col)
    bad = xq.copy()
    bad[6, 0, :2] = np.array([0x7C00], dtype=np.uint16).view(np.uint8)
    bad[6, 3, :2] = np.array([0x7E00], dtype=np.uint16).view(np.uint8)
    got = run(torch, t, w, bad, n_in, n_out, n_col)
    keep = np.arange(n_col) != 6
    assert np.array_equal(bits(got[keep]), bits(want[keep])) and np.isfinite(got[keep]).all()
    assert np.isnan(got[6]).all()
