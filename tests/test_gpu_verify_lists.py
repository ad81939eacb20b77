"""What VerifyWindow.begin hands out: keeping the counts keeps no rows alive, an empty window counts nothing."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_cache import dev, host, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def test_verify_begin_lists(torch):  # noqa: F811
    print("case: verify window's lists", flush=True)
    g = S.Geom(n_embd=256, n_ff=128, n_ff_shared=128, n_expert=16, top_k=4)
    w = S.synth_layer(g, 5)
    E = g.n_expert
    blobs = torch.cat([w[n].view(E, -1) for n in ("gate_exps", "up_exps", "down_exps")], dim=1)
    at = torch.arange(E, device="cuda") * blobs.shape[1] + blobs.data_ptr()
    held = torch.where(torch.arange(E, device="cuda") % 2 == 0, at, 0)
    vw = S.VerifyWindow(g, w, max_tokens=8)
    r = vw.begin(dev(torch, O.gen_normal(5, 100, 8 * 256).reshape(8, 256)), held)
    ids, counts, miss = host(torch, r["ids"]).ravel(), host(torch, r["counts"]), host(torch, r["miss_dst"])
    want = np.flatnonzero(ids % 2)
    assert counts[1] == 32 - len(want) and counts[2] == len(want) and counts[3] == 0
    assert np.array_equal(miss[:len(want)], want) and (miss[len(want):] == -1).all()
    assert r["counts"].untyped_storage().nbytes() <= 4 * (32 + 4)
    assert r["rows"].untyped_storage().nbytes() == 4 * (32 + 8) * 256
    assert (host(torch, vw.begin(torch.empty((0, 256), device="cuda"), held)["counts"]) == 0).all()
