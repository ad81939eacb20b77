"""Graph capture of the calls that change kernels with their size, on the side of the line that test_gpu_graph.py does not
reach: captured once and replayed three times with the program's own eager work between; every replay equals the eager
calls bit for bit."""
import numpy as np
import pytest

import oracle as O
import stratametal_amd as S
from test_gpu_hc import hc_dev, say, streams, torch  # noqa: F401
from test_gpu_native import native_layer

pytestmark = pytest.mark.gpu


def test_graph_replays_routes(torch):  # noqa: F811
    """The layer call with its read by rows (1, 17 tokens) and on the matrix cores (40, 130), its native shared expert in two
    launches (1), by stages and on the matrix cores (130); IQ2_S products on the row kernels (60) and the matrix cores
    (130); the f32 router's tiles; the junction in the router (60) and apart (90); the native GEMV by columns and in tiles;
    a verify window with its misses."""
    say("case: graph capture of the size-dependent routes, 3 replays")
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    H = 512
    gn = O.Geom(n_embd=H, n_ff=128, n_ff_shared=512, n_expert=16, top_k=3, sh_type=O.Q8_0, sh_down_type=O.IQ4_NL)
    ffn = S.FfnLayer(S.Geom(**vars(gn)), native_layer(torch, gn, 950)[1], hc_dev(torch, O.make_hc(H, 4, 960, 950), H), 130)
    gi = S.Geom(w_type=22, sh_type=22, n_embd=H, n_ff=512, n_ff_shared=512, n_expert=64, top_k=4)
    li = S.MoELayer(gi, S.synth_layer(gi, 951), max_tokens=130)
    gf = S.Geom(n_embd=H, n_ff=128, n_ff_shared=128, n_expert=200, top_k=4, router_dtype=S.ROUTER_F32)
    lf = S.MoELayer(gf, S.synth_layer(gf, 952), max_tokens=130)
    gb = S.Geom(n_embd=H, n_ff=128, n_ff_shared=128, n_expert=200, top_k=4)
    wb = S.synth_layer(gb, 953)
    lb, vw = S.MoELayer(gb, wb, max_tokens=100), S.VerifyWindow(gb, wb, max_tokens=4)
    blobs = torch.cat([wb[n].view(200, -1) for n in ("gate_exps", "up_exps", "down_exps")], dim=1)
    at = torch.arange(200, device="cuda") * blobs.shape[1] + blobs.data_ptr()
    held = torch.arange(200, device="cuda") % 4 != 0
    held, rest = torch.where(held, at, 0), torch.where(held, 0, at)
    x = {T: S.synth_normal(960 + T, 100, T * H).view(T, H) for T in (4, 6, 60, 90, 130)}
    r = {T: S.synth_normal(970 + T, 100, T * H).view(T, H) for T in (60, 90)}
    R = {T: to(streams(980 + T, T, 4, H)) for T in (1, 17, 40, 130)}
    wq = to(O.gen_native_blocks(O.Q6_K, 8, 3, 2047 * H))
    xq = {T: S.quantize_q8_1(x[T]) for T in (4, 130)}
    outs = {}

    def chain():
        for T in R:
            outs[("ffn", T)] = ffn.run(R[T])
        for T in (60, 130):
            outs[("iq2", T)] = li.forward(x[T])
        for T in (6, 130):
            outs[("f32", T)] = lf.forward(x[T])
        for T in (60, 90):
            xj = outs.setdefault(("xj", T), torch.empty_like(x[T]))
            outs[("res", T)] = lb.forward_residual(x[T], r[T], xj)
        for T in xq:
            outs[("q6_k", T)] = S.mmvq(O.Q6_K, wq, xq[T], H, 2047, T)
        v = vw.begin(x[4], held)
        groups = S.expert_group(v["ids"], gb.top_k, 200, rest)
        S.expert_grouped(gb, groups, xq[4], 4, v["rows"])
        outs["verify"] = vw.end(v)

    chain()
    torch.cuda.synchronize()
    want = {k: v.clone() for k, v in outs.items()}
    assert all(bool(torch.isfinite(w).all()) for w in want.values())
    graph, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        with torch.cuda.graph(graph, stream=st):
            chain()
    torch.cuda.synchronize()
    for rep in range(3):
        for v in outs.values():
            v.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for k, v in outs.items():
            assert torch.equal(v.view(torch.int32), want[k].view(torch.int32)), (rep, k)
        ffn.run(R[40])  # the program's own eager work between replays, on the same workspaces
        li.forward(x[6])
        lb.forward(x[60])
        torch.cuda.synchronize()
