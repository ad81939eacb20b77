"""The dispatch rules of stratametal_amd/csrc/smoe_rules.hpp at the sizes whose both sides were measured (the figures
stand beside the rules): host functions, compiled here and asked for their choice."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("c++")
pytestmark = pytest.mark.skipif(CXX is None, reason="no host compiler")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    """ask(expressions): their values, as whole numbers."""
    d = tmp_path_factory.mktemp("rules")

    def run(exprs):
        src, exe = str(d / "rules.cpp"), str(d / "rules")
        body = "".join(f'    std::printf("%lld\\n", (long long)({e}));\n' for e in exprs)
        with open(src, "w") as f:
            f.write('#include <cstdio>\n#include "smoe_rules.hpp"\nusing namespace smoe;\nint main() {\n' + body + "}\n")
        subprocess.run([CXX, "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "stratametal_amd", "csrc"), src, "-o",
                        exe], check=True, capture_output=True, text=True)
        out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
        return [int(v) for v in out]
    return run


def test_hc_slots(ask):
    """The read's slots hold the streams with few to spare: each is loaded."""
    shapes = [(n, hc) for n in range(8, 4097, 8) for hc in range(1, 9) if hc * n <= 16384]
    got = ask([e for n, hc in shapes for e in (f"hc_streams({hc})", f"hc_values({n})", f"hc_chunks({n}, {hc})")])
    for i, (n, hc) in enumerate(shapes):
        s, v, c = got[3 * i:3 * i + 3]
        need = (n + 255) // 256
        assert s >= hc and v >= need, (n, hc)
        assert s < 2 * hc or s == 2, (n, hc)  # fewer spare streams than streams (a second one beside a single one)
        assert v - need <= max(1, need // 4) or need == 1, (n, hc)
        assert 512 * c >= hc * n >= 0 and c - hc * n / 512 <= 8 and c in (8, 16, 24, 32), (n, hc)
        assert c <= (8 if s * v <= 16 else 16 if s * v <= 32 else 32), (n, hc)  # the kernels that exist


def test_hc_pieces(ask):
    """The same for a row of the gate products: no piece to spare up to five, fewer than needed beyond."""
    widths = list(range(8, 2049, 8))
    for lr, p in zip(widths, ask([f"hc_pieces({lr})" for lr in widths])):
        need = (lr + 63) // 64
        assert p >= need and (p == need if need <= 5 else p < 2 * need), lr


def test_hc_norm(ask):
    """Two waves per SIMD where they halve the rounds: hc, n, hc_lr, tokens -> the norm with the streams."""
    cases = [(4, 2048, 320, 1, 1), (4, 2048, 320, 16, 1), (4, 2560, 64, 16, 1), (6, 1536, 64, 16, 1), (6, 2048, 64, 14, 1),
             (6, 2048, 64, 16, 0), (5, 2048, 200, 6, 0), (3, 4096, 64, 16, 0), (8, 2048, 320, 4, 1), (6, 2560, 64, 16, 1)]
    got = ask([f"hc_norm_ahead(hc_streams({hc}) * hc_values({n}), 4 * hc_chunks({n}, {hc}), {(lr + hc + 3) // 4 * T}, "
               f"{lr * hc * n * 2})" for hc, n, lr, T, _ in cases])
    assert got == [c[-1] for c in cases]


def test_hc_matrix_cores(ask):
    """n, hc, hc_lr, tokens: the faster of the row-per-wave kernels (0) and the matrix cores (1); more tokens never go
    back (a workspace for more tokens holds every smaller call)."""
    cases = [(2048, 4, 320, 16, 0), (2048, 4, 320, 17, 1), (2048, 4, 320, 1000, 1), (512, 4, 320, 17, 0), (512, 4, 320, 64, 0),
             (512, 4, 320, 128, 1), (512, 2, 320, 32, 0), (512, 8, 320, 24, 0), (256, 8, 320, 64, 0), (256, 8, 320, 128, 1),
             (512, 8, 960, 24, 0), (2048, 4, 64, 24, 0), (2048, 4, 64, 64, 1), (2048, 2, 200, 24, 0), (1536, 4, 64, 24, 0),
             (2560, 2, 640, 17, 1), (4096, 1, 960, 17, 1), (4096, 4, 640, 17, 1), (1024, 8, 640, 24, 1)]
    assert ask([f"hc_mm_gains({T}, {n}, {hc}, {lr})" for n, hc, lr, T, _ in cases]) == [c[-1] for c in cases]
    shapes = [(n, hc, lr) for n in (64, 512, 2048, 4096) for hc in (1, 4, 8) for lr in (8, 320, 960)]
    tokens = (1, 16, 17, 40, 64, 100, 1000, 4096, 65535)
    got = ask([f"hc_mm_gains({T}, {n}, {hc}, {lr})" for n, hc, lr in shapes for T in tokens])
    for i, s in enumerate(shapes):
        g = got[i * len(tokens):(i + 1) * len(tokens)]
        assert g == sorted(g), s


def test_hc_write(ask):
    """n, hc, tokens: a value per thread (0), vectors stream by stream (1), vectors through all streams (2)."""
    cases = [(64, 8, 200, 0), (64, 8, 4000, 2), (72, 4, 64, 0), (32, 8, 4000, 0), (512, 8, 64, 1), (256, 8, 16, 1), (256, 8, 1000, 2),
             (2048, 4, 1, 1), (2048, 4, 64, 1), (2048, 4, 1000, 1), (2048, 4, 4000, 2), (4096, 4, 1000, 2)]
    assert ask([f"hc_write_kind({T}, {n}, {hc})" for n, hc, T, _ in cases]) == [c[-1] for c in cases]


def test_iq2_matrix_cores(ask):
    """n_expert, n_embd, n_ff, pairs per expert: the faster of the row kernels (0) and the matrix cores (1); more pairs
    never go back."""
    cases = [(512, 2048, 512, 6, 0), (512, 2048, 512, 8, 1), (512, 2048, 512, 11.7, 1), (128, 2048, 512, 6.25, 0),
             (128, 2048, 512, 8, 1), (64, 1024, 1024, 6.25, 0), (64, 512, 512, 8, 1), (16, 2048, 512, 8, 0),
             (16, 2048, 512, 12.5, 0), (16, 2048, 512, 38, 0), (16, 2048, 512, 200, 1), (8, 2048, 1024, 40, 0),
             (32, 2048, 512, 11, 0), (32, 1024, 2048, 11, 0), (32, 1024, 2048, 64, 1), (64, 512, 2048, 11, 0),
             (32, 2048, 2048, 12.5, 1)]
    assert ask([f"iq2_mm_gains({int(p * E)}, {E}, {H}, {F})" for E, H, F, p, _ in cases]) == [c[-1] for c in cases]
    for E, H, F in [(512, 2048, 512), (64, 512, 2048), (16, 1024, 1024), (1, 512, 512)]:
        got = ask([f"iq2_mm_gains({int(p * E)}, {E}, {H}, {F})" for p in (0.1, 1, 5, 7, 8, 16, 64, 100, 128, 1000)])
        assert got == sorted(got) and got[-1] == 1


def test_native_columns(ask):
    """type, n_in, n_out, columns, matrices: columns per work-group, 1 where a work-group per column is the faster."""
    q4k, q5k, q6k, q3k, iq4nl = 12, 13, 14, 11, 20
    cases = [(q4k, 256, 20000, 4, 1, 1), (q4k, 256, 20000, 5, 1, 1), (q4k, 2560, 640, 32, 1, 1), (q4k, 2560, 640, 48, 1, 4),
             (q5k, 512, 2048, 5, 1, 1), (q6k, 512, 2048, 5, 1, 1), (q6k, 512, 2048, 12, 1, 4), (q6k, 8192, 1000, 24, 1, 1),
             (q6k, 8192, 1000, 48, 1, 4), (q6k, 4096, 4096, 7, 1, 4), (q4k, 2048, 64, 250, 1, 4),
             (q3k, 2048, 512, 16, 1, 1), (q3k, 2048, 512, 16, 2, 4), (q3k, 2048, 512, 1000, 1, 16),
             (iq4nl, 512, 2048, 3, 1, 1), (iq4nl, 512, 2048, 32, 1, 8), (iq4nl, 512, 2048, 4, 1, 1), (8, 256, 20000, 4, 1, 4),
             (8, 256, 20000, 5, 1, 8)]
    assert ask([f"native_cols({t}, {i}, {o}, {c}, {z})" for t, i, o, c, z, _ in cases]) == [c[-1] for c in cases]
    assert ask(["native_cols(8, 32, 2147483647, 2147483647, 2)"]) == [1]  # the grid's y dimension


def test_native_shared(ask):
    """Tokens, n_embd, n_ff_shared: two launches (1) or the stage kernels (0); rows, columns, matrices: the matrix cores
    (1) or the row kernels (0), which alone a prompt of few tokens takes (traced or not, the same order)."""
    few = [(1, 2048, 512, 1), (4, 2048, 512, 1), (5, 2048, 512, 0), (2, 2048, 2048, 1), (3, 2048, 2048, 0), (4, 4096, 4096, 0),
           (2, 4096, 4096, 0), (2, 3072, 1536, 1), (3, 3072, 1536, 0), (4, 4096, 256, 1)]
    assert ask([f"native_few_gains({T}, {H}, {F})" for T, H, F, _ in few]) == [c[-1] for c in few]
    mm = [(512, 1, 2, 0), (512, 4, 2, 0), (512, 64, 2, 0), (512, 127, 2, 0), (512, 128, 2, 1), (512, 128, 1, 0), (512, 256, 1, 1),
          (2048, 128, 1, 1), (4096, 32, 1, 0), (256, 128, 1, 0), (256, 1000, 1, 1)]
    assert ask([f"native_mm_gains({n}, {c}, {z})" for n, c, z, _ in mm]) == [c[-1] for c in mm]


def test_router_tiles(ask):
    """Tokens, experts, n_embd, f32 rows: k_router (0) or the tiles (1)."""
    cases = [(4, 512, 2048, 0, 0), (5, 512, 2048, 0, 1), (5, 512, 2048, 1, 1), (5, 8, 512, 0, 1), (5, 32, 4096, 0, 0),
             (8, 8, 4096, 0, 0), (16, 64, 4096, 0, 0), (64, 8, 4096, 0, 1), (16, 128, 4096, 0, 1), (5, 512, 4096, 0, 1),
             (5, 8, 4096, 1, 1), (127, 8, 4096, 0, 1)]
    assert ask([f"router_tiles({T}, {E}, {H}, {f})" for T, E, H, f, _ in cases]) == [c[-1] for c in cases]


def test_router_tile_wide(ask):
    cases = [(111, 1024, 0), (112, 512, 1), (127, 256, 0), (224, 256, 1), (127, 64, 0), (300, 64, 0), (600, 128, 1), (600, 8, 0)]
    assert ask([f"router_tile_wide({T}, {E})" for T, E, _ in cases]) == [c[-1] for c in cases]


def test_router_tile_grid(ask):
    """A product whose tiles a launch's grid does not hold (152064 rows by 16384 tokens, 10 GB of logits) is refused
    before any launch; every smaller one is taken."""
    cases = [(16384, 152064, 2048, 0, 0), (4096, 152064, 2048, 0, 1), (2056, 1 << 20, 8, 0, 0), (2000, 1 << 20, 8, 0, 1),
             (65535, 1024, 4096, 1, 1), (100, 1 << 24, 8, 0, 0), (5, 1 << 24, 8, 0, 1)]
    assert ask([f"router_tile_fits({T}, {E}, {H}, {f})" for T, E, H, f, _ in cases]) == [c[-1] for c in cases]
    assert ask(["router_tile_grid(203, 700, 0, 4, 8)", "router_tile_grid(16, 513, 0, 4, 4)"]) == [26 * 48, 4 * 40]
    import stratametal_amd as S
    for T, E, H in ((16384, 152064, 2048), (2056, 1 << 20, 8), (1, 1 << 26, 8)):
        assert S.lib().smoe_bf16_gemv(1 << 20, 1 << 20, 1 << 20, H, E, T, None) == -1
        assert b"exceed a launch's grid" in S.lib().smoe_last_error()


def test_junction_apart(ask):
    """Tokens, experts, n_embd, f32 rows: the junction in the router kernel (0) or a kernel of its own (1)."""
    cases = [(11, 512, 2048, 0, 0), (12, 512, 2048, 0, 1), (12, 64, 2048, 0, 0), (16, 64, 2048, 0, 0), (32, 64, 2048, 0, 1),
             (16, 256, 512, 1, 0), (32, 256, 512, 0, 1), (12, 8, 4096, 0, 0), (16, 64, 4096, 0, 0), (32, 64, 4096, 0, 1),
             (12, 1024, 4096, 0, 1), (12, 8, 4096, 1, 1), (12, 8, 2048, 1, 0), (32, 8, 512, 0, 0), (127, 8, 512, 0, 1)]
    assert ask([f"junction_apart({T}, {E}, {H}, {f})" for T, E, H, f, _ in cases]) == [c[-1] for c in cases]


def test_workspaces_grow_with_tokens():
    """A workspace sized for more tokens holds every smaller call's, whatever kernels each takes."""
    import ctypes as C

    import stratametal_amd as S
    L, p = S.lib(), 0x10000
    geoms = [S.Geom(), S.Geom(w_type=22, sh_type=22, n_expert=64), S.Geom(sh_type=S.Q3_K, sh_down_type=S.IQ4_NL)]
    for hc, lr in ((4, 320), (2, 64), (8, 960), (1, 1000)):
        h = S._Hc(hc, lr, 1e-6, p, p, p, p)
        tokens = list(range(0, 140)) + [300, 301, 1000, 4096]
        sizes = [L.smoe_hc_read_workspace_bytes(C.byref(h), 2048, T) for T in tokens]
        assert sizes == sorted(sizes), (hc, lr)
        for g in geoms:
            sizes = [L.smoe_ffn_workspace_bytes(C.byref(g.c()), C.byref(h), T) for T in tokens]
            assert sizes == sorted(sizes) and sizes[-1] > 0, (hc, lr, vars(g))
