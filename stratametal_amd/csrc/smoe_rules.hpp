// stratametal_amd/csrc/smoe_rules.hpp - which kernel a call runs on, where the choice was measured: plain host
// functions of a call's sizes, so that a CPU test can hold them to the times they come from
// (tests/test_dispatch_rules.py).
#pragma once

#include <cstdint>
#include <initializer_list>

namespace smoe {

// The register slots of a token's streams in k_hc_proj and k_hc_act: HC streams of NM values per thread.  Every slot
// is loaded (the indices clamped into the row), so a spare one is a load too: the least that hold hc streams of n
// values (with 4 and 8 streams of 2, 8 and 16 alone the read of 16 tokens, hc 1, n 1024, hc_lr 320, took 14.0 us,
// with branches around the loads 13.4, so 10.1).
constexpr int kHcStreams[] = {2, 4, 8}, kHcValues[] = {2, 4, 6, 8, 10, 12, 16};
constexpr int hc_streams(int hc) {
    for (const int s : kHcStreams)
        if (hc <= s) return s;
    return 8;
}
constexpr int hc_values(int n) {
    for (const int v : kHcValues)
        if (n <= 256 * v) return v;
    return 16;
}
// 16-byte pieces of a weight row per lane: hc n / 512 rounded up to a multiple of eight.
constexpr int hc_chunks(int n, int hc) { return (hc * n / 8 + 511) / 512 * 8; }

// The same for the pieces of an `up` row per lane of k_hc_mix (hc_lr / 64 rounded up; five for one piece: the read of
// 64 tokens, hc 5, n 512, hc_lr 64, 14.5 us, with branches around the loads 13.7, with one 13.0).
constexpr int kHcPieces[] = {1, 2, 3, 4, 5, 8, 16, 32};
constexpr int hc_pieces(int hc_lr) {
    for (const int p : kHcPieces)
        if (hc_lr <= 64 * p) return p;
    return 32;
}

// The norm's slots are loaded with the streams' (one memory round trip less: 2 us of 13 at one token, n 2560, hc 4)
// where both fit 256 registers beside the weight row's `more`, two waves per SIMD.
constexpr bool hc_norm_fits(int slots, int more) { return 2 * slots + more <= 192; }
// Where they don't, the norm is loaded with the streams by one wave per SIMD or, where the streams and the weight row
// alone fit, after the scales are formed by two: by two where that halves the rounds of work-groups over the 256 CUs
// and an XCD's L2 holds the weights (n 2048, hc 6, hc_lr 64: 16 tokens, 288 work-groups, 26.7 us in two rounds of one
// wave, 21.7 in one of two waves; 14 tokens, 252, 17.6 against 20.2; hc 8, hc_lr 320: 4 tokens, 328, 32.3 against
// 34.3).
constexpr bool hc_norm_ahead(int slots, int more, int64_t groups, int64_t weight_bytes) {
    return hc_norm_fits(slots, more) || slots + more > 192 || (groups + 255) / 256 % 2 == 1 ||
           weight_bytes > (int64_t)5 << 20;
}

// Whether the read of a batch runs on the matrix cores: from 17 tokens (a second 16-token tile) and 2^23 products of
// the projection, where the row-per-wave kernels' time, which grows with the tokens, has passed the four launches',
// which hardly does but grows with the streams and hc_lr.  Fitted to 60 shapes of 8 to 400 tokens; rows and matrix
// cores, us: hc 4, hc_lr 320, n 2048 30 and 28 at 17 tokens, 82 and 31 at 64, 1965 and 66 at 1000; n 512 11 and 24 at
// 17, 24 and 26 at 64, 38 and 28 at 128; hc 8, n 256 45 and 36 at 128; hc 4, hc_lr 64, n 2048 17 and 20 at 24, 32 and
// 21 at 64; hc 1, hc_lr 960, n 4096 114 and 35 at 17.
constexpr bool hc_mm_gains(int64_t T, int n, int hc, int hc_lr) {
    return T >= 17 && T * hc * n * hc_lr >= (int64_t)1 << 23 &&
           120 * T * n * (hc * (hc_lr + 80) + hc_lr + 160) >= (int64_t)92 * 32768 * (960 + 360 * hc + hc_lr);
}

// The write of T tokens: kHcWriteValues a value per thread; else 16-byte vectors (n % 4 == 0 and aligned buffers), a
// work-group's piece of y through one stream (kHcWriteStream) or through all (kHcWriteStreams: y read once, from
// where the launch is long; rows of few values leave lanes idle in every piece, and one or two streams re-read
// little, so earlier).  us by value, by stream and through all: hc 8, n 64, 200 tokens 2.5, 2.6, 3.5, 4000 tokens
// 7.3, 13.0, 6.5; hc 8, n 512, 64 tokens 2.7, 2.5, 3.4; hc 4, n 2048, 64 tokens 3.3, 2.6, 2.9, 1000 tokens 21.5,
// 10.6, 11.6, 4000 tokens 98, 56, 44.
enum HcWrite { kHcWriteValues, kHcWriteStream, kHcWriteStreams };
constexpr HcWrite hc_write_kind(int64_t T, int n, int hc) {
    const int64_t limit = n < 512 ? 15 << 16 : n < 768 ? 15 << 17 : hc <= 2 ? 6 << 20 : 11 << 20;
    const bool all = T * hc * n >= limit;
    return n < 64 || (n < 256 && !all) ? kHcWriteValues : all ? kHcWriteStreams : kHcWriteStream;
}

// Whether an IQ2_S layer's products of P routed pairs run on the matrix cores (tiles of 16 columns; the row kernels'
// cost grows with the columns).  An item's tiles go one after the other, so few experts leave the chip idle: from
// seven or eight pairs per expert on where the products' work-groups, each as long as its rows, fill it; else from
// 64, or 128 with fewer than 32 experts, where an expert's pairs are several items.  Rows against matrix cores, the
// whole call: 512 experts of 2048 x 512 389 and 408 us at 5.9 pairs, 648 and 472 at 11.7; 128 experts of 2048 x 512,
// most pairs in 16 of them, 150 and 189 at 6.3, 1.05 times as fast at 8; 16 experts 70 and 102 at 12.5, 137 and 188
// at 38, 1.3 times as fast at 100; 32 experts of 1024 x 2048 0.84 times at 11, 1.34 at 64; of 2048 x 2048 187 and 161
// at 12.5.
constexpr bool iq2_mm_gains(int64_t P, int E, int H, int F) {
    const bool fills = (E >= 64 || (E >= 32 && H * F >= 2048 * 2048)) && (int64_t)E * F * 8 / H >= 128 &&
                       (int64_t)E * H * 4 / F >= 128;
    return P >= (int64_t)E * (fills ? E >= 128 ? 7 : 8 : E >= 32 ? 64 : 128);
}

// The native types' GEMV of n_col columns (nz matrices by one launch): columns per work-group of the column tiles, or
// 1 for a work-group per column and eight rows.  The most of 16, 8 and 4 that is not half empty and leaves the chip
// two work-groups per CU, else 4; a tile's chain of columns is the longer one, so few work-groups of 4 columns go by
// columns (512 x 2048 at 16 columns 3.9 to 6.6 us by type against 5.0 to 8.5 in tiles, at 32 5.8 to 10.9 against 4.1
// to 8.4).  Q4_K, Q5_K and Q6_K, whose decode the tiles save little of, from six or eight columns and more
// work-groups, long rows more yet (by columns and in tiles: Q4_K 256 x 20000 at 4 columns 8.3 and 12.4, Q5_K 512 x
// 2048 at 5 3.2 and 3.7, Q6_K 8192 x 1000 at 24 40 and 49, at 48 1.4 times as fast in tiles).
constexpr int kNativeTileRows = 16;
constexpr int native_cols(int type, int n_in, int n_out, int n_col, int nz) {
    const int64_t rg = ((int64_t)n_out + kNativeTileRows - 1) / kNativeTileRows * nz;
    const bool k = type == 12 || type == 13 || type == 14;
    const int64_t least = !k || n_col >= 128 ? 224 : n_in <= 4096 ? 336 : 480;
    if (n_col < (!k ? 4 : rg >= 256 ? 6 : 8) || n_col / 4 >= 65535 || rg * ((n_col + 3) / 4) < least) return 1;
    for (const int c : {16, 8})
        if (2 * n_col > c && rg * ((n_col + c - 1) / c) >= 512) return c;
    return 4;
}

// A native shared expert of T tokens in two launches (k_native_gu, k_native_down): every work-group quantises its
// token's whole row again and takes eight rows of it, so the stage kernels, whose tokens share a row's decode and one
// quantised row, win where tokens times weights are many (the layer's call with the two launches against it, Q8_0: 4
// tokens 2048 x 512 1.16 times as fast, 1 token 4096 x 4096 1.00, 2 tokens 3072 x 1536 1.05, 2048 x 2048 1.14, 4
// tokens 0.97, 4096 x 4096 0.63; Q4_K 3 tokens 3072 x 1536 0.93).
constexpr bool native_few_gains(int T, int H, int F) { return T <= 4 && (int64_t)T * H * F <= (int64_t)10 << 20; }

// The native shared expert's products of a prompt on the matrix cores (nz matrices of n_out rows by one launch): a
// chunk of K after the other is a chain of latencies, so from 128 columns, and 128 tiles of 32 rows by 32 columns
// (the layer's call on the matrix cores against the row kernels: Q8_0 2048 x 512 0.81 at 5 columns, 0.88 at 64, 0.98
// at 128, 1.05 at 200; gate and up apart 0.70 at 8, 0.89 at 128; Q3_K 1.07 at 128, 1.42 at 400).
constexpr bool native_mm_gains(int n_out, int n_col, int nz) {
    return n_col >= 128 && (int64_t)((n_out + 31) / 32) * ((n_col + 31) / 32) * nz >= 128;
}

// Whether the router of T tokens without the fused junction runs k_router_tile: from five tokens on, but for long
// bf16 rows of few experts, whose waves walk K in stages while most of the chip is idle.  512 rows of 2048, k_router
// and the tiles, us: bf16 6.3 and 6.3 at 5 tokens, 8.4 and 6.4 at 16, 19.8 and 7.7 at 64, 126 and 38 at 600; f32 7.8
// and 5.9 at 5, 27 and 7.1 at 64.  bf16 rows of 4096, the tiles' gain: 8 experts -1.0 at 8 tokens, +1.6 at 64; 32
// experts -1.8 at 5; 128 experts -0.4 at 8, +0.3 at 16; 512 experts 0.0 at 5, +2.4 at 16.
constexpr bool router_tiles(int64_t T, int E, int H, bool f32) {
    return T >= 5 && (f32 || H <= 2560 || T * (E > 64 ? E : 64) >= 2048);
}

// The tile: few tokens or experts need the work-groups (bf16 4 rows by 4 tokens, f32 2 by 8), many of both re-read
// less in tiles of 4 by 8 (512 rows of 2048, bf16 9.6 against 10.4 us at 100 tokens, 11.4 against 10.7 at 127; rows
// of 4096 at 127 tokens in tiles of 4 by 8 the same with 400 and 512 experts, 4.6 us longer with 256 and 4.8 with 64;
// f32 64 experts 3.1 us longer at 300 tokens, 128 experts 0.3 at 448).
constexpr bool router_tile_wide(int64_t T, int E) { return T >= 112 && T * E >= 112 * 512; }

// The tiled router's one-dimensional grid: the tiles of tt tokens by 4 rr rows, those of a row group, or by_tok of a
// token tile, on one XCD (whole groups of 8).  A launch holds kGridGroups work-groups of 256 threads in a dimension and
// takes a larger grid modulo that, with no error: a larger product, of some 2^31 outputs and more, is refused.
constexpr int64_t kGridGroups = 0xFFFFFFFFll / 256;
constexpr bool router_by_tok(int64_t T, int64_t E, bool f32) { return T * 4 > E * (f32 ? 4 : 2); }  // x, not W, on every XCD
constexpr int64_t router_tile_grid(int64_t T, int64_t E, bool f32, int rr, int tt) {
    const int64_t rb = (E + 4 * rr - 1) / (4 * rr), tb = (T + tt - 1) / tt;
    return router_by_tok(T, E, f32) ? (tb + 7) / 8 * 8 * rb : (rb + 7) / 8 * 8 * tb;
}
constexpr bool router_tile_fits(int64_t T, int E, int H, bool f32) {
    const bool wide = router_tile_wide(T, E);
    return router_tile_grid(T, E, f32, f32 && !wide ? 2 : 4, !f32 && !wide ? 4 : 8) + T + T * (H / 32) / 8 < kGridGroups;
}

// Whether the decode path runs the junction of T tokens as a kernel of its own: fused into the router kernel it saves
// the launch, and repeats the norm in every work-group of the router.  Apart from 12 tokens on where the tiled
// router's gain passes the launch, us: bf16, 512 experts of 2048 +0.4 at 10 tokens, +0.8 at 12, +3.6 at 16, 28.8 to
// 12.0 at 48; 64 experts of 2048 -0.6 at 12, -1.3 at 16, +0.3 at 32; of 4096 -1.4 at 12, +4.4 at 32; 256 experts of
// 512 +0.4 at 12, +1.1 at 32; 8 experts of 512 -0.6 at 32, +7 at 127; f32 rows longer than 2048 +4 and more at any
// number of experts.
constexpr bool junction_apart(int64_t T, int E, int H, bool f32) {
    return T >= 12 && ((f32 && H > 2048) || T >= (H >= 2048 ? 32 : 80) ||
                       T * E >= (H >= 2560 ? 2048 : H >= 2048 ? 4096 : 8192));
}

}  // namespace smoe
