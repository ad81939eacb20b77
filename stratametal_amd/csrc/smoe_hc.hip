// stratametal_amd/csrc/smoe_hc.hip - the hyper-connection ends of the layer call (gfx950, wave64).
//
// FfnExec::run reads the layer's input from hc residual streams through the gated residual and writes the MoE
// block's output back onto every stream (metal/src/layer_exec.cpp:469,531; metal/include/strata/metal/gr.hpp:1-48).
// Per token, R is [hc][n] f32 (stream c at c * n):
//   read:  xn = R * rs_c * w_norm (rs_c = 1 / sqrt(mean(R_c^2) + eps); w_norm is the stored (1 + w)), act = bf16(xn);
//          proj_r = act . down_r (r < hc_lr), lq = bf16(silu(proj_r / hc)); gate_i = lq . up_i (i < hc * n);
//          mixed_d = (sum_c xn_cd * sigmoid(gate_cd)) / hc;  inject_c = act . inj_c;
//   write: out_cd = R_cd + y_d * 2 sigmoid(inject_c / hc).
// For few tokens the read is two bandwidth-bound bf16 GEMVs in a chain (about 10.5 MB of weights per call at n 2048,
// hc 4, hc_lr 320, as much as the MoE block itself), so it is two launches: k_hc_proj (the norm, the activations staged
// in LDS, the down and inject rows) and k_hc_mix (lq, the up rows, the gated mean).  Their reduction orders are fixed
// and restated by the test oracle (or_hc_read_dev, or_hc_write_dev).  For a batch of tokens (hc_mm_gains) both products
// run on the matrix cores: k_hc_act, k_hc_proj_mm, k_hc_lq, k_hc_mix_mm.
#include "smoe_device.hpp"
#include "smoe_gemv.hpp"
#include "smoe_launch.hpp"
#include "smoe_rules.hpp"

#include <type_traits>

namespace smoe {

namespace {

// Per-stream scale rs_c of one token: thread i of 256 adds fmaf(v, v, acc) over d = i, i + 256, ... from 0, the wave
// butterfly 32..1, the four wave sums ((w0 + w1) + w2) + w3 (LDS `wsum`: 4 floats per stream); rs = 1 / sqrtf(ss / n
// + eps).  Every thread returns with rs of every stream in `rs_s` (LDS, hc floats).  `v[c][m]` holds R_c[tid + 256 m].
template <int HC, int NM>
__device__ __forceinline__ void stream_scales(const float (&v)[HC][NM], int hc, int n, float eps, float (*wsum)[4],
                                              float* rs_s) {
    const int tid = threadIdx.x;
    float acc[HC];
#pragma unroll
    for (int c = 0; c < HC; ++c) {
        acc[c] = 0.0f;
#pragma unroll
        for (int m = 0; m < NM; ++m)
            if (tid + 256 * m < n) acc[c] = __builtin_fmaf(v[c][m], v[c][m], acc[c]);
    }
    wave_sum_xor_fast_n<HC>(acc);
    if ((tid & 63) == 0) {
#pragma unroll
        for (int c = 0; c < HC; ++c) wsum[c][tid >> 6] = acc[c];
    }
    __syncthreads();
    if (tid < hc) {
        const float ss = ((wsum[tid][0] + wsum[tid][1]) + wsum[tid][2]) + wsum[tid][3];
        rs_s[tid] = 1.0f / __builtin_sqrtf(ss / (float)n + eps);
    }
    __syncthreads();
}

// A token's streams (or the norm's rows) in a thread's slots; those past hc or n hold the last ones' values.
template <int HC, int NM>
__device__ __forceinline__ void stream_slots(const float* __restrict__ rows, int n, int hc, float (&v)[HC][NM]) {
#pragma unroll
    for (int c = 0; c < HC; ++c)
#pragma unroll
        for (int m = 0; m < NM; ++m) v[c][m] = rows[min(c, hc - 1) * n + min((int)threadIdx.x + 256 * m, n - 1)];
}

}  // namespace

// k_hc_proj: grid (ceil((hc_lr + hc) / 4), T), 256 threads; block (b, t) takes rows 4b .. 4b + 3 of [down; inj] for
// token t, one row per wave (lane l adds the 8-element chunks l, l + 64, ... in element order, then the xor butterfly
// 32..1, as the router).  Every block forms the token's scales and stages act = bf16((R * rs) * w_norm) in LDS; block
// (0, t) also writes rs[t][c] for k_hc_mix.  Bound by latency at one token (81 work-groups): every load it needs (its
// streams, norm and weight row) is issued up front, unconditionally, so that one memory round trip covers them all
// (with the loads under their bounds' branches 13.1 us, of which the bytes take 1.2).  AHEAD: the norm among them
// (hc_norm_ahead).
template <int HC, int NM, int MAXC, bool AHEAD>
__global__ __launch_bounds__(256) void k_hc_proj(const float* __restrict__ R, const float* __restrict__ norm,
                                                  const uint16_t* __restrict__ down, const uint16_t* __restrict__ inj,
                                                  int n, int hc, int hc_lr, float eps, float* __restrict__ proj,
                                                  float* __restrict__ inject, float* __restrict__ rs_out) {
    extern __shared__ __align__(16) uint16_t act_s[];  // hc * n bf16
    __shared__ float wsum[HC][4];
    __shared__ float rs_s[HC];
    const int t = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int hd = hc * n;
    const int rows = hc_lr + hc;
    const int row = min((int)blockIdx.x * 4 + (tid >> 6), rows - 1);  // clamped: every load in bounds
    const uint16_t* wr = row < hc_lr ? down + (size_t)row * hd : inj + (size_t)(row - hc_lr) * hd;
    const int chunks = hd >> 3;
    const float* Rt = R + (size_t)t * hd;
    float v[HC][NM], nv[HC][NM];
    uint4 wv[MAXC];
    stream_slots<HC, NM>(Rt, n, hc, v);
    if constexpr (AHEAD) stream_slots<HC, NM>(norm, n, hc, nv);
#pragma unroll
    for (int j = 0; j < MAXC; ++j) wv[j] = *reinterpret_cast<const uint4*>(wr + 8 * min(lane + 64 * j, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    stream_scales<HC, NM>(v, hc, n, eps, wsum, rs_s);
    if (blockIdx.x == 0 && tid < hc) rs_out[(size_t)t * hc + tid] = rs_s[tid];
#pragma unroll
    for (int c = 0; c < HC; ++c) {
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int d = tid + 256 * m;
            if (c >= hc || d >= n) continue;
            const float w = AHEAD ? nv[c][m] : norm[c * n + d];
            act_s[c * n + d] = (uint16_t)f32_to_bf16((v[c][m] * rs_s[c]) * w);
        }
    }
    __syncthreads();
    if ((int)blockIdx.x * 4 + (tid >> 6) >= rows) return;
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < MAXC; ++j) {
        const int c = lane + 64 * j;
        if (c < chunks) {
            const uint4 xv = *reinterpret_cast<const uint4*>(act_s + 8 * c);
            const uint32_t xq[4] = {xv.x, xv.y, xv.z, xv.w};
            const uint32_t wq[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc = __builtin_fmaf(u2f(xq[q] << 16), u2f(wq[q] << 16), acc);
                acc = __builtin_fmaf(u2f(xq[q] & 0xFFFF0000u), u2f(wq[q] & 0xFFFF0000u), acc);
            }
        }
    }
    acc = wave_sum_xor_fast(acc);
    if (lane == 0) {
        if (row < hc_lr) proj[(size_t)t * hc_lr + row] = acc;
        else if (inject) inject[(size_t)t * hc + row - hc_lr] = acc;
    }
}

// k_hc_mix: grid (n / 8, T), 256 threads; block (b, t) forms mixed[t][8b .. 8b + 7].  lq = bf16(silu(proj / hc)) in
// LDS; the 8 hc rows i = c * n + d of `up` (hc_lr bf16 each) go 8 lanes per row (lane l adds the 8-element chunks
// l, l + 8, ... in element order, then the xor butterfly 4, 2, 1), wave w taking the rows of streams w, w + 4, ...;
// gated = xn * sigmoid(gate) with xn = (R * rs) * w_norm as k_hc_proj forms it; mixed = (((0 + g_0) + g_1) + ...) / hc.
template <int LQC>
__global__ __launch_bounds__(256) void k_hc_mix(const float* __restrict__ R, const float* __restrict__ norm,
                                                 const uint16_t* __restrict__ up, const float* __restrict__ proj,
                                                 const float* __restrict__ rs, int n, int hc, int hc_lr,
                                                 float* __restrict__ mixed) {
    __shared__ __align__(16) uint16_t lq_s[64 * LQC];
    __shared__ float gated[8][8];  // [stream][d - 8b], hc <= 8
    const int t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int d0 = blockIdx.x * 8;
    const int hd = hc * n;
    const int lchunks = hc_lr >> 3;  // 8-element chunks of a row
    const int g = lane >> 3, l = lane & 7;
    // the first row of this 8-lane group (stream `wave`, d0 + g), loaded before lq is formed
    uint4 wv[LQC];
    {
        const int c = min(wave, hc - 1);
        const uint16_t* wr = up + ((size_t)c * n + d0 + g) * hc_lr;
#pragma unroll
        for (int j = 0; j < LQC; ++j) {
            wv[j] = *reinterpret_cast<const uint4*>(wr + 8 * min(l + 8 * j, lchunks - 1));  // clamped: no branch
        }
    }
    for (int i = tid; i < hc_lr; i += 256) {
        const float z = proj[(size_t)t * hc_lr + i] / (float)hc;
        lq_s[i] = (uint16_t)f32_to_bf16(z / (1.0f + expf_smoe(-z)));
    }
    __syncthreads();
    for (int c = wave; c < hc; c += 4) {
        const size_t i = (size_t)c * n + d0 + g;
        if (c != wave) {  // streams beyond the first four: this wave's next row
            const uint16_t* wr = up + i * hc_lr;
#pragma unroll
            for (int j = 0; j < LQC; ++j) {
                wv[j] = *reinterpret_cast<const uint4*>(wr + 8 * min(l + 8 * j, lchunks - 1));
            }
        }
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < LQC; ++j) {
            const int ch = l + 8 * j;
            if (ch < lchunks) {
                const uint4 xq4 = *reinterpret_cast<const uint4*>(lq_s + 8 * ch);
                const uint32_t xq[4] = {xq4.x, xq4.y, xq4.z, xq4.w};
                const uint32_t wq[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    acc = __builtin_fmaf(u2f(xq[q] << 16), u2f(wq[q] << 16), acc);
                    acc = __builtin_fmaf(u2f(xq[q] & 0xFFFF0000u), u2f(wq[q] & 0xFFFF0000u), acc);
                }
            }
        }
        acc = acc + xor_swap<4>(acc);
        acc = acc + xor_swap<2>(acc);
        acc = acc + xor_swap<1>(acc);
        if (l == 0) {
            const float xn = (R[(size_t)t * hd + i] * rs[(size_t)t * hc + c]) * norm[i];
            gated[c][g] = xn * sigmoid(acc);
        }
    }
    __syncthreads();
    if (tid < 8) {
        float m = 0.0f;
        for (int c = 0; c < hc; ++c) m = m + gated[c][tid];
        mixed[(size_t)t * n + d0 + tid] = m / (float)hc;
    }
}

// k_hc_write: out[t][c][d] = R[t][c][d] + y[t][d] * (2 * sigmoid(inject[t][c] / hc)); out may be R.
__global__ __launch_bounds__(256) void k_hc_write(const float* R, const float* __restrict__ y,
                                                   const float* __restrict__ inject, int n, int hc, int64_t total,
                                                   float* out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t row = i / n;  // t * hc + c
    const int d = (int)(i - row * n);
    const int64_t t = row / hc;
    const float s = sigmoid(inject[row] / (float)hc);
    out[i] = R[i] + y[t * n + d] * (2.0f * s);
}

// The same with R, y and out as 16-byte vectors (n % 4 == 0): block (p, c) takes 256 four-value pieces of y of a token
// through stream c, or with one block in y through every stream, so y is read once (hc_write_kind).
__global__ __launch_bounds__(256) void k_hc_write4(const float* R, const float* __restrict__ y,
                                                    const float* __restrict__ inject, int n4, int hc, int parts,
                                                    float* out) {
    const int t = blockIdx.x / parts, d = (blockIdx.x % parts) * 256 + threadIdx.x;
    if (d >= n4) return;
    const float4 yv = reinterpret_cast<const float4*>(y)[(size_t)t * n4 + d];
    for (int c = blockIdx.y; c < hc; c += gridDim.y) {
        const float s = sigmoid(inject[(size_t)t * hc + c] / (float)hc), g = 2.0f * s;
        const size_t i = ((size_t)t * hc + c) * n4 + d;
        const float4 r = reinterpret_cast<const float4*>(R)[i];
        reinterpret_cast<float4*>(out)[i] = make_float4(r.x + yv.x * g, r.y + yv.y * g, r.z + yv.z * g, r.w + yv.w * g);
    }
}

// ------------------------------------------------------------------------------------------------ many tokens
// The read as two bf16 matrix products: every bf16 product is exact in f32 and the sums are the matrix core's f32
// accumulation, in the hardware's order and over the K slices below, so proj, inject and the gates are the exact dots
// to f32 sums' accuracy, not bit for bit the row-per-wave kernels' (each GEMV launch reads all the weights once per
// token from the caches: 1591 + 393 us at 1000 tokens of n 2048, hc 4, hc_lr 320).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// k_hc_act: one work-group per token: the stream scales (as k_hc_proj forms them) into rs, and act = bf16((R * rs) *
// w_norm) through LDS to memory as 16-byte pieces.  Bound by reading R once.
template <int HC, int NM>
__global__ __launch_bounds__(256) void k_hc_act(const float* __restrict__ R, const float* __restrict__ norm, int n,
                                                 int hc, float eps, uint16_t* __restrict__ act,
                                                 float* __restrict__ rs_out) {
    extern __shared__ __align__(16) uint16_t act_s[];  // hc * n bf16
    __shared__ float wsum[HC][4];
    __shared__ float rs_s[HC];
    const int t = blockIdx.x, tid = threadIdx.x;
    const int hd = hc * n;
    const float* Rt = R + (size_t)t * hd;
    float v[HC][NM], nv[HC][NM];
    stream_slots<HC, NM>(Rt, n, hc, v);
    if constexpr (hc_norm_fits(HC * NM, 0)) stream_slots<HC, NM>(norm, n, hc, nv);
    __builtin_amdgcn_sched_barrier(0);
    stream_scales<HC, NM>(v, hc, n, eps, wsum, rs_s);
    if (tid < hc) rs_out[(size_t)t * hc + tid] = rs_s[tid];
#pragma unroll
    for (int c = 0; c < HC; ++c)
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int d = tid + 256 * m;
            if (c >= hc || d >= n) continue;
            const float w = hc_norm_fits(HC * NM, 0) ? nv[c][m] : norm[c * n + d];
            act_s[c * n + d] = (uint16_t)f32_to_bf16((v[c][m] * rs_s[c]) * w);
        }
    __syncthreads();
    u32x4* dst = reinterpret_cast<u32x4*>(act + (size_t)t * hd);
    for (int p = tid; p < hd / 8; p += 256) dst[p] = reinterpret_cast<const u32x4*>(act_s)[p];
}

// k_hc_proj_mm: part[s][t][r] = act[t] . [down; inj][r] over K slice s.  Work-group tile 64 tokens x 128 rows (wave w:
// rows 32 w .. + 31, two row tiles by four token tiles), K in chunks of 64 through two LDS buffers (rows at a 144-byte
// pitch: a 16-row fragment read covers the 64 banks once), the next two chunks' loads in flight in registers, one
// barrier per chunk.  The product has few output tiles (48 at 1000 tokens of 324 rows) and a deep K (8192), so K is split
// over `splits` work-groups (hc_splits), whose partial sums k_hc_lq adds in slice order.  Slices are the fastest index
// and a power of two: the work-groups of an XCD share their K slices of the weights and activations, which its L2 holds.
constexpr int kHpTok = 64, kHpRows = 128, kHpK = 64, kHpPitch = kHpK * 2 + 16;
constexpr int kHpLa = kHpTok * 8 / 256, kHpLb = kHpRows * 8 / 256;  // 16-byte pieces of a chunk per thread

__global__ __launch_bounds__(256) void k_hc_proj_mm(const uint16_t* __restrict__ act, const uint16_t* __restrict__ down,
                                                     const uint16_t* __restrict__ inj, int hd, int hc_lr, int rows,
                                                     int ld, int T, int splits, int per, int n_rb,
                                                     float* __restrict__ part) {
    __shared__ __align__(16) uint8_t sa[2][kHpTok * kHpPitch];
    __shared__ __align__(16) uint8_t sb[2][kHpRows * kHpPitch];
    const int s = blockIdx.x % splits, tile = blockIdx.x / splits;
    const int t0 = (tile / n_rb) * kHpTok, r0 = (tile % n_rb) * kHpRows;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, i = lane & 15;
    const int nk = min(per, hd / kHpK - s * per);  // this slice's chunks, at least one
    // a thread's pieces of a chunk: piece tid % 8 of rows tid / 8 + 32 j (rows clamped: the tails' loads stay in bounds,
    // their results are not stored)
    const int pc = tid & 7, pr = tid >> 3;
    const uint16_t* asrc[kHpLa];
    const uint16_t* bsrc[kHpLb];
#pragma unroll
    for (int j = 0; j < kHpLa; ++j)
        asrc[j] = act + (size_t)min(t0 + pr + 32 * j, T - 1) * hd + (size_t)s * per * kHpK + 8 * pc;
#pragma unroll
    for (int j = 0; j < kHpLb; ++j) {
        const int r = min(r0 + pr + 32 * j, rows - 1);
        bsrc[j] = (r < hc_lr ? down + (size_t)r * hd : inj + (size_t)(r - hc_lr) * hd) + (size_t)s * per * kHpK + 8 * pc;
    }
    u32x4 ra[2][kHpLa], rw[2][kHpLb];
    auto load = [&](auto slot, int k0) {
        constexpr int P = decltype(slot)::value;
#pragma unroll
        for (int j = 0; j < kHpLa; ++j) ra[P][j] = *reinterpret_cast<const u32x4*>(asrc[j] + k0);
#pragma unroll
        for (int j = 0; j < kHpLb; ++j) rw[P][j] = *reinterpret_cast<const u32x4*>(bsrc[j] + k0);
    };
    auto stash = [&](auto slot) {
        constexpr int P = decltype(slot)::value;
#pragma unroll
        for (int j = 0; j < kHpLa; ++j) *reinterpret_cast<u32x4*>(&sa[P][(pr + 32 * j) * kHpPitch + 16 * pc]) = ra[P][j];
#pragma unroll
        for (int j = 0; j < kHpLb; ++j) *reinterpret_cast<u32x4*>(&sb[P][(pr + 32 * j) * kHpPitch + 16 * pc]) = rw[P][j];
    };
    using Zero = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    load(Zero{}, 0);
    load(One{}, min(1, nk - 1) * kHpK);
    stash(Zero{});
    __syncthreads();
    f32x4 acc[2][4];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[m][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto chunk = [&](int kc, auto parity) {
        constexpr int P = decltype(parity)::value;
        using Q = std::integral_constant<int, 1 - P>;
        load(parity, min(kc + 2, nk - 1) * kHpK);  // (past the end: the last chunk again, which nobody reads)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int st = 0; st < kHpK / 32; ++st) {
            bf16x8 w[2], a[4];
#pragma unroll
            for (int m = 0; m < 2; ++m)
                w[m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                                      &sb[P][(32 * wave + 16 * m + i) * kHpPitch + 64 * st + 16 * q]));
#pragma unroll
            for (int b = 0; b < 4; ++b)
                a[b] = __builtin_bit_cast(bf16x8,
                                          *reinterpret_cast<const u32x4*>(&sa[P][(16 * b + i) * kHpPitch + 64 * st + 16 * q]));
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[m], a[b], acc[m][b], 0, 0, 0);
        }
        stash(Q{});
        __syncthreads();
    };
    int kc = 0;
    for (; kc + 1 < nk; kc += 2) {
        chunk(kc, Zero{});
        chunk(kc + 1, One{});
    }
    if (kc < nk) chunk(kc, Zero{});
    // lane (q, i) holds rows 4 q .. + 3 of token i of each tile: one 16-byte store (ld % 4 == 0)
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int t = t0 + 16 * b + i, r = r0 + 32 * wave + 16 * m + 4 * q;
            if (t < T && r < ld) *reinterpret_cast<f32x4*>(part + ((size_t)s * T + t) * ld + r) = acc[m][b];
        }
}

// k_hc_lq: one work-group per token: the K slices' sums in slice order, lq = bf16(silu(proj / hc)) (zero from hc_lr to
// kp, the mix kernel's whole chunks) and inject.
__global__ __launch_bounds__(256) void k_hc_lq(const float* __restrict__ part, int T, int splits, int ld, int hc,
                                                int hc_lr, int kp, uint16_t* __restrict__ lq, float* __restrict__ inject) {
    const int t = blockIdx.x, n = max(kp, hc_lr + hc);
    for (int r = threadIdx.x; r < n; r += 256) {
        float v = 0.0f;
        if (r < hc_lr + hc) {
            const float* p = part + (size_t)t * ld + r;
            v = p[0];
#pragma unroll 8
            for (int s = 1; s < splits; ++s) v = v + p[(size_t)s * T * ld];
        }
        if (r < kp) {
            const float z = v / (float)hc;
            lq[(size_t)t * kp + r] = r < hc_lr ? (uint16_t)f32_to_bf16(z / (1.0f + expf_smoe(-z))) : (uint16_t)0;
        }
        if (inject && r >= hc_lr && r < hc_lr + hc) inject[(size_t)t * hc + r - hc_lr] = v;
    }
}

// k_hc_mix_mm: mixed[t][d] for 16 NT tokens x 64 values of d per work-group; wave w owns 16 values of d in every
// stream, so that a lane ends with the gates of all streams of its (token, d) and forms the gated mean in registers.
// lq of the tokens in LDS (pitch kp * 2 + 16 bytes); the wave's `up` rows stream from memory in chunks of 64 of K, the
// next chunk's loads in flight.  The d ranges are the fastest index, so that where n / 64 is a multiple of 8 the token
// blocks of a d range share an XCD, whose L2 serves the rows each of them reads again.  1000 tokens of n 2048, hc 4: 29 us,
// of which the bytes (R, the gates' rows, mixed: 52 MB) take 11 and VALU issue, a sigmoid per value and stream, half.
template <int HC, int NT>
__global__ __launch_bounds__(256) void k_hc_mix_mm(const float* __restrict__ R, const float* __restrict__ norm,
                                                    const uint16_t* __restrict__ up, const uint16_t* __restrict__ lq,
                                                    const float* __restrict__ rs, int n, int hc, int hc_lr, int kp,
                                                    int T, float* __restrict__ mixed) {
    extern __shared__ __align__(16) uint8_t lq_s[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, i = lane & 15;
    const int nd = n >> 6;
    const int t0 = (blockIdx.x / nd) * 16 * NT, d0 = (blockIdx.x % nd) * 64 + 16 * wave;
    const int hd = hc * n, pitch = kp * 2 + 16, pieces = kp >> 3;
    const uint16_t* wrow[HC];
#pragma unroll
    for (int c = 0; c < HC; ++c) wrow[c] = up + ((size_t)min(c, hc - 1) * n + d0 + i) * hc_lr;
    u32x4 w[2][HC][2];
    auto load = [&](auto slot, int k0) {
        constexpr int P = decltype(slot)::value;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const int k = k0 + 32 * st + 8 * q;  // (the tail past hc_lr: zeros, not the next row's values)
#pragma unroll
            for (int c = 0; c < HC; ++c)
                w[P][c][st] = k < hc_lr ? *reinterpret_cast<const u32x4*>(wrow[c] + k) : u32x4{0, 0, 0, 0};
        }
    };
    using Zero = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    load(Zero{}, 0);
    for (int p = tid; p < 16 * NT * pieces; p += 256) {
        const int r = p / pieces, o = p - r * pieces;
        *reinterpret_cast<u32x4*>(lq_s + (size_t)r * pitch + 16 * o) =
            *reinterpret_cast<const u32x4*>(lq + (size_t)min(t0 + r, T - 1) * kp + 8 * o);
    }
    __syncthreads();
    f32x4 acc[HC][NT];
#pragma unroll
    for (int c = 0; c < HC; ++c)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[c][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto chunk = [&](int k0, auto parity) {
        constexpr int P = decltype(parity)::value;
        load(std::integral_constant<int, 1 - P>{}, k0 + 64);  // (past the end: zeros)
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            bf16x8 a[NT];
#pragma unroll
            for (int b = 0; b < NT; ++b)
                a[b] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(lq_s + (size_t)(16 * b + i) * pitch +
                                                                                  2 * (k0 + 32 * st + 8 * q)));
#pragma unroll
            for (int c = 0; c < HC; ++c) {
                const bf16x8 wv = __builtin_bit_cast(bf16x8, w[P][c][st]);
#pragma unroll
                for (int b = 0; b < NT; ++b) acc[c][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, a[b], acc[c][b], 0, 0, 0);
            }
        }
    };
    // lane (q, i) ends with the gates of d .. d + 3 of token i of each tile; R of a token tile is loaded a tile ahead (the
    // first before the products)
    const int d = d0 + 4 * q;
    f32x4 xr[2][HC], nv[HC];
    auto load_r = [&](f32x4(&x)[HC], int b) {
        const float* p = R + (size_t)min(t0 + 16 * b + i, T - 1) * hd + d;
#pragma unroll
        for (int c = 0; c < HC; ++c) x[c] = *reinterpret_cast<const f32x4*>(p + (size_t)min(c, hc - 1) * n);
    };
#pragma unroll
    for (int c = 0; c < HC; ++c) nv[c] = *reinterpret_cast<const f32x4*>(norm + (size_t)min(c, hc - 1) * n + d);
    load_r(xr[0], 0);
    int k0 = 0;
    for (; k0 + 64 < kp; k0 += 128) {
        chunk(k0, Zero{});
        chunk(k0 + 64, One{});
    }
    if (k0 < kp) chunk(k0, Zero{});
#pragma unroll
    for (int b = 0; b < NT; ++b) {
        if (b + 1 < NT) load_r(xr[(b + 1) & 1], b + 1);
        const int t = t0 + 16 * b + i;
        f32x4 m = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < HC; ++c) {
            if (c >= hc) break;
            const float sc = rs[(size_t)min(t, T - 1) * hc + c];
#pragma unroll
            for (int r = 0; r < 4; ++r) m[r] = m[r] + ((xr[b & 1][c][r] * sc) * nv[c][r]) * sigmoid(acc[c][b][r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) m[r] = m[r] / (float)hc;
        if (t < T) *reinterpret_cast<f32x4*>(mixed + (size_t)t * n + d) = m;
    }
}

// go(HC, NM) with the slots of hc streams of n values
template <int V>
using Int = std::integral_constant<int, V>;
template <class Go>
static void hc_slots(int n, int hc, Go go) {
    auto values = [&](auto HC) {
        switch (hc_values(n)) {
            case 2: go(HC, Int<2>{}); break;
            case 4: go(HC, Int<4>{}); break;
            case 6: go(HC, Int<6>{}); break;
            case 8: go(HC, Int<8>{}); break;
            case 10: go(HC, Int<10>{}); break;
            case 12: go(HC, Int<12>{}); break;
            default: go(HC, Int<16>{}); break;
        }
    };
    switch (hc_streams(hc)) {
        case 2: values(Int<2>{}); break;
        case 4: values(Int<4>{}); break;
        default: values(Int<8>{}); break;
    }
}

// The shapes that run on the matrix cores where hc_mm_gains says so: whole 64-value chunks of a stream and an lq tile
// within 64 KiB of LDS; others keep the row-per-wave kernels.
constexpr int kHcMmMaxLr = 960;
static int hc_kp(int hc_lr) { return (hc_lr + 63) / 64 * 64; }
static int hc_ld(int hc_lr, int hc) { return (hc_lr + hc + 3) / 4 * 4; }
// K slices: a power of two up to 32 that fills the chip about once with two work-groups per CU.
constexpr int kHpGroups = 512;
static int hc_splits(int tiles, int chunks) {
    int s = 1;
    while (s < 32 && 2 * s <= chunks && 2 * s * tiles <= kHpGroups) s *= 2;
    return s;
}

bool hc_mm_shape(int64_t T, int n, int hc, int hc_lr) {
    return hc_shape_ok(n, hc, hc_lr) && hc_mm_gains(T, n, hc, hc_lr) && n % 64 == 0 && hc_lr <= kHcMmMaxLr;
}
// The scratch of the matrix-core read (act, the K slices' sums, lq), growing with T: part is bounded by the slices'
// largest count for few tokens, by the launch's work-groups' tiles, or by one slice.
void hc_mm_bytes(int64_t T, int n, int hc, int hc_lr, size_t* act, size_t* part, size_t* lq) {
    const size_t rows = (size_t)T * hc_ld(hc_lr, hc) * 4, tiles = (size_t)kHpGroups * kHpTok * kHpRows * 4;
    *act = (size_t)T * hc * n * 2;
    *part = rows > tiles ? rows : (32 * rows < tiles ? 32 * rows : tiles);
    *lq = (size_t)T * hc_kp(hc_lr) * 2;
}

hipError_t launch_hc_read_mm(const float* R, const float* norm, const uint16_t* down, const uint16_t* up,
                             const uint16_t* inj, int T, int n, int hc, int hc_lr, float eps, float* rs, uint16_t* act,
                             float* part, uint16_t* lq, float* mixed, float* inject, hipStream_t s) {
    if (!hc_mm_shape(T, n, hc, hc_lr)) return hipErrorInvalidValue;
    const int hd = hc * n, rows = hc_lr + hc, ld = hc_ld(hc_lr, hc), kp = hc_kp(hc_lr);
    const size_t lds = (size_t)hd * 2;
    hc_slots(n, hc, [&](auto HC, auto NM) {
        hipLaunchKernelGGL((k_hc_act<HC(), NM()>), dim3((unsigned)T), dim3(256), lds, s, R, norm, n, hc, eps, act, rs);
    });
    const int n_tb = (T + kHpTok - 1) / kHpTok, n_rb = (rows + kHpRows - 1) / kHpRows, chunks = hd / kHpK;
    int splits = hc_splits(n_tb * n_rb, chunks);
    const int per = (chunks + splits - 1) / splits;
    splits = (chunks + per - 1) / per;  // every slice holds a chunk
    hipLaunchKernelGGL(k_hc_proj_mm, dim3((unsigned)(splits * n_tb * n_rb)), dim3(256), 0, s, act, down, inj, hd, hc_lr,
                       rows, ld, T, splits, per, n_rb, part);
    hipLaunchKernelGGL(k_hc_lq, dim3((unsigned)T), dim3(256), 0, s, part, T, splits, ld, hc, hc_lr, kp, lq, inject);
    // 64-token tiles where they fill the chip (T 64, n 2048: 35.2 against 30.1 us the whole read; T 1000: 64.9 against 73.1)
    const int nt = (int64_t)((T + 63) / 64) * (n / 64) >= 256 && hc <= 4 && kp <= 448 ? 4 : 2;
    const unsigned grid = (unsigned)((T + 16 * nt - 1) / (16 * nt)) * (unsigned)(n / 64);
    const size_t tile = (size_t)16 * nt * (kp * 2 + 16);
#define SMOE_HCM(HCv, NTv)                                                                                         \
    hipLaunchKernelGGL((k_hc_mix_mm<HCv, NTv>), dim3(grid), dim3(256), tile, s, R, norm, up, lq, rs, n, hc, hc_lr, kp, T, \
                       mixed)
    if (hc <= 2) {
        if (nt == 4) SMOE_HCM(2, 4);
        else SMOE_HCM(2, 2);
    } else if (hc <= 4) {
        if (nt == 4) SMOE_HCM(4, 4);
        else SMOE_HCM(4, 2);
    } else {
        SMOE_HCM(8, 2);
    }
#undef SMOE_HCM
    return hipGetLastError();
}

bool hc_shape_ok(int n, int hc, int hc_lr) {
    if (n <= 0 || hc <= 0 || hc_lr <= 0) return false;
    if (n % 8 || hc_lr % 8 || n > 4096 || hc > 8 || hc_lr > 2048) return false;
    return (int64_t)hc * n <= 16384;  // the activations in LDS: 32 KiB of bf16
}

hipError_t launch_hc_read(const float* R, const float* norm, const uint16_t* down, const uint16_t* up, const uint16_t* inj,
                          int n_tok, int n, int hc, int hc_lr, float eps, float* proj, float* rs, float* mixed,
                          float* inject, hipStream_t s) {
    if (!hc_shape_ok(n, hc, hc_lr) || n_tok <= 0) return hipErrorInvalidValue;
    const int hd = hc * n;
    dim3 g1((unsigned)((hc_lr + hc + 3) / 4), (unsigned)n_tok);
    const size_t lds = (size_t)hd * 2;
    hc_slots(n, hc, [&](auto HC, auto NM) {
        constexpr int slots = HC() * NM();  // a row is at most slots / 2 pieces per lane
        auto go = [&](auto C) {
            constexpr int more = 4 * C();
            const auto k = hc_norm_ahead(slots, more, (int64_t)g1.x * g1.y, (int64_t)hc_lr * hd * 2)
                               ? k_hc_proj<HC(), NM(), C(), true>
                               : k_hc_proj<HC(), NM(), C(), hc_norm_fits(slots, more) || (slots + more > 192)>;
            hipLaunchKernelGGL(k, g1, dim3(256), lds, s, R, norm, down, inj, n, hc, hc_lr, eps, proj, inject, rs);
        };
        const int chunks = hc_chunks(n, hc);
        if (chunks == 8) go(Int<8>{});
        else if constexpr (slots > 16) {
            if (chunks == 16) go(Int<16>{});
            else if constexpr (slots > 32) {
                if (chunks == 24) go(Int<24>{});
                else go(Int<32>{});
            }
        }
    });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    dim3 g2((unsigned)(n / 8), (unsigned)n_tok);
    auto mix = [&](auto P) {
        hipLaunchKernelGGL((k_hc_mix<P()>), g2, dim3(256), 0, s, R, norm, up, proj, rs, n, hc, hc_lr, mixed);
    };
    switch (hc_pieces(hc_lr)) {
        case 1: mix(Int<1>{}); break;
        case 2: mix(Int<2>{}); break;
        case 3: mix(Int<3>{}); break;
        case 4: mix(Int<4>{}); break;
        case 5: mix(Int<5>{}); break;
        case 8: mix(Int<8>{}); break;
        case 16: mix(Int<16>{}); break;
        default: mix(Int<32>{}); break;
    }
    return hipGetLastError();
}

hipError_t launch_hc_write(const float* R, const float* y, const float* inject, int n_tok, int n, int hc, float* out,
                           hipStream_t s) {
    const int64_t total = (int64_t)n_tok * hc * n;
    if (total <= 0) return hipErrorInvalidValue;
    const int parts = (n / 4 + 255) / 256;
    const uintptr_t al = reinterpret_cast<uintptr_t>(R) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(out);
    const HcWrite kind = hc_write_kind(n_tok, n, hc);
    if (kind != kHcWriteValues && n % 4 == 0 && (al & 15) == 0 && (int64_t)n_tok * parts <= INT32_MAX) {
        const dim3 grid((unsigned)((int64_t)n_tok * parts), kind == kHcWriteStream ? (unsigned)hc : 1u);
        hipLaunchKernelGGL(k_hc_write4, grid, dim3(256), 0, s, R, y, inject, n / 4, hc, parts, out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_hc_write, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, R, y, inject, n, hc, total,
                       out);
    return hipGetLastError();
}

}  // namespace smoe
