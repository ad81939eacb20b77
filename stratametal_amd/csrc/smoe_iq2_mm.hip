// stratametal_amd/csrc/smoe_iq2_mm.hip - IQ2_S expert products of the decode contract on the matrix cores (gfx950), for
// items of many columns; bit for bit the results of smoe_iq2.hip's kernels.
//
// The contract's sub-block sum is an integer (metal/shaders/iq.metal:152-180): with s0, s1 the integer dots of a
// sub-block's two halves and ls0, ls1 their 4-bit scales, sumi = (s0 ls0 + s1 ls1 + (s0 + s1) / 2) / 4, both divisions
// truncating, and P = (f32(d_w) f32(d_x)) * sumi.  Two fp16 matrix products per sub-block (one 32-deep
// v_mfma_f32_16x16x32_f16 each) give its two linear parts exactly:
//     S = sum (w / 2) q = (s0 + s1) / 2,      V = sum (w ls / 4) q = (s0 ls0 + s1 ls1) / 4,
// w in {+-8, +-25, +-43} and q in -127 .. 127: w / 2 and w ls / 4 (|w ls| <= 645) are fp16 values, every product and every
// sum is a multiple of 1 / 4 below 2^22, so f32 holds them all; then sumi = trunc(V + trunc(S) / 4), again exact.  The f32
// steps are the other kernels': a block's P in sub-block order, the blocks of a row in the butterfly's order ((0 + 4) +
// (2 + 6)) + ((1 + 5) + (3 + 7)).
//
// smoe_iq2.hip spends eight dots and about twelve more instructions per row, column and sub-block on the VALU; here it is
// six, plus two matrix products that serve 16 x 16 of them and a costlier decode (fp16 pairs and their scaled copies), so a
// tile of 16 columns costs what about six columns cost there (iq2_mm_gains).  Still bound by VALU issue (83 to 85% of its
// slots, the matrix cores 12% busy): 600 tokens of 512 experts (2048, 512 wide) 648 us on the row kernels, 472 here.  A wave's block is loaded at its step (four waves per SIMD
// cover the load): prefetched a step ahead, its 21 registers spilled others, 482 us.
#include "smoe_gemv.hpp"
#include "smoe_launch.hpp"

namespace smoe {

namespace {

constexpr uint16_t kIq2sCodes[1024] = {
#include "iq2s_grid_codes.inc"
};
// Entry i: the grid entry's eight magnitudes halved, as fp16 pairs (j, j + 4): 4, 12.5 and 21.5.
struct Iq2sHalfTable {
    uint32_t e[1024][4];
};
constexpr Iq2sHalfTable make_half_table() {
    Iq2sHalfTable t{};
    constexpr uint32_t half[4] = {0x4400u, 0x4A40u, 0x4D60u, 0u};
    for (int i = 0; i < 1024; ++i)
        for (int j = 0; j < 4; ++j)
            t.e[i][j] = half[(kIq2sCodes[i] >> (2 * j)) & 3] | (half[(kIq2sCodes[i] >> (2 * (j + 4))) & 3] << 16);
    return t;
}
__device__ const Iq2sHalfTable kHalfTab = make_half_table();

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kCols = 16;                          // columns of a tile
constexpr int kPhaseBlocks = 4;                    // 256-value blocks of x in LDS at a time
constexpr int kXPitch = kPhaseBlocks * 512 + 16;   // bytes of a column's staged x (the pad spreads columns over the banks)
constexpr int kThreads = 512, kRows = 16;          // eight waves, 16 rows of each of two row sets per wave
constexpr int kHPitch = 8 * kRows + 4;             // floats of a column's h tile

struct MmLds {
    u32x4 tab[1024];
    alignas(16) uint8_t x[kCols * kXPitch];  // x tile; after the products the h tile of gate/up
    float dx[kCols][8 * kPhaseBlocks + 1];
    uint8_t qsc[16][32];
};
static_assert(sizeof(float) * kCols * kHPitch <= sizeof(uint8_t) * kCols * kXPitch, "the h tile fits the x tile");

// Column tile `c0` of the item against two row sets: wave w, lane (q, i) returns rows 16 w + 4 q .. + 3 of set s and
// column i in out[s].  row0 / row1: the lane's row i of the wave in each set; rowidx: image row of each column.  With
// `staged` the tile's x is in LDS from the call before (one phase: rows of at most four blocks).
template <int NB>
__device__ __forceinline__ void mm_tile(MmLds& s, const uint8_t* row0, const uint8_t* row1, const uint32_t* img,
                                        const int* rowidx, f32x4 (&out)[2], bool staged = false) {
    constexpr int PB = NB < kPhaseBlocks ? NB : kPhaseBlocks, PH = NB / PB;
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, q = lane >> 4;
    // block of step k in phase ph: the order whose pairwise sums are the butterfly's
    auto block_of = [](int ph, int k) {
        return NB == 8 ? ((k & 1) << 2 | (k >> 1) << 1) + ph : NB == 4 ? ((k & 1) << 1 | k >> 1) : k;
    };
    f32x4 sum[2][PH];
#pragma unroll
    for (int ph = 0; ph < PH; ++ph) {
        if (ph) __syncthreads();  // the phase before is done with s.x
        // x of the phase's blocks as fp16 in the weights' pair order, one group of 8 values per piece
        for (int p = staged ? kCols * PB * 32 : tid; p < kCols * PB * 32; p += kThreads) {
            const int c = p / (PB * 32), g = p % (PB * 32), k = g >> 5, sub = (g >> 2) & 7;
            const uint32_t* src = img + ((size_t)rowidx[c] * (8 * NB) + 8 * block_of(ph, k) + sub) * kImgDw;
            const uint2 w = *reinterpret_cast<const uint2*>(src + 2 * (g & 3));
            const uint32_t a = w.x ^ 0x80808080u, b = w.y ^ 0x80808080u;  // x + 128
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t pair = (((a >> (8 * j)) & 0xFFu) | (((b >> (8 * j)) & 0xFFu) << 16)) | 0x64006400u;
                const f16x2 v = __builtin_bit_cast(f16x2, pair) - f16x2{(_Float16)1152.0f, (_Float16)1152.0f};
                o[j] = __builtin_bit_cast(uint32_t, v);
            }
            *reinterpret_cast<u32x4*>(s.x + c * kXPitch + 16 * g) = o;
            if ((g & 3) == 0) s.dx[c][g >> 2] = u2f(src[8]);
        }
        if (!staged) __syncthreads();  // (uniform)
        f32x4 pair = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, tot = pair;
        // the steps of set 0, then of set 1 (not unrolled: one step's code is eight sub-blocks)
#pragma clang loop unroll(disable)
        for (int st = 0; st < 2 * PB; ++st) {
            const int k = st & (PB - 1);
            uint32_t raw[21];
            load_block_raw(st < PB ? row0 : row1, block_of(ph, k), raw);
            const uint32_t sh = (block_of(ph, k) & 1) ? 0u : 2u;  // load_block_raw's shift
            auto fd = [&](int m) { return __builtin_amdgcn_alignbyte(raw[m + 1], raw[m], sh); };
            {
                float dw[4];
                {
                    const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(sh ? raw[0] & 0xFFFFu : raw[20] >> 16));
#pragma unroll
                    for (int e = 0; e < 4; ++e) dw[e] = __shfl(d, 4 * q + e, kWave);
                }
                f32x4 L = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                // the grid entry of a sub-block is read a sub-block ahead
                auto entry = [&](int ib) {
                    const uint32_t lo = __builtin_amdgcn_ubfe(fd(ib), 8 * q, 8);
                    return s.tab[lo | (__builtin_amdgcn_ubfe(fd(16 + (ib >> 2)), 8 * (ib & 3) + 2 * q, 2) << 8)];
                };
                u32x4 ahead = entry(0);
#pragma unroll
                for (int ib = 0; ib < 8; ++ib) {
                    const uint32_t sg = fd(8 + ib), sc = fd(18 + (ib >> 2));
                    const u32x4 m = ahead;
                    if (ib < 7) ahead = entry(ib + 1);
                    uint32_t sgn = __umul24(__builtin_amdgcn_ubfe(sg, 8 * q, 8), 0x1001u);  // bit j at j and j + 12
                    asm("" : "+v"(sgn));  // (one multiply, then shifts: not a 32-bit multiply per pair)
                    const _Float16 ls = (_Float16)(uint16_t)__builtin_amdgcn_ubfe(sc, 8 * (ib & 3) + 4 * (q >> 1), 4) * (_Float16)0.5f;
                    u32x4 w, v;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {  // the signs of weights j and j + 4 to bits 15 and 31
                        const uint32_t wj = m[j] | ((sgn << (15 - j)) & 0x80008000u);
                        w[j] = wj;
                        v[j] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, wj) * f16x2{ls, ls});
                    }
                    const f16x8 x = __builtin_bit_cast(
                        f16x8, *reinterpret_cast<const u32x4*>(s.x + i * kXPitch + 16 * (32 * k + 4 * ib + q)));
                    const float dx = s.dx[i][8 * k + ib];
                    const f32x4 zero = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    const f32x4 S = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), x, zero, 0, 0, 0);
                    const f32x4 V = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, v), x, zero, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float sumi = __builtin_truncf(__builtin_fmaf(__builtin_truncf(S[e]), 0.25f, V[e]));
                        L[e] = L[e] + (dw[e] * dx) * sumi;
                    }
                }
                // ((L0 + L1) + (L2 + L3)) of the phase's steps (or L0 + L1)
                if (k & 1) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float t = pair[e] + L[e];
                        tot[e] = k == 1 ? t : tot[e] + t;
                    }
                } else {
                    pair = L;
                }
            }
            if (st == PB - 1) sum[0][ph] = tot;
        }
        sum[1][ph] = tot;
    }
#pragma unroll
    for (int set = 0; set < 2; ++set) {
        out[set] = sum[set][0];
        if constexpr (PH == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) out[set][e] = sum[set][0][e] + sum[set][1][e];
        }
    }
}

__device__ __forceinline__ void load_table(MmLds& s) {
    const u32x4* src = reinterpret_cast<const u32x4*>(kHalfTab.e);
    for (int p = threadIdx.x; p < 1024; p += kThreads) s.tab[p] = src[p];
}

}  // namespace

// Gate/up: work-group (item y, row block rt) computes h rows [128 rt, 128 rt + 128) of the item's columns, 16 at a time:
// wave w gate rows 16 w .. + 15 (set 0) and the same up rows (set 1), SwiGLU, then the natural-order q8_1 images of h.
template <int NB>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_iq2_mm_gu(
    const int4* __restrict__ items, int max_items, int n_rb, const uint32_t* __restrict__ ximg,
    const uint8_t* __restrict__ gate_exps, const uint8_t* __restrict__ up_exps, int F, int k,
    const uint8_t* __restrict__ gate_sh, const uint8_t* __restrict__ up_sh, const int32_t* __restrict__ perm,
    uint32_t* __restrict__ himg, int h_blocks) {
    __shared__ MmLds s;
    __shared__ int rowidx[kCols];
    int y, rt;
    if (!xcd_item(n_rb, max_items, y, rt)) return;
    Item item;
    if (!work_item(items, y, item)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, q = lane >> 4;
    constexpr size_t rb = (size_t)NB * 82;
    const size_t row = (size_t)128 * rt + 16 * wave + i;
    const uint8_t* g = (item.shared ? gate_sh : gate_exps + (size_t)item.e * F * rb) + row * rb;
    const uint8_t* u = (item.shared ? up_sh : up_exps + (size_t)item.e * F * rb) + row * rb;
    load_table(s);
    float* ht = reinterpret_cast<float*>(s.x);
    for (int c0 = 0; c0 < item.ncol; c0 += kCols) {
        const int nc = min(kCols, item.ncol - c0);
        if (tid < kCols) rowidx[tid] = item_token(item, perm, k, c0 + min(tid, nc - 1));  // dead columns: the last one again
        __syncthreads();
        f32x4 o[2];
        mm_tile<NB>(s, g, u, ximg, rowidx, o);
        __syncthreads();  // every wave is done with s.x
        f32x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = silu_mul(o[0][e], o[1][e]);
        *reinterpret_cast<f32x4*>(ht + i * kHPitch + 16 * wave + 4 * q) = h;
        __syncthreads();
        for (int b = tid >> 5; b < kCols * 4; b += kThreads / 32) {  // a half wave per 32-value block of a column
            const int c = b >> 2, hb = b & 3;
            const bool live = c < nc;
            const float v = live ? ht[c * kHPitch + 32 * hb + (tid & 31)] : 0.0f;
            q8_image_store(v, live, s.qsc[tid >> 5],
                           himg + ((size_t)(item.first + c0 + (live ? c : 0)) * h_blocks + 4 * rt + hb) * kImgDw, true);
        }
        __syncthreads();  // the h tile is read before the next tile's x
    }
}

// Down: work-group (item y, row block rt) computes down rows [256 RP rt, 256 RP rt + 256 RP) of the item's columns into
// Y[first + c] (the shared expert's times sigmoid(sg[t])), 256 rows a pass: wave w rows 32 w .. + 15 (set 0) and 32 w + 16
// .. + 15 (set 1).  The passes of a tile share its staged x, and the work-group its grid table.
template <int NB, int RP>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_iq2_mm_down(
    const int4* __restrict__ items, int max_items, int n_rb, const uint32_t* __restrict__ himg,
    const uint8_t* __restrict__ down_exps, const uint8_t* __restrict__ down_sh, int H, const float* __restrict__ sg,
    float* __restrict__ Y) {
    __shared__ MmLds s;
    __shared__ int rowidx[kCols];
    int y, rt;
    if (!xcd_item(n_rb, max_items, y, rt)) return;
    Item item;
    if (!work_item(items, y, item)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, q = lane >> 4;
    constexpr size_t rb = (size_t)NB * 82;
    static_assert(RP == 1 || NB <= kPhaseBlocks, "several passes: x staged in one phase");
    const int row = 256 * RP * rt + 32 * wave;
    const uint8_t* d = (item.shared ? down_sh : down_exps + (size_t)item.e * H * rb) + (size_t)(row + i) * rb;
    load_table(s);
    for (int c0 = 0; c0 < item.ncol; c0 += kCols) {
        const int nc = min(kCols, item.ncol - c0);
        if (tid < kCols) rowidx[tid] = item.first + c0 + min(tid, nc - 1);
        __syncthreads();
        const float gs = item.shared && i < nc ? sigmoid(sg[item.tok0 + c0 + i]) : 1.0f;
#pragma clang loop unroll(disable)
        for (int pass = 0; pass < RP; ++pass) {
            const uint8_t* dp = d + (size_t)(256 * pass) * rb;
            f32x4 o[2];
            mm_tile<NB>(s, dp, dp + 16 * rb, himg, rowidx, o, pass > 0);
            if (i < nc) {
#pragma unroll
                for (int set = 0; set < 2; ++set) {
                    f32x4 v = o[set];
                    if (item.shared) v = f32x4{v[0] * gs, v[1] * gs, v[2] * gs, v[3] * gs};
                    *reinterpret_cast<f32x4*>(Y + (size_t)(item.first + c0 + i) * H + row + 256 * pass + 16 * set + 4 * q) = v;
                }
            }
        }
        __syncthreads();  // every wave is done with s.x and rowidx
    }
}

// Shapes: rows of 512, 1024 or 2048 values on both sides (iq2_shape_ok), a shared expert as wide as the routed ones.
hipError_t launch_iq2_mm_gu(const uint8_t* gate_exps, const uint8_t* up_exps, const uint8_t* gate_sh, const uint8_t* up_sh,
                            const uint32_t* ximg, const int4* items, const int32_t* perm, int k, int H, int F,
                            int max_items, uint32_t* himg, int h_blocks, hipStream_t s) {
    if (!iq2_shape_ok(H) || !iq2_shape_ok(F) || h_blocks != F / 32) return hipErrorInvalidValue;
    const int n_rb = F / 128;
    const dim3 grid(xcd_grid(n_rb, max_items));
#define SMOE_MM_GU(NB)                                                                                              \
    hipLaunchKernelGGL((k_iq2_mm_gu<NB>), grid, dim3(kThreads), 0, s, items, max_items, n_rb, ximg, gate_exps, up_exps, F, \
                       k, gate_sh, up_sh, perm, himg, h_blocks)
    if (H == 512) SMOE_MM_GU(2);
    else if (H == 1024) SMOE_MM_GU(4);
    else SMOE_MM_GU(8);
#undef SMOE_MM_GU
    return hipGetLastError();
}

constexpr int kDownTwoPasses = 2048;
hipError_t launch_iq2_mm_down(const uint8_t* down_exps, const uint8_t* down_sh, const uint32_t* himg, int h_blocks,
                              const float* sg, const int4* items, int H, int F, int max_items, float* Y, hipStream_t s) {
    if (!iq2_shape_ok(H) || !iq2_shape_ok(F) || h_blocks != F / 32) return hipErrorInvalidValue;
    // two passes where the halved grid still fills the chip (two work-groups per CU) four times (600 tokens of 512
    // experts, 2048 rows of 512: 165 us one by one, 155 in twos; the whole call of 512 experts of 2048 x 1024 1.01 times
    // as fast; of 256 experts, 1300 work-groups, 1.01 at F 512 and 0.98 at F 1024, at 600 work-groups 0.96)
    const int rp = F <= 1024 && H % 512 == 0 && (int64_t)max_items * (H / 512) >= kDownTwoPasses ? 2 : 1;
    const int n_rb = H / (256 * rp);
    const dim3 grid(xcd_grid(n_rb, max_items));
#define SMOE_MM_DOWN(NB, RP)                                                                                       \
    hipLaunchKernelGGL((k_iq2_mm_down<NB, RP>), grid, dim3(kThreads), 0, s, items, max_items, n_rb, himg, down_exps, \
                       down_sh, H, sg, Y)
    if (F == 512 && rp == 2) SMOE_MM_DOWN(2, 2);
    else if (F == 512) SMOE_MM_DOWN(2, 1);
    else if (F == 1024 && rp == 2) SMOE_MM_DOWN(4, 2);
    else if (F == 1024) SMOE_MM_DOWN(4, 1);
    else SMOE_MM_DOWN(8, 1);
#undef SMOE_MM_DOWN
    return hipGetLastError();
}

// The columns of the items: chunks of four tiles, so that a hot expert's columns spread over work-groups.
int iq2_mm_chunk() { return 4 * kCols; }
int iq2_mm_shared_chunk() { return kCols; }

}  // namespace smoe
