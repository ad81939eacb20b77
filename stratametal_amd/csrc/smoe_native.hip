// stratametal_amd/csrc/smoe_native.hip - GEMV of the other native GGUF types of real layers (gfx950, wave64).
//
// The shared expert's projections and the down quants of real layers come in Q8_0, Q4_0, Q5_0, IQ4_NL, IQ4_XS,
// Q3_K, Q4_K, Q5_K and Q6_K (include/strata/kernels/shared_expert.hpp:54-58, metal/src/pack_parity.cpp:7782-7799).
// Each runs the reference's q8_1 MMVQ contract: a row is a sum of per-block integer partials against q8_1
// activations (metal/shaders/iq.metal:224-442), taken by 32 lanes -- lane l adds partials l, l + 32, ... in order
// from 0 -- then an xor butterfly 16, 8, 4, 2, 1 (iq_row / iq_mmvq_body, metal/shaders/iq.metal:458-513).  Here a
// 32-lane half wave owns one row, so that order runs unchanged (oracle: or_native_gemv, which is also the
// reference's own host order, metal/src/pack_parity.cpp:2785-3475).  One partial is decoded into registers once
// (NativePart) and taken against every column of a tile: a few columns read x from memory (k_mmvq_native), more stage
// it in LDS (k_mmvq_native_cols).
#include "smoe_device.hpp"
#include "smoe_gemv.hpp"
#include "smoe_launch.hpp"
#include "smoe_rules.hpp"

namespace smoe {

namespace {

// values, bytes, partials per block and the iqs step of each type (iq_row<QK, IPB, STEP, BLOCK>)
template <int TYPE>
struct NativeType;
template <> struct NativeType<8> { static constexpr int qk = 32, bytes = 34, ipb = 1, step = 1; };
template <> struct NativeType<2> { static constexpr int qk = 32, bytes = 18, ipb = 2, step = 2; };
template <> struct NativeType<6> { static constexpr int qk = 32, bytes = 22, ipb = 2, step = 2; };
template <> struct NativeType<20> { static constexpr int qk = 32, bytes = 18, ipb = 2, step = 2; };
template <> struct NativeType<23> { static constexpr int qk = 256, bytes = 136, ipb = 8, step = 4; };
template <> struct NativeType<11> { static constexpr int qk = 256, bytes = 110, ipb = 16, step = 1; };
template <> struct NativeType<12> { static constexpr int qk = 256, bytes = 144, ipb = 16, step = 2; };
template <> struct NativeType<13> { static constexpr int qk = 256, bytes = 176, ipb = 16, step = 2; };
template <> struct NativeType<14> { static constexpr int qk = 256, bytes = 210, ipb = 32, step = 1; };

// Block fields are 2-byte aligned (every block size is even); a 32-bit field is one load at that alignment.
__device__ __forceinline__ uint32_t rd16(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }
__device__ __forceinline__ int32_t rd32(const uint8_t* p) {
    int32_t v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 4);
    return v;
}
__device__ __forceinline__ float rdh(const uint8_t* p) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)rd16(p));  // exact fp16 -> f32
}
// the q8_1 block's int8 word w (4-byte aligned: blocks are 36 bytes)
__device__ __forceinline__ int32_t qword(const uint8_t* b, int w) {
    return *reinterpret_cast<const int32_t*>(b + 4 + 4 * w);
}
__device__ __forceinline__ int32_t dot4(int32_t a, int32_t b, int32_t c) { return __builtin_amdgcn_sdot4(a, b, c, false); }

// The IQ4 codebook as bytes: four signed values from four 4-bit indices (one per byte), two byte permutes of the
// table's halves and a select by the indices' top bit.
__device__ __forceinline__ int32_t nl4_bytes(uint32_t idx) {
    const uint32_t sel = idx & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(0xF6EADDCFu, 0xBFAD9881u, sel);  // -49 -35 -22 -10, -127 -104 -83 -65
    const uint32_t hi = __builtin_amdgcn_perm(0x71594535u, 0x26190D01u, sel);  // 53 69 89 113, 1 13 25 38
    const uint32_t m = (idx >> 3) & 0x01010101u, all = (m << 8) - m;  // 0xFF where the top bit is set
    return (int32_t)((hi & all) | (lo & ~all));
}

// Four bytes of v, each at most 127, less `off` (at most 128) in each: signed bytes, no borrow between them (shifts,
// subtractions and masks throughout: a 32-bit multiply takes four times as long).
__device__ __forceinline__ int32_t bytes_less(uint32_t v, uint32_t off) {
    return (int32_t)(((v | 0x80808080u) - off * 0x01010101u) ^ 0x80808080u);
}
// The four low bits of b as the lowest bits of four bytes.
__device__ __forceinline__ uint32_t spread4(uint32_t b) { return __umul24(b & 15u, 0x204081u) & 0x01010101u; }

// Q4_K / Q5_K: the 6-bit scale and min pair of two 32-value groups (iq_k_scale_min, metal/shaders/iq.metal:254-262)
__device__ __forceinline__ void k_scale_min(const uint8_t* s, int bq8_offset, int (&sc)[2], int (&mn)[2]) {
    const int j = bq8_offset / 2, jm = j & 1;
    const uint32_t s0 = rd16(s + 2 * (jm + 0)), s2 = rd16(s + 2 * (jm + 2)), s4 = rd16(s + 2 * (jm + 4));
    const uint32_t a0 = j >= 2 ? (((s4 >> 0) & 0x0F0Fu) | ((s0 & 0xC0C0u) >> 2)) : (s0 & 0x3F3Fu);
    const uint32_t a1 = j >= 2 ? (((s4 >> 4) & 0x0F0Fu) | ((s2 & 0xC0C0u) >> 2)) : (s2 & 0x3F3Fu);
    sc[0] = (int)(a0 & 0xFFu);
    sc[1] = (int)((a0 >> 8) & 0xFFu);
    mn[0] = (int)(a1 & 0xFFu);
    mn[1] = (int)((a1 >> 8) & 0xFFu);
}

// The activations of one 32-value block as the partials read them: the int8 words and the scale.  In memory a q8_1
// block (fp16 scale first), in LDS eight words and then the scale in f32 (kXlDw dwords per block: an odd pitch).
constexpr int kXlDw = 9;
struct XMem {
    const uint8_t* p;
    __device__ __forceinline__ XMem at(int block) const { return {p + (size_t)block * 36}; }
    __device__ __forceinline__ int32_t word(int w) const { return qword(p, w); }
    __device__ __forceinline__ float scale() const { return rdh(p); }
};
struct XLds {
    const uint32_t* p;
    __device__ __forceinline__ XLds at(int block) const { return {p + kXlDw * block}; }
    __device__ __forceinline__ int32_t word(int w) const { return (int32_t)p[w]; }
    __device__ __forceinline__ float scale() const { return __uint_as_float(p[8]); }
};

// One partial of a row (part iqs of a block), decoded once: signed bytes whose integer dots are the reference's (an
// offset it subtracts after the dot is subtracted from each byte: the same integer).  dot(x): the partial against a
// column's activations of the block (x its first 32-value block); the float steps are the reference's, one rounding
// each (no contraction).  A dot times its scale is a 24-bit multiply: every dot is below 2^20, every scale below 2^8.
// RAW: for one column, the codes stay unsigned and the offset is subtracted after the dot, as the reference has it: two to
// four dots of ones more for the column, eight to sixteen instructions fewer to decode.
template <int TYPE, bool RAW>
struct NativePart;

template <bool RAW>
struct NativePart<8, RAW> {  // Q8_0
    int32_t w[8];
    float d;
    __device__ __forceinline__ void decode(const uint8_t* blk, int) {
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = rd32(blk + 2 + 4 * j);
        d = rdh(blk);
    }
    template <class X>
    __device__ __forceinline__ float dot(const X& x, int) const {
        int32_t s = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) s = dot4(w[j], x.word(j), s);
        return (d * x.scale()) * (float)s;
    }
};

template <int TYPE, bool RAW>
struct NativePart16 {  // Q4_0, Q5_0, IQ4_NL: 16 values of a 32-value block, words iqs, iqs + 1 and 4 words on
    static constexpr int kOff = TYPE == 2 ? 8 : TYPE == 6 ? 16 : 0;
    int32_t lo[2], hi[2];
    float d;
    __device__ __forceinline__ void decode(const uint8_t* blk, int iqs) {
        const uint8_t* qs = blk + (TYPE == 6 ? 6 : 2);
        uint32_t h = 0;
        if constexpr (TYPE == 6) h = (uint32_t)rd32(blk + 2);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t v = (uint32_t)rd32(qs + 4 * (iqs + i));
            uint32_t a = v & 0x0F0F0F0Fu, b = (v >> 4) & 0x0F0F0F0Fu;
            if constexpr (TYPE == 20) {
                lo[i] = nl4_bytes(a);
                hi[i] = nl4_bytes(b);
                continue;
            }
            if constexpr (TYPE == 6) {
                const uint32_t hs = h >> (4 * (iqs + i));
                a |= spread4(hs) << 4;
                b |= spread4(hs >> 16) << 4;
            }
            lo[i] = RAW ? (int32_t)a : bytes_less(a, kOff);
            hi[i] = RAW ? (int32_t)b : bytes_less(b, kOff);
        }
        d = rdh(blk);
    }
    template <class X>
    __device__ __forceinline__ float dot(const X& x, int iqs) const {
        int32_t s = 0, a = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int32_t u0 = x.word(iqs + i), u1 = x.word(iqs + i + 4);
            s = dot4(lo[i], u0, s);
            s = dot4(hi[i], u1, s);
            if constexpr (RAW && kOff) a = dot4(0x01010101, u1, dot4(0x01010101, u0, a));
        }
        if constexpr (RAW && kOff) s -= kOff * a;
        return (d * x.scale()) * (float)s;
    }
};
template <bool RAW> struct NativePart<2, RAW> : NativePart16<2, RAW> {};
template <bool RAW> struct NativePart<6, RAW> : NativePart16<6, RAW> {};
template <bool RAW> struct NativePart<20, RAW> : NativePart16<20, RAW> {};

template <bool RAW>
struct NativePart<23, RAW> {  // IQ4_XS: 32-value group iqs / 4, its 6-bit scale - 32
    int32_t lo[4], hi[4], ls;
    float d;
    __device__ __forceinline__ void decode(const uint8_t* blk, int iqs) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t v = (uint32_t)rd32(blk + 8 + 4 * (iqs + j));
            lo[j] = nl4_bytes(v & 0x0F0F0F0Fu);
            hi[j] = nl4_bytes((v >> 4) & 0x0F0F0F0Fu);
        }
        ls = (((blk[4 + iqs / 8] >> (iqs & 4)) & 15) | (int)(((rd16(blk + 2) >> (iqs / 2)) & 3u) << 4)) - 32;
        d = rdh(blk);
    }
    template <class X>
    __device__ __forceinline__ float dot(const X& x0, int iqs) const {
        const X x = x0.at(iqs / 4);
        int32_t s = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s = dot4(lo[j], x.word(j), s);
            s = dot4(hi[j], x.word(j + 4), s);
        }
        return (d * x.scale()) * (float)__mul24(s, ls);
    }
};

template <int TYPE>
struct NativePartK {  // Q4_K, Q5_K: 8 values of two 32-value groups
    int32_t p[2][2];
    int sc[2], mn[2];
    float d, dmin;
    __device__ __forceinline__ void decode(const uint8_t* blk, int iqs) {
        constexpr bool q5 = TYPE == 13;
        const int bq8_offset = 2 * ((iqs / 2) / 4), qoff = (iqs / 2) % 4;
        const uint8_t* ql = blk + (q5 ? 48 : 16);
        const int byte = 16 * bq8_offset + 4 * qoff;
        const int32_t v0 = rd32(ql + byte), v1 = rd32(ql + byte + 16);
        int32_t vh0 = 0, vh1 = 0;
        if constexpr (q5) {
            vh0 = rd32(blk + 16 + 4 * qoff) >> bq8_offset;
            vh1 = rd32(blk + 32 + 4 * qoff) >> bq8_offset;
        }
        k_scale_min(blk + 4, bq8_offset, sc, mn);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            p[i][0] = (v0 >> (4 * i)) & 0x0F0F0F0F;
            p[i][1] = (v1 >> (4 * i)) & 0x0F0F0F0F;
            if constexpr (q5) {
                p[i][0] |= ((vh0 >> i) << 4) & 0x10101010;
                p[i][1] |= ((vh1 >> i) << 4) & 0x10101010;
            }
        }
        d = rdh(blk);
        dmin = rdh(blk + 2);
    }
    template <class X>
    __device__ __forceinline__ float dot(const X& x0, int iqs) const {
        const int bq8_offset = 2 * ((iqs / 2) / 4), qoff = (iqs / 2) % 4;
        float sum_d = 0.0f, sum_m = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const X x = x0.at(bq8_offset + i);
            const float d8 = x.scale();
            const int32_t u0 = x.word(qoff), u1 = x.word(qoff + 4);
            const int32_t dq = dot4(p[i][1], u1, dot4(p[i][0], u0, 0));
            const int32_t da = dot4(0x01010101, u1, dot4(0x01010101, u0, 0));
            sum_d = sum_d + d8 * (float)__mul24(dq, sc[i]);
            sum_m = sum_m + d8 * (float)__mul24(da, mn[i]);
        }
        return d * sum_d - dmin * sum_m;
    }
};
template <bool RAW> struct NativePart<12, RAW> : NativePartK<12> {};
template <bool RAW> struct NativePart<13, RAW> : NativePartK<13> {};

template <bool RAW>
struct NativePart<11, RAW> {  // Q3_K: 2 low bits, - 4 where the high bit is clear; scale - 32
    int32_t v[4];
    int sc[4];
    float d;
    __device__ __forceinline__ void decode(const uint8_t* blk, int iqs) {
        const int bq8_offset = 4 * (iqs / 8), scale_offset = iqs - (iqs % 8) + (iqs % 8) / 4;
        const uint32_t vl = (uint32_t)rd32(blk + 32 + 4 * iqs);
        const uint32_t vh = (~(uint32_t)rd32(blk + 4 * (iqs % 8))) >> bq8_offset;
        // scale j = scale_offset + 2 i: its low nibble in byte j % 8 (the high half of the byte from j = 8 on), its high
        // bits 2 (j / 4) of byte 8 + j % 4; scale_offset is 0, 1, 8 or 9
        const uint32_t sl[2] = {(uint32_t)rd32(blk + 96), (uint32_t)rd32(blk + 100)};
        const uint32_t sh = (uint32_t)rd32(blk + 104);
        const int odd = scale_offset & 1, half = scale_offset >> 3;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t lo = sl[i >> 1] >> (8 * (odd + 2 * (i & 1)) + 4 * half);
            const uint32_t hi = sh >> (8 * (odd + 2 * (i & 1)) + 2 * (2 * half + (i >> 1)));
            sc[i] = (int)((lo & 15u) | ((hi & 3u) << 4)) - 32;
            v[i] = (int32_t)(((vl >> (2 * i)) & 0x03030303u) | ((vh >> i) & 0x01010101u) * 0xFCu);
        }
        d = rdh(blk + 108);
    }
    template <class X>
    __device__ __forceinline__ float dot(const X& x0, int iqs) const {
        const X x = x0.at(4 * (iqs / 8));
        float sumf = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const X xi = x.at(i);
            sumf = sumf + xi.scale() * (float)__mul24(dot4(v[i], xi.word(iqs % 8), 0), sc[i]);
        }
        return d * sumf;
    }
};

template <bool RAW>
struct NativePart<14, RAW> {  // Q6_K: (low nibble | 2 high bits << 4) - 32 times an int8 scale
    int32_t v[2];
    int sc[2];
    float d;
    __device__ __forceinline__ void decode(const uint8_t* blk, int iqs) {
        const int scale_offset = 8 * (iqs / 16) + (iqs % 16) / 4, vh_shift = 2 * ((iqs % 16) / 8);
        const uint32_t vl = (uint32_t)rd32(blk + 4 * iqs);
        const uint32_t vh = (uint32_t)rd32(blk + 128 + 4 * (8 * (iqs / 16) + (iqs % 8))) >> vh_shift;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            sc[i] = (int)(int8_t)blk[192 + scale_offset + 4 * i];
            const uint32_t q = ((vl >> (4 * i)) & 0x0F0F0F0Fu) | (((vh >> (4 * i)) << 4) & 0x30303030u);
            v[i] = RAW ? (int32_t)q : bytes_less(q, 32);
        }
        d = rdh(blk + 208);
    }
    template <class X>
    __device__ __forceinline__ float dot(const X& x0, int iqs) const {
        const X x = x0.at(4 * (iqs / 16) + (iqs % 16) / 8);
        float sumf = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const X xi = x.at(2 * i);
            const int32_t u = xi.word(iqs % 8);
            int32_t dq = dot4(v[i], u, 0);
            if constexpr (RAW) dq -= dot4(0x20202020, u, 0);
            sumf = sumf + xi.scale() * (float)__mul24(dq, sc[i]);
        }
        return d * sumf;
    }
};

// A row against one column by 32 lanes: lane l (k = l) adds partials l, l + 32, ... in order, then the butterfly 16
// .. 1; every lane returns the sum.  (`acc`: the sum of the partials before k.)
template <int TYPE, class X>
__device__ __forceinline__ float native_row(const uint8_t* row, int npart, const X& col, float acc, int k) {
    using NT = NativeType<TYPE>;
    // four partials at a time: their loads are in flight together, their sums added in order (not the wider partials of
    // Q4_K and Q5_K, 3.3 us against 3.9 for 512 rows of 2048, nor Q4_0 and Q6_K, whose few instructions want the waves
    // instead: 4096 rows of 4096 4.7 against 5.0 and 5.7 against 6.7 us)
    constexpr bool four = TYPE == 8 || TYPE == 6 || TYPE == 20 || TYPE == 23 || TYPE == 11;
    for (; four && k + 96 < npart; k += 128) {
        NativePart<TYPE, false> p[4];
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j].decode(row + (size_t)((k + 32 * j) / NT::ipb) * NT::bytes, NT::step * ((k + 32 * j) % NT::ipb));
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = p[j].dot(col.at((k + 32 * j) / NT::ipb * (NT::qk / 32)), NT::step * ((k + 32 * j) % NT::ipb));
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = acc + v[j];
    }
    for (; k < npart; k += 32) {
        NativePart<TYPE, true> p;
        p.decode(row + (size_t)(k / NT::ipb) * NT::bytes, NT::step * (k % NT::ipb));
        acc = acc + p.dot(col.at(k / NT::ipb * (NT::qk / 32)), NT::step * (k % NT::ipb));
    }
    acc = acc + xor_swap<16>(acc);
    acc = acc + xor_swap<8>(acc);
    acc = acc + xor_swap<4>(acc);
    acc = acc + xor_swap<2>(acc);
    acc = acc + xor_swap<1>(acc);
    return acc;
}

// n values of x (n % 32 == 0) as q8_1 blocks in LDS, by the whole work-group (NTH threads): q8_1_value's int8 and scale,
// without the block sum, which no partial reads.
template <int NTH>
__device__ __forceinline__ void quantise_lds(const float* __restrict__ x, int n, uint32_t* xl) {
    uint8_t* xb = reinterpret_cast<uint8_t*>(xl);
    const int l = threadIdx.x & 31;
    for (int i0 = threadIdx.x; i0 < n; i0 += NTH * 4) {
        float v[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) v[m] = x[min(i0 + NTH * m, n - 32 + l)];  // past the end: the last block again
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const float a = half_max(__builtin_fabsf(v[m]));
            float d;
            const int q = q8_1_quant(v[m], a, d);
            const int i = i0 + NTH * m;
            if (i < n) {
                xb[(i >> 5) * (4 * kXlDw) + l] = (uint8_t)(int8_t)q;
                if (l == 0) xl[(i >> 5) * kXlDw + 8] = __float_as_uint((float)(_Float16)d);
            }
        }
    }
}

// A shared expert of native types for a few tokens, in two launches: h = silu(gate) * up of x in q8_1 (k_native_gu: grid
// (ceil(ff / 8), T), a half wave per row of each plane), then down rows of h in q8_1 (k_native_down: grid (ceil(n / 8),
// T)), each work-group quantising its token's row into LDS as the stage kernels form it.  Bound by launches and latency:
// one token of Q3_K gate and up, IQ4_NL down, 512 wide, took 4.0 + 7.8 + 7.0 + 2.4 + 3.3 us in five.
template <int TYPE>
__global__ __launch_bounds__(512) void k_native_gu(const float* __restrict__ x, const uint8_t* __restrict__ gate,
                                                   const uint8_t* __restrict__ up, int H, int F, float* __restrict__ h) {
    using NT = NativeType<TYPE>;
    extern __shared__ __align__(16) uint32_t xl[];  // [H / 32][kXlDw]
    __shared__ float rowv[16];                      // eight gate rows, the same up rows
    const int l = threadIdx.x & 31, hw = threadIdx.x >> 5, r = blockIdx.x * 8 + (hw & 7), t = blockIdx.y;
    quantise_lds<512>(x + (size_t)t * H, H, xl);
    __syncthreads();
    const float v = native_row<TYPE>((hw < 8 ? gate : up) + (size_t)min(r, F - 1) * (H / NT::qk) * NT::bytes,
                                     (H / NT::qk) * NT::ipb, XLds{xl}, 0.0f, l);
    if (l == 0) rowv[hw] = v;
    __syncthreads();
    if (hw < 8 && l == 0 && r < F) h[(size_t)t * F + r] = silu_mul(rowv[hw], rowv[hw + 8]);
}

template <int TYPE>
__global__ __launch_bounds__(256) void k_native_down(const float* __restrict__ h, const uint8_t* __restrict__ down, int F,
                                                     int H, const float* __restrict__ sg, int add, float* __restrict__ y) {
    using NT = NativeType<TYPE>;
    extern __shared__ __align__(16) uint32_t xl[];  // [F / 32][kXlDw]
    const int l = threadIdx.x & 31, r = blockIdx.x * 8 + (threadIdx.x >> 5), t = blockIdx.y;
    quantise_lds<256>(h + (size_t)t * F, F, xl);
    __syncthreads();
    const float acc = native_row<TYPE>(down + (size_t)min(r, H - 1) * (F / NT::qk) * NT::bytes, (F / NT::qk) * NT::ipb,
                                       XLds{xl}, 0.0f, l);
    if (r < H && l == 0) {
        const float v = acc * sigmoid(sg[t]);
        float* dst = y + (size_t)t * H + r;
        *dst = add ? *dst + v : v;
    }
}

// y[c * ldy + r] = row r . column c (times sigmoid(sg[c]) when sg is given).  Grid (ceil(n_out / 8), column
// groups, matrices: w into y, then w2 into y2); a 32-lane half wave per row; a work-group takes columns blockIdx.y,
// + gridDim.y, ...
template <int TYPE>
__global__ __launch_bounds__(256) void k_mmvq_native(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2,
                                                     int n_in, int n_out, int n_col, const uint8_t* __restrict__ xq,
                                                     float* __restrict__ y, float* __restrict__ y2, int ldy,
                                                     const float* __restrict__ sg) {
    using NT = NativeType<TYPE>;
    if (blockIdx.z) {
        w = w2;
        y = y2;
    }
    const int hw = threadIdx.x >> 5, l = threadIdx.x & 31;
    const int r = blockIdx.x * 8 + hw;
    const size_t rb = (size_t)(n_in / NT::qk) * NT::bytes, xb = (size_t)(n_in / 32) * 36;
    const uint8_t* row = w + (size_t)(r < n_out ? r : n_out - 1) * rb;  // a dead half wave reads the last row
    const int npart = (n_in / NT::qk) * NT::ipb;
    for (int c = blockIdx.y; c < n_col; c += gridDim.y) {
        const float acc = native_row<TYPE>(row, npart, XMem{xq + (size_t)c * xb}, 0.0f, l);
        if (r < n_out && l == 0) y[(size_t)c * ldy + r] = sg ? acc * sigmoid(sg[c]) : acc;
    }
}

// The same product for C columns at a time: a half wave owns kRw rows; x of the column tile in LDS, kXlChunk values of
// K at a time (a multiple of 32 partials of every type, so the order of a lane's partials is k_mmvq_native's); a partial
// is decoded once and taken against the C columns.  The butterflies of the kRw * C sums run as one scattering butterfly
// (each step halves the values a lane holds, 31 exchanges for 32 sums instead of 160), and the results go out through
// LDS as whole runs of a column's rows.  On 1000 columns, a work-group per column decoding the rows again and this: Q3_K
// 512 x 2048 232 and 58 us, IQ4_NL 2048 x 512 609 and 36 us.  Bound by the VALU: about nine instructions per 16 products
// for IQ4_NL, 22 for Q3_K (81 to 86% of its issue slots).
constexpr int kRw = 2, kXlChunk = 2048;
static_assert(8 * kRw == kNativeTileRows, "the rows of a work-group");
template <int TYPE, int C>
__global__ __launch_bounds__(256) void k_mmvq_native_cols(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2,
                                                          int n_in, int n_out, int n_col,
                                                          const uint8_t* __restrict__ xq, float* __restrict__ y,
                                                          float* __restrict__ y2, int ldy, const float* __restrict__ sg) {
    using NT = NativeType<TYPE>;
    constexpr int N = kRw * C;
    static_assert(N <= 32 && (N & (N - 1)) == 0, "a scattering butterfly over 32 lanes");
    extern __shared__ __align__(16) uint32_t xl[];  // [C][chunk blocks][kXlDw]
    __shared__ float ot[C][8 * kRw + 1];
    if (blockIdx.z) {
        w = w2;
        y = y2;
    }
    const int hw = threadIdx.x >> 5, l = threadIdx.x & 31;
    const int r0 = blockIdx.x * 8 * kRw, c0 = blockIdx.y * C;
    const size_t rb = (size_t)(n_in / NT::qk) * NT::bytes;
    const uint8_t* row[kRw];
#pragma unroll
    for (int j = 0; j < kRw; ++j) row[j] = w + (size_t)min(r0 + hw * kRw + j, n_out - 1) * rb;  // dead rows read the last
    const uint32_t* xd = reinterpret_cast<const uint32_t*>(xq);  // 36-byte blocks: whole dwords
    const int xb = n_in / 32 * 9;                                // dwords of a column
    float acc[N];
#pragma unroll
    for (int o = 0; o < N; ++o) acc[o] = 0.0f;
    for (int v0 = 0; v0 < n_in; v0 += kXlChunk) {
        const int vals = min(kXlChunk, n_in - v0), nb = vals / 32;  // 32-value blocks of this chunk
        const int npart = vals / NT::qk * NT::ipb, kb0 = v0 / NT::qk;
        if (v0) __syncthreads();
        for (int p = threadIdx.x; p < C * nb; p += 256) {  // a block per thread: its words, then its scale
            const int c = p / nb;
            const uint32_t* src = xd + (size_t)min(c0 + c, n_col - 1) * xb + (size_t)(v0 / 32 + p - c * nb) * 9;
            uint32_t v[9];
#pragma unroll
            for (int m = 0; m < 9; ++m) v[m] = src[m];
#pragma unroll
            for (int m = 1; m < 9; ++m) xl[p * kXlDw + m - 1] = v[m];
            xl[p * kXlDw + 8] = __float_as_uint((float)__builtin_bit_cast(_Float16, (uint16_t)(v[0] & 0xFFFFu)));
        }
        __syncthreads();
        for (int k = l; k < npart; k += 32) {
            const int kb = k / NT::ipb, iqs = NT::step * (k % NT::ipb);
            NativePart<TYPE, false> part[kRw];
#pragma unroll
            for (int j = 0; j < kRw; ++j) part[j].decode(row[j] + (size_t)(kb0 + kb) * NT::bytes, iqs);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const XLds x{xl + (c * nb + kb * (NT::qk / 32)) * kXlDw};
#pragma unroll
                for (int j = 0; j < kRw; ++j) acc[j * C + c] = acc[j * C + c] + part[j].dot(x, iqs);
            }
        }
    }
    scatter_step<16, N>(acc, l);
    scatter_step<8, (N > 2 ? N / 2 : 1)>(acc, l);
    scatter_step<4, (N > 4 ? N / 4 : 1)>(acc, l);
    scatter_step<2, (N > 8 ? N / 8 : 1)>(acc, l);
    scatter_step<1, (N > 16 ? N / 16 : 1)>(acc, l);
    constexpr int kDup = 32 / N;  // lanes that end with the same sum
    if (l % kDup == 0) {
        const int o = l / kDup, j = o / C, c = o % C;
        ot[c][hw * kRw + j] = acc[0];
    }
    __syncthreads();
    for (int p = threadIdx.x; p < C * 8 * kRw; p += 256) {
        const int c = p / (8 * kRw), r = p % (8 * kRw);
        if (c0 + c < n_col && r0 + r < n_out) {
            const float v = ot[c][r];
            y[(size_t)(c0 + c) * ldy + r0 + r] = sg ? v * sigmoid(sg[c0 + c]) : v;
        }
    }
}

// The product for a prompt's columns on the matrix cores, for the types whose weights are whole numbers (times a scale
// per 32 values, or per 256) that fp16 holds exactly, as it holds q8_1's: a 32-value dot is then exact in f32 and only
// fma(d_w d_x, dot, sum) rounds, once per 32 values (d_w d_x is exact: two fp16 values).  k_mmvq_native_cols spends 9 to
// 22 VALU instructions per 16 products on the row kernels' order of partials, which a prompt's contract does not ask for.
// A work-group takes 64 rows (16 per wave) or 32 (16 rows by 16 columns per wave) by 32 columns, 256 values of K at a time
// through LDS as fp16; the sums run 4 + 4 blocks, two chunks, then in order: short chains, for an error no larger than the
// row kernels'.  A word's four values lie in the order 0, 2, 1, 3 on both sides.  1000 columns, gate and up of Q3_K
// 512 x 2048 and down of IQ4_NL 2048 x 512: 124 and 37 us on the row kernels, 32 and 17 here: 60 to 65% of that VALU issue (the
// decode and expansion of both sides), the rest the latency of a chunk's loads; the matrix cores are 5% busy.
constexpr int kNmCols = 32, kNmPitch = 256 * 2 + 16;  // (the pad spreads 16 rows over the banks)
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// four signed bytes as fp16: values 0, 2 and 1, 3
__device__ __forceinline__ void word_f16(int32_t w, f16x2 (&o)[2]) {
    const uint32_t a = (uint32_t)w ^ 0x80808080u;  // value + 128, then 1024 + that as fp16 bits
    const f16x2 off{(_Float16)1152.0f, (_Float16)1152.0f};
    o[0] = __builtin_bit_cast(f16x2, (a & 0x00FF00FFu) | 0x64006400u) - off;
    o[1] = __builtin_bit_cast(f16x2, ((a >> 8) & 0x00FF00FFu) | 0x64006400u) - off;
}
__device__ __forceinline__ uint2 word_bits(int32_t w) {
    f16x2 o[2];
    word_f16(w, o);
    return make_uint2(__builtin_bit_cast(uint32_t, o[0]), __builtin_bit_cast(uint32_t, o[1]));
}

// Partial k of a row's 256-value chunk into its fp16 row and its blocks' scales (dw: [8][ROWS]).
template <int TYPE, int ROWS>
__device__ __forceinline__ void nm_put(const NativePart<TYPE, false>& p, int k, uint8_t* wrow, float* dw) {
    if constexpr (TYPE == 8) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint2 a = word_bits(p.w[2 * j]), b = word_bits(p.w[2 * j + 1]);
            *reinterpret_cast<u32x4*>(wrow + 64 * k + 16 * j) = u32x4{a.x, a.y, b.x, b.y};
        }
        dw[k * ROWS] = p.d;
    } else if constexpr (TYPE == 11) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f16x2 o[2];
            word_f16(p.v[i], o);
            const _Float16 sc = (_Float16)(int16_t)p.sc[i];
            const f16x2 a = o[0] * f16x2{sc, sc}, b = o[1] * f16x2{sc, sc};
            *reinterpret_cast<uint2*>(wrow + 64 * (4 * (k / 8) + i) + 8 * (k % 8)) =
                make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
        }
        if (k % 2 == 0) dw[k / 2 * ROWS] = p.d;
    } else {
        const int kb = k >> 1, iqs = 2 * (k & 1);
        const uint2 l0 = word_bits(p.lo[0]), l1 = word_bits(p.lo[1]), h0 = word_bits(p.hi[0]), h1 = word_bits(p.hi[1]);
        *reinterpret_cast<u32x4*>(wrow + 64 * kb + 8 * iqs) = u32x4{l0.x, l0.y, l1.x, l1.y};
        *reinterpret_cast<u32x4*>(wrow + 64 * kb + 8 * iqs + 32) = u32x4{h0.x, h0.y, h1.x, h1.y};
        if (iqs == 0) dw[kb * ROWS] = p.d;
    }
}

template <int TYPE, int ROWS>
__global__ __launch_bounds__(256) void k_native_mm(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2, int n_in,
                                                   int n_out, int n_col, const uint8_t* __restrict__ xq,
                                                   float* __restrict__ y, float* __restrict__ y2, int ldy,
                                                   const float* __restrict__ sg) {
    using NT = NativeType<TYPE>;
    constexpr int NP = 256 / NT::qk * NT::ipb;  // partials of a row's chunk
    constexpr int U = ROWS * NP / 256;          // per thread
    constexpr int CT = ROWS / 32;               // column tiles per wave
    static_assert(ROWS == 64 || ROWS == 32, "four waves over the tile");
    static_assert(NP == 8 || NP == 16, "whole partials per thread");
    __shared__ __align__(16) uint8_t ws[ROWS * kNmPitch];
    __shared__ __align__(16) uint8_t xs[kNmCols * kNmPitch];
    __shared__ __align__(16) float dw[8 * ROWS];
    __shared__ float dx[8][kNmCols];
    if (blockIdx.z) {
        w = w2;
        y = y2;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, q = lane >> 4;
    const int r0 = blockIdx.x * ROWS, c0 = blockIdx.y * kNmCols;
    const size_t rb = (size_t)(n_in / NT::qk) * NT::bytes;
    const uint32_t* xd = reinterpret_cast<const uint32_t*>(xq) + (size_t)min(c0 + (tid >> 3), n_col - 1) * (n_in / 32 * 9);
    const int wr = ROWS == 64 ? 16 * wave : 16 * (wave & 1), wc = ROWS == 64 ? 0 : 16 * (wave >> 1);
    f32x4 tot[CT], hold[CT];
#pragma unroll
    for (int b = 0; b < CT; ++b) tot[b] = hold[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int v0 = 0, ph = 0; v0 < n_in; v0 += 256, ph ^= 1) {
        const int nb = min(8, (n_in - v0) / 32);  // 32-value blocks of this chunk
        const int np = nb * 32 / NT::qk * NT::ipb;
        // a block of x per thread (past the end the chunk's last one), the thread's partials; dead rows read the last row
        uint32_t xw[9];
        const uint32_t* src = xd + (size_t)(v0 / 32 + min(tid & 7, nb - 1)) * 9;
#pragma unroll
        for (int m = 0; m < 9; ++m) xw[m] = src[m];
        NativePart<TYPE, false> part[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = tid + 256 * u, k = min(p % NP, np - 1);
            part[u].decode(w + (size_t)min(r0 + p / NP, n_out - 1) * rb + (size_t)(v0 / NT::qk + k / NT::ipb) * NT::bytes,
                           NT::step * (k % NT::ipb));
        }
        if (v0) __syncthreads();  // the chunk before is read
        {
            uint8_t* xr = xs + (tid >> 3) * kNmPitch + 64 * (tid & 7);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint2 a = word_bits((int32_t)xw[1 + 2 * j]), b = word_bits((int32_t)xw[2 + 2 * j]);
                *reinterpret_cast<u32x4*>(xr + 16 * j) = u32x4{a.x, a.y, b.x, b.y};
            }
            dx[tid & 7][tid >> 3] = (float)__builtin_bit_cast(_Float16, (uint16_t)(xw[0] & 0xFFFFu));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = tid + 256 * u, row = p / NP;
            nm_put<TYPE, ROWS>(part[u], p % NP, ws + row * kNmPitch, dw + row);
        }
        __syncthreads();
        f32x4 half[2][CT];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
            for (int b = 0; b < CT; ++b) half[hf][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int blk = 4 * hf + j;
                if (blk >= nb) break;  // (uniform)
                const f16x8 a = __builtin_bit_cast(
                    f16x8, *reinterpret_cast<const u32x4*>(ws + (wr + i) * kNmPitch + 64 * blk + 16 * q));
                const f32x4 d = *reinterpret_cast<const f32x4*>(dw + blk * ROWS + wr + 4 * q);
#pragma unroll
                for (int b = 0; b < CT; ++b) {
                    const f16x8 x = __builtin_bit_cast(
                        f16x8, *reinterpret_cast<const u32x4*>(xs + (wc + 16 * b + i) * kNmPitch + 64 * blk + 16 * q));
                    const float xsc = dx[blk][wc + 16 * b + i];
                    const f32x4 S =
                        __builtin_amdgcn_mfma_f32_16x16x32_f16(a, x, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) half[hf][b][e] = __builtin_fmaf(d[e] * xsc, S[e], half[hf][b][e]);
                }
            }
        }
#pragma unroll
        for (int b = 0; b < CT; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = half[0][b][e] + half[1][b][e];
                if (ph) {
                    tot[b][e] = tot[b][e] + (hold[b][e] + v);
                    hold[b][e] = 0.0f;
                } else {
                    hold[b][e] = v;
                }
            }
    }
    // lane (q, i) holds rows 4 q .. + 3 of column i of each tile
    const int r = r0 + wr + 4 * q;
#pragma unroll
    for (int b = 0; b < CT; ++b) {
        const int c = c0 + wc + 16 * b + i;
        if (c >= n_col || r >= n_out) continue;
        const float g = sg ? sigmoid(sg[c]) : 1.0f;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = tot[b][e] + hold[b][e];
            if (sg) v[e] = v[e] * g;
        }
        *reinterpret_cast<f32x4*>(y + (size_t)c * ldy + r) = v;
    }
}

// y[t][j] *= sigmoid(sg[t]) for the shared rows a Q2_0 / IQ2_S down projection wrote
__global__ __launch_bounds__(256) void k_sigmoid_rows(float* __restrict__ y, int n, const float* __restrict__ sg) {
    const int t = blockIdx.y;
    const float s = sigmoid(sg[t]);
    for (int j = blockIdx.x * 256 + threadIdx.x; j < n; j += gridDim.x * 256) y[(size_t)t * n + j] = y[(size_t)t * n + j] * s;
}

// y[t][j] = y[t][j] + r[t][j]: a native shared expert's rows added after a combine that left them out (the same last
// addition the combine makes)
__global__ __launch_bounds__(256) void k_add_rows(float* __restrict__ y, const float* __restrict__ r, int n) {
    const size_t o = (size_t)blockIdx.y * n;
    for (int j = blockIdx.x * 256 + threadIdx.x; j < n; j += gridDim.x * 256) y[o + j] = y[o + j] + r[o + j];
}

}  // namespace

bool native_type(int type) {
    switch (type) {
        case 8: case 2: case 6: case 20: case 23: case 11: case 12: case 13: case 14: return true;
        default: return false;
    }
}

int native_block_values(int type) {
    switch (type) {
        case 8: case 2: case 6: case 20: return 32;
        case 23: case 11: case 12: case 13: case 14: return 256;
        default: return 0;
    }
}

int64_t native_row_bytes(int type, int64_t n) {
    int bytes = 0;
    switch (type) {
        case 8: bytes = 34; break;
        case 2: case 20: bytes = 18; break;
        case 6: bytes = 22; break;
        case 23: bytes = 136; break;
        case 11: bytes = 110; break;
        case 12: bytes = 144; break;
        case 13: bytes = 176; break;
        case 14: bytes = 210; break;
        default: return -1;
    }
    const int qk = native_block_values(type);
    return (n <= 0 || n % qk) ? -1 : n / qk * bytes;
}

hipError_t launch_mmvq_native(int type, const uint8_t* w, const uint8_t* xq, int n_in, int n_out, int n_col, float* y,
                              int ldy, const float* sg, hipStream_t s, const uint8_t* w2, float* y2) {
    if (!native_type(type) || n_in % native_block_values(type)) return hipErrorInvalidValue;
    const int nz = w2 ? 2 : 1;
    const int rg = (n_out + kNativeTileRows - 1) / kNativeTileRows, cols = native_cols(type, n_in, n_out, n_col, nz);
    const int cg = n_col < 64 ? n_col : 64;
    const dim3 grid1((unsigned)((n_out + 7) / 8), (unsigned)cg, (unsigned)nz);
    const dim3 gridc((unsigned)rg, (unsigned)((n_col + cols - 1) / cols), (unsigned)nz);
    const size_t lds = (size_t)cols * (n_in < kXlChunk ? n_in : kXlChunk) / 32 * kXlDw * 4;
#define SMOE_NATC(T, C) \
    hipLaunchKernelGGL((k_mmvq_native_cols<T, C>), gridc, dim3(256), lds, s, w, w2, n_in, n_out, n_col, xq, y, y2, ldy, sg)
#define SMOE_NAT(T)                                                                                                  \
    if (cols == 16) SMOE_NATC(T, 16);                                                                                \
    else if (cols == 8) SMOE_NATC(T, 8);                                                                             \
    else if (cols == 4) SMOE_NATC(T, 4);                                                                             \
    else                                                                                                             \
        hipLaunchKernelGGL(k_mmvq_native<T>, grid1, dim3(256), 0, s, w, w2, n_in, n_out, n_col, xq, y, y2, ldy, sg)
    switch (type) {
        case 8: SMOE_NAT(8); break;
        case 2: SMOE_NAT(2); break;
        case 6: SMOE_NAT(6); break;
        case 20: SMOE_NAT(20); break;
        case 23: SMOE_NAT(23); break;
        case 11: SMOE_NAT(11); break;
        case 12: SMOE_NAT(12); break;
        case 13: SMOE_NAT(13); break;
        default: SMOE_NAT(14); break;
    }
#undef SMOE_NAT
#undef SMOE_NATC
    return hipGetLastError();
}

// The prompt's product on the matrix cores, where it is the faster: the types k_native_mm takes, rows stored four at a time.
bool native_mm_ok(int type, int n_out, int n_col, int nz) {
    return (type == 8 || type == 2 || type == 6 || type == 20 || type == 11) && n_out % 4 == 0 &&
           native_mm_gains(n_out, n_col, nz);
}

hipError_t launch_native_mm(int type, const uint8_t* w, const uint8_t* xq, int n_in, int n_out, int n_col, float* y,
                            int ldy, const float* sg, hipStream_t s, const uint8_t* w2, float* y2) {
    const uintptr_t al = reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(y2);
    const int cg = (n_col + kNmCols - 1) / kNmCols;
    const unsigned nz = w2 ? 2 : 1;
    if (!native_mm_ok(type, n_out, n_col, (int)nz) || native_row_bytes(type, n_in) <= 0 || cg > 65535 || ldy % 4 || (al & 15))
        return hipErrorInvalidValue;
    // 32 rows while 64 leave no second work-group per CU (the layer call at 128, 400 and 900 tokens: 221, 289 and 439 us
    // in 32 rows, 227, 290 and 427 in 64)
    const int rows = (int64_t)((n_out + 63) / 64) * cg * nz <= 256 ? 32 : 64;
    const dim3 grid((unsigned)((n_out + rows - 1) / rows), (unsigned)cg, nz);
#define SMOE_NMR(T, R) \
    hipLaunchKernelGGL((k_native_mm<T, R>), grid, dim3(256), 0, s, w, w2, n_in, n_out, n_col, xq, y, y2, ldy, sg)
#define SMOE_NM(T)                        \
    if (rows == 32) SMOE_NMR(T, 32);      \
    else SMOE_NMR(T, 64)
    switch (type) {
        case 8: SMOE_NM(8); break;
        case 2: SMOE_NM(2); break;
        case 6: SMOE_NM(6); break;
        case 20: SMOE_NM(20); break;
        default: SMOE_NM(11); break;
    }
#undef SMOE_NM
#undef SMOE_NMR
    return hipGetLastError();
}

// A native shared expert whose gate and up have one type and whose down is native, where two launches are the faster.
bool native_few_ok(int gu_type, int d_type, int T, int H, int F) {
    return native_few_gains(T, H, F) && native_row_bytes(gu_type, H) > 0 && native_row_bytes(d_type, F) > 0 && H <= 4096 &&
           F <= 4096;
}

hipError_t launch_native_few(int gu_type, int d_type, const float* x, const uint8_t* gate, const uint8_t* up,
                             const uint8_t* down, int T, int H, int F, float* h, const float* sg, int add, float* y,
                             hipStream_t s) {
    if (!native_few_ok(gu_type, d_type, T, H, F) || T < 1) return hipErrorInvalidValue;
    const dim3 g1((unsigned)((F + 7) / 8), (unsigned)T), g2((unsigned)((H + 7) / 8), (unsigned)T);
    const size_t l1 = (size_t)(H / 32) * kXlDw * 4, l2 = (size_t)(F / 32) * kXlDw * 4;
#define SMOE_EACH_NATIVE(type, CALL) \
    switch (type) {                  \
        case 8: CALL(8); break;      \
        case 2: CALL(2); break;      \
        case 6: CALL(6); break;      \
        case 20: CALL(20); break;    \
        case 23: CALL(23); break;    \
        case 11: CALL(11); break;    \
        case 12: CALL(12); break;    \
        case 13: CALL(13); break;    \
        default: CALL(14); break;    \
    }
#define SMOE_GU(T_) hipLaunchKernelGGL(k_native_gu<T_>, g1, dim3(512), l1, s, x, gate, up, H, F, h)
#define SMOE_DN(T_) hipLaunchKernelGGL(k_native_down<T_>, g2, dim3(256), l2, s, h, down, F, H, sg, add, y)
    SMOE_EACH_NATIVE(gu_type, SMOE_GU)
    SMOE_EACH_NATIVE(d_type, SMOE_DN)
#undef SMOE_DN
#undef SMOE_GU
#undef SMOE_EACH_NATIVE
    return hipGetLastError();
}

hipError_t launch_sigmoid_rows(float* y, int T, int n, const float* sg, hipStream_t s) {
    const int bx = (n + 255) / 256;
    hipLaunchKernelGGL(k_sigmoid_rows, dim3((unsigned)(bx < 16 ? bx : 16), (unsigned)T), dim3(256), 0, s, y, n, sg);
    return hipGetLastError();
}

hipError_t launch_add_rows(float* y, const float* r, int T, int n, hipStream_t s) {
    const int bx = (n + 255) / 256;
    hipLaunchKernelGGL(k_add_rows, dim3((unsigned)(bx < 16 ? bx : 16), (unsigned)T), dim3(256), 0, s, y, r, n);
    return hipGetLastError();
}

}  // namespace smoe
