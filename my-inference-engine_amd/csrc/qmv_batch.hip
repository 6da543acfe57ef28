/*
 * gfx950 kernels of the packed products of 2 to 32 positions on the matrix
 * cores, and of one position over short Q8_0 and Q5_0 rows with the RMSNorm.
 *
 * A workgroup takes a chunk of K (all of it where its activations fit LDS)
 * and a range of 16-row groups. It stages the chunk's activations in LDS
 * once, as matrix-core operands; then every wave streams weights on its own,
 * an item (row group, segment of K) after the other, with no barrier: an
 * activation is loaded and split once per workgroup, and a weight unit is
 * decoded once for all positions. Where the chunk is all of K the segments'
 * sums meet in LDS and the epilogue (RMSNorm's division, SwiGLU, addend) is
 * done here; else a second kernel adds them. What bounds it: up to 8 positions
 * the weight stream (gate|up 18944 x 3584 Q4_K with norm and SwiGLU at 8
 * positions 23.7 us, 76.6 MB: 3.2 TB/s with the launch, staging and epilogue;
 * 40.8 us before on split-K launches with bf16 limbs and a norm launch); at 32
 * the vector instructions that decode weights and apply scales, 33k of 48k
 * cycles of a SIMD, with the matrix cores' 19k (64 us before, 41 with its
 * reduction).
 *
 * Activations. x of one position and unit is scaled by the power of two that
 * brings the largest magnitude to [2^14, 2^15) and split into two f16 limbs,
 * xs = h + l * 2^-12 with h = f16(xs) and l = f16((xs - h) * 2^12). The two
 * limbs are summed apart, so l's range reaches 2^-36. That is one bit less
 * than a float: what h leaves takes up to 12 bits and l has 11, so a quarter of
 * all floats lose their last place. An activation within 2^28 of its unit's
 * largest is held to 2^-23 of itself; below, the error is at most 2^-51 of the
 * largest. The matvec kernels multiply the float, or three bf16 limbs that are
 * exact; the sums are still nearer to 64 bits here, because fewer roundings
 * follow (7B layers, relative 2-norm, matvec and prefill kernels / this: 4
 * positions 4.4e-7 / 3.3e-7, 13 4.6e-7 / 3.1e-7, 32 4.6e-7 / 3.1e-7; Q6_K
 * vocabulary at 4 2.1e-7 / 1.2e-7). Q4_K's sums of x are two limbs as well.
 * Sums of infinities and NaN are taken
 * again (finish_rows).
 *
 * Weights. An integer in the low bits of an f16 is a subnormal, so a mask and
 * one packed multiply-add with a sub-block's integer scale make exact f16
 * operands (Q4_K: scale * (code - 8), at most 504; Q6_K: two operands, scale *
 * (low nibble - 8) and scale * 8 (2 top bits - 3)). The sub-block scales are
 * thus inside the products, and a super-block needs no scaling of partial
 * sums: d and dmin are applied once to its sum. Codes are centred because the
 * matrix core's accumulation rounds with the size of what it adds: with codes
 * 0..15 the 7B q projection came out at 1.8-3.2e-7 of the 64-bit result,
 * centred at 1.5-1.7e-7 (2.2e-7 before this kernel). Lane kc of a column holds
 * any 8 k of a step, as long as the activations are staged in the same order,
 * so each lane reads whole 16-byte pieces of the planes and unpacks only its
 * own two (Q6_K: four) sub-blocks' scales. Q4_K's minimums, and the 8 of its
 * codes, are one product each of their integers with the sub-blocks' sums of
 * x. Q8_0 and Q5_0 have one f16 scale per 32 weights, a step, and scale each
 * step's sum.
 *
 * Up to 8 positions the limbs share the matrix core's 16 rows (h in rows
 * 0..7, l in rows 8..15), so a step is one MFMA and one LDS read.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qmv_kernels.h"

namespace qmv {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2_t as_h2(uint32_t v) { return __builtin_bit_cast(h2_t, v); }
__device__ __forceinline__ uint32_t as_u32(h2_t v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2_t h2_of(float v) { return h2_t{(_Float16)v, (_Float16)v}; }

__device__ __forceinline__ float half_bits(uint32_t bits)
{
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits & 0xffffu));
}

/* Two bytes of the words (hi, lo) by a v_perm selector, each with the high
 * byte 0x64 of the f16 1024 + byte. */
__device__ __forceinline__ h2_t bytes_plus_1024(uint32_t word, uint32_t sel)
{
    return as_h2(__builtin_amdgcn_perm(0x64646464u, word, sel));
}

/* v of the lane that DPP control CTRL names (all lanes active). */
template <int CTRL> __device__ __forceinline__ float dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ uint32_t dpp_bits(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL> __device__ __forceinline__ double dpp_double(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)dpp_bits<CTRL>((uint32_t)(u >> 32)) << 32 | dpp_bits<CTRL>((uint32_t)u));
}
#define DPP_XOR1 0xB1        /* quad_perm [1, 0, 3, 2] */
#define DPP_XOR2 0x4E        /* quad_perm [2, 3, 0, 1] */
#define DPP_HALF_MIRROR 0x141 /* lane i of 8 from 7 - i */
#define DPP_ROR8 0x128       /* rotate the 16-lane row by 8 */

/* ---- the formats ------------------------------------------------------------------
 * kUnit: weights per tiled unit (and staged at once); kSteps: MFMA steps of 32
 * k per unit. place(): where the float4 at k = 64 j + 4 i of a unit goes: the
 * step, the lane group kc and the half of its 8 slots. kSwap: the slots hold
 * elements 0, 2, 1, 3 of the float4 (nibbles come off a word as bytes 0, 2
 * and 1, 3). */
template <int FMT> struct BatchFmt;

template <> struct BatchFmt<QMV_FMT_Q4_K> {
    static constexpr int kUnit = 256, kSteps = 8, kUnitBytes = 144;
    static constexpr bool kSwap = true, kMins = true, kPerStep = false;
    struct W { u4_t h, a, b; };
    __device__ static void place(int j, int i, int &step, int &kc, int &half) { step = i & 7; kc = j; half = i >> 3; }
    /* lane (row, kc): both nibble halves of 64-weight chunk kc */
    __device__ static void load(W &w, const uint8_t *slab, int row, int kc)
    {
        w.h = *(const u4_t *)(slab + row * 16);
        w.a = *(const u4_t *)(slab + 1024 + kc * 2048 + row * 16);
        w.b = *(const u4_t *)(slab + 2048 + kc * 2048 + row * 16);
    }
};

template <> struct BatchFmt<QMV_FMT_Q6_K> {
    static constexpr int kUnit = 256, kSteps = 8, kUnitBytes = 210;
    static constexpr bool kSwap = true, kMins = false, kPerStep = false;
    struct W { u4_t a, b, q; u2_t s; uint32_t d; };
    __device__ static void place(int j, int i, int &step, int &kc, int &half)
    {
        step = 4 * (i >> 3) + (i & 3);
        kc = 2 * (j >> 1) + ((i >> 2) & 1);
        half = j & 1;
    }
    /* lane (row, kc): weights 128 (kc >> 1) + 16 (kc & 1) + {0, 32, 64, 96} + 0..15 */
    __device__ static void load(W &w, const uint8_t *slab, int row, int kc)
    {
        const int hf = kc >> 1, b = kc & 1;
        w.a = *(const u4_t *)(slab + (4 * hf + b) * 1024 + row * 16);
        w.b = *(const u4_t *)(slab + (4 * hf + 2 + b) * 1024 + row * 16);
        w.q = *(const u4_t *)(slab + (8 + 2 * hf + b) * 1024 + row * 16);
        w.s = *(const u2_t *)(slab + 12 * 1024 + row * 16 + 8 * hf);
        w.d = *(const uint16_t *)(slab + 13 * 1024 + row * 2);
    }
};

template <> struct BatchFmt<QMV_FMT_Q8_0> {
    static constexpr int kUnit = 128, kSteps = 4, kUnitBytes = 136;
    static constexpr bool kSwap = false, kMins = false, kPerStep = true;
    struct W { u2_t q[4]; u2_t d; };
    __device__ static void place(int j, int i, int &step, int &kc, int &half)
    {
        step = 2 * j + (i >> 3);
        kc = (i & 7) >> 1;
        half = i & 1;
    }
    /* lane (row, kc): weights 8 kc .. 8 kc + 7 of each block */
    __device__ static void load(W &w, const uint8_t *slab, int row, int kc)
    {
#pragma unroll
        for (int t = 0; t < 4; ++t)
            w.q[t] = *(const u2_t *)(slab + (2 * t + (kc >> 1)) * 1024 + row * 16 + 8 * (kc & 1));
        w.d = *(const u2_t *)(slab + 8 * 1024 + row * 8);
    }
};

template <> struct BatchFmt<QMV_FMT_Q5_0> {
    static constexpr int kUnit = 128, kSteps = 4, kUnitBytes = 88;
    static constexpr bool kSwap = true, kMins = false, kPerStep = true;
    struct W { uint32_t q[4]; u4_t h; u2_t d; };
    __device__ static void place(int j, int i, int &step, int &kc, int &half)
    {
        step = 2 * j + (i >> 3);
        kc = i & 3;
        half = (i & 7) >> 2;
    }
    /* lane (row, kc): weights 4 kc .. 4 kc + 3 and 16 more of each block */
    __device__ static void load(W &w, const uint8_t *slab, int row, int kc)
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) w.q[t] = *(const uint32_t *)(slab + t * 1024 + row * 16 + 4 * kc);
        w.h = *(const u4_t *)(slab + 4 * 1024 + row * 16);
        w.d = *(const u2_t *)(slab + 5 * 1024 + row * 8);
    }
};

/* ---- the staged activations of one unit ----------------------------------------------
 * NR rounds of 4 positions. F fragments: one with h in rows 0..7 and l in
 * rows 8..15 (up to 8 positions), or h and l of each block of 16 positions.
 * A fragment's step is [4 kc][kRows][16 bytes], padded by 64 bytes so that the
 * 16 lanes that write one position's float4s reach different banks. */
template <int FMT, int NR> struct BatchStage {
    using B = BatchFmt<FMT>;
    static constexpr int P = 4 * NR;               /* position slots */
    static constexpr int F = NR <= 2 ? 1 : NR / 2; /* MFMA per step and row group */
    static constexpr int kBlocks = (F + 1) / 2;   /* blocks of 16 positions (one of 8) */
    static constexpr int kRows = NR <= 2 ? 2 * P : 16;
    static constexpr int kStep = 4 * kRows * 16 + 64;
    static constexpr int kFrag = B::kSteps * kStep;
    static constexpr int kSumRows = F == 1 ? P : 16;
    static constexpr int kSums = F * kFrag; /* sums of x: [kBlocks][4 kc][kSumRows][h, h, l, l of two sub-blocks] */
    static constexpr int kInv = kSums + (B::kMins ? kBlocks * 4 * kSumRows * 8 : 0); /* 1 / scale: [P] floats */
    static constexpr int kSsq = kInv + (P < 8 ? 8 : P) * 4; /* sum of x^2 (the RMSNorm): [P] doubles */
    static constexpr int kBytes = (kSsq + P * 8 + 63) & ~63;
    __device__ static int h_frag(int pos) { return F == 1 ? 0 : 2 * (pos >> 4); }
    __device__ static int l_frag(int pos) { return F == 1 ? 0 : 2 * (pos >> 4) + 1; }
    __device__ static int h_row(int pos) { return F == 1 ? pos : pos & 15; }
    __device__ static int l_row(int pos) { return F == 1 ? P + pos : pos & 15; }
};

/* Stage one position's share of a unit: lane i = 0..15 of the position holds
 * v[j] = x[64 j + 4 i ..]. */
template <int FMT, int NR>
__device__ __forceinline__ void stage_position(uint8_t *lds, const f4_t (&v)[BatchFmt<FMT>::kUnit / 64], int pos, int i)
{
    using B = BatchFmt<FMT>;
    using L = BatchStage<FMT, NR>;
    constexpr int NJ = B::kUnit / 64;
    /* the largest magnitude as bits (a NaN counts as the largest) */
    uint32_t mx = 0;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = max(mx, __float_as_uint(v[j][e]) << 1);
    mx = max(mx, dpp_bits<DPP_XOR1>(mx));
    mx = max(mx, dpp_bits<DPP_XOR2>(mx));
    mx = max(mx, dpp_bits<DPP_HALF_MIRROR>(mx));
    mx = max(mx, dpp_bits<DPP_ROR8>(mx));
    /* 2^(14 - its exponent), at most 2^114 (all-zero and tiny units) */
    const int e = 268 - (int)(mx >> 24);
    const int b = e < 241 ? e : 241;
    const float s = __uint_as_float((uint32_t)b << 23), s12 = __uint_as_float((uint32_t)(b + 12) << 23);
    if (i == 0) *(float *)(lds + L::kInv + 4 * pos) = __uint_as_float((uint32_t)(254 - b) << 23);
    uint8_t *hp = lds + L::h_frag(pos) * L::kFrag + L::h_row(pos) * 16;
    uint8_t *lp = lds + L::l_frag(pos) * L::kFrag + L::l_row(pos) * 16;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        int step, kc, half;
        B::place(j, i, step, kc, half);
        const int at = step * L::kStep + kc * (L::kRows * 16) + half * 8;
        const f4_t x = v[j], t = x * s, u = x * s12;
        const float y0 = t[0], y1 = B::kSwap ? t[2] : t[1], y2 = B::kSwap ? t[1] : t[2], y3 = t[3];
        const float z0 = u[0], z1 = B::kSwap ? u[2] : u[1], z2 = B::kSwap ? u[1] : u[2], z3 = u[3];
        h2_t h01 = {(_Float16)y0, (_Float16)y1}, h23 = {(_Float16)y2, (_Float16)y3};
        asm("" : "+v"(h01), "+v"(h23)); /* else the conversions are repeated for the remainders */
        const h2_t l01 = {(_Float16)fmaf((float)h01[0], -4096.0f, z0), (_Float16)fmaf((float)h01[1], -4096.0f, z1)};
        const h2_t l23 = {(_Float16)fmaf((float)h23[0], -4096.0f, z2), (_Float16)fmaf((float)h23[1], -4096.0f, z3)};
        *(u2_t *)(hp + at) = u2_t{as_u32(h01), as_u32(h23)};
        *(u2_t *)(lp + at) = u2_t{as_u32(l01), as_u32(l23)};
        if constexpr (B::kMins) { /* the sum of each 32-weight sub-block, 8 lanes */
            float sum = (t[0] + t[1]) + (t[2] + t[3]);
            sum += dpp<DPP_XOR1>(sum);
            sum += dpp<DPP_XOR2>(sum);
            sum += dpp<DPP_HALF_MIRROR>(sum);
            if ((i & 7) == 0) {
                const float q = sum * 0x1p-6f; /* at most 2^14 */
                const _Float16 sh = (_Float16)q, sl = (_Float16)fmaf((float)sh, -4096.0f, q * 4096.0f);
                uint8_t *sp = lds + L::kSums + (((pos >> 4) * 4 + j) * L::kSumRows + (pos & (L::kSumRows - 1))) * 8;
                *(_Float16 *)(sp + 2 * (i >> 3)) = sh;
                *(_Float16 *)(sp + 2 * (i >> 3) + 4) = sl;
            }
        }
    }
}

/* ---- a unit's products --------------------------------------------------------------- */

__device__ __forceinline__ f4_t mma(h8_t a, u4_t b, f4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
}

/* One unit of 16 weight rows as matrix-core operands. */
template <int FMT> struct BatchB;

template <> struct BatchB<QMV_FMT_Q4_K> {
    u4_t b[8];
    h4_t mins, scales;
    float d, dm;
    __device__ __forceinline__ void decode(const BatchFmt<QMV_FMT_Q4_K>::W &w, int kc)
    {
        /* sub-blocks 0..3: the low 6 bits of u0 / u1; 4..7: the nibbles of u2
         * with the top bits of u0 / u1. One form for both: shifts and masks
         * by lane, no branch. */
        const uint32_t u0 = w.h[1], u1 = w.h[2], u2 = w.h[3];
        const uint32_t hs = kc & 2, hm = kc < 2 ? 0x3f3f3f3fu : 0x30303030u, lm = kc < 2 ? 0u : 0x0f0f0f0fu;
        const uint32_t sc = ((u0 >> hs) & hm) | (u2 & lm), mn = ((u1 >> hs) & hm) | ((u2 >> 4) & lm);
        const uint32_t sel = 0x04000400u | ((kc & 1) ? 0x00020002u : 0u);
        const h2_t k0 = bytes_plus_1024(sc, sel) - h2_of(1024.0f);
        const h2_t k1 = bytes_plus_1024(sc, sel + 0x00010001u) - h2_of(1024.0f);
        const h2_t s0 = k0 * h2_of(512.0f), s1 = k1 * h2_of(32.0f);
        const h2_t o0 = k0 * h2_of(-8 * 0x1p-15f), o1 = k1 * h2_of(-8 * 0x1p-15f);
        const h2_t m = bytes_plus_1024(mn, sel + 0x00010000u) - h2_of(1024.0f);
        const h2_t k = {k0[0], k1[0]}, lm2 = m * h2_of(0x1p-12f), lk = k * h2_of(0x1p-12f); /* for the l limbs */
        mins = h4_t{m[0], m[1], lm2[0], lm2[1]};
        scales = h4_t{k[0], k[1], lk[0], lk[1]};
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const uint32_t dw = t < 4 ? w.a[t & 3] : w.b[t & 3], od = dw >> 8;
            b[t] = u4_t{as_u32(__builtin_elementwise_fma(as_h2(dw & 0x000f000fu), s0, o0)),
                        as_u32(__builtin_elementwise_fma(as_h2(od & 0x000f000fu), s0, o0)),
                        as_u32(__builtin_elementwise_fma(as_h2(dw & 0x00f000f0u), s1, o1)),
                        as_u32(__builtin_elementwise_fma(as_h2(od & 0x00f000f0u), s1, o1))};
        }
        d = half_bits(w.h[0]) * 0x1p15f; /* products carry 2^-15, sums of x 2^-6 */
        dm = half_bits(w.h[0] >> 16) * -0x1p6f;
    }
};

/* Codes in the low bits of a half are q * 2^-24 (low nibbles), 16 q * 2^-24
 * (high), top bits h * 2^-20 or h * 2^-18; every operand carries 2^-16. q - 32
 * = (nibble - 8) + 8 (2 h - 3), each times the scale exact in an f16. */
template <> struct BatchB<QMV_FMT_Q6_K> {
    u4_t b[8], c[8];
    float d;
    __device__ __forceinline__ void decode(const BatchFmt<QMV_FMT_Q6_K>::W &w, int kc)
    {
        h2_t sn[4], sh[4], on[4], oh[4];
        const uint32_t sel = 0x04000400u | ((kc & 1) ? 0x00010001u : 0u);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const h2_t sc =
                bytes_plus_1024(w.s[k >> 1] ^ 0x80808080u, sel + ((k & 1) ? 0x00020002u : 0u)) - h2_of(1152.0f);
            sn[k] = sc * h2_of(k < 2 ? 256.0f : 16.0f);
            sh[k] = sc * h2_of(k & 1 ? 64.0f : 256.0f);
            on[k] = sc * h2_of(-8 * 0x1p-16f);
            oh[k] = sc * h2_of(-24 * 0x1p-16f);
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            /* steps 0..3: sub-blocks 0 (low nibbles) and 2 (high); 4..7: 1 and 3 */
            constexpr uint32_t kLo = 0x000f000fu, kHi = 0x00f000f0u;
            const int k0 = t < 4 ? 0 : 1, k1 = k0 + 2;
            const uint32_t top = t < 4 ? 0x00300030u : 0x00c000c0u;
            const uint32_t dw = t < 4 ? w.a[t & 3] : w.b[t & 3], q = w.q[t & 3], od = dw >> 8;
            b[t] = u4_t{as_u32(__builtin_elementwise_fma(as_h2(dw & kLo), sn[k0], on[k0])),
                        as_u32(__builtin_elementwise_fma(as_h2(od & kLo), sn[k0], on[k0])),
                        as_u32(__builtin_elementwise_fma(as_h2(dw & kHi), sn[k1], on[k1])),
                        as_u32(__builtin_elementwise_fma(as_h2(od & kHi), sn[k1], on[k1]))};
            c[t] = u4_t{as_u32(__builtin_elementwise_fma(as_h2((q << 4) & top), sh[k0], oh[k0])),
                        as_u32(__builtin_elementwise_fma(as_h2((q >> 4) & top), sh[k0], oh[k0])),
                        as_u32(__builtin_elementwise_fma(as_h2(q & top), sh[k1], oh[k1])),
                        as_u32(__builtin_elementwise_fma(as_h2((q >> 8) & top), sh[k1], oh[k1]))};
        }
        d = half_bits(w.d) * 0x1p16f;
    }
};

template <> struct BatchB<QMV_FMT_Q8_0> {
    u4_t b[4];
    float d[4];
    __device__ __forceinline__ void decode(const BatchFmt<QMV_FMT_Q8_0>::W &w, int)
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t q0 = w.q[t][0] ^ 0x80808080u, q1 = w.q[t][1] ^ 0x80808080u; /* q + 128 */
            const h2_t k = h2_of(1152.0f);
            b[t] = u4_t{as_u32(bytes_plus_1024(q0, 0x04010400u) - k), as_u32(bytes_plus_1024(q0, 0x04030402u) - k),
                        as_u32(bytes_plus_1024(q1, 0x04010400u) - k), as_u32(bytes_plus_1024(q1, 0x04030402u) - k)};
            d[t] = half_bits(w.d[t >> 1] >> (16 * (t & 1)));
        }
    }
};

template <> struct BatchB<QMV_FMT_Q5_0> {
    u4_t b[4];
    float d[4];
    __device__ __forceinline__ void decode(const BatchFmt<QMV_FMT_Q5_0>::W &w, int kc)
    {
        /* nibble | fifth bit << 4 in the low bits of each half, q * 2^-24
         * (high nibbles 4 bits up), to (q - 16) * 2^-9 */
        const h2_t lo = h2_of(32768.0f), hi = h2_of(2048.0f), off = h2_of(-0x1p-5f);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t q = w.q[t], od = q >> 8, bits = w.h[t] >> (4 * kc), hb = bits >> 16;
            const uint32_t e0 = (bits & 1u) << 4 | (bits & 4u) << 18, e1 = (bits & 2u) << 3 | (bits & 8u) << 17;
            const uint32_t e2 = (hb & 1u) << 8 | (hb & 4u) << 22, e3 = (hb & 2u) << 7 | (hb & 8u) << 21;
            b[t] = u4_t{as_u32(__builtin_elementwise_fma(as_h2((q & 0x000f000fu) | e0), lo, off)),
                        as_u32(__builtin_elementwise_fma(as_h2((od & 0x000f000fu) | e1), lo, off)),
                        as_u32(__builtin_elementwise_fma(as_h2((q & 0x00f000f0u) | e2), hi, off)),
                        as_u32(__builtin_elementwise_fma(as_h2((od & 0x00f000f0u) | e3), hi, off))};
            d[t] = half_bits(w.d[t >> 1] >> (16 * (t & 1))) * 512.0f;
        }
    }
};

/* Fragment f of a staged unit: a lane's 16 bytes of every step. */
template <int FMT, int NR>
__device__ __forceinline__ void read_fragment(h8_t (&a)[BatchFmt<FMT>::kSteps], const uint8_t *stage, int f, int row,
                                              int kc)
{
    using L = BatchStage<FMT, NR>;
#pragma unroll
    for (int t = 0; t < BatchFmt<FMT>::kSteps; ++t)
        a[t] = *(const h8_t *)(stage + f * L::kFrag + t * L::kStep + (kc * L::kRows + row) * 16);
}

/* Add one unit's products to y: R row groups, the staged unit in LDS. A
 * fragment's reads are issued before the products of the one before it (the
 * first one's by the caller, before the weights are decoded): left to itself
 * the compiler puts each read next to its use, and the wave then waits out
 * the LDS latency at every step (151936 x 3584 Q6_K at 32 positions 241 us
 * against 212). The K-quants run two chains of 4 MFMA each on the h limbs
 * (Q6_K: four), which keeps the accumulators' rounding below that of a chain
 * of 8; l sums, 2^-12 of them, need one. y: lanes of F == 1
 * hold h sums (lanes 0..31) or l sums, joined at the end of the item;
 * otherwise h and l are joined here, per block of 16 positions. */
template <int FMT, int NR, int R>
__device__ __forceinline__ void unit_product(const BatchB<FMT> (&w)[R], h8_t (&a)[BatchFmt<FMT>::kSteps],
                                             const uint8_t *stage, int row, int kc,
                                             f4_t (&y)[R][BatchStage<FMT, NR>::kBlocks])
{
    using B = BatchFmt<FMT>;
    using L = BatchStage<FMT, NR>;
    constexpr int kLimbs = L::F == 1 ? 1 : 2;
    const f4_t zero = {0, 0, 0, 0};
#pragma unroll
    for (int blk = 0; blk < L::kBlocks; ++blk) {
        const int at = L::F == 1 ? (L::P == 4 ? 0 : (kc & 1) * 4) : blk * 16 + kc * 4;
        const f4_t inv = *(const f4_t *)(stage + L::kInv + 4 * at);
        f4_t s[R]; /* h + 2^-12 l of the codes' products with the scales */
        h4_t sa;   /* both limbs of the sub-blocks' sums of x (in the h rows) */
        if constexpr (B::kMins) {
            const int sr = L::F == 1 ? row & (L::P - 1) : row;
            const u2_t v = *(const u2_t *)(stage + L::kSums + ((blk * 4 + kc) * L::kSumRows + sr) * 8);
            sa = __builtin_bit_cast(h4_t, L::F == 1 && row >= L::P ? u2_t{0, 0} : v);
        }
#pragma unroll
        for (int limb = 0; limb < kLimbs; ++limb) {
            const int f = blk * kLimbs + limb;
            const bool low = limb == 1;
            h8_t an[B::kSteps];
            if (f + 1 < L::F) {
                read_fragment<FMT, NR>(an, stage, f + 1, row, kc);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (B::kPerStep) {
#pragma unroll
                for (int t = 0; t < B::kSteps; ++t)
#pragma unroll
                    for (int g = 0; g < R; ++g) {
                        const f4_t p = mma(a[t], w[g].b[t], zero);
                        const float d = low ? w[g].d[t] * 0x1p-12f : w[g].d[t];
#pragma unroll
                        for (int r = 0; r < 4; ++r) s[g][r] = !low && t == 0 ? d * p[r] : fmaf(d, p[r], s[g][r]);
                    }
            } else {
                f4_t c0[R], c1[R], c2[R], c3[R];
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int g = 0; g < R; ++g) {
                        c0[g] = mma(a[t], w[g].b[t], t ? c0[g] : zero);
                        if constexpr (FMT == QMV_FMT_Q6_K) c2[g] = mma(a[t], w[g].c[t], t ? c2[g] : zero);
                        if (low) continue;
                        c1[g] = mma(a[t + 4], w[g].b[t + 4], t ? c1[g] : zero);
                        if constexpr (FMT == QMV_FMT_Q6_K) c3[g] = mma(a[t + 4], w[g].c[t + 4], t ? c3[g] : zero);
                    }
                if (low) {
#pragma unroll
                    for (int t = 4; t < 8; ++t)
#pragma unroll
                        for (int g = 0; g < R; ++g) {
                            c0[g] = mma(a[t], w[g].b[t], c0[g]);
                            if constexpr (FMT == QMV_FMT_Q6_K) c2[g] = mma(a[t], w[g].c[t], c2[g]);
                        }
                }
#pragma unroll
                for (int g = 0; g < R; ++g) {
                    f4_t sum = low ? c0[g] : c0[g] + c1[g];
                    if constexpr (FMT == QMV_FMT_Q6_K) sum += low ? c2[g] : c2[g] + c3[g];
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[g][r] = low ? fmaf(sum[r], 0x1p-12f, s[g][r]) : sum[r];
                }
            }
            if (f + 1 < L::F) {
#pragma unroll
                for (int t = 0; t < B::kSteps; ++t) a[t] = an[t];
            }
        }
#pragma unroll
        for (int g = 0; g < R; ++g) {
            f4_t m, e;
            if constexpr (B::kMins) {
                m = __builtin_amdgcn_mfma_f32_16x16x16f16(sa, w[g].mins, zero, 0, 0, 0);
                e = __builtin_amdgcn_mfma_f32_16x16x16f16(sa, w[g].scales, zero, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = s[g][r];
                if constexpr (B::kMins) v = fmaf(e[r], 0x1p-6f, v); /* the codes' 8: 8 * 2^6 * 2^-15 */
                if constexpr (!B::kPerStep) v *= w[g].d;
                if constexpr (B::kMins) v = fmaf(w[g].dm, m[r], v);
                y[g][blk][r] = fmaf(inv[r], v, y[g][blk][r]);
            }
        }
    }
}

/* ---- the kernels ---------------------------------------------------------------------- */

__device__ __forceinline__ float silu_product(float g, float u) { return u * (g / (1.0f + expf(-g))); }

/* First unit of segment s. */
__device__ __forceinline__ int segment_begin(const BatchParams &p, int s)
{
    return s * p.seg_units + (s < p.seg_more ? s : p.seg_more);
}

/* Tensor and row group of the launch's row group `group`: the jobs' groups in
 * turn, or gate and up groups alternating (SwiGLU). */
__device__ __forceinline__ void locate_group(const BatchParams &p, int group, int &job, int &rg)
{
    if (p.swiglu) {
        job = group & 1;
        rg = group >> 1;
        return;
    }
    job = 0;
#pragma unroll
    for (int i = 1; i < QMV_MAX_JOBS; ++i) job = group >= p.job[i].group_begin ? i : job;
    rg = group - p.job[job].group_begin;
}

/* The same, and the tensor's weights, by selects among every job's fields
 * (unused slots begin past the last group): the fields are read once, at the
 * kernel's start, so no memory round trip stands before an item's weights. */
__device__ __forceinline__ const uint8_t *group_weights(const BatchParams &p, int group, int &rg)
{
    if (p.swiglu) {
        rg = group >> 1;
        return group & 1 ? p.job[1].w : p.job[0].w;
    }
    const uint8_t *w = p.job[0].w;
    int begin = 0;
#pragma unroll
    for (int i = 1; i < QMV_MAX_JOBS; ++i) {
        const bool past = group >= p.job[i].group_begin;
        w = past ? p.job[i].w : w;
        begin = past ? p.job[i].group_begin : begin;
    }
    rg = group - begin;
    return w;
}

/* The sum of n values (or vectors) s[0], s[stride], ...: four running sums of
 * every fourth value, then those, loads eight at a time. The four keep the
 * rounding of long rows' many segments down. */
template <typename T, typename S>
__device__ __forceinline__ T strided_sum(const S *s, size_t stride, int n)
{
    T v[4] = {T(0), T(0), T(0), T(0)};
    const auto add = [&](int i, auto count) { /* s[i ..], as many as count */
        constexpr int N = decltype(count)::value;
        T q[N];
#pragma unroll
        for (int j = 0; j < N; ++j) q[j] = *(const T *)(s + (i + j < n ? i + j : n - 1) * stride);
#pragma unroll
        for (int j = 0; j < N; ++j) v[j & 3] += i + j < n ? q[j] : T(0);
    };
    if (n <= 4)
        add(0, std::integral_constant<int, 4>());
    else
        for (int i = 0; i < n; i += 8) add(i, std::integral_constant<int, 8>());
    return (v[0] + v[1]) + (v[2] + v[3]);
}

/* Weight i of the row in lane `row` of a tile, in the unit at slab. */
template <int FMT> __device__ float tiled_weight(const uint8_t *slab, int row, int i)
{
    const auto byte = [&](int j) { return (int)slab[(j >> 4) * 1024 + row * 16 + (j & 15)]; }; /* of the 16-byte planes */
    const auto half = [&](int at) { return half_bits(*(const uint16_t *)(slab + at)); };
    if constexpr (FMT == QMV_FMT_Q8_0) return half(8 * 1024 + row * 8 + 2 * (i >> 5)) * (float)(int8_t)byte(i);
    if constexpr (FMT == QMV_FMT_Q5_0) {
        const int b = i >> 5, j = i & 31, q = byte(16 * b + (j & 15)) >> (j < 16 ? 0 : 4) & 15;
        const int top = byte(64 + 4 * b + (j >> 3)) >> (j & 7) & 1;
        return half(5 * 1024 + row * 8 + 2 * b) * (float)((q | top << 4) - 16);
    }
    if constexpr (FMT == QMV_FMT_Q6_K) {
        const int h = i >> 7, k = i >> 5 & 3, l = i & 31;
        const int q = byte(64 * h + 32 * (k & 1) + l) >> (k < 2 ? 0 : 4) & 15, top = byte(128 + 32 * h + l) >> 2 * k & 3;
        return half(13 * 1024 + row * 2) * (float)(int8_t)byte(192 + (i >> 4)) * (float)((q | top << 4) - 32);
    }
    const int k = i >> 5, q = byte(16 + 32 * (i >> 6) + (i & 31)) >> (k & 1 ? 4 : 0) & 15;
    const int lo = byte(4 + (k & 3)), mid = byte(8 + (k & 3)), hi = k < 4 ? 0 : byte(8 + k);
    const int sc = k < 4 ? lo & 63 : (hi & 15) | (lo >> 6) << 4, m = k < 4 ? mid & 63 : hi >> 4 | (mid >> 6) << 4;
    return __fsub_rn(__fmul_rn(half(row * 16), (float)sc) * (float)q, __fmul_rn(half(row * 16 + 2), (float)m));
}

/* One row's product with one position of x, as the reference's loops take it. */
template <int FMT>
__device__ float plain_row(const BatchParams &p, const uint8_t *w, int row, int pos, float denom)
{
    constexpr int kUnit = BatchFmt<FMT>::kUnit;
    constexpr size_t kSlab = 64 * BatchFmt<FMT>::kUnitBytes;
    const uint8_t *tile = w + (size_t)(row >> 6) * p.units * kSlab;
    const float *x = p.x + (size_t)pos * p.cols;
    float sum = 0.0f;
#pragma unroll 1
    for (int k = 0; k < p.cols; ++k) {
        const float v = p.norm_w ? x[k] / denom * p.norm_w[k] : x[k];
        sum += v * tiled_weight<FMT>(tile + (k / kUnit) * kSlab, row & 63, k % kUnit);
    }
    return sum;
}

__device__ __forceinline__ float lane_of(float v, int) { return v; }
__device__ __forceinline__ float lane_of(const f4_t &v, int e) { return v[e]; }

/* Where N rows (1 or 4) from `r` of a row group and one position go, and what is
 * added to them: read before their segments are summed, so that these reads
 * and the sums' run together. */
template <int N> struct RowsOut {
    float *y;
    const uint8_t *w;
    int row, left; /* rows of the tensor from `row` on */
    bool whole;    /* N of them, and y aligned */
    float add[N];
};

template <int N> __device__ __forceinline__ RowsOut<N> rows_out(const BatchParams &p, int pos, int group, int r)
{
    RowsOut<N> o;
    int job, rg;
    locate_group(p, group, job, rg);
    const BatchJob &j = p.job[job];
    o.row = rg * 16 + r;
    o.left = j.rows - o.row;
    o.w = j.w;
    o.y = j.y + (size_t)pos * j.rows + o.row;
    o.whole = o.left >= N && (N == 1 || ((size_t)j.y | (size_t)j.rows * 4) % 16 == 0);
#pragma unroll
    for (int e = 0; e < N; ++e) o.add[e] = j.add && e < o.left ? j.add[(size_t)pos * j.ldadd + o.row + e] : 0.0f;
    return o;
}

/* What is left of the rows once their segments are summed (v2: the up
 * projection's, with SwiGLU): the norm's division, SwiGLU, the addend, the
 * store. Sums that are not finite, which two limbs of an infinity (inf - inf)
 * never are, are taken again in the plain way: an infinity gives the infinity
 * of its weight's sign. */
template <int FMT, int N, bool NORM, typename T>
__device__ __forceinline__ void finish_rows(const BatchParams &p, int pos, const RowsOut<N> &o, T v, T v2, float denom)
{
    float out[N];
    bool finite = true;
#pragma unroll
    for (int e = 0; e < N; ++e) {
        float a = lane_of(v, e), b = lane_of(v2, e);
        finite = finite && __builtin_isfinite(a) && (!p.swiglu || __builtin_isfinite(b));
        if (NORM) a /= denom;
        if (p.swiglu) a = silu_product(a, NORM ? b / denom : b);
        out[e] = a + o.add[e];
    }
    if (__builtin_expect(!finite, 0)) {
#pragma unroll 1
        for (int e = 0; e < N && e < o.left; ++e) {
            float a = plain_row<FMT>(p, o.w, o.row + e, pos, denom);
            if (p.swiglu) a = silu_product(a, plain_row<FMT>(p, p.job[1].w, o.row + e, pos, denom));
            float add = o.add[0];
#pragma unroll
            for (int i = 1; i < N; ++i) add = e == i ? o.add[i] : add;
            o.y[e] = a + add;
        }
        return;
    }
    if (N == 4 && o.whole) {
        *(f4_t *)o.y = f4_t{out[0], out[1 % N], out[2 % N], out[3 % N]};
        return;
    }
#pragma unroll
    for (int e = 0; e < N; ++e)
        if (e < o.left) o.y[e] = out[e];
}

/* A workgroup stages the activations of a chunk of K (segments [seg0, seg1))
 * for all positions, once; its waves then take the items (R row groups, one
 * segment) of its rows in turn, reading weights one unit ahead. FUSED: the
 * chunk is all of K, the segments' sums meet in LDS and the workgroup writes
 * the rows. DIRECT: a wave takes all segments of a row group and writes its
 * rows (no norm, no SwiGLU) when it has them, while others read weights.
 * CHUNKS: the sums go to memory, [segment][position][row], and
 * reduce_kernel adds them. A row's segments are always added in their
 * order; how many there are depends on the format, K, the launch's rows in all
 * and, up to 8 positions or with a norm or SwiGLU, on those (batch_shape), so a
 * grouped launch may sum in another order than its tensors alone. */
template <int FMT, int NR, int R, int WAVES, bool NORM, int MODE>
__global__ void __launch_bounds__(WAVES * 64) chunk_kernel(BatchParams p)
{
    constexpr bool FUSED = MODE != QMV_BATCH_CHUNKS;
    using B = BatchFmt<FMT>;
    using L = BatchStage<FMT, NR>;
    constexpr int F = L::F, P = L::P, NJ = B::kUnit / 64;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = (int)(blockDim.x >> 6), n = lane & 15, kc = lane >> 4;

    const int chunk = FUSED ? 0 : (int)blockIdx.x / p.chunk_wgs;
    const int g0 = (FUSED ? (int)blockIdx.x : (int)blockIdx.x % p.chunk_wgs) * p.wg_groups;
    const int ng = p.groups - g0 < p.wg_groups ? p.groups - g0 : p.wg_groups;
    const int seg0 = FUSED ? 0 : chunk * p.chunk_segs;
    const int nseg = FUSED ? p.segs : p.segs - seg0 < p.chunk_segs ? p.segs - seg0 : p.chunk_segs;
    const int u0 = segment_begin(p, seg0), nu = segment_begin(p, seg0 + nseg) - u0;
    const size_t tile_bytes = (size_t)p.units * 64 * B::kUnitBytes;

    /* The items of this wave: (ig, is) = row group set and segment. */
    constexpr bool DIRECT = MODE == QMV_BATCH_DIRECT; /* a wave takes all segments of its row groups */
    const int step_g = DIRECT ? nw : nw / nseg, step_s = DIRECT ? 1 : nw % nseg;
    int ig = DIRECT ? wave : wave / nseg, is = DIRECT ? 0 : wave % nseg, u = 0, uend = 0;
    const uint8_t *wp[R];
    int wrow[R];
    const auto open_item = [&]() {
        u = segment_begin(p, seg0 + is);
        uend = segment_begin(p, seg0 + is + 1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int group = g0 + ig * R + r;
            int rg;
            const uint8_t *w0 = group_weights(p, group < p.groups ? group : p.groups - 1, rg);
            wp[r] = w0 + (size_t)(rg >> 2) * tile_bytes;
            wrow[r] = (rg & 3) * 16 + n;
        }
    };
    typename B::W w[R];
    const auto load_w = [&](int unit) {
#pragma unroll
        for (int r = 0; r < R; ++r) B::load(w[r], wp[r] + (size_t)unit * (64 * B::kUnitBytes), wrow[r], kc);
    };
    bool more = ig * R < ng;
    if (more) {
        open_item();
        load_w(u);
    }

    /* Stage the chunk: a wave per unit and round of 4 positions, up to four
     * loads ahead of the first split. */
    const int stages = nu * NR;
    for (int s0 = wave; s0 < stages; s0 += 4 * nw) {
        f4_t v[4][NJ];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int s = s0 + q * nw;
            if (s >= stages) break;
            const int pos = s % NR * 4 + kc, at = pos < p.positions ? pos : p.positions - 1;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int k = (u0 + s / NR) * B::kUnit + 64 * j + 4 * n;
                const bool in = B::kUnit == 256 || k < p.cols; /* whole units of 256, or whole blocks of 32 */
                v[q][j] = in ? *(const f4u_t *)(p.x + (size_t)at * p.cols + k) : f4_t{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int s = s0 + q * nw;
            if (s >= stages) break;
            const int pos = s % NR * 4 + kc, su = s / NR;
            uint8_t *out = lds + su * L::kBytes;
            if (NORM) {
                /* in 64 bits: its error is common to all of a position's rows */
                double ssq = 0.0;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int k = (u0 + su) * B::kUnit + 64 * j + 4 * n;
                    const bool in = B::kUnit == 256 || k < p.cols;
                    const f4_t nw4 = in ? *(const f4u_t *)(p.norm_w + k) : f4_t{0, 0, 0, 0};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ssq = fma((double)v[q][j][e], (double)v[q][j][e], ssq);
                        v[q][j][e] *= nw4[e];
                    }
                }
                ssq += dpp_double<DPP_XOR1>(ssq);
                ssq += dpp_double<DPP_XOR2>(ssq);
                ssq += dpp_double<DPP_HALF_MIRROR>(ssq);
                ssq += dpp_double<DPP_ROR8>(ssq);
                if (n == 0) {
                    *(double *)(out + L::kSsq + 8 * pos) = ssq;
                    if (!FUSED && g0 == 0) p.ssq[(u0 + su) * P + pos] = ssq;
                }
            }
            stage_position<FMT, NR>(out, v[q], pos, n);
        }
    }
    __syncthreads();

    const int arow = F == 1 ? (n >> 3) * P + (n & (P - 1)) : n; /* this lane's row of a fragment */
    /* FUSED: [segment][row group][position][16]; DIRECT: of each wave [segment][position][16] */
    float *part = (float *)(lds + nu * L::kBytes);
    if (DIRECT) part += wave * (nseg * P * 16);
    f4_t y[R][L::kBlocks];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int f = 0; f < L::kBlocks; ++f) y[r][f] = f4_t{0, 0, 0, 0};
    while (more) {
        const uint8_t *stage = lds + (u - u0) * L::kBytes;
        h8_t a[B::kSteps];
        read_fragment<FMT, NR>(a, stage, 0, arow, kc);
        __builtin_amdgcn_sched_barrier(0);
        BatchB<FMT> b[R];
#pragma unroll
        for (int r = 0; r < R; ++r) b[r].decode(w[r], kc);
        const int set = ig, seg = is;
        const bool last = ++u == uend;
        if (last) { /* the next item's first unit */
            is += step_s;
            if (!DIRECT) ig += step_g;
            if (is >= nseg) {
                is -= nseg;
                ig += DIRECT ? step_g : 1;
            }
            more = ig * R < ng;
            if (DIRECT && is) /* the same rows */
                uend = segment_begin(p, is + 1);
            else if (more)
                open_item();
        }
        load_w(more ? u : u - 1); /* past the last: that one again */
        unit_product<FMT, NR, R>(b, a, stage, arow, kc, y);
        if (!last) continue;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int g = set * R + r; /* of the workgroup */
            float *o = DIRECT  ? part + seg * (P * 16) + n
                       : FUSED ? part + ((size_t)seg * p.wg_groups + g) * (P * 16) + n
                             : p.partials + (size_t)(seg0 + seg) * p.positions * p.groups * 16 +
                                   (size_t)(g0 + g) * 16 + n;
            const size_t ld = FUSED ? 16 : (size_t)p.groups * 16;
            const bool real = R == 1 || g < ng;
#pragma unroll
            for (int f = 0; f < L::kBlocks; ++f)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    /* F == 1: lanes 0..31 hold h sums of positions 4 (kc & 1)
                     * + e, lanes 32..63 their l sums */
                    float v = y[r][f][e];
                    if (F == 1) v = fmaf(__shfl_xor(v, 32, 64), 0x1p-12f, v);
                    const int pos = F == 1 ? 4 * (kc & 1) + e : 16 * f + 4 * kc + e;
                    const bool mine = F == 1 ? kc < 2 && pos < P : true;
                    if (real && mine && (FUSED || pos < p.positions)) o[pos * ld] = v;
                }
#pragma unroll
            for (int f = 0; f < L::kBlocks; ++f) y[r][f] = f4_t{0, 0, 0, 0};
        }
        if constexpr (DIRECT) { /* the row group's rows, four a lane */
            if (seg + 1 < nseg) continue;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (int o = lane; o < 4 * p.positions; o += 64) {
                const int pos = o >> 2, q = (o & 3) * 4;
                const float *s = part + pos * 16 + q;
                const f4_t v = nseg == 1 ? f4_t{0, 0, 0, 0} + *(const f4_t *)s : strided_sum<f4_t>(s, P * 16, nseg);
                finish_rows<FMT, 4, false>(p, pos, rows_out<4>(p, pos, g0 + set, q), v, v, 0.0f);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    if constexpr (MODE == QMV_BATCH_FUSED) {
        __syncthreads();
        float *denom = part + (size_t)p.segs * p.wg_groups * (P * 16);
        if (NORM) {
            if ((int)threadIdx.x < P) {
                const double t = strided_sum<double>((const double *)(lds + L::kSsq) + threadIdx.x, L::kBytes / 8, nu);
                denom[threadIdx.x] = sqrtf((float)(t / p.cols + p.norm_eps));
            }
            __syncthreads();
        }
        /* A row a thread, or four where that takes several rounds */
        const int rows = (p.swiglu ? ng / 2 : ng) * 16;
        const size_t stride = (size_t)p.wg_groups * (P * 16);
        const auto finish = [&](auto width, int o) {
            constexpr int N = decltype(width)::value;
            typedef std::conditional_t<N == 4, f4_t, float> T;
            const int pos = o / (rows / N), lr = o % (rows / N) * N, group = p.swiglu ? lr >> 4 << 1 : lr >> 4;
            const float *s = part + (size_t)group * (P * 16) + pos * 16 + (lr & 15);
            const RowsOut<N> out = rows_out<N>(p, pos, g0 + group, lr & 15);
            const T v = strided_sum<T>(s, stride, p.segs);
            finish_rows<FMT, N, NORM>(p, pos, out, v, p.swiglu ? strided_sum<T>(s + P * 16, stride, p.segs) : v,
                                      NORM ? denom[pos] : 0.0f);
        };
        if (rows * p.positions <= 2 * (int)blockDim.x)
            for (int o = threadIdx.x; o < rows * p.positions; o += blockDim.x) finish(std::integral_constant<int, 1>(), o);
        else
            for (int o = threadIdx.x; o < rows / 4 * p.positions; o += blockDim.x) finish(std::integral_constant<int, 4>(), o);
    }
}

/* The segments' sums of one position, four rows a thread (of gate and up:
 * four of each), and the epilogue. Seven waves a SIMD (72 registers, 5 of them
 * spilled) stream the partial sums best: time over 28 launches of 4 to 32
 * positions to that of the kernel without the check for infinities, seven waves
 * 0.987, eight (11 spilled) 0.995, six 0.991, five (what the compiler takes by
 * itself, 84 registers) 0.988; 151936 x 2048 Q6_K at 32 positions 101.7, 105.0,
 * 103.9, 103.8 us. */
template <int FMT, bool NORM>
__global__ void __launch_bounds__(256, 7) reduce_kernel(BatchParams p, int ssq_ld)
{
    const int pos = blockIdx.y, lr = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4, g = lr >> 4;
    __shared__ float denom;
    if (NORM && threadIdx.x < 64) { /* a lane per unit: 74 units by one thread were 1.7 us that the others waited */
        double t = 0.0;
        for (int u = threadIdx.x; u < p.units; u += 64) t += p.ssq[(size_t)u * ssq_ld + pos];
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) t += __shfl_xor(t, m, 64);
        if (threadIdx.x == 0) denom = sqrtf((float)(t / p.cols + p.norm_eps));
    }
    const int group = p.swiglu ? 2 * g : g;
    const bool in = group < p.groups;
    const size_t stride = (size_t)p.positions * p.groups * 16;
    const float *s = p.partials + (size_t)pos * p.groups * 16 + (size_t)(in ? group : 0) * 16 + (lr & 15);
    f4_t v = strided_sum<f4_t>(s, stride, p.segs), v2 = {0, 0, 0, 0};
    if (p.swiglu) v2 = strided_sum<f4_t>(s + 16, stride, p.segs);
    const RowsOut<4> out = rows_out<4>(p, pos, in ? group : 0, lr & 15);
    if (NORM) __syncthreads();
    if (in) finish_rows<FMT, 4, NORM>(p, pos, out, v, v2, NORM ? denom : 0.0f);
}

template <int FMT, int NR, int R, int WAVES, bool NORM, int MODE>
static hipError_t launch_chunks(const BatchParams &p, int waves, hipStream_t s)
{
    using L = BatchStage<FMT, NR>;
    constexpr bool FUSED = MODE != QMV_BATCH_CHUNKS;
    if (MODE == QMV_BATCH_DIRECT && (R != 1 || p.swiglu)) return hipErrorInvalidValue;
    if (waves > WAVES || p.wg_groups % R || p.wg_groups < 1 || p.segs < 1 || p.segs > p.units) return hipErrorInvalidValue;
    const int most = (p.units + p.segs - 1) / p.segs * p.chunk_segs; /* units of a chunk, at most */
    const size_t units = FUSED ? p.units : most < p.units ? most : p.units;
    const size_t sums = MODE == QMV_BATCH_DIRECT  ? (size_t)waves * p.segs * L::P * 16
                        : MODE == QMV_BATCH_FUSED ? (size_t)p.segs * p.wg_groups * L::P * 16 + L::P
                                                  : 0;
    const size_t bytes = units * L::kBytes + sums * sizeof(float);
    if (bytes > 160 * 1024) return hipErrorInvalidValue;
    const int chunks = FUSED ? 1 : (p.segs + p.chunk_segs - 1) / p.chunk_segs;
    chunk_kernel<FMT, NR, R, WAVES, NORM, MODE><<<chunks * p.chunk_wgs, waves * 64, bytes, s>>>(p);
    if (!FUSED) {
        const int rows = (p.swiglu ? p.groups / 2 : p.groups) * 16;
        reduce_kernel<FMT, NORM><<<dim3((rows + 1023) / 1024, p.positions), 256, 0, s>>>(p, L::P);
    }
    return hipGetLastError();
}

template <int FMT, int NR, int R, int WAVES>
static hipError_t launch_shape(const BatchParams &p, int mode, int waves, hipStream_t s)
{
    if (mode == QMV_BATCH_DIRECT) {
        if constexpr (NR >= 4 && R == 1)
            if (!p.norm_w) return launch_chunks<FMT, NR, R, WAVES, false, QMV_BATCH_DIRECT>(p, waves, s);
        return hipErrorInvalidValue;
    }
    if (mode == QMV_BATCH_FUSED)
        return p.norm_w ? launch_chunks<FMT, NR, R, WAVES, true, QMV_BATCH_FUSED>(p, waves, s)
                        : launch_chunks<FMT, NR, R, WAVES, false, QMV_BATCH_FUSED>(p, waves, s);
    if constexpr (WAVES <= 12) /* what batch_shape cuts chunks for */
        return p.norm_w ? launch_chunks<FMT, NR, R, WAVES, true, QMV_BATCH_CHUNKS>(p, waves, s)
                        : launch_chunks<FMT, NR, R, WAVES, false, QMV_BATCH_CHUNKS>(p, waves, s);
    return hipErrorInvalidValue;
}

template <int FMT>
static hipError_t launch_fmt(const BatchParams &p, int nr, int r, int mode, int waves, hipStream_t s)
{
#define QMV_BATCH(NR, R, W) \
    if (nr == NR && r == R && waves <= W) return launch_shape<FMT, NR, R, W>(p, mode, waves, s);
    QMV_BATCH(1, 1, 12)
    QMV_BATCH(2, 1, 12)
    if constexpr (FMT == QMV_FMT_Q6_K) {
        QMV_BATCH(4, 1, 8)
        QMV_BATCH(8, 1, 8)
    } else {
        QMV_BATCH(1, 1, 16)
        QMV_BATCH(2, 1, 16)
        QMV_BATCH(4, 1, 12)
        QMV_BATCH(8, 1, 12)
    }
    if constexpr (FMT == QMV_FMT_Q4_K || FMT == QMV_FMT_Q8_0) {
        QMV_BATCH(4, 2, 8)
    }
#undef QMV_BATCH
    return hipErrorInvalidValue;
}

size_t batch_stage_bytes(int fmt, int nr)
{
#define QMV_BYTES(F)                                \
    (nr == 1   ? BatchStage<F, 1>::kBytes           \
     : nr == 2 ? BatchStage<F, 2>::kBytes           \
     : nr == 4 ? BatchStage<F, 4>::kBytes           \
               : BatchStage<F, 8>::kBytes)
    return fmt == QMV_FMT_Q8_0   ? QMV_BYTES(QMV_FMT_Q8_0)
           : fmt == QMV_FMT_Q5_0 ? QMV_BYTES(QMV_FMT_Q5_0)
           : fmt == QMV_FMT_Q4_K ? QMV_BYTES(QMV_FMT_Q4_K)
                                 : QMV_BYTES(QMV_FMT_Q6_K);
#undef QMV_BYTES
}

hipError_t launch_batch(int fmt, const BatchParams &p, int nr, int r, int mode, int waves, hipStream_t s)
{
    switch (fmt) {
    case QMV_FMT_Q8_0: return launch_fmt<QMV_FMT_Q8_0>(p, nr, r, mode, waves, s);
    case QMV_FMT_Q5_0: return launch_fmt<QMV_FMT_Q5_0>(p, nr, r, mode, waves, s);
    case QMV_FMT_Q4_K: return launch_fmt<QMV_FMT_Q4_K>(p, nr, r, mode, waves, s);
    case QMV_FMT_Q6_K: return launch_fmt<QMV_FMT_Q6_K>(p, nr, r, mode, waves, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace qmv
