// qg_prefill_wide.hip -- batched prefill of long prompts: up to kWideMax
// tokens through a layer at a time (qg_model_prefill, include/qgmodel.h).
//
// The same computation as qg_prefill.hip (model.rs:361-365 token by token;
// here every projection is one GEMM on the matrix cores over exact f16
// products), arranged for chunks of more than 64 tokens:
//
//   * wide_planes_k: one workgroup per token holds the token's whole input
//     vector x (the RMSNorm of the residual stream, the attention output, or
//     silu(g) * u), so the norm is complete; every 256-element group g of x has
//     its own power-of-two scale 2^e_g (the group's largest magnitude into
//     [512, 1024)), as in qg_prefill.hip, and xs = x 2^e_g goes out as two f16
//     pieces (hi + lo, 22 significant bits of everything down to 2^-12 of the
//     group's maximum, and an absolute 2^-35 of it below) in the layout of the
//     GEMM's LDS buffers, with the sums of xs per 32 elements and 2^-e_g;
//   * wide_gemm_k: tiles of 128 tokens x 256 rows,
//     y = sum over blocks of 2^-e_g (d D - dmin Dm): D the block's exact
//     integer products accumulated by v_mfma_f32_16x16x32_f16, Dm its min terms
//     by v_mfma_f32_16x16x16_f16;
//   * wide_attention_k: causal attention, 64 tokens of a head per workgroup,
//     on v_mfma_f32_16x16x4f32 (f32 products and sums).
//
// MFMA operand layouts: qg_prefill.hip.
#include <hip/hip_runtime.h>

#include <cmath>

#include "qg_common.h"

namespace qgw {

using qg::T_Q4_K;
using qg::T_Q5_K;
using qg::T_Q6_K;
using qg::T_Q8_0;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
// Q6_K's row groups are 210 bytes a block: their pieces and scales start at any
// even address
typedef uint32_t v4u_2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32_2 __attribute__((aligned(2)));

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u(h2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ float h2f(uint32_t h16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(h16 & 0xFFFFu)); }
__device__ __forceinline__ h2 splat(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ uint32_t fma2(uint32_t a, h2 b, h2 c) { return as_u(__builtin_elementwise_fma(as_h2(a), b, c)); }

// bytes i and i + 2 of c as the f16 pair 1024 + byte
__device__ __forceinline__ uint32_t mag02(uint32_t c) { return __builtin_amdgcn_perm(0x64646464u, c, 0x04020400u); }
__device__ __forceinline__ uint32_t mag13(uint32_t c) { return __builtin_amdgcn_perm(0x64646464u, c, 0x04030401u); }
// 1024 + the byte of v selected by sel's low bytes, twice, less 1024
__device__ __forceinline__ h2 byte_pair(uint32_t v, uint32_t sel)
{
    return as_h2(__builtin_amdgcn_perm(0x64646464u, v, sel)) - splat(1024.f);
}

// ------------------------------------------------------------ weight types
//
// A chunk is 128 consecutive elements of a row (half a K-quant block, four
// Q8_0 blocks), four MFMA steps m = 0..3 of 32 elements.  Lane kq = lane / 16
// of a row loads the chunk's weights from the repacked layout (repack_k) with
// 16-byte loads and supplies 8 elements per step; which 8 is the type's choice
// (its 16-byte slot slot0(kq) ^ mx(m) of the chunk), the x operand is read
// from the same slot.  Inside a slot the elements go in the order 0 2 1 3 4 6 5
// 7: two codes that sit two bytes apart in a word become an f16 pair with one
// and-or.
//   load(W, cs, v, c, L, ni): chunk c of the row whose group starts v bytes
//     after W; the part of the address that depends on the chunk only is in
//     the scalar W (cs = c), or in the lane's (cs = 0): rows of one group
//     start at different chunks;
//   half(h, half): what a half's scales need of the block header;
//   scale(x, n, kq): of the low (n = 0: steps 0, 1) or high codes;
//   decode(raw, sc, m, kq, b): the step's B operands (NB of them; Q6_K's
//     second is the part of sc (q - 32) that f16 cannot hold).
template <uint32_t T> struct Wt;

// A multiply-add pair: code -> scaled code, see decode
struct Sc2 {
    h2 s, o;
};

// A K-quant header (d, dmin and the 12 bytes of 6-bit scales and mins) as the
// lane needs it: the scales of the two halves' sub-blocks (a byte each), the
// mins of the lane's half (kq >> 1) and d | dmin << 16
struct KHead {
    uint32_t lo, hi, m4, dd;
};
__device__ __forceinline__ KHead khead(v4u h, uint32_t mhalf)
{
    const uint32_t ml = h.z & 0x3F3F3F3Fu, mh = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
    return KHead{h.y & 0x3F3F3F3Fu, (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u), mhalf ? mh : ml, h.x};
}
// low codes: fma(1024 + q, s, -1024 s); high: fma(1024 + 16 q, s / 16, -64 s),
// s the scale of sub-block 2 (kq >> 1) (+ 1 for the high codes) of the half
__device__ __forceinline__ Sc2 kscale(uint32_t sc4, uint32_t n, uint32_t kq)
{
    const h2 a = byte_pair(sc4, 0x04000400u + n * 0x00010001u + (kq >> 1) * 0x00020002u);
    return n ? Sc2{a * splat(0.0625f), a * splat(-64.f)} : Sc2{a, a * splat(-1024.f)};
}
// B operand of the min terms of a whole block (v_mfma_f32_16x16x16_f16, K slot
// 2 j + p = piece p of the sum of sub-block j): lane kq holds the mins of
// sub-blocks 2 kq, 2 kq + 1, each twice.  Of one half (four sub-blocks, K slots
// 0..7): the lanes kq >= 2 hold zeros.
__device__ __forceinline__ uint2 kmins(uint32_t m4, uint32_t kq)
{
    const uint32_t sel = 0x04000400u + (kq & 1u) * 0x00020002u;
    return make_uint2(as_u(byte_pair(m4, sel)), as_u(byte_pair(m4, sel + 0x00010001u)));
}

template <> struct Wt<T_Q4_K> {
    static constexpr int NB = 1;
    static constexpr bool KQ = true;               // header with scales and mins
    struct Raw { uint4 v; };
    __device__ static uint32_t slot0(uint32_t kq) { return ((kq >> 1) << 3) | ((kq & 1u) << 1); }
    __device__ static constexpr uint32_t mx(uint32_t m) { return ((m >> 1) << 2) | (m & 1u); }
    __device__ static Raw load(const uint8_t *W, uint32_t cs, uint32_t v, uint32_t c, uint32_t kq, uint32_t ni)
    {
        return Raw{*(const uint4 *)(W + (size_t)cs * 16u + (v + 8u * ni + kq * ni * 16u + c * 16u))};
    }
    __device__ static void decode(const Raw &w, const Sc2 &s, uint32_t m, uint32_t, uint4 (&b)[NB])
    {
        const uint32_t c0 = (m & 1u) ? w.v.z : w.v.x, c1 = (m & 1u) ? w.v.w : w.v.y;
        const uint32_t M = 0x64006400u, k = m < 2u ? 0x000F000Fu : 0x00F000F0u;
        b[0] = make_uint4(fma2((c0 & k) | M, s.s, s.o), fma2(((c0 >> 8) & k) | M, s.s, s.o),
                          fma2((c1 & k) | M, s.s, s.o), fma2(((c1 >> 8) & k) | M, s.s, s.o));
    }
};

template <> struct Wt<T_Q5_K> {
    static constexpr int NB = 1;
    static constexpr bool KQ = true;
    struct Raw { uint4 v; uint32_t w; };           // w: the fifth bits of the lane's 32 codes
    __device__ static uint32_t slot0(uint32_t kq) { return Wt<T_Q4_K>::slot0(kq); }
    __device__ static constexpr uint32_t mx(uint32_t m) { return Wt<T_Q4_K>::mx(m); }
    __device__ static Raw load(const uint8_t *W, uint32_t cs, uint32_t v, uint32_t c, uint32_t kq, uint32_t ni)
    {
        return Raw{*(const uint4 *)(W + (size_t)cs * 32u + (v + 4u * ni + (kq & 1u) * ni * 16u + (kq >> 1) * 16u + c * 32u)),
                   *(const uint32_t *)(W + (size_t)cs * 16u + (v + 36u * ni + (kq >> 1) * 8u + (kq & 1u) * 4u + c * 16u))};
    }
    __device__ static void decode(const Raw &w, const Sc2 &s, uint32_t m, uint32_t, uint4 (&b)[NB])
    {
        // word t' of the piece: bit 8 bb + 2 t' + n of w is the fifth bit of
        // byte bb's low (n = 0) or high (n = 1) code; moved to bit 8 bb + 4
        // (low) or 8 bb + 8 (high)
        const uint32_t M = 0x64006400u;
        const uint32_t c0 = (m & 1u) ? w.v.z : w.v.x, c1 = (m & 1u) ? w.v.w : w.v.y;
        auto sh = [](uint32_t x, int l) { return l >= 0 ? x << l : x >> -l; };
        const uint32_t k = m < 2u ? 0x000F000Fu : 0x00F000F0u, f = m < 2u ? 0x00100010u : 0x01000100u;
        const int l0 = (m < 2u ? 4 : 7) - 4 * (int)(m & 1u), l1 = l0 - 2;
        b[0] = make_uint4(fma2((sh(w.w, l0) & f) | ((c0 & k) | M), s.s, s.o),
                          fma2((sh(w.w, l0 - 8) & f) | (((c0 >> 8) & k) | M), s.s, s.o),
                          fma2((sh(w.w, l1) & f) | ((c1 & k) | M), s.s, s.o),
                          fma2((sh(w.w, l1 - 8) & f) | (((c1 >> 8) & k) | M), s.s, s.o));
    }
};

// Q6_K: value d sc (q - 32).  B1 = f16(sc (q - 32)) and B2 = what B1 leaves
// (0 or +-1: |sc (q - 32)| <= 4096), both exact f16.  All four products of the
// pieces are formed (down of Llama-3-8B over 1001 tokens about 350 us, 310
// without the low piece's with B2): without that one a product was off by up
// to 2^-22 of it, as much again as x's own split.
template <> struct Wt<T_Q6_K> {
    static constexpr int NB = 2;
    static constexpr bool KQ = false;
    struct Raw { v4u l, h; uint32_t sc; uint32_t d; };
    __device__ static uint32_t slot0(uint32_t kq) { return ((kq >> 1) << 2) | ((kq & 1u) << 1); }
    __device__ static constexpr uint32_t mx(uint32_t m) { return ((m >> 1) << 3) | (m & 1u); }
    __device__ static Raw load(const uint8_t *W, uint32_t cs, uint32_t v, uint32_t c, uint32_t kq, uint32_t ni)
    {
        const uint8_t *p = W + (size_t)cs * 32u;
        const uint32_t o = v + c * 32u + (kq & 1u) * 16u;
        return Raw{*(const v4u_2 *)(p + (o + (kq >> 1) * ni * 16u)), *(const v4u_2 *)(p + (o + 32u * ni)),
                   *(const u32_2 *)(W + (size_t)cs * 8u + (v + 48u * ni + (kq & 1u) * 4u + c * 8u)),
                   (uint32_t)*(const uint16_t *)(W + (size_t)(cs >> 1) * 2u + (v + 52u * ni + (c >> 1) * 2u))};
    }
    __device__ static Sc2 scale(const Raw &w, uint32_t n, uint32_t kq)
    {
        // bytes kq >> 1 and + 2: sub-blocks kq >> 1 and + 2 of the half
        const _Float16 a = (_Float16)(int16_t)(int8_t)((w.sc >> (8u * (kq >> 1) + 16u * n)) & 0xFFu);
        return Sc2{h2{a, a}, h2{a, a}};
    }
    __device__ static void decode(const Raw &w, const Sc2 &s, uint32_t m, uint32_t kq, uint4 (&b)[NB])
    {
        const uint32_t M = 0x64006400u;
        const uint32_t c[2] = {(m & 1u) ? w.l.z : w.l.x, (m & 1u) ? w.l.w : w.l.y};
        const uint32_t g[2] = {(m & 1u) ? w.h.z : w.h.x, (m & 1u) ? w.h.w : w.h.y};
        uint32_t r1[4], r2[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            // the two high bits of the low codes (bits 2 (kq >> 1) of every
            // byte of g) and of the high codes (4 bits further)
            const uint32_t z = g[i] >> (2u * (kq >> 1)), z0 = z << 4, z1 = z >> 4, c1 = c[i] >> 8;
            h2 q[2];
            if (m < 2u) {
                const uint32_t k = 0x000F000Fu, f = 0x00300030u;
                q[0] = as_h2((z0 & f) | ((c[i] & k) | M)) + splat(-1056.f);
                q[1] = as_h2((z1 & f) | ((c1 & k) | M)) + splat(-1056.f);
            } else {
                const uint32_t k = 0x00F000F0u, f = 0x03000300u;
                q[0] = __builtin_elementwise_fma(as_h2((z0 & f) | ((c[i] & k) | M)), splat(0.0625f), splat(-96.f));
                q[1] = __builtin_elementwise_fma(as_h2((z1 & f) | ((c1 & k) | M)), splat(0.0625f), splat(-96.f));
            }
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const h2 p = q[e] * s.s;
                r1[2 * i + e] = as_u(p);
                r2[2 * i + e] = as_u(__builtin_elementwise_fma(q[e], s.s, -p));
            }
        }
        b[0] = make_uint4(r1[0], r1[1], r1[2], r1[3]);
        b[1] = make_uint4(r2[0], r2[1], r2[2], r2[3]);
    }
};

// Q8_0: value d q, one d per 32 elements; step m is block m of the chunk.
template <> struct Wt<T_Q8_0> {
    static constexpr int NB = 1;
    static constexpr bool KQ = false;
    struct Raw { uint2 q[4]; uint32_t d0, d1; };
    __device__ static uint32_t slot0(uint32_t kq) { return kq; }
    __device__ static constexpr uint32_t mx(uint32_t m) { return m << 2; }
    __device__ static Raw load(const uint8_t *W, uint32_t cs, uint32_t v, uint32_t c, uint32_t kq, uint32_t ni)
    {
        Raw r;
        const uint8_t *p = W + (size_t)cs * 32u;
        const uint32_t o = v + c * 32u + (kq >> 1) * ni * 16u + (kq & 1u) * 8u;
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) r.q[i] = *(const uint2 *)(p + (o + (i & 1u) * 32u * ni + (i >> 1) * 16u));
        const uint8_t *d = W + (size_t)cs * 8u + (v + 64u * ni + c * 8u);
        r.d0 = *(const uint32_t *)d;
        r.d1 = *(const uint32_t *)(d + 4u);
        return r;
    }
    __device__ static Sc2 scale(const Raw &, uint32_t, uint32_t) { return Sc2{}; }
    __device__ static float dscale(const Raw &w, uint32_t m) { return h2f((m < 2u ? w.d0 : w.d1) >> (16u * (m & 1u))); }
    __device__ static void decode(const Raw &w, const Sc2 &, uint32_t m, uint32_t, uint4 (&b)[NB])
    {
        const uint32_t c0 = w.q[m].x ^ 0x80808080u, c1 = w.q[m].y ^ 0x80808080u;
        const h2 o = splat(-1152.f);
        b[0] = make_uint4(as_u(as_h2(mag02(c0)) + o), as_u(as_h2(mag13(c0)) + o), as_u(as_h2(mag02(c1)) + o),
                          as_u(as_h2(mag13(c1)) + o));
    }
};

// ------------------------------------------------------------------ GEMM

constexpr uint32_t kR = 2;                         // 16-row tiles per wave
constexpr uint32_t kTok = 128;                     // tokens per workgroup tile: two x images of 64
constexpr uint32_t kRowsWG = 8u * 16u * kR;        // rows per workgroup tile
constexpr uint32_t kImg = 2u * 64u * 256u;         // bytes of a chunk's x image of 64 tokens
constexpr uint32_t kBufX = 2u * kImg;              // ... of a workgroup's two halves
// A chunk's record of 64 tokens: the sums of its four sub-blocks, then 2^-e_g
constexpr uint32_t kRec = 5u * 64u;                // dwords
constexpr uint32_t kBufS = 2u * kRec * 4u;         // bytes of a workgroup's two halves
constexpr uint32_t kLds = 2u * kBufX + 4u * kBufS; // two x buffers, four of the records

__device__ __forceinline__ void dma16(const void *gp, uint32_t lds_addr)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gp), "{m0}"(lds_addr) : "memory");
}

__device__ __forceinline__ void dma4(const void *gp, uint32_t lds_addr)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(gp), "{m0}"(lds_addr) : "memory");
}

// The registers of x are (re)defined here: no computation on them moves above.
template <class X> __device__ __forceinline__ void pin(X &x)
{
    static_assert(sizeof(X) % 4 == 0, "whole dwords");
    uint32_t w[sizeof(X) / 4];
    __builtin_memcpy(w, &x, sizeof(X));
#pragma unroll
    for (uint32_t i = 0; i < sizeof(X) / 4; i++) asm volatile("" : "+v"(w[i]));
    __builtin_memcpy(&x, w, sizeof(X));
}

struct Job {
    const uint8_t *w;
    float *y;
    uint32_t rows, tiles;
    uint32_t g, ni;
    uint64_t gb;
};
struct Jobs {
    Job j[3];
};

// One tile of 128 tokens x 256 rows of a K slice: eight waves of 32 rows, each
// over all 128 tokens, so that a weight is decoded once per workgroup.  Chunks
// of 128 elements of x (64 KB) are copied straight to LDS, two buffers in
// turn; a wave's weights go to registers one chunk ahead.
//
// What bounds it: two waves a SIMD that issue or wait together.  A chunk of
// Q4_K or Q5_K is 136 MFMAs of 16 cycles per wave, two waves to a SIMD (4352
// cycles), and 72 LDS reads; gate and up of Llama-3-8B over 1001 tokens in Q5_K
// (526-555 us, 3.5 tiles a CU in 4 rounds) take about 8500 cycles a chunk.  Of
// its wave cycles 30 % issue, 32 % wait to issue and 38 % wait for data and at
// the barriers; the matrix cores are busy in 45 % of all SIMD cycles (Q6_K down:
// 68 %), the LDS in 25 % of the CUs'.  Without the copies and weight
// loads a chunk took 30 % less, without the decode 25 % less.  Measured against
// it, with three products of Q6_K (Q5_K gate and up / Q6_K down, us): this shape
// 610 / 327; wave tiles of 64 tokens x 48 rows 666
// / 437, of 64 x 64 1221 / 914 (registers spill); four waves of 128 x 64, one
// to a SIMD, 820 / 410; copies and loads all requested at the start of a
// chunk instead of between its steps 734 / 590 (64 x 48: the memory pipe's
// queue fills and the waves wait to issue).  64-token chunks through
// qg_prefill.hip's kernel, 16 of them: 1120 / 800.
//
// ONE: one row per row group (blocks end with every second chunk for the whole
// wave, and a block is a group of x); otherwise rows may start in the middle of
// a block and every chunk ends D.  At the end of D the token's 2^-e_g comes
// from the record, one multiply per element more than a scale common to the
// row would take: nothing to see of it in the time (1001 tokens of two
// Llama-3-8B layers, Q5_K and Q6_K: 2.73 ms with the common scale, 2.70 so),
// and without it an outlier takes the bits of the whole row.
//
// Blocks go to XCDs so that the token tiles of a row tile run beside each
// other on one XCD: its L2 then holds the row tile's open weight lines.
template <uint32_t T, bool ONE>
__global__ void __launch_bounds__(512) wide_gemm_k(Jobs jobs, uint32_t row_tiles, uint32_t tok_tiles, uint32_t slices,
                                                   uint32_t nchunk, uint32_t cps, const uint8_t *__restrict__ xp,
                                                   const uint32_t *__restrict__ rec, uint32_t ntok, uint32_t ldy,
                                                   uint64_t sstride)
{
    using P = Wt<T>;
    constexpr bool Q8 = T == T_Q8_0;
    constexpr uint32_t BLK = ONE && !Q8 ? 2u : 1u;         // chunks per flush of D
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t j8 = blockIdx.x >> 3, tt0 = j8 % tok_tiles;
    uint32_t tile = (j8 / tok_tiles) * 8u + (blockIdx.x & 7u);
    if (tile >= row_tiles * slices) return;
    const uint32_t slice = tile / row_tiles;
    tile -= slice * row_tiles;
    Job J = jobs.j[0];
    if (tile >= J.tiles) {
        tile -= J.tiles;
        J = jobs.j[1];
        if (tile >= J.tiles) {
            tile -= J.tiles;
            J = jobs.j[2];
        }
    }
    const uint32_t k0 = slice * cps, k1 = min(nchunk, k0 + cps);
    const uint32_t lane = threadIdx.x & 63u, kq = lane >> 4, c16 = lane & 15u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t row0 = tile * kRowsWG + wave * 16u * kR, tg0 = 2u * tt0;
    // byte offset of each row's group, and the row's first chunk in it
    uint32_t off[kR], f0[kR];
#pragma unroll
    for (uint32_t i = 0; i < kR; i++) {
        const uint32_t r = min(row0 + 16u * i + c16, J.rows - 1u);
        off[i] = (ONE ? r : r / J.g) * (uint32_t)J.gb;
        f0[i] = ONE ? 0u : (r % J.g) * nchunk;
    }
    // part `part` (of 4) of the copies of chunk c into buffer c' & 1 (c' = c, or
    // the chunk after the slice's last, whose buffers no one reads): wave w
    // copies 1 KB blocks 8 w .. 8 w + 7 of the chunk's 64 KB and the sums of one
    // sub-block of a half; waves 0 and 4 the halves' scales
    auto stage = [&](uint32_t c, uint32_t cd, uint32_t part) {
        const uint32_t b0 = lds0 + (cd & 1u) * kBufX;
        const size_t img = (size_t)(tg0 + (wave >> 2)) * nchunk + c;
        const uint8_t *src = xp + img * kImg + (wave & 3u) * 8192u;
#pragma unroll
        for (uint32_t v = 2u * part; v < 2u * part + 2u; v++)
            dma16(src + v * 1024u + 16u * lane, b0 + wave * 8192u + v * 1024u);
        if (part == 0u) {
            const uint32_t *r = rec + img * kRec + lane;
            const uint32_t rl = lds0 + 2u * kBufX + (cd & 3u) * kBufS + (wave >> 2) * 4u * kRec;
            if (P::KQ) dma4(r + (wave & 3u) * 64u, rl + (wave & 3u) * 256u);
            if ((wave & 3u) == 0u) dma4(r + 256u, rl + 1024u);
        }
    };
    typename P::Raw cw[kR], nw[kR];
    v4u nh[kR];                                                   // K-quants: the next block's headers
    KHead hd[kR];
    auto load = [&](uint32_t c, uint32_t i) {
        nw[i] = P::load(J.w, ONE ? c : 0u, off[i], ONE ? 0u : f0[i] + c, kq, J.ni);
    };
    auto load_head = [&](uint32_t c) {
#pragma unroll
        for (uint32_t i = 0; i < kR; i++)
            nh[i] = *(const v4u *)(J.w + (ONE ? (size_t)(c >> 1) * 16u : 0u) + (off[i] + (ONE ? 0u : ((f0[i] + c) >> 1) * 16u)));
    };
    v4f acc[kR][8], D[kR][8];
#pragma unroll
    for (uint32_t i = 0; i < kR; i++)
#pragma unroll
        for (uint32_t t = 0; t < 8; t++) acc[i][t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t part = 0; part < 4; part++) stage(k0, k0, part);
#pragma unroll
    for (uint32_t i = 0; i < kR; i++) load(k0, i);
    if constexpr (P::KQ) load_head(k0);
    const uint32_t slot = P::slot0(kq) ^ c16;                       // this lane's slot position at step 0
    for (uint32_t cb = k0; cb < k1; cb += BLK) {
#pragma unroll
        for (uint32_t hc = 0; hc < BLK; hc++) {
            const uint32_t c = cb + hc, cn = min(c + 1u, k1 - 1u);
            __builtin_amdgcn_s_waitcnt(0x0F70);                     // vmcnt(0): this chunk's copies and weights
            __syncthreads();
#pragma unroll
            for (uint32_t i = 0; i < kR; i++) {
                cw[i] = nw[i];
                pin(cw[i]);
                if constexpr (P::KQ) {
                    if (hc == 0) {
                        pin(nh[i]);
                        hd[i] = khead(nh[i], ONE ? kq >> 1 : (f0[i] + c) & 1u);
                    }
                }
            }
            // the next chunk's copies and weights are requested between this
            // one's steps (all at once they fill the memory pipe's queue and
            // the waves wait to issue them)
            auto request = [&](uint32_t m) {
                stage(cn, c + 1u, m);
                if (m < kR) load(cn, m);
                if constexpr (P::KQ) {
                    if (hc + 1u == BLK && m == 3u) load_head(cn);
                }
            };
            const uint8_t *xb = lds + (c & 1u) * kBufX + c16 * 256u;
            Sc2 sc[kR];
#pragma unroll
            for (uint32_t m = 0; m < 4; m++) {
                // steps stay apart: moved together, their operands pass the 256 registers
                if constexpr (!Q8) __builtin_amdgcn_sched_barrier(0);
                request(m);
                const uint8_t *xa = xb + ((slot ^ P::mx(m)) << 4);
                uint4 b[kR][P::NB];
#pragma unroll
                for (uint32_t i = 0; i < kR; i++) {
                    if ((m & 1u) == 0u) {
                        if constexpr (P::KQ)
                            sc[i] = kscale((ONE ? hc != 0u : ((f0[i] + c) & 1u) != 0u) ? hd[i].hi : hd[i].lo, m >> 1, kq);
                        else
                            sc[i] = P::scale(cw[i], m >> 1, kq);
                    }
                    P::decode(cw[i], sc[i], m, kq, b[i]);
                }
                const bool first = hc == 0 && m == 0;               // D starts at zero
#pragma unroll
                for (uint32_t t = 0; t < 8; t++) {
                    const h8 a0 = *(const h8 *)(xa + (t & 3u) * 4096u + (t >> 2) * 32768u), a1 = *(const h8 *)(xa + (t & 3u) * 4096u + (t >> 2) * 32768u + 16384u);
                    if constexpr (Q8) {                             // a block per step: d times its products
                        v4f q[kR];
#pragma unroll
                        for (uint32_t i = 0; i < kR; i++)
                            q[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, __builtin_bit_cast(h8, b[i][0]),
                                                                          v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (uint32_t i = 0; i < kR; i++)
                            q[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, __builtin_bit_cast(h8, b[i][0]), q[i], 0, 0, 0);
#pragma unroll
                        for (uint32_t i = 0; i < kR; i++) {
                            const float d = Wt<T_Q8_0>::dscale(cw[i], m);
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                D[i][t][e] = first ? d * q[i][e] : __builtin_fmaf(d, q[i][e], D[i][t][e]);
                        }
                        continue;
                    }
#pragma unroll
                    for (uint32_t i = 0; i < kR; i++)
                        D[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, __builtin_bit_cast(h8, b[i][0]),
                                                                         first ? v4f{0.f, 0.f, 0.f, 0.f} : D[i][t], 0, 0, 0);
                    if constexpr (P::NB == 2)
#pragma unroll
                        for (uint32_t i = 0; i < kR; i++)
                            D[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, __builtin_bit_cast(h8, b[i][1]), D[i][t], 0, 0, 0);
#pragma unroll
                    for (uint32_t n = 0; n < (uint32_t)P::NB; n++)
#pragma unroll
                        for (uint32_t i = 0; i < kR; i++)
                            D[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, __builtin_bit_cast(h8, b[i][n]), D[i][t], 0, 0, 0);
                }
            }
            if (hc + 1u == BLK) {
                // the end of D: acc += 2^-e_g (d D - dmin Dm), Dm the min terms
                const uint8_t *sb = lds + 2u * kBufX;
                float d[kR], dm[kR];
                uint2 bm[kR];
#pragma unroll
                for (uint32_t i = 0; i < kR; i++) {
                    if constexpr (P::KQ) {
                        d[i] = h2f(hd[i].dd);
                        dm[i] = -h2f(hd[i].dd >> 16);
                        bm[i] = kmins(hd[i].m4, kq);
                        if (BLK == 1u && kq >= 2u) bm[i] = make_uint2(0u, 0u);
                    } else if constexpr (!Q8) {
                        d[i] = h2f(cw[i].d);
                    }
                }
#pragma unroll
                for (uint32_t t = 0; t < 8; t++) {
                    const uint32_t to = (t & 3u) * 64u + (t >> 2) * 4u * kRec;
                    const v4f sg = *(const v4f *)(sb + (c & 3u) * kBufS + 1024u + to + 16u * kq);
                    h4 sa = {};
                    if constexpr (P::KQ) {
                        // lane kq: the sums of sub-blocks 2 kq, 2 kq + 1 of the block (kq >> 1: its
                        // chunk), or of the chunk's 2 (kq & 1), + 1
                        const uint32_t cs = BLK == 2u ? cb + (kq >> 1) : c;
                        const uint8_t *s = sb + (cs & 3u) * kBufS + (kq & 1u) * 512u + to + 4u * c16;
                        sa = __builtin_bit_cast(h4, make_uint2(*(const uint32_t *)s, *(const uint32_t *)(s + 256u)));
                    }
#pragma unroll
                    for (uint32_t i = 0; i < kR; i++) {
                        if constexpr (P::KQ) {
                            const v4f Dm = __builtin_amdgcn_mfma_f32_16x16x16f16(sa, __builtin_bit_cast(h4, bm[i]),
                                                                                 v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[i][t][e] = __builtin_fmaf(sg[e], __builtin_fmaf(d[i], D[i][t][e], dm[i] * Dm[e]),
                                                              acc[i][t][e]);
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[i][t][e] = __builtin_fmaf(Q8 ? sg[e] : d[i] * sg[e], D[i][t][e], acc[i][t][e]);
                        }
                    }
                }
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                             // the last chunk's surplus copies
    float *y = J.y + (size_t)slice * sstride;
    const uint32_t tb = tg0 * 64u;
#pragma unroll
    for (uint32_t t = 0; t < 8; t++)
#pragma unroll
        for (uint32_t e = 0; e < 4; e++) {
            const uint32_t tok = tb + 16u * t + 4u * kq + e;
            if (tok < ntok)
#pragma unroll
                for (uint32_t i = 0; i < kR; i++) {
                    const uint32_t r = row0 + 16u * i + c16;
                    if (r < J.rows) y[(size_t)tok * ldy + r] = acc[i][t][e];
                }
        }
}

// ---------------------------------------------------------------- planes

// sum of v over a workgroup of 512 threads (every thread the same value); red: 8 floats
__device__ __forceinline__ float block_sum(float v, float *red)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int i = 1; i < 8; i++) r += red[i];
    return r;
}

__device__ __forceinline__ float silu1(float x)
{
    // math.rs:137-146's two branches
    const float e = expf(x >= 0.0f ? -x : x);
    return x >= 0.0f ? x / (1.0f + e) : x * e / (1.0f + e);
}

// elements e0 .. e0 + 7 of the sum of ns slices, in slice order
__device__ __forceinline__ void sum8(const float *p, uint32_t ns, uint64_t sstride, float (&v)[8])
{
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    for (uint32_t s = 1; s < ns; s++) {
        const float4 c = *(const float4 *)(p + s * sstride), d = *(const float4 *)(p + s * sstride + 4);
        v[0] += c.x; v[1] += c.y; v[2] += c.z; v[3] += c.w;
        v[4] += d.x; v[5] += d.y; v[6] += d.z; v[7] += d.w;
    }
}

// The input vector x of token blockIdx.x -- mode 0: a; mode 1: rmsnorm(a + b)
// * nw, with a + b stored to sum_out when given; mode 2: silu(a) * b -- as the
// GEMM's x images: xs = x 2^e_g (the largest magnitude of the 256-element group
// g into [512, 1024)) in two f16 pieces, slot j (8 elements) of a chunk at
// position j ^ (t & 15) of the token's 256 bytes, the sums of xs per 32
// elements (two f16 pieces) and 2^-e_g (NaN when the group's x is not finite),
// of each of the group's chunks.  32 threads hold a group.  a, b: sums of na,
// nb slices.  PM: 8-element pieces per thread (n <= 4096 PM); instances of 1, 2,
// 5 and 8, so rows of 14336 (3.5 pieces) and 18944 (4.6) share one.
template <int PM>
__global__ void __launch_bounds__(512) wide_planes_k(const float *__restrict__ a, uint32_t na, const float *__restrict__ b,
                                                     uint32_t nb, uint64_t sstride, float *__restrict__ sum_out,
                                                     const float *__restrict__ nw, uint32_t n, uint32_t lda,
                                                     uint32_t mode, float eps, uint8_t *__restrict__ xp,
                                                     uint32_t *__restrict__ rec)
{
    __shared__ float red[8];
    const uint32_t t = blockIdx.x, tid = threadIdx.x, np = n / 8u, nchunk = n / 128u;
    const float *at = a + (size_t)t * lda, *bt = b ? b + (size_t)t * lda : nullptr;
    float v[PM][8];
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < PM; p++) {
        const uint32_t j = tid + 512u * (uint32_t)p;
#pragma unroll
        for (int e = 0; e < 8; e++) v[p][e] = 0.f;
        if (j >= np) continue;
        sum8(at + 8u * j, na, sstride, v[p]);
        if (bt) {
            float u[8];
            sum8(bt + 8u * j, nb, sstride, u);
#pragma unroll
            for (int e = 0; e < 8; e++) v[p][e] = mode == 2u ? silu1(v[p][e]) * u[e] : v[p][e] + u[e];
        }
        if (mode == 1u) {
            if (sum_out) {
                float *so = sum_out + (size_t)t * lda + 8u * j;
                *(float4 *)so = make_float4(v[p][0], v[p][1], v[p][2], v[p][3]);
                *(float4 *)(so + 4) = make_float4(v[p][4], v[p][5], v[p][6], v[p][7]);
            }
#pragma unroll
            for (int e = 0; e < 8; e++) ss += v[p][e] * v[p][e];
        }
    }
    if (mode == 1u) {
        // math.rs:237-257: x * (1 / rms) * w
        const float r = 1.0f / sqrtf(block_sum(ss, red) / (float)n + eps);
#pragma unroll
        for (int p = 0; p < PM; p++) {
            const uint32_t j = tid + 512u * (uint32_t)p;
            if (j < np) {
                const float4 w0 = *(const float4 *)(nw + 8u * j), w1 = *(const float4 *)(nw + 8u * j + 4u);
                const float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
                for (int e = 0; e < 8; e++) v[p][e] = v[p][e] * r * w[e];
            }
        }
    }
    uint8_t *xt = xp + (size_t)(t >> 6) * nchunk * kImg + (t & 63u) * 256u;
    uint32_t *rt = rec + (size_t)(t >> 6) * nchunk * kRec + (t & 63u);
#pragma unroll
    for (int p = 0; p < PM; p++) {
        const uint32_t j = tid + 512u * (uint32_t)p;
        const bool live = j < np;
        float mx = 0.f;
        bool bad = false;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            bad |= !__builtin_isfinite(v[p][e]);
            mx = fmaxf(mx, fabsf(v[p][e]));
        }
        // a NaN passes fmaxf by: it goes through the maximum as an infinity
        if (bad) mx = INFINITY;
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        bad = !__builtin_isfinite(mx);
        int E = 0;
        (void)frexpf(mx, &E);
        const int e2 = bad || mx == 0.f ? 0 : min(max(10 - E, -126), 126);
        const float sc = ldexpf(1.0f, e2);
        _Float16 h[8], l[8];
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x = v[p][e] * sc;
            h[e] = (_Float16)x;
            l[e] = (_Float16)(x - (float)h[e]);
            v[p][e] = x;
        }
        s = ((v[p][0] + v[p][1]) + (v[p][2] + v[p][3])) + ((v[p][4] + v[p][5]) + (v[p][6] + v[p][7]));
        s += __shfl_xor(s, 1, 64);
        s += __shfl_xor(s, 2, 64);
        if (!live) continue;
        const h8 hh = {h[0], h[2], h[1], h[3], h[4], h[6], h[5], h[7]};
        const h8 ll = {l[0], l[2], l[1], l[3], l[4], l[6], l[5], l[7]};
        uint8_t *d = xt + (size_t)(j >> 4) * kImg + (((j & 15u) ^ (t & 15u)) << 4);
        *(h8 *)d = hh;
        *(h8 *)(d + 16384u) = ll;
        if ((j & 3u) == 0u) {
            const _Float16 sh = (_Float16)s, sl = (_Float16)(s - (float)sh);
            rt[(j >> 4) * kRec + ((j >> 2) & 3u) * 64u] = as_u(h2{sh, sl});
        }
        if ((j & 15u) == 0u)
            rt[(j >> 4) * kRec + 256u] = __builtin_bit_cast(uint32_t, bad ? __builtin_nanf("") : ldexpf(1.0f, -e2));
    }
}

// ------------------------------------------------------------- attention

// Causal attention of query head blockIdx.x for the chunk's tokens t0 .. t0 +
// 63, token t over cache slots 0 .. slot0 + t (attention.rs:93-121,
// math.rs:63-70 / 104-118).
// Four waves of 16 tokens; positions in tiles of 32 rows of K and V, staged in
// LDS for the four and requested one tile ahead.  A wave computes S = Q K^T
// (2 x hd / 4 v_mfma_f32_16x16x4f32, Q in registers), its running maximum per
// token, P = exp(S - M) through its own LDS rows into the A layout, and O = O
// exp(M' - M) + P V (8 x hd / 16 MFMAs).  f32 products and sums throughout;
// bound by the f32 matrix rate (32 cycles per MFMA): three workgroups per CU
// overlap the softmax and the barriers of one with the MFMAs of the others.
// The MFMAs take their four-element k steps from four consecutive elements
// per lane (element 16 k + 4 g + j of lane group g at step 4 k + j), so K, Q
// and P are read 16 bytes at a time.
constexpr uint32_t kAttTok = 64, kAttPos = 32;
__host__ __device__ constexpr uint32_t att_lds(uint32_t hd)
{
    return (2u * kAttPos * (hd + 4u) + 4u * 16u * (kAttPos + 4u)) * 4u;
}

template <int CTRL> __device__ __forceinline__ float row_dpp(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// over the 16 lanes of a row, to all of them (quad_perm, row_half_mirror, row_mirror)
__device__ __forceinline__ float row_max(float v)
{
    v = fmaxf(v, row_dpp<0xB1>(v));
    v = fmaxf(v, row_dpp<0x4E>(v));
    v = fmaxf(v, row_dpp<0x141>(v));
    return fmaxf(v, row_dpp<0x140>(v));
}
__device__ __forceinline__ float row_sum(float v)
{
    v += row_dpp<0xB1>(v);
    v += row_dpp<0x4E>(v);
    v += row_dpp<0x141>(v);
    return v + row_dpp<0x140>(v);
}

template <uint32_t HD>
__global__ void __launch_bounds__(256) wide_attention_k(const float *__restrict__ qkv, uint32_t ldq,
                                                        const float *__restrict__ kc, const float *__restrict__ vc,
                                                        float *__restrict__ out, uint32_t kv_dim, uint32_t n_rep,
                                                        float scale, uint32_t slot0, uint32_t ntok)
{
    constexpr uint32_t LK = HD + 4u, LP = kAttPos + 4u, KS = HD / 16u, NT = HD / 16u;
    constexpr uint32_t LD = kAttPos * HD / 4u / 256u;      // float4 of K (and of V) per thread and tile
    extern __shared__ __align__(16) float att[];
    float *ks = att, *vs = ks + kAttPos * LK;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, c = lane & 15u, g = lane >> 4;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *ps = vs + kAttPos * LK + w * 16u * LP;
    // token tiles: the later half from the last on, then the earlier half from
    // the first on, so that a CU's second workgroup is the shorter the longer
    // its first (1001 tokens of 32 heads: 130 us; all from the last on 139;
    // eight waves, four of them for the second half of tiles of 64 positions,
    // 154)
    const uint32_t ny = gridDim.y, by = blockIdx.y, late = (ny + 1u) / 2u;
    const uint32_t h = blockIdx.x, t0 = (by < late ? ny - 1u - by : by - late) * kAttTok, kvh = (h / n_rep) * HD;
    const uint32_t tw = t0 + 16u * w;                      // this wave's first token
    const uint32_t npos = slot0 + min(ntok, t0 + kAttTok); // positions any token of the workgroup sees
    // A of S: q[token c][16 k + 4 g + j] (tokens past the chunk: the last one's, never stored)
    v4f qa[KS];
    {
        const float *q = qkv + (size_t)min(tw + c, ntok - 1u) * ldq + (size_t)h * HD + 4u * g;
#pragma unroll
        for (uint32_t k = 0; k < KS; k++) qa[k] = *(const v4f *)(q + 16u * k);
    }
    v4f nk[LD], nv[LD];
    auto request = [&](uint32_t base) {
#pragma unroll
        for (uint32_t i = 0; i < LD; i++) {
            const uint32_t x = tid + 256u * i, p = x / (HD / 4u), d4 = x % (HD / 4u);
            const size_t o = (size_t)min(base + p, npos - 1u) * kv_dim + kvh + 4u * d4;
            nk[i] = *(const v4f *)(kc + o);
            nv[i] = *(const v4f *)(vc + o);
        }
    };
    float m[4], l[4];                                      // of tokens 4 g + i (l: this lane's positions only)
    v4f o[NT];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) { m[i] = -INFINITY; l[i] = 0.f; }
#pragma unroll
    for (uint32_t b = 0; b < NT; b++) o[b] = v4f{0.f, 0.f, 0.f, 0.f};
    request(0);
    for (uint32_t base = 0; base < npos; base += kAttPos) {
        __syncthreads();                                   // the previous tile's readers are done
#pragma unroll
        for (uint32_t i = 0; i < LD; i++) {
            const uint32_t x = tid + 256u * i, p = x / (HD / 4u), d4 = x % (HD / 4u);
            *(v4f *)(ks + p * LK + 4u * d4) = nk[i];
            *(v4f *)(vs + p * LK + 4u * d4) = nv[i];
        }
        __syncthreads();
        if (base + kAttPos < npos) request(base + kAttPos);
        if (base > slot0 + tw + 15u || tw >= ntok) continue;   // no token of this wave sees the tile
        v4f s[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (uint32_t k = 0; k < KS; k++) {
            const v4f b0 = *(const v4f *)(ks + c * LK + 16u * k + 4u * g);
            const v4f b1 = *(const v4f *)(ks + (16u + c) * LK + 16u * k + 4u * g);
            s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].x, b0.x, s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].x, b1.x, s[1], 0, 0, 0);
            s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].y, b0.y, s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].y, b1.y, s[1], 0, 0, 0);
            s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].z, b0.z, s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].z, b1.z, s[1], 0, 0, 0);
            s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].w, b0.w, s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[k].w, b1.w, s[1], 0, 0, 0);
        }
        // masked (after the token's own slot): -inf.  Position 0 is in the
        // first tile, so every maximum is finite from there on.
        float al[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const uint32_t last = slot0 + tw + 4u * g + i;
            const float s0 = base + c <= last ? s[0][i] * scale : -INFINITY;
            const float s1 = base + 16u + c <= last ? s[1][i] * scale : -INFINITY;
            const float mn = fmaxf(m[i], row_max(fmaxf(s0, s1)));
            al[i] = expf(m[i] - mn);
            const float p0 = expf(s0 - mn), p1 = expf(s1 - mn);
            m[i] = mn;
            l[i] = l[i] * al[i] + (p0 + p1);
            ps[(4u * g + i) * LP + c] = p0;
            ps[(4u * g + i) * LP + 16u + c] = p1;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t b = 0; b < NT; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) o[b][i] *= al[i];
#pragma unroll
        for (uint32_t k = 0; k < kAttPos / 16u; k++) {
            const v4f pa = *(const v4f *)(ps + c * LP + 16u * k + 4u * g);
            const float *vr = vs + (16u * k + 4u * g) * LK + c;
#pragma unroll
            for (uint32_t b = 0; b < NT; b++) o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa.x, vr[16u * b], o[b], 0, 0, 0);
#pragma unroll
            for (uint32_t b = 0; b < NT; b++) o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa.y, vr[LK + 16u * b], o[b], 0, 0, 0);
#pragma unroll
            for (uint32_t b = 0; b < NT; b++) o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa.z, vr[2u * LK + 16u * b], o[b], 0, 0, 0);
#pragma unroll
            for (uint32_t b = 0; b < NT; b++) o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa.w, vr[3u * LK + 16u * b], o[b], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const uint32_t t = tw + 4u * g + i;
        const float inv = 1.0f / row_sum(l[i]);
        if (t < ntok) {
            float *dst = out + ((size_t)t * gridDim.x + h) * HD + c;
#pragma unroll
            for (uint32_t b = 0; b < NT; b++) dst[16u * b] = o[b][i] * inv;
        }
    }
}

}  // namespace qgw

namespace qg {

bool wide_mat_ok(const PfMat &m, size_t cols)
{
    if (!prefill_type_supported(m.type) || !m.rp || m.rows == 0 || m.rows > 0xFFFFFFFFull || cols % 128 != 0 ||
        cols > kWideCols || m.g == 0 || m.rows % m.g != 0 || m.ni == 0 || m.gb == 0 ||
        m.rows / m.g > 0xFFFFFFFFull / m.gb)                             // 32-bit byte offsets
        return false;
    // a row group's whole blocks: rows of one group start at multiples of a chunk
    return m.g > 1 || m.type == T_Q8_0 || cols % 256 == 0;
}

uint32_t wide_tiles(size_t rows) { return (uint32_t)((rows + qgw::kRowsWG - 1) / qgw::kRowsWG); }

static uint32_t wide_slice_len(uint32_t nchunk, uint32_t slices)
{
    const uint32_t nb = nchunk / 2u, b = (nb + slices - 1u) / slices;
    return nchunk % 2u ? (nchunk + slices - 1u) / slices : 2u * b;
}

// One workgroup per CU at a time: rounds of n_cu workgroups, each as long as
// its slice's blocks plus what a slice costs beside them (filling the
// pipeline, writing 128 KB of products and reading them back: about 4
// blocks' time).
uint32_t wide_split(uint32_t row_tiles, uint32_t tok_tiles, size_t cols, int n_cu)
{
    const uint32_t nchunk = (uint32_t)(cols / 128u), tiles = row_tiles * tok_tiles, ncu = n_cu > 0 ? (uint32_t)n_cu : 256u;
    uint32_t best = 1, cost = 0xFFFFFFFFu;
    for (uint32_t s = 1; s <= kWideSlices; s++) {
        const uint32_t len = wide_slice_len(nchunk, s);
        if (len == 0 || (nchunk + len - 1u) / len != s) continue;         // no empty slice
        const uint32_t c = ((tiles * s + ncu - 1u) / ncu) * (len + 8u);
        if (c < cost) {
            cost = c;
            best = s;
        }
    }
    return best;
}

template <uint32_t T, bool ONE>
static void wide_launch(const qgw::Jobs &j, uint32_t tiles, uint32_t tok_tiles, uint32_t slices, uint32_t nchunk,
                        const uint8_t *xp, const uint32_t *rec, uint32_t ntok, uint32_t ldy, size_t sstride,
                        hipStream_t st)
{
    const uint32_t cps = wide_slice_len(nchunk, slices);
    const dim3 grid((tiles * slices + 7u) / 8u * 8u * tok_tiles);
    hipLaunchKernelGGL((qgw::wide_gemm_k<T, ONE>), grid, dim3(512), qgw::kLds, st, j, tiles, tok_tiles, slices, nchunk,
                       cps, xp, rec, ntok, ldy, (uint64_t)sstride);
}

int launch_wide_gemm(const PfMat *mats, int n_mats, size_t cols, const uint8_t *xp, const uint32_t *rec,
                     uint32_t ntok, uint32_t ldy, uint32_t slices, size_t sstride, ihipStream_t *stream)
{
    if (ntok == 0) return 0;
    if (n_mats < 1 || n_mats > 3 || ntok > kWideMax || slices < 1 || slices > kWideSlices) return -1;
    qgw::Jobs j = {};
    uint32_t tiles = 0;
    for (int i = 0; i < n_mats; i++) {
        const PfMat &m = mats[i];
        if (!wide_mat_ok(m, cols) || m.type != mats[0].type || (m.g == 1) != (mats[0].g == 1)) return -1;
        j.j[i] = qgw::Job{m.w, m.y, (uint32_t)m.rows, wide_tiles(m.rows), m.g, m.ni, (uint64_t)m.gb};
        tiles += j.j[i].tiles;
    }
    const uint32_t nchunk = (uint32_t)(cols / 128), tt = (ntok + qgw::kTok - 1) / qgw::kTok;
    const uint32_t len = wide_slice_len(nchunk, slices);
    if (len == 0 || (nchunk + len - 1u) / len != slices) return -1;
    hipStream_t st = (hipStream_t)stream;
    const bool one = mats[0].g == 1;
    switch (mats[0].type) {
    case T_Q4_K:
        if (one) wide_launch<T_Q4_K, true>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        else wide_launch<T_Q4_K, false>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        break;
    case T_Q5_K:
        if (one) wide_launch<T_Q5_K, true>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        else wide_launch<T_Q5_K, false>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        break;
    case T_Q6_K:
        if (one) wide_launch<T_Q6_K, true>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        else wide_launch<T_Q6_K, false>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        break;
    case T_Q8_0:
        if (!one) return -1;
        wide_launch<T_Q8_0, true>(j, tiles, tt, slices, nchunk, xp, rec, ntok, ldy, sstride, st);
        break;
    default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_wide_planes(const float *a, uint32_t na, const float *b, uint32_t nb, size_t sstride, float *sum_out,
                       const float *nw, size_t n, size_t lda, int mode, float eps, uint8_t *xp, uint32_t *rec,
                       uint32_t ntok, ihipStream_t *stream)
{
    if (ntok == 0) return 0;
    if (n % 128 != 0 || n == 0 || n > kWideCols || ntok > kWideMax || na < 1 || (b && nb < 1) || (mode == 2 && !b) ||
        (mode == 1 && !nw) || lda % 4 != 0 || sstride % 4 != 0 || ((uintptr_t)a & 15u) || ((uintptr_t)b & 15u) ||
        ((uintptr_t)sum_out & 15u) || ((uintptr_t)nw & 15u))
        return -1;
    hipStream_t st = (hipStream_t)stream;
    const uint32_t pm = (uint32_t)((n / 8 + 511) / 512);
    auto go = [&](auto fn) {
        hipLaunchKernelGGL(fn, dim3(ntok), dim3(512), 0, st, a, na, b, nb, (uint64_t)sstride, sum_out, nw, (uint32_t)n,
                           (uint32_t)lda, (uint32_t)mode, eps, xp, rec);
    };
    if (pm <= 1) go(qgw::wide_planes_k<1>);
    else if (pm <= 2) go(qgw::wide_planes_k<2>);
    else if (pm <= 5) go(qgw::wide_planes_k<5>);
    else go(qgw::wide_planes_k<8>);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_wide_attention(const float *qkv, uint32_t ldq, const float *kc, const float *vc, float *out,
                          uint32_t n_heads, uint32_t hd, uint32_t kv_dim, uint32_t n_rep, float scale, uint32_t slot0,
                          uint32_t ntok, ihipStream_t *stream)
{
    if (ntok == 0) return 0;
    if (ntok > kWideMax || n_rep == 0 || n_heads % n_rep != 0 || ldq % 4 != 0 || kv_dim % 4 != 0 ||
        ((uintptr_t)qkv & 15u) || ((uintptr_t)kc & 15u) || ((uintptr_t)vc & 15u) ||
        (uint64_t)n_heads * hd > ldq || (uint64_t)(n_heads / n_rep) * hd > kv_dim)
        return -1;
    const dim3 grid(n_heads, (ntok + qgw::kAttTok - 1) / qgw::kAttTok), block(256);
    hipStream_t st = (hipStream_t)stream;
    switch (hd) {
    case 64:
        hipLaunchKernelGGL(qgw::wide_attention_k<64>, grid, block, qgw::att_lds(64), st, qkv, ldq, kc, vc, out, kv_dim,
                           n_rep, scale, slot0, ntok);
        break;
    case 128:
        hipLaunchKernelGGL(qgw::wide_attention_k<128>, grid, block, qgw::att_lds(128), st, qkv, ldq, kc, vc, out,
                           kv_dim, n_rep, scale, slot0, ntok);
        break;
    case 256:
        hipLaunchKernelGGL(qgw::wide_attention_k<256>, grid, block, qgw::att_lds(256), st, qkv, ldq, kc, vc, out,
                           kv_dim, n_rep, scale, slot0, ntok);
        break;
    default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace qg
