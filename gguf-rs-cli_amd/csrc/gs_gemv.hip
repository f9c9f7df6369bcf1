// gs_gemv.hip -- gfx950 quantized projection that produces the logits (the
// reference's output projection, src/model/llama.rs:333-334 on the GPU path,
// :405-407 on the CPU path), for Q4_0, Q4_1, Q8_0, Q3_K, Q4_K, Q5_K and Q6_K
// weights: out[b][r] = sum_c W[r][c] x[b][c] for B vectors.
//
// Two kernels, for up to 4 vectors and for more, on the matrix cores, for
// every type and row length.  The stored integers of a weight are exact in
// f16 (at most 8 bits; Q3_K's scaled by its 6-bit sub-block scale: at most
// 9), and x is split into three f16 parts that hold its 24 bits, whose
// products the MFMA adds in f32.  What is left for the vector units is the
// unpacking of the integers (about 1.3 instructions per weight for the 4-bit
// types) and, per sub-block, row and vector, an addition and a multiply-add.
//
// Why: the weights have to be read once per call, and that read is the bound
// for a few vectors.  Byte-to-float conversions and FMAs took 3.2-3.4
// instructions per weight, as long as the read itself, for one vector, and a
// pass over the weights for each further one.  Measured (MI355X, us per call;
// before: one pass of the vector units per vector):
//   Q4_K 152064 x 3584:  1 vector 61 -> 54 (5.7 TB/s), 16: 980 -> 93,
//                        32: 1975 -> 151
//   Q6_K 152064 x 3584:  1 vector 70 -> 72 (6.2 TB/s), 16: 1157 -> 148,
//                        32: 2330 -> 235
//   Q5_K 152064 x 3584:  1 vector 70 -> 71; 32000 x 8192: 121 -> 38
//   Q8_0 32000 x 4096:   4 vectors 96 -> 26
// With x in two parts (23 bits at best) instead of three and their products
// in one sum: 50, 78 and 116 us for Q4_K, 70, 109 and 162 for Q6_K, 64 for
// Q5_K.
//
// Error against 64-bit sums (2-norm, relative; x normal, channels of unequal
// size; 1024 to 8192 columns, 1 to 32 vectors, means of 4 to 8 runs), before
// -> now:
//   Q4_0 2.0-2.3e-7 -> 0.7-1.0e-7     Q4_K 1.4-1.5e-7 -> 0.9-1.3e-7
//   Q4_1 1.3-1.8e-7 -> 1.3e-7         Q5_K 1.3-1.5e-7 -> 0.9-1.3e-7
//   Q8_0 1.7-2.4e-7 -> 0.8-1.1e-7     Q6_K 2.1-2.2e-7 -> 0.9-1.2e-7
//   Q3_K 1.9-2.0e-7 -> 0.8-1.1e-7
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>
#include <new>

#include "../../include/gs_gemv.h"
#include "../../include/gs_sampler.h"

namespace gs {

constexpr int kMaxCols = 16384;
constexpr int kPair = 256;              // columns of a record (eight K steps of 32)

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float h2f(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }
__device__ __forceinline__ h2_t as_h2(uint32_t w) { return __builtin_bit_cast(h2_t, w); }
__device__ __forceinline__ h2_t splat(float f) { return h2_t{(_Float16)f, (_Float16)f}; }
__device__ __forceinline__ h8_t cat(h2_t a, h2_t b, h2_t c, h2_t d) { return h8_t{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y}; }
__device__ __forceinline__ h4_t cat(h2_t a, h2_t b) { return h4_t{a.x, a.y, b.x, b.y}; }
__device__ __forceinline__ float ub(uint32_t w, int t) { return (float)((w >> (8 * t)) & 0xffu); }

// The records are read through an opaque scalar address in the global address
// space: one scalar base per record and 32-bit lane offsets (a generic one
// would make flat loads, whose waits are for everything).  Non-temporal: each
// byte is used once, and kept out of the way of what is not (Q4_K 152064 x
// 3584, one vector: 59 us against 62).
#define GS_GLOBAL __attribute__((address_space(1)))
typedef const GS_GLOBAL uint8_t *gptr;
__device__ __forceinline__ gptr opaque(const uint8_t *p)
{
    uint64_t a = (uint64_t)p;
    asm volatile("" : "+s"(a));
    return (gptr)a;
}
template <class T> __device__ __forceinline__ T ld(gptr p, uint32_t off)
{
    return __builtin_nontemporal_load((const GS_GLOBAL T *)(p + off));
}

// Integers in 16-bit halves to f16: 0x6400 | n is 1024 + n for n < 1024.
// n0: n in the low bits of the halves; n4: 16 n in bits 4 and up (a nibble in
// place, not shifted down): (1024 + 16 n) / 16 = 64 + n, exact in one fma.
constexpr uint32_t kMagic = 0x64006400u;
// A constant that the compiler keeps in a scalar (vector) register: with
// literals (w & mask) | c takes two instructions, the three-operand form has
// none.  (No instruction in the asm: the compiler does not see the hazards
// between one and the MFMAs around it.)
__device__ __forceinline__ uint32_t sreg(uint32_t c)
{
    uint32_t r;
    asm("" : "=s"(r) : "0"(c));
    return r;
}
__device__ __forceinline__ uint32_t vreg(uint32_t c)
{
    uint32_t r;
    asm("" : "=v"(r) : "0"(c));
    return r;
}
__device__ __forceinline__ uint32_t and_or(uint32_t w, uint32_t mask, uint32_t c)
{
    uint32_t d = (w & sreg(mask)) | c;
    asm("" : "+v"(d));          // (two in a row stay two: not two ands and a three-way or)
    return d;
}
__device__ __forceinline__ h2_t n0(uint32_t w, float off) { return as_h2(w) - splat(1024.0f + off); }
__device__ __forceinline__ h2_t n4(uint32_t w, float off)
{
    return __builtin_elementwise_fma(as_h2(w), splat(0.0625f), splat(-64.0f - off));
}
__device__ __forceinline__ h2_t u0(uint32_t w, float off) { return n0(and_or(w, 0x000F000Fu, vreg(kMagic)), off); }
__device__ __forceinline__ h2_t u4(uint32_t w, float off) { return n4(and_or(w, 0x00F000F0u, vreg(kMagic)), off); }

// ------------------------------------------------------- operand layouts ---
// v_mfma_f32_16x16x32_f16, lane L = 16 g + n: operand A holds row n, k = 8 g
// .. 8 g + 7 (x); operand B column n, the same k (weight row n of the tile);
// D column n, rows 4 g .. 4 g + 3.  With the weights as B, everything of a
// weight row (bits, scales, sums) sits in the lanes with that n.
__device__ __forceinline__ f4_t mfma(h8_t a, h8_t b, f4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
constexpr f4_t kZero = {0.0f, 0.0f, 0.0f, 0.0f};

// ------------------------------------------------------------- formats -----
// A record holds 256 columns of 16 rows, in the order the lanes read them:
// 16-byte pieces for all 64 lanes first (lane L at 16 L), then what is per
// row.  Records of a tile follow each other, so a wave reads one run of
// memory.  Each format has
//   kRec   bytes of a record;
//   kSplit a lane's columns of K step ks: 32 ks + 4 g .. + 3 and + 16 (true)
//          or 32 ks + 8 g .. + 7;
//   kSwap  within four columns the unpacked order is 0, 2, 1, 3 (bytes 0 and
//          2 of a word, then 1 and 3);
//   kHalf  a scale for each 16 columns (a lane's first four of a step, and the
//          other four), so a sum for each;
//   kRecScale a factor of the whole record, rec();
//   kMin   a term min_scale() * (min_frag() . the sums of x over 32 columns),
//          min_frag() with the factor of the sums' parts (low()) where that
//          is exact (kMinLow);
//   Item, load(); frag(): the operand of a step; sub(): its scale (its half's);
//   put(): a lane's part of a record from the 256 (or 8 x 32) GGUF blocks of
//          its row.

// A row's blocks from a record on: b, bb bytes each, n of them left (0 bytes
// past the row's end).
struct Src {
    const uint8_t *b;
    int bb, n;
    __device__ uint32_t at(int j, int i) const { return j < n ? b[(size_t)j * bb + i] : 0u; }
    __device__ uint32_t word(int j, int i) const   // four bytes, no alignment
    {
        return at(j, i) | at(j, i + 1) << 8 | at(j, i + 2) << 16 | at(j, i + 3) << 24;
    }
    __device__ uint32_t half(int j, int i) const { return at(j, i) | at(j, i + 1) << 8; }
};

// x's parts b and c carry this factor (below); of its sums' parts, group g of
// an operand's lanes holds part g.
constexpr float kLow = 2048.0f;
__device__ __forceinline__ float low() { return (threadIdx.x & 63) < 16 ? 1.0f : 1.0f / kLow; }

// Bytes 2 i, 2 i + 1 of w as integers less off.
__device__ __forceinline__ h2_t two(uint32_t w, int i, float off)
{
    h2_t d = as_h2(__builtin_amdgcn_perm(kMagic, w, i ? 0x07030702u : 0x07010700u)) - splat(1024.0f + off);
    asm("" : "+v"(d));          // (one packed subtraction, also where the halves are used apart)
    return d;
}

// Q4_0 (src/tensor/dequant.rs:26-41) w = (q - 8) d; Q4_1 (:42-54) w = q d + m;
// byte l of a block's 16 holds weight l (low nibble) and l + 16 (high).
template <bool Q41> struct Q4Fmt {
    static constexpr int kRec = 2048 + 256 + (Q41 ? 256 : 0), kBlock = Q41 ? 20 : 18, kCols = 32;
    static constexpr bool kSplit = true, kSwap = true, kHalf = false, kRecScale = false, kMin = Q41, kMinLow = false;
    struct Item { u4_t q[2], d, m; };
    static __device__ __forceinline__ void load(Item &it, gptr r, uint32_t lane)
    {
        it.q[0] = ld<u4_t>(r, 16 * lane);
        it.q[1] = ld<u4_t>(r, 1024 + 16 * lane);
        it.d = ld<u4_t>(r, 2048 + 16 * (lane & 15));
        if (Q41) it.m = ld<u4_t>(r, 2304 + 16 * (lane & 15));
    }
    static __device__ __forceinline__ h8_t frag(const Item &it, int ks)
    {
        constexpr float off = Q41 ? 0.0f : 8.0f;
        const uint32_t w = it.q[ks >> 2][ks & 3], h = w >> 8;
        return cat(u0(w, off), u0(h, off), u4(w, off), u4(h, off));
    }
    static __device__ __forceinline__ float sub(const Item &it, int ks, int) { return h2f(it.d[ks >> 1] >> (16 * (ks & 1))); }
    static __device__ __forceinline__ float rec(const Item &) { return 1.0f; }
    static __device__ __forceinline__ h8_t min_frag(const Item &it) { return __builtin_bit_cast(h8_t, it.m); }
    static __device__ __forceinline__ float min_scale(const Item &) { return 64.0f; }
    static __device__ void put(uint8_t *r, const Src &s, int lane)
    {
        const int g = lane >> 4, n = lane & 15, o = Q41 ? 4 : 2;
        for (int ks = 0; ks < 8; ks++)
            reinterpret_cast<uint32_t *>(r + 1024 * (ks >> 2) + 16 * lane)[ks & 3] = s.word(ks, o + 4 * g);
        for (int k = 0; k < 2; k++) {
            const int ks = 2 * g + k;
            reinterpret_cast<uint16_t *>(r + 2048 + 16 * n)[ks] = (uint16_t)s.half(ks, 0);
            if (Q41) reinterpret_cast<uint16_t *>(r + 2304 + 16 * n)[ks] = (uint16_t)s.half(ks, 2);
        }
    }
};

// Q8_0: w = q d, int8 q, stored as q + 128.
struct Q8Fmt {
    static constexpr int kRec = 4096 + 256, kBlock = 34, kCols = 32;
    static constexpr bool kSplit = false, kSwap = false, kHalf = false, kRecScale = false, kMin = false, kMinLow = false;
    struct Item { u4_t q[4], d; };
    static __device__ __forceinline__ void load(Item &it, gptr r, uint32_t lane)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) it.q[i] = ld<u4_t>(r, 1024 * i + 16 * lane);
        it.d = ld<u4_t>(r, 4096 + 16 * (lane & 15));
    }
    static __device__ __forceinline__ h8_t frag(const Item &it, int ks)
    {
        const uint32_t w0 = it.q[ks >> 1][2 * (ks & 1)], w1 = it.q[ks >> 1][2 * (ks & 1) + 1];
        return cat(two(w0, 0, 128.0f), two(w0, 1, 128.0f), two(w1, 0, 128.0f), two(w1, 1, 128.0f));
    }
    static __device__ __forceinline__ float sub(const Item &it, int ks, int) { return h2f(it.d[ks >> 1] >> (16 * (ks & 1))); }
    static __device__ __forceinline__ float rec(const Item &) { return 1.0f; }
    static __device__ void put(uint8_t *r, const Src &s, int lane)
    {
        const int g = lane >> 4, n = lane & 15;
        for (int ks = 0; ks < 8; ks++)
            for (int k = 0; k < 2; k++)
                reinterpret_cast<uint32_t *>(r + 1024 * (ks >> 1) + 16 * lane)[2 * (ks & 1) + k] =
                    s.word(ks, 2 + 8 * g + 4 * k) ^ 0x80808080u;
        for (int k = 0; k < 2; k++)
            reinterpret_cast<uint16_t *>(r + 4096 + 16 * n)[2 * g + k] = (uint16_t)s.half(2 * g + k, 0);
    }
};

// get_scale_min_k4 (src/tensor/dequant.rs:141-148): the 6-bit scale (min) of
// sub-block j from the 12 packed bytes at `o`.
__device__ inline uint32_t k4_scale(const Src &s, int o, int j)
{
    return j < 4 ? s.at(0, o + j) & 63u : (s.at(0, o + j + 4) & 15u) | (s.at(0, o + j - 4) >> 6) << 4;
}
__device__ inline uint32_t k4_min(const Src &s, int o, int j)
{
    return j < 4 ? s.at(0, o + j + 4) & 63u : s.at(0, o + j + 4) >> 4 | (s.at(0, o + j) >> 6) << 4;
}

// Q4_K / Q5_K (src/tensor/dequant.rs:149-196): w = (d sc_i) q - dmin m_i per
// sub-block i of 32; byte 32 s + l of qs holds weight 64 s + l (low nibble,
// i = 2 s) and 64 s + 32 + l (high, i = 2 s + 1); Q5_K adds bit i of qh[l]
// as 16.  A lane's bits of qh for two steps s are one word: bits b, b + 16
// (low nibbles) and b + 1, b + 17 (high), b = 8 (s & 1) + 2 q, for the bytes
// 0 and 2 of the lane's first word (q = 0), 1 and 3 of it (1), and the
// second word's (2, 3): one shift and mask moves a pair to the places above
// the nibbles.
template <bool Q5> struct KFmt {
    static constexpr int kRec = 2048 + (Q5 ? 512 : 0) + 256 + 64, kBlock = Q5 ? 176 : 144, kCols = 256;
    static constexpr bool kSplit = false, kSwap = true, kHalf = false, kRecScale = true, kMin = true, kMinLow = true;
    struct Item { u4_t q[2]; u2_t h, sc, mn; uint32_t dd; };
    static constexpr int kH = 2048, kS = 2048 + (Q5 ? 512 : 0), kM = kS + 128, kD = kS + 256;
    static __device__ __forceinline__ void load(Item &it, gptr r, uint32_t lane)
    {
        it.q[0] = ld<u4_t>(r, 16 * lane);
        it.q[1] = ld<u4_t>(r, 1024 + 16 * lane);
        if (Q5) it.h = ld<u2_t>(r, kH + 8 * lane);
        it.sc = ld<u2_t>(r, kS + 8 * (lane & 15));
        it.mn = ld<u2_t>(r, kM + 8 * (lane & 15));
        it.dd = ld<uint32_t>(r, kD + 4 * (lane & 15));
    }
    static __device__ __forceinline__ h8_t frag(const Item &it, int ks)
    {
        const int st = ks >> 1;
        const uint32_t w0 = it.q[st >> 1][2 * (st & 1)], w1 = it.q[st >> 1][2 * (st & 1) + 1];
        const bool hi = ks & 1;
        uint32_t w[4] = {w0, w0 >> 8, w1, w1 >> 8};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            w[q] = and_or(w[q], hi ? 0x00F000F0u : 0x000F000Fu, vreg(kMagic));
            if constexpr (Q5) {
                const uint32_t hw = it.h[st >> 1];
                const int up = (hi ? 7 : 4) - (8 * (st & 1) + 2 * q);      // to bit 4, or 8 (from b + 1)
                w[q] = and_or(up > 0 ? hw << up : hw >> -up, hi ? 0x01000100u : 0x00100010u, w[q]);
            }
        }
        return hi ? cat(n4(w[0], 0.0f), n4(w[1], 0.0f), n4(w[2], 0.0f), n4(w[3], 0.0f))
                  : cat(n0(w[0], 0.0f), n0(w[1], 0.0f), n0(w[2], 0.0f), n0(w[3], 0.0f));
    }
    static __device__ __forceinline__ float sub(const Item &it, int ks, int) { return ub(it.sc[ks >> 2], ks & 3); }
    static __device__ __forceinline__ float rec(const Item &it) { return h2f(it.dd & 0xffffu); }
    static __device__ __forceinline__ h8_t min_frag(const Item &it)
    {
        const h2_t f = splat(low());
        return cat(two(it.mn[0], 0, 0.0f) * f, two(it.mn[0], 1, 0.0f) * f, two(it.mn[1], 0, 0.0f) * f, two(it.mn[1], 1, 0.0f) * f);
    }
    static __device__ __forceinline__ float min_scale(const Item &it) { return -64.0f * h2f(it.dd >> 16); }
    static __device__ void put(uint8_t *r, const Src &s, int lane)
    {
        const int g = lane >> 4, n = lane & 15, qs = Q5 ? 48 : 16;
        for (int st = 0; st < 4; st++)
            for (int k = 0; k < 2; k++)
                reinterpret_cast<uint32_t *>(r + 1024 * (st >> 1) + 16 * lane)[2 * (st & 1) + k] =
                    s.word(0, qs + 32 * st + 8 * g + 4 * k);
        if (Q5) {
            for (int hw = 0; hw < 2; hw++) {
                uint32_t w = 0;
                for (int st = 0; st < 2; st++)
                    for (int q = 0; q < 4; q++)
                        for (int e = 0; e < 2; e++) {
                            const uint32_t qh = s.at(0, 16 + 8 * g + 4 * (q >> 1) + (q & 1) + 2 * e);
                            const int i = 2 * (2 * hw + st), b = 8 * st + 2 * q + 16 * e;
                            w |= (qh >> i & 1u) << b | (qh >> (i + 1) & 1u) << (b + 1);
                        }
                reinterpret_cast<uint32_t *>(r + kH + 8 * lane)[hw] = w;
            }
        }
        for (int k = 0; k < 2; k++) {
            r[kS + 8 * n + 2 * g + k] = (uint8_t)k4_scale(s, 4, 2 * g + k);
            r[kM + 8 * n + 2 * g + k] = (uint8_t)k4_min(s, 4, 2 * g + k);
        }
        if (g == 0) reinterpret_cast<uint32_t *>(r + kD)[n] = s.word(0, 0);   // d | dmin << 16
    }
};

// Q6_K (src/tensor/dequant.rs:203-214): w = (d sc) (u - 32), an int8 scale
// per 16 weights; weight 128 h + 32 j + l takes a nibble of
// ql[64 h + 32 (j & 1) + l] (low for j < 2) and bits 2 j of qh[32 h + l].
// The scales' products need 12 bits, more than an f16 holds: each 16 columns
// are summed apart and scaled in f32.
struct Q6Fmt {
    static constexpr int kRec = 2048 + 1024 + 256 + 32, kBlock = 210, kCols = 256;
    static constexpr bool kSplit = true, kSwap = true, kHalf = true, kRecScale = true, kMin = false, kMinLow = false;
    struct Item { u4_t q[2], c, sc; uint32_t d; };
    static __device__ __forceinline__ void load(Item &it, gptr r, uint32_t lane)
    {
        it.q[0] = ld<u4_t>(r, 16 * lane);
        it.q[1] = ld<u4_t>(r, 1024 + 16 * lane);
        it.c = ld<u4_t>(r, 2048 + 16 * lane);
        it.sc = ld<u4_t>(r, 3072 + 16 * (lane & 15));
        it.d = ld<uint16_t>(r, 3328 + 2 * (lane & 15));
    }
    // columns 16 i .. + 15 of step ks = 4 h + j
    static __device__ __forceinline__ h4_t half(const Item &it, int ks, int i)
    {
        const int h = ks >> 2, j = ks & 3;
        const uint32_t a = it.q[h][2 * (j & 1) + i], c = it.c[2 * h + i], e = j & 1 ? c << 2 : c << 4, f = j & 1 ? c >> 6 : c >> 4;
        return j < 2 ? cat(n0(and_or(e, 0x00300030u, and_or(a, 0x000F000Fu, vreg(kMagic))), 32.0f),
                           n0(and_or(f, 0x00300030u, and_or(a >> 8, 0x000F000Fu, vreg(kMagic))), 32.0f))
                     : cat(n4(and_or(e, 0x03000300u, and_or(a, 0x00F000F0u, vreg(kMagic))), 32.0f),
                           n4(and_or(f, 0x03000300u, and_or(a >> 8, 0x00F000F0u, vreg(kMagic))), 32.0f));
    }
    static __device__ __forceinline__ h8_t frag(const Item &it, int ks)
    {
        const h4_t a = half(it, ks, 0), b = half(it, ks, 1);
        return h8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    }
    // (an f16: two scales in two instructions, and the multiply-add takes it as it is)
    static __device__ __forceinline__ float sub(const Item &it, int ks, int i) { return (float)two(it.sc[ks >> 1], ks & 1, 128.0f)[i]; }
    static __device__ __forceinline__ float rec(const Item &it) { return h2f(it.d); }
    static __device__ void put(uint8_t *r, const Src &s, int lane)
    {
        const int g = lane >> 4, n = lane & 15;
        for (int h = 0; h < 2; h++) {
            for (int i = 0; i < 2; i++) {
                uint32_t *q = reinterpret_cast<uint32_t *>(r + 1024 * h + 16 * lane);
                q[i] = s.word(0, 64 * h + 16 * i + 4 * g);
                q[2 + i] = s.word(0, 64 * h + 32 + 16 * i + 4 * g);
                reinterpret_cast<uint32_t *>(r + 2048 + 16 * lane)[2 * h + i] = s.word(0, 128 + 32 * h + 16 * i + 4 * g);
            }
        }
        reinterpret_cast<uint32_t *>(r + 3072 + 16 * n)[g] = s.word(0, 192 + 4 * g) ^ 0x80808080u;    // scale + 128
        if (g == 0) reinterpret_cast<uint16_t *>(r + 3328)[n] = (uint16_t)s.half(0, 208);
    }
};

// Q3_K in the GGUF layout: w = d sc (u - 4), a signed 6-bit scale per 16
// weights; weight 128 h + 32 j + l has low bits (qs[32 h + l] >> 2 j) & 3 and
// third bit (hmask[l] >> (4 h + j)) & 1.  The three bits are merged into a
// nibble here (146 bytes per block on the device for the file's 110): a
// lane's eight weights of a step are the nibbles 0, 4, 1, 5, 2, 6, 3, 7 of
// its word.  |sc (u - 4)| <= 128 is exact in f16, so the scale goes into the
// weights.
struct Q3Fmt {
    static constexpr int kRec = 2048 + 256 + 32, kBlock = 110, kCols = 256;
    static constexpr bool kSplit = false, kSwap = false, kHalf = false, kRecScale = true, kMin = false, kMinLow = false;
    struct Item { u4_t q[2]; u2_t sc; uint32_t d; };
    static __device__ __forceinline__ void load(Item &it, gptr r, uint32_t lane)
    {
        it.q[0] = ld<u4_t>(r, 16 * lane);
        it.q[1] = ld<u4_t>(r, 1024 + 16 * lane);
        it.sc = ld<u2_t>(r, 2048 + 8 * (lane & 15) + 128 * (lane >> 5));
        it.d = ld<uint16_t>(r, 2304 + 2 * (lane & 15));
    }
    static __device__ __forceinline__ h8_t frag(const Item &it, int ks)
    {
        const uint32_t w = it.q[ks >> 2][ks & 3], h = w >> 8, p = ks & 3;
        const h2_t sc = as_h2(__builtin_amdgcn_perm(kMagic, it.sc[ks >> 2], 0x07000700u | p << 16 | p)) - splat(1024.0f + 32.0f);
        return cat(u0(w, 4.0f) * sc, u4(w, 4.0f) * sc, u0(h, 4.0f) * sc,
                   u4(h, 4.0f) * sc);
    }
    static __device__ __forceinline__ float sub(const Item &, int, int) { return 1.0f; }
    static __device__ __forceinline__ float rec(const Item &it) { return h2f(it.d); }
    // The scale of sub-block is, plus 32: low nibble from byte is % 8 (bits
    // 0-3 for is < 8, 4-7 above), top two bits from bits 2 (is / 4) of byte
    // 8 + is % 4.
    static __device__ uint32_t scale(const Src &s, int is)
    {
        const int k = is >> 2, j = is & 3;
        const uint32_t b = s.at(0, 96 + (k & 1) * 4 + j);
        return (k < 2 ? b & 15u : b >> 4) | (s.at(0, 104 + j) >> (2 * k) & 3u) << 4;
    }
    static __device__ void put(uint8_t *r, const Src &s, int lane)
    {
        const int g = lane >> 4, n = lane & 15;
        for (int ks = 0; ks < 8; ks++) {
            const int h = ks >> 2, j = ks & 3;
            uint32_t w = 0;
            for (int i = 0; i < 8; i++) {
                const int l = 8 * g + i;
                const uint32_t u = (s.at(0, 32 + 32 * h + l) >> (2 * j) & 3u) | (s.at(0, l) >> (4 * h + j) & 1u) << 2;
                w |= u << (4 * (i >> 1) + 16 * (i & 1));
            }
            reinterpret_cast<uint32_t *>(r + 1024 * h + 16 * lane)[j] = w;
        }
        if ((g & 1) == 0)       // lanes 16 g, 16 (g + 1) share the 16-column half g / 2 of a step
            for (int ks = 0; ks < 8; ks++)
                r[2048 + 8 * n + 128 * (g >> 1) + ks] = (uint8_t)scale(s, 2 * ks + (g >> 1));
        if (g == 0) reinterpret_cast<uint16_t *>(r + 2304)[n] = (uint16_t)s.half(0, 108);
    }
};

// ------------------------------------------------------- x in f16 parts ----
// x s = a + (b + c) 2^-11, three f16 parts with their 11 bits each, s =
// 2^(15 - e) for the largest |x| in [2^e, 2^(e+1)) of the record's 256 columns
// of the vector.  Every x of at least 2^-27 of that largest is held exactly
// (24 bits: the parts are cut off, not rounded, and c has two bits left to
// hold); a smaller one to half of f16's last step in c, 2^-51 of the largest.
// (b and c are summed apart from a, so their factor costs nothing: without it
// the limits were 2^-16 and 2^-40.)  (kMin) the sums of x s over 32 columns,
// over 64, go into three parts too: whole from 2^-21 of the largest x, to
// 2^-45 of it below.
//
// A wave converts a record of a vector: lane L holds columns 4 L .. 4 L + 3,
// those of step L / 8.
__device__ __forceinline__ void x_scale(float mx, float &s, float &inv)
{
    // 2^(15 - e), at most 2^126, and its inverse (exact; e of a subnormal as
    // -127, of an infinity as 128)
    const int e = (int)(__float_as_uint(mx) >> 23) - 127;
    const int se = mx > 0.0f ? min(15 - e, 126) : 0;
    s = __uint_as_float((uint32_t)(se + 127) << 23);
    inv = __uint_as_float((uint32_t)(127 - se) << 23);
}
__device__ __forceinline__ h2_t cut(float x, float y) { return __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_pkrtz(x, y)); }
// (For an infinite t the difference is a NaN, which the clamp drops: a alone
// decides the sum.)
__device__ __forceinline__ float rest(float t, _Float16 a) { return __builtin_amdgcn_fmed3f(t - (float)a, -32.0f, 32.0f); }
__device__ __forceinline__ void x_split2(float x, float y, h2_t (&q)[3])
{
    q[0] = cut(x, y);
    x = rest(x, q[0].x) * kLow;
    y = rest(y, q[0].y) * kLow;
    q[1] = cut(x, y);
    q[2] = h2_t{(_Float16)(x - (float)q[1].x), (_Float16)(y - (float)q[1].y)};
}
// The sum of x's products, from those of a and those of b and c.
__device__ __forceinline__ float whole(float a, float bc) { return fmaf(bc, 1.0f / kLow, a); }
// The value of a lane paired with this one (of 2, 4, 8 or 16 lanes that hold
// equal halves).
template <int C> __device__ __forceinline__ float pair(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), C, 0xf, 0xf, true));
}
constexpr int kPair1 = 0xB1, kPair2 = 0x4E, kPair4 = 0x141, kPair8 = 0x140;    // quad_perm, row_half_mirror, row_mirror
struct XRec {
    h4_t q[3];          // the parts of the lane's columns, in operand order
    _Float16 sum[3];    // (kMin) of the lane's step
    float inv;          // 1 / s
};
template <class F> __device__ __forceinline__ XRec x_convert(f4_t x)
{
    XRec r;
    float mx = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
    mx = fmaxf(mx, pair<kPair1>(mx));
    mx = fmaxf(mx, pair<kPair2>(mx));
    mx = fmaxf(mx, pair<kPair4>(mx));
    mx = fmaxf(mx, pair<kPair8>(mx));
    const int b = __float_as_int(mx);
    mx = fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(b, 0)), __int_as_float(__builtin_amdgcn_readlane(b, 16))),
               fmaxf(__int_as_float(__builtin_amdgcn_readlane(b, 32)), __int_as_float(__builtin_amdgcn_readlane(b, 48))));
    float s;
    x_scale(mx, s, r.inv);
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] *= s;
    h2_t u[3], v[3];
    x_split2(x[0], x[F::kSwap ? 2 : 1], u);
    x_split2(x[F::kSwap ? 1 : 2], x[3], v);
#pragma unroll
    for (int i = 0; i < 3; i++) r.q[i] = cat(u[i], v[i]);
    if constexpr (F::kMin) {
        float t = (x[0] + x[1]) + (x[2] + x[3]);
        t += pair<kPair1>(t);
        t += pair<kPair2>(t);
        t += pair<kPair4>(t);
        h2_t w[3];
        x_split2(t * 0.015625f, 0.0f, w);
#pragma unroll
        for (int i = 0; i < 3; i++) r.sum[i] = w[i].x;
    }
    return r;
}
// Where a lane's columns of its step go: operand group g, half h of the eight.
template <class F> __device__ __forceinline__ void x_place(int lane, int &g, int &h)
{
    const int i = lane & 7;     // columns 4 i .. 4 i + 3
    g = F::kSplit ? i & 3 : i >> 1;
    h = F::kSplit ? i >> 2 : i & 1;
}

// The order of every addition is the same in the two kernels below, so a
// vector's result does not depend on the others of the call: the sum of a's
// products with a step's weights (of a half's, kHalf) from zero, that of c's
// from zero and of b's onto it, and the two added (an MFMA that adds onto a
// sum cuts what falls below the largest term's last bits, always downwards:
// a's products onto those of b and c, 1.6e-7 against 64 bits for Q4_0 x 8192
// where this has 1.1e-7); the steps of a record; the record's factor and its
// minimums; record after record, kChunk at a time, and the chunks.
constexpr int kChunk = 16;

// ------------------------------------------------- up to 4 vectors (GEMV) ---
// (and more over few rows, four to a block)
// Rows 4 v and 4 v + 1 of the first MFMA's A = parts a and c of vector v (the
// others zero), row 4 v + 1 of the second one's = b: a lane's sums of vector
// g are D[0] and D[1].  Formats with a scale for each 16 columns (kHalf) use
// all four rows: x of the first 16 columns of the step (zeros for the others)
// in 4 v and 4 v + 2, and of the second in 4 v + 1 and 4 v + 3.
//
// A block takes tpb tiles of 16 rows; its waves share the columns, a record
// each, with the operand of a and c in registers for all tiles and that of b
// in LDS (both in registers take more than the 128 of 4 waves per SIMD).  D tiles are in
// flight: a record's registers are loaded again, for the tile D further on,
// as soon as it has been used.  The waves' sums meet in LDS every kBatch
// tiles (two buffers: one barrier per batch); within a batch a wave's
// priority falls with its progress, so that the waves of a SIMD arrive
// together (with equal priorities the youngest came late and ran the end of
// each batch alone: Q4_K 152064 x 3584 59 us against 52, Q6_K 84 against 74).
// Bound: the read of the weights (5.1-6.5 TB/s at 152064 x 3584; Q3_K and Q5_K,
// the slowest, by the unpacking).  Four tiles in flight instead of two: 57 us
// against 52 (Q4_K; these figures with x in two parts).  Rows of more columns
// than the waves hold (MULTI) go in chunks: a batch's tiles take one chunk
// after the other, and the running sums stay with the waves that add them.
constexpr int kVecs = 4, kBatch = 8, kMaxWaves = kChunk, kInFlight = 2;
// A wave's f16s of x in LDS: rows of 256, padded: two for each vector, one of
// zeros for the unused rows of A, then [v][part][8] of the sums.
constexpr int kXRow = 264, kXZeros = 2 * kVecs * kXRow, kXWave = (2 * kVecs + 1) * kXRow + 112;
// floats of a tile's sums (16 more: the rows of four tiles in different banks)
__host__ __device__ constexpr int lds_tile(int nw) { return nw * 64 + 16; }
constexpr size_t gemv_lds(int nw)
{
    return sizeof(float) * 2 * kBatch * lds_tile(nw) + sizeof(_Float16) * kXWave * nw;
}

struct XOps {
    h8_t ac[8];
    const _Float16 *b;  // in LDS, + 32 ks
    h8_t sx;
    float inv;          // 1 / s of vector g
};
__device__ __forceinline__ void lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// The operands of a record's columns [c0, c0 + 256) from the lane's columns
// 4 L .. + 3 of each vector.  The parts pass through a vector's two rows of
// LDS: a and c, then b stays in the second one; kHalf: the halves of a, of c
// and of b, which stay, each with the other half's columns zero.
template <class F>
__device__ __forceinline__ void x_ops(XOps &o, const f4_t (&raw)[kVecs], _Float16 *lds, int nv, int cols, int c0)
{
    const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15, k = lane >> 3, q = m & 3;
    const bool on = (m >> 2) < nv;
    _Float16 *sxs = lds + kXZeros + kXRow;
    int pg, ph;
    x_place<F>(lane, pg, ph);
    auto put = [&](int v, int row, h4_t x) {
        *reinterpret_cast<h4_t *>(lds + (2 * v + row) * kXRow + 32 * k + 8 * pg + 4 * ph) = x;
    };
    auto from = [&](bool is, int row) { return lds + (on && is ? (2 * (m >> 2) + row) * kXRow : kXZeros) + 8 * g; };
    const h4_t z = {0, 0, 0, 0};
    *reinterpret_cast<h4_t *>(lds + kXZeros + 4 * lane) = z;
    XRec r[kVecs];
    o.inv = 1.0f;
#pragma unroll
    for (int v = 0; v < kVecs; v++)
        if (v < nv) {
            r[v] = x_convert<F>(c0 + 4 * lane < cols ? raw[v] : kZero);
            o.inv = g == v ? r[v].inv : o.inv;
            if constexpr (F::kMin)
                if ((lane & 7) < 3) sxs[24 * v + 8 * (lane & 7) + k] = (lane & 7) == 0 ? r[v].sum[0] : (lane & 7) == 1 ? r[v].sum[1] : r[v].sum[2];
            put(v, F::kHalf ? ph : 0, r[v].q[0]);
            put(v, F::kHalf ? 1 - ph : 1, F::kHalf ? z : r[v].q[2]);
        }
    lds_fence();
    const _Float16 *p = from(q < 2, q & 1);
#pragma unroll
    for (int ks = 0; ks < 8; ks++) o.ac[ks] = *reinterpret_cast<const h8_t *>(p + 32 * ks);
    lds_fence();
    if constexpr (F::kHalf) {
#pragma unroll
        for (int v = 0; v < kVecs; v++)
            if (v < nv) put(v, ph, r[v].q[2]);
        lds_fence();
        p = from(q >= 2, q & 1);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) o.ac[ks] = q >= 2 ? *reinterpret_cast<const h8_t *>(p + 32 * ks) : o.ac[ks];
        lds_fence();
    }
#pragma unroll
    for (int v = 0; v < kVecs; v++)
        if (v < nv) put(v, F::kHalf ? ph : 1, r[v].q[1]);
    lds_fence();
    o.b = F::kHalf ? from(q >= 2, q & 1) : from(q == 1, 1);
    if constexpr (F::kMin)      // part g of the sums in row 4 v (not kMinLow: b's and c's in row 4 v + 1)
        o.sx = *reinterpret_cast<const h8_t *>(on && g < 3 && q == (!F::kMinLow && g > 0) ? sxs + 24 * (m >> 2) + 8 * g : lds + kXZeros);
}

// A record's sum for the lane's row and vector, times s.
template <class F> __device__ __forceinline__ float dot(const typename F::Item &it, const XOps &x)
{
    float v = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 8; ks++) {
        const h8_t w = F::frag(it, ks);
        const f4_t D = mfma(*reinterpret_cast<const h8_t *>(x.b + 32 * ks), w, mfma(x.ac[ks], w, kZero));
        v = fmaf(whole(D[0], D[F::kHalf ? 2 : 1]), F::sub(it, ks, 0), v);
        if constexpr (F::kHalf) v = fmaf(whole(D[1], D[3]), F::sub(it, ks, 1), v);
    }
    if constexpr (F::kRecScale) v *= F::rec(it);
    if constexpr (F::kMin) {
        const f4_t D = mfma(x.sx, F::min_frag(it), kZero);
        v = fmaf(F::kMinLow ? D[0] : whole(D[0], D[1]), F::min_scale(it), v);
    }
    return v;
}

template <class F, bool MULTI>
__global__ void __launch_bounds__(64 * kMaxWaves)
qgemv_kernel(const uint8_t *W, const float *x, float *out, int rows, int cols, int np, int B, int tiles, int tpb)
{
    extern __shared__ __align__(16) float red[];    // [2][batch] sums of a tile, then the waves' x
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6, ts = lds_tile(nw);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t0 = blockIdx.x * tpb, t1 = min(t0 + tpb, tiles);
    const int v0 = kVecs * blockIdx.y, nv = min(kVecs, B - v0);
    if (t0 >= t1) return;
    x += (size_t)v0 * cols;
    out += (size_t)v0 * rows;
    _Float16 *xl = reinterpret_cast<_Float16 *>(red + 2 * kBatch * ts) + kXWave * w;
    XOps xo;
    typename F::Item it[kInFlight];
    auto load = [&](int d, int t, int p) {      // (past the block's tiles: the last one, not used)
        F::load(it[d], opaque(W + ((size_t)min(t, t1 - 1) * np + p) * F::kRec), lane);
    };
    auto start = [&](int t, int p) {        // (x first: loads return in order)
        f4_t raw[kVecs];
#pragma unroll
        for (int v = 0; v < kVecs; v++)     // (cols is a multiple of 32)
            raw[v] = *reinterpret_cast<const f4_t *>(x + (size_t)min(v, nv - 1) * cols + min(kPair * p + 4 * lane, cols - 4));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < kInFlight; d++) load(d, t + d, p);
        __builtin_amdgcn_sched_barrier(0);
        x_ops<F>(xo, raw, xl, nv, cols, kPair * p);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (!MULTI) start(t0, w);
    int buf = 0;
    for (int tb = t0; tb < t1; tb += kBatch) {
        const int nb = min(kBatch, t1 - tb);
        float sum = 0.0f;       // of the chunks (MULTI: a wave adds for at most one vector and four tiles)
        for (int c = 0; c < (MULTI ? np : 1); c += nw, buf ^= 1) {
            float *rb = red + buf * kBatch * ts;
            const int p = c + w;
            if (!MULTI || p < np) {
                if (MULTI) start(tb, p);
                for (int k0 = 0; k0 < nb; k0 += kInFlight) {
                    switch (k0 * 4 / kBatch) {
                    case 0: __builtin_amdgcn_s_setprio(3); break;
                    case 1: __builtin_amdgcn_s_setprio(2); break;
                    case 2: __builtin_amdgcn_s_setprio(1); break;
                    default: __builtin_amdgcn_s_setprio(0); break;
                    }
#pragma unroll
                    for (int d = 0; d < kInFlight; d++) {
                        const int k = k0 + d;
                        if (d > 0 && k >= nb) break;
                        const float v = dot<F>(it[d], xo) * xo.inv;
                        __builtin_amdgcn_sched_barrier(0);
                        load(d, tb + k + kInFlight, p);
                        rb[k * ts + w * 64 + lane] = v;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            __builtin_amdgcn_s_setprio(3);
            // a wave adds four tiles of a vector at a time: vector v, row n is in
            // lane 16 v + n
            const int cnt = min(nw, np - c);
            for (int u = w; u < nv * (kBatch / 4); u += nw) {
                const int v = u / (kBatch / 4), rr = (u % (kBatch / 4)) * 64 + lane;
                const uint32_t r = 16u * tb + rr;
                const float *q = rb + (rr >> 4) * ts + v * 16 + (lane & 15);
                float s = 0.0f;
#pragma unroll
                for (int i = 0; i < kMaxWaves; i++)
                    if (i < cnt) s += q[i * 64];
                if (MULTI) sum = s = c > 0 ? sum + s : s;
                if (c + nw >= np && rr < 16 * nb && r < (uint32_t)rows) out[(size_t)v * rows + r] = s;
            }
        }
    }
}

// ------------------------------------------- more vectors, up to 32 (GEMM) ---
// VT tiles of 16 vectors: row m of A's tile vt is vector 16 vt + m, an MFMA
// for each part of x, the rows of D (of a) and E (of b and c) the vectors.
//
// A block of 8 waves (one per CU, 2 waves per SIMD: 256 registers each) takes
// up to 8 RT tiles of 16 rows at a time, RT to a wave, through all columns.
// The x of a record is converted once per block into LDS (each wave 2 VT of
// the vectors; two buffers, one barrier per record) and read from there for
// two or three groups of the wave's tiles; a group's registers are loaded
// again, for the next record, as soon as it has been used.  (x of 32 vectors
// in registers for all columns would fill the CU's register file.)
constexpr int kGemmWaves = 8;
// f16s of a step's part in LDS: lane 16 g + m reads the eight at m, m ^ 8 in
// the odd groups (so, and with the steps shifted by eight, the lanes that
// write a vector's columns, four each, use all banks)
constexpr int kXStep = 520;
template <class F, int VT> constexpr int kXBuf = VT * (3 * 8 * kXStep + (F::kMin ? 512 : 0));     // of a record's x
__device__ __forceinline__ int x_lane(int lane) { return 8 * (lane ^ (lane >> 1 & 8)); }

template <class F, int VT, int N>
__device__ __forceinline__ void group(const typename F::Item *it, const _Float16 *xb, const float *inv, float (*acc)[VT][4])
{
    const int lane = threadIdx.x & 63;
    const _Float16 *xr = xb + x_lane(lane);
    float sum[N][VT][4] = {};   // of the record: shorter chains of additions
    h8_t nx[3];                 // the next vector tile's x, read ahead
    auto read = [&](int ks, int v) {
#pragma unroll
        for (int q = 0; q < 3; q++) nx[q] = *reinterpret_cast<const h8_t *>(xr + ((3 * v + q) * 8 + ks) * kXStep);
    };
    read(0, 0);
#pragma unroll
    for (int ks = 0; ks < 8; ks++) {
        h8_t f[N];
        float s[N][2];
#pragma unroll
        for (int r = 0; r < N; r++) {
            f[r] = F::frag(it[r], ks);
#pragma unroll
            for (int i = 0; i < (F::kHalf ? 2 : 1); i++) s[r][i] = F::sub(it[r], ks, i);
        }
#pragma unroll
        for (int v = 0; v < VT; v++) {
            const h8_t xa = nx[0], xb = nx[1], xc = nx[2];
            if (v + 1 < VT) read(ks, v + 1);
            else if (ks < 7) read(ks + 1, 0);
#pragma unroll
            for (int r = 0; r < N; r++)
#pragma unroll
                for (int i = 0; i < (F::kHalf ? 2 : 1); i++) {
                    const h8_t w = !F::kHalf ? f[r] : i == 0 ? h8_t{f[r][0], f[r][1], f[r][2], f[r][3], 0, 0, 0, 0}
                                                             : h8_t{0, 0, 0, 0, f[r][4], f[r][5], f[r][6], f[r][7]};
                    const f4_t E = mfma(xb, w, mfma(xc, w, kZero)), D = mfma(xa, w, kZero);
#pragma unroll
                    for (int j = 0; j < 4; j++) sum[r][v][j] = fmaf(whole(D[j], E[j]), s[r][i], sum[r][v][j]);
                }
            // these sums are done here (else the steps of a record are mixed
            // until the registers spill)
#pragma unroll
            for (int r = 0; r < N; r++)
#pragma unroll
                for (int j = 0; j < 4; j++) asm volatile("" : "+v"(sum[r][v][j]));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The minimums join the record's own sum first: the two nearly cancel
    // where the weights are centred, and the running sum then takes the small
    // difference.
#pragma unroll
    for (int v = 0; v < VT; v++) {
        const f4_t iv = *reinterpret_cast<const f4_t *>(inv + 16 * v + 4 * (lane >> 4));
        h8_t sa, sb;            // the sums' parts (not kMinLow: a, and b and c)
        if constexpr (F::kMin) {
            constexpr h8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
            const h8_t sx = *reinterpret_cast<const h8_t *>(xb + VT * 3 * 8 * kXStep + 512 * v + 8 * lane);
            sa = F::kMinLow || lane < 16 ? sx : z;
            sb = lane < 16 ? z : sx;
        }
#pragma unroll
        for (int r = 0; r < N; r++) {
            f4_t D, E;
            if constexpr (F::kMin) {
                const h8_t w = F::min_frag(it[r]);
                D = mfma(sa, w, kZero);
                if constexpr (!F::kMinLow) E = mfma(sb, w, kZero);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float t = sum[r][v][j];
                if constexpr (F::kRecScale) t *= F::rec(it[r]);
                if constexpr (F::kMin) t = fmaf(F::kMinLow ? D[j] : whole(D[j], E[j]), F::min_scale(it[r]), t);
                acc[r][v][j] += t * iv[j];
            }
        }
    }
    // The additions are done here: put off past the branches that follow they
    // keep the products of all steps in registers.
#pragma unroll
    for (int r = 0; r < N; r++)
#pragma unroll
        for (int v = 0; v < VT; v++)
#pragma unroll
            for (int j = 0; j < 4; j++) asm volatile("" : "+v"(acc[r][v][j]));
}

template <class F, int VT, int RT>
__global__ void __launch_bounds__(64 * kGemmWaves)
qgemm_kernel(const uint8_t *W, const float *x, float *out, int rows, int cols, int np, int B, int per, int tiles, int tpb)
{
    // RT > 1: the wave's tiles in groups of N; RT = 1: two records of its tile
    constexpr int N = RT <= 3 ? (RT + 1) / 2 : VT == 2 ? 2 : (RT + 1) / 2, NI = RT > 1 ? RT : 2;
    __shared__ __align__(16) _Float16 xs[2][kXBuf<F, VT>];
    __shared__ __align__(16) float si[2][VT * 16];      // 1 / s of the vectors
    const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int v0 = blockIdx.y * per, nv = min(per, B - v0);
    const int t0 = blockIdx.x * tpb, t1 = min(t0 + tpb, tiles);
    if (t0 >= t1) return;
    x += (size_t)v0 * cols;
    out += (size_t)v0 * rows;

    typename F::Item it[NI];
    f4_t raw[2 * VT];           // columns 4 lane .. + 3 of vectors w, w + 8, ..
    auto xload = [&](int p) {   // (cols is a multiple of 32)
        const int c = min(kPair * p + 4 * lane, cols - 4);
#pragma unroll
        for (int i = 0; i < 2 * VT; i++) raw[i] = *reinterpret_cast<const f4_t *>(x + (size_t)min(w + 8 * i, nv - 1) * cols + c);
    };
    int pg, ph;
    x_place<F>(lane, pg, ph);
    const int at = (lane >> 3) * kXStep + 4 * ph;
    auto xput = [&](int p) {
        _Float16 *b = xs[p & 1];
#pragma unroll
        for (int i = 0; i < 2 * VT; i++) {
            const int v = w + 8 * i, vt = i >> 1, vm = v & 15;
            const XRec r = x_convert<F>(v < nv && kPair * p + 4 * lane < cols ? raw[i] : kZero);
#pragma unroll
            for (int q = 0; q < 3; q++) *reinterpret_cast<h4_t *>(b + (3 * vt + q) * 8 * kXStep + at + x_lane(16 * pg + vm)) = r.q[q];
            if (lane == 0) si[p & 1][v] = r.inv;
            if constexpr (F::kMin) {        // lanes 16 g + m hold part g of the sums over the steps
                const int q = lane & 7;
                if (q < 4)
                    b[VT * 3 * 8 * kXStep + 512 * vt + 8 * (16 * q + vm) + (lane >> 3)] =
                        q == 0 ? r.sum[0] : q == 1 ? r.sum[1] : q == 2 ? r.sum[2] : (_Float16)0.0f;
            }
        }
    };
    auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    const int rounds = (t1 - t0 + kGemmWaves * RT - 1) / (kGemmWaves * RT);
    for (int rd = 0; rd < rounds; rd++) {
        // the round's tiles, spread evenly over the waves
        const int ra = t0 + (int)((long)(t1 - t0) * rd / rounds), nt = t0 + (int)((long)(t1 - t0) * (rd + 1) / rounds) - ra;
        const int q = nt / kGemmWaves, rem = nt - q * kGemmWaves;
        const int cnt = q + (w < rem), tw = ra + w * q + min(w, rem);
        auto load = [&](int i, int r, int p) {      // past the wave's tiles or the records: the last, not used
            F::load(it[i], opaque(W + ((size_t)min(tw + r, t1 - 1) * np + min(p, np - 1)) * F::kRec), lane);
        };
        xload(0);
#pragma unroll
        for (int i = 0; i < NI; i++) load(i, RT > 1 ? i : 0, RT > 1 ? 0 : i);
        float acc[RT][VT][4] = {};
        // The sums of a chunk that ends before record p: onto those of the
        // chunks before it, which wait in out.
        auto flush = [&](int p) {
            // (opaque: else the addresses and conditions are kept in registers through the loop)
            size_t ld = rows;
            int lim = nv, most = cnt;
            asm volatile("" : "+s"(ld), "+s"(lim), "+s"(most));
#pragma unroll
            for (int v = 0; v < VT; v++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int vec = 16 * v + 4 * g + j;
#pragma unroll
                    for (int r = 0; r < RT; r++) {
                        const uint32_t row = 16u * (tw + r) + m;
                        if (r < most && vec < lim && row < ld) {
                            float *o = out + vec * ld + row;
                            __builtin_nontemporal_store(p > kChunk ? *o + acc[r][v][j] : acc[r][v][j], o);
                        }
                        acc[r][v][j] = 0.0f;
                    }
                }
        };
        xput(0);
        xload(1);
        sync();
        for (int p = 0; p < np; p += RT > 1 ? 1 : 2) {
            const _Float16 *xb = xs[p & 1];
            const float *sb = si[p & 1];
            __builtin_amdgcn_s_setprio(3);
            __builtin_amdgcn_sched_barrier(0);
            group<F, VT, N>(it, xb, sb, acc);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < N; i++) load(i, i, p + (RT > 1 ? 1 : 2));
            xput(p + 1);
            xload(p + 2);
            if constexpr (RT > 1) {
#pragma unroll
                for (int r = N; r < RT; r += N) {
                    constexpr int M = RT % N;       // the last group's, if it is smaller
                    if (r == N) __builtin_amdgcn_s_setprio(1);
                    else __builtin_amdgcn_s_setprio(0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (M == 0 || r + N <= RT) group<F, VT, N>(it + r, xb, sb, acc + r);
                    else group<F, VT, M ? M : 1>(it + r, xb, sb, acc + r);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = r; i < r + N; i++)
                        if (i < RT) load(i, i, p + 1);
                }
            } else {
                sync();
                if (p + 1 < np) {
                    __builtin_amdgcn_sched_barrier(0);
                    group<F, VT, 1>(it + 1, xs[1], si[1], acc);
                    __builtin_amdgcn_sched_barrier(0);
                    load(1, 0, p + 3);
                    xput(p + 2);
                    xload(p + 3);
                }
            }
            sync();
            if (const int q = p + (RT > 1 ? 1 : 2); q % kChunk == 0 && q < np) flush(q);
        }
        flush(np);
    }
}

// GGUF blocks of rows [16 t0, 16 (t0 + tiles)) of the matrix (raw, nb blocks
// of F::kBlock bytes per row, rows_here of them given) to records; one lane
// of a record per thread.
template <class F>
__global__ void __launch_bounds__(256) repack_kernel(const uint8_t *raw, uint8_t *W, int rows_here, int nb, int np, int tiles)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int lane = (int)(i & 63);
    const size_t rec = i >> 6;
    if (rec >= (size_t)tiles * np) return;
    const int t = (int)(rec / np), p = (int)(rec - (size_t)t * np);
    const int row = 16 * t + (lane & 15), j = p * (kPair / F::kCols);
    const Src s{raw + ((size_t)(row < rows_here ? row : 0) * nb + j) * F::kBlock, F::kBlock, row < rows_here ? nb - j : 0};
    F::put(W + rec * F::kRec, s, lane);
}

} // namespace gs

// ------------------------------------------------------------- host side ---
struct gs_qmatrix {
    uint32_t qtype;
    size_t rows, cols;
    int np, tiles;             // records per row tile, row tiles
    int device;
    int cus;
    uint8_t *base;             // the records
};

namespace {

// Calls f with a value of the format of `qtype`.
template <class Fn> int with_format(uint32_t qtype, Fn f)
{
    switch (qtype) {
    case GS_QTYPE_Q4_0: return f(gs::Q4Fmt<false>());
    case GS_QTYPE_Q4_1: return f(gs::Q4Fmt<true>());
    case GS_QTYPE_Q8_0: return f(gs::Q8Fmt());
    case GS_QTYPE_Q3_K: return f(gs::Q3Fmt());
    case GS_QTYPE_Q4_K: return f(gs::KFmt<false>());
    case GS_QTYPE_Q5_K: return f(gs::KFmt<true>());
    case GS_QTYPE_Q6_K: return f(gs::Q6Fmt());
    default: return GS_ERR_UNSUPPORTED;
    }
}

constexpr size_t kStage = (size_t)64 << 20;     // raw blocks on the device at a time

// The matrix's blocks, a group of row tiles at a time, through a staging
// buffer on the device to records.
template <class F> int upload(gs_qmatrix *m, const uint8_t *src)
{
    const size_t nb = m->cols / F::kCols, row_bytes = nb * F::kBlock;
    const size_t step = kStage / (16 * row_bytes) > 0 ? kStage / (16 * row_bytes) : 1;
    const size_t most = step < (size_t)m->tiles ? step : (size_t)m->tiles;
    if (hipMalloc((void **)&m->base, (size_t)m->tiles * m->np * F::kRec) != hipSuccess) {
        (void)hipGetLastError();
        m->base = nullptr;
        return GS_ERR_NOMEM;
    }
    uint8_t *raw = nullptr;
    if (hipMalloc((void **)&raw, most * 16 * row_bytes) != hipSuccess) {
        (void)hipGetLastError();
        return GS_ERR_NOMEM;
    }
    int rc = GS_OK;
    for (size_t t = 0; t < (size_t)m->tiles && rc == GS_OK; t += step) {
        const size_t n = (size_t)m->tiles - t < step ? (size_t)m->tiles - t : step;
        const size_t rows = m->rows - 16 * t < 16 * n ? m->rows - 16 * t : 16 * n;
        if (hipMemcpy(raw, src + 16 * t * row_bytes, rows * row_bytes, hipMemcpyHostToDevice) != hipSuccess) { rc = GS_ERR_HIP; break; }
        const size_t threads = n * m->np * 64;
        hipLaunchKernelGGL(gs::repack_kernel<F>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, nullptr, raw,
                           m->base + t * m->np * F::kRec, (int)rows, (int)nb, m->np, (int)n);
        if (hipGetLastError() != hipSuccess) rc = GS_ERR_HIP;
    }
    if (hipStreamSynchronize(nullptr) != hipSuccess) rc = GS_ERR_HIP;
    (void)hipFree(raw);
    return rc;
}

template <class F, bool MULTI>
int gemv(const gs_qmatrix *m, const float *x, float *out, int B, hipStream_t st)
{
    const int nw = MULTI ? gs::kMaxWaves : m->np;
    int blocks = m->cus * (gs::kMaxWaves / nw);         // 16 waves per CU
    const int tpb = (m->tiles + blocks - 1) / blocks;
    blocks = (m->tiles + tpb - 1) / tpb;
    hipLaunchKernelGGL((gs::qgemv_kernel<F, MULTI>), dim3(blocks, (B + gs::kVecs - 1) / gs::kVecs), dim3(64 * nw), gs::gemv_lds(nw), st, m->base, x, out,
                       (int)m->rows, (int)m->cols, m->np, B, m->tiles, tpb);
    return hipGetLastError() == hipSuccess ? GS_OK : GS_ERR_HIP;
}

template <class F, int VT, int RT>
int gemm_rt(const gs_qmatrix *m, const float *x, float *out, int B, int per, int groups, int blocks, int tpb, hipStream_t st)
{
    hipLaunchKernelGGL((gs::qgemm_kernel<F, VT, RT>), dim3(blocks, groups), dim3(64 * gs::kGemmWaves), 0, st, m->base, x,
                       out, (int)m->rows, (int)m->cols, m->np, B, per, m->tiles, tpb);
    return hipGetLastError() == hipSuccess ? GS_OK : GS_ERR_HIP;
}

template <class F, int VT>
int gemm(const gs_qmatrix *m, const float *x, float *out, int B, int per, int groups, hipStream_t st)
{
    int blocks = m->cus / groups;
    if (blocks < 1) blocks = 1;
    const int tpb = (m->tiles + blocks - 1) / blocks;
    blocks = (m->tiles + tpb - 1) / tpb;
    const int rounds = (tpb + 5 * gs::kGemmWaves - 1) / (5 * gs::kGemmWaves);
    const int rt = ((tpb + rounds - 1) / rounds + gs::kGemmWaves - 1) / gs::kGemmWaves;
    switch (rt) {
    case 1: return gemm_rt<F, VT, 1>(m, x, out, B, per, groups, blocks, tpb, st);
    case 2: return gemm_rt<F, VT, 2>(m, x, out, B, per, groups, blocks, tpb, st);
    case 3: return gemm_rt<F, VT, 3>(m, x, out, B, per, groups, blocks, tpb, st);
    case 4: return gemm_rt<F, VT, 4>(m, x, out, B, per, groups, blocks, tpb, st);
    default: return gemm_rt<F, VT, 5>(m, x, out, B, per, groups, blocks, tpb, st);
    }
}

template <class F>
int project(const gs_qmatrix *m, const float *x, float *out, int B, hipStream_t st)
{
    // More than 4 vectors over few rows: a wave of the second kernel takes row
    // tiles through all columns, so fewer tiles than its waves (8 per CU) leave
    // some without work, and the time is that of one tile.  There the first
    // kernel takes the vectors four at a time (the same bits).  The line: 6
    // (row tile, four vectors) pairs per CU.  us per call by the second kernel
    // and the first, on the near and far side of it:
    //                     4000 rows: 5, 16, 24, 32 vectors         8000 rows: 8, 12, 16
    //   Q4_K x 3584       30.8 11.8  31.0 26.6  51.2 38.3 50.8 49.8  30.8 16.3  30.8 23.7  30.7 31.1
    //   Q6_K x 8192       79.4 33.6  78.3 71.0  131 104   132 137    85.4 50.4  85.4 74.5  83.1 93.7
    //   Q8_0 x 3584       27.1 12.8  28.1 25.9  45.9 38.5 46.2 49.6  29.1 17.5  29.5 25.8  28.7 35.6
    // (one vector after the other on the vector units, 4000 rows, 5 vectors:
    // Q6_K x 8192 68, Q8_0 x 3584 26.9)
    const bool few = (size_t)((B + gs::kVecs - 1) / gs::kVecs) * m->tiles <= 6 * (size_t)m->cus;
    if (B <= gs::kVecs || few)
        return m->np <= gs::kMaxWaves ? gemv<F, false>(m, x, out, B, st) : gemv<F, true>(m, x, out, B, st);
    const int groups = (B + 31) / 32, per = (B + groups - 1) / groups;
    return per <= 16 ? gemm<F, 1>(m, x, out, B, per, groups, st) : gemm<F, 2>(m, x, out, B, per, groups, st);
}

} // namespace

extern "C" {

int gs_qmatrix_upload(uint32_t qtype, const void *blocks, size_t rows, size_t cols, gs_qmatrix **out)
{
    if (!out) return GS_ERR_INVALID;
    *out = nullptr;
    if (!blocks || rows == 0 || cols == 0) return GS_ERR_INVALID;
    size_t bw = 0;
    if (int rc = with_format(qtype, [&](auto f) { bw = decltype(f)::kCols; return GS_OK; })) return rc;
    if (cols % bw != 0 || cols > (size_t)gs::kMaxCols || rows > 0x7fffffffu) return GS_ERR_UNSUPPORTED;
    // the size limits of each type's matrices
    const bool q4 = qtype == GS_QTYPE_Q4_0 || qtype == GS_QTYPE_Q4_1;
    const bool q68 = qtype == GS_QTYPE_Q6_K || qtype == GS_QTYPE_Q8_0;
    if (rows * (cols / 64) >= (q4 ? 1ull << 29 : q68 ? 1ull << 28 : 1ull << 27)) return GS_ERR_UNSUPPORTED;
    gs_qmatrix *m = new (std::nothrow) gs_qmatrix();
    if (!m) return GS_ERR_NOMEM;
    m->qtype = qtype; m->rows = rows; m->cols = cols;
    m->np = (int)((cols + gs::kPair - 1) / gs::kPair);
    m->tiles = (int)((rows + 15) / 16);
    if (hipGetDevice(&m->device) != hipSuccess ||
        hipDeviceGetAttribute(&m->cus, hipDeviceAttributeMultiprocessorCount, m->device) != hipSuccess) {
        delete m; return GS_ERR_HIP;
    }
    if (m->cus <= 0) m->cus = 256;
    const int rc = with_format(qtype, [&](auto f) { return upload<decltype(f)>(m, (const uint8_t *)blocks); });
    if (rc != GS_OK) { if (m->base) (void)hipFree(m->base); delete m; return rc; }
    *out = m;
    return GS_OK;
}

int gs_qmatrix_destroy(gs_qmatrix *m)
{
    if (!m) return GS_ERR_INVALID;
    int dev;
    (void)hipGetDevice(&dev);
    (void)hipSetDevice(m->device);
    (void)hipDeviceSynchronize();
    (void)hipFree(m->base);
    (void)hipSetDevice(dev);
    delete m;
    return GS_OK;
}

int gs_qmatrix_shape(const gs_qmatrix *m, uint32_t *qtype, size_t *rows, size_t *cols)
{
    if (!m) return GS_ERR_INVALID;
    if (qtype) *qtype = m->qtype;
    if (rows) *rows = m->rows;
    if (cols) *cols = m->cols;
    return GS_OK;
}

int gs_gemv(const gs_qmatrix *m, const float *d_x, size_t B, float *d_out, void *stream)
{
    if (!m || (B > 0 && (!d_x || !d_out))) return GS_ERR_INVALID;
    if (((uintptr_t)d_x & 15u) != 0) return GS_ERR_INVALID;     // x is read as float4 (columns: a multiple of 32)
    // up to 16384 vectors per launch (groups of 4, or of up to 32, along the grid's y)
    for (size_t b = 0; b < B; b += 16384) {
        const int n = (int)(B - b < 16384 ? B - b : 16384);
        const int rc = with_format(m->qtype, [&](auto f) {
            return project<decltype(f)>(m, d_x + b * m->cols, d_out + b * m->rows, n, (hipStream_t)stream);
        });
        if (rc != GS_OK) return rc;
    }
    return GS_OK;
}

} // extern "C"
