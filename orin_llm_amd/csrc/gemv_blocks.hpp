// The block formats on the matrix cores (Q4_K, Q5_K, Q6_K, Q8_0), apart from the kernels that multiply by them
// (gemv_mfma.hip): the activation's int8 digits in LDS, and per format how a lane turns a block's
// bytes into operands of v_mfma_i32_16x16x64_i8 and the accumulator into a part of the row's sum.  gemv_mfma.hip's
// head says how the arithmetic works.
#pragma once

#include "layer_common.hpp"

namespace orin_fa {
namespace {

constexpr int kMaxWaves = 8; // waves per workgroup: 4; 8 where a matrix has few 16-row tiles and long rows; 2 or 3 where many and short ones
constexpr float kDigitRange = 8388608.0f - 65536.0f; // largest |integer| the three signed digits hold

struct XPair {
    float scale, sum; // of one sub-block of the activation
};

// LDS: digit planes [3][n_in] | XPair [n_in / G] | 16 zero bytes | partial row sums [kMaxWaves][2][16]
template <int G>
struct Lds {
    static __host__ __device__ int pairs_off(int n_in) { return 3 * n_in; }
    static __host__ __device__ int zero_off(int n_in) { return 3 * n_in + n_in / G * 8; }
    static __host__ __device__ int red_off(int n_in) { return zero_off(n_in) + 16; }
    static __host__ __device__ size_t bytes(int n_in) { return (size_t)red_off(n_in) + kMaxWaves * 2 * 16 * 4; }
};

// Eight consecutive elements (x, already multiplied by the norm's weights) of a group of G into the digit planes;
// the G / 8 threads of a group sit in one quad (n_in is a multiple of 32, so a quad is never split) and meet
// by DPP moves.
template <int G>
__device__ __forceinline__ void digits8(const float (&x)[8], int e, int n_in, unsigned char* smem, XPair* pairs, int tid) {
    float mx = 0.0f, sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        mx = fmaxf(mx, fabsf(x[i]));
        sum += x[i];
    }
    mx = fmaxf(mx, dpp_xor_step(mx, 0));
    sum += dpp_xor_step(sum, 0);
    if constexpr (G == 32) {
        mx = fmaxf(mx, dpp_xor_step(mx, 1));
        sum += dpp_xor_step(sum, 1);
    }
    // A group that holds an infinity or a NaN gets a NaN scale (sum - sum), so that every row sum it enters is NaN, as the
    // products of the vector-ALU kernel are (fmaxf above drops a NaN and the conversion would turn it into 0; the sum
    // does not lose it: a sum of floats is finite only if every term is).  The smallest normal number stands in for a
    // scale below it (a group of zeros, too): the reciprocal stays finite.  One Newton step on the hardware's
    // reciprocal: x inv scale = x to the rounding of a division.  (Divisions spelled "/" are ten instructions each, and
    // every wave of a product passes here with each of its chunks: 135 vector instructions a pass with them, 109 without.)
    const float scale = fmaxf(mx * (1.0f / kDigitRange), 1.17549435e-38f) + (sum - sum);
    float inv = __builtin_amdgcn_rcpf(scale);
    inv = __builtin_fmaf(__builtin_fmaf(-scale, inv, 1.0f), inv, inv);
    // X + 0x808080 carries 128 into each of the three byte positions, so its bytes are the signed
    // digits plus 128 (byte k of X + 0x808080 is ((X >> 8 k) + 128) & 255 with the lower digits'
    // carries already taken out); the exclusive-or takes the 128 off again, byte by byte.
    unsigned z[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = (unsigned)((int)rintf(x[i] * inv)) + 0x808080u; // (to even: most of these are halves or quarters, and halves rounded up add up over a row of weights of one sign)
    // byte k of four consecutive elements into one word of plane 2 - k (plane 0 holds the top digits)
    u32x2 plane[3];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const unsigned lo01 = __builtin_amdgcn_perm(z[4 * w + 1], z[4 * w + 0], 0x05010400u), lo23 = __builtin_amdgcn_perm(z[4 * w + 3], z[4 * w + 2], 0x05010400u); // bytes 0, 0, 1, 1 of two elements
        const unsigned hi01 = __builtin_amdgcn_perm(z[4 * w + 1], z[4 * w + 0], 0x0c0c0602u), hi23 = __builtin_amdgcn_perm(z[4 * w + 3], z[4 * w + 2], 0x0c0c0602u); // bytes 2, 2
        plane[2][w] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u) ^ 0x80808080u;
        plane[1][w] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u) ^ 0x80808080u;
        plane[0][w] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u) ^ 0x80808080u;
    }
    *reinterpret_cast<u32x2*>(smem + e) = plane[0];
    *reinterpret_cast<u32x2*>(smem + n_in + e) = plane[1];
    *reinterpret_cast<u32x2*>(smem + 2 * n_in + e) = plane[2];
    if ((tid & (G / 8 - 1)) == 0) pairs[e / G] = XPair{scale, sum};
}

// A workgroup barrier that waits for this wave's LDS traffic only: weight requests in flight stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16-byte loads of the kernels that fetch 64 bytes of each of 16 rows per instruction: ordinary ones, because the
// neighbouring pieces of a line are fetched by other instructions and meet in the CU's cache (as streaming loads,
// which pass that cache, these kernels take half as long again).  p may be 2-byte aligned.
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
__device__ __forceinline__ u32x4 load16(const unsigned char* p) { return *reinterpret_cast<const u32x4_a2*>(p); }
__device__ __forceinline__ u32x4 load16_aligned(const unsigned char* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ float half_of(unsigned bits) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits); }
__device__ __forceinline__ unsigned from_lane(int src_lane4, unsigned v) {
    return (unsigned)__builtin_amdgcn_ds_bpermute(src_lane4, (int)v);
}
// (the upper two digits' sums are put together as integers: below 2^30 for every block type, and rounded once on
// conversion where the fused multiply-add of the converted parts would round, to the same value)
__device__ __forceinline__ float digits_sum(const i32x4& acc) {
    return (float)(acc[0] * 256 + acc[1]) * 256.0f + (float)acc[2];
}
// Every byte's low nibble from a, its high nibble from b, in one instruction (as a three-input operation: of AND and OR the
// compiler, which knows which bits of b can be set, narrows the mask and then needs two).  Not as inline assembly: what
// it writes goes straight into a matrix instruction, which needs two instructions between (the compiler's business, and it does
// not see into assembly).
__device__ __forceinline__ unsigned low_nibbles_of(unsigned a, unsigned b) {
    return __builtin_amdgcn_bitop3_b32(0x0f0f0f0fu, a, b, 0xca); // first ? second : third
}
// LDS byte offset of a lane's A operand: base + x for a lane that holds digits (step 1), base (the zero bytes) for
// one whose rows are zero (step 0); x is the same in every lane.  One 24-bit multiply-add.
__device__ __forceinline__ int operand_at(int base, int step, int x) {
    return (int)(__umul24((unsigned)x, (unsigned)step) + (unsigned)base);
}
// (the step as a value the compiler knows nothing of: told that it is 0 or 1, it replaces the multiply-add by a
// move, a select and an add)
__device__ __forceinline__ int opaque_step(bool on) {
    int step = on ? 1 : 0;
    asm volatile("" : "+v"(step));
    return step;
}

// What a lane needs to know of itself: as a loader (row ln of the tile, 16-byte piece lg), as a lane of
// the matrix instruction (weight row / column n, element group g; the loader of its data is lane
// 4 n + g, whose piece is g as well), and as a lane of the A operand (accumulator row am = 4 p + digit).
struct LaneCtx {
    int n, g, ln, lg, src_lane4, am;
    const unsigned char* smem;
    const XPair* pairs;
    int n_in, zero_off;
};

template <int T>
struct MF;

// Q4_K and Q5_K (reference: src/quant.h:14-31): per 128-element half of a block, the lane's 16 bytes of
// nibbles are 16 elements of sub-block 2 (g / 2) (low nibbles) and of 2 (g / 2) + 1 (high nibbles); the two
// matrix instructions of a half add into one accumulator whose row group p is sub-block p of the half.
// Q5_K keeps a fifth bit per element in 32 bytes behind the header: bit p of byte e belongs to element e of
// sub-block p.
template <bool FIVE>
struct MFK45 {
    static constexpr int kGroup = 32, kBlockBytes = FIVE ? 176 : 144, kQs = FIVE ? 48 : 16;
    struct Raw {
        u32x4 hdr, q1, q2; // a block's header and this lane's 16 bytes of each half of its nibbles
        u32x4 qh;          // (Q5_K) the 16 bytes of fifth bits that cover this lane's elements
    };
    struct Addr {
        int lo_base, hi_base, lo_step, hi_step; // LDS byte offsets of this lane's A operands and whether they move with the block (1); a lane whose row is zero reads the 16 zero bytes (0)
    };
    static __device__ __forceinline__ void load(const unsigned char* blk, int lg, Raw& r) {
        r.hdr = load16_aligned(blk);
        if constexpr (FIVE) r.qh = load16_aligned(blk + 16 + 16 * (lg & 1));
        r.q1 = load16_aligned(blk + kQs + 16 * lg);
        r.q2 = load16_aligned(blk + kQs + 64 + 16 * lg);
    }
    static __device__ __forceinline__ Addr addr(const LaneCtx& c) {
        const int ap = c.am >> 2, ad = c.am & 3, g = c.g;
        const bool live = ad < 3 && (ap >> 1) == (g >> 1);
        const int elem = 64 * (g >> 1) + 16 * (g & 1);
        const bool lo = live && (ap & 1) == 0, hi = live && (ap & 1) == 1;
        return Addr{lo ? ad * c.n_in + elem : c.zero_off, hi ? ad * c.n_in + elem + 32 : c.zero_off, opaque_step(lo), opaque_step(hi)};
    }
    static __device__ __forceinline__ float block(const Raw& r, const LaneCtx& c, const Addr& ad, int b) {
        // (the loading lane holds piece lg of its row, and lane (n, g) wants piece g of row n: the bytes of
        // the packed pairs it needs are bytes lg of the loading lane's three words)
        const unsigned mine = ((r.hdr.y >> (8 * c.lg)) & 0xffu) | (((r.hdr.z >> (8 * c.lg)) & 0xffu) << 8) |
                              (((r.hdr.w >> (8 * c.lg)) & 0xffu) << 16);
        const unsigned dd = from_lane(c.src_lane4, r.hdr.x), bb = from_lane(c.src_lane4, mine);
        u32x4 fifth = {0u, 0u, 0u, 0u}, q1, q2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (FIVE) fifth[i] = from_lane(c.src_lane4, r.qh[i]) >> (2 * (c.g >> 1));
            q1[i] = from_lane(c.src_lane4, r.q1[i]);
            q2[i] = from_lane(c.src_lane4, r.q2[i]);
        }
        const unsigned b0 = bb & 0xffu, b1 = (bb >> 8) & 0xffu, b2 = (bb >> 16) & 0xffu;
        // pairs g (first half of the block) and 4 + g (second half) of the twelve packed bytes
        const float sc[2] = {(float)(b0 & 63u), (float)((b2 & 0x0fu) | ((b0 >> 6) << 4))};
        const float mn[2] = {(float)(b1 & 63u), (float)((b2 >> 4) | ((b1 >> 6) << 4))};
        return math(dd, sc, mn, q1, q2, fifth, [&](int h) { return digits(c, ad, b, h); });
    }
    // What half a block's product takes from the activation: A operands and sub-block pairs.
    struct Digits {
        i32x4 lo, hi;
        XPair xp;
    };
    static __device__ __forceinline__ Digits digits(const LaneCtx& c, const Addr& ad, int b, int h) {
        return Digits{*reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.lo_base, ad.lo_step, 256 * b + 128 * h)),
                      *reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.hi_base, ad.hi_step, 256 * b + 128 * h)), c.pairs[8 * b + 4 * h + c.g]};
    }
    // A block laid out in LDS piece after piece (the kernel that reads rows in long runs): piece k is the block's
    // bytes 16 k ...
    static constexpr int kPieces = kBlockBytes / 16;
    static constexpr bool kRun = false;
    static constexpr int kAlign = 16;
    static __host__ __device__ constexpr int piece_off(int k) { return 16 * k; }
    struct Words {
        u32x4 hdr, q1, q2, fifth;
    };
    static __device__ __forceinline__ Words words(const unsigned char* blk, const LaneCtx& c) {
        Words w{*reinterpret_cast<const u32x4*>(blk), *reinterpret_cast<const u32x4*>(blk + kQs + 16 * c.g),
                *reinterpret_cast<const u32x4*>(blk + kQs + 64 + 16 * c.g), u32x4{0u, 0u, 0u, 0u}};
        if constexpr (FIVE) w.fifth = *reinterpret_cast<const u32x4*>(blk + 16 + 16 * (c.g & 1));
        return w;
    }
    // `of_half`(h): the digits of half h
    template <typename X>
    static __device__ __forceinline__ float product(const Words& w, const X& of_half, const LaneCtx& c) {
        // the six-bit pairs straight out of the three words (bit fields at 8 g: no byte is put together first)
        const unsigned s8 = 8 * c.g;
        const float sc[2] = {(float)__builtin_amdgcn_ubfe(w.hdr.y, s8, 6), (float)(__builtin_amdgcn_ubfe(w.hdr.w, s8, 4) | ((w.hdr.y >> (s8 + 2)) & 0x30u))};
        const float mn[2] = {(float)__builtin_amdgcn_ubfe(w.hdr.z, s8, 6), (float)(__builtin_amdgcn_ubfe(w.hdr.w, s8 + 4, 4) | ((w.hdr.z >> (s8 + 2)) & 0x30u))};
        return math(w.hdr.x, sc, mn, w.q1, w.q2, FIVE ? w.fifth >> (unsigned)(2 * (c.g >> 1)) : w.fifth, of_half);
    }
    template <typename X>
    static __device__ __forceinline__ float from_lds(const unsigned char* blk, const X& of_half, const LaneCtx& c) { return product(words(blk, c), of_half, c); }
    // In lane (n, g): dd = the block's two fp16 scales, sc / mn = the six-bit scales and minima of sub-blocks g (first
    // half of the block) and 4 + g (second half), q1 / q2 = piece g of each half of the nibbles, fifth = the fifth
    // bits of this lane's elements shifted down to bit 0 (Q5_K).
    template <typename X>
    static __device__ __forceinline__ float math(unsigned dd, const float (&sc)[2], const float (&mn)[2], const u32x4& q1, const u32x4& q2,
                                                 const u32x4& fifth, const X& of_half) {
        const float d = half_of(dd & 0xffffu), dmin = half_of(dd >> 16);
        float scaled[2], offset[2]; // sum of sc * q * x and of mn * x over a sub-block pair; the block's two scales come last
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const Digits x = of_half(h);
            const u32x4 qs = h ? q2 : q1;
            i32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned q = qs[i];
                unsigned l = q & 0x0f0f0f0fu, u = (q >> 4) & 0x0f0f0f0fu;
                if constexpr (FIVE) { // sub-blocks 4 h + 2 (g / 2) and + 1: bits 4 h and 4 h + 1 of the shifted bytes
                    const unsigned f = fifth[i] >> (4 * h);
                    l |= (f & 0x01010101u) << 4;
                    u |= (f & 0x02020202u) << 3;
                }
                lo[i] = (int)l;
                hi[i] = (int)u;
            }
            i32x4 acc = {0, 0, 0, 0};
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.lo, lo, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.hi, hi, acc, 0, 0, 0);
            scaled[h] = sc[h] * (digits_sum(acc) * x.xp.scale);
            offset[h] = mn[h] * x.xp.sum;
        }
        return d * (scaled[0] + scaled[1]) - dmin * (offset[0] + offset[1]);
    }
};
template <>
struct MF<kQ4_K> : MFK45<false> {};
template <>
struct MF<kQ5_K> : MFK45<true> {};

// Q8_0 (reference: src/quant.h:42-45; blocks of 34 bytes, 2-byte aligned): eight blocks make up the 256
// elements the kernel walks at a time.  Per 128-element half, the lane's 16 bytes are half of block
// 2 run + g / 2 of the half, for run = 0, 1: one matrix instruction per run, both adding into one accumulator
// whose row group p is block p of the half.
template <>
struct MF<kQ8_0> {
    static constexpr int kGroup = 32, kBlockBytes = 272;
    struct Raw {
        u32x4 q[2][2]; // [half][run]
        unsigned d[2]; // scales of blocks lg and 4 + lg
    };
    typedef MFK45<false>::Addr Addr;
    template <typename V>
    struct __attribute__((packed, aligned(2))) Loose {
        V v;
    };
    static __device__ __forceinline__ void load(const unsigned char* blk, int lg, Raw& r) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int run = 0; run < 2; ++run)
                r.q[h][run] = load16(blk + 34 * (4 * h + 2 * run + (lg >> 1)) + 2 + 16 * (lg & 1));
            r.d[h] = *reinterpret_cast<const uint16_t*>(blk + 34 * (4 * h + lg));
        }
    }
    static __device__ __forceinline__ Addr addr(const LaneCtx& c) {
        const int ap = c.am >> 2, ad = c.am & 3, g = c.g;
        const bool live = ad < 3 && (ap & 1) == (g >> 1);
        const int elem = 32 * ap + 16 * (g & 1);
        const bool r0 = live && (ap >> 1) == 0, r1 = live && (ap >> 1) == 1;
        return Addr{r0 ? ad * c.n_in + elem : c.zero_off, r1 ? ad * c.n_in + elem : c.zero_off, opaque_step(r0), opaque_step(r1)};
    }
    static __device__ __forceinline__ float block(const Raw& r, const LaneCtx& c, const Addr& ad, int b) {
        float out[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const i32x4 a0 = *reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.lo_base, ad.lo_step, 256 * b + 128 * h));
            const i32x4 a1 = *reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.hi_base, ad.hi_step, 256 * b + 128 * h));
            const XPair xp = c.pairs[8 * b + 4 * h + c.g];
            const float d = half_of(from_lane(c.src_lane4, r.d[h]));
            i32x4 w0, w1;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                w0[i] = (int)from_lane(c.src_lane4, r.q[h][0][i]);
                w1[i] = (int)from_lane(c.src_lane4, r.q[h][1][i]);
            }
            i32x4 acc = {0, 0, 0, 0};
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, w0, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, w1, acc, 0, 0, 0);
            out[h] = d * (digits_sum(acc) * xp.scale);
        }
        return out[0] + out[1];
    }
    // 256 elements laid out in LDS as they are in memory: eight blocks of 34 bytes are seventeen whole 16-byte pieces (a
    // matrix whose base is 16-byte aligned has only such pieces).  A lane's 16 weights start 2 bytes off a word in the
    // even blocks: five words and a byte shift that is the same for every block a lane reads.
    static constexpr int kPieces = 17;
    static constexpr bool kRun = false;
    static constexpr int kAlign = 16;
    static __host__ __device__ constexpr int piece_off(int k) { return 16 * k; }
    struct Digits {
        i32x4 a[2]; // of the runs
        XPair xp;
    };
    static __device__ __forceinline__ Digits digits(const LaneCtx& c, const Addr& ad, int b, int h) {
        return Digits{{*reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.lo_base, ad.lo_step, 256 * b + 128 * h)),
                       *reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.hi_base, ad.hi_step, 256 * b + 128 * h))}, c.pairs[8 * b + 4 * h + c.g]};
    }
    struct HalfWords {
        unsigned v[2][5]; // of the runs
        uint16_t d;
    };
    struct Words {
        HalfWords half[2];
    };
    static __device__ __forceinline__ HalfWords half_words(const unsigned char* blk, const LaneCtx& c, int h) {
        const unsigned char* const mine = blk + 34 * (c.g >> 1) + 2 + 16 * (c.g & 1) - (c.g < 2 ? 2u : 0u); // (word aligned)
        HalfWords w;
        w.d = *reinterpret_cast<const uint16_t*>(blk + 34 * (4 * h + c.g));
#pragma unroll
        for (int run = 0; run < 2; ++run)
#pragma unroll
            for (int i = 0; i < 5; ++i) w.v[run][i] = reinterpret_cast<const unsigned*>(mine + 34 * (4 * h + 2 * run))[i];
        return w;
    }
    static __device__ __forceinline__ Words words(const unsigned char* blk, const LaneCtx& c) { return Words{{half_words(blk, c, 0), half_words(blk, c, 1)}}; }
    static __device__ __forceinline__ float half_product(const HalfWords& words, const Digits& x, const LaneCtx& c) {
        const unsigned shift = c.g < 2 ? 2u : 0u;
        i32x4 w[2], acc = {0, 0, 0, 0};
#pragma unroll
        for (int run = 0; run < 2; ++run) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[run][i] = (int)__builtin_amdgcn_alignbyte(words.v[run][i + 1], words.v[run][i], shift);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.a[run], w[run], acc, 0, 0, 0);
        }
        return half_of(words.d) * (digits_sum(acc) * x.xp.scale);
    }
    // `of_half`(h): the digits of half h
    template <typename X>
    static __device__ __forceinline__ float product(const Words& w, const X& of_half, const LaneCtx& c) {
        return half_product(w.half[0], of_half(0), c) + half_product(w.half[1], of_half(1), c);
    }
    template <typename X>
    static __device__ __forceinline__ float from_lds(const unsigned char* blk, const X& of_half, const LaneCtx& c) {
        float out[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const Digits x = of_half(h);
            out[h] = half_product(half_words(blk, c, h), x, c);
        }
        return out[0] + out[1];
    }
};

// Q6_K (reference: src/quant.h:34-40; blocks of 210 bytes, 2-byte aligned): per 128-element half, piece g
// of the half's 64 low-nibble bytes holds sub-block g (elements 16 g .. 16 g + 15 of the half) in its low
// nibbles and sub-block 4 + g in its high nibbles; their high bit pairs sit in high byte 16 (g & 1) + i at
// bits 2 (g / 2) and 4 + 2 (g / 2).  One matrix instruction and one accumulator per nibble; the element
// group g of the instruction is sub-block g (or 4 + g), so the A operand's row group p is live in group p.
template <>
struct MF<kQ6_K> {
    static constexpr int kGroup = 16, kBlockBytes = 210;
    struct Raw {
        u32x4 ql[2], qh[2], sc;
        unsigned d;
    };
    struct Addr {
        int base, step;
    };
    template <typename V>
    struct __attribute__((packed, aligned(2))) Loose {
        V v;
    };
    static __device__ __forceinline__ void load(const unsigned char* blk, int lg, Raw& r) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            r.ql[h] = load16(blk + 64 * h + 16 * lg);
            r.qh[h] = load16(blk + 128 + 32 * h + 16 * (lg & 1));
        }
        r.sc = load16(blk + 192);
        r.d = *reinterpret_cast<const uint16_t*>(blk + 208);
    }
    static __device__ __forceinline__ Addr addr(const LaneCtx& c) {
        const int ap = c.am >> 2, ad = c.am & 3;
        const bool live = ad < 3 && ap == c.g;
        return Addr{live ? ad * c.n_in + 16 * c.g : c.zero_off, opaque_step(live)};
    }
    static __device__ __forceinline__ float block(const Raw& r, const LaneCtx& c, const Addr& ad, int b) {
        // scales 8 h + g and 8 h + 4 + g of both halves: byte lg of each of the loading lane's four words
        const unsigned mine = ((r.sc.x >> (8 * c.lg)) & 0xffu) | (((r.sc.y >> (8 * c.lg)) & 0xffu) << 8) |
                              (((r.sc.z >> (8 * c.lg)) & 0xffu) << 16) | (((r.sc.w >> (8 * c.lg)) & 0xffu) << 24);
        const unsigned ss = from_lane(c.src_lane4, mine);
        const unsigned dd = from_lane(c.src_lane4, r.d);
        u32x4 ql[2], qh[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ql[h][i] = from_lane(c.src_lane4, r.ql[h][i]);
                qh[h][i] = from_lane(c.src_lane4, r.qh[h][i]);
            }
        }
        const int sc[4] = {(int)(ss << 24) >> 24, (int)(ss << 16) >> 24, (int)(ss << 8) >> 24, (int)ss >> 24};
        return math(sc, dd, ql, qh, c, [&](int h) { return digits(c, ad, b, h); });
    }
    // A block laid out in LDS piece after piece (the kernel that reads rows in long runs): pieces 0 ... 12 are the
    // block's bytes 16 k ..., piece 13 its last 16 bytes (194 ... 209: the fp16 scale in its last two), so that no
    // piece reaches past the block.
    static constexpr int kPieces = 14;
    static constexpr bool kRun = false;
    static constexpr int kAlign = 2;
    static __host__ __device__ constexpr int piece_off(int k) { return k < 13 ? 16 * k : 194; }
    struct Words {
        u32x4 ql[2], qh[2];
        int sc[4];
        unsigned d;
    };
    static __device__ __forceinline__ Words words(const unsigned char* blk, const LaneCtx& c) {
        Words w;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w.ql[h] = *reinterpret_cast<const u32x4*>(blk + 64 * h + 16 * c.g);
            w.qh[h] = *reinterpret_cast<const u32x4*>(blk + 128 + 32 * h + 16 * (c.g & 1));
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) w.sc[k] = reinterpret_cast<const signed char*>(blk)[192 + 4 * k + c.g];
        w.d = *reinterpret_cast<const unsigned*>(blk + 13 * 16 + 12) >> 16;
        return w;
    }
    struct Digits {
        i32x4 lo, hi;
        XPair xlo, xhi;
    };
    static __device__ __forceinline__ Digits digits(const LaneCtx& c, const Addr& ad, int b, int h) {
        return Digits{*reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.base, ad.step, 256 * b + 128 * h)),
                      *reinterpret_cast<const i32x4*>(c.smem + operand_at(ad.base, ad.step, 256 * b + 128 * h + 64)),
                      c.pairs[16 * b + 8 * h + c.g], c.pairs[16 * b + 8 * h + 4 + c.g]};
    }
    template <typename X>
    static __device__ __forceinline__ float product(const Words& w, const X& of_half, const LaneCtx& c) { return math(w.sc, w.d, w.ql, w.qh, c, of_half); }
    template <typename X>
    static __device__ __forceinline__ float from_lds(const unsigned char* blk, const X& of_half, const LaneCtx& c) { return product(words(blk, c), of_half, c); }
    // In lane (n, g): sc = the scales g, 4 + g, 8 + g and 12 + g, dd = the block's fp16 scale, ql / qh = piece g of each half's low nibbles and the piece of high bit pairs that covers it.
    template <typename X>
    static __device__ __forceinline__ float math(const int (&sc)[4], unsigned dd, const u32x4 (&ql)[2], const u32x4 (&qh)[2], const LaneCtx& c,
                                                 const X& of_half) {
        const float d = half_of(dd & 0xffffu);
        const int s1 = 2 * (c.g >> 1);
        float out[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const Digits x = of_half(h);
            i32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // u: this lane's two bit pairs of every byte at bits 0, 1 and 4, 5, nothing else; each lands in the
                // high nibble of its element by one bit-field insert
                const unsigned l = ql[h][i], u = (qh[h][i] >> s1) & 0x33333333u;
                lo[i] = (int)low_nibbles_of(l, u << 4);
                hi[i] = (int)low_nibbles_of(l >> 4, u);
            }
            const i32x4 zero = {0, 0, 0, 0};
            const i32x4 acc_lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.lo, lo, zero, 0, 0, 0);
            const i32x4 acc_hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.hi, hi, zero, 0, 0, 0);
            const float sc_lo = (float)sc[2 * h], sc_hi = (float)sc[2 * h + 1];
            out[h] = sc_lo * (digits_sum(acc_lo) * x.xlo.scale - 32.0f * x.xlo.sum) + sc_hi * (digits_sum(acc_hi) * x.xhi.scale - 32.0f * x.xhi.sum);
        }
        return d * (out[0] + out[1]);
    }
};

// Q6_K read in runs of two blocks that start on a word: 420 bytes are 27 pieces one behind the other, the last of them the run's
// last sixteen bytes.  A block fetched as pieces of its own starts on a word only every other time, and its last piece overlaps the one
// before: reads alone (48 MB) 10.25 us against 9.2, and 43.3 against 38.6 over 255 MB, as fast as 16-byte aligned ones.
// For rows of an even number of blocks, cut (shares, chunks) at even blocks, and a matrix that starts on a word.  Per launch, the same
// matrix two bytes off a word (block by block) and on one (in runs): down projection of Qwen2.5-7B 15.1 and 12.9 us (55.7 MB, 4.3
// TB/s), Llama-3-8B 13.0 and 11.7, its logits 80.3 and 71.8 (6.0 TB/s), Llama-3.2-1B's 42.9 and 37.1, Qwen2.5-7B's gate/up 26.6 and 23.8.
// In LDS the run lies as it does in memory: block 1 starts two bytes into a piece, and a lane's sixteen bytes there are that
// piece and the word behind it, shifted down (LDS takes 64 clocks for wide reads off their alignment, 9 on it).
constexpr int kQ6_KRun = 0x100 + kQ6_K;
template <>
struct MF<kQ6_KRun> : MF<kQ6_K> {
    static constexpr bool kRun = true;
    static constexpr int kAlign = 4, kRunBytes = 2 * kBlockBytes, kRunPieces = (kRunBytes + 15) / 16, kLastPiece = kRunBytes - 16;
    template <int J>
    static __device__ __forceinline__ Words run_words(const unsigned char* row, const LaneCtx& c) {
        constexpr int kShift = J * kBlockBytes % 16, kFloor = J * kBlockBytes - kShift;
        auto piece = [&](int off) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(row + kFloor + off);
            if constexpr (kShift == 0) {
                return v;
            } else {
                const unsigned behind = *reinterpret_cast<const unsigned*>(row + kFloor + off + 16);
                return u32x4{__builtin_amdgcn_alignbyte(v[1], v[0], kShift), __builtin_amdgcn_alignbyte(v[2], v[1], kShift),
                             __builtin_amdgcn_alignbyte(v[3], v[2], kShift), __builtin_amdgcn_alignbyte(behind, v[3], kShift)};
            }
        };
        Words w;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w.ql[h] = piece(64 * h + 16 * c.g);
            w.qh[h] = piece(128 + 32 * h + 16 * (c.g & 1));
        }
        // (what lies behind the run's last whole piece is in the last one, further on by as much as that overlaps)
        constexpr int kWhole = kRunBytes / 16 * 16, kOn = kWhole - kLastPiece;
        const int lane_on = J == 1 && c.g >= 2 ? kOn : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            static_assert(kBlockBytes + 192 + 4 * 2 + 3 < kWhole && kBlockBytes + 192 + 4 * 3 + 1 < kWhole && kBlockBytes + 192 + 4 * 3 + 2 >= kWhole, "scales 14 and 15 of block 1");
            w.sc[k] = reinterpret_cast<const signed char*>(row)[J * kBlockBytes + 192 + 4 * k + c.g + (k == 3 ? lane_on : 0)];
        }
        w.d = *reinterpret_cast<const uint16_t*>(row + J * kBlockBytes + 208 + (J == 1 ? kOn : 0));
        return w;
    }
};

// Rows read in long runs (gemv_mfma.hip, gemv_rows_kernel): an item is CB <= 2 consecutive blocks of each of 16 rows, in
// LDS piece after piece with rows padded to an odd number of pieces.
constexpr int kRowsMaxCb = 2; // blocks of a row in an item, at most
constexpr int kRowsRedBytes = 2 * kMaxWaves * 2 * 16 * 4 + 64; // two sets of partial row sums (tiles alternate: one barrier a tile), the waves' sums of squares

template <int T, int CB>
struct RowsGeom {
    static constexpr int P = MF<T>::kPieces;                 // pieces of a block
    static constexpr bool kRun = MF<T>::kRun;
    static_assert(!kRun || CB == 2, "runs of two blocks");
    static constexpr int kRowPieces = kRun ? (2 * MF<T>::kBlockBytes + 15) / 16 : CB * P; // pieces of a row in an item
    static constexpr int kUnit = kRun ? 2 : 1;               // blocks that stay together where a row is cut into shares
    static constexpr int R = kRowPieces | 1;                 // LDS row stride, pieces
    static constexpr int NL = (16 * kRowPieces + 63) / 64;   // load instructions an item
    static constexpr int kWaveBytes = (16 * R + 1) * 16;     // (one more piece: where lanes past the item's end write)
    static __host__ __device__ size_t lds_bytes(int n_in, int waves) {
        return (size_t)Lds<MF<T>::kGroup>::red_off(n_in) + kRowsRedBytes + (size_t)waves * kWaveBytes;
    }
};

} // namespace
} // namespace orin_fa
