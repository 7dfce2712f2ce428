// The wave64 trellis reader and the two codebooks.
//
// A packed tile holds 256 codewords in "code position" order; weight t's codeword is the 16-bit window of the tile's
// circular MSB-first bitstream that ends at bit ((t + 1) n) >> 4, n the tile's halfwords (turboexl3
// src/core/format.zig:176-222). Position p = 8 L + i maps to tile row 2 (L % 4) + {0, 1, 8, 9}[i % 4] and column
// L / 4 + 8 (i / 4) (format.zig:237-256).
//
// One wave64 reads one tile, four consecutive positions a lane ("a quad"): lane l, with c = l % 16 and g = l / 16,
// takes positions P..P+3, P = 8 (4 (c % 8) + g) + 4 (c / 8): the weights of output column c at input rows
// 2g + {0, 1, 8, 9}. That is the A fragment of v_mfma_f32_16x16x32_f16 when every weight fills a pair of K slots
// (M = column c = l % 16, K slots 8g..8g+7), so decoded registers feed the matrix core with no shuffle.
//
// A quad's four windows span at most 3n/16 + 17 bits. Up to n = 84 they fit one 32-bit register R (the 32 stream bits
// ending at the last window's end): two word loads, one v_alignbit, one v_bfe a weight (kNarrow). Wider rates read the
// first two windows from a second register ending at window 1's end: cut from the same two words where every quad's
// span lies inside them (kWidePair: n = 86..90, 96, 128), from two more words otherwise (kWide).
#pragma once

#include <type_traits>

#include "t3_common.hpp"

namespace t3 {

// format.zig Codebook's numbering, extended with the two GEMV-only forms
enum Codebook : int {
    kMul1 = 0,      // exact f16 weight, fma(f16(1024 + t), A, B)
    kMcg = 1,       // exact f16 weight, f16(lo + hi)
    kMul1Defer = 2, // h = 1024 + t as the weight; the affine map applied once an output (A acc + B sum x)
    kMcgPair = 3,   // the hashed pair (lo, hi) as two K slots: x lo + x hi, the weight never rounded to f16
};

constexpr uint32_t kMcgMult = 0xCBAC1FEDu;
constexpr uint32_t kMul1Mult = 0x83DCD12Du;

// What the vector ALU takes for the decode's operations, measured (ns of a SIMD's issue a wave64 operation, four waves a SIMD):
//   1.0      and, or, xor, right shift, add, f16 add, f32 multiply; v_bitop3 over three VECTOR registers whose second and
//            third operand have register numbers of different parity
//   1.8-1.9  v_alignbit, v_bfe, v_mul_lo_u32 (and v_mul_u32_u24: no split over the 24-bit multiplier pays), v_sad_u8,
//            sub-dword adds; v_bitop3 and the plain operations above with a scalar register among their operands, v_bitop3
//            with its second and third operand of one parity
// So where a kernel's waves are few the constants of its inner loop sit in vector registers, MCG's two in an aligned pair
// (neighbours differ in parity), and a window that ends where its register ends is cut with an and. A lane's quad of MCG
// weights, 17 operations in a row: 27.4 -> 26.4 ns of a SIMD at four waves, 36.5 -> 31.6 at one.
struct DecodeConsts {
    static constexpr bool kLean = false;
    uint2v mcg;     // the hash's mask, then its exclusive or
    uint32_t mask;  // a window's bits: (1 << wbits) - 1
};
// Where a launch's waves are many, its kernel keeps no constants: their three registers are a wave of occupancy for the routed
// GEMVs at four tiles a load (96 registers are five waves a SIMD, 98 four; 78 six, 81 five), and the adds of two weights stand by
// themselves, between other weights' operations, instead of four to a block. The other form against this one, us a routed call on
// one box: 512 experts of 2048 x 512 top-10 K3 with a shared expert at 8 / 16 rows 55.0 / 95.2 -> 53.5 / 92.7, 512 of 2560 x 640
// K4 at 8 rows 84.4 -> 82.0, 64 of 4096 x 1024 top-8 K5 at 4 / 8 rows 89.5 / 128.5 -> 85.1 / 120.8, K8 at 8 rows 143.0 -> 134.6,
// 256 of 7168 x 2048 K3 at 1 / 2 rows 72.3 / 126.6 -> 70.8 / 123.7. With few waves the other form is the faster: one row of the
// first 19.98 against 20.10, of the K5 bank 31.9 against 33.1, one dense row of 4096 x 12288 K3 12.08 against 12.23, of
// 2048 x 2048 6.28 against 6.43.
struct LeanConsts {
    static constexpr bool kLean = true;
};
template <bool LEAN = false>
__device__ __forceinline__ auto decode_consts(uint32_t wbits) {
    if constexpr (LEAN) {
        (void)wbits;
        return LeanConsts{};
    } else {
        DecodeConsts c;
        c.mcg = uint2v{0x8FFF8FFFu, 0x3B603B60u};
        c.mask = (1u << wbits) - 1u;
        asm volatile("" : "+v"(c.mcg), "+v"(c.mask));  // in vector registers, their values unknown to the compiler
        return c;
    }
}

// cw times a 32-bit constant, modulo 2^32
template <uint32_t M>
__device__ __forceinline__ uint32_t hash_mul(uint32_t cw) {
    return cw * M;
}

// MUL1's h = 0x6400 + byte sum of the hashed codeword: the f16 bit pattern of 1024 + t, t in [0, 1020]
__device__ __forceinline__ uint32_t mul1_h(uint32_t cw) {
    return __builtin_amdgcn_sad_u8(hash_mul<kMul1Mult>(cw), 0u, 0x6400u);
}
__device__ __forceinline__ uint32_t mul1_t(uint32_t cw) { return mul1_h(cw) - 0x6400u; }

// MCG's hashed pair: two f16 with fixed exponent range, sign and mantissa from the hash
__device__ __forceinline__ uint32_t mcg_pair(uint32_t cw) {
    return 0x3B603B60u ^ (hash_mul<kMcgMult>(cw) & 0x8FFF8FFFu);
}
__device__ __forceinline__ uint32_t mcg_pair(uint32_t cw, const DecodeConsts& k) {
    // (a builtin, not an asm statement: the compiler keeps the wait states before a matrix instruction reads its result)
    return __builtin_amdgcn_bitop3_b32(hash_mul<kMcgMult>(cw), k.mcg[0], k.mcg[1], 0x6A);
}

__device__ __forceinline__ uint32_t mcg_pair(uint32_t cw, const LeanConsts&) { return mcg_pair(cw); }

// Exact decoders (format.zig:149-167). MCG: both halves have exponents in [2^-3, 2^0], so their f32 sum is exact and
// one f16 add rounds as f16(f32(lo) + f32(hi)) does. MUL1: (1024 + t) A + B is a multiple of 2^-18 below 4, exact in
// f32, so one fused f16 multiply-add rounds as f16(fmaf(...)) does.
__device__ __forceinline__ uint16_t decode_mcg(uint32_t cw) {
    const uint32_t p = mcg_pair(cw);
    const _Float16 lo = __builtin_bit_cast(_Float16, static_cast<uint16_t>(p & 0xFFFFu));
    const _Float16 hi = __builtin_bit_cast(_Float16, static_cast<uint16_t>(p >> 16));
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(lo + hi));
}
__device__ __forceinline__ uint16_t decode_mul1(uint32_t cw) {
    const _Float16 h = __builtin_bit_cast(_Float16, static_cast<uint16_t>(mul1_h(cw)));
    const _Float16 a = __builtin_bit_cast(_Float16, static_cast<uint16_t>(0x1EEEu));
    const _Float16 b = __builtin_bit_cast(_Float16, static_cast<uint16_t>(0xC931u));
    return __builtin_bit_cast(uint16_t, __builtin_fmaf16(h, a, b));
}
template <int CB>
__device__ __forceinline__ uint16_t decode_exact(uint32_t cw) {
    if constexpr (CB == kMcg || CB == kMcgPair) return decode_mcg(cw);
    else return decode_mul1(cw);
}

// A weight as the GEMV's matrix core takes it where a quad fills the fragment: 32 bits = two f16 K slots (the second zero
// unless kMcgPair).
template <int CB, typename Consts>
__device__ __forceinline__ uint32_t weight_pair(uint32_t cw, const Consts& k) {
    if constexpr (CB == kMcgPair) return mcg_pair(cw, k);
    else if constexpr (CB == kMul1Defer) return mul1_h(cw);
    else return static_cast<uint32_t>(decode_exact<CB>(cw));
}

// Eight weights as an A fragment's eight f16 K slots: c0's four, then c1's. Exact, or MUL1's h = 1024 + t where its map is
// deferred.
template <int CB, typename Consts>
__device__ __forceinline__ uint4v weight_halves8(const uint32_t (&c0)[4], const uint32_t (&c1)[4], const Consts& k) {
    uint4v a;
    if constexpr (CB == kMcg) {
        // A weight is one f16 add of its hashed pair's halves, and the sub-dword forms of v_add_f16 write the low half,
        // then the high half of the same register. A sub-dword write wants one wait state before the add that keeps it
        // (two registers' adds take turns, or an s_nop) and two before a matrix instruction reads it (the s_nop at the
        // end); the compiler adds them for its own sub-dword instructions, not for these.
        uint32_t r[4];
        if constexpr (Consts::kLean) {
            // a wait state behind every add: other waves issue in it (without the second one the routed launches of
            // eight rows measured 1 to 2 % longer)
            auto two = [&](uint32_t w0, uint32_t w1) {
                uint32_t d;
                asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
                    "s_nop 0"
                    : "=v"(d)
                    : "v"(mcg_pair(w0, k)));
                asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\t"
                    "s_nop 0"
                    : "+v"(d)
                    : "v"(mcg_pair(w1, k)));
                return d;
            };
            r[0] = two(c0[0], c0[1]);
            r[1] = two(c0[2], c0[3]);
            r[2] = two(c1[0], c1[1]);
            r[3] = two(c1[2], c1[3]);
        } else {
            auto two = [&](uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t& lo, uint32_t& hi) {
                asm("v_add_f16_sdwa %0, %2, %2 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
                    "v_add_f16_sdwa %1, %4, %4 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
                    "v_add_f16_sdwa %0, %3, %3 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\t"
                    "v_add_f16_sdwa %1, %5, %5 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1"
                    : "=&v"(lo), "=&v"(hi)
                    : "v"(mcg_pair(w0, k)), "v"(mcg_pair(w1, k)), "v"(mcg_pair(w2, k)), "v"(mcg_pair(w3, k)));
            };
            two(c0[0], c0[1], c0[2], c0[3], r[0], r[1]);
            two(c1[0], c1[1], c1[2], c1[3], r[2], r[3]);
        }
        a = uint4v{r[0], r[1], r[2], r[3]};
        asm("s_nop 1" : "+v"(a));
    } else {
        // h = 0x6400 + byte sum, twice: the second sum goes to the high half of the first one's register by itself; then, the
        // map not being deferred, decode_mul1's fused multiply-add on both halves
        auto two = [](uint32_t lo, uint32_t hi) {
            const uint32_t h = __builtin_amdgcn_sad_hi_u8(hash_mul<kMul1Mult>(hi), 0u,
                                                          __builtin_amdgcn_sad_u8(hash_mul<kMul1Mult>(lo), 0u, 0x64006400u));
            if constexpr (CB == kMul1Defer) return h;
            const half2 map_a = __builtin_bit_cast(half2, 0x1EEE1EEEu), map_b = __builtin_bit_cast(half2, 0xC931C931u);
            return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2, h), map_a, map_b));
        };
        a = uint4v{two(c0[0], c0[1]), two(c0[2], c0[3]), two(c1[0], c1[1]), two(c1[2], c1[3])};
    }
    return a;
}

// ---- the quad plan --------------------------------------------------------------------------------------------

__device__ __forceinline__ uint32_t quad_first_position(uint32_t lane) {
    const uint32_t c = lane & 15u, g = lane >> 4;
    return 8u * (4u * (c & 7u) + g) + 4u * (c >> 3);
}

// How a lane reads its quad at rate n.
enum Reader : int { kNarrow = 0, kWide = 1, kWidePair = 2 };

// Whether some quad's four windows overflow one 32-bit register at rate n (host and device agree on this rule).
__host__ __device__ inline bool quad_needs_wide(uint32_t n) {
    for (uint32_t q = 0; q < 64u; ++q) {
        const uint32_t e0 = ((4u * q + 1u) * n) >> 4, e3 = ((4u * q + 4u) * n) >> 4;
        if (e3 - e0 > 16u) return true;
    }
    return false;
}
// Whether every quad's four windows lie inside the two words that hold the 32 stream bits ending at window 3's end.
__host__ __device__ inline bool quad_in_two_words(uint32_t n) {
    for (uint32_t q = 0; q < 64u; ++q) {
        const uint32_t e0 = ((4u * q + 1u) * n) >> 4, e3 = ((4u * q + 4u) * n) >> 4;
        const uint32_t w = (e3 + 16u * n - 1u) >> 5;  // one period added, as the plan does
        if (e0 + 16u * n - 16u < 32u * (w - 1u)) return false;
    }
    return true;
}
__host__ __device__ inline int quad_reader(uint32_t n) {
    return !quad_needs_wide(n) ? kNarrow : quad_in_two_words(n) ? kWidePair : kWide;
}

// Host side: call f with the rate's reader as a compile-time constant.
template <typename F>
inline auto with_reader(uint32_t n, F&& f) {
    switch (quad_reader(n)) {
        case kWide: return f(std::integral_constant<int, kWide>{});
        case kWidePair: return f(std::integral_constant<int, kWidePair>{});
        default: return f(std::integral_constant<int, kNarrow>{});
    }
}

template <int WIDE>
struct QuadPlan {
    uint32_t ib_prev, ib_last, shb;  // register B: the 32 stream bits ending at window 3's end
    uint32_t ia_prev, ia_last, sha;  // register A (wide readers): ... ending at window 1's end
    uint32_t a_low;                  // kWidePair: register A's low word is B's previous word (else B's last)
    uint32_t o[4];                   // window m's right shift inside its register
};

template <int WIDE>
__device__ __forceinline__ QuadPlan<WIDE> quad_plan(uint32_t n, uint32_t lane) {
    const uint32_t p = quad_first_position(lane);
    const uint32_t nw = n >> 1, total = 16u * n;
    uint32_t e[4];
#pragma unroll
    for (uint32_t m = 0; m < 4u; ++m) e[m] = ((p + m + 1u) * n) >> 4;
    QuadPlan<WIDE> q;
    {
        // one period added keeps the word index positive: w is in [nw, 2 nw), so the modulo is one subtraction
        const uint32_t end = e[3] + total;
        const uint32_t w = (end - 1u) >> 5;
        q.shb = 32u * (w + 1u) - end;
        q.ib_last = w - nw;
        q.ib_prev = w - 1u >= nw ? w - 1u - nw : w - 1u;
    }
    q.a_low = 0u;
    if constexpr (WIDE == kWidePair) {
        // the 64 bits {previous, last} shifted right until window 1's end is bit 0: by less than 32, one v_alignbit of
        // the pair; by 32 or more, the previous word alone (its own bits fill the top, above the two windows)
        const uint32_t sa = q.shb + (e[3] - e[1]);
        q.a_low = sa >= 32u ? 1u : 0u;
        q.sha = sa & 31u;
        q.ia_last = q.ia_prev = 0u;
        q.o[0] = e[1] - e[0];
        q.o[1] = 0u;
        q.o[2] = e[3] - e[2];
        q.o[3] = 0u;
    } else if constexpr (WIDE == kWide) {
        const uint32_t end = e[1] + total;
        const uint32_t w = (end - 1u) >> 5;
        q.sha = 32u * (w + 1u) - end;
        q.ia_last = w - nw;
        q.ia_prev = w - 1u >= nw ? w - 1u - nw : w - 1u;
        q.o[0] = e[1] - e[0];
        q.o[1] = 0u;
        q.o[2] = e[3] - e[2];
        q.o[3] = 0u;
    } else {
        q.sha = q.ia_last = q.ia_prev = 0u;
#pragma unroll
        for (uint32_t m = 0; m < 4u; ++m) q.o[m] = e[3] - e[m];
    }
    return q;
}

// The words a lane holds of one tile, loaded ahead of their use.
template <int WIDE>
struct QuadWords {
    uint32_t b_prev, b_last, a_prev, a_last;  // the a words: kWide only
};

template <int WIDE>
__device__ __forceinline__ QuadWords<WIDE> quad_load(const uint32_t* tile, const QuadPlan<WIDE>& q) {
    QuadWords<WIDE> w;
    w.b_prev = tile[q.ib_prev];
    w.b_last = tile[q.ib_last];
    if constexpr (WIDE == kWide) {
        w.a_prev = tile[q.ia_prev];
        w.a_last = tile[q.ia_last];
    } else {
        w.a_prev = w.a_last = 0u;
    }
    return w;
}

// The quad's four codewords, masked to the pack's window width `wbits` (8..16). The last window of each register ends at its
// bit 0 (o[3] = 0, and o[1] = 0 of the wide readers): an and where the others take a v_bfe, if its mask is in a register.
template <int WIDE, typename Consts>
__device__ __forceinline__ void quad_codewords(const QuadWords<WIDE>& w, const QuadPlan<WIDE>& q, uint32_t wbits,
                                               const Consts& k, uint32_t (&cw)[4]) {
    const auto last = [&](uint32_t r) -> uint32_t {
        if constexpr (Consts::kLean) return __builtin_amdgcn_ubfe(r, 0u, wbits);
        else return r & k.mask;
    };
    const uint32_t rb = __builtin_amdgcn_alignbit(w.b_prev, w.b_last, q.shb);
    uint32_t ra = rb;
    if constexpr (WIDE == kWide) ra = __builtin_amdgcn_alignbit(w.a_prev, w.a_last, q.sha);
    if constexpr (WIDE == kWidePair) ra = __builtin_amdgcn_alignbit(w.b_prev, q.a_low ? w.b_prev : w.b_last, q.sha);
    cw[0] = __builtin_amdgcn_ubfe(ra, q.o[0], wbits);
    cw[1] = WIDE == kNarrow ? __builtin_amdgcn_ubfe(ra, q.o[1], wbits) : last(ra);
    cw[2] = __builtin_amdgcn_ubfe(rb, q.o[2], wbits);
    cw[3] = last(rb);
}

// Tile row of a quad's weight m, and its column: the inverse of the permutation for one lane.
__device__ __forceinline__ uint32_t quad_row(uint32_t lane, uint32_t m) {
    return 2u * (lane >> 4) + (m & 1u) + 8u * (m >> 1);
}
__device__ __forceinline__ uint32_t quad_col(uint32_t lane) { return lane & 15u; }

}  // namespace t3
