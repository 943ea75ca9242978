// math.hpp - per-element integer arithmetic of the Ozaki Scheme II path,
// shared by the gfx950 kernels and by the host build used to test it on the
// CPU (csrc/test/emu.cpp).  Everything here is exact integer work except the
// fixed-point CRT quotient estimate, whose error is bounded far below its margin.
#pragma once
#include <cstdint>
#include <type_traits>

#include "plan.hpp"

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define OZ2_HD __host__ __device__ __forceinline__
#define OZ2_UNROLL _Pragma("unroll")
#else
#include <cmath>
#define OZ2_HD inline
#define OZ2_UNROLL
#endif

namespace oz2 {
namespace math {

// The functions below take the constant tables as a pointer of any type with
// TabSet's members.  Kernels pass const_tab(p): loads through an address-space-4
// (constant) pointer compile to scalar loads even where the kernel also stores
// through pointers that could alias the tables (int8 planes, byte residues).
#if defined(__HIPCC__)
using ConstTab = const __attribute__((address_space(4))) TabSet*;
__device__ __forceinline__ ConstTab const_tab(const TabSet* p) { return (ConstTab)p; }
#endif

#if defined(__HIP_DEVICE_COMPILE__)
// The LLVM intrinsics behind v_mul_hi_u32_u24 and v_mul_i32_i24 (no clang builtin names
// them).  Called directly they take the low 24 bits of each operand themselves, so no
// masking instructions are emitted, and the optimizer cannot turn a 24-bit product whose
// low bits alone are used into a full 32- or 64-bit multiply (quarter rate).
extern "C" __device__ uint32_t oz2_llvm_mulhi_u24(uint32_t, uint32_t) __asm("llvm.amdgcn.mulhi.u24");
extern "C" __device__ int32_t oz2_llvm_mul_i24(int32_t, int32_t) __asm("llvm.amdgcn.mul.i24");
#endif

// v_mad_i32_i24: a * b + c with a, b sign-extended from 24 bits (low 32 bits of the result)
OZ2_HD uint32_t mad_i24(int32_t a, int32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return static_cast<uint32_t>(oz2_llvm_mul_i24(a, b)) + c;
#else
    const int64_t sa = static_cast<int64_t>(static_cast<uint64_t>(a) << 40) >> 40;
    const int64_t sb = static_cast<int64_t>(static_cast<uint64_t>(b) << 40) >> 40;
    return static_cast<uint32_t>(static_cast<uint64_t>(sa * sb)) + c;
#endif
}
// v_mul_hi_u32_u24: high 16 bits of a 24 x 24-bit product
OZ2_HD uint32_t mulhi24(uint32_t a, uint32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return oz2_llvm_mulhi_u24(a, b);
#else
    return static_cast<uint32_t>((static_cast<uint64_t>(a & 0xFFFFFFu) * static_cast<uint64_t>(b & 0xFFFFFFu)) >> 32);
#endif
}

// v_mul_hi_u32
OZ2_HD uint32_t mulhi32(uint32_t a, uint32_t b) { return static_cast<uint32_t>((static_cast<uint64_t>(a) * b) >> 32); }

// v_dot2_u32_u16: c + a.lo * b.lo + a.hi * b.hi (16-bit halves, no clamping)
OZ2_HD uint32_t udot2(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_udot2(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b), c, false);
#else
    return c + (a & 0xFFFFu) * (b & 0xFFFFu) + (a >> 16) * (b >> 16);
#endif
}

// v_dot4_u32_u8: c + the sum of the four byte products (no clamping)
OZ2_HD uint32_t udot4(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_udot4(a, b, c, false);
#else
    for (int i = 0; i < 32; i += 8) c += ((a >> i) & 0xFFu) * ((b >> i) & 0xFFu);
    return c;
#endif
}

OZ2_HD int clz32(uint32_t x) { return x ? __builtin_clz(x) : 32; }
OZ2_HD int clz64(uint64_t x) { return x ? __builtin_clzll(x) : 64; }

// frexp exponent of a positive finite double given by its bit pattern (bits != 0)
OZ2_HD int frexp_exp_bits(uint64_t b) {
    const int bexp = static_cast<int>(b >> 52);
    if (bexp) return bexp - 1022;
    return (64 - clz64(b & 0xFFFFFFFFFFFFFull)) - 1074;
}

// exponent rule of the scaling step (hpp:360-377): 0 for an all-zero row,
// kNonFinite for Inf/NaN (bit patterns >= the infinity pattern), else tk - frexp_exp(max)
OZ2_HD int32_t exponent_from_maxbits(uint64_t b, int tk) {
    if (b >= 0x7FF0000000000000ull) return INT32_MIN;
    if (b == 0) return 0;
    return tk - frexp_exp_bits(b);
}

OZ2_HD double ldexp_(double v, int e) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ldexp(v, e);
#else
    return std::ldexp(v, e);
#endif
}

// RNE(|v| * 2^e) for |v * 2^e| < 2^62 (narrow values) in straight-line code: the
// mantissa moves left by max(sh, 0) and right by min(max(-sh, 0), 63) with the
// round-to-nearest-even increment rem + lsb > half (half = 2^(rs-1); none if rs = 0).
OZ2_HD uint64_t scaled_mag62(uint64_t bits, int e) {
    const int bexp = static_cast<int>((bits >> 52) & 0x7FF);
    const uint64_t mant = (bits & 0xFFFFFFFFFFFFFull) | (bexp ? 0x10000000000000ull : 0);
    const int sh = (bexp ? bexp : 1) - 1075 + e;
    const int ls = sh > 0 ? sh : 0;
    const int rs = sh < 0 ? (-sh < 63 ? -sh : 63) : 0;
    const uint64_t up = mant << ls;
    const uint64_t q = up >> rs;
    const uint64_t rem = up & ((1ull << rs) - 1);
    const uint64_t half = rs ? (1ull << (rs - 1)) : ~0ull;
    return q + (rem + (q & 1) > half ? 1 : 0);
}

// Words of x = RNE(v 2^e) in base 2^31, x = sum_w (a[w] - 2^31) 2^(31 w): the residue chain takes one v_dot4 a word
//   Words2  two words, |x| <= 2^61;   Words3  three, |x| <= 2^92 (every plan has tk <= 91);
//   Words4  four, |x| <= 2^100.
enum class Limbs { Words2, Words3, Words4 };
template <Limbs F>
inline constexpr int kLimbWords = F == Limbs::Words2 ? 2 : F == Limbs::Words3 ? 3 : 4;

// Adding 1.5 2^52 + 2^31 units of 2^(31 w) leaves word w, rounded to nearest, in the low half of the sum's bits;
// subtracting that is exact, and the remainder of at most half a unit goes to the next word.  So the top word is
// at most 2^30 from 2^31 and the others too, none wraps, and the last sum is the rounding to nearest even, ties
// included (the words above are even).  Subnormal v scale exactly; what vanishes below 2^-1074 rounds to 0.
// 8 instructions an element for three words; with shifts and masks of the mantissa in 64-bit halves it was about
// 60, and 35 for two words.  With sym_float, split on MI355X, us: 2048 x 200000 by 200000 x 2048 s = 24 5380 ->
// 5215, 256 products of 64 .. 4096 with 17 to 24 moduli 1882 -> 1712, 1024^3 s = 14 14.7 -> 11.9, 1537 x 771 x
// 3001 s = 15 36.6 -> 31.5, complex 4096^2 twice s = 16 510 -> 454, complex 777 x 1023 x 515 39 -> 23.
// zero: the element is outside the matrix or its row is non-finite, giving x = 0.
template <Limbs F>
OZ2_HD void to_limbs(uint64_t bits, int e, bool zero, uint32_t (&a)[4]) {
    double y = ldexp_(__builtin_bit_cast(double, zero ? uint64_t{0} : bits), e);
    OZ2_UNROLL
    for (int w = kLimbWords<F> - 1; w >= 0; --w) {
        const double c = (6755399441055744.0 + 2147483648.0) * (w > 2 ? 0x1p93 : w > 1 ? 0x1p62 : w > 0 ? 0x1p31 : 1.0);
        const double t = y + c;
        a[w] = static_cast<uint32_t>(__builtin_bit_cast(uint64_t, t));
        y -= t - c;
    }
}

// Exact quotient by a modulus 129 <= m <= 255 for 0 <= v < 2^23: with mu = ceil(2^31 / m)
// (< 2^24) and e = mu m - 2^31 in [0, m), v mu / 2^31 = v/m + v e / (m 2^31), and
// v e < 2^23 * 255 < 2^31 keeps the excess below 1/m, so q = mulhi24(2v, mu) =
// floor(v mu / 2^31) = floor(v/m) and v - q m (one v_mad_i32_i24) is v mod m.
OZ2_HD uint32_t mod_m23(uint32_t v, uint32_t m, uint32_t mu) {
    const uint32_t q = mulhi24(v + v, mu);
    return mad_i24(static_cast<int32_t>(q), -static_cast<int32_t>(m), v);
}

// (v mod m) - h for w = v - h (mod 2^32), v < 2^23: the exact quotient of v = w + h
// takes (w << 1) + 2h (one v_lshl_add_u32) and w - q m = (v mod m) - h needs no
// separate subtraction of h.
OZ2_HD uint32_t sym_m23(uint32_t w, uint32_t m, uint32_t mu, uint32_t h2) {
    const uint32_t q = mulhi24((w << 1) + h2, mu);
    return mad_i24(static_cast<int32_t>(q), -static_cast<int32_t>(m), w);
}

OZ2_HD float as_float(uint32_t x) { return __builtin_bit_cast(float, x); }
// Low byte: v - m round(v / m), the symmetric residue of v, for F = v + B (B = TabSet::fb) as the bits of a float
// in [2^23, 2^24): F is 2^23 ulps up, so a chain of integer additions that starts at the bits of B's float leaves
// the float itself.  One fma with 1.5 2^23 rounds F / m to the integer in its low bits.  B is a multiple of m;
// F 2^-24 / m is up to half the distance of a quotient from its tie, so whether rounding 1/m to a float moves a
// quotient over one depends on m: for the moduli in use none of the chains' values does (all checked in the tests)
// except with m = 255, which takes sym_m23.  The high byte of the fma's bits does not enter, 2^22 m and 2^23 are
// multiples of 256.
OZ2_HD uint32_t sym_float(uint32_t F, uint32_t m, float rm) {
    const uint32_t q = __builtin_bit_cast(uint32_t, __builtin_fmaf(as_float(F), rm, 12582912.0f));
    return mad_i24(static_cast<int32_t>(q), -static_cast<int32_t>(m), F);
}

// Chain of x's words for modulus index t from `start`: start + sum over the words' bytes of byte (2^(31 w + 8 j) mod m)
template <Limbs F, typename Tab>
OZ2_HD uint32_t word_chain(const uint32_t (&a)[4], Tab tb, int t, uint32_t start) {
    uint32_t w = udot4(a[0], tb->c8[t][0], start);
    w = udot4(a[1], tb->c8[t][1], w);
    if (kLimbWords<F> > 2) w = udot4(a[2], tb->c8[t][2], w);
    if (kLimbWords<F> > 3) w = udot4(a[3], tb->c8[t][3], w);
    return w;
}

// Symmetric residues (low byte) of x, of y and of x + y for modulus index t >= 1 (m <= 255).
//   EXACT, t = 1 (m = 255 in the sets of up to six moduli) and four words: w = v - h by sym_m23 with v = x + h (mod m), v < 2^20;
//   else sym_float: one instruction less, also for the sum.
template <Limbs F>
inline constexpr bool kFloatResidues = F != Limbs::Words4;
template <Limbs F, bool EXACT, typename Tab>
OZ2_HD uint32_t sym_residue(const uint32_t (&a)[4], Tab tb, int t) {
    constexpr int f = static_cast<int>(F);
    if (EXACT) return sym_m23(word_chain<F>(a, tb, t, tb->offh[f][t]), tb->m[t], tb->mu[t], tb->h2[t]);
    return sym_float(word_chain<F>(a, tb, t, tb->fstart[f][t]), tb->m[t], tb->rm[t]);
}
template <Limbs F, bool EXACT, typename Tab>
OZ2_HD void sym_residues(const uint32_t (&a)[4], const uint32_t (&b)[4], Tab tb, int t, uint32_t (&out)[3]) {
    constexpr int f = static_cast<int>(F);
    const uint32_t m = tb->m[t];
    if (EXACT) {
        const uint32_t mu = tb->mu[t], h2 = tb->h2[t];
        out[0] = sym_m23(word_chain<F>(a, tb, t, tb->offh[f][t]), m, mu, h2);
        out[1] = sym_m23(word_chain<F>(b, tb, t, tb->offh[f][t]), m, mu, h2);
        out[2] = sym_m23(out[0] + out[1] + m, m, mu, h2);  // both in [-h, h]: v = the sum + m + h > 0
        return;
    }
    const uint32_t x = word_chain<F>(a, tb, t, tb->fstart[f][t]), y = word_chain<F>(b, tb, t, tb->fstart[f][t]);
    const float rm = tb->rm[t];
    out[0] = sym_float(x, m, rm);
    out[1] = sym_float(y, m, rm);
    out[2] = sym_float(x + y - tb->fb[t], m, rm);
}

// The moduli t0 .. t1 - 1 of a split, by the form of their residues: low() for t = 0 (m = 256: the words' units are
// multiples of it, the low byte of word 0 is the residue), plane(t, exact) for the others (sym_residue).
template <Limbs F, typename Low, typename Plane>
OZ2_HD void for_moduli(int t0, int t1, const Low& low, const Plane& plane) {
    if (t0 == 0) low();
    if (t0 <= 1 && t1 > 1) plane(1, std::true_type{});
    for (int t = t0 > 2 ? t0 : 2; t < t1; ++t) plane(t, std::bool_constant<!kFloatResidues<F>>{});
}

// the low bytes of b0..b3 packed into one word (b0 lowest): two v_perm_b32 (each
// takes byte 0 of two registers) and an or
OZ2_HD uint32_t pack_lo_bytes(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
#if defined(__HIP_DEVICE_COMPILE__)
    // v_perm_b32 D, S0, S1, sel: selector byte values 0-3 pick bytes of S1, 4-7 bytes of S0, 0x0c gives 0
    return __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u) | __builtin_amdgcn_perm(b3, b2, 0x04000c0cu);
#else
    return (b0 & 0xFFu) | (b1 & 0xFFu) << 8 | (b2 & 0xFFu) << 16 | (b3 & 0xFFu) << 24;
#endif
}

// the low halves of a and b in one word (a lowest)
OZ2_HD uint32_t pack_lo_halves(uint32_t a, uint32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_perm(b, a, 0x05040100u);
#else
    return (a & 0xFFFFu) | b << 16;
#endif
}

// GEMM epilogue: int32 dot product x of one k-chunk -> x mod m in [0, m), m <= 255.  A chunk holds at most
// kMaxKChunk = 65408 k, so |x| <= 65408 * 2^14 <= 2^30 - 2^21, and with c30 = m ceil(2^30 / m) in
// [2^30, 2^30 + m) the value u = x + c30 lies in [0, 2^31) and keeps x's residue; the sums start at c30, so u
// is what the matrix cores leave.  With mg = ceil(2^39 / m), u mg / 2^39 = u/m + u e / (m 2^39), e < m < 2^8:
// the excess stays below 1/m, so q = floor(u mg / 2^39) = floor(u/m).  q may exceed 23 bits, so only the low
// byte of the returned word is u - q m.  m = 256 has mg = c30 = 0: the low byte of x.
OZ2_HD uint32_t residue_word(uint32_t u, uint32_t m, uint32_t mg) {
    return mad_i24(static_cast<int32_t>(mulhi32(u, mg) >> 7), -static_cast<int32_t>(m), u);
}

// Exact reconstruction of one entry from its limb and quotient sums (as rows of the matrix product of TabSet::Wd and
// Kc, or by dot products); NL = 32-bit words of M.  The quotient q = round(sum_t r_t y_t / m_t) is taken in 16.16 fixed
// point: with F_t = round(2^16 y_t / m_t) the sum sum_t r_t F_t / 2^16 is within s * 255 * 2^-17 < 0.05 of the exact
// one, which lies within 1/4 of q whenever |C'| <= M/4 (the scaling guarantees it), so rounding it gives q (the
// reference's fp32 estimate gives the same q for the same reason).

// keeps the compiler from merging the operations before and after
OZ2_HD void settle(int32_t& x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(x));
#else
    (void)x;
#endif
}

// V = 2^up C' = sum_t r_t (2^up W_t) - q (2^up M) as NL little-endian words (two's complement, mod 2^(32 NL);
// |V| < 2^(32 NL - 2)) from its 2 NL limb sums, each with q Mc16 below 2^30 in magnitude.  Per limb one
// v_mad_i32_i24 and one add whose carry operand is the high half of its register (SDWA); without settle()
// the compiler takes a multiplication, a shift and a three-way addition.
template <int NL, typename Tab, typename Limb>
OZ2_HD void crt_carry(Tab tb, uint32_t uq, Limb limb, uint32_t (&w)[NL]) {
    int32_t q = static_cast<int32_t>(uq) >> 16;
    settle(q);
    int32_t prev = 0;
    OZ2_UNROLL for (int i = 0; i < NL; ++i) {
        int32_t v[2];
        OZ2_UNROLL for (int h = 0; h < 2; ++h) {
            const int l = 2 * i + h;
            int32_t x = static_cast<int32_t>(limb(l));
            settle(x);
            x = static_cast<int32_t>(mad_i24(q, static_cast<int32_t>(tb->Mc16[l]), static_cast<uint32_t>(x)));
            settle(x);
            v[h] = x + (prev >> 16);
            prev = v[h];
        }
        w[i] = pack_lo_halves(static_cast<uint32_t>(v[0]), static_cast<uint32_t>(v[1]));
    }
}

// from the rows of the matrix product: limb l is x[2l] + 256 x[2l+1] (24 * 128 * 128 * 257 + 24 * 128 * 65535
// + 24 * 255 * 65535 < 2^30); the 2^15 of q's rounding is in
// Kc, which signed residues (SYM, of any representative in [-128, 127]) do without: q may then be negative
template <int NL, bool SYM = false, typename Tab, typename Row>
OZ2_HD void crt_words(Tab tb, Row x, uint32_t (&w)[NL]) {
    const uint32_t uq = (SYM ? 0x8000u : 0u) + static_cast<uint32_t>(x(4 * NL)) + ((static_cast<uint32_t>(x(4 * NL + 1)) +
                                                            (static_cast<uint32_t>(x(4 * NL + 2)) << 8)) << 8);
    crt_carry<NL>(tb, uq, [&](int l) { return static_cast<uint32_t>(x(2 * l)) + (static_cast<uint32_t>(x(2 * l + 1)) << 8); }, w);
}

// the limb and quotient sums by 16-bit dot products: moduli 2i and 2i+1 at once (r1 = 0 past s), one dot2
// per limb (r < 256, W16 < 2^16: sums below 2^29)
template <int NL>
struct CrtAcc {
    uint32_t uq = 0x8000u, acc[2 * NL] = {};
    template <typename Tab>
    OZ2_HD void add2(Tab tb, int i, uint32_t r0, uint32_t r1) {
        const uint32_t rr = r0 | (r1 << 16);
        uq = udot2(rr, tb->F16p[i], uq);
        OZ2_UNROLL for (int l = 0; l < 2 * NL; ++l) acc[l] = udot2(rr, tb->W16p[i][l], acc[l]);
    }
    template <typename Tab>
    OZ2_HD void words(Tab tb, uint32_t (&w)[NL]) const {
        crt_carry<NL>(tb, uq, [&](int l) { return acc[l]; }, w);
    }
};

// RNE(V) * 2^-shift (shift includes up), any V.  The window is 64 bits of V from its sign bit on, every lower
// bit folded into the window's last one (sticky).  It stays in two's complement: the fold moves the value
// towards the next odd number, and the rounding boundaries of a 53-bit result are even, so negative values
// round as their magnitudes do.
template <int NL>
OZ2_HD double crt_round_any(const uint32_t (&w)[NL], int shift) {
    constexpr int G = (NL + 1) / 2;
    static_assert(G <= 3, "at most 6 words");
    int64_t g[G];
    OZ2_UNROLL for (int i = 0; i < G; ++i) {
        const uint32_t top = 2 * i + 1 < NL ? w[2 * i + 1] : static_cast<uint32_t>(static_cast<int32_t>(w[NL - 1]) >> 31);
        g[i] = static_cast<int64_t>(w[2 * i] | static_cast<uint64_t>(top) << 32);
    }
    int64_t hi = g[G - 1], lo = G >= 2 ? g[G - 2] : 0;
    bool below = G == 3 && g[0] != 0;
    int base = 64 * (G - 1);  // log2 weight of hi's lowest bit
    OZ2_UNROLL for (int step = 0; step + 1 < G; ++step) {  // step down past groups that only extend the sign
        const bool z = hi == lo >> 63;
        const int idx = G - 2 - step;            // lo is group idx
        hi = z ? lo : hi;
        lo = z ? (idx >= 1 ? g[idx - 1] : 0) : lo;
        base -= z ? 64 : 0;
        below = z ? false : below;               // with G <= 3 nothing lies below the new lo
    }
    const int sh = clz64(static_cast<uint64_t>(hi ^ (hi >> 63))) - 1;  // sign bits but one: 0 .. 63
    uint64_t top = (static_cast<uint64_t>(hi) << sh) | ((static_cast<uint64_t>(lo) >> 1) >> (63 - sh));
    const uint64_t rest = static_cast<uint64_t>(lo) << sh;
    top |= (below || rest != 0) ? 1u : 0u;
    // the window's lsb weighs 2^(base - sh); one RNE here, a second only if subnormal
    return ldexp_(static_cast<double>(static_cast<int64_t>(top)), base - sh - shift);
}

// RNE(V) * 2^-shift: the top 96 bits of V as a sum of two 48-bit doubles, a 2^48 + b, exact but for the last
// bit of b, which folds in every lower word; one addition rounds it.  The fold is right where a unit of the
// result is at least four of b's (the rounding boundaries are then even): |a| >= 65, that is |C'| above about
// 2^-40 of its bound, or where nothing was folded (every V of at most 3 words, and V = 0).  For the rest, rare,
// `any` is set and crt_round_any has the value.
template <int NL>
OZ2_HD double crt_round(const uint32_t (&w)[NL], int shift, bool& any) {
    any = false;
    if (NL == 2) {
        const double v = __builtin_fma(static_cast<double>(static_cast<int32_t>(w[1])), 4294967296.0, static_cast<double>(w[0]));
        return ldexp_(v, -shift);
    }
    constexpr int T = NL >= 3 ? NL : 3;  // (the words below exist for NL >= 3)
    uint32_t low = 0;
    OZ2_UNROLL for (int i = 0; i + 3 < NL; ++i) low |= w[i];
    const double a = __builtin_fma(static_cast<double>(static_cast<int32_t>(w[T - 1])), 65536.0, static_cast<double>(w[T - 2] >> 16));
    const uint32_t w0 = w[T - 3] | (low < 1u ? low : 1u);
    const double b = __builtin_fma(static_cast<double>(w[T - 2] & 0xFFFFu), 4294967296.0, static_cast<double>(w0));
    any = NL > 3 && __builtin_fabs(a) < 65.0 && low != 0;
    return ldexp_(__builtin_fma(a, 281474976710656.0, b), 32 * (NL - 3) - shift);
}

}  // namespace math
}  // namespace oz2
