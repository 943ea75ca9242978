// crt_tile.hpp - CRT of four entries per lane on the matrix cores (device only).
//
// The CRT of an entry is linear in its residues up to the final rounding: limb sums
// sum_t r_t W_t and the quotient sum sum_t r_t F_t.  As 16-bit dot products on the VALU
// (v_dot2_u32_u16, two moduli a step) they are s/2 (2 NL + 1) instructions an entry, 72 at
// s = 16 and 156 at s = 24, most of the reconstruction.  Here they are rows of one int8
// product (TabSet::Wd: digits of W_t and F_t by modulus, times residues by entry): two
// v_mfma_i32_32x32x32_i8 give all rows of 64 entries for up to 16 moduli, four for 24.
//
// Operands of the MFMA (lane l: row l mod 32 of A, column l mod 32 of B, k = 16 (l / 32) ..
// + 15): a lane holds its own entry's residues of moduli 0 .. 15 as its 16 bytes of B, so
// columns of lanes 0 .. 31 sit in k 0 .. 15 and those of lanes 32 .. 63 in k 16 .. 31; A has
// the digits in one half of k and zeros in the other, once per half of the lanes.  The two
// results hold rows 8 (v/4) + 4 (l/32) + v % 4 of entry l mod 32 (+ 32): v_permlane32_swap
// of their registers gives every lane all rows of its own entry.
#pragma once
#include "kernels.hpp"
#include "math.hpp"

namespace oz2 {
namespace k {

typedef int crt_v4i __attribute__((ext_vector_type(4)));
typedef int crt_v16i __attribute__((ext_vector_type(16)));

// digits and constants of one modulus set, held by a wave for all its entries.  SYM: the residues come as
// signed bytes in [-128, 127] (any representative), else as bytes in [0, m).
template <int NL, bool SYM = false>
struct CrtTile {
    static constexpr int SC = 4 * NL;  // moduli of NL words of M: at most 4 NL
    crt_v4i a[NL > 4 ? 2 : 1][2];      // [moduli 0 .. 15, 16 .. 31][lanes 0 .. 31, 32 .. 63]
    crt_v16i init;
    math::ConstTab tb;

    __device__ __forceinline__ explicit CrtTile(const TabSet* tab) : tb(math::const_tab(tab)) {
        const int lane = threadIdx.x & 63, half = lane >> 5;
        const crt_v4i zero = {0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < (NL > 4 ? 2 : 1); ++u) {
            const crt_v4i d = *reinterpret_cast<const crt_v4i*>(&tab->Wd[lane & 31][16 * u]);
            a[u][0] = half ? zero : d;
            a[u][1] = half ? d : zero;
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const crt_v4i c = *reinterpret_cast<const crt_v4i*>(&tab->Kc[8 * b + 4 * half]);
#pragma unroll
            for (int i = 0; i < 4; ++i) init[4 * b + i] = SYM ? 0 : c[i];
        }
    }

    // r[t]: residues of modulus t of the lane's four entries, one byte each (any value past s);
    // out(e, w): words of V of entry e.  All lanes of the wave take part.
    template <typename Out>
    __device__ __forceinline__ void four(const uint32_t (&r)[SC], const Out& out) const {
        // 4 x 4 byte transposes: b[e] = residues of entry e, minus 128, by modulus
        uint32_t b[4][NL];
#pragma unroll
        for (int g = 0; g < NL; ++g) {
            const uint32_t lo01 = __builtin_amdgcn_perm(r[4 * g + 1], r[4 * g], 0x05010400u);
            const uint32_t hi01 = __builtin_amdgcn_perm(r[4 * g + 1], r[4 * g], 0x07030602u);
            const uint32_t lo23 = __builtin_amdgcn_perm(r[4 * g + 3], r[4 * g + 2], 0x05010400u);
            const uint32_t hi23 = __builtin_amdgcn_perm(r[4 * g + 3], r[4 * g + 2], 0x07030602u);
            b[0][g] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u) ^ (SYM ? 0u : 0x80808080u);
            b[1][g] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u) ^ (SYM ? 0u : 0x80808080u);
            b[2][g] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u) ^ (SYM ? 0u : 0x80808080u);
            b[3][g] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u) ^ (SYM ? 0u : 0x80808080u);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            crt_v4i v = {0, 0, 0, 0};
#pragma unroll
            for (int g = 0; g < 4 && g < NL; ++g) v[g] = static_cast<int>(b[e][g]);
            crt_v16i o0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0][0], v, init, 0, 0, 0);
            crt_v16i o1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0][1], v, init, 0, 0, 0);
            if constexpr (NL > 4) {
                crt_v4i v2 = {static_cast<int>(b[e][4]), NL > 5 ? static_cast<int>(b[e][NL - 1]) : 0, 0, 0};
                o0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[NL > 4][0], v2, o0, 0, 0, 0);
                o1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[NL > 4][1], v2, o1, 0, 0, 0);
            }
            int32_t row[32];
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                const int at = 8 * (x >> 2) + (x & 3);
                if (at < 4 * NL + 3) {
                    const auto sw = __builtin_amdgcn_permlane32_swap(o0[x], o1[x], false, false);
                    row[at] = static_cast<int32_t>(sw[0]);
                    row[at + 4] = static_cast<int32_t>(sw[1]);
                }
            }
            uint32_t w[NL];
            math::crt_words<NL, SYM>(tb, [&](int x) { return row[x]; }, w);
            out(e, w);
        }
    }
};

// RNE(V) 2^-shift of four entries from their sums (CrtTile or the dot products)
template <int NL, typename Sums>
__device__ __forceinline__ void crt_four(const Sums& sums, const uint32_t (&r)[4 * NL], const int32_t (&shift)[4],
                                         double (&v)[4]) {
    // entries far below their bound, rare, take the general window: up to 16 moduli the wave takes the quad
    // again (all lanes are needed), above, where holding the residues for that would spill, entry by entry
    bool any = false;
    sums.four(r, [&](int e, const uint32_t (&w)[NL]) {
        bool f;
        v[e] = math::crt_round<NL>(w, shift[e], f);
        if (NL > 4 && f) v[e] = math::crt_round_any<NL>(w, shift[e]);
        any |= f;
    });
    if (NL == 4 && __any(any))
        sums.four(r, [&](int e, const uint32_t (&w)[NL]) { v[e] = math::crt_round_any<NL>(w, shift[e]); });
}

}  // namespace k
}  // namespace oz2
