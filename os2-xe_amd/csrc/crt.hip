// crt.hip - CRT reconstruction fused with the alpha/beta epilogue, for gfx950.
//
// Bounds: HBM up to s = 16 (s + 8 or 16 bytes an entry; 5.3 TB/s at 8192 x 8192 s = 16, the rate of a plain
// copy), the VALU above (4.0 TB/s at s = 24).
//
// Reference behaviour: src/ozaki2_gpu.hpp:526-664.  For each entry the s
// residues r_t (bytes from the GEMM epilogue; k-chunks are summed mod m_t)
// determine the exact integer C' with |C'| <= M/4:
//   q  = round(sum_t r_t F_t / 2^16)            (F_t = round(2^16 y_t / m_t); error < 0.05, so q is exact)
//   C' = sum_t r_t W_t - q M                     (limb sums of crt_tile.hpp or 16-bit dot products)
// C' is rounded once to 53 bits (sticky bit) and scaled by 2^-(D_i + E_j),
// which rounds again only for subnormal results, as in the reference.
// Rows / columns with a non-finite exponent give NaN.  The epilogue is
// C = alpha*v (beta == 0, C not read) or fma(alpha, v, beta*C); complex:
// Re = P0 - P1, Im = P2 - P0 - P1 in residue space (3M form), then
// (ar*vr - ai*vi, ar*vi + ai*vr) + beta*C, each product pair fused as one fma.
#include "crt_tile.hpp"
#include "grouped.hpp"
#include "kernels.hpp"
#include "math.hpp"

namespace oz2 {
namespace k {
using namespace math;

namespace {

// Residue words (4 entries) of SC moduli summed over the k-chunks mod m_t: all words of a chunk are
// loaded before they are added, as bytes 0, 2 and bytes 1, 3 in 16-bit halves.
template <int SC>
__device__ __forceinline__ void chunk_words(const uint8_t* base, const CrtArgs& a, ConstTab tb,
                                            uint32_t (&r)[SC]) {
    uint32_t even[SC] = {}, odd[SC] = {};
    auto reduce = [&](uint32_t x, int t) {  // both halves mod m_t
        const uint32_t m = tb->m[t], mu = tb->mu[t];
        return m == 256 ? x & 0x00FF00FFu : mod_m23(x & 0xFFFFu, m, mu) | mod_m23(x >> 16, m, mu) << 16;
    };
    for (int c = 0; c < a.kch; ++c) {
        uint32_t w[SC];
#pragma unroll
        for (int t = 0; t < SC; ++t)
            w[t] = t < a.s ? *reinterpret_cast<const uint32_t*>(base + c * a.chunk_r + t * a.plane_r) : 0u;
#pragma unroll
        for (int t = 0; t < SC; ++t) {
            even[t] += w[t] & 0x00FF00FFu;
            odd[t] += (w[t] >> 8) & 0x00FF00FFu;
        }
        if ((c & 127) == 127) {  // sums stay below 256 + 128 * 255 < 2^16
#pragma unroll
            for (int t = 0; t < SC; ++t)
                if (t < a.s) {
                    even[t] = reduce(even[t], t);
                    odd[t] = reduce(odd[t], t);
                }
        }
    }
#pragma unroll
    for (int t = 0; t < SC; ++t) r[t] = t < a.s ? reduce(even[t], t) | reduce(odd[t], t) << 8 : 0u;
}

// 3M residues of modulus m: Re = P0 - P1 and Im = P2 - P0 - P1, reduced into [0, m)
__device__ __forceinline__ void from_3m(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t m, uint32_t& re, uint32_t& im) {
    uint32_t xr[4], xi[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t x0 = (w0 >> (8 * e)) & 0xFFu, x1 = (w1 >> (8 * e)) & 0xFFu, x2 = (w2 >> (8 * e)) & 0xFFu;
        uint32_t r = x0 + m - x1;  // [0, 2m)
        xr[e] = r >= m ? r - m : r;
        r = x2 + 2 * m - x0 - x1;  // [0, 3m)
        r = r >= m ? r - m : r;
        xi[e] = r >= m ? r - m : r;
    }
    re = pack_lo_bytes(xr[0], xr[1], xr[2], xr[3]);
    im = pack_lo_bytes(xi[0], xi[1], xi[2], xi[3]);
}

// Matrix cores or dot products for the limb and quotient sums.  With few moduli the kernel is bound by its
// loads, and the dot products' registers (44 to 78, against 87 and more) keep more waves in flight; with many
// it is bound by the sums.  Measured on MI355X, beta != 0, matrix / dot products, us: 4096 x 4096
// s = 8 72 / 62, s = 16 124 / 109, s = 20 131 / 160, s = 24 150 / 192; 8192 x 8192 s = 16 459 / 414;
// complex 4096 x 4096 s = 16 324 / 357, s = 24 430 / 489 (before the two-double rounding of crt_round, which
// took 2 to 7 % off each: 8192 x 8192 s = 16 404, 4096 x 4096 s = 24 135, complex 315 and 411).
// No scalar load may be left for the end of the kernel: one (the scaling exponent, from the tables) made it
// 30 % slower, so that comes as an argument.
constexpr bool crt_matrix(int nl, bool cplx) { return cplx ? nl >= 4 : nl >= 5; }

template <int NL, bool MAT>
struct CrtSums : CrtTile<NL> {
    using CrtTile<NL>::CrtTile;
};
template <int NL>
struct CrtSums<NL, false> {
    ConstTab tb;
    __device__ __forceinline__ explicit CrtSums(const TabSet* tab) : tb(const_tab(tab)) {}
    template <typename Out>
    __device__ __forceinline__ void four(const uint32_t (&r)[4 * NL], const Out& out) const {
        CrtAcc<NL> acc[4];
#pragma unroll
        for (int t = 0; t < 4 * NL; t += 2) {
            if (t >= tb->s) break;  // (also keeps the tables' scalar loads apart: together they spill)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e].add2(tb, t >> 1, (r[t] >> (8 * e)) & 0xFFu, (r[t + 1] >> (8 * e)) & 0xFFu);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t w[NL];
            acc[e].words(tb, w);
            out(e, w);
        }
    }
};

// 4 consecutive rows per thread; residues are bytes packed 4 per 32-bit load.  CHUNKS: k-chunks to sum.
template <int NL, bool CPLX, bool CHUNKS>
__device__ __forceinline__ void crt_body(const CrtArgs& a, uint32_t bx) {
    constexpr int SC = 4 * NL;
    const auto tb = const_tab(a.tab);
    const CrtSums<NL, crt_matrix(NL, CPLX)> sums(a.tab);
    // row quads of a column; the block's first quad by one uniform division, the lane's from there in
    // 32 bits (a 64-bit division per lane is about as long as the reconstruction of an entry)
    const uint32_t mq = static_cast<uint32_t>((a.mb + 3) >> 2);
    const uint64_t first = static_cast<uint64_t>(bx) * 256;
    const int64_t jb = static_cast<int64_t>(first / mq);
    const uint32_t in = static_cast<uint32_t>(first - static_cast<uint64_t>(jb) * mq) + threadIdx.x;
    const uint32_t dj = in / mq;
    // every lane takes part in the matrix products: the ones past the end repeat the last column's start
    const bool ok = jb + dj < a.nb;
    const int64_t j = ok ? jb + dj : a.nb - 1;
    const int64_t i0 = ok ? static_cast<int64_t>(in - dj * mq) * 4 : 0;
    const int32_t Ej = a.E[j];
    const uint8_t* base = a.R + j * a.ldr + i0;
    const int s = a.s;
    const int64_t gs = static_cast<int64_t>(s) * a.plane_r;

    uint32_t re[SC], im[CPLX ? SC : 1];
#pragma unroll
    for (int t = 0; t < SC; ++t) {
        re[t] = 0;
        if (CPLX) im[t] = 0;
    }
    if (!CPLX && !CHUNKS) {
        // all s residue words are loaded before any arithmetic
#pragma unroll
        for (int t = 0; t < SC; ++t)
            if (t < s) re[t] = *reinterpret_cast<const uint32_t*>(base + t * a.plane_r);
    } else if (!CPLX) {
        chunk_words<SC>(base, a, tb, re);
    } else if (!CHUNKS) {
        // the same for the three 3M groups, in two halves of the moduli to bound the words held at once
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            constexpr int H = SC / 2;
            uint32_t w0[H], w1[H], w2[H];
#pragma unroll
            for (int u = 0; u < H; ++u) {
                const int t = half * H + u;
                const uint8_t* b = base + t * a.plane_r;
                w0[u] = t < s ? *reinterpret_cast<const uint32_t*>(b) : 0u;
                w1[u] = t < s ? *reinterpret_cast<const uint32_t*>(b + gs) : 0u;
                w2[u] = t < s ? *reinterpret_cast<const uint32_t*>(b + 2 * gs) : 0u;
            }
#pragma unroll
            for (int u = 0; u < H; ++u) {
                const int t = half * H + u;
                if (t < s) from_3m(w0[u], w1[u], w2[u], tb->m[t], re[t], im[CPLX ? t : 0]);
            }
        }
    } else {
        uint32_t w[3][SC];
#pragma unroll
        for (int g = 0; g < 3; ++g) chunk_words<SC>(base + g * gs, a, tb, w[g]);
#pragma unroll
        for (int t = 0; t < SC; ++t)
            if (t < s) from_3m(w[0][t], w[1][t], w[2][t], tb->m[t], re[t], im[CPLX ? t : 0]);
    }

    int32_t shift[4];
    bool nonfinite[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int32_t Di = a.D[min(i0 + e, a.mb - 1)];
        nonfinite[e] = Di == INT32_MIN || Ej == INT32_MIN;
        shift[e] = Di + Ej + a.up;
    }
    double v[4], vi[4];
    crt_four<NL>(sums, re, shift, v);
    if constexpr (CPLX)
        crt_four<NL>(sums, im, shift, vi);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (nonfinite[e]) v[e] = vi[e] = __builtin_nan("");
    if (!ok) return;
    if constexpr (!CPLX) {
        double* cp = a.C + i0 + j * a.ldc;
        if (i0 + 4 <= a.mb && (reinterpret_cast<uintptr_t>(cp) & 15) == 0) {
            // four entries of one column: 16-byte accesses to C when it is aligned for them
            double2* c2 = reinterpret_cast<double2*>(cp);
            if (a.br == 0.0) {
                c2[0] = make_double2(a.ar * v[0], a.ar * v[1]);
                c2[1] = make_double2(a.ar * v[2], a.ar * v[3]);
            } else {
                const double2 x0 = c2[0], x1 = c2[1];
                c2[0] = make_double2(__builtin_fma(a.ar, v[0], a.br * x0.x), __builtin_fma(a.ar, v[1], a.br * x0.y));
                c2[1] = make_double2(__builtin_fma(a.ar, v[2], a.br * x1.x), __builtin_fma(a.ar, v[3], a.br * x1.y));
            }
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i0 + e < a.mb) cp[e] = a.br == 0.0 ? a.ar * v[e] : __builtin_fma(a.ar, v[e], a.br * cp[e]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t i = i0 + e;
            if (i >= a.mb) break;
            double* cp = a.C + 2 * (i + j * a.ldc);
            double orr = __builtin_fma(a.ar, v[e], -(a.ai * vi[e]));
            double oi = __builtin_fma(a.ar, vi[e], a.ai * v[e]);
            if (a.br != 0.0 || a.bi != 0.0) {
                const double cr = cp[0], ci = cp[1];
                orr = orr + __builtin_fma(a.br, cr, -(a.bi * ci));
                oi = oi + __builtin_fma(a.br, ci, a.bi * cr);
            }
            cp[0] = orr;
            cp[1] = oi;
        }
    }
}

// waves per SIMD to compile for (below 256 registers the products' results stay out of the accumulation
// registers, which the VALU cannot read)
constexpr int crt_waves(int nl, bool cplx, bool chunks) {
    return cplx ? (nl > 4 ? 2 : 3) : nl > 4 || chunks ? 4 : 6;
}

template <int NL, bool CPLX, bool CHUNKS>
__global__ void __launch_bounds__(256, crt_waves(NL, CPLX, CHUNKS)) crt_kernel(CrtArgs a, uint64_t* ts) {
    const Stamp st(ts);
    crt_body<NL, CPLX, CHUNKS>(a, blockIdx.x);
    st.end();
}

template <int NL, bool CHUNKS>
__global__ void __launch_bounds__(256, crt_waves(NL, false, CHUNKS)) crt_grouped_kernel(const CrtArgs* __restrict__ items,
                                                          const uint32_t* __restrict__ start, uint32_t n) {
    const uint32_t p = owner_of(start, n, blockIdx.x);
    crt_body<NL, false, CHUNKS>(items[p], blockIdx.x - start[p]);
}

uint32_t crt_blocks(const CrtArgs& a) {
    const int64_t threads = ((a.mb + 3) / 4) * a.nb;
    return static_cast<uint32_t>((threads + 255) / 256);
}

__global__ void scale_c_kernel(double* C, int64_t ldc, int64_t m, int64_t n, double br, double bi, int cplx) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= m * n) return;
    const int64_t j = idx / m, i = idx - j * m;
    if (!cplx) {
        double* cp = C + i + j * ldc;
        *cp = br == 0.0 ? 0.0 : br * *cp;
    } else {
        double* cp = C + 2 * (i + j * ldc);
        if (br == 0.0 && bi == 0.0) {
            cp[0] = 0.0;
            cp[1] = 0.0;
        } else {
            const double r = cp[0], im = cp[1];
            cp[0] = __builtin_fma(br, r, -(bi * im));
            cp[1] = __builtin_fma(br, im, bi * r);
        }
    }
}

template <int NL>
void launch_crt_nl(const Stream& st, const CrtArgs& a) {
    const unsigned blocks = crt_blocks(a);
    if (a.cplx && a.kch > 1) launch(st, crt_kernel<NL, true, true>, dim3(blocks), dim3(256), a);
    else if (a.cplx) launch(st, crt_kernel<NL, true, false>, dim3(blocks), dim3(256), a);
    else if (a.kch > 1) launch(st, crt_kernel<NL, false, true>, dim3(blocks), dim3(256), a);
    else launch(st, crt_kernel<NL, false, false>, dim3(blocks), dim3(256), a);
}

}  // namespace

void crt(const Stream& st, const CrtArgs& a) {
    if (a.mb <= 0 || a.nb <= 0) return;
    switch (a.L16 / 2) {
        case 2: launch_crt_nl<2>(st, a); break;
        case 3: launch_crt_nl<3>(st, a); break;
        case 4: launch_crt_nl<4>(st, a); break;
        case 5: launch_crt_nl<5>(st, a); break;
        case 6: launch_crt_nl<6>(st, a); break;
        default: break;
    }
}

// grouped CRT (real products): one launch per (limb count, one k-chunk / several)
void prep_crt(std::vector<GroupedLaunch>& out, const std::vector<CrtArgs>& jobs) {
    GroupedLaunch by[14];
    for (const CrtArgs& a : jobs) {
        if (a.mb <= 0 || a.nb <= 0) continue;
        const int v = (a.L16 / 2) * 2 + (a.kch > 1 ? 1 : 0);
        by[v].kind = v;
        by[v].add(a, crt_blocks(a));
    }
    for (GroupedLaunch& g : by)
        if (g.n) out.push_back(std::move(g));
}

void launch_crt_grouped(hipStream_t st, const GroupedLaunch& g) {
    if (g.n == 0) return;
    const CrtArgs* items = static_cast<const CrtArgs*>(g.d_items);
    switch (g.kind) {
#define OZ2_NL(NL)                                                                                        \
    case 2 * NL:                                                                                          \
        hipLaunchKernelGGL((crt_grouped_kernel<NL, false>), dim3(g.blocks), dim3(256), 0, st, items, g.d_start, g.n); \
        break;                                                                                            \
    case 2 * NL + 1:                                                                                      \
        hipLaunchKernelGGL((crt_grouped_kernel<NL, true>), dim3(g.blocks), dim3(256), 0, st, items, g.d_start, g.n); \
        break;
        OZ2_NL(2) OZ2_NL(3) OZ2_NL(4) OZ2_NL(5) OZ2_NL(6)
#undef OZ2_NL
        default: break;
    }
}

void scale_c(hipStream_t st, double* C, int64_t ldc, int64_t m, int64_t n, double br, double bi, bool cplx) {
    const int64_t total = m * n;
    if (total <= 0) return;
    hipLaunchKernelGGL(scale_c_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, st, C, ldc, m,
                       n, br, bi, cplx ? 1 : 0);
}

}  // namespace k
}  // namespace oz2
