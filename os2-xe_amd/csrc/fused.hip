// fused.hip - INT8 GEMMs of all planes and the CRT of one tile of C in one workgroup.
#include <algorithm>

#include "crt_tile.hpp"
#include "grouped.hpp"
#include "kernels.hpp"
#include "math.hpp"

namespace oz2 {
namespace k {
using namespace math;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(1))) void* glb_ptr;

namespace {

constexpr int KT = 128;  // k bytes per LDS stage

constexpr int vm_wait(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
constexpr int kLgkmWait0 = 0xC07F & ~0x0F00;

// blockIdx -> work item: workgroups are dispatched round-robin over the 8 XCDs; each XCD takes a
// contiguous range of the n items (any n)
__device__ __forceinline__ uint32_t xcd_range(uint32_t b, uint32_t n) {
    const uint32_t x = b & 7, q = n >> 3, r = n & 7;
    return x * q + min(x, r) + (b >> 3);
}

template <int TM, int TN, int GM, int GN, int NS, int NL>
__device__ __forceinline__ void fused_tile(const FusedArgs& p, uint32_t tm, uint32_t tn, v4i* smem) {
    constexpr int NWV = GM * GN;
    constexpr int WTM = TM / GM, WTN = TN / GN;
    constexpr int FM = WTM / 32, FN = WTN / 32;
    constexpr int LA = TM / 16 / NWV, LB = TN / 16 / NWV;  // 16-row bands per wave and stage
    static_assert(LA * NWV * 16 == TM && LB * NWV * 16 == TN);
    constexpr int STAGE = (TM + TN) * KT;
    constexpr int NF = FM * FN;
    constexpr int ND = 2 * (LA + LB);
    constexpr int NW = NF * 4;       // residue words (4 rows of a column) per lane and plane
    constexpr int SC = 4 * NL;       // moduli of NL words of M: at most 4 NL

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / GN, wn = wave % GN;
    const int fr = lane & 31, fc = lane >> 5;
    const int S = p.s;
    const int nst = static_cast<int>(p.kp / KT);
    const int64_t band = p.kp * 16;  // bytes of a 16-row band of a plane
    const auto tb0 = const_tab(p.tab);
    const int8_t* Ab = p.A + (static_cast<int64_t>(tm) * (TM / 16) + wave * LA) * band;
    const int8_t* Bb = p.B + (static_cast<int64_t>(tn) * (TN / 16) + wave * LB) * band;
    uint32_t va[LA], vb[LB];
#pragma unroll
    for (int d = 0; d < LA; ++d) va[d] = static_cast<uint32_t>(d * band) + lane * 16 - (d & 1) * 2048;
#pragma unroll
    for (int d = 0; d < LB; ++d) vb[d] = static_cast<uint32_t>(d * band) + lane * 16 - (d & 1) * 2048;
    char* sbase = reinterpret_cast<char*>(smem);
    const int rowoff = (fr >> 4) * 2048 + (fr & 15) * 64;
    int offa[2], offb[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int ch = ((2 * ks + fc) ^ ((fr >> 2) & 3)) << 4;
        offa[ks] = wm * WTM * KT + rowoff + ch;
        offb[ks] = (TM + wn * WTN) * KT + rowoff + ch;
    }
    // DMA stream, plane-major: stage `left` stages before the end, at k byte dko of its plane
    int left = S * nst, dko = 0, dbuf = 0;
    const int kend = nst * 2048;
    auto rsrc = [](const int8_t* q) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(q), 0, 0xFFFFFFFFu, 0x00027000);
    };
    auto dma = [&](int d) {  // d-th 1 KB block of the stage
        const int u = d >> 1, h = d & 1;
        if (u < LA) {
            auto ra = rsrc(Ab);
            lds_ptr dst = (lds_ptr)(sbase + dbuf + (wave * LA + (u & ~1)) * 2048);
            if ((u & 1) == 0) {
                if (h == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst, 16, va[u], dko, 0, 0);
                else __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst, 16, va[u], dko, 1024, 0);
            } else {
                if (h == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst, 16, va[u], dko, 2048, 0);
                else __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst, 16, va[u], dko, 3072, 0);
            }
        } else {
            const int x = u - LA;
            auto rb = rsrc(Bb);
            lds_ptr dst = (lds_ptr)(sbase + dbuf + TM * KT + (wave * LB + (x & ~1)) * 2048);
            if ((x & 1) == 0) {
                if (h == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst, 16, vb[x], dko, 0, 0);
                else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst, 16, vb[x], dko, 1024, 0);
            } else {
                if (h == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst, 16, vb[x], dko, 2048, 0);
                else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst, 16, vb[x], dko, 3072, 0);
            }
        }
    };
    // next stage; past the last one the same stage is fetched again into a buffer that is not read
    auto dma_next = [&] {
        dbuf = dbuf == (NS - 1) * STAGE ? 0 : dbuf + STAGE;
        const int last = --left <= 0;
        dko += last ? 0 : 2048;
        const bool wrap = dko == kend;
        dko = wrap ? 0 : dko;
        Ab += wrap ? p.plane_a : 0;
        Bb += wrap ? p.plane_b : 0;
    };

    v16i acc[FM][FN];
    // residue words by plane: vectors that a uniform index addresses in registers
    constexpr int SL = SC < 16 ? SC : 16, SH = SC > 16 ? SC - 16 : 4;
    typedef uint32_t lo_t __attribute__((ext_vector_type(SL == 12 ? 16 : SL)));
    typedef uint32_t hi_t __attribute__((ext_vector_type(SH)));
    lo_t rlo[NW];
    hi_t rhi[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        rlo[w] = 0;
        rhi[w] = 0;
    }

#pragma unroll
    for (int s0 = 0; s0 < NS - 1; ++s0) {
#pragma unroll
        for (int d = 0; d < ND; ++d) dma(d);
        dma_next();
    }
    // exponents of the tile's rows and columns (past the end: the last one's)
    {
        int32_t* ex = reinterpret_cast<int32_t*>(sbase + NS * STAGE);
        for (int x = threadIdx.x; x < TM + TN; x += 64 * NWV)
            ex[x] = x < TM ? p.D[min(static_cast<int64_t>(tm) * TM + x, p.mb - 1)]
                           : p.E[min(static_cast<int64_t>(tn) * TN + x - TM, p.nb - 1)];
    }
    const CrtTile<NL> tile(p.tab);
    int rbuf = 0;
    for (int t = 0; t < S; ++t) {
        const uint32_t m = tb0->m[t], c30 = tb0->c30[t], mu = tb0->mu[t], c8 = tb0->c8[t][0];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = c30;
        for (int kt = 0; kt < nst; ++kt) {
            v4i fa[4][FM], fb[4][FN];
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(vm_wait((NS - 2) * ND));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            const char* pa[2] = {sbase + rbuf + offa[0], sbase + rbuf + offa[1]};
            const char* pb[2] = {sbase + rbuf + offb[0], sbase + rbuf + offb[1]};
            auto rd = [&](int q) {  // fragments of k step q
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    fa[q][i] = *reinterpret_cast<const v4i*>(pa[q & 1] + (q >> 1) * 1024 + i * 4096);
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    fb[q][j] = *reinterpret_cast<const v4i*>(pb[q & 1] + (q >> 1) * 1024 + j * 4096);
            };
            rd(0);
            rd(1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q < 2) rd(q + 2);
#pragma unroll
                for (int u = 0; u < NF; ++u) {
                    const int i = u / FN, j = u % FN;
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[q][i], fb[q][j], acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int d = 0; d < ND; ++d)
                        if (d * (4 * NF) / ND == q * NF + u) dma(d);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            dma_next();
            rbuf = rbuf == (NS - 1) * STAGE ? 0 : rbuf + STAGE;
        }
        uint32_t w[NW];
        if (m == 256) {
#pragma unroll
            for (int x = 0; x < NW; ++x) {
                const auto& c = acc[x / 4 / FN][x / 4 % FN];
                const int q = x % 4;
                w[x] = pack_lo_bytes(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]);
            }
        } else {
#pragma unroll
            for (int x = 0; x < NW; x += 2) {
                // eight entries step by step (a dot product's result is not ready for three slots)
                uint32_t y[8], z[8];
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const auto& c = acc[x / 4 / FN][x / 4 % FN];
                    y[b] = udot4(static_cast<uint32_t>(c[4 * (x % 4) + b]), c8, 0u);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < 8; ++b) z[b] = y[b] + y[b];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < 8; ++b) z[b] = mulhi24(z[b], mu);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < 8; ++b) y[b] = mad_i24(static_cast<int32_t>(z[b]), -static_cast<int32_t>(m), y[b]);
                __builtin_amdgcn_sched_barrier(0);
                w[x] = pack_lo_bytes(y[0], y[1], y[2], y[3]);
                w[x + 1] = pack_lo_bytes(y[4], y[5], y[6], y[7]);
            }
        }
        if (SC <= 16 || t < 16) {
#pragma unroll
            for (int x = 0; x < NW; ++x) rlo[x][t] = w[x];
        } else {
#pragma unroll
            for (int x = 0; x < NW; ++x) rhi[x][t - 16] = w[x];
        }
    }
    __builtin_amdgcn_s_waitcnt(vm_wait(0));

    const int rw = wm * WTM + 4 * fc, cw = wn * WTN + fr;  // the lane's first row and column in the tile
    const int64_t row0 = static_cast<int64_t>(tm) * TM + rw, col0 = static_cast<int64_t>(tn) * TN + cw;
    const int32_t* eD = reinterpret_cast<const int32_t*>(sbase + NS * STAGE);
    const int32_t* eE = eD + TM;
    // C entries of word x, one word ahead of its use
    double cn[4];
    auto load_c = [&](int x, double (&c)[4]) {
        const int i = x / 4 / FN, j = x / 4 % FN, q = x % 4;
        const int64_t col = min(col0 + j * 32, p.nb - 1), row = row0 + i * 32 + 8 * q;
        const double* cp = p.C + col * p.ldc;
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = cp[min(row + e, p.mb - 1)];
    };
    const bool beta = p.br != 0.0;
    if (beta) load_c(0, cn);
#pragma unroll
    for (int x = 0; x < NW; ++x) {
        const int i = x / 4 / FN, j = x / 4 % FN, q = x % 4;
        __builtin_amdgcn_sched_barrier(0);
        double c[4];
        if (beta) {
#pragma unroll
            for (int e = 0; e < 4; ++e) c[e] = cn[e];
            if (x + 1 < NW) load_c(x + 1, cn);
        }
        const int64_t col = col0 + j * 32, row = row0 + i * 32 + 8 * q;
        const bool ok = col < p.nb && row < p.mb;
        const int32_t Ej = eE[cw + j * 32];
        uint32_t r[SC];
#pragma unroll
        for (int t = 0; t < SC; ++t) r[t] = t < 16 ? rlo[x][t < SL ? t : 0] : rhi[x][t < 16 ? 0 : t - 16];
        double v[4];
        tile.four(r, [&](int e, const uint32_t (&w)[NL]) {
            const int32_t Di = eD[rw + i * 32 + 8 * q + e];
            const bool nonfinite = Di == INT32_MIN || Ej == INT32_MIN;
            v[e] = nonfinite ? __builtin_nan("") : crt_round<NL>(w, Di + Ej + tb0->up);
        });
        double* cp = p.C + row + col * p.ldc;
        if (!ok) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = beta ? __builtin_fma(p.ar, v[e], p.br * c[e]) : p.ar * v[e];
        if (row + 4 <= p.mb && (reinterpret_cast<uintptr_t>(cp) & 15) == 0) {
            double2* c2 = reinterpret_cast<double2*>(cp);
            c2[0] = make_double2(v[0], v[1]);
            c2[1] = make_double2(v[2], v[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (row + e < p.mb) cp[e] = v[e];
        }
    }
}

template <int TM, int TN, int GM, int GN, int NS, int NL, int MINB>
__global__ void __launch_bounds__(64 * GM * GN, MINB) fused_kernel(FusedArgs p, uint64_t* ts) {
    const Stamp st(ts);
    __shared__ v4i smem[(NS * (TM + TN) * KT + (TM + TN) * 4) / 16];
    const uint32_t w = xcd_range(blockIdx.x, gridDim.x);
    const uint32_t G = 8, per = G * p.tiles_n, g = w / per, first = g * G;
    const uint32_t gs = min(G, static_cast<uint32_t>(p.tiles_m) - first), in = w - g * per;
    fused_tile<TM, TN, GM, GN, NS, NL>(p, first + in % gs, in / gs, smem);
    st.end();
}

}  // namespace

void fused(const Stream& st, int code, const FusedArgs& a) {
    const uint32_t n = static_cast<uint32_t>(a.tiles_m) * a.tiles_n;
    if (n == 0) return;
#define OZ2_L(TM, TN, GM, GN, NS, NL, MINB) launch(st, fused_kernel<TM, TN, GM, GN, NS, NL, MINB>, dim3(n), dim3(64 * GM * GN), a)
#define OZ2_S(TM, TN, GM, GN, NS, M2, M3, M4, M5, M6) \
    switch (a.nl) { case 2: OZ2_L(TM, TN, GM, GN, NS, 2, M2); break; case 3: OZ2_L(TM, TN, GM, GN, NS, 3, M3); break; \
        case 4: OZ2_L(TM, TN, GM, GN, NS, 4, M4); break; case 5: OZ2_L(TM, TN, GM, GN, NS, 5, M5); break; case 6: OZ2_L(TM, TN, GM, GN, NS, 6, M6); break; }
    if (code == 64) { OZ2_S(64, 64, 2, 2, 3, 3, 3, 3, 2, 2) }
    else if (code == 12864) { OZ2_S(128, 64, 2, 2, 3, 2, 2, 2, 2, 2) }
    else if (code == 128) { OZ2_S(128, 128, 2, 4, 4, 2, 2, 2, 2, 2) }
#undef OZ2_L
}

}  // namespace k
}  // namespace oz2
