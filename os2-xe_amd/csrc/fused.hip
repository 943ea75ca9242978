// fused.hip - the INT8 GEMMs of all planes and the CRT of a tile of C in one workgroup (real products of
// one k-chunk).
//
// The separate path writes s residue bytes per entry of C and reads them back in the CRT: with a short k
// that traffic and the residue epilogues take longer than the matrix products (4096 x 4096 x 256 s = 16:
// 244 us, the products 43 of them at the matrix cores' rate).  Here one workgroup takes all s planes of its
// tile, keeps the residues in registers, four rows of a column to a word as the CRT takes them, and writes
// C once.  The k loops of the planes are one loop: the LDS-DMA stream runs on through the reductions between them.
//
//   128 x 128 tiles: 8 waves of 64 x 32, one workgroup per CU (208 of 256 registers at NL = 4: 128 of them
//   residues), 4 stages of 128 k (128 KB of LDS).  64 x 64 tiles: 4 waves of 32 x 32, 3 workgroups per CU
//   (2 above 16 moduli), 3 stages.
//
// Bound: VALU (reduction 4 instructions an entry and plane, CRT 85 to 100 an entry) and the latency of the
// short k loops; the matrix cores are busy 27 % of the time at k = 256, 42 % at k = 1024.  Measured on
// MI355X, separate -> fused, us (GEMM + CRT): 4096 x 4096 s = 16 k = 128 214 -> 126, k = 256 244 -> 160,
// k = 512 308 -> 229, k = 1024 439 -> 410; s = 20 k = 256 314 -> 201; s = 8 k = 256 131 -> 116;
// 2048 x 2048 x 256 s = 16 62 -> 40.  With longer k the separate path's larger tiles win (fused_tile in
// planner.cpp).  Tried without gain: reducing a plane in the shadow of the next one's products (a second
// set of accumulators spills at 128 x 128 and is slower at 64 x 64); 128 x 64 tiles of 4 waves, two
// workgroups per CU (1 to 2 % either way against 128 x 128).
#include "crt_tile.hpp"
#include "grouped.hpp"
#include "kernels.hpp"
#include "math.hpp"

namespace oz2 {
namespace k {
using namespace math;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

namespace {

constexpr int KT = 128;  // k bytes per LDS stage: two block columns of a plane

// s_waitcnt immediate waiting for vmcnt <= n only
constexpr int vm_wait(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// Tile TM x TN by GM x GN waves, NS stages of LDS, NL words of M.
//
// Stage layout in LDS: the 16-row bands of A, then of B, each 2 KB: its two 1 KB plane blocks.  The blocks
// are dealt to the waves in turn.  Fragments, MFMA operand layout and bank pattern as in igemm.hip.
template <int TM, int TN, int GM, int GN, int NS, int NL>
__device__ __forceinline__ void fused_tile(const FusedArgs& p, uint32_t tm, uint32_t tn, v4i* smem, const Stamp& st) {
    constexpr int NWV = GM * GN;
    constexpr int WTM = TM / GM, WTN = TN / GN;
    constexpr int FM = WTM / 32, FN = WTN / 32;
    constexpr int STAGE = (TM + TN) * KT;
    constexpr int NF = FM * FN;
    constexpr int ND = (TM + TN) / 8 / NWV;  // 1 KB blocks that a wave fetches per stage
    static_assert(ND * 8 * NWV == TM + TN);
    constexpr int NW = NF * 4;       // residue words (4 rows of a column) per lane and plane
    constexpr int SC = 4 * NL;       // moduli of NL words of M: at most 4 NL

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / GN, wn = wave % GN;
    const int fr = lane & 31, fc = lane >> 5;
    const int S = p.s;
    const int nst = static_cast<int>(p.kp / KT);  // kp is a multiple of 128
    const auto tb = const_tab(p.tab);
    // block b of a stage: k half b % 2 of band b / 2 (bands of A, then of B); this wave's are d NWV + wave
    const PlaneMap map = PlaneMap::by_group(p.kp);
    const int8_t* src[ND];
    int64_t step[ND];  // next plane
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const int b = d * NWV + wave;
        const bool isa = b < TM / 8;
        const int64_t row = isa ? static_cast<int64_t>(tm) * (TM / 16) + (b >> 1)
                                : static_cast<int64_t>(tn) * (TN / 16) + (b >> 1) - TM / 16;
        src[d] = (isa ? p.A : p.B) + (row >> 2) * map.group + (row & 3) * map.band + (b & 1) * map.blk;
        step[d] = isa ? p.plane_a : p.plane_b;
    }
    char* sbase = reinterpret_cast<char*>(smem);
    const int rowoff = (fr >> 4) * 2048 + (fr & 15) * 64;
    int offa[2], offb[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int ch = ((2 * ks + fc) ^ ((fr >> 2) & 3)) << 4;
        offa[ks] = wm * WTM * KT + rowoff + ch;
        offb[ks] = (TM + wn * WTN) * KT + rowoff + ch;
    }
    // DMA stream, plane-major: stage `left` stages before the end, at offset dko of its plane
    const int kstep = static_cast<int>(2 * map.blk), kend = nst * kstep;
    int left = S * nst, dko = 0, dbuf = 0;
    auto dma = [&](int d) { block_to_lds(src[d], dko, lane, sbase + dbuf + (d * NWV + wave) * 1024); };  // the wave's d-th block
    // next stage; past the last one the same stage is fetched again into a buffer that is not read
    auto dma_next = [&] {
        dbuf = dbuf == (NS - 1) * STAGE ? 0 : dbuf + STAGE;
        dko += --left <= 0 ? 0 : kstep;
        const bool wrap = dko == kend;
        dko = wrap ? 0 : dko;
#pragma unroll
        for (int d = 0; d < ND; ++d) src[d] += wrap ? step[d] : 0;
    };

    // residue words by plane: vectors that a uniform index addresses in registers
    constexpr int SL = SC < 16 ? SC : 16, SH = SC > 16 ? SC - 16 : 4;
    typedef uint32_t lo_t __attribute__((ext_vector_type(SL)));
    typedef uint32_t hi_t __attribute__((ext_vector_type(SH)));
    lo_t rlo[NW];
    hi_t rhi[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        rlo[w] = 0;
        rhi[w] = 0;
    }
    v16i acc[FM][FN];
    int rbuf = 0;
    // one stage: its DMAs have landed (own, then everyone's), and everyone is done with the buffer that the
    // DMAs issued here refill
    auto stage = [&] {
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
    };

#pragma unroll
    for (int s0 = 0; s0 < NS - 1; ++s0) {
#pragma unroll
        for (int d = 0; d < ND; ++d) dma(d);
        dma_next();
    }
    // exponents of the tile's rows and columns (past the end: the last one's), read after the last stage; at
    // least two stages' barriers lie between
    {
        int32_t* ex = reinterpret_cast<int32_t*>(sbase + NS * STAGE);
        for (int x = threadIdx.x; x < TM + TN; x += 64 * NWV)
            ex[x] = x < TM ? p.D[min(static_cast<int64_t>(tm) * TM + x, p.mb - 1)]
                           : p.E[min(static_cast<int64_t>(tn) * TN + x - TM, p.nb - 1)];
    }
    // The sums start at c30 + 128: the residue of x + 128, xored with 0x80, is x's as a signed byte in
    // [-128, 126], as CrtTile takes it.
    uint32_t c30 = tb->c30[0] + 128;
    for (int t = 0; t < S; ++t) {
        const uint32_t m = tb->m[t], mg = tb->mg[t];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = c30;
        c30 = tb->c30[t + 1 < kMaxModuli ? t + 1 : t] + 128;
        for (int kt = 0; kt < nst; ++kt) stage();
        uint32_t w[NW];
#pragma unroll
        for (int x = 0; x < NW; ++x) {
            uint32_t r[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t u = static_cast<uint32_t>(acc[x / 4 / FN][x / 4 % FN][4 * (x % 4) + b]);
                r[b] = residue_word(u, m, mg);
            }
            w[x] = pack_lo_bytes(r[0], r[1], r[2], r[3]) ^ 0x80808080u;
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

    st.inner(0);
    const CrtTile<NL, true> tile(p.tab);
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
        int32_t shift[4];
        bool nonfinite[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int32_t Di = eD[rw + i * 32 + 8 * q + e];
            nonfinite[e] = Di == INT32_MIN || Ej == INT32_MIN;
            shift[e] = Di + Ej + p.up;
        }
        double v[4];
        tile.four(r, [&](int e, const uint32_t (&w)[NL]) {
            bool f;
            v[e] = crt_round<NL>(w, shift[e], f);
            if (f) v[e] = crt_round_any<NL>(w, shift[e]);
        });
        double* cp = p.C + row + col * p.ldc;
        if (!ok) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (nonfinite[e]) v[e] = __builtin_nan("");
            v[e] = beta ? __builtin_fma(p.ar, v[e], p.br * c[e]) : p.ar * v[e];
        }
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

// tile (tm, tn) of index w: columns of 8 tile-rows, walking tile-columns inside a group
__device__ __forceinline__ void tile_coords(const FusedArgs& p, uint32_t w, uint32_t& tm, uint32_t& tn) {
    const uint32_t G = 8, per = G * p.tiles_n, g = w / per, first = g * G;
    const uint32_t gs = min(G, static_cast<uint32_t>(p.tiles_m) - first), in = w - g * per;
    tm = first + in % gs;
    tn = in / gs;
}

// The tile, or where half of it holds the rows or the columns left (128 x 128), that half.  256 products of
// 64 .. 4096 in 128 x 128 tiles: 11.53 -> 11.38 ms.
template <int T, int GM, int GN, int NS, int NL>
__device__ __forceinline__ void fused_edge(const FusedArgs& p, uint32_t tm, uint32_t tn, v4i* smem, const Stamp& st) {
    if constexpr (T == 128) {
        if (p.mb - static_cast<int64_t>(tm) * T <= T / 2) return fused_tile<T / 2, T, 2, 4, NS, NL>(p, 2 * tm, tn, smem, st);
        if (p.nb - static_cast<int64_t>(tn) * T <= T / 2) return fused_tile<T, T / 2, 4, 2, NS, NL>(p, tm, 2 * tn, smem, st);
    }
    fused_tile<T, T, GM, GN, NS, NL>(p, tm, tn, smem, st);
}

template <int T, int NL>
struct Shape;
template <int NL>
struct Shape<128, NL> {
    static constexpr int GM = 2, GN = 4, NS = 4, MINB = 2;
};
template <int NL>
struct Shape<64, NL> {
    static constexpr int GM = 2, GN = 2, NS = 3, MINB = NL > 4 ? 2 : 3;
};
template <int T, int NL>
constexpr int kThreads = 64 * Shape<T, NL>::GM * Shape<T, NL>::GN;
template <int T, int NL>
constexpr int kSmem = (Shape<T, NL>::NS * 2 * T * KT + 2 * T * 4) / 16;

template <int T, int NL, int THREADS = kThreads<T, NL>, int MINB = Shape<T, NL>::MINB>
__global__ void __launch_bounds__(THREADS, MINB) fused_kernel(FusedArgs p, uint64_t* ts) {
    using S = Shape<T, NL>;
    const Stamp st(ts);
    __shared__ v4i smem[kSmem<T, NL>];
    // workgroups go round-robin over the 8 XCDs: each takes a contiguous range of the tiles (any count), so
    // that tiles sharing A and B bands meet in one L2
    const uint32_t x = blockIdx.x & 7, q = gridDim.x >> 3, r = gridDim.x & 7;
    uint32_t tm, tn;
    tile_coords(p, x * q + min(x, r) + (blockIdx.x >> 3), tm, tn);
    fused_edge<T, S::GM, S::GN, S::NS, NL>(p, tm, tn, smem, st);
    st.inner(1);
    st.end();
}

// Tiles of many products, listed by decreasing cost; in each run of 256 workgroups an XCD takes 32
// consecutive tiles.
template <int T, int NL, int THREADS = kThreads<T, NL>, int MINB = Shape<T, NL>::MINB>
__global__ void __launch_bounds__(THREADS, MINB) fused_grouped_kernel(const FusedArgs* __restrict__ items,
                                                                  const uint32_t* __restrict__ start,
                                                                  const uint32_t* __restrict__ owner) {
    using S = Shape<T, NL>;
    __shared__ v4i smem[kSmem<T, NL>];
    const uint32_t b = blockIdx.x, run = b & ~255u;
    const uint32_t w = run + 256 <= gridDim.x ? run + (b & 7) * 32 + ((b & 255) >> 3) : b;
    const uint32_t it = owner[w];
    const FusedArgs& p = items[it];
    uint32_t tm, tn;
    tile_coords(p, w - start[it], tm, tn);
    const Stamp none(nullptr);
    fused_edge<T, S::GM, S::GN, S::NS, NL>(p, tm, tn, smem, none);
}

}  // namespace

#define OZ2_FUSED_CASES(F) F(64, 2) F(64, 3) F(64, 4) F(64, 5) F(64, 6) F(128, 2) F(128, 3) F(128, 4) F(128, 5) F(128, 6)

void fused(const Stream& st, int tile, const FusedArgs& a) {
    const uint32_t n = static_cast<uint32_t>(a.tiles_m) * a.tiles_n;
    if (n == 0) return;
    switch (tile * 8 + a.nl) {
#define OZ2_CASE(T, NL) \
    case T * 8 + NL: launch(st, fused_kernel<T, NL>, dim3(n), dim3(kThreads<T, NL>), a); break;
        OZ2_FUSED_CASES(OZ2_CASE)
#undef OZ2_CASE
    }
}

// one launch per (tile, limb count)
void prep_fused(std::vector<GroupedLaunch>& out, const std::vector<FusedJob>& jobs) {
    std::vector<GroupedLaunch> by(128 * 8 + 8);
    for (const FusedJob& j : jobs) {
        const uint32_t n = static_cast<uint32_t>(j.args.tiles_m) * j.args.tiles_n;
        if (n == 0) continue;
        GroupedLaunch& g = by[j.tile * 8 + j.args.nl];
        g.kind = j.tile * 8 + j.args.nl;
        g.owner.insert(g.owner.end(), n, g.n);
        g.add(j.args, n);
    }
    for (GroupedLaunch& g : by)
        if (g.n) out.push_back(std::move(g));
}

void launch_fused_grouped(hipStream_t st, const GroupedLaunch& g) {
    const FusedArgs* items = static_cast<const FusedArgs*>(g.d_items);
    switch (g.kind) {
#define OZ2_CASE(T, NL)                                                                                           \
    case T * 8 + NL:                                                                                              \
        hipLaunchKernelGGL((fused_grouped_kernel<T, NL>), dim3(g.blocks), dim3(kThreads<T, NL>), 0, st, items,    \
                           g.d_start, g.d_owner);                                                                 \
        break;
        OZ2_FUSED_CASES(OZ2_CASE)
#undef OZ2_CASE
    }
}

}  // namespace k
}  // namespace oz2
