// planner.cpp - workspace layout and panel planner (see planner.hpp).
#include "planner.hpp"

#include <algorithm>
#include <cmath>
#include <limits>
#include <stdexcept>
#include <string>

#include "plan.hpp"

namespace oz2 {

namespace {
inline int64_t round_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }
inline int64_t ceil_div(int64_t v, int64_t a) { return (v + a - 1) / a; }
inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Plane strides that are multiples of 64 KiB put the same offset of every plane
// on the same HBM channels; the GEMM (one plane per XCD range) and the CRT (all
// planes of one entry) read those offsets at the same time.  Tuning::pad_lda
// staggers such strides by 4 KiB, the counterpart of the reference's ld pad
// for cache-set conflicts (ozaki2_gpu.hpp:669-672).
constexpr int64_t kPlanePadPeriod = 64 << 10;
constexpr int64_t kPlanePad = 4 << 10;
inline int64_t plane_stride(int64_t bytes, bool pad) {
    return pad && bytes % kPlanePadPeriod == 0 ? bytes + kPlanePad : bytes;
}

// Rates of this library's kernels on MI355X.  Only their ratios steer the choice.
// GEMM: a macro tile's k loop runs at `peak` (all CUs busy) and its prologue and
// residue epilogue cost as much as `k0` more k (fitted to 256 x 256 at 8192^3 2.5,
// 2048^3 2.1 and 4096 x 4096 x 256 0.77 Pop/s; 256 x 128 at 2.0 and 0.96).
struct TileRate {
    double peak;  // int8 op/s of the whole GPU
    double k0;    // k-equivalent fixed cost per tile
};
constexpr TileRate kTileRate[4] = {
    {2.60e15, 450.0},  // T256
    {2.07e15, 420.0},  // T128
    {1.00e15, 300.0},  // T64
    {2.12e15, 310.0},  // T256x128
};
// scale, split and CRT move their algorithmic bytes at 4.4-5.2 TB/s; one launch ~6 us
constexpr double kStreamRate = 4.7e12;
constexpr double kLaunchSec = 6e-6;

// Seconds of the INT8 GEMM tiles on MI355X: a tile with a k loop of `len` takes a + b len where c + 1 of its kind
// share the CU (fitted to 512^2 .. 4096^2, s = 16, k = 128 .. 8192, within 8 %).
struct TileTime {
    double a[4], b[4];
};
constexpr TileTime kTileTime[4] = {
    {{6.0e-6}, {12.2e-9}},                                                    // T256
    {{2.2e-6, 3.0e-6}, {4.1e-9, 7.4e-9}},                                     // T128
    {{2.3e-6, 2.3e-6, 2.4e-6, 2.5e-6}, {3.0e-9, 3.8e-9, 4.8e-9, 5.9e-9}},     // T64
    {{3.0e-6, 3.6e-6}, {7.9e-9, 14.2e-9}},                                    // T256x128
};
// share of a tile's time that a half tile at the edge takes
constexpr double kHalfTile = 0.62;

// tiles along an extent, the last one a half tile where that holds what is left
double edge_tiles(int64_t x, int64_t t, int64_t pad) {
    const int64_t full = x / t, left = x - full * t;
    return static_cast<double>(full) + (left == 0 ? 0.0 : left <= t / 2 && pad < t ? kHalfTile : 1.0);
}

// GEMM of rows x cols in tiles t: rounds that fill every CU, then what is left over, fewer to a CU
double tile_seconds(k::Tile t, int64_t rows, int64_t cols, int planes, int64_t len, int cus) {
    const TileTime& R = kTileTime[static_cast<int>(t)];
    const int per = k::tile_blocks_per_cu(t);
    auto time = [&](int c) { return R.a[c - 1] + R.b[c - 1] * static_cast<double>(len); };
    const double per_cu = edge_tiles(rows, k::tile_m(t), k::tile_pad_m(t)) * edge_tiles(cols, k::tile_n(t), k::tile_pad_n(t)) *
                          planes / cus;
    const double full = std::floor(per_cu / per);
    const int left = static_cast<int>(std::ceil(per_cu - full * per));
    return full * time(per) + (left ? time(left) : 0.0);
}

// distinct balanced panel extents of x: x itself, then round_up(ceil(x / p), 64)
// for p = 2, 3, ... down to 64 (each value once, largest first)
template <class F>
void for_each_panel(int64_t x, F&& f) {
    f(x);
    int64_t b = x;
    int64_t p = 2;
    while (b > 64) {
        const int64_t nb = round_up(ceil_div(x, p), 64);
        if (nb < b) {
            b = nb;
            f(b);
        }
        if (b <= 64) break;
        // the next panel count that gives a smaller extent: ceil(x / p') <= b - 64
        p = std::max(p + 1, ceil_div(x, b - 64));
    }
}

// GEMM seconds of one launch over r x c of the panel grid (tile t, k loops of klen)
double gemm_seconds(const CallShape& c, const Layout& L, k::Tile tile, int64_t rows, int64_t cols) {
    const TileRate& R = kTileRate[static_cast<int>(tile)];
    const int64_t TM = k::tile_m(tile), TN = k::tile_n(tile);
    const double tiles = static_cast<double>(ceil_div(rows, TM)) * static_cast<double>(ceil_div(cols, TN)) * L.planes;
    const double slots = static_cast<double>(c.cus) * k::tile_blocks_per_cu(tile);
    const double waves = std::ceil(tiles / slots);
    double t = 0;
    for (int64_t k0 = 0; k0 < L.kp; k0 += L.klen) {
        const double len = static_cast<double>(std::min(L.klen, L.kp - k0));
        // one wave of `slots` tiles takes 2 TM TN (len + k0) slots / peak
        t += waves * 2.0 * TM * TN * (len + R.k0) * slots / R.peak;
    }
    return t;
}
}  // namespace

namespace {
// longest k at which 128 x 128 tiles of the fused kernel are ahead of the separate ones in full rounds, us on
// MI355X, separate / fused: 4096 x 4096 x 768 s = 8 192 / 181, x 1024 220 / 227; x 1024 s = 16 439 / 410;
// 2048 x 2048 x 1024 s = 16 109 / 93, x 1536 139 / 129, 4096 x 4096 x 1024 s = 24 679 / 676
int64_t fused_k(int s) { return limbs_for(s) == 2 ? 512 : limbs_for(s) == 6 ? 768 : 1024; }
}  // namespace

int fused_tile(const CallShape& c, const Layout& L, int64_t mb, int64_t nb) {
    if (c.cplx || L.kch != 1 || c.per_plane || c.forced_tile != -1) return 0;
    const int nl = limbs_for(c.s);
    const double area = static_cast<double>(mb) * static_cast<double>(nb), cus = c.cus;
    // 64 x 64 tiles, three (two) per CU, pay at short k, where the separate path is mostly traffic, also with
    // ragged rounds; with less than 0.6 of a round (1024 x 1024 x 256 s = 16: 19.3 / 19.3 us) nothing is gained.
    // Separate / 64 tiles: 1408 x 1408 x 256 s = 16 35 / 26, 3000 x 3000 x 256 131 / 97, x 1024 241 / 268,
    // 2304 x 2304 s = 20 k = 128 81 / 71, k = 256 92 / 90.  Above 20 moduli the 128 tiles spill: 8192 x 8192
    // x 128 s = 24 1261 / 891, 128 tiles 1084.
    const bool t64 = L.kp <= (nl > 4 ? 128 : 256) && area >= 0.6 * 64 * 64 * fused_per_cu(64, c.s) * cus;
    if (nl == 6 && t64) return 64;
    // 128 x 128 tiles, one per CU, want their rounds full: the fused rounds are long (s planes each), the
    // separate path's are a plane each.  3000 x 3000 x 256 s = 16 (72 %) 131 / 118, x 1024 241 / 253; s = 8
    // x 256 72 / 80; 2816 x 2816 (95 %) x 256 s = 8 61 / 59.
    const double rounds = std::ceil(static_cast<double>(ceil_div(mb, 128)) * static_cast<double>(ceil_div(nb, 128)) / cus);
    if (L.kp <= fused_k(c.s) && area >= 0.8 * 128 * 128 * cus * rounds && L.TM % 128 == 0 && L.TN % 128 == 0) return 128;
    return t64 ? 64 : 0;
}

int fused_batch_tile(k::Tile tile, int64_t kp, int64_t kch, int s) {
    if (kch != 1 || kp > fused_k(s)) return 0;
    return tile == k::Tile::T64 ? 64 : 128;
}

bool same_call(const CallShape& a, const CallShape& b) {
    return a.m == b.m && a.n == b.n && a.k == b.k && a.s == b.s && a.cplx == b.cplx && a.partial_a == b.partial_a &&
           a.partial_b == b.partial_b && a.cus == b.cus && a.pad_planes == b.pad_planes && a.pow2 == b.pow2 &&
           a.per_plane == b.per_plane && a.forced_tile == b.forced_tile;
}

k::Tile pick_tile(int64_t mb, int64_t nb, int64_t klen, int planes, int forced_code) {
    k::Tile forced;
    if (k::tile_from_code(forced_code, forced)) return forced;
    // never pad a small tile up to a bigger macro tile
    const int64_t lim = std::min(mb, nb);
    if (lim <= 64) return k::Tile::T64;
    auto blocks = [&](int64_t tm, int64_t tn) { return ceil_div(mb, tm) * ceil_div(nb, tn) * planes; };
    // k loops of at most 1024: 256 x 128 tiles, two workgroups per CU (measured
    // ahead of both square tiles there, behind 256 x 256 for long k)
    if (klen <= 1024 && mb > 128 && nb > 64 && blocks(256, 128) >= 512) return k::Tile::T256x128;
    // largest square tile that still gives every CU two workgroups
    if (lim > 128 && blocks(256, 256) >= 512) return k::Tile::T256;
    if (blocks(128, 128) >= 512) return k::Tile::T128;
    return blocks(128, 128) >= 256 ? k::Tile::T128 : k::Tile::T64;
}

k::Tile call_tile(int64_t mb, int64_t nb, int64_t klen, int planes, int forced_code, int cus) {
    k::Tile forced;
    if (k::tile_from_code(forced_code, forced)) return forced;
    // never pad a small tile up to a bigger macro tile
    if (std::min(mb, nb) <= 64) return k::Tile::T64;
    // The fastest by tile_seconds.  GEMM, us, pick_tile's / this one: 1024^3 s = 14 20.2 (128 x 128) / 17.0
    // (256 x 128), 2048^3 s = 10 89.0 / 82.6, 2048 x 300 x 4096 s = 16 55.4 / 53.5; of 20 sizes from 100^3 to 4096^2
    // one was slower (130 x 8000 x 1000 35.6 / 37.8, the call the same).  In a batch the neighbours fill the chip,
    // and its tiles lose (64 products of 64 .. 1024: 513 / 597).
    k::Tile best = k::Tile::T64;
    double least = std::numeric_limits<double>::infinity();
    for (k::Tile t : {k::Tile::T256, k::Tile::T256x128, k::Tile::T128, k::Tile::T64}) {
        if ((t == k::Tile::T256 && std::min(mb, nb) <= 128) || (t == k::Tile::T256x128 && mb <= 128)) continue;
        const double s = tile_seconds(t, mb, nb, planes, klen, cus);
        if (s < least) {
            least = s;
            best = t;
        }
    }
    return best;
}

k::Tile panel_tile(const CallShape& c, int64_t mb, int64_t nb) {
    const int planes = (c.cplx ? 3 : 1) * c.s;
    const int64_t klen = k_chunk_len(round_up(c.k, kKStep));
    // (panels of a call that does not fit keep the simpler rule, whose cost the search over them can rely on to
    // fall with larger panels)
    return mb == c.m && nb == c.n ? call_tile(mb, nb, klen, planes, c.forced_tile, c.cus)
                                  : pick_tile(mb, nb, klen, planes, c.forced_tile);
}

Layout layout(const CallShape& c, int64_t mb, int64_t nb, k::Tile tile) {
    Layout L;
    L.g = c.cplx ? 3 : 1;
    L.planes = L.g * c.s;
    L.kp = round_up(c.k, kKStep);
    L.klen = k_chunk_len(L.kp);
    L.kch = k_chunks(L.kp);
    L.tile = tile;
    L.TM = k::tile_m(L.tile);
    L.TN = k::tile_n(L.tile);
    L.mpad = round_up(mb, L.TM);
    L.npad = round_up(nb, L.TN);
    L.planeA = plane_stride(L.mpad * L.kp, c.pad_planes);
    L.planeB = plane_stride(L.npad * L.kp, c.pad_planes);
    L.planeR = plane_stride(L.npad * L.mpad, c.pad_planes);
    size_t off = 0;
    auto carve = [&](size_t bytes) {
        const size_t o = off;
        off = align_up(off + bytes, 256);
        return o;
    };
    L.oD = carve(static_cast<size_t>(c.m) * 4);
    L.oE = carve(static_cast<size_t>(c.n) * 4);
    L.oPA = carve(c.partial_a);
    L.oPB = carve(c.partial_b);
    L.oA = carve(static_cast<size_t>(L.planes) * L.planeA);
    L.oB = carve(static_cast<size_t>(L.planes) * L.planeB);
    L.oR = carve(static_cast<size_t>(L.kch) * L.planes * L.planeR);
    L.total = off + 4096;
    return L;
}

double panel_cost(const CallShape& c, int64_t mb, int64_t nb, k::Tile layout_tile) {
    const Layout L = layout(c, mb, nb, layout_tile);
    const int64_t pm = ceil_div(c.m, mb), pn = ceil_div(c.n, nb);
    const int64_t mlast = c.m - (pm - 1) * mb, nlast = c.n - (pn - 1) * nb;
    // GEMM launches: (pm - 1) x (pn - 1) full panel pairs, the ragged last row and column
    // (priced with the tiles of a panel, the whole call too, so that the panel counts compare)
    double gemm = 0;
    const k::Tile tile = pick_tile(mb, nb, L.klen, L.planes, c.forced_tile);
    gemm += static_cast<double>((pm - 1) * (pn - 1)) * gemm_seconds(c, L, tile, mb, nb);
    gemm += static_cast<double>(pn - 1) * gemm_seconds(c, L, tile, mlast, nb);
    gemm += static_cast<double>(pm - 1) * gemm_seconds(c, L, tile, mb, nlast);
    gemm += gemm_seconds(c, L, tile, mlast, nlast);
    // bandwidth-bound bytes: each split reads its operand and writes the padded planes;
    // op(A) is split once when it is one row panel, else once per panel pair; the CRT
    // reads every residue byte and reads and writes C
    const double elem = c.cplx ? 16.0 : 8.0;
    const double mpad_all = static_cast<double>((pm - 1) * round_up(mb, L.TM) + round_up(mlast, L.TM));
    const double npad_all = static_cast<double>((pn - 1) * round_up(nb, L.TN) + round_up(nlast, L.TN));
    const double kd = static_cast<double>(c.k), kpd = static_cast<double>(L.kp);
    const double split_b = static_cast<double>(c.n) * kd * elem + L.planes * npad_all * kpd;
    const double split_a = static_cast<double>(pm > 1 ? pn : 1) * (static_cast<double>(c.m) * kd * elem + L.planes * mpad_all * kpd);
    const double crt = static_cast<double>(c.m) * static_cast<double>(c.n) * (L.planes * L.kch + 2.0 * elem);
    const double launches = static_cast<double>(pn + (pm > 1 ? pm * pn : 1) + pm * pn) +
                            static_cast<double>(pm * pn * L.kch) * (c.per_plane ? L.planes : 1);
    return gemm + (split_a + split_b + crt) / kStreamRate + launches * kLaunchSec;
}

TileInfo plan_tiling(const CallShape& c, size_t limit) {
    // A call that fits whole only with the padding of pick_tile's tile takes that one: 294 x 525 x 87 s = 16 needs 4.6 MiB
    // with 64 x 64 tiles, 5.8 with call_tile's.  At limits between, us, in panels / whole: this one 31.8 / 17.7, 783 x 507
    // x 73 s = 24 41.1 / 27.2, complex 163 x 180 x 414 s = 20 48.7 / 31.6, 2404 x 655 x 10945 s = 8 362 / 335.
    const k::Tile small = pick_tile(c.m, c.n, k_chunk_len(round_up(c.k, kKStep)), (c.cplx ? 3 : 1) * c.s, c.forced_tile);
    const k::Tile whole = layout(c, c.m, c.n).total <= limit ? panel_tile(c, c.m, c.n) : small;
    auto tile_of = [&](int64_t mb, int64_t nb) { return mb == c.m && nb == c.n ? whole : panel_tile(c, mb, nb); };
    auto fits = [&](int64_t mb, int64_t nb) { return layout(c, mb, nb, tile_of(mb, nb)).total <= limit; };
    double best = std::numeric_limits<double>::infinity();
    TileInfo bt;
    auto consider = [&](int64_t mb, int64_t nb) {
        if (!fits(mb, nb)) return;
        const k::Tile tile = tile_of(mb, nb);
        const double t = panel_cost(c, mb, nb, tile);
        // strictly cheaper only: among equal costs the first (fewest panels) stays
        if (t < best * (1.0 - 1e-12)) {
            best = t;
            const Layout L = layout(c, mb, nb, tile);
            bt = TileInfo{mb, nb, ceil_div(c.m, mb), ceil_div(c.n, nb), L.kch, L.total, tile};
        }
    };
    auto try_rows = [&](int64_t mb) {
        // largest column panel that fits: all of n, else bisection over multiples of 64
        int64_t nbmax = 0;
        if (fits(mb, c.n)) {
            nbmax = c.n;
        } else {
            int64_t lo = 0, hi = ceil_div(c.n, 64);  // fits(64 lo) (lo = 0: nothing yet), !fits(64 hi)
            while (hi - lo > 1) {
                const int64_t mid = (lo + hi) / 2;
                if (fits(mb, 64 * mid)) lo = mid;
                else hi = mid;
            }
            nbmax = 64 * lo;
        }
        if (nbmax == 0) return;
        // the fewest column panels that fit, and two more (less padding or better waves)
        const int64_t pn0 = ceil_div(c.n, nbmax);
        for (int64_t pn = pn0; pn <= pn0 + 2; ++pn) {
            const int64_t nb = pn == 1 ? c.n : round_up(ceil_div(c.n, pn), 64);
            if (nb > nbmax && nb != c.n) continue;
            if (ceil_div(c.n, nb) != pn) continue;  // this count is not reachable with balanced panels
            consider(mb, nb);
        }
        if (c.pow2)
            for (int64_t nb = 1024; nb < std::min(c.n, nbmax + 1); nb *= 2) consider(mb, nb);
    };
    for_each_panel(c.m, try_rows);
    if (c.pow2)
        for (int64_t mb = 1024; mb < c.m; mb *= 2) try_rows(mb);
    if (!std::isfinite(best))
        throw std::runtime_error("oz2: not enough device memory for workspace (limit " + std::to_string(limit >> 20) +
                                 " MiB)");
    return bt;
}

}  // namespace oz2
