// scale_split.hip - scaling (row/column max -> power-of-two exponents) and the
// exact split of op(A) / op(B) into s int8 residue planes, for gfx950.
//
// Reference behaviour: src/ozaki2_gpu.hpp:309-377 (max |x| per row / column,
// exponent D = tk - frexp_exp(max), 0 for an all-zero row, kNonFinite for
// Inf/NaN) and hpp:251-303, 407-520 (x = RNE(v 2^e) taken exactly from the
// IEEE bits, symmetric residues per modulus; complex: Re, +-Im, Re+-Im).
//
// Both operands are written in one blocked plane layout (PlaneMap: 1 KB
// blocks of 16 rows x 64 k), so the GEMM copies A and B tiles the same way.
// A thread's 16 k lie in one 16-byte chunk of a block (block_k order), so each
// plane store is one aligned vector store.  Rows of op(X)
// that are strided in memory (op(A) = N, op(B) = T) are read column-by-column
// with lanes along rows, so no separate transpose pass is needed.
#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "grouped.hpp"
#include "kernels.hpp"
#include "math.hpp"

namespace oz2 {
namespace k {
using namespace math;

namespace {

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int mask) {
    const uint32_t lo = __shfl_xor(static_cast<uint32_t>(v), mask, 64);
    const uint32_t hi = __shfl_xor(static_cast<uint32_t>(v >> 32), mask, 64);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

__device__ __forceinline__ uint64_t absbits(const double* p) {
    return __double_as_longlong(*p) & 0x7FFFFFFFFFFFFFFFll;
}

// Maximum of every row of op(X).  Rows strided in memory over several k-blocks leave a partial maximum each.
struct ScaleItem {
    const double* X;
    int64_t ldx, len, k;
    int64_t kper;         // strided rows: k of a block
    int kcontig, cplx, tk, nkb;
    uint64_t* partial;    // strided rows with nkb > 1
    int32_t* ex;
    uint32_t gx;          // blocks along the rows
    uint32_t blocks;
};
// One wave per row of op(X), row contiguous in memory: n doubles from base.
__device__ __forceinline__ void scale_kcontig_body(const ScaleItem& it, uint32_t bx) {
    const int lane = threadIdx.x & 63;
    const int64_t r = static_cast<int64_t>(bx) * 4 + (threadIdx.x >> 6);
    if (r >= it.len) return;
    const int64_t ndbl = it.cplx ? 2 * it.k : it.k;
    const double* row = it.X + (it.cplx ? 2 : 1) * r * it.ldx;
    uint64_t mx = 0;
    if ((reinterpret_cast<uintptr_t>(row) & 15) == 0) {
        const int64_t n2 = ndbl >> 1;
        const double2* row2 = reinterpret_cast<const double2*>(row);
        constexpr int U = 8;  // loads in flight per step, all at i < n2
        int64_t i = lane;
        for (; i + 64 * (U - 1) < n2; i += 64 * U) {
            double2 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = row2[i + 64 * u];
#pragma unroll
            for (int u = 0; u < U; ++u)
                mx = max(mx, max(static_cast<uint64_t>(__double_as_longlong(v[u].x) & 0x7FFFFFFFFFFFFFFFll),
                                 static_cast<uint64_t>(__double_as_longlong(v[u].y) & 0x7FFFFFFFFFFFFFFFll)));
        }
        for (; i < n2; i += 64) {
            const double2 v = row2[i];
            const uint64_t a = __double_as_longlong(v.x) & 0x7FFFFFFFFFFFFFFFll;
            const uint64_t b = __double_as_longlong(v.y) & 0x7FFFFFFFFFFFFFFFll;
            mx = max(mx, max(a, b));
        }
        if ((ndbl & 1) && lane == 0) mx = max(mx, absbits(row + ndbl - 1));
    } else {  // a row that is only 8-byte aligned (odd leading dimension): single doubles
        constexpr int U = 8;
        int64_t i = lane;
        for (; i + 64 * (U - 1) < ndbl; i += 64 * U) {
            uint64_t v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = absbits(row + i + 64 * u);
#pragma unroll
            for (int u = 0; u < U; ++u) mx = max(mx, v[u]);
        }
        for (; i < ndbl; i += 64) mx = max(mx, absbits(row + i));
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = max(mx, shfl_xor_u64(mx, o));
    if (lane == 0) it.ex[r] = exponent_from_maxbits(mx, it.tk);
}

// Rows strided in memory: block = 64 rows x 4 k-lanes over a k range; partial max per (k block, row), the
// exponent itself with one k block.
__device__ __forceinline__ void scale_kstrided_body(const ScaleItem& it, uint32_t bx, uint32_t by) {
    __shared__ uint64_t red[4][64];
    const int rl = threadIdx.x & 63, kl = threadIdx.x >> 6;
    const int64_t r = static_cast<int64_t>(bx) * 64 + rl;
    const int64_t p0 = static_cast<int64_t>(by) * it.kper;
    const int64_t p1 = min(it.k, p0 + it.kper);
    const double* X = it.X;
    const int64_t ldx = it.ldx;
    uint64_t mx = 0;
    if (r < it.len) {
        // U loads in flight per step (all of them at k < p1), then the remainder one by one:
        // a single load per step leaves each wave waiting out the full memory latency
        constexpr int U = 8;
        int64_t p = p0 + kl;
        if (it.cplx) {
            for (; p + 4 * (U - 1) < p1; p += 4 * U) {
                double2 v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const double2*>(X + 2 * (r + (p + 4 * u) * ldx));
#pragma unroll
                for (int u = 0; u < U; ++u)
                    mx = max(mx, max(static_cast<uint64_t>(__double_as_longlong(v[u].x) & 0x7FFFFFFFFFFFFFFFll),
                                     static_cast<uint64_t>(__double_as_longlong(v[u].y) & 0x7FFFFFFFFFFFFFFFll)));
            }
            for (; p < p1; p += 4) {
                const double2 v = *reinterpret_cast<const double2*>(X + 2 * (r + p * ldx));
                mx = max(mx, max(static_cast<uint64_t>(__double_as_longlong(v.x) & 0x7FFFFFFFFFFFFFFFll),
                                 static_cast<uint64_t>(__double_as_longlong(v.y) & 0x7FFFFFFFFFFFFFFFll)));
            }
        } else {
            for (; p + 4 * (U - 1) < p1; p += 4 * U) {
                uint64_t v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = absbits(X + r + (p + 4 * u) * ldx);
#pragma unroll
                for (int u = 0; u < U; ++u) mx = max(mx, v[u]);
            }
            for (; p < p1; p += 4) mx = max(mx, absbits(X + r + p * ldx));
        }
    }
    red[kl][rl] = mx;
    __syncthreads();
    if (kl == 0 && r < it.len) {
        mx = max(max(red[0][rl], red[1][rl]), max(red[2][rl], red[3][rl]));
        if (it.nkb == 1) it.ex[r] = exponent_from_maxbits(mx, it.tk);
        else it.partial[static_cast<int64_t>(by) * it.len + r] = mx;
    }
}

__device__ __forceinline__ void scale_body(const ScaleItem& it, uint32_t l) {
    if (it.kcontig) scale_kcontig_body(it, l);
    else scale_kstrided_body(it, l % it.gx, l / it.gx);
}

__device__ __forceinline__ void scale_finalize_body(const ScaleItem& it, uint32_t bx) {
    const int64_t r = static_cast<int64_t>(bx) * 256 + threadIdx.x;
    if (r >= it.len) return;
    uint64_t mx = 0;
    int b = 0;
    for (; b + 3 < it.nkb; b += 4) {  // four loads in flight, all at b < nkb
        uint64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = it.partial[static_cast<int64_t>(b + u) * it.len + r];
        mx = max(mx, max(max(v[0], v[1]), max(v[2], v[3])));
    }
    for (; b < it.nkb; ++b) mx = max(mx, it.partial[static_cast<int64_t>(b) * it.len + r]);
    it.ex[r] = exponent_from_maxbits(mx, it.tk);
}

// Both operands of a product in one launch: the first a.blocks blocks are a's.  A launch of its own for each
// costs 3 us where the operands are small, and leaves the chip half empty.  MI355X, scale and split of both, us,
// launches of their own / together (exponents from partials in the split included): 64^3 s = 16 23.5 / 9.4,
// 1024^3 s = 14 32 / 22, 4096 x 256 by 256 x 4096 s = 16 40 / 21.
__global__ void __launch_bounds__(256) scale_kernel(ScaleItem a, ScaleItem b, uint64_t* ts) {
    const Stamp st(ts);
    const bool second = blockIdx.x >= a.blocks;
    const ScaleItem it = second ? b : a;
    scale_body(it, second ? blockIdx.x - a.blocks : blockIdx.x);
    st.end();
}
// ex of the rows of a and of b from their partials; na blocks are a's
__global__ void __launch_bounds__(256) scale_finalize_kernel(ScaleItem a, ScaleItem b, uint32_t na, uint64_t* ts) {
    const Stamp st(ts);
    const bool second = blockIdx.x >= na;
    const ScaleItem it = second ? b : a;
    scale_finalize_body(it, second ? blockIdx.x - na : blockIdx.x);
    st.end();
}

constexpr int64_t kScaleRowsPerBlock = 64;
// Up to this many partial maxima a row the split reads them itself (512 bytes a block each, beside its 32 KB
// of operand), instead of a launch that reduces them: 2.2 to 4.3 us at k = 257 to 4096, where calls take 50 to
// 200.  With more of them the launch's 5 to 20 us are a thousandth of the call.
constexpr int kScaleFold = 16;
// Blocks that a split of few blocks deals its moduli to: one a CU, four for complex data, whose blocks take three
// groups of planes.  64^3 s = 16, 2 blocks: 7.8 us an operand undealt, 5.2 for both.  Calls, us, 256 / 512 / 1024 /
// 2048: complex 777 x 1023 x 515 (300 blocks) 94.6 / 94.5 / 91.5 / 92.3, 1024^3 s = 14 (512) 47.2 / 47.0 / 48.2 /
// 50.4, 1500 x 900 x 2000 in panels (256) 132.4 / 132.3 / 134.1 / 134.5.
constexpr uint32_t kSplitBlocks = 256, kSplitBlocksCplx = 1024;

int64_t scale_kblocks(int64_t len, int64_t k) {
    const int64_t rb = (len + kScaleRowsPerBlock - 1) / kScaleRowsPerBlock;
    int64_t kb = (4096 + rb - 1) / rb;
    kb = std::max<int64_t>(1, std::min<int64_t>(kb, (k + 255) / 256));
    return std::min<int64_t>(kb, 65535);
}

ScaleItem scale_item(const ScaleJob& j) {
    ScaleItem it{j.X, j.ldx, j.len, j.k, j.k, j.kcontig ? 1 : 0, j.cplx ? 1 : 0, j.tk, 1, j.partial, j.ex, 0, 0};
    if (j.len <= 0) return it;
    if (j.kcontig) {
        it.blocks = it.gx = static_cast<uint32_t>((j.len + 3) / 4);
    } else {
        it.nkb = static_cast<int>(scale_kblocks(j.len, j.k));
        it.kper = (j.k + it.nkb - 1) / it.nkb;
        it.gx = static_cast<uint32_t>((j.len + kScaleRowsPerBlock - 1) / kScaleRowsPerBlock);
        it.blocks = it.gx * static_cast<uint32_t>(it.nkb);
    }
    return it;
}
// blocks of the launch that finalizes the item's exponents: none where the scale kernel wrote them or the split does
uint32_t finalize_blocks(const ScaleJob& j, const ScaleItem& it) {
    return it.blocks && it.nkb > 1 && !(j.fold && scale_folds(j.len, j.k, j.kcontig)) ? static_cast<uint32_t>((j.len + 255) / 256) : 0;
}

// ---------------------------------------------------------------------------
// split
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint64_t bits_of(const double* p) { return static_cast<uint64_t>(__double_as_longlong(*p)); }
__device__ __forceinline__ uint64_t word64(uint32_t lo, uint32_t hi) { return static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32); }

// Thread slot of a split: Q bytes (Q = 16: a whole 16-byte chunk, Q = 8: half of one) of
// one row of the planes.  ck counts the slots along the row.
template <int Q>
struct SplitSlot {
    static_assert(Q == 16 || Q == 8, "a slot is a chunk or half a chunk");
    int64_t blk;  // 64-k block
    int c;        // chunk in the block
    int q0;       // first byte of the chunk filled by this slot
    int64_t kb;   // byte q of the chunk holds k = kb + 8 (q >> 1) + (q & 1)
    __device__ __forceinline__ explicit SplitSlot(int64_t ck) {
        constexpr int per_blk = 64 / Q;
        blk = ck / per_blk;
        const int ib = static_cast<int>(ck % per_blk);
        c = ib / (16 / Q);
        q0 = (ib % (16 / Q)) * Q;
        kb = blk * 64 + 2 * c;
    }
    __device__ __forceinline__ int64_t k_of(int q) const { return kb + 8 * ((q0 + q) >> 1) + ((q0 + q) & 1); }
};

// A split of one operand.  Rows contiguous in memory (X[p + r*ldx]): a block covers 256 slots, 1 << lg of
// each row.  Rows strided (X[r + p*ldx]): a block is one 64-k block of 4 bands (2 for half chunks), lanes along
// rows, so a wave (16 rows x 4 slots) reads one 128-byte line per load, and the block 512 bytes of a column,
// and writes a run of plane blocks.
struct SplitItem {
    SplitArgs a;
    int lg;
    int tper;         // moduli of a block (all of them, or a part where the blocks are few)
    uint32_t gx, gy;  // blocks along the rows, along k
    uint32_t blocks;  // gx gy, times the parts of the moduli
};

constexpr uint32_t kStrip = 16;

// What a thread of a split works on.  SCALE: the block holds all k of its 64 rows, 256 threads for each 64-k block.
template <int Q, bool SCALE = false>
struct SplitThread {
    int64_t r, ck;    // row, slot
    int t0, t1;       // moduli
    bool ok;          // inside the planes
    int32_t ex;       // exponent of the row (INT32_MIN outside the matrix)

    __device__ __forceinline__ SplitThread(const SplitItem& it, uint32_t l) {
        const SplitArgs& a = it.a;
        t0 = 0;
        t1 = a.s;
        if (it.tper < a.s) {
            const uint32_t per = it.gx * it.gy, g = __builtin_amdgcn_readfirstlane(l / per);
            l -= g * per;
            t0 = static_cast<int>(g) * it.tper;
            t1 = min(a.s, t0 + it.tper);
        }
        // rows first; contiguous rows in strips of kStrip blocks along k, so that what runs together reads runs of
        // 8 KB of a row, not 512 bytes at a stride that a power of two puts on few channels (MI355X, calls, us,
        // rows first / strips: 4096^3 s = 8 654 / 640, complex 4096^3 3410 / 3363, k = 200000 20863 / 20810)
        uint32_t bx, by;
        if (SCALE) {
            by = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
            bx = l;
        } else if (a.kcontig) {
            const uint32_t strip = __builtin_amdgcn_readfirstlane(l / (it.gx * kStrip)), in = l - strip * it.gx * kStrip;
            const uint32_t n = min(kStrip, it.gy - strip * kStrip);
            bx = __builtin_amdgcn_readfirstlane(in / n);
            by = strip * kStrip + in - bx * n;
        } else {
            by = __builtin_amdgcn_readfirstlane(l / it.gx);
            bx = l - by * it.gx;
        }
        constexpr int slots = 64 / Q;
        const int tid = SCALE ? threadIdx.x & 255 : threadIdx.x, wq = tid >> 4;  // strided rows: 16 rows x one slot
        if (a.kcontig) {
            r = static_cast<int64_t>(bx) * (256 >> it.lg) + (tid >> it.lg);
            ck = (static_cast<int64_t>(by) << it.lg) + (tid & ((1 << it.lg) - 1));
        } else {
            r = static_cast<int64_t>(bx) * (256 / slots) + wq / slots * 16 + (tid & 15);
            ck = static_cast<int64_t>(by) * slots + wq % slots;
        }
        ok = r < a.rows_pad && ck < a.kp / Q;
        const bool in = ok && r < a.rows;
        ex = INT32_MIN;
        if (SCALE) return;
        if (a.part) {
            // the row's maximum from the scale kernel's partials: the four lanes of a wave that hold the row
            // (16 apart) take every fourth
            uint64_t mx = 0;
            if (in)
                for (int b = (threadIdx.x >> 4) & 3; b < a.nkb; b += 4) mx = max(mx, a.part[static_cast<int64_t>(b) * a.part_ld + r]);
            mx = max(mx, shfl_xor_u64(mx, 16));
            mx = max(mx, shfl_xor_u64(mx, 32));
            if (in) {
                ex = exponent_from_maxbits(mx, a.tk);
                if (ck == 0 && t0 == 0) a.ex_out[r] = ex;
            }
        } else if (in) {
            ex = a.ex[r];
        }
    }
};

// Q bytes packed little-endian from 32-bit words: one Q-byte store
template <int Q>
__device__ __forceinline__ void store_bytes(int8_t* p, const uint32_t (&w)[4]) {
    if (Q == 16) *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
    else *reinterpret_cast<uint2*>(p) = make_uint2(w[0], w[1]);
}

// Real split: Q bytes (Q of the k of one row, block_k order) per thread -> one
// Q-byte store per plane.  All loads are issued before any arithmetic and stay
// inside the matrix: padding rows read row 0 and k past the end reads k - 1, and
// those values are then zeroed.
template <int FORM, int Q, bool SCALE = false>
__device__ __forceinline__ void split_real_body(const SplitItem& it, uint32_t l, const Stamp* st = nullptr) {
    const SplitArgs& a = it.a;
    const auto tb = const_tab(a.tab);
    SplitThread<Q, SCALE> th(it, l);
    if (!SCALE && !th.ok) return;
    const SplitSlot<Q> sl(th.ck);
    const int64_t rl = th.r < a.rows ? th.r : 0;

    uint64_t bits[Q];
    const bool full = sl.blk * 64 + 64 <= a.k;
    if (full && a.kcontig) {
        const double* rowp = a.X + rl * a.ldx + sl.kb;
        if ((reinterpret_cast<uintptr_t>(rowp) & 15) == 0) {
#pragma unroll
            for (int i = 0; i < Q / 2; ++i) {
                const uint4 v = *reinterpret_cast<const uint4*>(rowp + sl.k_of(2 * i) - sl.kb);
                bits[2 * i] = word64(v.x, v.y);
                bits[2 * i + 1] = word64(v.z, v.w);
            }
        } else {
#pragma unroll
            for (int q = 0; q < Q; ++q) bits[q] = bits_of(rowp + (sl.k_of(q) - sl.kb));
        }
    } else if (full) {
#pragma unroll
        for (int q = 0; q < Q; ++q) bits[q] = bits_of(a.X + rl + sl.k_of(q) * a.ldx);
    } else {
        const int64_t sr = a.kcontig ? a.ldx : 1, sp = a.kcontig ? 1 : a.ldx;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int64_t p = sl.k_of(q);
            bits[q] = bits_of(a.X + rl * sr + (p < a.k ? p : a.k - 1) * sp);
            bits[q] = p < a.k ? bits[q] : 0;
        }
    }

    if constexpr (SCALE) {
        // the rows' maxima: the four threads that share a row in a 64-k block, then the k blocks
        static_assert(Q == 16, "four threads a row");
        __shared__ uint64_t red[4][64];
        uint64_t mx = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) mx = max(mx, bits[q] & 0x7FFFFFFFFFFFFFFFull);
        mx = max(mx, shfl_xor_u64(mx, a.kcontig ? 1 : 16));
        mx = max(mx, shfl_xor_u64(mx, a.kcontig ? 2 : 32));
        const int row = static_cast<int>(th.r & 63);
        if ((th.ck & 3) == 0) red[threadIdx.x >> 8][row] = mx;
        __syncthreads();
        mx = 0;
        for (int b = 0; b < static_cast<int>(blockDim.x >> 8); ++b) mx = max(mx, red[b][row]);
        if (th.r < a.rows) {
            th.ex = exponent_from_maxbits(mx, a.tk);
            if (th.ck == 0 && th.t0 == 0) a.ex_out[th.r] = th.ex;
        }
        st->inner(0);
    }
    const bool rowzero = th.ex == INT32_MIN;
    const int e = rowzero ? 0 : th.ex;

    // two to four words (limb_form of tk)
    constexpr Limbs F = static_cast<Limbs>(FORM);
    uint32_t limbs[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) to_limbs<F>(rowzero ? 0 : bits[q], e, false, limbs[q]);
    int8_t* out = a.P + chunk_offset(th.r, sl.blk, sl.c, a.map) + sl.q0;
    uint32_t w[4] = {0, 0, 0, 0};
    auto low = [&] {
#pragma unroll
        for (int g = 0; g < Q / 4; ++g)
            w[g] = pack_lo_bytes(limbs[4 * g][0], limbs[4 * g + 1][0], limbs[4 * g + 2][0], limbs[4 * g + 3][0]);
        store_bytes<Q>(out, w);
    };
    auto plane = [&](int t, auto exact) {
        constexpr bool E = decltype(exact)::value;
#pragma unroll
        for (int g = 0; g < Q / 4; ++g)
            w[g] = pack_lo_bytes(sym_residue<F, E>(limbs[4 * g], tb, t), sym_residue<F, E>(limbs[4 * g + 1], tb, t),
                                 sym_residue<F, E>(limbs[4 * g + 2], tb, t), sym_residue<F, E>(limbs[4 * g + 3], tb, t));
        store_bytes<Q>(out + t * a.plane, w);
    };
    for_moduli<F>(th.t0, th.t1, low, plane);
}

// Complex split: three plane groups Re, Im (negated for conj: the sign of the bits), Re+Im, each
// reduced to the symmetric range [-h, m-1-h]; slots, k order and loads as in the
// real split, one Q-byte store per plane of each group.
template <int FORM, int Q>
__device__ __forceinline__ void split_cplx_body(const SplitItem& it, uint32_t l) {
    const SplitArgs& a = it.a;
    const auto tb = const_tab(a.tab);
    const SplitThread<Q> th(it, l);
    if (!th.ok) return;
    const SplitSlot<Q> sl(th.ck);
    const bool rowzero = th.ex == INT32_MIN;
    const int e = rowzero ? 0 : th.ex;
    const int64_t rl = th.r < a.rows ? th.r : 0;

    uint64_t br[Q], bi[Q];
    const bool full = sl.blk * 64 + 64 <= a.k;
    const double* rowp = a.X + 2 * rl * a.ldx + 2 * sl.kb;
    if (a.kcontig && full && (reinterpret_cast<uintptr_t>(rowp) & 15) == 0) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint4 v = *reinterpret_cast<const uint4*>(rowp + 2 * (sl.k_of(q) - sl.kb));
            br[q] = word64(v.x, v.y);
            bi[q] = word64(v.z, v.w);
        }
    } else {
        const int64_t sr = a.kcontig ? a.ldx : 1, sp = a.kcontig ? 1 : a.ldx;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int64_t p = sl.k_of(q);
            const double* x = a.X + 2 * (rl * sr + (p < a.k ? p : a.k - 1) * sp);
            br[q] = bits_of(x);
            bi[q] = bits_of(x + 1);
            br[q] = p < a.k ? br[q] : 0;
            bi[q] = p < a.k ? bi[q] : 0;
        }
    }
    const uint64_t flip = a.conj ? 1ull << 63 : 0;
    constexpr Limbs F = static_cast<Limbs>(FORM);
    uint32_t lr[Q][4], li[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        to_limbs<F>(rowzero ? 0 : br[q], e, false, lr[q]);
        to_limbs<F>(rowzero ? 0 : bi[q] ^ flip, e, false, li[q]);
    }
    int8_t* out = a.P + chunk_offset(th.r, sl.blk, sl.c, a.map) + sl.q0;
    // plane t of the three groups; residues(x, y, r) of an element
    auto plane = [&](int t, const auto& residues) {
        uint32_t w0[4] = {0, 0, 0, 0}, w1[4] = {0, 0, 0, 0}, w2[4] = {0, 0, 0, 0};
#pragma unroll
        for (int g = 0; g < Q / 4; ++g) {
            uint32_t r[4][3];
#pragma unroll
            for (int q = 0; q < 4; ++q) residues(lr[4 * g + q], li[4 * g + q], r[q]);
            w0[g] = pack_lo_bytes(r[0][0], r[1][0], r[2][0], r[3][0]);
            w1[g] = pack_lo_bytes(r[0][1], r[1][1], r[2][1], r[3][1]);
            w2[g] = pack_lo_bytes(r[0][2], r[1][2], r[2][2], r[3][2]);
        }
        store_bytes<Q>(out + t * a.plane, w0);
        store_bytes<Q>(out + a.group + t * a.plane, w1);
        store_bytes<Q>(out + 2 * a.group + t * a.plane, w2);
    };
    typedef const uint32_t (&words)[4];
    typedef uint32_t (&bytes)[3];
    for_moduli<F>(
        th.t0, th.t1,
        [&] {
            plane(0, [](words x, words y, bytes r) {
                r[0] = x[0];
                r[1] = y[0];
                r[2] = x[0] + y[0];
            });
        },
        [&](int t, auto exact) {
            plane(t, [&](words x, words y, bytes r) { sym_residues<F, decltype(exact)::value>(x, y, tb, t, r); });
        });
}

// bytes per thread slot: half chunks for wide complex values (their 2 x 4 words
// per element would not fit 16 elements in registers), whole chunks otherwise
constexpr int split_q(int form, bool cplx) { return form != 0 && cplx ? 8 : 16; }
template <int FORM, bool CPLX>
__device__ __forceinline__ void split_body(const SplitItem& it, uint32_t l) {
    if constexpr (CPLX) split_cplx_body<FORM, split_q(FORM, true)>(it, l);
    else split_real_body<FORM, split_q(FORM, false)>(it, l);
}
// one operand, or both of a product (scale_kernel)
template <int FORM, bool CPLX>
__global__ void __launch_bounds__(256) split_kernel(SplitItem a, SplitItem b, uint64_t* ts) {
    const Stamp st(ts);
    const bool second = blockIdx.x >= a.blocks;
    const SplitItem it = second ? b : a;
    split_body<FORM, CPLX>(it, second ? blockIdx.x - a.blocks : blockIdx.x);
    st.end();
}

// Scale and split of both operands where a block can hold all k of its rows (kp <= 256): one pass over the
// operands and one launch.  MI355X, calls, us, scale and split / this: 64^3 s = 16 22 / 17, 4096 x 4096 x 256
// s = 16 201.6 / 197.5.
template <int FORM>
__global__ void __launch_bounds__(1024) scale_split_kernel(SplitItem a, SplitItem b, uint64_t* ts) {
    const Stamp st(ts);
    const bool second = blockIdx.x >= a.blocks;
    const SplitItem it = second ? b : a;
    split_real_body<FORM, 16, true>(it, second ? blockIdx.x - a.blocks : blockIdx.x, &st);
    st.inner(1);
    st.end();
}

// grid of one split: contiguous rows: rows x slot groups (tpr threads per row); strided: 64 rows x 4 slots (32 x 8 for half chunks).
// Contiguous rows take at most one 64-k block each (tpr <= 64 / Q), so a wave fills whole
// 1 KB plane blocks (16 rows x 64 k; 8 rows for 8-byte slots) and every 128-byte line of
// a plane is written by one wave.  With a whole row per workgroup (256 slots) the two
// rows sharing a line came from different workgroups, usually on different XCDs, and
// the L2s wrote half lines: 0.79 against 0.69 ms for both operands at 8192^3 s = 16.
SplitItem split_item(const SplitArgs& a) {
    const int q = split_q(a.form, a.cplx);
    const int64_t nck = a.kp / q;
    SplitItem it{a, 0, a.s, 0, 0, 0};
    if (a.rows_pad <= 0) return it;
    if (a.kcontig) {
        int tpr = 1;
        while (tpr < 64 / q && tpr < nck) {
            tpr <<= 1;
            ++it.lg;
        }
        it.gx = static_cast<uint32_t>((a.rows_pad + (256 / tpr) - 1) / (256 / tpr));
        it.gy = static_cast<uint32_t>((nck + tpr - 1) / tpr);
    } else {
        const int slots = 64 / q;
        it.gx = static_cast<uint32_t>((a.rows_pad + 256 / slots - 1) / (256 / slots));
        it.gy = static_cast<uint32_t>((nck + slots - 1) / slots);
    }
    it.blocks = it.gx * it.gy;
    return it;
}
// Few blocks leave the chip idle while each goes through all its moduli: these are then dealt to up to four
// times as many, which read the operand again (from the caches).
void split_parts(SplitItem& it, uint32_t launch_blocks) {
    const int parts = static_cast<int>(std::min<uint32_t>((it.a.cplx ? kSplitBlocksCplx : kSplitBlocks) / std::max(launch_blocks, 1u), 4));
    if (it.blocks == 0 || parts < 2) return;
    it.tper = (it.a.s + parts - 1) / parts;
    it.blocks *= static_cast<uint32_t>((it.a.s + it.tper - 1) / it.tper);
}

// both operands of a product in one launch, or in one each where a launch cannot hold the blocks of both: operands
// of 2^26 contiguous rows and more together (m = 67108856, n = 8), each of which one can hold
template <typename Item>
void launch_pair(const Stream& st, void (*kernel)(Item, Item, uint64_t*), uint32_t threads, const Item& a, const Item& b) {
    if (b.blocks <= max_blocks(threads) - std::min(a.blocks, max_blocks(threads))) {
        launch(st, kernel, dim3(a.blocks + b.blocks), dim3(threads), a, b);
    } else {
        launch(st, kernel, dim3(a.blocks), dim3(threads), a, b);
        launch(st, kernel, dim3(b.blocks), dim3(threads), b, a);
    }
}

template <int FORM, bool CPLX>
void launch_split(const Stream& st, const SplitItem& a, const SplitItem& b) {
    launch_pair(st, split_kernel<FORM, CPLX>, 256, a, b);
}

// ---- grouped forms: block b of the launch runs block (b - start[p]) of item p
enum GroupKind { kScale = 0, kScaleFin = 1, kSplitBase = 16 };

template <bool FIN>
__global__ void __launch_bounds__(256) grouped_scale_kernel(const ScaleItem* __restrict__ items,
                                                            const uint32_t* __restrict__ start, uint32_t n) {
    const uint32_t p = owner_of(start, n, blockIdx.x);
    const uint32_t l = blockIdx.x - start[p];
    if constexpr (FIN) scale_finalize_body(items[p], l);
    else scale_body(items[p], l);
}

template <int FORM>
__global__ void __launch_bounds__(256) grouped_split_kernel(const SplitItem* __restrict__ items,
                                                            const uint32_t* __restrict__ start, uint32_t n) {
    const uint32_t p = owner_of(start, n, blockIdx.x);
    split_body<FORM, false>(items[p], blockIdx.x - start[p]);
}

}  // namespace

size_t scale_partial_elems(int64_t len, int64_t k, bool kcontig) {
    if (kcontig) return 0;
    return static_cast<size_t>(scale_kblocks(len, k)) * static_cast<size_t>(len);
}

int scale_partials(int64_t len, int64_t k, bool kcontig) {
    return kcontig || len <= 0 ? 1 : static_cast<int>(scale_kblocks(len, k));
}

bool scale_folds(int64_t len, int64_t k, bool kcontig) {
    const int n = scale_partials(len, k, kcontig);
    return n > 1 && n <= kScaleFold;
}

void scale(const Stream& st, const ScaleJob& ja, const ScaleJob& jb) {
    const ScaleItem a = scale_item(ja), b = scale_item(jb);
    if (a.blocks + b.blocks == 0) return;
    launch_pair(st, scale_kernel, 256, a, b);
    const uint32_t fa = finalize_blocks(ja, a), fb = finalize_blocks(jb, b);
    if (fa + fb) launch(st, scale_finalize_kernel, dim3(fa + fb), dim3(256), a, b, fa);
}

void split(const Stream& st, const SplitArgs& x, const SplitArgs& y) {
    SplitItem a = split_item(x), b = split_item(y);
    const uint32_t n = a.blocks + b.blocks;
    if (n == 0) return;
    split_parts(a, n);
    split_parts(b, n);
    switch (x.form * 2 + (x.cplx ? 1 : 0)) {
        case 0: launch_split<0, false>(st, a, b); break;
        case 1: launch_split<0, true>(st, a, b); break;
        case 2: launch_split<1, false>(st, a, b); break;
        case 3: launch_split<1, true>(st, a, b); break;
        case 4: launch_split<2, false>(st, a, b); break;
        case 5: launch_split<2, true>(st, a, b); break;
        default: throw std::logic_error("oz2: no split kernel for this variant");
    }
}

bool split_scales(int64_t kp, bool cplx, int form) { return !cplx && form < 2 && kp <= 256; }

void scale_split(const Stream& st, const SplitArgs& x, const SplitArgs& y) {
    SplitItem a = split_item(x), b = split_item(y);
    a.blocks = a.gx;
    b.blocks = b.gx;
    a.gy = b.gy = 1;
    const uint32_t n = a.blocks + b.blocks;
    if (n == 0) return;
    // a workgroup fills half a CU or more, so the moduli are dealt out until every CU has one
    const int parts = static_cast<int>(std::clamp<uint32_t>(256 / n, 1, 4));
    for (SplitItem* i : {&a, &b}) {
        i->tper = (i->a.s + parts - 1) / parts;
        i->blocks *= static_cast<uint32_t>((i->a.s + i->tper - 1) / i->tper);
    }
    const uint32_t threads = static_cast<uint32_t>(4 * x.kp);
    if (x.form == 0) launch_pair(st, scale_split_kernel<0>, threads, a, b);
    else launch_pair(st, scale_split_kernel<1>, threads, a, b);
}

void split(const Stream& st, const SplitArgs& a) {
    SplitArgs none = a;
    none.rows_pad = 0;
    split(st, a, none);
}

void prep_scale(std::vector<GroupedLaunch>& out, const std::vector<ScaleJob>& jobs) {
    std::vector<GroupedLaunch> all, fin;
    for (const ScaleJob& j : jobs) {
        const ScaleItem it = scale_item(j);
        if (it.blocks == 0) continue;
        add_item(all, kScale, it, it.blocks);
        if (const uint32_t f = finalize_blocks(j, it)) add_item(fin, kScaleFin, it, f);
    }
    for (auto* v : {&all, &fin})
        for (GroupedLaunch& g : *v) out.push_back(std::move(g));
}

void prep_split(std::vector<GroupedLaunch>& out, const std::vector<SplitArgs>& jobs) {
    std::vector<GroupedLaunch> by[3];
    for (const SplitArgs& a : jobs) {
        const SplitItem it = split_item(a);
        if (it.blocks == 0) continue;
        add_item(by[a.form], kSplitBase + a.form, it, it.blocks);
    }
    for (auto& v : by)
        for (GroupedLaunch& g : v) out.push_back(std::move(g));
}

bool launch_scale_split_grouped(hipStream_t st, const GroupedLaunch& g) {
    if (g.n == 0) return true;
    const dim3 grid(g.blocks), block(256);
    switch (g.kind) {
        case kScale:
            hipLaunchKernelGGL((grouped_scale_kernel<false>), grid, block, 0, st, static_cast<const ScaleItem*>(g.d_items),
                               g.d_start, g.n);
            return true;
        case kScaleFin:
            hipLaunchKernelGGL((grouped_scale_kernel<true>), grid, block, 0, st, static_cast<const ScaleItem*>(g.d_items),
                               g.d_start, g.n);
            return true;
        // the batch takes real products only, whose plans all have tk <= 91 (forms 0 and 1)
        case kSplitBase:
            hipLaunchKernelGGL((grouped_split_kernel<0>), grid, block, 0, st, static_cast<const SplitItem*>(g.d_items),
                               g.d_start, g.n);
            return true;
        case kSplitBase + 1:
            hipLaunchKernelGGL((grouped_split_kernel<1>), grid, block, 0, st, static_cast<const SplitItem*>(g.d_items),
                               g.d_start, g.n);
            return true;
        default: return false;
    }
}

}  // namespace k
}  // namespace oz2
