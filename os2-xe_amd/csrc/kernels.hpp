// kernels.hpp - host-side launch interface of the gfx950 kernels.
//
// Data layout in HBM (all owned by the engine's workspace):
//   planes   int8  [group][t] of op(A) and op(B)^T in 1 KB blocks of 16 rows x 64 k (PlaneMap).  The split writes
//                  zeros up to kp along k and up to a multiple of the half tile of the GEMM (tile_pad_m, tile_pad_n; 64
//                  for the fused kernel) along the rows; a plane has room for whole tiles.  A tile may read the rows
//                  behind those written, whatever they hold: they only enter sums of rows or columns that lie outside C
//                  and are not stored to it.
//   residues uint8 [chunk][group][t][j][ldr]  GEMM results reduced mod m_t, i contiguous
//   D, E     int32 exponents per row of op(A) / column of op(B)
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include <vector>

#include "grouped.hpp"
#include "plan.hpp"
#include "planner.hpp"

namespace oz2 {
namespace k {

// Source of a timed launch's stamps (stage times): kStampWords device words of its own.
inline constexpr uint32_t kStampWords = 16, kStampEnds = 8, kStampInner = 9;
struct LaunchTimer {
    virtual uint64_t* next() = 0;

protected:
    ~LaunchTimer() = default;
};

// The stages that launches are timed as.  Fused: GEMM and CRT in one launch, ScaleSplit: scale and split; their time is
// divided as the launch's first workgroup divided its own.
enum class Stage : uint8_t { Scale, Split, Gemm, Crt, Fused, ScaleSplit };
inline constexpr int kStageSums = 4;  // scale, split, GEMM, CRT

// adds the time of one launch, in ticks of the clock, from its stamps
__host__ __device__ inline void add_stage_ticks(const uint64_t* w, Stage st, double* sums) {
    uint64_t e = 0;
    for (uint32_t i = 1; i <= kStampEnds; ++i) e = e > w[i] ? e : w[i];
    const uint64_t b = w[0], second = w[kStampInner], end = w[kStampInner + 1];
    const double ticks = e > b ? static_cast<double>(e - b) : 0.0;
    if (st != Stage::Fused && st != Stage::ScaleSplit) {
        sums[static_cast<int>(st)] += ticks;
        return;
    }
    const double f = end > second && second > b ? static_cast<double>(end - second) / static_cast<double>(end - b) : 0.0;
    const int first = st == Stage::Fused ? static_cast<int>(Stage::Gemm) : static_cast<int>(Stage::Scale);
    sums[first] += ticks * (1.0 - f);
    sums[first + 1] += ticks * f;
}

// Sums of the stages over the first n of the stamps at ts, added to sums (first: stored).  A handle has the stamps of
// kStampSlots launches; a longer region is summed on the stream, a launch of 3.4 us in 256, so that no call allocates
// for its stamps or waits for the GPU.
inline constexpr uint32_t kStampSlots = 256;
struct StampStages {
    Stage s[kStampSlots];
};
void sum_stamps(hipStream_t st, const uint64_t* ts, const StampStages& stages, uint32_t n, double* sums, bool first);

// Where a launch goes: a stream and, for timed calls, the timer of its stage.  The kernel stamps the
// GPU's constant-rate clock itself (Stamp below).  Events recorded around the launches are barrier
// packets of their own, about 10 us of idle GPU between any two stages (DGEMM 64^3 s = 16: 68 us a call
// with them, 29 us with timing off; 1024^3 s = 14: 112 and 76 us), and events handed to the launch cost
// 12 us of host time each; the stamps cost nothing that shows.
struct Stream {
    hipStream_t s;
    LaunchTimer* timer = nullptr;
    Stream(hipStream_t st, LaunchTimer* t = nullptr) : s(st), timer(t) {}
};

#if defined(__HIPCC__)
// Begin of a kernel in ts[0], ends in the next kStampEnds words, one an XCD (ts null: not timed).  Workgroups start in
// order, so the first one stamps the begin.  Any can be the last to end (64 x 64 x 200000, T,T: 16 blocks of op(A)'s
// rows outlast the 782 of op(B) behind them: 208 us of scaling, 81 by the last workgroups alone), so all store the
// time at which their first wave ends into their XCD's word.  The stores of an XCD meet in its L2, and the last one
// stands, which gives the end to within the flight of a store.  That costs nothing that shows, us:
// 64^3 s = 16 14.0 / 14.0, 1024^3 s = 14 46.4 / 46.4 (atomicMax of all workgroups: 1 us more with a line an XCD, 7 to 15
// with one for all).  The clock only grows, so words left by an earlier launch do not count.
struct Stamp {
    uint64_t* ts;
    uint32_t b;
    __device__ __forceinline__ explicit Stamp(uint64_t* t) : ts(t), b(blockIdx.y * gridDim.x + blockIdx.x) {
        if (ts && b == 0 && threadIdx.x == 0) ts[0] = wall_clock64();
    }
    __device__ __forceinline__ void end() const {
        constexpr int kXccId = 20 | 3 << 11;  // hardware register 20, four bits from bit 0
        if (ts && threadIdx.x == 0) ts[1 + (__builtin_amdgcn_s_getreg(kXccId) & (kStampEnds - 1))] = wall_clock64();
    }
    // a moment inside the first workgroup (a kernel of two stages)
    __device__ __forceinline__ void inner(int i) const {
        if (ts && b == 0 && threadIdx.x == 0) ts[kStampInner + i] = wall_clock64();
    }
};

// kernels launched this way take the stamps as their last parameter
template <typename... P, typename... A>
void launch(const Stream& st, void (*kernel)(P...), dim3 grid, dim3 block, A&&... args) {
    uint64_t* ts = st.timer ? st.timer->next() : nullptr;
    hipLaunchKernelGGL(kernel, grid, block, 0, st.s, args..., ts);
}
#endif

// Layout of one operand plane: 1 KB blocks of 16 rows (a band) x 64 k, 64 bytes per row as four 16-byte
// chunks.  Byte b of chunk c holds k = block_k(c, b) of the block: chunk c takes the pair (2c, 2c+1) of each
// group of 8 consecutive k, so the four threads that fill the chunks of one row read 64 contiguous bytes of a
// k-contiguous row per load.  The GEMM's dot products do not depend on the k order
// inside a block, which both operands share.  The chunks of row r are permuted by
// XOR with (r >> 2) & 3: the GEMM's DMA copies blocks verbatim to LDS, where that
// permutation makes the MFMA operand reads free of bank conflicts.
__host__ __device__ constexpr int block_k(int c, int b) { return 8 * (b >> 1) + 2 * c + (b & 1); }
// Bytes from one group of 4 bands to the next, from band to band in it, and from block column to block column.
// A stage of a GEMM tile reads one block column of 4 to 16 bands.
//   by_band:  a band's blocks side by side (the documented layout of the kernel-level entry points).  With kp
//             a multiple of 256 the blocks of a stage lie on a few of the L2's channels.
//   by_group: the four bands of a block column side by side, 4 KB, which cover the channels evenly; a tile's
//             operand is a few runs of memory.  For 128 x 128 and 64 x 64 tiles and the fused kernel.
//   by_k:     all bands of a block column side by side.  For the tiles of 256 rows: the split's writes are
//             whole runs too, where a long k makes the groups' strides powers of two.
// MI355X, us, by_band / by_group / by_k: GEMM 1024^3 s = 14 (128 x 128) 32.0 / 25.8 / 28.9, 512 x 512 x 2048
// s = 16 22.7 / 16.8 / 15.0, 1024 x 1024 x 1152 s = 14 (256 x 256) 25.7 / 26.0 / 25.0, 8192^3 s = 16 6900 /
// 6680 / 6670, 4096^3 s = 8 498 / 479 / 476; split of 2048 x 65000 by 65000 x 2048 s = 24 1965 / 2032 / 1890,
// of 8192 x 8192 both s = 16 665 / 625 / 628.
struct PlaneMap {
    int64_t group, band, blk;
    static constexpr PlaneMap by_band(int64_t kp) { return {kp * 64, kp * 16, 1024}; }
    static constexpr PlaneMap by_group(int64_t kp) { return {kp * 64, 1024, 4096}; }
    static constexpr PlaneMap by_k(int64_t rows_pad) { return {4096, 1024, rows_pad * 64}; }
    static constexpr PlaneMap of(Tile t, bool fused, int64_t rows_pad, int64_t kp) {
        return !fused && (t == Tile::T256 || t == Tile::T256x128) ? by_k(rows_pad) : by_group(kp);
    }
};
__host__ __device__ inline int64_t chunk_offset(int64_t r, int64_t blk, int c, const PlaneMap& map) {
    return (r >> 6) * map.group + ((r >> 4) & 3) * map.band + blk * map.blk + ((r & 15) << 6) + ((c ^ static_cast<int>((r >> 2) & 3)) << 4);
}

#if defined(__HIPCC__)
// blockIdx -> work item.  Workgroups go round-robin over the 8 XCDs, each with an L2 of its own; of every
// `window` items (a multiple of 8: what the chip holds at once) each XCD takes a contiguous share, so that
// the tiles it runs together share A and B bands, of large planes and of small ones.  With each plane's tiles
// spread over all XCDs, as large planes like it, an XCD held two tiles of 8 planes at 512 x 512 and read three
// times the planes' bytes from memory; with tile counts that 8 does not divide left as they came, five times
// (1537 x 771 x 3001 s = 15).  Before -> after, us: 512 x 512 x 2048 s = 16 16.4 -> 10.5, 1024 x 1024 x 2048
// 45.2 -> 35.0, 1537 x 771 x 3001 87.4 -> 68.4 (all 128 x 128), 2048^3 135 -> 128, 8192^3 the same.
__device__ __forceinline__ uint32_t xcd_window(uint32_t b, uint32_t n, uint32_t window) {
    const uint32_t base = b / window * window, i = b - base, len = min(window, n - base);
    const uint32_t x = i & 7, q = len >> 3, r = len & 7;
    return base + x * q + min(x, r) + (i >> 3);
}
// one plane block, at src + offset (both uniform), to LDS by DMA: lane l moves bytes 16 l .. 16 l + 15
__device__ __forceinline__ void block_to_lds(const int8_t* src, int offset, int lane, char* lds) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer resources are a device type
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(src), 0, 0xFFFFFFFFu, 0x00027000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds, 16, lane * 16, offset, 0, 0);
#endif
}
#endif

// ---- scaling -----------------------------------------------------------------
// Exponents of the `len` rows of op(X) over k columns.  kcontig: row r of op(X)
// is contiguous (X[p + r*ldx]); otherwise rows are strided (X[r + p*ldx]).
// Complex data (interleaved re, im) scales by the max over both parts.
// `partial` needs scale_partial_elems(len, k) u64 entries when !kcontig.
struct ScaleJob {
    const double* X;
    int64_t ldx, len, k;
    bool kcontig, cplx;
    int tk;
    uint64_t* partial;    // [scale_partials][len] maxima (strided rows only)
    int32_t* ex;
    bool fold = false;    // where scale_folds() the exponents are left to the split (SplitArgs::part)
};
size_t scale_partial_elems(int64_t len, int64_t k, bool kcontig);
int scale_partials(int64_t len, int64_t k, bool kcontig);
bool scale_folds(int64_t len, int64_t k, bool kcontig);
void scale(const Stream& st, const ScaleJob& a, const ScaleJob& b);  // both operands of a product

// ---- split -------------------------------------------------------------------
struct SplitArgs {
    const double* X;      // op(X) rows start at row r0 (already offset)
    int64_t ldx;
    int64_t rows;         // valid rows of this block
    int64_t rows_pad;     // rows written (>= rows, multiple of 32, in scale_split of 64)
    int64_t k;            // valid k
    int64_t kp;           // padded k (multiple of 128)
    const int32_t* ex;    // exponent per row (already offset); unused with part
    const uint64_t* part; // strided rows: the scale kernel's partial maxima (already offset), or null
    int64_t part_ld;      // from one k-block's maxima to the next
    int nkb, tk;          // with part (tk: scale_split too)
    int32_t* ex_out;      // with part, and in scale_split: the exponents are written here
    int8_t* P;            // planes
    PlaneMap map;
    int64_t plane;        // bytes from plane to plane (at least rows_pad * kp)
    int64_t group;        // bytes per group of s planes (complex)
    int s;
    bool kcontig, cplx, conj;
    int form;             // limb_form(tk): two, three or four words of base 2^31
    const TabSet* tab;    // device tables of this s
};
void split(const Stream& st, const SplitArgs& a);
void split(const Stream& st, const SplitArgs& a, const SplitArgs& b);  // both operands of a product (one form)
// where split_scales(): the split of both operands (or of one: rows_pad 0) with their exponents, no scale() before;
// rows_pad a multiple of 64, tk and ex_out set
bool split_scales(int64_t kp, bool cplx, int form);
void scale_split(const Stream& st, const SplitArgs& a, const SplitArgs& b);

// ---- INT8 GEMM with residue epilogue ------------------------------------------
struct GemmArgs {
    const int8_t* A;      // planes of op(A): nplanes x (mpad x kp, blocked as map_a says)
    const int8_t* B;      // planes of op(B): nplanes x (npad x kp, blocked as map_b says)
    uint8_t* R;           // residues [nplanes][npad_c][ldr]
    PlaneMap map_a, map_b;
    int64_t plane_a, plane_b, plane_r;
    int64_t ldr;          // column stride of residues (= mpad)
    int64_t k0, klen;     // k range (multiples of 128)
    int tiles_m, tiles_n;
    int64_t rows, cols;   // of the planes: multiples of tile_pad_m and tile_pad_n
    int nplanes;          // planes of this launch (s or 3s; 1 for per-plane launches)
    int plane0;           // global index of this launch's first plane: its modulus is (plane0 + plane) mod s
    int s;
    const TabSet* tab;    // device tables of this s
    int64_t kb_extra;     // op(B) reads k range k0 + kb_extra .. (0 for Scheme II)
    int32_t* R32;         // igemm_int32: sums [nplanes][npad_c][ldr] as int32 (R unused)
};
void igemm_residue(const Stream& st, Tile tile, const GemmArgs& a);
// the same GEMM with the int32 sums stored as they are (|sums| < 2^31 is the caller's to keep):
// the digit products of Ozaki Scheme I
void igemm_int32(hipStream_t st, Tile tile, const GemmArgs& a);

// ---- CRT + alpha/beta epilogue -------------------------------------------------
struct CrtArgs {
    const uint8_t* R;     // residues of this tile
    int64_t plane_r;      // bytes per (plane) residue matrix
    int64_t chunk_r;      // bytes per k-chunk (nplanes * plane_r)
    int kch;
    int64_t ldr;
    int64_t mb, nb;       // tile extent
    const int32_t* D;     // per row (offset to tile)
    const int32_t* E;     // per column (offset to tile)
    double* C;            // offset to tile; complex: interleaved
    int64_t ldc;
    double ar, ai, br, bi;
    bool cplx;
    int s, L16;
    int up;               // Plan::up()
    const TabSet* tab;    // device tables of this s
};
void crt(const Stream& st, const CrtArgs& a);

// ---- INT8 GEMMs of all planes and the CRT of a tile in one workgroup --------------
// a real product of one k-chunk; tile 128 or 64 (square): the planes hold rows up to a multiple of 64
struct FusedArgs {
    const int8_t *A, *B;      // planes of op(A), op(B): PlaneMap::by_group
    int64_t kp, plane_a, plane_b;
    int tiles_m, tiles_n;
    int s, nl, up;            // moduli, Plan::NL, Plan::up()
    const TabSet* tab;
    const int32_t *D, *E;     // exponents per row, per column (offset to the panel)
    double* C;                // offset to the panel
    int64_t mb, nb, ldc;      // panel extent
    double ar, br;
};
void fused(const Stream& st, int tile, const FusedArgs& a);

// ---- Ozaki Scheme I (the accuracy benchmark's comparison baseline) --------------------
// L balanced base-128 digits of RNE(op(X)[r][p] 2^ex[r]) per element into one extended
// plane of rows_pad x (L kp) bytes (PlaneMap::by_k): digit i
// (most significant first) at k-slot i, or L - 1 - i with rev
struct Oz1SliceArgs {
    const double* X;
    int64_t ldx, rows, rows_pad, k, kp;
    const int32_t* ex;
    int8_t* P;
    bool kcontig, rev;
};
void oz1_slices(hipStream_t st, const Oz1SliceArgs& a, int L);
// Horner step of anti-diagonal d over the int32 chunk sums Ct[c][j][ldt] (m x n entries)
struct Oz1HornerArgs {
    const int32_t* Ct;
    int64_t ldt, chunk;   // column stride and chunk stride of Ct (elements)
    int nchunks;
    double *Th, *Tl;      // running double-double T (m x n)
    bool first, last;
    int shift;            // 7 (L - 1)
    const int32_t *D, *E;
    double* C;
    int64_t m, n, ldc;
};
void oz1_horner(hipStream_t st, const Oz1HornerArgs& a);

// ---- C = beta * C for k == 0 or alpha == 0 --------------------------------------
void scale_c(hipStream_t st, double* C, int64_t ldc, int64_t m, int64_t n, double br, double bi, bool cplx);

// ---- grouped launches over many problems (batched GEMMs) -------------------------
// prep_* append launches (one per kernel variant the jobs need) whose blocks
// run exactly the single-problem kernels' blocks; launch order = vector order.
struct GemmJob {
    Tile tile;
    GemmArgs args;
};
struct FusedJob {
    int tile;
    FusedArgs args;
};
void prep_scale(std::vector<GroupedLaunch>& out, const std::vector<ScaleJob>& jobs);
void prep_split(std::vector<GroupedLaunch>& out, const std::vector<SplitArgs>& jobs);
void prep_gemm(std::vector<GroupedLaunch>& out, const std::vector<GemmJob>& jobs);
void prep_crt(std::vector<GroupedLaunch>& out, const std::vector<CrtArgs>& jobs);
void prep_fused(std::vector<GroupedLaunch>& out, const std::vector<FusedJob>& jobs);
bool launch_scale_split_grouped(hipStream_t st, const GroupedLaunch& g);
// persistent (128 x 128 and 64 x 64 tiles at their blocks per CU, 256 x 128 at one per CU):
// min(blocks, cus x that) workgroups pull tiles through counter[0 .. kGemmCounters) (reset
// first; one per XCD range of the work); else, and always for 256 x 256 tiles, one workgroup
// per tile (counters unused)
inline constexpr int kGemmCounters = 8;
void launch_gemm_grouped(hipStream_t st, const GroupedLaunch& g, uint32_t* counter, int cus, bool persistent);
int gemm_grouped_launches(const GroupedLaunch& g, bool persistent);  // kernels launch_gemm_grouped enqueues
void launch_crt_grouped(hipStream_t st, const GroupedLaunch& g);
void launch_fused_grouped(hipStream_t st, const GroupedLaunch& g);

}  // namespace k
}  // namespace oz2
