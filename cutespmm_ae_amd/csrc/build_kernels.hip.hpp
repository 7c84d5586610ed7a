// gfx950 kernels that build the two MFMA layouts (brick tiles, quad lists) from a CSR matrix that already
// lives on the device -- the device-side counterpart of HRPB::DATASTRUCT (reference data.cu:94-335), whose
// output the host functions cute_hrpb_build + cute_hrpb_retile and cute_quad_census + cute_quad_pack
// define word for word.
//
// Both layouts are orderings of the matrix entries: the brick tiles hold the entries of a 16-row panel
// sorted by (column, row) -- active column a of the panel is column a%4 of brick (a%16)/4 of block a/16, and
// inside a brick the lane-order bitmap runs column-major -- and the quad lists hold the entries of a 4-row
// strip in the same order.  Rows are sorted and duplicate-free (checked first).
//
// A panel of up to kPanelCap entries in a window of up to kPanelSpan columns is one work-group's, and nothing is sorted: the
// window is a bitmap in LDS, the running popcount of its words (number_columns) numbers the active columns, and one word per active column
// collects which of the 16 rows hold it.  Positions, list places, header lines and records all follow from prefix sums over
// those words; lines and records are written by the 16 lanes that stand for their 16 columns, so nothing is cleared beforehand
// and no global atomic is needed.  About six LDS operations an entry; ranking it by binary searches over the panel's other rows
// takes 50 to 100 (LDS merges of the rows, measured: census 57, strip lists 52 us on the graph below, 44 and 40 on the
// finite-element matrix).
// R-MAT graph of 65 536 nodes, 1.24 million entries: strip lists 40 us, where the entry-parallel kernels
// over the whole matrix took 64; finite-element matrix of 24 000 rows, 1.44 million entries: brick tiles
// 15 (before: 37).  The census (panel_census) numbers nothing.  What bounds it is latency: a dozen dependent steps a panel, four to six work-groups a compute unit.
// Other panels (hub rows of a graph, windows too wide for the bitmap) take the entry-parallel path at the end, where an entry's
// position is a sum of binary searches over the panel's rows in global memory; both write the same words.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cutespmm.h"

namespace cute_build {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kScanItems = 8;                               // entries per thread of a scan block
constexpr uint32_t kScanBlock = kThreads * kScanItems;      // entries per scan block

// Entries of a panel that one work-group holds, eight a thread: 512 threads for up to kPanelCap; the launches over all panels
// take 256 threads and up to kPanelFirst (list kernel: kPanelList, whose LDS lets six work-groups share a compute unit instead
// of three, 60 -> 40 us on the graph above), panels between have a launch that is given their list, or, for the strip lists, a
// work-group a strip.
// Where no panel has more than kPanelShort entries, 128 threads take one.  With that and LDS for the widest window there is, not for the most that the
// matrix could have, a compute unit holds 16 panels instead of 4: bricks of a 9-point stencil of 300 x 300 points 31 -> 14 us.
constexpr uint32_t kPanelCap = 4096, kPanelFirst = 2048, kPanelList = 1024, kPanelShort = 512;
constexpr uint32_t kPanelSpan = 1u << 17;                   // columns of its window: a bitmap of 16 KB and 2 KB of running counts

enum : uint32_t { kErrRange = 1, kErrUnsorted = 2, kAnyError = kErrRange | kErrUnsorted };
constexpr uint32_t kLongStrip = 16;                         // << strip, beside the errors: the strip has more than kPanelList entries

// What the planner wants to know about a panel; one 48-byte record each, written to host memory.
struct PanelCensus {
    uint32_t nnz, maxRow;      // entries, longest row
    uint32_t cols, span;       // distinct (active) columns, last column - first column + 1
    uint32_t pairs[4];         // distinct columns of each 4-row strip
    uint32_t stored;           // entries that are not zero
    uint32_t error;            // kErrRange | kErrUnsorted, with either of which the other fields mean nothing; kLongStrip
    uint32_t first, end;       // first column, last column + 1; of a panel without entries ~0 and 0
};
static_assert(sizeof(PanelCensus) == 48, "written as twelve words");

// The panels beyond kPanelCap or kPanelSpan, in ascending order.
struct LargePanels {
    const uint32_t *panel;     // [count]
    const uint32_t *prefix;    // [count + 1] running number of entries
    uint32_t count, total;
};

__device__ __forceinline__ uint64_t global_id() { return uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; }

// Inclusive scan over the 64 lanes of a wavefront by data-parallel-primitive moves: shifts by 1, 2, 4, 8 inside the rows of 16
// lanes, then the last lane of row 0 (2) to row 1 (3) and of lane 31 to rows 2 and 3.  No LDS round trip a step, which a
// shuffle is: 29.9 -> 25.2 us for the list kernel, 32.0 -> 27.8 for the census of the graph above.  op(IDENTITY, x) = x.
template <uint32_t IDENTITY, class Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t x, Op op)
{
#define CUTE_DPP(ctrl, rows) x = op(x, uint32_t(__builtin_amdgcn_update_dpp(int(IDENTITY), int(x), ctrl, rows, 0xf, false)))
    CUTE_DPP(0x111, 0xf);                    // row_shr:1
    CUTE_DPP(0x112, 0xf);
    CUTE_DPP(0x114, 0xf);
    CUTE_DPP(0x118, 0xf);
    CUTE_DPP(0x142, 0xa);                    // row_bcast:15
    CUTE_DPP(0x143, 0xc);                    // row_bcast:31
#undef CUTE_DPP
    return x;
}
// x of every eight lanes together: the other lane of a pair, the other pair of four lanes, the other four (mirrored).
__device__ __forceinline__ uint32_t or_of_eight(uint32_t x)
{
#define CUTE_DPP(ctrl) x |= uint32_t(__builtin_amdgcn_update_dpp(0, int(x), ctrl, 0xf, 0xf, true))
    CUTE_DPP(0xb1);                          // quad_perm:[1,0,3,2]
    CUTE_DPP(0x4e);                          // quad_perm:[2,3,0,1]
    CUTE_DPP(0x141);                         // row_half_mirror
#undef CUTE_DPP
    return x;
}
__device__ __forceinline__ uint32_t wave_add(uint32_t x) { return wave_scan<0u>(x, [](uint32_t a, uint32_t b) { return a + b; }); }

// ------------------------------------------------------------------------------------------------
// Inclusive prefix sum of uint32 values, in three steps: block sums, their prefix sum (by the same three
// steps), block-local prefix sums shifted by the sums of the blocks before.  Several arrays of one length, `pitch` apart, are
// summed by one launch (grid.y).
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void scan_block_sums(const uint32_t *__restrict__ in, uint64_t n, uint64_t pitch, uint32_t *__restrict__ sums,
                                                            uint64_t sums_pitch)
{
    in += blockIdx.y * pitch;
    sums += blockIdx.y * sums_pitch;
    __shared__ uint32_t wave_sum[kThreads / 64];
    const uint64_t base = uint64_t(blockIdx.x) * kScanBlock + uint64_t(threadIdx.x) * kScanItems;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i)
        if (base + i < n) s += in[base + i];
    s = wave_add(s);
    if ((threadIdx.x & 63) == 63) wave_sum[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w) t += wave_sum[w];
        sums[blockIdx.x] = t;
    }
}

// `sums` holds the inclusive prefix sums of the block sums (nullptr when there is one block).
__global__ __launch_bounds__(kThreads) void scan_block_apply(uint32_t *data, uint64_t n, uint64_t pitch, const uint32_t *__restrict__ sums, uint64_t sums_pitch)
{
    data += blockIdx.y * pitch;
    if (sums) sums += blockIdx.y * sums_pitch;
    __shared__ uint32_t wave_total[kThreads / 64];
    const uint64_t base = uint64_t(blockIdx.x) * kScanBlock + uint64_t(threadIdx.x) * kScanItems;
    uint32_t v[kScanItems];
    uint32_t t = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        t += base + i < n ? data[base + i] : 0u;
        v[i] = t;
    }
    const uint32_t incl = wave_add(t), lane = threadIdx.x & 63u;       // inclusive sum over the lanes of this wavefront
    if (lane == 63u) wave_total[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint32_t offset = (sums && blockIdx.x) ? sums[blockIdx.x - 1] : 0u;
    for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) offset += wave_total[w];
    offset += incl - t;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i)
        if (base + i < n) data[base + i] = offset + v[i];
}

// From pinned host memory into device memory.
__global__ __launch_bounds__(kThreads) void copy_words(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, uint64_t n)
{
    for (uint64_t i = global_id(); i < n; i += uint64_t(gridDim.x) * kThreads) dst[i] = src[i];
}

// table[i] by a vector load: the table may stand in host memory, 1.5 us away, and what waits for a scalar load waits for LDS as well.
__device__ __forceinline__ uint32_t table_word(const uint32_t *__restrict__ table, uint32_t i)
{
    asm volatile("" : "+v"(i));
    return table[i];
}

__device__ __forceinline__ uint32_t row_in_panel(const uint32_t *rp, uint32_t e)
{
    uint32_t lo = 0, hi = 15u;                               // the row r with rp[r] <= e < rp[r+1]
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (rp[mid + 1] <= e) lo = mid + 1u;
        else hi = mid;
    }
    return lo;
}

// ------------------------------------------------------------------------------------------------
// A panel in LDS.
// ------------------------------------------------------------------------------------------------
constexpr uint32_t panel_threads(uint32_t cap) { return cap == kPanelCap ? 512u : cap == kPanelShort ? 128u : 256u; }
struct Two { uint32_t x, y; };
template <uint32_t CAP> struct PanelLds {
    static constexpr uint32_t kBlock = panel_threads(CAP);
    uint32_t rp[17];                         // row starts, from the panel's first entry
    uint32_t lo, hi;                         // first and last column
    Two waveSum[kBlock / 64];
    uint32_t col[CAP];                       // active columns
    uint32_t rows[CAP];                      // and the rows that hold them: bits 0..15 any entry, bits 16..31 one that is not zero
};

// The entries t, t + (threads), .. of a panel in one thread's registers.
template <uint32_t CAP> struct PanelEntries {
    static constexpr uint32_t kEach = CAP / panel_threads(CAP);
    uint32_t active[kEach];                  // index of the entry's column among the panel's active columns
    uint32_t row[kEach];
    float val[kEach];
};

// Dynamic LDS of the panel kernels: the window's bitmap and the running counts of its words, later reused.
constexpr __host__ __device__ uint32_t panel_window_words(uint32_t max_span) { return (max_span + 31u) / 32u; }
// Of number_columns: words of the bitmap, and where word w of it stands.  Fours of words change places among four of them, so that
// threads that read runs of two or four of them ask for different banks.
constexpr __host__ __device__ uint32_t window_room(uint32_t max_span) { return (panel_window_words(max_span) + 15u) & ~15u; }
constexpr __host__ __device__ uint32_t bank_word(uint32_t w) { return w ^ ((w >> 4) & 12u); }

// Sum over the threads before this one, and over the whole work-group in `total`, of two words at once.
template <uint32_t WAVES> __device__ __forceinline__ Two block_exclusive_over(Two (&waveSum)[WAVES], Two own, Two &total)
{
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const Two incl = {wave_add(own.x), wave_add(own.y)};
    if (lane == 63u) waveSum[wave] = incl;
    __syncthreads();
    Two before = {incl.x - own.x, incl.y - own.y};
    total = {0u, 0u};
#pragma unroll 8
    for (uint32_t w = 0; w < WAVES; ++w) {
        const Two v = waveSum[w];
        if (w < wave) { before.x += v.x; before.y += v.y; }
        total.x += v.x;
        total.y += v.y;
    }
    __syncthreads();
    return before;
}
template <uint32_t CAP> __device__ __forceinline__ Two block_exclusive(PanelLds<CAP> &l, Two own, Two &total) { return block_exclusive_over(l.waveSum, own, total); }
template <uint32_t CAP> __device__ __forceinline__ uint32_t block_exclusive(PanelLds<CAP> &l, uint32_t own, uint32_t &total)
{
    Two sum;
    const uint32_t before = block_exclusive(l, Two{own, 0u}, sum).x;
    total = sum.x;
    return before;
}

// Row starts into LDS; returns the number of entries, or ~0u when the pointers do not ascend within [0, nnz].
// (every panel checks its own 17, so together they check all of them before anything is indexed through them)
template <uint32_t CAP> __device__ __forceinline__ uint32_t panel_rows(PanelLds<CAP> &l, const uint32_t *__restrict__ rowPtr, uint32_t p, uint32_t P, uint32_t nnz,
                                               uint32_t &start)
{
    const uint32_t t = threadIdx.x;
    int bad = 0;
    const uint32_t s = rowPtr[uint64_t(p) * 16u];
    if (t < 17u) {
        const uint32_t v = rowPtr[uint64_t(p) * 16u + t];
        l.rp[t] = v - s;
        if (t < 16u) bad = v > rowPtr[uint64_t(p) * 16u + t + 1u];
        else bad = v > nnz || (p == P - 1u && v != nnz);
        if (t == 0u && p == 0u && v != 0u) bad = 1;
    }
    if (t == 0u) { l.lo = ~0u; l.hi = 0u; }
    bad = __syncthreads_or(bad);
    start = s;
    return bad ? ~0u : l.rp[16];
}

// The same for one strip: the other rows are empty.
template <uint32_t CAP> __device__ __forceinline__ uint32_t strip_rows(PanelLds<CAP> &l, const uint32_t *__restrict__ rowPtr, uint32_t p, uint32_t strip, uint32_t &start)
{
    const uint32_t t = threadIdx.x, s = rowPtr[uint64_t(p) * 16u + 4u * strip];
    if (t < 17u) l.rp[t] = rowPtr[uint64_t(p) * 16u + min(max(t, 4u * strip), 4u * strip + 4u)] - s;
    if (t == 0u) { l.lo = ~0u; l.hi = 0u; }
    __syncthreads();
    start = s;
    return l.rp[16];
}

// How many of the entries [begin, end) are not zero; every thread of the work-group has the answer.
template <uint32_t CAP> __device__ __forceinline__ uint32_t values_in(PanelLds<CAP> &l, const float *__restrict__ vals, uint32_t begin, uint32_t end)
{
    uint32_t own = 0, total;
#pragma unroll 8
    for (uint32_t i = begin + threadIdx.x; i < end; i += PanelLds<CAP>::kBlock) own += vals[i] != 0.0f ? 1u : 0u;
    block_exclusive(l, own, total);
    return total;
}

template <uint32_t CAP> __device__ __forceinline__ bool panel_fits(const PanelLds<CAP> &l, uint32_t max_span) { return l.hi - l.lo < max_span; }

// Loads the entries of a panel of up to CAP of them (the census has checked them), finds its column window and clears the LDS that
// numbers it while the loads are on their way.
template <uint32_t CAP>
__device__ __forceinline__ void load_panel(PanelLds<CAP> &l, PanelEntries<CAP> &e, uint32_t *window, const uint32_t *__restrict__ cols,
                                           const float *__restrict__ vals, uint32_t start, uint32_t n, uint32_t max_span)
{
    const uint32_t t = threadIdx.x;
    uint32_t lo = ~0u, hi = 0u;
#pragma unroll
    for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
        if (k * PanelLds<CAP>::kBlock >= n) break;
        const uint32_t i = k * PanelLds<CAP>::kBlock + t;
        if (i >= n) continue;
        e.active[k] = cols[uint64_t(start) + i];             // its column until number_columns
        e.val[k] = vals[uint64_t(start) + i];
    }
    for (uint32_t w = t; w < window_room(max_span) / 4u; w += PanelLds<CAP>::kBlock) reinterpret_cast<uint4 *>(window)[w] = make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t i = t; i < n; i += PanelLds<CAP>::kBlock) l.rows[i] = 0u;
#pragma unroll
    for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
        if (k * PanelLds<CAP>::kBlock >= n) break;
        const uint32_t i = k * PanelLds<CAP>::kBlock + t;
        if (i >= n) continue;
        e.row[k] = row_in_panel(l.rp, i);
        const uint32_t c = e.active[k];
        lo = min(lo, c);
        hi = max(hi, c);
    }
    lo = wave_scan<~0u>(lo, [](uint32_t a, uint32_t b) { return min(a, b); });
    hi = wave_scan<0u>(hi, [](uint32_t a, uint32_t b) { return max(a, b); });
    if ((t & 63u) == 63u) { atomicMin(&l.lo, lo); atomicMax(&l.hi, hi); }
    __syncthreads();
}

// Numbers the active columns and fills l.col and l.rows; returns how many there are.  A thread counts a run of the bitmap's words, four at a
// time, which stay in its registers until their counts are known; there is a count for every four words, and an entry reads these four as well.
// (A word at a time, each read twice and with a count of its own, sixteen words a thread and so sixteen lanes to a bank: lists of an R-MAT graph of
// 131 072 nodes and 6 edges a node 91.5 us, with the words spread over the banks 82.5, this way 59.3.)
template <uint32_t CAP>
__device__ __forceinline__ uint32_t number_columns(PanelLds<CAP> &l, PanelEntries<CAP> &e, uint32_t *window, uint32_t n)
{
    constexpr uint32_t kBlock = PanelLds<CAP>::kBlock, kMost = (kPanelSpan / 128u + kBlock - 1u) / kBlock;
    const uint32_t t = threadIdx.x, lo = l.lo, words = window_room(l.hi - lo + 1u), fours = words / 4u;
    const uint4 *four = reinterpret_cast<const uint4 *>(window);
    uint16_t *count = reinterpret_cast<uint16_t *>(window + words);
#pragma unroll
    for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
        if (k * kBlock >= n) break;
        if (k * kBlock + t < n) atomicOr(&window[bank_word((e.active[k] - lo) >> 5)], 1u << ((e.active[k] - lo) & 31u));
    }
    __syncthreads();
    const uint32_t per = (fours + kBlock - 1u) / kBlock, f0 = t * per;
    auto bits_of = [](const uint4 &v) { return uint32_t(__popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w)); };
    uint32_t own = 0, of[kMost];
#pragma unroll
    for (uint32_t j = 0; j < kMost; ++j) {
        if (j >= per) break;
        of[j] = f0 + j < fours ? bits_of(four[bank_word(4u * (f0 + j)) / 4u]) : 0u;
        own += of[j];
    }
    uint32_t total;
    uint32_t run = block_exclusive(l, own, total);
#pragma unroll
    for (uint32_t j = 0; j < kMost; ++j) {
        if (j >= per) break;
        if (f0 + j < fours) count[f0 + j] = uint16_t(run);
        run += of[j];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
        if (k * kBlock >= n) break;
        if (k * kBlock + t >= n) continue;
        const uint32_t c = e.active[k], at = c - lo, below = (1u << (at & 31u)) - 1u, w = (at >> 5) & 3u;
        const uint4 v = four[bank_word(at >> 7 << 2) / 4u];
        const uint32_t a = count[at >> 7] + uint32_t(__popc(v.x & (w > 0u ? ~0u : below)) + __popc(v.y & (w > 1u ? ~0u : w == 1u ? below : 0u)) +
                                                     __popc(v.z & (w > 2u ? ~0u : w == 2u ? below : 0u)) + __popc(v.w & (w == 3u ? below : 0u)));
        e.active[k] = a;
        l.col[a] = c;
        atomicOr(&l.rows[a], (1u << e.row[k]) | (e.val[k] != 0.0f ? 1u << (16u + e.row[k]) : 0u));
    }
    __syncthreads();
    return total;
}

// Does strip s hold the column?  Strips 0 and 1 in the halves of x, 2 and 3 in those of y; half() takes one out again.
__device__ __forceinline__ Two strips_of(uint32_t rows)
{
    return {(rows & 0xfu ? 1u : 0u) | (rows & 0xf0u ? 0x10000u : 0u), (rows & 0xf00u ? 1u : 0u) | (rows & 0xf000u ? 0x10000u : 0u)};
}
__device__ __forceinline__ uint32_t half(const Two &v, uint32_t s) { return ((s & 2u ? v.y : v.x) >> (16u * (s & 1u))) & 0xffffu; }

// The panel kernels take every panel of up to CAP entries (list_of = nullptr), or the panels of a list (with CAP = kPanelCap; a
// second launch over all panels would spend 15 us on work-groups that only leave).
// A launch has at most 2^32 - 1 threads along a dimension of its grid, so all panels are kPanelRow to a row of the grid.
constexpr uint32_t kPanelRow = 1u << 22;

// Counts every panel for the planner and checks its rows.  A strip's pairs are the entries that find their column's bit clear in the
// strip's bitmap of the panel's window, the panel's active columns those that find it clear in the panel's: nothing is numbered and no bitmap
// is read through.  The bitmaps of four strips at a time where the window leaves room for them, else of two strips or of one.
// Panels of more entries than the registers hold, up to kBigEntries, are walked strip after strip.
// A chain of memory and LDS round trips a panel bounds this -- row starts, entries, window, bits -- so what counts is how many work-groups a compute unit
// holds, hence the choice of census_words.  Numbering the columns in the
// census as the builders below do took twice the steps and a second launch, with a wait for the first, for panels of more than 2 048 entries.
// us, then (both launches) / now: R-MAT graph of 65 536 nodes 68 / 36.5; finite-element matrix of 24 000 rows 22.7 / 12.5; 9-point stencil of
// 128 x 128 points 7.3 / 6.2; 65 536 rows of 32 in a band of 500, format to product, 156 / 147; 131 072 rows of 8 at random columns 280 / 219.
// COPY: the arrays are the caller's and are copied to `to` as well.  With a launch of its own for that, format to product took, us: stencil of
// 128 x 128 points, N = 32 78.6 (75.6 now), 65 536 rows of 32 in a band 147 (138 now), 50 000 rows of 16 at random columns 178 (173 now).
// Dynamic LDS: lds_words, two bitmaps of max_span columns at least.
constexpr uint32_t kBigEntries = 49152;
constexpr uint32_t kCensusEach = 8;                          // entries a thread has on their way
// Three bitmaps up to 65 536 columns (24 KB a work-group), then two (32 KB).  Four of 65 536 columns and their sums by reading them through took
// 50 000 rows of 16 at random columns 22.3 us (16.0 now), 65 536 rows in a band of 500 26.9 (17.8 now), R-MAT graph of 131 072 nodes and 4
// edges a node 109 (68 now).
constexpr uint32_t census_words(uint32_t max_span) { return panel_window_words(max_span) * (max_span <= 65536u ? 3u : 2u); }

// Of panel_census_waves: a hash table of kWaveEntries entries for each wavefront where five bitmaps of the widest window need more.
constexpr uint32_t kWaveEntries = 512, kWaveMean = 512, kWaveFront = 1024;      // up to kWaveFront panels: one in front each
constexpr uint32_t wave_census_words(uint32_t max_span)
{
    const uint32_t maps = 5u * panel_window_words(max_span), table = 2u * kWaveEntries, all = census_words(max_span);
    const uint32_t four = 4u * (maps < table ? maps : table);
    return all > four ? (all + 3u) / 4u * 4u : four;
}

struct CsrCopy {
    uint32_t *rowPtr, *cols;
    float *vals;
};

// Panel p by a whole work-group; `res` and `lo_hi` are shared.  With COPY the work-group also copies the panel's row pointers and its share of
// the entries, the same for every work-group (beside the rest its own entries would take registers).
template <bool COPY>
__device__ __forceinline__ void census_by_group(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols, const float *__restrict__ vals, uint32_t p,
                                                uint32_t P, uint32_t K, uint32_t nnz, uint32_t max_span, uint32_t lds_words, uint32_t share, const CsrCopy &to,
                                                uint32_t *bits, PanelCensus &res, uint32_t (&lo_hi)[2])
{
    constexpr uint32_t kQuarter = kThreads / 4u;             // threads of a strip
    const uint32_t t = threadIdx.x;
    // the row pointers are the work-group's (scalar registers); every panel checks its own, so together they check all of them before
    // anything is indexed through them
    uint32_t rp[17];
#pragma unroll
    for (uint32_t k = 0; k < 17u; ++k) rp[k] = rowPtr[uint64_t(p) * 16u + k];
    const uint32_t start = rp[0];
    bool bad = rp[16] > nnz || (p == P - 1u && rp[16] != nnz) || (p == 0u && start != 0u);
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) bad = bad || rp[k] > rp[k + 1u];
#pragma unroll
    for (uint32_t k = 0; k < 17u; ++k) rp[k] -= start;
    // row starts of a strip, and the end of its last row
    auto at_row = [&](uint32_t s, uint32_t k) { return s == 0u ? rp[k] : s == 1u ? rp[4u + k] : s == 2u ? rp[8u + k] : rp[12u + k]; };
    const uint32_t n = bad ? 0u : rp[16];
    if (t < 12u) reinterpret_cast<uint32_t *>(&res)[t] = 0u;
    if (COPY && t < (p == P - 1u ? 17u : 16u)) to.rowPtr[uint64_t(p) * 16u + t] = rowPtr[uint64_t(p) * 16u + t];
    if (n) {
        const uint32_t *const c = cols + start;
        const float *const v = vals + start;
        uint32_t range = 0, unsorted = 0, stored = 0, pairs = 0, active = 0, lo = 0, reach = 0, words = 0, longest = 0;
        uint32_t at_once = 4;                                // strips whose bitmaps are in LDS at one time
        bool fits = false;
        struct Entries { uint32_t col[kCensusEach], before[kCensusEach]; float val[kCensusEach]; };
        // entries i0 + k * step below `end`; the thread's own is `mine` further
        auto fetch = [&](Entries &e, uint32_t i0, uint32_t mine, uint32_t step, uint32_t end) {
#pragma unroll
            for (uint32_t k = 0; k < kCensusEach; ++k) {
                if (i0 + k * step >= end) break;
                const uint32_t i = min(i0 + mine + k * step, n - 1u);
                e.col[k] = c[i];
                e.before[k] = c[i ? i - 1u : 0u];
                e.val[k] = v[i];
            }
        };
        auto window = [&] {                                  // and LDS cleared for it
            if (t < 64u) {
                uint32_t low = ~0u, high = 0u, row = 0u;
                if (t < 16u) {
                    const uint32_t b = rowPtr[uint64_t(p) * 16u + t], e = rowPtr[uint64_t(p) * 16u + t + 1u];
                    if (e > b) { low = cols[b]; high = cols[e - 1u]; row = e - b; }
                }
                low = wave_scan<~0u>(low, [](uint32_t a, uint32_t b) { return min(a, b); });
                high = wave_scan<0u>(high, [](uint32_t a, uint32_t b) { return max(a, b); });
                longest = wave_scan<0u>(row, [](uint32_t a, uint32_t b) { return max(a, b); });
                if (t == 63u) { lo_hi[0] = low; lo_hi[1] = high; }
            }
            __syncthreads();
            // (rows that are not sorted may lie outside the window: they are not marked, and the census refuses the matrix)
            lo = lo_hi[0];
            reach = lo_hi[1] - lo;
            words = reach / 32u + 1u;
            fits = lo_hi[1] >= lo && reach < max_span;
            at_once = !fits || 5u * words <= lds_words ? 4u : 3u * words <= lds_words ? 2u : 1u;
            if (fits)                                        // (the panel's bitmap first)
                for (uint32_t w = t; w < (at_once + 1u) * words; w += kThreads) bits[w] = 0u;
            __syncthreads();
        };
        // mark(word, bit) for every column
        auto take = [&](const Entries &e, uint32_t i0, uint32_t mine, uint32_t step, uint32_t s, auto mark) {
            const uint32_t r0 = at_row(s, 0), r1 = at_row(s, 1), r2 = at_row(s, 2), r3 = at_row(s, 3), end = at_row(s, 4);
#pragma unroll
            for (uint32_t k = 0; k < kCensusEach; ++k) {
                if (i0 + k * step >= end) break;
                const uint32_t i = i0 + mine + k * step;
                if (i >= end) continue;
                range |= e.col[k] >= K ? 1u : 0u;
                unsorted |= i != r0 && i != r1 && i != r2 && i != r3 && e.before[k] >= e.col[k] ? 1u : 0u;
                stored += e.val[k] != 0.0f ? 1u : 0u;
                const uint32_t at = e.col[k] - lo;
                if (fits && at <= reach) mark(at >> 5, 1u << (at & 31u));
            }
        };
        auto add_pairs = [&](uint32_t s) {
            pairs = wave_add(pairs);
            if ((t & 63u) == 63u) atomicAdd(&res.pairs[s], pairs);
            pairs = 0;
        };
        bool held = n <= 4u * kCensusEach * kQuarter;
#pragma unroll
        for (uint32_t s = 0; s < 4u; ++s) held = held && rp[4u * s + 4u] - rp[4u * s] <= kCensusEach * kQuarter;
        if (held) {
            // every strip has at most kCensusEach entries for each thread of its quarter of the work-group: asked for before the window is known
            const uint32_t strip = __builtin_amdgcn_readfirstlane(t / kQuarter), mine = t % kQuarter, from = at_row(strip, 0), end = at_row(strip, 4);
            Entries e;
            fetch(e, from, mine, kQuarter, end);
            window();
#pragma unroll 1
            for (uint32_t s = 0; s < 4u; s += at_once) {
                uint32_t *const marked = bits + (strip - s + 1u) * words;
                if (strip - s < at_once)
                    take(e, from, mine, kQuarter, strip, [&](uint32_t w, uint32_t bit) {
                        pairs += atomicOr(&marked[w], bit) & bit ? 0u : 1u;
                        active += atomicOr(&bits[w], bit) & bit ? 0u : 1u;
                    });
                if (s + at_once == 4u || !fits) continue;
                __syncthreads();
                if (strip - s < at_once)                     // the next strips' bits begin clear
#pragma unroll
                    for (uint32_t k = 0; k < kCensusEach; ++k) {
                        if (from + k * kQuarter >= end) break;
                        if (e.col[k] - lo <= reach) marked[(e.col[k] - lo) >> 5] = 0u;
                    }
                __syncthreads();
            }
            add_pairs(strip);
        } else {
            window();
            if (t < 4u && at_row(t, 4) - at_row(t, 0) > kPanelList) atomicOr(&res.error, kLongStrip << t);
            if (n <= kBigEntries) {
                // (so many entries that their strip's bitmap is soon read through)
#pragma unroll 1
                for (uint32_t s = 0; s < 4u; ++s) {
#pragma unroll 1
                    for (uint32_t i0 = at_row(s, 0); i0 < at_row(s, 4); i0 += kCensusEach * kThreads) {
                        Entries e;
                        fetch(e, i0, t, kThreads, at_row(s, 4));
                        take(e, i0, t, kThreads, s, [&](uint32_t w, uint32_t bit) { atomicOr(&bits[words + w], bit); });
                    }
                    __syncthreads();
                    if (fits)
                        for (uint32_t w = t; w < words; w += kThreads) {          // (a thread's words are its own from strip to strip)
                            const uint32_t b = bits[words + w], all = bits[w] | b;
                            pairs += uint32_t(__popc(b));
                            if (s == 3u) active += uint32_t(__popc(all));
                            bits[w] = all;
                            bits[words + w] = 0u;
                        }
                    add_pairs(s);
                    __syncthreads();
                }
            }
        }
        if (range | unsorted) atomicOr(&res.error, (range ? uint32_t(kErrRange) : 0u) | (unsorted ? uint32_t(kErrUnsorted) : 0u));
        active = wave_add(active);
        stored = wave_add(stored);
        if ((t & 63u) == 63u) {
            atomicAdd(&res.cols, active);
            atomicAdd(&res.stored, stored);
        }
        if (t == 63u) {                                      // (its wavefront's `longest` is in its last lane)
            res.nnz = n;
            res.maxRow = longest;
            res.first = lo;
            res.span = reach + 1u;
            res.end = lo + reach + 1u;
        }
    } else if (t == 0u) {
        res.first = ~0u;
        res.error = bad ? uint32_t(kErrRange) : 0u;
    }
    if (COPY) {
        const uint64_t upto = min(uint64_t(nnz), (p + uint64_t(1)) * share);
#pragma unroll 4
        for (uint64_t i = p * uint64_t(share) + t; i < upto; i += kThreads) { to.cols[i] = cols[i]; to.vals[i] = vals[i]; }
    }
    __syncthreads();
}

template <bool COPY>
__global__ __launch_bounds__(kThreads, 7) void panel_census(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                         const float *__restrict__ vals, uint32_t P, uint32_t K, uint32_t nnz, uint32_t max_span,
                                                         uint32_t lds_words, uint32_t share, CsrCopy to, PanelCensus *__restrict__ out)
{
    extern __shared__ uint32_t bits[];
    __shared__ PanelCensus res;
    __shared__ uint32_t lo_hi[2];
    const uint32_t p = blockIdx.y * gridDim.x + blockIdx.x, t = threadIdx.x;
    if (p >= P) return;
    census_by_group<COPY>(rowPtr, cols, vals, p, P, K, nnz, max_span, lds_words, share, to, bits, res, lo_hi);
    if (t < 12u) reinterpret_cast<uint32_t *>(out + p)[t] = reinterpret_cast<const uint32_t *>(&res)[t];
}

// The same where panels are short (up to kWaveMean entries on average): a wavefront a panel and no barrier.  A panel of up to kWaveEntries entries
// stays in the wavefront's registers; columns are told apart by five bitmaps of its window or, where these do not fit the wavefront's share of the
// LDS, in a hash table of twice the entries (column from the window's start, plus one, and a bit a strip).  The first `front` work-groups take
// the longer panels, one after the other, and mostly find none: of one panel each, or of the same fours of panels, which come from four quarters of
// the matrix, `skew` panels apart, because a graph's long panels stand together at its beginning and at the quarters.  Those are copied by the
// work-group that has them among its wavefronts' panels, not by the one that counts them.
// A work-group a panel takes as long for these as for others, its chain of round trips: us, that way / this way, 131 072 rows of 12 at random columns
// 54.4 / 24.6; 9-point stencils of 300 x 300 points 23.2 / 16.2, 128 x 128 6.8 / 5.5; 65 536 rows of 32 in a band 18.7 / 17.5; R-MAT graph of 65 536
// nodes, bound by its longest panel, 39.1 / 40.3.  (Longer panels after the wavefronts' own: graph 49.  Up to 1 024 entries a wavefront: 16.1 for the
// stencil of 300 x 300.)
template <bool COPY>
__global__ __launch_bounds__(kThreads, 6) void panel_census_waves(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                               const float *__restrict__ vals, uint32_t P, uint32_t K, uint32_t nnz, uint32_t max_span,
                                                               uint32_t lds_words, uint32_t quarter, uint32_t skew, uint32_t front, CsrCopy to, PanelCensus *__restrict__ out)
{
    extern __shared__ uint32_t bits[];
    __shared__ PanelCensus res;
    __shared__ uint32_t lo_hi[2], starts_of[4][kWaveEntries / 32u];
    const uint32_t id = blockIdx.y * gridDim.x + blockIdx.x, t = threadIdx.x, lane = t & 63u, wave = __builtin_amdgcn_readfirstlane(t / 64u);
    if (id >= front + quarter) return;
    const uint32_t group = id < front ? id : id - front;
    auto panel_of = [&](uint32_t w) {
        const uint32_t x = group + w * skew;
        return w * quarter + (x >= quarter ? x - quarter : x);
    };
    if (id < front) {
        const bool one = front != quarter;
        uint32_t entries[4];
#pragma unroll
        for (uint32_t w = 0; w < 4u; ++w) {
            const uint32_t q = one ? (w ? P : id) : panel_of(w), in = min(q, P - 1u);
            entries[w] = q < P ? rowPtr[uint64_t(in) * 16u + 16u] - rowPtr[uint64_t(in) * 16u] : 0u;
        }
#pragma unroll 1
        for (uint32_t w = 0; w < 4u; ++w) {
            if ((w == 0u ? entries[0] : w == 1u ? entries[1] : w == 2u ? entries[2] : entries[3]) <= kWaveEntries) continue;
            const uint32_t q = one ? id : panel_of(w);
            census_by_group<false>(rowPtr, cols, vals, q, P, K, nnz, max_span, lds_words, 0u, to, bits, res, lo_hi);
            if (t < 12u) reinterpret_cast<uint32_t *>(out + q)[t] = reinterpret_cast<const uint32_t *>(&res)[t];
            __syncthreads();
        }
        return;
    }
    const uint32_t p = panel_of(wave);
    if (p < P) {
        const uint32_t own = rowPtr[uint64_t(p) * 16u + min(lane, 16u)];
        const uint32_t next = uint32_t(__builtin_amdgcn_update_dpp(0, int(own), 0x130, 0xf, 0xf, true));      // wave_shl:1, the next lane's
        auto row_start = [&](int r) { return uint32_t(__builtin_amdgcn_readlane(int(own), r)); };
        const uint32_t start = row_start(0), stop = row_start(16);
        if (COPY && lane < (p == P - 1u ? 17u : 16u)) to.rowPtr[uint64_t(p) * 16u + lane] = own;
        const bool bad = stop > nnz || (p == P - 1u && stop != nnz) || (p == 0u && start != 0u) || __ballot(lane < 16u && own > next) != 0u;
        const uint32_t n = bad ? 0u : stop - start;
        if (stop - start <= kWaveEntries) {
            uint32_t word = lane == 10u ? ~0u : lane == 9u && bad ? uint32_t(kErrRange) : 0u;       // the record, a word a lane
            if (n) {
                constexpr uint32_t kEach = kWaveEntries / 64u;
                const uint32_t *const c = cols + start;
                const float *const v = vals + start;
                uint32_t col[kEach];
                float val[kEach];
#pragma unroll
                for (uint32_t k = 0; k < kEach; ++k) {
                    if (k * 64u >= n) break;
                    col[k] = c[min(k * 64u + lane, n - 1u)];
                    val[k] = v[min(k * 64u + lane, n - 1u)];
                }
                const uint32_t region = lds_words / 4u;
                uint32_t *const mine = bits + wave * region, *const starts = starts_of[wave];
                if (lane < kWaveEntries / 32u) starts[lane] = 0u;
                __builtin_amdgcn_wave_barrier();
                const uint32_t at_row = own - start;
                if (lane < 16u && at_row < n) atomicOr(&starts[at_row >> 5], 1u << (at_row & 31u));
                uint32_t lo = ~0u, hi = 0u;
#pragma unroll
                for (uint32_t k = 0; k < kEach; ++k) {
                    if (k * 64u >= n) break;
                    lo = min(lo, col[k]);
                    hi = max(hi, col[k]);
                    if (COPY && k * 64u + lane < n) { to.cols[uint64_t(start) + k * 64u + lane] = col[k]; to.vals[uint64_t(start) + k * 64u + lane] = val[k]; }
                }
                lo = uint32_t(__builtin_amdgcn_readlane(int(wave_scan<~0u>(lo, [](uint32_t a, uint32_t b) { return min(a, b); })), 63));
                hi = uint32_t(__builtin_amdgcn_readlane(int(wave_scan<0u>(hi, [](uint32_t a, uint32_t b) { return max(a, b); })), 63));
                const uint32_t longest = uint32_t(__builtin_amdgcn_readlane(
                    int(wave_scan<0u>(lane < 16u ? next - own : 0u, [](uint32_t a, uint32_t b) { return max(a, b); })), 63));
                const uint32_t reach = hi - lo, words = reach / 32u + 1u;
                const bool fits = reach < max_span, maps = fits && 5u * words <= region;
                const uint32_t log = 32u - uint32_t(__builtin_clz(max(2u * n - 1u, 1u)));          // of the table
                const uint32_t clear = maps ? 5u * words : fits ? 1u << log : 0u;
                for (uint32_t w = lane; w < clear; w += 64u) mine[w] = 0u;
                __builtin_amdgcn_wave_barrier();
                const uint32_t s1 = row_start(4) - start, s2 = row_start(8) - start, s3 = row_start(12) - start;
                uint32_t range = 0, unsorted = 0, stored = 0, active = 0, pairs[4] = {}, front = 0;
#pragma unroll
                for (uint32_t k = 0; k < kEach; ++k) {
                    if (k * 64u >= n) break;
                    const uint32_t i = k * 64u + lane, at = col[k] - lo;
                    const uint32_t before = uint32_t(__builtin_amdgcn_update_dpp(int(front), int(col[k]), 0x138, 0xf, 0xf, false));       // wave_shr:1
                    front = uint32_t(__builtin_amdgcn_readlane(int(col[k]), 63));
                    const uint32_t strip = (i >= s1 ? 1u : 0u) + (i >= s2 ? 1u : 0u) + (i >= s3 ? 1u : 0u);
                    bool first = false, pair = false;
                    if (i < n) {
                        range |= col[k] >= K ? 1u : 0u;
                        unsorted |= before >= col[k] && !(starts[i >> 5] >> (i & 31u) & 1u) ? 1u : 0u;
                        if (maps) {
                            const uint32_t bit = 1u << (at & 31u);
                            first = !(atomicOr(&mine[at >> 5], bit) & bit);
                            pair = !(atomicOr(&mine[(1u + strip) * words + (at >> 5)], bit) & bit);
                        } else if (fits) {
                            uint32_t slot = (at * 0x9e3779b1u) >> (32u - log), held;
                            while ((held = atomicCAS(&mine[slot], 0u, at + 1u)) != 0u && (held & 0xfffffu) != at + 1u) slot = (slot + 1u) & ((1u << log) - 1u);
                            first = held == 0u;
                            pair = !(atomicOr(&mine[slot], 0x100000u << strip) & (0x100000u << strip));
                        }
                    }
                    stored += uint32_t(__popcll(__ballot(i < n && val[k] != 0.0f)));
                    active += uint32_t(__popcll(__ballot(first)));
#pragma unroll
                    for (uint32_t s = 0; s < 4u; ++s) pairs[s] += uint32_t(__popcll(__ballot(pair && strip == s)));
                }
                const uint32_t error = (__ballot(range) ? uint32_t(kErrRange) : 0u) | (__ballot(unsorted) ? uint32_t(kErrUnsorted) : 0u);
                const uint32_t record[12] = {n, longest, active, reach + 1u, pairs[0], pairs[1], pairs[2], pairs[3], stored, error, lo, lo + reach + 1u};
#pragma unroll
                for (uint32_t k = 0; k < 12u; ++k) word = lane == k ? record[k] : word;
            }
            if (lane < 12u) reinterpret_cast<uint32_t *>(out + p)[lane] = word;
        }
    }
    if (!COPY) return;
#pragma unroll 1
    for (uint32_t w = 0; w < 4u; ++w) {                      // the longer panels are copied here, beside their census
        const uint32_t q = panel_of(w);
        if (q >= P) continue;
        const uint32_t begin = min(rowPtr[uint64_t(q) * 16u], nnz), end = min(rowPtr[uint64_t(q) * 16u + 16u], nnz);
        if (end < begin || end - begin <= kWaveEntries) continue;
        for (uint64_t i0 = begin; i0 < end; i0 += 8u * kThreads) {
            uint32_t x[8];
            float y[8];
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) { x[k] = cols[min(i0 + k * kThreads + t, end - uint64_t(1))]; y[k] = vals[min(i0 + k * kThreads + t, end - uint64_t(1))]; }
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k)
                if (i0 + k * kThreads + t < end) { to.cols[i0 + k * kThreads + t] = x[k]; to.vals[i0 + k * kThreads + t] = y[k]; }
        }
    }
}

// Brick tiles of the panels that fit: hdr lines and values (cute_hrpb_retile defines both).  brp: first block of every
// panel.  Block 0 also writes the wavefront of zeros behind the values.
template <uint32_t CAP>
__global__ __launch_bounds__(panel_threads(CAP)) void panel_bricks(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                         const float *__restrict__ vals, uint32_t P, uint32_t nnz, uint32_t max_span,
                                                         const uint32_t *__restrict__ list_of, const uint32_t *__restrict__ brp, uint32_t *__restrict__ hdr, float *__restrict__ tile_vals)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t window[];
    __shared__ PanelLds<CAP> l;
    const uint32_t p = list_of ? list_of[blockIdx.x] : blockIdx.y * gridDim.x + blockIdx.x, t = threadIdx.x;
    if (p >= P) return;
    if (!list_of && p == 0u && t < 64u) tile_vals[uint64_t(nnz) + t] = 0.0f;
    uint32_t start;
    const uint32_t n = panel_rows(l, rowPtr, p, P, nnz, start);
    if (n == 0u || n > CAP) return;
    PanelEntries<CAP> e;
    load_panel(l, e, window, cols, vals, start, n, max_span);
    if (!panel_fits(l, max_span)) return;
    const uint32_t block_word = table_word(brp, p);
    const uint32_t active = number_columns(l, e, window, n);
    uint16_t *first = reinterpret_cast<uint16_t *>(window);   // position of every active column's first entry, and n behind the last
    {
        uint32_t own = 0;
#pragma unroll
        for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
            const uint32_t a = t * PanelEntries<CAP>::kEach + k;
            own += a < active ? uint32_t(__popc(l.rows[a] & 0xffffu)) : 0u;
        }
        uint32_t total;
        uint32_t run = block_exclusive(l, own, total);
#pragma unroll
        for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
            const uint32_t a = t * PanelEntries<CAP>::kEach + k;
            if (a <= active) first[a] = uint16_t(run);
            run += a < active ? uint32_t(__popc(l.rows[a] & 0xffffu)) : 0u;
        }
        if (t == 0u && active == CAP) first[CAP] = uint16_t(n);
    }
    __syncthreads();
    const uint32_t slots = ((active + 15u) / 16u) * 16u, block0 = __builtin_amdgcn_readfirstlane(block_word);
    for (uint32_t a = t; a < slots; a += PanelLds<CAP>::kBlock) {          // sixteen lanes are the sixteen columns of one block
        const uint32_t b = first[min(a, active)];
        const uint32_t mask = a < active ? l.rows[a] & 0xffffu : 0u;
        const uint32_t slot = a & 15u, j = slot >> 2, k = slot & 3u;
        uint32_t *h = hdr + (uint64_t(block0) + (a >> 4)) * CUTE_TILED_HDR_WORDS;
        h[k * 4u + j] = a < active ? l.col[a] : 0u;
        const uint32_t upper = __shfl_xor(mask, 1);           // bit k*16 + row of the brick's bitmap: two columns to a word
        if ((k & 1u) == 0u) h[16u + 2u * j + (k >> 1)] = mask | (upper << 16);
        if (k == 0u) h[24u + j] = start + b;                  // a brick of padding columns only points at the panel's end
        if (slot < 4u) h[28u + slot] = slot == 0u ? uint32_t(first[min((a | 15u) + 1u, active)]) - first[a & ~15u] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
        if (k * PanelLds<CAP>::kBlock >= n) break;
        if (k * PanelLds<CAP>::kBlock + t >= n) continue;
        const uint32_t a = e.active[k];
        tile_vals[uint64_t(start) + first[a] + uint32_t(__popc(l.rows[a] & ((1u << e.row[k]) - 1u)))] = e.val[k];
    }
}

// Quad lists of the panels that fit (cute_quad_pack defines them).  STRIPS: one list per strip, groups[4p + s] its first group;
// else four lockstep lists per panel, groups[p].  valBase: first stored value of every panel.  A thread is one
// (row group, column) pair; the running number of stored values over the pairs of the panel is at once the place of
// their values and, at a group's first pair, the record's index word.  Block 0 writes the zeros behind the values.
// Dynamic LDS: the window, then (in its place) the list places of every column, four 16-bit numbers each.
// The first `listed` work-groups of STRIPS take a strip each of panels of more than CAP entries (4 panel + strip, kHasZeros), which have no
// launch of their own: three launches one after the other took 27 + 25 + 18 us (big_quads, panels of up to 1 024, of up to 4 096 entries) on the
// graph above, now big_quads runs beside this one on a second stream, 36 us from first to last; format to product 346 -> 322.  Without
// STRIPS `listed` says that `list` names the panels.
constexpr uint32_t kHasZeros = 1u << 31;
template <bool STRIPS, uint32_t CAP>
__global__ __launch_bounds__(panel_threads(CAP)) void panel_quads(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                        const float *__restrict__ vals, uint32_t P, uint32_t nnz, uint32_t max_span,
                                                        const uint32_t *__restrict__ list_of, uint32_t listed,
                                                        const uint32_t *__restrict__ groups, const uint32_t *__restrict__ valBase, uint32_t stored,
                                                        uint32_t *__restrict__ recs, float *__restrict__ packed)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t window[];
    __shared__ PanelLds<CAP> l;
    __shared__ uint16_t list[CAP], place[CAP];    // pair -> active column, and -> its first value from the panel's first
    const uint32_t id = blockIdx.y * gridDim.x + blockIdx.x, t = threadIdx.x;
    const bool one_strip = STRIPS && id < listed;
    const uint32_t word = id < listed ? list_of[id] : 0u, strip = one_strip ? word & 3u : 0u;
    const uint32_t p = one_strip ? (word & ~kHasZeros) >> 2 : STRIPS ? id - listed : listed ? word : id;
    if (p >= P || (!STRIPS && listed && id >= listed)) return;
    if (p == 0u && t < 64u && (STRIPS ? !one_strip : !listed)) packed[uint64_t(stored) + t] = 0.0f;
    uint32_t start;
    const uint32_t n = one_strip ? strip_rows(l, rowPtr, p, strip, start) : panel_rows(l, rowPtr, p, P, nnz, start);
    if (n == 0u || n > CAP) return;
    PanelEntries<CAP> e;
    load_panel(l, e, window, cols, vals, start, n, max_span);
    if (!panel_fits(l, max_span)) return;
    const uint32_t group_word = table_word(groups, p * (STRIPS ? 4u : 1u) + strip), value_word = table_word(valBase, p);
    // values of the strips in front
    uint32_t front = 0;
    if (one_strip && strip) {
        const uint32_t panel = rowPtr[uint64_t(p) * 16u];
        front = word & kHasZeros ? values_in(l, vals, panel, start) : start - panel;
    }
    const uint32_t active = number_columns(l, e, window, n);
    Two *before = reinterpret_cast<Two *>(window);            // pairs in front of an active column's, in each strip's list
    Two lens;
    {
        Two own = {0u, 0u};
#pragma unroll
        for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
            const uint32_t a = t * PanelEntries<CAP>::kEach + k;
            const Two here = strips_of(a < active ? l.rows[a] : 0u);
            own.x += here.x;
            own.y += here.y;
        }
        Two run = block_exclusive(l, own, lens);
        // (a strip's pairs stand behind those of the strips in front of it)
        const uint32_t front = half(lens, 0) + half(lens, 1);
        run.x += half(lens, 0) << 16;
        run.y += front | ((front + half(lens, 2)) << 16);
#pragma unroll
        for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
            const uint32_t a = t * PanelEntries<CAP>::kEach + k;
            if (a >= active) break;
            const Two here = strips_of(l.rows[a]);
            before[a] = run;
#pragma unroll
            for (uint32_t s = 0; s < 4u; ++s)
                if (half(here, s)) list[half(run, s)] = uint16_t(a);
            run.x += here.x;
            run.y += here.y;
        }
    }
    __syncthreads();
    uint32_t len[4], list0[4], group_before[4], total = 0;    // list lengths and starts; STRIPS: groups in front of each strip
#pragma unroll
    for (uint32_t s = 0; s < 4u; ++s) {
        len[s] = half(lens, s);
        list0[s] = s ? list0[s - 1] + len[s - 1] : 0u;
        group_before[s] = total;
        total = STRIPS ? total + (len[s] + 15u) / 16u : max(total, (len[s] + 3u) / 4u);
    }
    const uint32_t slots = total * 16u, group0 = __builtin_amdgcn_readfirstlane(group_word), value0 = __builtin_amdgcn_readfirstlane(value_word + front);
    uint32_t base = 0;
    for (uint32_t x0 = 0; x0 < slots; x0 += PanelLds<CAP>::kBlock) {
        const uint32_t x = x0 + t, g = x >> 4, pair = x & 15u;
        const bool live = x < slots;
        const uint32_t s = STRIPS ? (g >= group_before[1] ? 1u : 0u) + (g >= group_before[2] ? 1u : 0u) + (g >= group_before[3] ? 1u : 0u) : pair & 3u;
        auto of_strip = [&](const uint32_t (&v)[4]) { return s == 0u ? v[0] : s == 1u ? v[1] : s == 2u ? v[2] : v[3]; };
        const uint32_t q = STRIPS ? 16u * (g - of_strip(group_before)) + pair : 4u * g + (pair >> 2);
        const uint32_t my_len = of_strip(len), my_list = of_strip(list0);
        uint32_t col = 0, mask = 0;
        if (live && my_len) {
            const uint32_t a = list[my_list + min(q, my_len - 1u)];           // padding repeats the last column of its list
            col = l.col[a];
            mask = q < my_len ? (l.rows[a] >> (16u + 4u * s)) & 15u : 0u;     // an explicit zero is an empty slot
        }
        uint32_t sum;
        const uint32_t at = base + block_exclusive(l, uint32_t(__popc(mask)), sum);
        base += sum;
        const uint32_t word = or_of_eight(mask << (4u * (pair & 7u)));       // slot 4*pair + row: eight pairs to a mask word
        if (live) {
            uint32_t *rec = recs + (uint64_t(group0) + g) * CUTE_QUAD_RECORD_WORDS;
            rec[pair] = col;
            if (pair == 0u) { rec[16] = word; rec[18] = value0 + at; }
            if (pair == 8u) { rec[17] = word; rec[19] = 0u; }
            if (q < my_len) place[my_list + q] = uint16_t(at);
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < PanelEntries<CAP>::kEach; ++k) {
        if (k * PanelLds<CAP>::kBlock >= n) break;
        if (k * PanelLds<CAP>::kBlock + t >= n || e.val[k] == 0.0f) continue;
        const uint32_t a = e.active[k], s = e.row[k] >> 2, mask = (l.rows[a] >> (16u + 4u * s)) & 15u;
        const uint32_t pr = half(before[a], s);
        packed[uint64_t(value0) + place[pr] + uint32_t(__popc(mask & ((1u << (e.row[k] & 3u)) - 1u)))] = e.val[k];
    }
}

// ------------------------------------------------------------------------------------------------
// Strips of more than kPanelList entries (the hub rows of a graph) whose panel's window the bitmap takes: a work-group of sixteen wavefronts
// walks the entries of a strip instead of holding them, for the strip lists.  LDS holds the bitmap, its counts and the
// rows of every active column, and the rest follows from prefix sums over the columns, a thread a run of them.
// The entry-parallel kernels below need sixteen binary searches an entry, two scans and a launch for each step: R-MAT graph of 65 536
// nodes, 449 000 entries in 79 such panels, lists 70 -> 34 us.
// ------------------------------------------------------------------------------------------------
constexpr uint32_t kBigThreads = 1024;        // (with kBigEntries the sums of a panel fit 16 bits)

constexpr __host__ __device__ uint32_t big_window_words(uint32_t window_words) { return window_words + (window_words + 1u) / 2u; }   // bitmap and 16-bit counts

// Running counts of the bitmap's words; returns how many columns are active.
__device__ __forceinline__ uint32_t big_counts(Two (&waveSum)[kBigThreads / 64], const uint32_t *window, uint16_t *count, uint32_t words)
{
    const uint32_t t = threadIdx.x, per = (words + kBigThreads - 1u) / kBigThreads, w0 = min(t * per, words), w1 = min(w0 + per, words);
    uint32_t own = 0;
    for (uint32_t w = w0; w < w1; ++w) own += uint32_t(__popc(window[w]));
    Two total;
    uint32_t run = block_exclusive_over(waveSum, {own, 0u}, total).x;
    for (uint32_t w = w0; w < w1; ++w) { count[w] = uint16_t(run); run += uint32_t(__popc(window[w])); }
    __syncthreads();
    return total.x;
}

__device__ __forceinline__ uint32_t big_number(const uint32_t *window, const uint16_t *count, uint32_t c)      // c: from the window's start
{
    return count[c >> 5] + uint32_t(__popc(window[c >> 5] & ((1u << (c & 31u)) - 1u)));
}

// The listed strips of more than kPanelList entries (panel_quads<true> defines the lists), a work-group each: a strip's entries are one piece of the arrays, its
// active columns are its pairs.  row_words: a byte a column, the rows that hold it and those whose entry is not zero; step_words: three
// words for every 64 columns.  (One work-group for all four strips of a panel: 81 us against 34.)
// A wavefront takes 64 columns of the list at a time: where their entries stand in each row, and where their values go, is the sum of what
// the columns before them hold and a count of bits below the lane, so the loads of a step are whole pieces of the rows and no step waits
// for another.  Graph above: 34.8 us with a thread walking a run of columns, one after the other, 26.5 this way; what is left is the first strip,
// of 15 000 entries: loads and bits 14 400 cycles, numbers 10 800, values 14 000.
__global__ __launch_bounds__(kBigThreads) void big_quads(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols, const float *__restrict__ vals,
                                                         const uint32_t *__restrict__ list, uint32_t window_words, uint32_t row_words,
                                                         const uint32_t *__restrict__ groups, const uint32_t *__restrict__ valBase,
                                                         uint32_t *__restrict__ recs, float *__restrict__ packed)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t window[];
    __shared__ Two waveSum[kBigThreads / 64];
    __shared__ uint32_t lo_hi[2], front;      // front: values stored for the strips in front of this one
    uint16_t *count = reinterpret_cast<uint16_t *>(window + window_words);
    uint32_t *rows = window + big_window_words(window_words), *steps = rows + row_words;
    const uint32_t word = list[blockIdx.x], p = (word & ~kHasZeros) >> 2, s = word & 3u, t = threadIdx.x, lane = t & 63u;
    const uint32_t group0 = groups[uint64_t(p) * 4u + s], num_groups = groups[uint64_t(p) * 4u + s + 1u] - group0;
    if (num_groups == 0u) return;
    uint32_t rp[5];                           // the strip's rows
#pragma unroll
    for (uint32_t k = 0; k < 5u; ++k) rp[k] = rowPtr[uint64_t(p) * 16u + 4u * s + k];
    const uint32_t panel = rowPtr[uint64_t(p) * 16u], start = rp[0], end = rp[4], value0 = valBase[p];
    uint32_t *const strip_recs = recs + uint64_t(group0) * CUTE_QUAD_RECORD_WORDS;
    for (uint32_t w = t; w < window_words; w += kBigThreads) window[w] = 0u;
    for (uint32_t w = t; w < row_words; w += kBigThreads) rows[w] = 0u;
    if (t == 0u) { lo_hi[0] = ~0u; lo_hi[1] = 0u; front = word & kHasZeros ? 0u : start - panel; }
    __syncthreads();
    if (t < 4u && rowPtr[uint64_t(p) * 16u + 4u * s + t + 1u] > rowPtr[uint64_t(p) * 16u + 4u * s + t]) {
        atomicMin(&lo_hi[0], cols[rowPtr[uint64_t(p) * 16u + 4u * s + t]]);
        atomicMax(&lo_hi[1], cols[rowPtr[uint64_t(p) * 16u + 4u * s + t + 1u] - 1u]);
    }
    uint32_t before = 0;
    for (uint32_t i0 = word & kHasZeros ? panel : start; i0 < start; i0 += 16u * kBigThreads) {          // (sixteen loads on their way, whatever is left)
        float v[16];
#pragma unroll
        for (uint32_t k = 0; k < 16u; ++k) {
            if (i0 + k * kBigThreads >= start) break;
            v[k] = vals[min(i0 + k * kBigThreads + t, start - 1u)];
        }
#pragma unroll
        for (uint32_t k = 0; k < 16u; ++k) {
            if (i0 + k * kBigThreads >= start) break;
            before += i0 + k * kBigThreads + t < start && v[k] != 0.0f ? 1u : 0u;
        }
    }
    __syncthreads();
    const uint32_t lo = lo_hi[0], words = (lo_hi[1] - lo) / 32u + 1u;
    // the strip's columns stay in registers until they are numbered, with a bit for every value that is not zero
    constexpr uint32_t kEach = kBigEntries / kBigThreads;
    static_assert(kEach <= 64u, "a bit an entry");
    uint32_t col[kEach];
    uint64_t not_zero = 0;
#pragma unroll
    for (uint32_t k = 0; k < kEach; ++k) {
        if (start + k * kBigThreads >= end) break;
        col[k] = cols[min(start + k * kBigThreads + t, end - 1u)];
    }
    for (uint32_t k0 = 0; start + k0 * kBigThreads < end; k0 += 16u) {
        float v[16];
#pragma unroll
        for (uint32_t k = 0; k < 16u; ++k) {
            if (start + (k0 + k) * kBigThreads >= end) break;
            v[k] = vals[min(start + (k0 + k) * kBigThreads + t, end - 1u)];
        }
#pragma unroll
        for (uint32_t k = 0; k < 16u; ++k) {
            if (start + (k0 + k) * kBigThreads >= end) break;
            not_zero |= uint64_t(v[k] != 0.0f ? 1u : 0u) << (k0 + k);
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kEach; ++k) {
        if (start + k * kBigThreads >= end) break;
        atomicOr(&window[(col[k] - lo) >> 5], 1u << ((col[k] - lo) & 31u));
    }
    __syncthreads();
    const uint32_t active = big_counts(waveSum, window, count, words);
#pragma unroll
    for (uint32_t k = 0; k < kEach; ++k) {
        if (start + k * kBigThreads >= end) break;
        const uint32_t i = start + k * kBigThreads + t;
        if (i >= end) continue;
        const uint32_t a = big_number(window, count, col[k] - lo), r = (i >= rp[1] ? 1u : 0u) + (i >= rp[2] ? 1u : 0u) + (i >= rp[3] ? 1u : 0u);
        atomicOr(&rows[a >> 2], ((1u << r) | (not_zero >> k & 1u ? 16u << r : 0u)) << (8u * (a & 3u)));
        strip_recs[(a >> 4) * CUTE_QUAD_RECORD_WORDS + (a & 15u)] = col[k];       // (every entry of the column writes it)
    }
    __syncthreads();
    const uint8_t *row_of = reinterpret_cast<const uint8_t *>(rows);
    const uint32_t num_steps = (active + 63u) / 64u;
    auto rows_at = [&](uint32_t a) -> uint32_t { return a < active ? row_of[a] : 0u; };
    // what the 64 columns of a step hold, entries of each row and values: sixteen lanes of four columns each (the bytes behind the last are clear)
    for (uint32_t i = t; i < num_steps * 16u; i += kBigThreads) {
        const uint32_t m = i < row_words ? rows[i] : 0u;
        uint32_t x = uint32_t(__popc(m & 0x01010101u)) | uint32_t(__popc(m & 0x02020202u)) << 16;
        uint32_t y = uint32_t(__popc(m & 0x04040404u)) | uint32_t(__popc(m & 0x08080808u)) << 16;
        uint32_t z = uint32_t(__popc(m & 0xf0f0f0f0u));
#define CUTE_DPP(v, ctrl) v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), ctrl, 0xf, 0xf, true))
#define CUTE_SUM(ctrl) CUTE_DPP(x, ctrl); CUTE_DPP(y, ctrl); CUTE_DPP(z, ctrl)
        CUTE_SUM(0x111);                      // row_shr:1, 2, 4, 8
        CUTE_SUM(0x112);
        CUTE_SUM(0x114);
        CUTE_SUM(0x118);
#undef CUTE_SUM
#undef CUTE_DPP
        if ((i & 15u) == 15u) { steps[3u * (i >> 4)] = x; steps[3u * (i >> 4) + 1u] = y; steps[3u * (i >> 4) + 2u] = z; }
    }
    before = wave_add(before);
    if (lane == 63u && before) atomicAdd(&front, before);
    __syncthreads();
    if (t < 64u) {                            // and in front of each
        Two row = {0u, 0u};
        uint32_t held = 0;
        for (uint32_t first = 0; first < num_steps; first += 64u) {
            uint32_t *const of = steps + 3u * (first + lane);
            const bool mine = first + lane < num_steps;
            const uint32_t x = mine ? of[0] : 0u, y = mine ? of[1] : 0u, z = mine ? of[2] : 0u, xs = wave_add(x), ys = wave_add(y), zs = wave_add(z);
            if (mine) { of[0] = row.x + xs - x; of[1] = row.y + ys - y; of[2] = held + zs - z; }
            row.x += uint32_t(__builtin_amdgcn_readlane(int(xs), 63));
            row.y += uint32_t(__builtin_amdgcn_readlane(int(ys), 63));
            held += uint32_t(__builtin_amdgcn_readlane(int(zs), 63));
        }
    }
    __syncthreads();
    const uint32_t first_value = __builtin_amdgcn_readfirstlane(value0 + front);
    float *const strip_vals = packed + first_value;
    const float *const strip_in = vals + start;
    constexpr uint32_t kTurn = 6, kApart = kBigThreads / 64u;     // steps a wavefront has on their way
    for (uint32_t step0 = t / 64u; step0 < num_steps; step0 += kTurn * kApart) {
        uint32_t rows_here[kTurn], value[kTurn];
        float v[kTurn][4];
#pragma unroll
        for (uint32_t u = 0; u < kTurn; ++u) {
            const uint32_t step = min(step0 + u * kApart, num_steps - 1u), m = rows_at(step * 64u + lane);
            const Two row = {steps[3u * step], steps[3u * step + 1u]};
            rows_here[u] = m;
            value[u] = steps[3u * step + 2u];
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) {
                const uint64_t in_row = __ballot(m >> k & 1u), held = __ballot(m >> (4u + k) & 1u);
                const uint32_t at = __builtin_amdgcn_mbcnt_hi(uint32_t(in_row >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(in_row), rp[k] - start + half(row, k)));
                v[u][k] = strip_in[m >> k & 1u ? at : 0u];
                value[u] = __builtin_amdgcn_mbcnt_hi(uint32_t(held >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(held), value[u]));
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kTurn; ++u) {
            if (step0 + u * kApart >= num_steps) break;
            const uint32_t a = (step0 + u * kApart) * 64u + lane, pair = a & 15u, mask = rows_here[u] >> 4;
            const uint32_t word = or_of_eight(mask << (4u * (pair & 7u)));
            uint32_t *rec = strip_recs + (a >> 4) * CUTE_QUAD_RECORD_WORDS, to = value[u];
            if ((a >> 4) < num_groups) {
                if (a >= active) rec[pair] = lo_hi[1];        // padding repeats the last column
                if (pair == 0u) { rec[16] = word; rec[18] = first_value + to; rec[19] = 0u; }
                if (pair == 8u) rec[17] = word;
            }
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k)
                if (mask >> k & 1u) strip_vals[to++] = v[u][k];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The other panels: a thread per entry, searches over the rows in global memory, positions and numbers in temporary
// arrays over the entries of these panels alone (index id = prefix[k] + position in the panel).
// ------------------------------------------------------------------------------------------------
// First index whose column is not below c[k] in each of R sorted ranges [lo[k], lo[k] + len[k]); left in lo.  The searches
// advance together, so their reads overlap: 57 -> 41 us for the hub panels of the graph above.
template <int R>
__device__ __forceinline__ void lower_bounds(const uint32_t *__restrict__ cols, uint32_t (&lo)[R], uint32_t (&len)[R], uint32_t c)
{
    uint32_t left;
    do {
        left = 0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t half = len[k] >> 1, probe = len[k] ? lo[k] + half : 0u;
            const bool less = cols[probe] < c && len[k] != 0u;
            lo[k] = less ? probe + 1u : lo[k];
            len[k] = less ? len[k] - half - 1u : half;
            left |= len[k];
        }
    } while (left);
}

__device__ __forceinline__ uint32_t upper_index(const uint32_t *__restrict__ prefix, uint32_t count, uint32_t id)
{
    uint32_t lo = 0, hi = count - 1u;                        // the k with prefix[k] <= id < prefix[k+1]
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (prefix[mid + 1] <= id) lo = mid + 1u;
        else hi = mid;
    }
    return lo;
}

// Position of every entry in the (column, row) order of its panel (posP) and of its strip (posS), and, at those positions,
// whether the entry is the first of its column there (firstP, firstS).  Also counts the stored values and checks the columns.
__global__ __launch_bounds__(kThreads) void large_positions(LargePanels L, const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                            const float *__restrict__ vals, uint32_t K, uint32_t *__restrict__ posP,
                                                            uint32_t *__restrict__ posS, uint32_t *__restrict__ firstP,
                                                            uint32_t *__restrict__ firstS, PanelCensus *__restrict__ res)
{
    const uint64_t id64 = global_id();
    const bool live = id64 < L.total;
    const uint32_t id = live ? uint32_t(id64) : L.total - 1u;
    const uint32_t k = upper_index(L.prefix, L.count, id), base = L.prefix[k];
    const uint32_t *rp = rowPtr + uint64_t(L.panel[k]) * 16u;
    const uint32_t panel_start = rp[0], e = panel_start + (id - base), me = row_in_panel(rp, e), strip0 = me & ~3u;
    const uint32_t c = cols[e];
    if (res) {
        uint32_t err = 0;
        if (c >= K) err |= kErrRange;
        if (e > rp[me] && cols[e - 1u] >= c) err |= kErrUnsorted;
        if (live && err) atomicOr(&res[k].error, err);
        // one addition per wavefront where its entries belong to one panel, which is nearly always
        const bool stored = live && vals[e] != 0.0f;
        const uint32_t k0 = __shfl(k, 0);
        if (__ballot(k != k0) == 0ull) {
            const uint64_t m = __ballot(stored);
            if ((threadIdx.x & 63u) == 0u && m) atomicAdd(&res[k].stored, uint32_t(__popcll(m)));
        } else if (stored) atomicAdd(&res[k].stored, 1u);
    }
    if (!live) return;
    uint32_t below = 0, above_same = 0, below_s = 0, above_same_s = 0;
#pragma unroll
    for (uint32_t i0 = 0; i0 < 16u; i0 += 4u) {              // a strip's rows at a time
        uint32_t lo[4], len[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) { lo[k] = rp[i0 + k]; len[k] = rp[i0 + k + 1u] - lo[k]; }
        lower_bounds<4>(cols, lo, len, c);
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            const uint32_t i = i0 + k, cnt = lo[k] - rp[i];  // (the entry's own row counts the entries in front of it)
            const uint32_t has = (i < me && lo[k] < rp[i + 1u] && cols[lo[k]] == c) ? 1u : 0u;
            below += cnt;
            above_same += has;
            if (i0 == strip0) { below_s += cnt; above_same_s += has; }
        }
    }
    // (columns that are not sorted give positions that mean nothing, but never ones outside the panel: the census refuses them)
    const uint32_t last = L.prefix[k + 1] - 1u;
    const uint32_t pp = min(base + below + above_same, last), ps = min(base + (rp[strip0] - panel_start) + below_s + above_same_s, last);
    posP[id] = pp;
    posS[id] = ps;
    firstP[pp] = above_same == 0u ? 1u : 0u;
    firstS[ps] = above_same_s == 0u ? 1u : 0u;
}

// Active columns and list pairs of the large panels, from the prefix sums DP, DS of the first flags.
__global__ __launch_bounds__(kThreads) void large_counts(LargePanels L, const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ DP,
                                                         const uint32_t *__restrict__ DS, const PanelCensus *__restrict__ res, PanelCensus *__restrict__ out)
{
    const uint64_t k = global_id();
    if (k >= L.count) return;
    const uint32_t p = L.panel[k], base = L.prefix[k], end = L.prefix[k + 1];
    const uint32_t *rp = rowPtr + uint64_t(p) * 16u;
    auto run = [](const uint32_t *__restrict__ D, uint32_t b, uint32_t e) { return e > b ? D[e - 1u] - (b ? D[b - 1u] : 0u) : 0u; };
    out[p].cols = run(DP, base, end);
    for (uint32_t s = 0; s < 4u; ++s) out[p].pairs[s] = run(DS, base + (rp[4u * s] - rp[0]), base + (rp[4u * s + 4u] - rp[0]));
    out[p].stored = res[k].stored;
    out[p].error = res[k].error;
}

// unit[k]: first block (group) of large panel k in the layout; unitPrefix: running number of blocks (groups) over the large
// panels.  Clears their header lines (records), which the scatter below fills with atomics.
__global__ __launch_bounds__(kThreads) void large_clear(const uint32_t *__restrict__ unit, const uint32_t *__restrict__ unitPrefix,
                                                        uint32_t count, uint32_t words, uint32_t *__restrict__ dst)
{
    const uint64_t id = global_id();
    if (id >= uint64_t(unitPrefix[count]) * words) return;
    const uint32_t u = uint32_t(id / words), k = upper_index(unitPrefix, count, u);
    dst[(uint64_t(unit[k]) + (u - unitPrefix[k])) * words + uint32_t(id % words)] = 0u;
}

__global__ __launch_bounds__(kThreads) void large_bricks(LargePanels L, const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                         const float *__restrict__ vals, const uint32_t *__restrict__ posP,
                                                         const uint32_t *__restrict__ DP, const uint32_t *__restrict__ unit,
                                                         uint32_t *hdr, float *__restrict__ tile_vals)
{
    const uint64_t id = global_id();
    if (id >= L.total) return;
    const uint32_t k0 = upper_index(L.prefix, L.count, uint32_t(id)), base = L.prefix[k0];
    const uint32_t *rp = rowPtr + uint64_t(L.panel[k0]) * 16u;
    const uint32_t start = rp[0], e = start + (uint32_t(id) - base), row = row_in_panel(rp, e), pos = posP[id];
    const uint32_t a = DP[pos] - DP[base];                   // index of the entry's column among the panel's active columns
    const uint32_t j = (a >> 2) & 3u, k = a & 3u;
    uint32_t *h = hdr + (uint64_t(unit[k0]) + (a >> 4)) * CUTE_TILED_HDR_WORDS;
    tile_vals[start + (pos - base)] = vals[e];
    const uint32_t bit = k * 16u + row;                      // the A operand slot of lane `bit` in v_mfma_f32_16x16x4_f32
    atomicOr(h + 16u + 2u * j + (bit >> 5), 1u << (bit & 31u));
    if (pos == base || DP[pos] != DP[pos - 1u]) {            // first entry of its column: the column's own words
        h[k * 4u + j] = cols[e];
        if (k == 0u) h[24u + j] = start + (pos - base);
    }
}

// Per block of a large panel: value offsets of bricks that hold padding columns only (they point at the end of the block,
// where a running offset would stand) and the number of entries in the block.
__global__ __launch_bounds__(kThreads) void large_brick_ends(LargePanels L, const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ unit,
                                                             const uint32_t *__restrict__ unitPrefix, const uint32_t *__restrict__ panelCols,
                                                             uint32_t *hdr)
{
    const uint64_t b = global_id();
    if (b >= unitPrefix[L.count]) return;
    const uint32_t k = upper_index(unitPrefix, L.count, uint32_t(b)), local = uint32_t(b) - unitPrefix[k];
    uint32_t *h = hdr + (uint64_t(unit[k]) + local) * CUTE_TILED_HDR_WORDS;
    const bool last = b + 1u == unitPrefix[k + 1u];
    const uint32_t end = last ? rowPtr[uint64_t(L.panel[k]) * 16u + 16u] : h[CUTE_TILED_HDR_WORDS + 24u];
    const uint32_t live = min(16u, panelCols[k] - 16u * local);
    for (uint32_t j = 1; j < 4u; ++j)
        if (4u * j >= live) h[24u + j] = end;
    h[28] = end - h[24];
}

// Where the pair of an entry of large panel k stands.  STRIPS: one list per 4-row strip (a group = 16 consecutive pairs of one
// strip, group[4k + s] its first); else four lockstep lists per panel (pair 4*step + list, group[k] the panel's first).
template <bool STRIPS>
__device__ __forceinline__ void large_place(uint32_t k, uint32_t row, uint32_t stripBase, uint32_t pos, const uint32_t *__restrict__ DS,
                                            const uint32_t *__restrict__ group, uint32_t &g, uint32_t &pair, bool &first)
{
    const uint32_t s = row >> 2;
    const uint32_t q = DS[pos] - DS[stripBase];              // index of the entry's column in the strip's list
    if (STRIPS) {
        g = group[4u * k + s] + (q >> 4);
        pair = q & 15u;
    } else {
        g = group[k] + (q >> 2);
        pair = 4u * (q & 3u) + s;
    }
    first = pos == stripBase || DS[pos] != DS[pos - 1u];
}

// VALUES false: columns and slot masks of the records (cleared before); true: the stored values, once the records are whole.
template <bool STRIPS, bool VALUES>
__global__ __launch_bounds__(kThreads) void large_quads(LargePanels L, const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                        const float *__restrict__ vals, const uint32_t *__restrict__ posS,
                                                        const uint32_t *__restrict__ DS, const uint32_t *__restrict__ group,
                                                        uint32_t *recs, float *__restrict__ packed)
{
    const uint64_t id = global_id();
    if (id >= L.total) return;
    const uint32_t k = upper_index(L.prefix, L.count, uint32_t(id)), base = L.prefix[k];
    const uint32_t *rp = rowPtr + uint64_t(L.panel[k]) * 16u;
    const uint32_t e = rp[0] + (uint32_t(id) - base), row = row_in_panel(rp, e);
    const float v = vals[e];
    if (VALUES && v == 0.0f) return;
    uint32_t g, pair;
    bool first;
    large_place<STRIPS>(k, row, base + (rp[row & ~3u] - rp[0]), posS[id], DS, group, g, pair, first);
    uint32_t *rec = recs + uint64_t(g) * CUTE_QUAD_RECORD_WORDS;
    const uint32_t slot = 4u * pair + (row & 3u);
    if (VALUES) {
        const uint64_t mask = (uint64_t(rec[17]) << 32) | rec[16];
        packed[rec[18] + uint32_t(__popcll(mask & ((1ull << slot) - 1ull)))] = v;
    } else {
        if (v != 0.0f) atomicOr(rec + 16u + (slot >> 5), 1u << (slot & 31u));   // an explicit zero is an empty slot
        if (first) rec[pair] = cols[e];
    }
}

// Per group of a large panel: the number of stored values (counts, for the prefix sum that gives each group its first value)
// and the columns of padding pairs, which repeat the last column of their list (0 for an empty list).
template <bool STRIPS>
__global__ __launch_bounds__(kThreads) void large_groups(LargePanels L, const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols,
                                                         const uint32_t *__restrict__ group, const uint32_t *__restrict__ groupPrefix,
                                                         const uint32_t *__restrict__ stripPairs, uint32_t *recs, uint32_t *__restrict__ counts)
{
    const uint64_t id = global_id();
    if (id >= groupPrefix[L.count]) return;
    const uint32_t k = upper_index(groupPrefix, L.count, uint32_t(id)), local = uint32_t(id) - groupPrefix[k];
    const uint32_t g = (STRIPS ? group[4u * k] : group[k]) + local;
    uint32_t *rec = recs + uint64_t(g) * CUTE_QUAD_RECORD_WORDS;
    counts[id] = uint32_t(__popc(rec[16]) + __popc(rec[17]));
    for (uint32_t s = 0; s < 4u; ++s) {
        const uint32_t len = stripPairs[4u * k + s];
        uint32_t first_step, per;                            // steps of this list inside the group: 16 (strips) or 4 (lockstep)
        if (STRIPS) {
            const uint32_t g0 = group[4u * k + s];
            if (g < g0 || g >= g0 + (len + 15u) / 16u) continue;
            first_step = 16u * (g - g0); per = 16u;
        } else { first_step = 4u * local; per = 4u; }
        if (first_step + per <= len) continue;               // no padding in this list here
        uint32_t last = 0;
        const uint32_t *rp = rowPtr + uint64_t(L.panel[k]) * 16u + 4u * s;
        if (len)
            for (uint32_t i = 0; i < 4u; ++i)
                if (rp[i + 1u] > rp[i]) last = max(last, cols[rp[i + 1u] - 1u]);
        for (uint32_t x = 0; x < per; ++x)
            if (first_step + x >= len) rec[STRIPS ? x : 4u * x + s] = last;
    }
}

// counts holds the inclusive prefix sums of the stored values per group: word 18 of a record is the index of the group's first.
__global__ __launch_bounds__(kThreads) void large_first_values(const uint32_t *__restrict__ unit, const uint32_t *__restrict__ groupPrefix, const uint32_t *__restrict__ valBase,
                                                               uint32_t count, const uint32_t *__restrict__ counts, uint32_t *recs)
{
    const uint64_t id = global_id();
    if (id >= groupPrefix[count]) return;
    const uint32_t k = upper_index(groupPrefix, count, uint32_t(id)), b = groupPrefix[k];
    const uint32_t before = (id ? counts[id - 1u] : 0u) - (b ? counts[b - 1u] : 0u);
    recs[(uint64_t(unit[k]) + (uint32_t(id) - b)) * CUTE_QUAD_RECORD_WORDS + 18u] = valBase[k] + before;
}

// The tables of a plan, from its staged host copy, in one launch: chunk descriptors -- or, for the quad kernels (recs given),
// one 128-byte head per work item: its descriptor and a copy of its first group's record --, the list of cut panels, the
// row kernel's list of a mixed plan, expanded from panels: every row with its row pointers, {row, first entry, end, 0}, and what the
// pieces of cut panels add themselves up with.
struct PlanTables {
    const uint4 *chunks;       // staged
    const uint4 *fixups;
    const uint32_t *rowPanels;
    uint32_t numChunks, numFixups, numRowPanels;
    uint4 *dChunks;            // device
    uint32_t *dHeads;
    uint4 *dFixups, *dRowList;
    const uint4 *cut;          // staged: what the pieces of cut panels add themselves up with, and their counters behind it
    uint4 *dCut;               // device
    uint64_t numCut, counterWords;
};

__global__ __launch_bounds__(kThreads) void plan_tables(PlanTables T, const uint32_t *__restrict__ recs, uint32_t head_words,
                                                        const uint32_t *__restrict__ rowPtr)
{
    uint64_t id = global_id();
    const uint64_t chunk_items = uint64_t(T.numChunks) * (recs ? head_words : 1u);
    if (id < chunk_items) {
        if (!recs) { T.dChunks[id] = T.chunks[id]; return; }
        const uint32_t w = uint32_t(id % head_words);
        const uint4 ck = T.chunks[id / head_words];
        uint32_t v = 0;
        if (w == 0) v = ck.x;
        else if (w == 1) v = ck.y;
        else if (w == 2) v = ck.z;
        else if (w == 3) v = ck.w;
        else if (w < 4u + CUTE_QUAD_RECORD_WORDS && ck.x < ck.y) v = recs[uint64_t(ck.x) * CUTE_QUAD_RECORD_WORDS + (w - 4u)];
        T.dHeads[id] = v;
        return;
    }
    id -= chunk_items;
    if (id < T.numFixups) { T.dFixups[id] = T.fixups[id]; return; }
    id -= T.numFixups;
    if (id < uint64_t(T.numRowPanels) * 16u) {
        const uint32_t r = T.rowPanels[id >> 4] * 16u + uint32_t(id & 15u);
        T.dRowList[id] = make_uint4(r, rowPtr[r], rowPtr[r + 1u], 0u);
        return;
    }
    id -= uint64_t(T.numRowPanels) * 16u;
    if (id < T.numCut) T.dCut[id] = T.cut[id];
    else if (id - T.numCut < (T.counterWords + 3u) / 4u) T.dCut[id] = make_uint4(0u, 0u, 0u, 0u);      // (an array ends on 256 bytes)
}

// Hub plans (hrpb_quad_hub_f32): how often every column occurs in the quad records, and a copy of the records in
// which the columns that have a slot in the LDS table of hub rows (slot_of[col] != ~0u) name that slot instead.
__global__ __launch_bounds__(kThreads) void count_record_columns(const uint32_t *__restrict__ recs, uint64_t numGroups,
                                                                 uint32_t *__restrict__ counts)
{
    const uint64_t id = global_id();
    if (id >= numGroups * 16u) return;
    atomicAdd(&counts[recs[(id >> 4) * CUTE_QUAD_RECORD_WORDS + (id & 15u)]], 1u);
}

__global__ __launch_bounds__(kThreads) void mark_hub_columns(const uint32_t *__restrict__ recs, uint64_t numGroups,
                                                             const uint32_t *__restrict__ slot_of, uint32_t hub_flag,
                                                             uint32_t *__restrict__ out)
{
    const uint64_t id = global_id();
    if (id >= numGroups * CUTE_QUAD_RECORD_WORDS) return;
    uint32_t w = recs[id];
    if (id % CUTE_QUAD_RECORD_WORDS < 16u) {
        const uint32_t slot = slot_of[w];
        if (slot != ~0u) w = hub_flag | slot;
    }
    out[id] = w;
}

// The entries of csr_rows_window (which describes them): a work-group is a slice.  The slice's part of the CSR arrays is one piece,
// so it is read, and the quads are written, whole lines at a time, and four lanes a row sort in between in
// LDS (a lane that walks its row in global memory touches a line an entry: 33.5 million entries 2 400 us; one lane a row in LDS
// 300, this way 94, 5 TB/s).  The order inside a row, (slot + row / 2) mod 8, is a counting sort by the eight bytes of one
// word: rows of fewer than 256 entries.  `staged`: {first quad, -, quads, -} of every slice, and the tiles' windows, in host memory
// (asked for behind the entries, which would wait for it); slices[] gets the quads that no row of the slice pads besides.
struct WindowTables {
    const uint4 *slices;       // staged
    const uint2 *tiles;
    uint32_t numTiles;
    uint4 *dSlices;            // device
    uint2 *dTiles;
};

// rows of 32 entries do not start in one bank
__device__ __forceinline__ uint32_t skewed(uint32_t i) { return i + (i >> 5); }
__device__ __forceinline__ uint32_t skewed_half(uint32_t i) { return i + 2u * (i >> 5); }

__global__ __launch_bounds__(kThreads) void window_entries(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols, const float *__restrict__ vals,
                                                     uint32_t M, uint32_t ring_rows, WindowTables T, uint32_t longest, uint2 *__restrict__ slots,
                                                     f32x4 *__restrict__ out)
{
    static_assert(kThreads == 4 * 64, "four lanes a row");
    extern __shared__ uint32_t lds[];
    __shared__ uint32_t least_of[kThreads / 64];
    const uint32_t slice = blockIdx.x, tid = threadIdx.x, row0 = slice * 64u;
    float *val_of = reinterpret_cast<float *>(lds), *placed_val = val_of + skewed(64u * longest);
    uint16_t *placed_slot = reinterpret_cast<uint16_t *>(placed_val + 64u * longest), *slot_of = placed_slot + 64u * longest;
    const uint32_t lane = tid >> 2, part = tid & 3u, row = row0 + lane, begin = rowPtr[row0], end = rowPtr[min(row0 + 64u, M)],
                   s = rowPtr[min(row, M)], n = rowPtr[min(row + 1u, M)] - s;
    for (uint32_t base = begin; base < end; base += 8u * kThreads) {
        uint32_t col[8];
        float val[8];
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
            const uint32_t i = base + u * kThreads + tid;
            if (i < end) { col[u] = cols[i]; val[u] = vals[i]; }
        }
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
            const uint32_t i = base + u * kThreads + tid;
            if (i < end) { slot_of[skewed_half(i - begin)] = uint16_t(col[u] % ring_rows); val_of[skewed(i - begin)] = val[u]; }
        }
    }
    uint4 d = T.slices[slice];
    for (uint32_t t = slice * kThreads + tid; t < T.numTiles; t += gridDim.x * kThreads) T.dTiles[t] = T.tiles[t];
    __syncthreads();
    {
        const uint32_t turn = lane >> 1, first = s - begin, per = (n + 3u) / 4u, i0 = min(part * per, n), i1 = min(i0 + per, n);
        uint64_t mine = 0;
        for (uint32_t i = i0; i < i1; ++i) mine += 1ull << (8u * ((slot_of[skewed_half(first + i)] + turn) & 7u));
        uint64_t upto = mine;
#pragma unroll
        for (int step = 1; step < 4; step *= 2) {
            const uint64_t other = __shfl_up(static_cast<unsigned long long>(upto), step, 4);
            if (part >= uint32_t(step)) upto += other;
        }
        // where the entries of each of the eight begin, and this lane's among them
        const uint64_t all = __shfl(static_cast<unsigned long long>(upto), 3, 4);
        uint64_t place = all * 0x0101010101010100ull + (upto - mine);
        auto at = [&](uint32_t k) { return (k / 4u * 64u + lane) * 4u + k % 4u; };
        for (uint32_t i = i0; i < i1; ++i) {
            const uint32_t slot = slot_of[skewed_half(first + i)], shift = 8u * ((slot + turn) & 7u), to = at(uint32_t(place >> shift) & 255u);
            place += 1ull << shift;
            placed_slot[to] = uint16_t(slot);
            placed_val[to] = val_of[skewed(first + i)];
        }
        for (uint32_t k = n + part; k < d.z * 4u; k += 4u) {
            placed_slot[at(k)] = uint16_t(0xffffu);
            placed_val[at(k)] = 0.0f;
        }
        uint32_t least = n / 4u;
#pragma unroll
        for (int step = 1; step < 64; step *= 2) least = min(least, uint32_t(__shfl_xor(int(least), step)));
        if ((tid & 63u) == 0u) least_of[tid >> 6] = least;
    }
    __syncthreads();
    if (tid == 0u) {
        d.y = min(min(least_of[0], least_of[1]), min(least_of[2], least_of[3]));
        T.dSlices[slice] = d;
    }
    const uint2 *slots_in = reinterpret_cast<const uint2 *>(placed_slot);
    const f32x4 *vals_in = reinterpret_cast<const f32x4 *>(placed_val);
    for (uint32_t i = tid; i < d.z * 64u; i += kThreads) {
        slots[size_t(d.x) * 64u + i] = slots_in[i];
        out[size_t(d.x) * 64u + i] = vals_in[i];
    }
}

// LDS of window_entries for rows of up to `longest` entries (a multiple of four, so that what is read 16 bytes at a time begins at them).
inline uint32_t window_entries_lds(uint32_t longest) { return 64u * longest * 12u + 2u * longest * 4u + 4u * longest * 2u; }

}  // namespace cute_build
