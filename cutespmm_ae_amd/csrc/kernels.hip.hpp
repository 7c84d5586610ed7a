// gfx950 device kernels of libcutespmm.
//
//   hrpb_brick_f32_rolling   one wavefront per (row-panel chunk, N slab) over the brick tiles; every non-empty
//                    16x4 brick is one v_mfma_f32_16x16x4_f32 A operand taken straight from the lane-order
//                    bitmap; B rows are gathered in the MFMA B-operand layout (16 lanes read one contiguous
//                    row segment), so no LDS transpose is needed.  One operand set, refilled behind the MFMAs.
//   hrpb_brick_f32   the same work with two whole operand sets in flight and 64-bit addressing (operands
//                    beyond the 32-bit offsets of the rolling variant).
//   hrpb_brick_bf16x3   the brick tiles on the bf16 matrix pipeline: operands split into bf16 high and low
//                    parts in registers, three v_mfma_f32_16x16x16_bf16 per block and 16 columns.
//   hrpb_quad_f32    quad lists: v_mfma_f32_4x4x1_16B_f32 over 16 (row group, column) pairs at a time, so
//                    only occupied 4-row column pieces cost matrix time.
//   csr_rows_batched one lane group per CSR row, lanes span N, 8 (col, val) pairs in flight; the kernel
//                    for panels with too little reuse for the matrix cores.
//   csr_rows_window  rows whose columns move along with them: their window of B slides through LDS.
//   csr_rows_split   products of a few columns: several lane groups share a row.
//   hrpb_quad_rows_f32 / hrpb_brick_rows_f32   MFMA work items and sparse rows of a mixed plan in one launch.
//   reduce_partials  adds up the partial tiles of panels that were cut, where their pieces do not do it themselves (store_piece).
//   blocked_ell_f32  fp32 MFMA over the dense blocks of a Blocked-ELL matrix.
//   csr_rows / csr_thread_per_element / csr_wave_scalar   the simple CSR comparison kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cutespmm.h"

namespace cute_dev {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

template <int VEC> struct Vec;
template <> struct Vec<1> { typedef float type; };
template <> struct Vec<2> { typedef f32x2 type; };
template <> struct Vec<4> { typedef f32x4 type; };

// B and C rows are N floats apart, so a lane's VEC consecutive columns are VEC-aligned only when N is a multiple of VEC.
// Global memory needs dword alignment for loads and stores of any width, so every N >= VEC moves VEC columns per lane:
// a lane whose columns would pass column N takes the row's last VEC columns instead (first_column), and the few columns
// two lanes then share are computed twice, in the same order, and stored twice with the same bits.  The alternative, the
// widest VEC that divides N, made odd N one float per lane: R-MAT graph of 65 536 nodes, N = 47: 85.3 us a product
// against 36.4, 9-point stencil of 200 x 200 points, N = 101: 17.3 against 11.4.
template <int VEC> struct VecInMemory { typedef typename Vec<VEC>::type type __attribute__((aligned(4))); };
template <int VEC> __device__ __forceinline__ typename Vec<VEC>::type load_vec(const void *p)
{
    return *reinterpret_cast<const typename VecInMemory<VEC>::type *>(p);
}
template <int VEC> __device__ __forceinline__ void store_vec_streaming(const typename Vec<VEC>::type &v, void *p)
{
    // C is not read again by the launch that writes it: keep it out of the L2
    __builtin_nontemporal_store(v, reinterpret_cast<typename VecInMemory<VEC>::type *>(p));
}
template <int VEC> __device__ __forceinline__ uint32_t first_column(uint32_t c, uint32_t N) { return min(c, N - uint32_t(VEC)); }

template <int VEC> __device__ __forceinline__ float vec_get(const typename Vec<VEC>::type &v, int i) { return v[i]; }
template <> __device__ __forceinline__ float vec_get<1>(const float &v, int) { return v; }
template <int VEC> __device__ __forceinline__ void vec_set(typename Vec<VEC>::type &v, int i, float x) { v[i] = x; }
template <> __device__ __forceinline__ void vec_set<1>(float &v, int, float x) { v = x; }

constexpr int kWaveSize = 64;
constexpr int kWavesPerGroup = 4;
constexpr int kHdrWords = 32;
constexpr int kNumXcd = 8;
constexpr int kQuadRecordWords = CUTE_QUAD_RECORD_WORDS;   // device record of one quad-list group: 16 columns, mask lo/hi, first value, pad
constexpr int kQuadHeadWords = 32;     // quad kernels, per chunk: descriptor (4 words), first group's record, padding to 128 bytes

// Work-groups are handed to the 8 XCDs round-robin; this maps the hardware id to a
// logical id such that each XCD walks one contiguous range of logical ids (neighbouring
// row panels share B rows, which then stay in that XCD's L2).
__device__ __forceinline__ uint32_t xcd_contiguous_id(uint32_t bid, uint32_t groups_per_xcd)
{
    return (bid % kNumXcd) * groups_per_xcd + bid / kNumXcd;
}

// The same idea with ranges of unequal length (balanced by work, not by count): range x holds the
// logical blocks [first[x], first[x+1]); the launch has kNumXcd * (longest range) blocks.
struct XcdRanges {
    uint32_t first[kNumXcd + 1];
};

__device__ __forceinline__ bool xcd_range_id(const XcdRanges &r, uint32_t bid, uint32_t x, uint32_t &logical)
{
    logical = r.first[x] + bid / kNumXcd;
    return logical < r.first[x + 1];
}

// Which eighth of the list a work-group takes, and in which slab.  In row order (column_slabs = 0) XCD x walks eighth x of every
// slab, slab after slab: neighbouring rows share B rows in its L2.  A matrix whose rows read columns from all over B gains
// nothing from that, and every XCD fetches all of B from behind its L2.  By columns, the slabs' eighths are dealt in slab order:
// XCD x takes the column_slabs eighths from x * column_slabs on, that is 1/8 of the columns and (almost) all rows of them, and
// the L2 has to hold those columns only.  The same eighths, only permuted: every (slab, eighth) is still taken once.
// 16 384 rows of 8 random columns, N = 512: 35.4 us in row order, 18.3 by columns (32-column slabs, 2 MB of B each).
// The kernels of the default plans are compiled for each order (COLUMNS): deciding at run time put the argument and the
// division by it in front of a wavefront's first fetch, 0.5 of 13.8 us on the 9-point stencil of 256 x 256 points, N = 128.
__device__ __forceinline__ uint32_t xcd_share(uint32_t bid, uint32_t &slab, uint32_t column_slabs)
{
    const uint32_t x = bid % kNumXcd;
    if (!column_slabs) return x;
    const uint32_t e = x * column_slabs + slab;
    slab = e / kNumXcd;
    return e % kNumXcd;
}

struct BlockHeader {          // one 128-byte header line as a wavefront sees it
    uint64_t bitmap[4];       // wave-uniform (scalar loads)
    uint32_t voff[4];         // wave-uniform
    uint4 cols;               // per lane: the (lane/16)-th active column of bricks 0..3
};

template <int VEC, int NG>
struct BlockOperands {
    float a[4];                                   // value at (brick offset + lane rank), before masking
    uint64_t bitmap[4];                           // wave-uniform: lane L is a nonzero iff bit L
    typename Vec<VEC>::type b[4][NG];             // B operand vectors per brick and column group
};

__device__ __forceinline__ BlockHeader load_header(const uint32_t *__restrict__ hdr, uint32_t blk, uint32_t lane)
{
    const uint32_t *h = hdr + size_t(blk) * kHdrWords;
    BlockHeader r;
    r.cols = reinterpret_cast<const uint4 *>(h)[lane >> 4];
    const uint64_t *bm = reinterpret_cast<const uint64_t *>(h + 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) r.bitmap[j] = bm[j];
#pragma unroll
    for (int j = 0; j < 4; ++j) r.voff[j] = h[24 + j];
    return r;
}

// Issues every load of one block without a branch: bricks that consist of padding only
// have an all-zero bitmap and padding columns point at B row 0, so they contribute
// 0 * B[0][.] (B must be finite, as in the reference, kernel.cu:26-27,149).  vals[] is
// padded by one wavefront of floats so that the unconditional A load never leaves it.
template <int VEC, int NG, bool FULL>
__device__ __forceinline__ void load_operands(BlockOperands<VEC, NG> &o, const BlockHeader &hd,
                                              const float *__restrict__ vals, const float *__restrict__ B,
                                              uint32_t N, uint32_t col0, uint32_t lane)
{
    const uint32_t cols[4] = {hd.cols.x, hd.cols.y, hd.cols.z, hd.cols.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint64_t bm = hd.bitmap[j];
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(uint32_t(bm >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(bm), 0u));
        o.a[j] = vals[hd.voff[j] + below];       // masked when consumed, so nothing waits here
        o.bitmap[j] = bm;
        const float *brow = B + size_t(cols[j]) * N;
#pragma unroll
        for (int ng = 0; ng < NG; ++ng) {
            // lanes beyond column N re-read the row's last VEC columns and store nothing:
            // a branch around the load would split the pipeline's basic blocks
            const uint32_t c = col0 + uint32_t(ng) * 16u * VEC;
            o.b[j][ng] = load_vec<VEC>(brow + (FULL ? c : first_column<VEC>(c, N)));
        }
    }
}

template <int VEC, int NG>
__device__ __forceinline__ void mfma_block(const BlockOperands<VEC, NG> &o, f32x4 (&acc)[NG][VEC], uint32_t lane)
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float a = ((o.bitmap[j] >> lane) & 1ull) ? o.a[j] : 0.0f;
#pragma unroll
        for (int ng = 0; ng < NG; ++ng)
#pragma unroll
            for (int v = 0; v < VEC; ++v)
                acc[ng][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vec_get<VEC>(o.b[j][ng], v), acc[ng][v], 0, 0, 0);
    }
}

// chunks[i] = {first block, end block, row panel, piece}.  piece = 0: the chunk is its panel's only one and
// stores the C tile; piece = k > 0: the panel is cut, and this chunk stores its partial tile as "panel" k-1
// of the partials matrix (same row pitch as C); store_piece says who adds them up.  A work item is (chunk, slab);
// slab s covers columns [s*16*VEC*NG, (s+1)*16*VEC*NG).  Lane L = 16*g + j owns, inside
// column group ng, the VEC consecutive columns starting at s*slab + ng*16*VEC + j*VEC;
// MFMA tile v of that group therefore holds the columns {.. + j*VEC + v}, and after the
// MFMA lane L holds rows 4g..4g+3 of exactly those VEC columns -> one vector store per row.
// FULL: N is a multiple of the slab width, so no column guard is compiled in.
struct BrickItem {
    uint32_t start, end, panel, piece, col0, slab;
    bool valid;
};

// The launch is a 2-D grid: x walks the chunks (kWavesPerGroup per work-group, remapped so that
// each XCD owns a contiguous range), y is the slab.  gridDim.x is a multiple of the XCD count,
// so the slabs of one chunk run on the same XCD and share its B rows in that L2.
template <int VEC, int NG>
__device__ __forceinline__ BrickItem brick_item(const uint4 *__restrict__ chunks, uint32_t num_chunks,
                                                uint32_t groups_per_xcd, uint32_t lane, uint32_t block_x, uint32_t block_y, uint32_t column_slabs)
{
    BrickItem it;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const uint32_t x = xcd_share(block_x, block_y, column_slabs);
    const uint32_t chunk = (x * groups_per_xcd + block_x / kNumXcd) * kWavesPerGroup + wave;
    it.valid = chunk < num_chunks;
    if (!it.valid) return it;
    const uint4 ck = chunks[chunk];
    it.start = __builtin_amdgcn_readfirstlane(ck.x);
    it.end = __builtin_amdgcn_readfirstlane(ck.y);
    it.panel = __builtin_amdgcn_readfirstlane(ck.z);
    it.piece = __builtin_amdgcn_readfirstlane(ck.w);
    it.slab = block_y;
    it.col0 = block_y * (16u * VEC * NG) + (lane & 15u) * VEC;
    return it;
}

// ---------------------------------------------------------------------------------------
// Panels (or 4-row strips) that the planner cut: every piece stores its partial tile, and the pieces are added up in an order
// that depends on their number alone -- eight consecutive pieces one after the other, then the sums of these eights one after
// the other -- so the same product gives the same bits every time, whoever does the adding.
//
// Inside the launch (a CutPieces given) the pieces of an eight count themselves in behind their tiles, the one that comes last adds
// the eight up, and of those, where there are several eights, the last one adds the sums up.  Nobody waits for anybody, and a
// counter returns to zero by itself (atomicInc wraps), so the next launch finds it as this one did.  What a piece stores for
// others, and what it reads of theirs, passes by the XCD's own L2 (agent-scope accesses): counting in then needs the stores to have
// arrived, not the write-back of everything the L2 holds that a device-wide release is on this part (which made counting in 1.1 to 5.5
// times slower than a second launch).  A plan without cut panels runs the kernels that are compiled without any of this (CUT = false): the branch and
// the registers behind it cost 0.5 to 1 % of a short launch (9-point stencil of 200 x 200 points, N = 101, 9.54 -> 9.65 us; hrpb_quad_half_f32 46 -> 50
// vector registers).
// With a second launch (reduce_partials), as calls whose scratch comes without counters and kernels that are no plan's default have it, and
// without, us: R-MAT graph of 131 072 nodes, N = 64 45.0 / 44.0; 65 536 nodes, N = 47 26.6 / 23.9.
// ---------------------------------------------------------------------------------------
constexpr uint32_t kPiecesAtOnce = 8;
constexpr uint32_t kEightsOfOne = 2;          // up to so many eights the last piece of all adds them up, and nobody an eight

struct CutPieces {             // in device memory: an argument more would be in registers from a wavefront's start
    const uint4 *of_piece;     // {first piece of the unit, pieces, first counter, unit}
    uint32_t *counters;        // an eight's counters, then one for the eights; a word for each slab
    uint64_t slabs;
};

// Loads and stores of W columns with the scope bit that the compiler gives agent-scope atomics (sc1), which the language has for single words only.  A word
// a lane, bricks of two or four columns left every line in pieces that memory has to put together: R-MAT graph of 32 768 nodes and 9 edges a node, N = 84, bf16x3
// 58.9 us, 16 384 nodes and 4 edges, N = 24 13.5; with whole vectors 35.6 ... 36.5 and 8.9 ... 9.3 (a second launch instead: 36.5 and 9.5).
constexpr int kAgentScope = 16;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t shared_tiles(float *partials) { return __builtin_amdgcn_make_buffer_rsrc(partials, 0, ~0u, 0x00020000); }
template <int W> __device__ __forceinline__ typename Vec<W>::type load_shared(float *partials, uint32_t at, uint32_t further)
{
    if constexpr (W == 4) return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(shared_tiles(partials), at, further, kAgentScope));
    else if constexpr (W == 2) return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(shared_tiles(partials), at, further, kAgentScope));
    else return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(shared_tiles(partials), at, further, kAgentScope));
}
template <int W> __device__ __forceinline__ void store_shared(float *partials, uint32_t at, const typename Vec<W>::type &x)
{
    if constexpr (W == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), shared_tiles(partials), at, 0, kAgentScope);
    else if constexpr (W == 2) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), shared_tiles(partials), at, 0, kAgentScope);
    else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), shared_tiles(partials), at, 0, kAgentScope);
}

// The lane, without a register that holds it: what the end of a piece needs is not kept through its main loop.
__device__ __forceinline__ uint32_t lane_again() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// Counts the wavefront in; true for the last of `members`.
__device__ __forceinline__ bool last_to_arrive(uint32_t *counter, uint32_t members)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // what this wavefront stored has arrived
    uint32_t before = 0;
    if (lane_again() == 0u) before = atomicInc(counter, members - 1u);
    const bool last = __builtin_amdgcn_readfirstlane(before) == members - 1u;
    asm volatile("" ::: "memory");
    return last;
}

// sum (of the values so far), then v[0] .. v[n - 1] one after the other
template <class T> __device__ __forceinline__ T add_pieces(T sum, bool none_so_far, uint32_t n, const T (&v)[kPiecesAtOnce])
{
#pragma unroll
    for (uint32_t k = 0; k < kPiecesAtOnce; ++k) {
        const T next = k == 0u && none_so_far ? v[0] : sum + v[k];
        sum = k < n ? next : sum;
    }
    return sum;
}

// A lane's part of the tile of a piece: E vectors of W columns, at(unit, e) the byte offset of vector e of tile (or panel, or strip) `unit`.  Near the last
// column two lanes, or two vectors of one, hold the same columns: the last own(e) of a vector are the lane's.  (The sums of an eight
// stand where its first tile does, so a place that was read again after it was written would count twice.)  pitch: bytes from a tile to the next; ragged: a
// vector may be partly owned.
template <int W, int E, class At, class Own>
__device__ __forceinline__ void store_piece(const CutPieces *__restrict__ cut, uint32_t piece, uint32_t slab, const typename Vec<W>::type (&mine)[E], At at, Own own,
                                            uint32_t pitch, bool ragged, float *__restrict__ partials, float *__restrict__ C)
{
    typedef typename Vec<W>::type V;
    float *tiles = partials;
    asm volatile("" : "+s"(tiles));        // other wavefronts write here too: not the argument that nothing else points to
    auto put = [&](uint32_t unit, int e, const V &v, auto whole, auto word) {
        const uint32_t n = own(e);
        if (n == uint32_t(W)) whole(at(unit, e), v);
        if constexpr (W > 1)
            if (ragged)
#pragma unroll
                for (int j = 1; j < W; ++j)
                    if (n < uint32_t(W) && uint32_t(W - j) <= n) word(at(unit, e) + uint32_t(j) * 4u, vec_get<W>(v, j));
    };
    auto to_tile = [&](uint32_t tile, int e, const V &v) {
        put(tile, e, v, [&](uint32_t to, const V &x) { store_shared<W>(tiles, to, x); }, [&](uint32_t to, float x) { store_shared<1>(tiles, to, x); });
    };
    auto to_c = [&](uint32_t unit, int e, const V &v) {
        char *const c = reinterpret_cast<char *>(C);
        put(unit, e, v, [&](uint32_t to, const V &x) { store_vec_streaming<W>(x, c + to); },
            [&](uint32_t to, float x) { __builtin_nontemporal_store(x, reinterpret_cast<float *>(c + to)); });
    };
    // (a fence behind a few stores, or the addresses of all of them take registers first)
    if (!cut) {               // a second launch reads them; columns that two lanes hold get the same bits twice
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if (own(e)) store_vec_streaming<W>(mine[e], reinterpret_cast<char *>(partials) + at(piece - 1u, e));
            if (W > 1 || e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        to_tile(piece - 1u, e, mine[e]);
        if (W > 1 || e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    const uint4 of = cut->of_piece[piece - 1u];
    uint32_t *const counters = cut->counters + slab;
    const uint32_t slabs = uint32_t(cut->slabs);
    const uint32_t first = __builtin_amdgcn_readfirstlane(of.x), pieces = __builtin_amdgcn_readfirstlane(of.y),
                   counter = __builtin_amdgcn_readfirstlane(of.z), unit = __builtin_amdgcn_readfirstlane(of.w);
    const uint32_t eights = (pieces + kPiecesAtOnce - 1u) / kPiecesAtOnce, eight = (piece - 1u - first) / kPiecesAtOnce,
                   tile0 = first + eight * kPiecesAtOnce, members = min(kPiecesAtOnce, pieces - eight * kPiecesAtOnce);
    // (one loop for every E, a few words of a lane a turn: the tile is not held in registers again)
    constexpr int kTurn = W == 4 ? 1 : W == 1 && E == 4 ? 4 : 2;
    static_assert(E % kTurn == 0, "whole turns");
    // the turn's vectors of n tiles, `apart` bytes from one to the next, added up: all are on their way before the first is added
    auto add_all = [&](int e0, V (&sum)[kTurn], bool none_so_far, uint32_t n, uint32_t tile, uint32_t apart) {
        V v[kTurn][kPiecesAtOnce];
        uint32_t further = 0;          // (behind the last the same again)
#pragma unroll
        for (uint32_t k = 0; k < kPiecesAtOnce; ++k) {
#pragma unroll
            for (int e = 0; e < kTurn; ++e) v[e][k] = load_shared<W>(tiles, at(tile, e0 + e), further);
            further += k + 1u < n ? apart : 0u;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < kTurn; ++e) sum[e] = add_pieces(sum[e], none_so_far, n, v[e]);
    };
    const bool by_eights = eights > kEightsOfOne;
    if (by_eights) {
        if (!last_to_arrive(counters + size_t(counter + eight) * slabs, members)) return;
#pragma unroll 1
        for (int e0 = 0; e0 < E; e0 += kTurn) {
            V sum[kTurn];
#pragma unroll
            for (int e = 0; e < kTurn; ++e) sum[e] = V(0.0f);
            add_all(e0, sum, true, members, tile0, pitch);
#pragma unroll
            for (int e = 0; e < kTurn; ++e) to_tile(tile0, e0 + e, sum[e]);
        }
    }
    if (!last_to_arrive(counters + size_t(counter + eights) * slabs, by_eights ? eights : pieces)) return;
    // the sums of the eights, or what they are the sums of
    const uint32_t of_all = by_eights ? eights : pieces, apart = by_eights ? kPiecesAtOnce * pitch : pitch, step = by_eights ? kPiecesAtOnce * kPiecesAtOnce : kPiecesAtOnce;
#pragma unroll 1
    for (int e0 = 0; e0 < E; e0 += kTurn) {
        V sum[kTurn];
#pragma unroll
        for (int e = 0; e < kTurn; ++e) sum[e] = V(0.0f);
        uint32_t tile = first;
#pragma unroll 1
        for (uint32_t base = 0; base < of_all; base += kPiecesAtOnce, tile += step) {
            V part[kTurn];
#pragma unroll
            for (int e = 0; e < kTurn; ++e) part[e] = sum[e];
            add_all(e0, part, !by_eights || base == 0u, min(kPiecesAtOnce, of_all - base), tile, apart);
#pragma unroll
            for (int e = 0; e < kTurn; ++e) sum[e] = by_eights || base == 0u ? part[e] : sum[e] + part[e];
        }
#pragma unroll
        for (int e = 0; e < kTurn; ++e) to_c(unit, e0 + e, sum[e]);
    }
}

template <int VEC, int NG, bool FULL>
__device__ __forceinline__ void brick_store(const BrickItem &it, const f32x4 (&acc)[NG][VEC], float *__restrict__ C,
                                            float *__restrict__ partials, uint32_t N, uint32_t lane)
{
    typedef typename Vec<VEC>::type V;
    float *out_base = it.piece ? partials : C;
    const uint32_t row0 = (it.piece ? it.piece - 1u : it.panel) * 16u + (lane >> 4) * 4u;
#pragma unroll
    for (int ng = 0; ng < NG; ++ng) {
        const uint32_t c = it.col0 + uint32_t(ng) * 16u * VEC;
        if (!FULL && c >= N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            V out;
#pragma unroll
            for (int v = 0; v < VEC; ++v) vec_set<VEC>(out, v, acc[ng][v][r]);
            store_vec_streaming<VEC>(out, out_base + size_t(row0 + r) * N + (FULL ? c : first_column<VEC>(c, N)));
        }
    }
}

// Variant "pipelined": two operand sets per wavefront ping-pong, so a wavefront overlaps its
// own loads with its own MFMAs.  Best when work items are long (many blocks per chunk) and
// few wavefronts fit per SIMD anyway.
template <int VEC, int NG, bool FULL>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup) void hrpb_brick_f32(
    const uint4 *__restrict__ chunks, uint32_t num_chunks, uint32_t groups_per_xcd,
    const uint32_t *__restrict__ hdr, const float *__restrict__ vals, const float *__restrict__ B,
    float *__restrict__ C, float *__restrict__ partials, uint32_t N, uint32_t column_slabs)
{
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const BrickItem it = brick_item<VEC, NG>(chunks, num_chunks, groups_per_xcd, lane, blockIdx.x, blockIdx.y, column_slabs);
    if (!it.valid) return;
    const uint32_t end = it.end, col0 = it.col0;

    f32x4 acc[NG][VEC];
#pragma unroll
    for (int ng = 0; ng < NG; ++ng)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[ng][v] = f32x4(0.0f);

    // Software pipeline, unrolled by two so that the operand sets ping-pong without copies:
    // header lines run two blocks ahead of the MFMAs, operand loads one block ahead.  The
    // steady-state loop is a single basic block (every prefetch in it is in range), so the
    // scheduling barriers really keep each load group ahead of the MFMAs that hide it.
    BlockOperands<VEC, NG> opA, opB;
    BlockHeader hd, hn;
    uint32_t blk = it.start;
    if (blk < end) {
        hd = load_header(hdr, blk, lane);
        if (blk + 1 < end) hn = load_header(hdr, blk + 1, lane);
        load_operands<VEC, NG, FULL>(opA, hd, vals, B, N, col0, lane);
        hd = hn;
    }
    // Inside a stage the next header line is requested before the operand loads: loads
    // return in order, so the later wait for that header then leaves the operand loads in flight.
    while (blk + 4 <= end) {          // opA holds block blk, hd the header of blk+1
        hn = load_header(hdr, blk + 2, lane);
        __builtin_amdgcn_sched_barrier(0);
        load_operands<VEC, NG, FULL>(opB, hd, vals, B, N, col0, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opA, acc, lane);
        __builtin_amdgcn_sched_barrier(0);
        hd = load_header(hdr, blk + 3, lane);
        __builtin_amdgcn_sched_barrier(0);
        load_operands<VEC, NG, FULL>(opA, hn, vals, B, N, col0, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opB, acc, lane);
        __builtin_amdgcn_sched_barrier(0);
        blk += 2;
    }
    const uint32_t rem = end - blk;   // 0 (empty chunk), 1, 2 or 3 blocks left; opA/hd as above
    if (rem == 1) {
        mfma_block<VEC, NG>(opA, acc, lane);
    } else if (rem == 2) {
        load_operands<VEC, NG, FULL>(opB, hd, vals, B, N, col0, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opA, acc, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opB, acc, lane);
    } else if (rem == 3) {
        hn = load_header(hdr, blk + 2, lane);
        __builtin_amdgcn_sched_barrier(0);
        load_operands<VEC, NG, FULL>(opB, hd, vals, B, N, col0, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opA, acc, lane);
        __builtin_amdgcn_sched_barrier(0);
        load_operands<VEC, NG, FULL>(opA, hn, vals, B, N, col0, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opB, acc, lane);
        __builtin_amdgcn_sched_barrier(0);
        mfma_block<VEC, NG>(opA, acc, lane);
    }
    brick_store<VEC, NG, FULL>(it, acc, C, partials, N, lane);
}

// One brick's loads -- the unit of the rolling pipeline below -- written for a SIMD whose
// matrix and vector instructions share one issue stream (on gfx950 an fp32 MFMA of one
// wavefront and the vector ALU work of another do not overlap), so every vector instruction
// saved is time saved:
//   * the A value is fetched already masked: lanes whose bitmap bit is clear read the zero
//     stored behind the values (the bitmap itself, a scalar register pair, is the select mask);
//   * the brick's value offset rides in the addend of the lane-rank count;
//   * both addresses are 32-bit byte offsets from a scalar base (the planner checks that B and
//     the value array are smaller than 4 GiB and that column * row pitch fits 24 x 24 bits).
struct BrickOperands {
    float a;
    f32x4 b;
};

struct LeanHeader {           // like BlockHeader, plus nothing: kept separate so the scalar parts stay scalar
    uint64_t bitmap[4];
    uint32_t voff[4];
    u32x4 cols;
};

__device__ __forceinline__ LeanHeader load_lean_header(const uint32_t *__restrict__ hdr, uint32_t blk, uint32_t lane)
{
    const uint32_t *h = hdr + size_t(blk) * kHdrWords;
    LeanHeader r;
    r.cols = *reinterpret_cast<const u32x4 *>(h + (lane >> 4) * 4u);
    const uint64_t *bm = reinterpret_cast<const uint64_t *>(h + 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) r.bitmap[j] = bm[j];
#pragma unroll
    for (int j = 0; j < 4; ++j) r.voff[j] = h[24 + j];
    return r;
}

// col_offs[ng]: byte offset inside a B row of the lane's VEC columns in column group ng.  When N is not a multiple of
// the slab width, the lanes of the last slab that stand beyond column N, or whose columns would pass it, point at the
// row's last VEC columns instead: they load valid memory, compute values nobody stores, and the loop keeps the one basic
// block per iteration that its pipeline needs -- a branch around those loads cost 29 % (N = 192 against N = 256).
template <int VEC, int NG, bool FULL>
__device__ __forceinline__ void brick_column_offsets(uint32_t (&col_offs)[NG], uint32_t col0, uint32_t N)
{
#pragma unroll
    for (int ng = 0; ng < NG; ++ng) {
        const uint32_t c = col0 + uint32_t(ng) * 16u * VEC;
        col_offs[ng] = (FULL ? c : first_column<VEC>(c, N)) * 4u;
    }
}

template <int VEC, int NG, bool FULL>
__device__ __forceinline__ void load_brick_lean(typename Vec<VEC>::type (&b_out)[NG], float &a_out, int j,
                                                const LeanHeader &hd, const float *__restrict__ vals,
                                                uint32_t zero_index, const float *__restrict__ B, uint32_t row_pitch,
                                                const uint32_t (&col_offs)[NG])
{
    const uint64_t bm = hd.bitmap[j];
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi(uint32_t(bm >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(bm), hd.voff[j]));
    const uint32_t aoff = (__builtin_amdgcn_inverse_ballot_w64(bm) ? rank : zero_index) * 4u;
    a_out = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(vals) + aoff);
    const uint32_t row = __umul24(hd.cols[j], row_pitch);
    if constexpr (FULL) {       // one address, the column groups at constant offsets from it
        const char *brow = reinterpret_cast<const char *>(B) + (row + col_offs[0]);
#pragma unroll
        for (int ng = 0; ng < NG; ++ng) b_out[ng] = load_vec<VEC>(brow + ng * 64 * VEC);
    } else {
#pragma unroll
        for (int ng = 0; ng < NG; ++ng)
            b_out[ng] = load_vec<VEC>(reinterpret_cast<const char *>(B) + (row + col_offs[ng]));
    }
}

template <int VEC, int NG, bool FULL>
__device__ __forceinline__ void brick_store_piece(const BrickItem &it, const f32x4 (&acc)[NG][VEC], float *__restrict__ C,
                                                  float *__restrict__ partials, uint32_t N, const CutPieces *__restrict__ cut)
{
    const uint32_t lane = lane_again(), col0 = it.slab * (16u * VEC * NG) + (lane & 15u) * VEC;
    typename Vec<VEC>::type mine[NG * 4];        // four rows of each column group
#pragma unroll
    for (int e = 0; e < NG * 4; ++e)
#pragma unroll
        for (int v = 0; v < VEC; ++v) vec_set<VEC>(mine[e], v, acc[e / 4][v][e % 4]);
    auto column = [&](int e) { return col0 + uint32_t(e / 4) * 16u * VEC; };
    auto at = [&](uint32_t unit, int e) {
        return __umul24(unit * 16u + (lane >> 4) * 4u + uint32_t(e % 4), N * 4u) + (FULL ? column(e) : first_column<VEC>(column(e), N)) * 4u;
    };
    auto own = [&](int e) -> uint32_t { return FULL ? uint32_t(VEC) : column(e) < N ? min(N - column(e), uint32_t(VEC)) : 0u; };
    store_piece<VEC>(cut, it.piece, it.slab, mine, at, own, 64u * N, !FULL && N % uint32_t(VEC) != 0u, partials, C);
}

// C tile of one item, addressed like the loads: 32-bit byte offsets from a scalar base.
template <int VEC, int NG, bool FULL, bool CUT>
__device__ __forceinline__ void brick_store_lean(const BrickItem &it, const f32x4 (&acc)[NG][VEC], float *__restrict__ C,
                                                 float *__restrict__ partials, uint32_t N, uint32_t lane, const CutPieces *__restrict__ cut)
{
    typedef typename Vec<VEC>::type V;
    if (CUT && it.piece) return brick_store_piece<VEC, NG, FULL>(it, acc, C, partials, N, cut);
    if (CUT) lane = lane_again();
    char *out_base = reinterpret_cast<char *>(C);
    const uint32_t row0 = it.panel * 16u + (lane >> 4) * 4u;
#pragma unroll
    for (int ng = 0; ng < NG; ++ng) {
        const uint32_t c = it.col0 + uint32_t(ng) * 16u * VEC;
        if (!FULL && c >= N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t off = __umul24(row0 + r, N * 4u) + (FULL ? c : first_column<VEC>(c, N)) * 4u;
            V out;
#pragma unroll
            for (int v = 0; v < VEC; ++v) vec_set<VEC>(out, v, acc[ng][v][r]);
            store_vec_streaming<VEC>(out, out_base + off);
        }
    }
}

// Variant "rolling": ONE operand set per wavefront, refilled brick by brick -- as soon as the
// MFMAs of brick j of block i are issued, the loads of brick j of block i+1 go out into the
// same registers.  Loads are therefore always in flight behind the MFMAs, and the register
// budget is small enough that a launch of short panels is resident as a whole.  Padding-only
// bricks skip their MFMAs.  NG = 2 lets one wavefront cover two column groups, which halves the
// header traffic and shares the A-side index arithmetic between them.
template <int VEC, int NG, bool FULL, bool TOGETHER, bool CUT>
__device__ __forceinline__ void brick_rolling_body(uint32_t block_x, uint32_t block_y, const uint4 *__restrict__ chunks,
                                                   uint32_t num_chunks, uint32_t groups_per_xcd,
                                                   const uint32_t *__restrict__ hdr, const float *__restrict__ vals,
                                                   uint32_t zero_index, const float *__restrict__ B, float *__restrict__ C,
                                                   float *__restrict__ partials, uint32_t N, uint32_t column_slabs, const CutPieces *__restrict__ cut)
{
    typedef typename Vec<VEC>::type V;
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const BrickItem it = brick_item<VEC, NG>(chunks, num_chunks, groups_per_xcd, lane, block_x, block_y, column_slabs);
    if (!it.valid) return;
    const uint32_t end = it.end;
    const uint32_t row_pitch = N * 4u;
    uint32_t col_offs[NG];
    brick_column_offsets<VEC, NG, FULL>(col_offs, it.col0, N);

    f32x4 acc[NG][VEC];
#pragma unroll
    for (int ng = 0; ng < NG; ++ng)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[ng][v] = f32x4(0.0f);

    uint32_t blk = it.start;
    if (blk < end) {
        V b[4][NG];
        float a[4];
        uint64_t bitmap[4];
        LeanHeader h1, h2;
        {
            LeanHeader h0 = load_lean_header(hdr, blk, lane);
            h1 = load_lean_header(hdr, min(blk + 1, end - 1), lane);
            // TOGETHER: h1 is asked for before h0's scalars are waited for (the compiler moves it behind them, a round trip later).  Tied to a scalar, and no fence: what
            // comes after keeps its order.  With a fence for it the operand loads mix with what they wait for: rows of odd widths are 4 % faster, 200 x 200 points,
            // N = 101 11.4 -> 10.9 us, but 256 x 256, N = 128 13.6 -> 13.8, finite elements of 232 nodes, N = 512 10.6 -> 11.4, from HBM 396 x 396 points, N = 512
            // 147 -> 154, and in some variants the loop then waits for nearly all loads.
            if constexpr (TOGETHER) asm volatile("" : "+s"(h0.bitmap[0])::"memory");
            // h1's load must be complete before the loop is entered.  The wait in front of its first use in
            // the loop is compiled once for both ways into the loop; were the load still in flight here (the
            // compiler would sink it behind the operand loads below), that wait would allow only two younger
            // loads and would drain the whole operand set on every iteration.  Waiting here costs nothing:
            // the operand addresses below need h0, which was requested together with h1.
            asm volatile("" ::"v"(h1.cols[0]), "v"(h1.cols[1]), "v"(h1.cols[2]), "v"(h1.cols[3]));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                load_brick_lean<VEC, NG, FULL>(b[j], a[j], j, h0, vals, zero_index, B, row_pitch, col_offs);
                bitmap[j] = h0.bitmap[j];
            }
        }
        // One basic block per iteration and a scheduling fence after every group, so the order
        // "MFMAs of brick j, then the loads that refill brick j" survives instruction scheduling.
        // Only the last block of a panel can hold padding-only bricks; it is peeled below.
        for (; blk + 1 < end; ++blk) {       // a/b hold block blk, h1 the header line of blk+1
            h2 = load_lean_header(hdr, min(blk + 2, end - 1), lane);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int ng = 0; ng < NG; ++ng)
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        acc[ng][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], vec_get<VEC>(b[j][ng], v), acc[ng][v], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                load_brick_lean<VEC, NG, FULL>(b[j], a[j], j, h1, vals, zero_index, B, row_pitch, col_offs);
                bitmap[j] = h1.bitmap[j];
                __builtin_amdgcn_sched_barrier(0);
            }
            h1 = h2;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (bitmap[j] == 0) continue;     // wave-uniform: a brick made of padding columns only
#pragma unroll
            for (int ng = 0; ng < NG; ++ng)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    acc[ng][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], vec_get<VEC>(b[j][ng], v), acc[ng][v], 0, 0, 0);
        }
    }
    brick_store_lean<VEC, NG, FULL, CUT>(it, acc, C, partials, N, lane, cut);
}

template <int VEC, int NG, bool FULL, bool COLUMNS, bool TOGETHER, bool CUT>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup, (NG == 1 ? 8 : 4)) void hrpb_brick_f32_rolling(
    const uint4 *__restrict__ chunks, uint32_t num_chunks, uint32_t groups_per_xcd, const uint32_t *__restrict__ hdr,
    const float *__restrict__ vals, uint32_t zero_index, const float *__restrict__ B, float *__restrict__ C,
    float *__restrict__ partials, uint32_t N, uint32_t column_slabs, const CutPieces *__restrict__ cut)
{
    brick_rolling_body<VEC, NG, FULL, TOGETHER, CUT>(blockIdx.x, blockIdx.y, chunks, num_chunks, groups_per_xcd, hdr, vals, zero_index, B, C,
                                      partials, N, COLUMNS ? column_slabs : 0u, cut);
}

// ---------------------------------------------------------------------------------------
// Reduced-precision brick kernel: the same tiles, loads and C layout as the rolling fp32 kernel, but the
// products run on the bf16 matrix pipeline.  Every fp32 operand x is split in registers into two bf16
// numbers, hi = bf16(x) and lo = bf16(x - hi) (round to nearest; x - hi is exact in fp32), and a block
// contributes  A_hi.B_hi + A_lo.B_hi + A_hi.B_lo  -- three v_mfma_f32_16x16x16_bf16 with fp32
// accumulation.  What is dropped (A_lo.B_lo and the rounding of the lo parts) is below 2^-16 of each
// product.  One such instruction spans the 16 active columns of a whole block: k slot 4g+i of lane
// group g is column g of brick i, which is exactly what lane group g of the fp32 kernel fetches for
// brick i -- so the block header, the masked A fetch through the lane-order bitmaps and the B gathers are
// those of the fp32 kernel unchanged, and only the arithmetic between the loads differs.  An fp32 block
// costs 4 bricks x 32 cycles per 16 columns on the matrix pipeline, this one 3 x 16; the split costs
// three vector instructions per B value, which (unlike next to fp32 MFMAs) overlap with bf16 MFMAs.
// ---------------------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// hi and lo parts of four fp32 values as two packed bf16 quadruples
__device__ __forceinline__ void split_bf16x4(float x0, float x1, float x2, float x3, s16x4 &hi, s16x4 &lo)
{
    const uint32_t h01 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x0, x1}, bf16x2));
    const uint32_t h23 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x2, x3}, bf16x2));
    const float r0 = x0 - __uint_as_float(h01 << 16), r1 = x1 - __uint_as_float(h01 & 0xffff0000u);
    const float r2 = x2 - __uint_as_float(h23 << 16), r3 = x3 - __uint_as_float(h23 & 0xffff0000u);
    const uint32_t l01 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){r0, r1}, bf16x2));
    const uint32_t l23 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){r2, r3}, bf16x2));
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    hi = __builtin_bit_cast(s16x4, (u32x2){h01, h23});
    lo = __builtin_bit_cast(s16x4, (u32x2){l01, l23});
}

template <int NG>
struct Bf16Operands {
    s16x4 a_hi, a_lo;
    s16x4 b_hi[NG][4], b_lo[NG][4];
};

template <int NG>
__device__ __forceinline__ void split_block(Bf16Operands<NG> &o, const float (&a)[4], const f32x4 (&b)[4][NG])
{
    split_bf16x4(a[0], a[1], a[2], a[3], o.a_hi, o.a_lo);
#pragma unroll
    for (int ng = 0; ng < NG; ++ng)
#pragma unroll
        for (int v = 0; v < 4; ++v) split_bf16x4(b[0][ng][v], b[1][ng][v], b[2][ng][v], b[3][ng][v], o.b_hi[ng][v], o.b_lo[ng][v]);
}

template <int NG>
__device__ __forceinline__ void mfma_block_bf16x3(const Bf16Operands<NG> &o, f32x4 (&acc)[NG][4])
{
#pragma unroll
    for (int ng = 0; ng < NG; ++ng)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            acc[ng][v] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(o.a_hi, o.b_hi[ng][v], acc[ng][v], 0, 0, 0);
            acc[ng][v] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(o.a_lo, o.b_hi[ng][v], acc[ng][v], 0, 0, 0);
            acc[ng][v] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(o.a_hi, o.b_lo[ng][v], acc[ng][v], 0, 0, 0);
        }
}

template <int NG, bool FULL, bool COLUMNS, bool CUT>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup, (NG == 1 ? 6 : 4)) void hrpb_brick_bf16x3(
    const uint4 *__restrict__ chunks, uint32_t num_chunks, uint32_t groups_per_xcd, const uint32_t *__restrict__ hdr,
    const float *__restrict__ vals, uint32_t zero_index, const float *__restrict__ B, float *__restrict__ C,
    float *__restrict__ partials, uint32_t N, uint32_t column_slabs, const CutPieces *__restrict__ cut)
{
    constexpr int VEC = 4;
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const BrickItem it = brick_item<VEC, NG>(chunks, num_chunks, groups_per_xcd, lane, blockIdx.x, blockIdx.y, COLUMNS ? column_slabs : 0u);
    if (!it.valid) return;
    const uint32_t end = it.end;
    const uint32_t row_pitch = N * 4u;
    uint32_t col_offs[NG];
    brick_column_offsets<VEC, NG, FULL>(col_offs, it.col0, N);

    f32x4 acc[NG][VEC];
#pragma unroll
    for (int ng = 0; ng < NG; ++ng)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[ng][v] = f32x4(0.0f);

    uint32_t blk = it.start;
    if (blk < end) {
        f32x4 b[4][NG];
        float a[4];
        LeanHeader h1;
        {
            LeanHeader h0 = load_lean_header(hdr, blk, lane);
            h1 = load_lean_header(hdr, min(blk + 1, end - 1), lane);
            asm volatile("" : "+s"(h0.bitmap[0])::"memory");                                         // as in the fp32 kernel
            asm volatile("" ::"v"(h1.cols[0]), "v"(h1.cols[1]), "v"(h1.cols[2]), "v"(h1.cols[3]));
#pragma unroll
            for (int j = 0; j < 4; ++j) load_brick_lean<VEC, NG, FULL>(b[j], a[j], j, h0, vals, zero_index, B, row_pitch, col_offs);
        }
        Bf16Operands<NG> o;
        // per block: split what has arrived, ask for the next block into the same registers, multiply
        for (; blk + 1 < end; ++blk) {       // a/b hold block blk, h1 the header line of blk+1
            const LeanHeader h2 = load_lean_header(hdr, min(blk + 2, end - 1), lane);
            __builtin_amdgcn_sched_barrier(0);
            split_block<NG>(o, a, b);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) load_brick_lean<VEC, NG, FULL>(b[j], a[j], j, h1, vals, zero_index, B, row_pitch, col_offs);
            __builtin_amdgcn_sched_barrier(0);
            mfma_block_bf16x3<NG>(o, acc);
            __builtin_amdgcn_sched_barrier(0);
            h1 = h2;
        }
        split_block<NG>(o, a, b);
        mfma_block_bf16x3<NG>(o, acc);
    }
    brick_store_lean<VEC, NG, FULL, CUT>(it, acc, C, partials, N, lane, cut);
}

// ---------------------------------------------------------------------------------------
// Quad kernel: v_mfma_f32_4x4x1_16B_f32 over the quad lists (see cute_quad_lists).
//
// With cbsz = 4 the instruction takes the four A values of lanes 4p..4p+3 (abid = p), and
// multiplies them into all 64 B lanes: D[i][lane] += A[4p+i] * B[lane].  One instruction is
// therefore "one column of one 4-row group times 64 output columns" -- 8 cycles of the SIMD
// instead of the 36 a 16x16x4 tile costs, and a panel only pays for the (row group, column)
// pairs that hold a nonzero.
//
// Lane L owns output column slab*64 + L of all 16 rows: acc[rg][i] is row 4*rg+i.  A group's
// 64 values are one coalesced dword per lane and ARE the A register (lane 4p+i = pair p, row i);
// its 16 columns are wave-uniform (scalar registers); its 16 B operands are one dword per lane
// each, a contiguous 256-byte piece of a B row.  Two operand sets roll: as soon as the MFMA of
// pair p is issued, B operand p of the group after next is requested into the same register.
//
// chunks[i] = {first group, end group, row panel (or 4-row strip), piece} (piece as for the brick kernels); launch: x walks
// the chunks, y the slabs.  STRIPS: one list per 4-row strip (cute_quad_build_strips) instead of four
// lockstep lists per panel; the instruction stream is the same, only the accumulators mean something else.
// Addresses are 32-bit byte offsets from scalar bases; the planner checks the sizes.
// ---------------------------------------------------------------------------------------
template <int P>
__device__ __forceinline__ void quad_mfma(float a, float b, f32x4 (&acc)[4])
{
    acc[P & 3] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc[P & 3], 4, P, 0);
}

// HUB: the column words of the records a hub plan reads may name a slot of the work-group's LDS table of hub
// rows instead of a B row (kHubFlag | slot): that operand then comes out of LDS (see hrpb_quad_hub_f32).
constexpr uint32_t kHubFlag = 0x80000000u;

template <bool HUB>
__device__ __forceinline__ float quad_load_b(const float *__restrict__ B, uint32_t col, uint32_t row_pitch, uint32_t col_off,
                                             const float *hub)
{
    if (HUB && (col & kHubFlag))        // wave-uniform: the column is a scalar
        return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(hub) + ((col & 0x00ffffffu) * (kWaveSize * 4u) + (threadIdx.x & (kWaveSize - 1)) * 4u));
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(B) + (__umul24(col, row_pitch) + col_off));
}

template <bool FULL, bool STRIPS, bool HUB, bool CUT>
__device__ __forceinline__ void quad_chunk(uint32_t chunk, uint32_t block_y, const uint32_t *__restrict__ heads,
                                           const uint32_t *__restrict__ qrecs, const float *__restrict__ qvals, uint32_t zero_index,
                                           const float *__restrict__ B, float *__restrict__ C, float *__restrict__ partials,
                                           uint32_t N, const CutPieces *__restrict__ cut, const float *hub);

template <bool FULL, bool STRIPS, bool CUT>
__device__ __forceinline__ void quad_body(uint32_t block_x, uint32_t block_y, const uint32_t *__restrict__ heads,
                                          uint32_t num_chunks, uint32_t groups_per_xcd, const uint32_t *__restrict__ qrecs,
                                          const float *__restrict__ qvals, uint32_t zero_index,
                                          const float *__restrict__ B, float *__restrict__ C,
                                          float *__restrict__ partials, uint32_t N, uint32_t column_slabs, const CutPieces *__restrict__ cut)
{
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const uint32_t x = xcd_share(block_x, block_y, column_slabs);
    const uint32_t chunk = (x * groups_per_xcd + block_x / kNumXcd) * kWavesPerGroup + wave;
    if (chunk >= num_chunks) return;
    quad_chunk<FULL, STRIPS, false, CUT>(chunk, block_y, heads, qrecs, qvals, zero_index, B, C, partials, N, cut, nullptr);
}

template <bool FULL, bool STRIPS, bool HUB, bool CUT>
__device__ __forceinline__ void quad_chunk(uint32_t chunk, uint32_t block_y, const uint32_t *__restrict__ heads,
                                           const uint32_t *__restrict__ qrecs, const float *__restrict__ qvals, uint32_t zero_index,
                                           const float *__restrict__ B, float *__restrict__ C, float *__restrict__ partials,
                                           uint32_t N, const CutPieces *__restrict__ cut, const float *hub)
{
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    // One entry of kQuadHeadWords per chunk: its descriptor and, behind it, the record of its first group, so
    // that the first B rows can be requested after one scalar fetch instead of two dependent ones.
    const uint32_t *head = heads + size_t(chunk) * kQuadHeadWords;
    uint32_t g = head[0];
    const uint32_t g_end = head[1];
    const uint32_t panel = head[2];
    const uint32_t piece = head[3];
    uint32_t head_rec[kQuadRecordWords];
#pragma unroll
    for (int p = 0; p < kQuadRecordWords; ++p) head_rec[p] = head[4 + p];
    // one wait for the whole entry: the compiler would otherwise sink the later words to their first use
    asm volatile("" ::"s"(head_rec[11]), "s"(head_rec[12]), "s"(head_rec[15]), "s"(head_rec[16]), "s"(head_rec[17]), "s"(head_rec[18]));

    const uint32_t n = block_y * kWaveSize + lane;
    const bool live = FULL || n < N;
    const uint32_t row_pitch = N * 4u;
    const uint32_t col_off = (live ? n : N - 1u) * 4u;      // dead lanes re-read the last column and store nothing

    f32x4 acc[4];
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) acc[rg] = f32x4(0.0f);

    if (g < g_end) {
        // Two operand sets, so every B operand is requested two groups before its MFMA: set 0 holds
        // group g, set 1 group g+1 (or a harmless re-read of the last group when there is none).
        float b0[16], b1[16], a0, a1;
        // records of the groups being requested (scalar registers): 16 columns, the 64-bit occupancy mask of
        // the group's 64 value slots and the position of its first stored value
        uint32_t ca[kQuadRecordWords], cb[kQuadRecordWords];
        const uint32_t last = g_end - 1u;
        auto fetch_cols = [&](uint32_t (&c)[kQuadRecordWords], uint32_t grp) {
            const uint32_t *src = qrecs + size_t(min(grp, last)) * kQuadRecordWords;
#pragma unroll
            for (int p = 0; p < kQuadRecordWords; ++p) c[p] = src[p];
        };
        // only occupied slots are stored: lane L's value sits (number of occupied slots below L) behind the
        // group's first one; an empty slot reads the zero kept behind the last value
        auto fetch_a = [&](const uint32_t (&c)[kQuadRecordWords]) {
            const uint64_t mask = (uint64_t(c[17]) << 32) | c[16];
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(c[17], __builtin_amdgcn_mbcnt_lo(c[16], c[18]));
            const uint32_t off = (__builtin_amdgcn_inverse_ballot_w64(mask) ? rank : zero_index) * 4u;
            return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(qvals) + off);
        };
#pragma unroll
        for (int p = 0; p < kQuadRecordWords; ++p) ca[p] = head_rec[p];
        fetch_cols(cb, g + 1);
        a0 = fetch_a(ca);
        a1 = fetch_a(cb);
#pragma unroll
        for (int p = 0; p < 16; ++p) b0[p] = quad_load_b<HUB>(B, ca[p], row_pitch, col_off, hub);
#pragma unroll
        for (int p = 0; p < 16; ++p) b1[p] = quad_load_b<HUB>(B, cb[p], row_pitch, col_off, hub);
#define CUTE_QUAD_ROLL(P, A, BSET, COLS)                          \
    quad_mfma<P>(A, BSET[P], acc);                                \
    __builtin_amdgcn_sched_barrier(0);                            \
    BSET[P] = quad_load_b<HUB>(B, COLS[P], row_pitch, col_off, hub); \
    __builtin_amdgcn_sched_barrier(0);
#define CUTE_QUAD_ROLL_REST(A, BSET, COLS)                                                                 \
    CUTE_QUAD_ROLL(1, A, BSET, COLS) CUTE_QUAD_ROLL(2, A, BSET, COLS)                                      \
    CUTE_QUAD_ROLL(3, A, BSET, COLS) CUTE_QUAD_ROLL(4, A, BSET, COLS) CUTE_QUAD_ROLL(5, A, BSET, COLS)    \
    CUTE_QUAD_ROLL(6, A, BSET, COLS) CUTE_QUAD_ROLL(7, A, BSET, COLS) CUTE_QUAD_ROLL(8, A, BSET, COLS)    \
    CUTE_QUAD_ROLL(9, A, BSET, COLS) CUTE_QUAD_ROLL(10, A, BSET, COLS) CUTE_QUAD_ROLL(11, A, BSET, COLS)  \
    CUTE_QUAD_ROLL(12, A, BSET, COLS) CUTE_QUAD_ROLL(13, A, BSET, COLS) CUTE_QUAD_ROLL(14, A, BSET, COLS) \
    CUTE_QUAD_ROLL(15, A, BSET, COLS)
#define CUTE_QUAD_MFMA16(A, BSET)                                                                          \
    quad_mfma<0>(A, BSET[0], acc);   quad_mfma<1>(A, BSET[1], acc);   quad_mfma<2>(A, BSET[2], acc);       \
    quad_mfma<3>(A, BSET[3], acc);   quad_mfma<4>(A, BSET[4], acc);   quad_mfma<5>(A, BSET[5], acc);       \
    quad_mfma<6>(A, BSET[6], acc);   quad_mfma<7>(A, BSET[7], acc);   quad_mfma<8>(A, BSET[8], acc);       \
    quad_mfma<9>(A, BSET[9], acc);   quad_mfma<10>(A, BSET[10], acc); quad_mfma<11>(A, BSET[11], acc);     \
    quad_mfma<12>(A, BSET[12], acc); quad_mfma<13>(A, BSET[13], acc); quad_mfma<14>(A, BSET[14], acc);     \
    quad_mfma<15>(A, BSET[15], acc);
        fetch_cols(ca, g + 2);
        while (g + 2 < g_end) {              // groups g, g+1 and g+2 exist
            // group g from set 0; set 0 is refilled with group g+2.  The other column list is
            // asked for right after this one's first use (where it is waited for), so that wait
            // never covers a fetch just issued; it is first used 15 pairs later.
            const float a0n = fetch_a(ca);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_QUAD_ROLL(0, a0, b0, ca)
            fetch_cols(cb, g + 3);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_QUAD_ROLL_REST(a0, b0, ca)
            a0 = a0n;
            // group g+1 from set 1; set 1 is refilled with group g+3 (clamped to the last one)
            const float a1n = fetch_a(cb);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_QUAD_ROLL(0, a1, b1, cb)
            fetch_cols(ca, g + 4);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_QUAD_ROLL_REST(a1, b1, cb)
            a1 = a1n;
            g += 2;
        }
        CUTE_QUAD_MFMA16(a0, b0)
        if (g + 1 < g_end) { CUTE_QUAD_MFMA16(a1, b1) }
#undef CUTE_QUAD_ROLL
#undef CUTE_QUAD_ROLL_REST
#undef CUTE_QUAD_MFMA16
    }
    if (CUT && !HUB && piece) {      // (the partials matrix: rows (piece-1)*16.., same pitch as C)
        constexpr int E = STRIPS ? 4 : 16;
        float mine[E];
        const f32x4 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
        for (int e = 0; e < E; ++e) mine[e] = STRIPS ? sum[e] : acc[e / 4][e % 4];
        const uint32_t column = block_y * kWaveSize + lane_again(), offset = min(column, N - 1u) * 4u;
        auto at = [&](uint32_t unit, int e) { return __umul24(unit * uint32_t(E) + uint32_t(e), N * 4u) + offset; };
        store_piece<1>(cut, piece, block_y, mine, at, [&](int) { return FULL || column < N ? 1u : 0u; }, uint32_t(E) * N * 4u, false, partials, C);
    } else if (live) {
        // (pieces of a hub plan are added up by reduce_partials: store_piece here takes hrpb_quad_hub_f32<true> from 64 to 65 vector registers, and a
        // compute unit then holds one of its work-groups instead of two)
        char *out_base = reinterpret_cast<char *>(HUB && piece ? partials : C);
        const uint32_t unit = HUB && piece ? piece - 1u : panel;
        if (STRIPS) {
            // all 16 pairs of a group belong to one 4-row strip; the four accumulators only break
            // the dependency chain and are summed here
            const f32x4 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            uint32_t off = __umul24(unit * 4u, row_pitch) + n * 4u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                __builtin_nontemporal_store(sum[i], reinterpret_cast<float *>(out_base + off));
                off += row_pitch;
            }
        } else {
            uint32_t off = __umul24(unit * 16u, row_pitch) + n * 4u;
#pragma unroll
            for (int rg = 0; rg < 4; ++rg)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // not read again by this launch: keep it out of the L2
                    __builtin_nontemporal_store(acc[rg][i], reinterpret_cast<float *>(out_base + off));
                    off += row_pitch;
                }
        }
    }
}

template <bool FULL, bool STRIPS, bool COLUMNS, bool CUT>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup, 8) void hrpb_quad_f32(
    const uint32_t *__restrict__ heads, uint32_t num_chunks, uint32_t groups_per_xcd, const uint32_t *__restrict__ qrecs,
    const float *__restrict__ qvals, uint32_t zero_index, const float *__restrict__ B, float *__restrict__ C,
    float *__restrict__ partials, uint32_t N, uint32_t column_slabs, const CutPieces *__restrict__ cut)
{
    quad_body<FULL, STRIPS, CUT>(blockIdx.x, blockIdx.y, heads, num_chunks, groups_per_xcd, qrecs, qvals, zero_index, B, C,
                            partials, N, COLUMNS ? column_slabs : 0u, cut);
}

// ---------------------------------------------------------------------------------------
// The quad kernel on slabs of 32 columns, for products by columns (xcd_share) whose window of B does not fit the L2s in
// slabs of 64: what an XCD has to hold is halved, a 128-byte line of every B row.
//
// With cbsz = 3 the A block that abid names is broadcast inside each half of the wavefront: lanes 0..31 multiply by pair P,
// lanes 32..63 by pair P + 8, so eight instructions do the sixteen pairs of a group for 32 columns and the lists are read
// as they are.  Pairs P and P + 8 belong to the same row group (P & 3); the two halves' sums are added at the end, half a
// wavefront storing rows 0..7 of the panel and the other rows 8..15.  Same rate per element as the 64-column kernel; two
// operand sets of eight loads keep half its bytes in flight (four sets were slower: 85.0 against 80.6 us on 50 000 rows of 7
// random columns, N = 512, where the 64-column kernel takes 90.8).
// ---------------------------------------------------------------------------------------
template <int P>
__device__ __forceinline__ void quad_half_mfma(float a, float b, f32x4 (&acc)[4])
{
    acc[P & 3] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc[P & 3], 3, P, 0);
}

// the sums of rows r (lo) and r' (hi) over both halves: row r in lanes 0..31, row r' in lanes 32..63
__device__ __forceinline__ float add_halves(float lo, float hi)
{
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

template <bool STRIPS, bool CUT>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup, 8) void hrpb_quad_half_f32(
    const uint32_t *__restrict__ heads, uint32_t num_chunks, uint32_t groups_per_xcd, const uint32_t *__restrict__ qrecs,
    const float *__restrict__ qvals, uint32_t zero_index, const float *__restrict__ B, float *__restrict__ C,
    float *__restrict__ partials, uint32_t N, uint32_t column_slabs, const CutPieces *__restrict__ cut)
{
    constexpr uint32_t kHalf = kWaveSize / 2;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    uint32_t slab = blockIdx.y;
    const uint32_t share = xcd_share(blockIdx.x, slab, column_slabs);
    const uint32_t chunk = (share * groups_per_xcd + blockIdx.x / kNumXcd) * kWavesPerGroup + wave;
    if (chunk >= num_chunks) return;
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t *head = heads + size_t(chunk) * kQuadHeadWords;
    uint32_t g = head[0];
    const uint32_t g_end = head[1], panel = head[2], piece = head[3];
    uint32_t ca[kQuadRecordWords], cb[kQuadRecordWords];       // as in quad_chunk
#pragma unroll
    for (int p = 0; p < kQuadRecordWords; ++p) ca[p] = head[4 + p];
    asm volatile("" ::"s"(ca[11]), "s"(ca[12]), "s"(ca[15]), "s"(ca[16]), "s"(ca[17]), "s"(ca[18]));

    const uint32_t n = slab * kHalf + (lane & (kHalf - 1));
    const bool live = n < N;
    const uint32_t row_pitch = N * 4u;
    const uint32_t col_off = (live ? n : N - 1u) * 4u;
    const uint32_t upper = lane >= kHalf ? 0xffffffffu : 0u;

    f32x4 acc[4];
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) acc[rg] = f32x4(0.0f);

    if (g < g_end) {
        float b0[8], b1[8], a0, a1;
        const uint32_t last = g_end - 1u;
        auto fetch_cols = [&](uint32_t (&c)[kQuadRecordWords], uint32_t grp) {
            const uint32_t *src = qrecs + size_t(min(grp, last)) * kQuadRecordWords;
#pragma unroll
            for (int p = 0; p < kQuadRecordWords; ++p) c[p] = src[p];
        };
        auto fetch_a = [&](const uint32_t (&c)[kQuadRecordWords]) {
            const uint64_t mask = (uint64_t(c[17]) << 32) | c[16];
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(c[17], __builtin_amdgcn_mbcnt_lo(c[16], c[18]));
            const uint32_t off = (__builtin_amdgcn_inverse_ballot_w64(mask) ? rank : zero_index) * 4u;
            return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(qvals) + off);
        };
        // the row offsets are products of scalars; the upper half adds the difference of its own (modulo 2^32)
        auto load_b = [&](const uint32_t (&c)[kQuadRecordWords], int p) {
            const uint32_t lo = c[p] * row_pitch, hi = c[p + 8] * row_pitch;
            return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(B) + (((hi - lo) & upper) + lo + col_off));
        };
        fetch_cols(cb, g + 1);
        a0 = fetch_a(ca);
        a1 = fetch_a(cb);
#pragma unroll
        for (int p = 0; p < 8; ++p) b0[p] = load_b(ca, p);
#pragma unroll
        for (int p = 0; p < 8; ++p) b1[p] = load_b(cb, p);
#define CUTE_HALF_ROLL(P, A, BSET, COLS)       \
    quad_half_mfma<P>(A, BSET[P], acc);        \
    __builtin_amdgcn_sched_barrier(0);         \
    BSET[P] = load_b(COLS, P);                 \
    __builtin_amdgcn_sched_barrier(0);
#define CUTE_HALF_ROLL_REST(A, BSET, COLS)                                                             \
    CUTE_HALF_ROLL(1, A, BSET, COLS) CUTE_HALF_ROLL(2, A, BSET, COLS) CUTE_HALF_ROLL(3, A, BSET, COLS) \
    CUTE_HALF_ROLL(4, A, BSET, COLS) CUTE_HALF_ROLL(5, A, BSET, COLS) CUTE_HALF_ROLL(6, A, BSET, COLS) \
    CUTE_HALF_ROLL(7, A, BSET, COLS)
#define CUTE_HALF_MFMA8(A, BSET)                                                                                     \
    quad_half_mfma<0>(A, BSET[0], acc); quad_half_mfma<1>(A, BSET[1], acc); quad_half_mfma<2>(A, BSET[2], acc);      \
    quad_half_mfma<3>(A, BSET[3], acc); quad_half_mfma<4>(A, BSET[4], acc); quad_half_mfma<5>(A, BSET[5], acc);      \
    quad_half_mfma<6>(A, BSET[6], acc); quad_half_mfma<7>(A, BSET[7], acc);
        fetch_cols(ca, g + 2);
        while (g + 2 < g_end) {              // the pipeline of quad_chunk: groups g, g+1 and g+2 exist
            const float a0n = fetch_a(ca);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_HALF_ROLL(0, a0, b0, ca)
            fetch_cols(cb, g + 3);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_HALF_ROLL_REST(a0, b0, ca)
            a0 = a0n;
            const float a1n = fetch_a(cb);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_HALF_ROLL(0, a1, b1, cb)
            fetch_cols(ca, g + 4);
            __builtin_amdgcn_sched_barrier(0);
            CUTE_HALF_ROLL_REST(a1, b1, cb)
            a1 = a1n;
            g += 2;
        }
        CUTE_HALF_MFMA8(a0, b0)
        if (g + 1 < g_end) { CUTE_HALF_MFMA8(a1, b1) }
#undef CUTE_HALF_ROLL
#undef CUTE_HALF_ROLL_REST
#undef CUTE_HALF_MFMA8
    }
    // a lane's rows of the tile: those from first_row on, each the halves' sums of rows e and e + E
    constexpr int E = STRIPS ? 2 : 8;
    const uint32_t first_row = upper & uint32_t(E);
    const f32x4 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    auto row = [&](int e) { return STRIPS ? add_halves(sum[e], sum[(e + 2) % 4]) : add_halves(acc[e / 4][e % 4], acc[(e / 4 + 2) % 4][e % 4]); };
    if (CUT && piece) {
        float mine[E];
#pragma unroll
        for (int e = 0; e < E; ++e) mine[e] = row(e);
        auto at = [&](uint32_t unit, int e) { return __umul24(unit * uint32_t(2 * E) + first_row + uint32_t(e), row_pitch) + col_off; };
        store_piece<1>(cut, piece, slab, mine, at, [&](int) { return live ? 1u : 0u; }, uint32_t(2 * E) * row_pitch, false, partials, C);
        return;
    }
    uint32_t off = __umul24(panel * uint32_t(2 * E) + first_row, row_pitch) + n * 4u;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const float v = row(e);
        if (live) __builtin_nontemporal_store(v, reinterpret_cast<float *>(reinterpret_cast<char *>(C) + off));
        off += row_pitch;
    }
}

// ---------------------------------------------------------------------------------------
// The quad kernel with the most referenced B rows staged in LDS (the reference stages the B rows of a block in
// shared memory for the warps of its thread block, kernel.cu:123-124,143-164; here what is staged is what many
// work items share: the rows of hub columns).  A work-group of sixteen wavefronts copies, once, the 64-column
// pieces of `num_hub` hub rows of its slab into LDS (num_hub * 256 bytes) and then stays: its wavefronts walk the
// chunk list with a stride of the whole launch, so the table is filled once per work-group, not once per chunk.
// A column word of the plan's records that carries kHubFlag names a slot of that table, and the operand is an
// LDS read instead of a gather through the vector memory path.  Strip lists only (graphs with hub vertices).
// ---------------------------------------------------------------------------------------
constexpr int kHubWaves = 16;

template <bool FULL>
__global__ __launch_bounds__(kWaveSize *kHubWaves) void hrpb_quad_hub_f32(
    const uint32_t *__restrict__ heads, uint32_t num_chunks, const uint32_t *__restrict__ qrecs, const float *__restrict__ qvals,
    uint32_t zero_index, const uint32_t *__restrict__ hub_rows, uint32_t num_hub, const float *__restrict__ B,
    float *__restrict__ C, float *__restrict__ partials, uint32_t N)
{
    extern __shared__ float hub[];
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const uint32_t n = blockIdx.y * kWaveSize + lane;
    for (uint32_t h = wave; h < num_hub; h += kHubWaves)
        hub[h * kWaveSize + lane] = (FULL || n < N) ? B[size_t(hub_rows[h]) * N + n] : 0.0f;
    __syncthreads();
    // consecutive chunks of the list (longest first) go to different work-groups
    const uint32_t stride = gridDim.x * kHubWaves;
    for (uint32_t chunk = wave * gridDim.x + blockIdx.x; chunk < num_chunks; chunk += stride)
        quad_chunk<FULL, true, true, true>(chunk, blockIdx.y, heads, qrecs, qvals, zero_index, B, C, partials, N, nullptr, hub);
}

// ---------------------------------------------------------------------------------------
// Blocked-ELL SpMM (the format of inc/prepareBlkEll.hpp): dense blockSize x blockSize blocks,
// ellColIdx[height x width] block-column ids (ascending, -1 padded), ellValues row-major
// [height*blockSize x width*blockSize].  One wavefront per (16-row strip, slab of 16*VEC columns).
// A 16x16 tile of A is one 16-byte load per lane: lane (row = L%16, q = L/16) holds
// A[row][4q..4q+3].  MFMA number e of the tile takes element e of that vector, i.e. k index
// 4q+e from lane group q -- so lane group q fetches B rows 4q+e, e = 0..3, itself, and no
// cross-lane move is needed.  Accumulator layout and the column interleave that gives every
// lane VEC consecutive C columns are those of the brick kernel.
// ACCUMULATE: C += A.B (for the heavy part of a split matrix), else C = A.B.
// ---------------------------------------------------------------------------------------
constexpr int kEllDepth = 3;

template <int VEC, bool FULL, bool ACCUMULATE>
__global__ __launch_bounds__(256) void blocked_ell_f32(const int32_t *__restrict__ ell_col, const float *__restrict__ ell_val,
                                                       uint32_t block_size, uint32_t width, uint32_t num_strips,
                                                       uint32_t num_rows, const float *__restrict__ B, float *__restrict__ C,
                                                       uint32_t N)
{
    typedef typename Vec<VEC>::type V;
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    // neighbouring strips reference neighbouring block columns: keep them on one XCD, whose L2 then holds
    // their B rows (gridDim.x is a multiple of the XCD count)
    const uint32_t strip = xcd_contiguous_id(blockIdx.x, gridDim.x / kNumXcd) * (blockDim.x / kWaveSize) +
                           __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    if (strip >= num_strips) return;
    const uint32_t row16 = lane & 15u, q = lane >> 4;
    const uint32_t c0 = blockIdx.y * (16u * VEC) + row16 * VEC;       // this lane's VEC columns of the slab
    const bool col_live = FULL || c0 < N;
    const uint32_t block_row = (strip * 16u) / block_size;
    const uint32_t tiles_per_block = block_size / 16u;                // 16-wide k tiles of one block
    const size_t pitch = size_t(width) * block_size;
    const float *a_row = ell_val + size_t(strip * 16u + row16) * pitch + q * 4u;
    const int32_t *cols = ell_col + size_t(block_row) * width;
    const float *b_base = B + size_t(q * 4u) * N + (col_live ? c0 : 0u);

    f32x4 acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = f32x4(0.0f);

    struct Operands {
        f32x4 a;
        V b[4];
        bool past;                    // wave-uniform: the set holds a re-read of the last tile and must not count
    };
    // Block ids are taken 64 at a time into one vector register (lane i holds block w0 + i);
    // the padding (-1) that follows the last block ends the row.  Inside such a batch the k
    // tiles roll through kEllDepth operand sets: a set is refilled with tile t+kEllDepth right
    // after the MFMAs of tile t, and the id of a tile's block comes out of the register by readlane, so no load
    // depends on another load.
    for (uint32_t w0 = 0; w0 < width; w0 += kWaveSize) {
        const uint32_t in_batch = min(width - w0, uint32_t(kWaveSize));
        const int32_t ids = lane < in_batch ? cols[w0 + lane] : -1;
        const uint64_t pad = __ballot(ids < 0);
        const uint32_t valid = pad ? uint32_t(__builtin_ctzll(pad)) : uint32_t(kWaveSize);
        const uint32_t tiles = valid * tiles_per_block;
        if (tiles == 0) break;
        auto fetch = [&](uint32_t t, Operands &o) {
            o.past = t >= tiles;                                      // past the end: re-read the last tile
            t = min(t, tiles - 1u);
            const uint32_t w = t / tiles_per_block, kt = (t % tiles_per_block) * 16u;
            const uint32_t bc = uint32_t(__builtin_amdgcn_readlane(ids, w));
            o.a = *reinterpret_cast<const f32x4 *>(a_row + size_t(w0 + w) * block_size + kt);
            const float *b_row = b_base + size_t(bc * block_size + kt) * N;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.b[e] = *reinterpret_cast<const V *>(b_row + size_t(e) * N);
        };
        auto multiply = [&](const Operands &o) {
            const f32x4 a = o.past ? f32x4(0.0f) : o.a;               // masked here, where the data is waited for anyway
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    acc[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], vec_get<VEC>(o.b[e], v), acc[v], 0, 0, 0);
        };
        Operands o[kEllDepth];
#pragma unroll
        for (int k = 0; k < kEllDepth; ++k) fetch(uint32_t(k), o[k]);
        __builtin_amdgcn_sched_barrier(0);
        for (uint32_t t = 0; t < tiles; t += kEllDepth) {
#pragma unroll
            for (int k = 0; k < kEllDepth; ++k) {
                // the fences keep the compiler from sinking the loads to their first use
                multiply(o[k]);
                __builtin_amdgcn_sched_barrier(0);
                fetch(t + uint32_t(k) + kEllDepth, o[k]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (valid < in_batch) break;
    }
    if (!col_live) return;
    const uint32_t r0 = strip * 16u + q * 4u;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (r0 + r >= num_rows) break;
        V *dst = reinterpret_cast<V *>(C + size_t(r0 + r) * N + c0);
        V out;
#pragma unroll
        for (int v = 0; v < VEC; ++v) vec_set<VEC>(out, v, acc[v][r]);
        if (ACCUMULATE) out += *dst;
        *dst = out;
    }
}

// Adds up the partial tiles of the panels (16 rows) or strips (4 rows) that were cut into several chunks, for calls whose pieces do
// not do it themselves: fixups[i] = {panel or strip, first piece, number of pieces, -}; piece k is rows [k*rows, (k+1)*rows) of the
// partials matrix, whose row pitch is N like C's.  A block of sixteen wavefronts works on tile i in segments
// of 64 elements.  With up to eight pieces every wavefront takes a segment of its own; with more, G = 2..16 wavefronts share a
// segment, each an eight of the pieces, and the sums are added in order: store_piece's order, hence its bits.
// The launch has one block per (tile, segment); blocks past the last segment group exit.
constexpr int kReduceWaves = 16;
constexpr __host__ __device__ uint32_t reduce_waves(uint32_t pieces) { return pieces <= 8u ? 1u : pieces <= 16u ? 2u : pieces <= 32u ? 4u : pieces <= 64u ? 8u : 16u; }

__global__ __launch_bounds__(kWaveSize *kReduceWaves) void reduce_partials(const uint4 *__restrict__ fixups, uint32_t count,
                                                                           uint32_t rows, const float *__restrict__ partials,
                                                                           float *__restrict__ C, uint32_t N)
{
    __shared__ float sums[kReduceWaves][kWaveSize];
    const uint32_t lane = threadIdx.x & (kWaveSize - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    if (blockIdx.x >= count) return;
    const uint4 fx = fixups[blockIdx.x];
    const uint32_t pieces = __builtin_amdgcn_readfirstlane(fx.z), eights = (pieces + kPiecesAtOnce - 1u) / kPiecesAtOnce;
    const uint32_t G = reduce_waves(pieces);
    const uint32_t segs_per_block = kReduceWaves / G;
    const uint32_t tile = rows * N;
    if (blockIdx.y * segs_per_block * kWaveSize >= tile) return;      // whole block: nothing left of this tile
    const uint32_t seg = blockIdx.y * segs_per_block + wave / G, g = wave % G;
    const uint32_t e = seg * kWaveSize + lane;
    const bool valid = e < tile;
    const float *src = partials + size_t(fx.y) * tile + (valid ? e : 0u);
    float total = 0.0f;
    auto sum_of = [&](uint32_t piece0) {
        const uint32_t n = min(kPiecesAtOnce, pieces - piece0);
        float v[kPiecesAtOnce];
#pragma unroll
        for (uint32_t k = 0; k < kPiecesAtOnce; ++k) v[k] = src[size_t(piece0 + min(k, n - 1u)) * tile];
        return add_pieces(0.0f, true, n, v);
    };
    for (uint32_t base = 0; base < eights; base += G) {               // (a block works on one unit: the rounds are the same for all of it)
        const uint32_t eight = base + g, piece0 = eight * kPiecesAtOnce;
        float sum = 0.0f;
        if (eight < eights) sum = sum_of(piece0);
        if (G == 1u) { total = sum; break; }
        sums[wave][lane] = sum;
        __syncthreads();
        if (g == 0u)
            for (uint32_t w = 0; w < min(G, eights - base); ++w) total = base + w == 0u ? sums[wave][lane] : total + sums[wave + w][lane];
        __syncthreads();
    }
    if (valid && g == 0u) __builtin_nontemporal_store(total, C + size_t(fx.x) * tile + e);
}

// One group of L = 1<<LOG_L lanes per row; lane t of the group owns VEC consecutive columns
// starting at slab*L*VEC + t*VEC.  Nonzeros are fetched L at a time, one per lane, then
// broadcast one after the other, so each C element accumulates its row in storage order.
// row_list == nullptr: rows 0..num_rows-1.
template <int VEC, int LOG_L>
__global__ __launch_bounds__(256) void csr_rows(const uint32_t *__restrict__ row_list, uint32_t num_rows,
                                                uint32_t num_slabs, const uint32_t *__restrict__ rowPtr,
                                                const uint32_t *__restrict__ cols, const float *__restrict__ vals,
                                                const float *__restrict__ B, float *__restrict__ C, uint32_t N)
{
    typedef typename Vec<VEC>::type V;
    constexpr uint32_t L = 1u << LOG_L;
    const uint32_t t = threadIdx.x & (L - 1);
    const uint64_t gid = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> LOG_L;
    // whole groups leave together, so shuffles below never read a retired lane of the same group
    if (gid >= uint64_t(num_rows) * num_slabs) return;
    const uint32_t ridx = uint32_t(gid / num_slabs);
    const uint32_t slab = uint32_t(gid % num_slabs);
    const uint32_t row = row_list ? row_list[ridx] : ridx;
    const bool live = slab * L * VEC + t * VEC < N;
    const uint32_t c0 = first_column<VEC>(slab * L * VEC + t * VEC, N);
    const uint32_t s = rowPtr[row], e = rowPtr[row + 1];
    V acc = V(0.0f);
    for (uint32_t base = s; base < e; base += L) {
        const uint32_t mine = base + t;
        uint32_t my_col = 0;
        float my_val = 0.0f;
        if (mine < e) { my_col = cols[mine]; my_val = vals[mine]; }
        const uint32_t cnt = min(L, e - base);
        for (uint32_t q = 0; q < cnt; ++q) {
            const uint32_t c = __shfl(my_col, int(q), int(L));
            const float a = __shfl(my_val, int(q), int(L));
            if (live) {
                const V b = load_vec<VEC>(B + size_t(c) * N + c0);
                acc += a * b;
            }
        }
    }
    if (live) *reinterpret_cast<typename VecInMemory<VEC>::type *>(C + size_t(row) * N + c0) = acc;
}

// The sparse-panel kernel of the library: same work split as csr_rows, but the nonzeros of a
// row are consumed in batches whose B-row loads are all issued before the first FMA, so a
// row costs about one memory round trip per batch instead of one per nonzero.  Each C
// element still accumulates its row in storage order.
// AHEAD: the entries of the next round are asked for ahead of this round's B rows (loads return in order), so a row longer than
// a round waits for one round trip per round, not for two (131 072 rows of 20, N = 64: 93.2 -> 89.4 us).  The fused kernels
// leave that out where the entries take several registers: their 64 would not do (nor would they for entries that are held
// from one round to the next in any other way: a register spilled to scratch in four of them).  They also leave it out for
// sixteen lanes a row in row order, where most rows are one round and the lists fill the launch: R-MAT graph of 131 072 nodes,
// N = 64: 45.5 us with it, 45.0 without; by columns, N = 128: 95.8 and 96.4.
template <int VEC, int LOG_L, int BATCH, bool AHEAD>
__device__ __forceinline__ void rows_batched_body(uint32_t block_id, uint32_t slab, const uint4 *__restrict__ row_list,
                                                  uint32_t num_rows, const uint32_t *__restrict__ rowPtr,
                                                  const uint32_t *__restrict__ cols, const float *__restrict__ vals,
                                                  const float *__restrict__ B, float *__restrict__ C, uint32_t N)
{
    typedef typename Vec<VEC>::type V;
    constexpr uint32_t L = 1u << LOG_L;
    constexpr uint32_t STEP = BATCH;
    constexpr uint32_t PER = uint32_t(BATCH) > L ? uint32_t(BATCH) / L : 1u;      // entries a lane holds of a round
    constexpr uint32_t ROUND = L * PER;
    const uint32_t t = threadIdx.x & (L - 1);
    const uint64_t gid = (uint64_t(block_id) * blockDim.x + threadIdx.x) >> LOG_L;
    if (gid >= num_rows) return;
    const uint32_t ridx = uint32_t(gid);
    // a listed row comes with its row pointers {row, first entry, end, -}: one fetch, where the row index in one array
    // and the row pointers in another would be two, the second waiting for the first
    uint32_t row, s, e;
    if (row_list) {
        const uint4 entry = row_list[ridx];
        row = entry.x; s = entry.y; e = entry.z;
    } else {
        row = ridx; s = rowPtr[row]; e = rowPtr[row + 1];
    }
    const bool live = slab * L * VEC + t * VEC < N;
    const uint32_t c0 = first_column<VEC>(slab * L * VEC + t * VEC, N);
    const float *bcol = B + c0;
    V acc = V(0.0f);
    // A lane group narrower than a batch takes a whole batch a round all the same, a few consecutive entries in each lane
    // (what it reads past the row's end is the next row's or the padding behind the arrays, and is not used): one entry per
    // lane and round, N = 4 walked a row of 30 entries in 30 round trips.  Bands of 400 000 rows of 30 entries, N = 4:
    // 365 -> 47 us, N = 1: 351 -> 44.
    struct Entries {
        uint32_t col[PER];
        float val[PER];
    };
    auto fetch = [&](uint32_t first, Entries &m) {
        if constexpr (PER == 1) {
            m.col[0] = 0;
            m.val[0] = 0.0f;
            if (first + t < e) { m.col[0] = cols[first + t]; m.val[0] = vals[first + t]; }
        } else if (first < e) {
            __builtin_memcpy(m.col, cols + first + t * PER, sizeof m.col);
            __builtin_memcpy(m.val, vals + first + t * PER, sizeof m.val);
        }
    };
    Entries mine, next;
    if (AHEAD) fetch(s, mine);
    for (uint32_t base = s; base < e; base += ROUND) {
        if (AHEAD) fetch(base + ROUND, next);
        else fetch(base, mine);
        const uint32_t cnt = min(ROUND, e - base);
        for (uint32_t q0 = 0; q0 < cnt; q0 += STEP) {
            V b[STEP];
            float a[STEP];
#pragma unroll
            for (uint32_t u = 0; u < STEP; ++u) {
                // slots past the end of the row are skipped
                const bool taken = q0 + u < cnt;
                const uint32_t c = __shfl(mine.col[u % PER], int((q0 + u) / PER), int(L));
                a[u] = __shfl(mine.val[u % PER], int((q0 + u) / PER), int(L));
                if (PER > 1) a[u] = taken ? a[u] : 0.0f;
                b[u] = V(0.0f);
                if (live && taken) b[u] = load_vec<VEC>(bcol + size_t(c) * N);
            }
#pragma unroll
            for (uint32_t u = 0; u < STEP; ++u) acc += a[u] * b[u];
        }
        if (AHEAD) mine = next;
    }
    // (narrow groups work it out again: kept through the loop it took the register of the row's number in one of the fused kernels, which went to scratch)
    const uint32_t column = slab * L * VEC + (AHEAD ? t : lane_again() & (L - 1)) * VEC;
    if (AHEAD ? live : column < N) store_vec_streaming<VEC>(acc, C + size_t(row) * N + first_column<VEC>(column, N));
}

template <int VEC, int LOG_L, int BATCH, bool COLUMNS>
__global__ __launch_bounds__(256) void csr_rows_batched(const uint4 *__restrict__ row_list, uint32_t num_rows,
                                                        const uint32_t *__restrict__ rowPtr,
                                                        const uint32_t *__restrict__ cols,
                                                        const float *__restrict__ vals, const float *__restrict__ B,
                                                        float *__restrict__ C, uint32_t N, XcdRanges ranges, uint32_t column_slabs)
{
    // each XCD walks one contiguous range of rows (ranges of equal work), so the B rows that neighbouring
    // rows share stay in that XCD's L2.  A product wider than one lane group's slab (2^LOG_L * VEC columns) is
    // walked slab by slab, each over all rows (y is the slower index of the order in which work-groups start):
    // what the resident rows read of B at one time is then one slab wide, whatever N is.
    uint32_t block_id, slab = blockIdx.y;
    const uint32_t x = xcd_share(blockIdx.x, slab, COLUMNS ? column_slabs : 0u);
    if (!xcd_range_id(ranges, blockIdx.x, x, block_id)) return;
    rows_batched_body<VEC, LOG_L, BATCH, true>(block_id, slab, row_list, num_rows, rowPtr, cols, vals, B, C, N);
}

// Rows of products of a few columns: 2^log_parts lane groups share a row's entries, each group 2^log_lanes lanes of VEC columns, and add their
// sums up by exchanges.  With one group a row, as csr_rows_batched has it, a lane walks its row alone, and the chain of round trips is
// what such a product takes: finite elements, 12 000 rows of 60, N = 1 12.9 us in the brick kernel, 3.6 with sixteen groups a row.
template <int VEC>
__global__ __launch_bounds__(256) void csr_rows_split(const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols, const float *__restrict__ vals,
                                                      const float *__restrict__ B, float *__restrict__ C, uint32_t M, uint32_t N, uint32_t log_lanes,
                                                      uint32_t log_parts, uint32_t blocks_per_xcd)
{
    constexpr uint32_t kTurn = 4;                             // entries a lane has on their way
    const uint64_t at = uint64_t(xcd_contiguous_id(blockIdx.x, blocks_per_xcd)) * 256u + threadIdx.x;
    const uint32_t log_row = log_lanes + log_parts, in_row = uint32_t(at) & ((1u << log_row) - 1u);
    if (at >> log_row >= M) return;
    const uint32_t row = uint32_t(at >> log_row), part = in_row >> log_lanes, parts = 1u << log_parts;
    const uint32_t c = min((in_row & ((1u << log_lanes) - 1u)) * VEC, N - uint32_t(VEC));       // the last lanes may share columns: the same bits
    const uint32_t end = rowPtr[row + 1u];
    float acc[VEC] = {};
    for (uint64_t i0 = uint64_t(rowPtr[row]) + part; i0 < end; i0 += kTurn * parts) {
        uint32_t col[kTurn];
        float val[kTurn];
        typename Vec<VEC>::type b[kTurn];
#pragma unroll
        for (uint32_t k = 0; k < kTurn; ++k) {
            const uint64_t i = min(i0 + k * parts, uint64_t(end) - 1u);
            col[k] = cols[i];
            val[k] = vals[i];
        }
#pragma unroll
        for (uint32_t k = 0; k < kTurn; ++k) b[k] = load_vec<VEC>(B + size_t(col[k]) * N + c);
#pragma unroll
        for (uint32_t k = 0; k < kTurn; ++k)
            if (i0 + k * parts < end) {                       // (left out, not multiplied by zero: B may hold what is not finite)
                const float *x = reinterpret_cast<const float *>(&b[k]);
#pragma unroll
                for (int j = 0; j < VEC; ++j) acc[j] += val[k] * x[j];
            }
    }
    for (uint32_t apart = 1u << log_lanes; apart < 1u << log_row; apart <<= 1)
#pragma unroll
        for (int j = 0; j < VEC; ++j) acc[j] += __shfl_xor(acc[j], int(apart));
    if (part == 0u) {
        typename Vec<VEC>::type out;
        float *x = reinterpret_cast<float *>(&out);
#pragma unroll
        for (int j = 0; j < VEC; ++j) x[j] = acc[j];
        store_vec_streaming<VEC>(out, C + size_t(row) * N + c);
    }
}

// Rows whose columns lie in a window that moves along with them (banded matrices, operators in a local numbering): the piece of B
// they read is kept in LDS, W columns of it for one work-group, as a ring that slides over B, and the gathers are LDS reads.
// csr_rows_batched gathers through the vector memory path, which returns about 40 bytes a clock and CU (20 TB/s in all) whatever
// level of the caches answers; LDS returns 128.  A chain is a run of tiles of kWindowTile rows that one work-group of sixteen
// wavefronts walks, a row a lane, all W columns of it; every row of B enters the ring once a chain.
//
// What bounds it: a CU has about 64 lines on their way from the L2 (measured: 59 to 74), and a tile asks for one 128-byte line
// a row of B (of which W floats are used) and for 6 bytes an entry, once for each slab of W columns.  So W is as wide as the
// window allows, 8 or 16, an entry is a ring slot of 16 bits beside its value, four entries of a row are fetched at once, and the
// slabs of a chain run on one XCD at the same time: they ask its L2 for the same entries and lines and fill the same lines of C.
// Then LDS: 16 bytes a lane, rows at random, so the pieces of a row are read in an order that depends on the lane (the low bits
// of the address all differ across Q lanes), and the entries of a row stand in the order of (slot + row / 2) mod 8, which lets
// neighbouring lanes ask for different banks (LDS cycles 98 600 -> 74 900 a CU, 65 536 rows of 32, N = 256: 60.4 -> 56.7 us).
// Row kernel / this one, us: 1 048 576 rows of 32 entries, band of 2 048 on either side, N = 256 1 720 / 1 007 (34 TB/s of gathers; the
// operands take 440 at a copy's rate), 262 144 rows 414 / 258, N = 47 and 30 entries 87 / 51; band of 700 (16 columns) 414 / 211.
// At the first of these 52 % of the time are LDS cycles, 44 % vector instructions, and 59 lines are on their way on average.
// Tried and slower: B asked for a whole tile ahead (258 -> 276), wavefronts of their own for it (258 -> 292 and more, fewer of
// them add up), non-temporal loads or stores (+ 10 ... 25 %: the sharing goes).
constexpr uint32_t kWindowTile = 1024, kWindowBytes = 160u << 10, kWindowPad = 0xffffu;
template <int W> constexpr uint32_t kWindowRows = kWindowBytes / (W * 4u);     // rows of B in the ring

// x of lane (l ^ XOR) of each four lanes
template <int XOR> __device__ __forceinline__ f32x4 quad_xor(const f32x4 &v)
{
    constexpr int perm = (0 ^ XOR) | (1 ^ XOR) << 2 | (2 ^ XOR) << 4 | (3 ^ XOR) << 6;
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = v[i];
        r[i] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), perm, 0xf, 0xf, true));
    }
    return r;
}

// slices[i], 64 rows: {first quad, quads without padding, quads, -}; a quad is four entries of each of the 64 rows, slot and value
// lane after lane.  tiles[t]: columns [lo, hi) that the rows of tile t and, by lo, of every later tile, by hi, of every earlier one
// read; hi - lo is at most the ring.  Column c of B stands in slot c mod kWindowRows.
// WARM: operands from HBM.  The lines of B that the tile after next brings are asked for here, each by one of the work-groups that share
// them, so that all of them find it in the L2 (262 144 rows, N = 256: 12 entries a row 245 -> 188 us, 32 entries 257 -> 248; from the
// Infinity Cache, 65 536 rows of 32, 56.6 -> 61.5).
template <int W, bool WARM>
__global__ __launch_bounds__(1024) void csr_rows_window(const uint4 *__restrict__ slices, const uint2 *__restrict__ slots, const f32x4 *__restrict__ vals,
                                                        const uint2 *__restrict__ tiles, uint32_t num_tiles, uint32_t tiles_per_chain,
                                                        uint32_t num_chains, uint32_t num_slabs, const float *__restrict__ B,
                                                        float *__restrict__ C, uint32_t M, uint32_t N)
{
    constexpr uint32_t Q = W / 4, S = kWindowRows<W>, ROW_LOG = W == 8 ? 5 : 6;    // 16-byte pieces, rows of the ring; bytes of a row
    constexpr uint32_t STEP = 1024u / Q, AHEAD = kWindowTile / STEP, FIRST = S / STEP;   // rows of B a round; rounds ahead, of the first window
    constexpr uint32_t HOLD = W == 8 ? 4 : 2;                                      // quads of a row in registers
    static_assert(W == 8 || W == 16, "a slot and its bytes are packed for these");
    __shared__ f32x4 ring[S * Q];
    // the slabs of a chain are neighbours on one XCD
    const uint32_t local = blockIdx.x / kNumXcd, chain = blockIdx.x % kNumXcd + kNumXcd * (local / num_slabs), slab = local % num_slabs;
    const uint32_t t0 = chain * tiles_per_chain, t1 = min(t0 + tiles_per_chain, num_tiles);
    if (chain >= num_chains || t0 >= t1) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize), l = lane % Q;
    const uint32_t c0 = min(slab * W, N - uint32_t(W));       // the last slab may share columns with the one before: the same bits
    const float *Bc = B + c0 + l * 4u;
    const uint32_t r_in = tid / Q;
    auto load_row = [&](uint32_t r) { return load_vec<4>(Bc + size_t(r) * N); };
    auto keep_row = [&](uint32_t r, const f32x4 &v) { ring[(r % S) * Q + l] = v; };
    auto lds_barrier = [] {                                   // (global loads and stores stay under way)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    struct Quad {
        uint2 slot;
        f32x4 val;
    };
    auto fetch = [&](const uint4 &d, uint32_t q) {            // (a slice has a quad at least)
        const size_t at = (size_t(d.x) + min(q, d.z - 1u)) * kWaveSize + lane;
        Quad m;
        m.slot = slots[at];
        m.val = vals[at];
        return m;
    };
    const uint32_t num_slices = (M + 63u) / 64u;
    auto slice_of = [&](uint32_t t) { return slices[min(t * (kWindowTile / 64u) + wave, num_slices - 1u)]; };
    uint4 d = slice_of(t0);
    Quad held[HOLD];
    uint32_t have = tiles[t0].x;
    {
        f32x4 first[FIRST];
        const uint32_t hi = tiles[t0].y;
#pragma unroll
        for (uint32_t i = 0; i < FIRST; ++i)
            if (have + i * STEP + r_in < hi) first[i] = load_row(have + i * STEP + r_in);
#pragma unroll
        for (uint32_t j = 0; j < HOLD; ++j) held[j] = fetch(d, j);
#pragma unroll
        for (uint32_t i = 0; i < FIRST; ++i)
            if (have + i * STEP + r_in < hi) keep_row(have + i * STEP + r_in, first[i]);
        have = hi;
    }
    lds_barrier();
    const char *lds = reinterpret_cast<const char *>(ring);
    // piece j of the lane is piece j ^ l of the row, a lane's pieces differ from its neighbours' in every read
    auto read = [&](uint32_t slot, f32x4 (&b)[Q]) {
        const uint32_t at = slot << ROW_LOG | l << 4;
#pragma unroll
        for (uint32_t j = 0; j < Q; ++j) b[j] = *reinterpret_cast<const f32x4 *>(lds + (at ^ (j * 16u)));
    };
    auto add_quad = [&](const Quad &m, f32x4 (&acc)[Q]) {
        const uint32_t slot[4] = {m.slot.x & 0xffffu, m.slot.x >> 16, m.slot.y & 0xffffu, m.slot.y >> 16};
        constexpr int G = 16 / (2 * int(Q));                  // entries whose pieces are on their way together: the registers' share
#pragma unroll
        for (int g = 0; g < 4; g += G) {
            f32x4 b[G][Q];
#pragma unroll
            for (int u = 0; u < G; ++u) read(slot[g + u], b[u]);
#pragma unroll
            for (int u = 0; u < G; ++u)
#pragma unroll
                for (uint32_t j = 0; j < Q; ++j) acc[j] += m.val[g + u] * b[u][j];
            if (G < 4) __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto add_padded = [&](const Quad &m, f32x4 (&acc)[Q]) {   // padding is left out, not multiplied by zero: B may hold what is not finite
        const uint32_t slot[4] = {m.slot.x & 0xffffu, m.slot.x >> 16, m.slot.y & 0xffffu, m.slot.y >> 16};
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (slot[u] != kWindowPad) {
                f32x4 b[Q];
                read(slot[u], b);
#pragma unroll
                for (uint32_t j = 0; j < Q; ++j) acc[j] += m.val[u] * b[j];
            }
    };
    const uint32_t lines = WARM ? (N * 4u + 127u) / 128u : 1u;
    float warm = 0.0f;
    for (uint32_t t = t0; t < t1; ++t) {
        // (what lies between two windows is left out)
        const uint2 coming = t + 1u < t1 ? tiles[t + 1u] : make_uint2(have, have);
        const uint32_t from = max(have, coming.x), next = coming.y;
        const uint4 dn = slice_of(min(t + 1u, t1 - 1u));
        f32x4 acc[Q];
#pragma unroll
        for (uint32_t j = 0; j < Q; ++j) acc[j] = f32x4(0.0f);
        // loads return in order: what is asked for behind the rows of B waits for them, so those come last in a tile, before the
        // next tile's first entries, and are covered by the HOLD quads at hand
        uint32_t q = 0;
        for (; q + HOLD < d.z && q + HOLD <= d.y; q += HOLD) {
#pragma unroll
            for (uint32_t j = 0; j < HOLD; ++j) {
                const Quad now = held[j];
                held[j] = fetch(d, q + HOLD + j);
                add_quad(now, acc);
            }
        }
        for (; q + HOLD < d.z; q += HOLD) {
#pragma unroll
            for (uint32_t j = 0; j < HOLD; ++j) {
                const Quad now = held[j];
                held[j] = fetch(d, q + HOLD + j);
                if (q + j < d.y) add_quad(now, acc);
                else add_padded(now, acc);
            }
        }
        f32x4 ahead[AHEAD];
#pragma unroll
        for (uint32_t i = 0; i < AHEAD; ++i)
            if (from + i * STEP + r_in < next) ahead[i] = load_row(from + i * STEP + r_in);
#pragma unroll
        for (uint32_t j = 0; j < HOLD; ++j) {
            const Quad now = held[j];
            held[j] = fetch(dn, j);
            if (q + j < d.y) add_quad(now, acc);
            else if (q + j < d.z) add_padded(now, acc);
        }
        d = dn;
        if (WARM) {
            asm volatile("" ::"v"(warm));
            if (t + 2u < t1) {
                const uint2 later = tiles[t + 2u];
                const uint32_t line = tid * num_slabs + slab, r = max(next, later.x) + line / lines;
                if (r < later.y) warm = B[size_t(r) * N + min(line % lines * 32u, N - 1u)];
            }
        }
        // acc[j] is piece j ^ l of the lane's row; after these exchanges y[k] is piece l of row k of the Q lanes, and a store
        // fills whole pieces of rows
        f32x4 y[Q];
        y[0] = acc[0];
        y[1] = quad_xor<1>(acc[1]);
        if constexpr (Q == 4) {
            y[2] = quad_xor<2>(acc[2]);
            y[3] = quad_xor<3>(acc[3]);
        }
#pragma unroll
        for (uint32_t bit = 1; bit < Q; bit *= 2)
#pragma unroll
            for (uint32_t k = 0; k < Q; ++k)
                if (!(k & bit)) {
                    const f32x4 a = y[k], b = y[k | bit];
                    const bool swap = l & bit;
                    y[k] = swap ? b : a;
                    y[k | bit] = swap ? a : b;
                }
        const uint32_t row = (t * (kWindowTile / 64u) + wave) * 64u + lane - l;
#pragma unroll
        for (uint32_t k = 0; k < Q; ++k)      // (through the L2: the slabs beside this one fill the rest of the line)
            if (row + k < M) *reinterpret_cast<VecInMemory<4>::type *>(C + size_t(row + k) * N + c0 + l * 4u) = y[k];
        lds_barrier();                        // the rows that leave the window are not read any more
#pragma unroll
        for (uint32_t i = 0; i < AHEAD; ++i)
            if (from + i * STEP + r_in < next) keep_row(from + i * STEP + r_in, ahead[i]);
        for (uint32_t r = from + kWindowTile + r_in; r < next; r += STEP) keep_row(r, load_row(r));     // a window that jumps
        have = next;
        lds_barrier();
    }
}

// One launch for a plan that uses both the quad kernel and the row kernel: they write disjoint
// panels, and the row kernel's short, even work fills the SIMDs that the quad kernel's long chunks
// leave idle.  Blocks [0, quad_blocks) are the quad kernel's 2-D grid flattened (x fastest, so the
// XCD of a block is still x % 8); the rest are the row kernel's blocks, dealt to the XCDs in
// contiguous ranges like the row kernel's own launch does.
template <bool FULL, bool STRIPS, int LOG_L, bool COLUMNS, bool CUT>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup, 8) void hrpb_quad_rows_f32(
    uint32_t quad_blocks_x, uint32_t quad_blocks, const uint32_t *__restrict__ heads, uint32_t num_chunks,
    uint32_t groups_per_xcd, const uint32_t *__restrict__ qrecs, const float *__restrict__ qvals, uint32_t zero_index,
    const uint4 *__restrict__ row_list, uint32_t num_rows, uint32_t row_blocks_per_slab, XcdRanges row_ranges, uint32_t column_slabs, uint32_t row_column_slabs,
    const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols, const float *__restrict__ vals,
    const float *__restrict__ B, float *__restrict__ C, float *__restrict__ partials, uint32_t N, const CutPieces *__restrict__ cut)
{
    static_assert(kWaveSize * kWavesPerGroup == 256, "both bodies are written for 256-thread blocks");
    if (blockIdx.x < quad_blocks) {
        quad_body<FULL, STRIPS, CUT>(blockIdx.x % quad_blocks_x, blockIdx.x / quad_blocks_x, heads, num_chunks, groups_per_xcd,
                                qrecs, qvals, zero_index, B, C, partials, N, COLUMNS ? column_slabs : 0u, cut);
    } else {   // quad_blocks is a multiple of the XCD count, so the XCD of a row block is (its index) % 8 as well
        const uint32_t rb = blockIdx.x - quad_blocks;
        uint32_t slab = rb / row_blocks_per_slab;      // slab by slab, as in csr_rows_batched
        const uint32_t bid = rb - slab * row_blocks_per_slab;
        uint32_t block_id;
        const uint32_t x = xcd_share(bid, slab, COLUMNS ? row_column_slabs : 0u);
        if (!xcd_range_id(row_ranges, bid, x, block_id)) return;
        rows_batched_body<4, LOG_L, 8, (LOG_L > 4 || COLUMNS)>(block_id, slab, row_list, num_rows, rowPtr, cols, vals, B, C, N);
    }
}

// The same for a plan that pairs the rolling brick kernel with the row kernel.
template <int VEC, int NG, bool FULL, int LOG_L, bool COLUMNS, bool CUT>
__global__ __launch_bounds__(kWaveSize *kWavesPerGroup, (NG == 1 ? 8 : 4)) void hrpb_brick_rows_f32(
    uint32_t brick_blocks_x, uint32_t brick_blocks, const uint4 *__restrict__ chunks, uint32_t num_chunks,
    uint32_t groups_per_xcd, const uint32_t *__restrict__ hdr, const float *__restrict__ tile_vals, uint32_t zero_index,
    const uint4 *__restrict__ row_list, uint32_t num_rows, uint32_t row_blocks_per_slab, XcdRanges row_ranges, uint32_t column_slabs, uint32_t row_column_slabs,
    const uint32_t *__restrict__ rowPtr, const uint32_t *__restrict__ cols, const float *__restrict__ vals,
    const float *__restrict__ B, float *__restrict__ C, float *__restrict__ partials, uint32_t N, const CutPieces *__restrict__ cut)
{
    if (blockIdx.x < brick_blocks) {
        brick_rolling_body<VEC, NG, FULL, true, CUT>(blockIdx.x % brick_blocks_x, blockIdx.x / brick_blocks_x, chunks, num_chunks,
                                          groups_per_xcd, hdr, tile_vals, zero_index, B, C, partials, N, COLUMNS ? column_slabs : 0u, cut);
    } else {
        const uint32_t rb = blockIdx.x - brick_blocks;
        uint32_t slab = rb / row_blocks_per_slab;
        const uint32_t bid = rb - slab * row_blocks_per_slab;
        uint32_t block_id;
        const uint32_t x = xcd_share(bid, slab, COLUMNS ? row_column_slabs : 0u);
        if (!xcd_range_id(row_ranges, bid, x, block_id)) return;
        rows_batched_body<4, LOG_L, 8, (LOG_L > 3)>(block_id, slab, row_list, num_rows, rowPtr, cols, vals, B, C, N);
    }
}

// Thread per C element (inc/SPMM.cuh:898-920 restated for fp32 and a 64x4 thread tile).
__global__ __launch_bounds__(256) void csr_thread_per_element(const uint32_t *__restrict__ rowPtr,
                                                              const uint32_t *__restrict__ cols,
                                                              const float *__restrict__ vals,
                                                              const float *__restrict__ B, float *__restrict__ C,
                                                              uint32_t M, uint32_t N)
{
    const uint32_t col = blockIdx.x * 64u + threadIdx.x;
    const uint32_t row = blockIdx.y * 4u + threadIdx.y;
    if (row >= M || col >= N) return;
    float sum = 0.0f;
    for (uint32_t i = rowPtr[row]; i < rowPtr[row + 1]; ++i) sum += vals[i] * B[size_t(cols[i]) * N + col];
    C[size_t(row) * N + col] = sum;
}

// Wavefront per row, lane L handles columns L, L+64, ...; every lane reads (col, val) itself.
__global__ __launch_bounds__(256) void csr_wave_scalar(const uint32_t *__restrict__ rowPtr,
                                                       const uint32_t *__restrict__ cols,
                                                       const float *__restrict__ vals, const float *__restrict__ B,
                                                       float *__restrict__ C, uint32_t M, uint32_t N)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t row = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
    if (row >= M) return;
    const uint32_t s = rowPtr[row], e = rowPtr[row + 1];
    for (uint32_t c = lane; c < N; c += 64u) {
        float sum = 0.0f;
        for (uint32_t i = s; i < e; ++i) sum += vals[i] * B[size_t(cols[i]) * N + c];
        C[row * N + c] = sum;
    }
}

}  // namespace cute_dev
