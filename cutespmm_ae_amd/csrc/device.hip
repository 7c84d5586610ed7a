// Device side of libcutespmm: upload, plan, launch, plain CSR kernels, timing helpers.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <functional>
#include <mutex>
#include <string>
#include <unordered_map>

#include "common.hpp"
#include "kernels.hip.hpp"
#include "build_kernels.hip.hpp"

using namespace cute;

namespace {

thread_local std::string g_hip_error;
thread_local hipError_t g_hip_status = hipSuccess;      // of the call g_hip_error describes

// The planner's default thresholds (measured on the five benchmark matrices and on the reference's 43).
constexpr float kMinReuse = 1.25f;          // a panel with fewer nonzeros per B row the MFMA side would fetch goes to the row kernel
constexpr uint64_t kWideWindowBytes = 16ull << 20;   // ... whose window of B is wider than this (four L2s' worth)
constexpr float kWideReuse = 0.98f;          // ... the bar for products of 256 columns or more over large matrices (see cute_spmm_plan_create)
constexpr uint32_t kMaxRowForRows = 48;      // ... unless it holds a row longer than this: one lane group would serialise it
constexpr uint32_t kRowBatch = 8;           // entries the row kernel has in flight per row
constexpr uint32_t kTilePanels = cute_dev::kWindowTile / CUTE_TM;   // panels of a tile of csr_rows_window
// A panel is scattered when the window of B it reads (at most 256 columns of it at a time) is wider than this: its rows then
// come from behind the L2s, which deliver about 8 TB/s against the 20 an L2 gives.  One and a half L2s: bands of 4 100
// rows by 256 columns still come out of an L2 (92 % hits), 8 192 rows at random do not (N = 512: 25 us in row order, 12 with
// an XCD per column slab).
constexpr uint64_t kScatteredBytes = 6ull << 20;
constexpr float kGraphReuse = 2.0f;          // scattered panels of large products (see cute_spmm_plan_create)
constexpr uint32_t kGraphMaxRow = 96;
constexpr uint64_t kGraphProduct = 1ull << 24;   // rows times columns from which on those two apply
constexpr uint32_t kMaxHubRows = 256;       // hub plans: B rows a work-group keeps in LDS (64 KiB of 256-byte pieces; two work-groups per CU)
constexpr uint32_t kUnevenRowFloor = 16;     // row kernel vs MFMA kernel: a panel whose longest row exceeds this and ...
constexpr uint32_t kUnevenRowRatio = 2;      // ... this many mean rows of the panel goes to the MFMA kernel while rows share wavefronts
constexpr float kHybridFill = 0.15f;         // cute_hybrid: a tile goes to the Blocked-ELL part from this fill on (threshold 0)
constexpr uint64_t kSlotsPerBrick = 8;      // quad lists when the MFMA panels need fewer list slots per 16x4 brick, else brick tiles
// B and C together larger than the Infinity Cache: whatever the caller does between launches, their rows come
// from HBM.  There the brick kernel's wider row pieces (16 lanes x 16 bytes per row and column group, two groups
// per wavefront from N = 128 on) beat the quad kernel's 256-byte pieces by 20-25 % (9-point stencils of 0.25 to
// 1 million rows) -- as long as its matrix work, 32 cycles per brick and 16 columns however empty the brick,
// stays below the time the operands take to stream at 4 TB/s; on R-MAT graphs, where it is 1.4 to 1.7 times
// that, the two kernels are within 10 % of each other either way and the rule above keeps deciding.  While the
// operands fit the cache the quad kernel is level or ahead.
constexpr double kStreamBytesPerSecond = 4.0e12, kSimdCyclesPerSecond = 1024 * 2.4e9, kCyclesPerBrickTile = 32.0;

// Which MFMA kernel serves the panels that go to the matrix cores (1 brick tiles, 2 quad lists).
//   slots   list slots of the quad lists (pairs plus padding): the quad kernel pays 8 matrix cycles and one
//           256-byte piece of a B row per slot and 64 columns
//   bricks  16x4 bricks: the brick kernel pays 32 matrix cycles per brick and 16 columns, however empty the brick
//   blocks  16-column blocks: the brick kernel requests 16 row pieces per block (padding columns included)
// A launch fed from a cache is bound by what it issues, and the two kernels cross at about 8 slots per brick
// (measured on the benchmark matrices and on the reference's 43).  A launch fed from HBM is bound by the
// memory system, and what counts there is how many row pieces a kernel requests and how wide they are: the
// brick kernel asks for a B row once per panel, in pieces of 512 contiguous bytes from N = 128 on; the quad
// kernel once per 4-row group that uses it, in 256-byte pieces that two wavefronts request at different
// times.  Measured with operands no cache holds: 9-point stencils (1.25 slots per brick-kernel fetch) run
// 7-25 % faster through the brick kernel at 16 384 to 262 144 rows and N = 64..512, 5-point stencils (1.0)
// 5-8 % slower; from a cache the quad kernel is level or up to 20 % ahead on both.  So unless the caller
// says that the operands stay cache-resident (operand_residency = 2, a tight loop over the same buffers that
// fit the Infinity Cache), a matrix whose quad lists need more than 1.1 fetches per brick-kernel fetch goes to
// the brick kernel -- as long as its matrix work stays below the time the operands take to stream at 4 TB/s
// (on R-MAT graphs it is 1.4-1.7 times that, and the quad kernel keeps them).
// A graph's panels pass that test as well while N is small, but their bricks are nearly empty and what streams is not B but
// the gathered rows: only lists whose slots carry 1.4 entries or more (9-point stencils 1.8, finite elements 2.8; R-MAT graphs
// 1.03 ... 1.25) go to the brick kernel.  R-MAT graph of 131 072 nodes, N = 32: 74.5 us through bricks, 37.3 through lists;
// 65 536 nodes, N = 47: 36.5 against 26.2.  Products of less than 32 columns keep the bricks (their narrow tiles; a list
// slot always spans 64 columns): 32 768 nodes, N = 16: 11.5 against 16.1.
int choose_mfma_shape(uint64_t slots, uint64_t bricks, uint64_t blocks, uint64_t entries, uint64_t rows_and_cols, uint64_t nnz, uint32_t N,
                      uint32_t residency, uint64_t cache_bytes)
{
    int shape = slots < kSlotsPerBrick * bricks ? 2 : 1;
    const bool resident = residency == 2 && rows_and_cols * N * sizeof(float) <= cache_bytes;
    if (shape == 2 && !resident && slots * 10u > blocks * 16u * 11u && (N < 32u || entries * 10u >= slots * 14u)) {
        const double matrix_s = double(bricks) * double((N + 15u) / 16u) * kCyclesPerBrickTile / kSimdCyclesPerSecond;
        const double stream_s = (double(rows_and_cols) * N * 4.0 + double(nnz) * 8.0) / kStreamBytesPerSecond;
        if (matrix_s <= stream_s) shape = 1;
    }
    return shape;
}

// Floats per lane of a B or C row: four wherever a row has four (the kernels need no alignment beyond a float).
inline int lane_floats(uint32_t N) { return N >= 4u ? 4 : N >= 2u ? 2 : 1; }

// (an error that is returned is not left behind for the next launch to find)
inline int hip_fail(hipError_t e, const char *what, int line)
{
    (void)hipGetLastError();
    g_hip_status = e;
    g_hip_error = std::string(hipGetErrorString(e)) + " (" + what + ", device.hip:" + std::to_string(line) + ")";
    return CUTE_ERR_HIP;
}
#define HIP_TRY(expr)                                                    \
    do {                                                                 \
        hipError_t e_ = (expr);                                          \
        if (e_ != hipSuccess) return hip_fail(e_, #expr, __LINE__);      \
    } while (0)

struct DeviceContext {
    int status = CUTE_ERR_NO_DEVICE;
    int device = 0;
    int num_cus = 0;
    int wave_size = 0;
    // What the planner assumes about the part of the chip this device is.  A whole MI355X (SPX mode) shows 256
    // compute units in 8 XCDs of 32, each XCD with its own 4 MiB L2, and 256 MiB of Infinity Cache; in the
    // partitioned modes a device is 4, 2 or 1 of those XCDs with its share of the cache.  The kernels' mapping of
    // work-groups to contiguous panel ranges is written for 8 XCDs and stays a valid, locality-preserving order
    // on fewer (a device with x XCDs walks 8/x ranges per XCD); the model of where wavefronts land, which only
    // orders work items, is used on the whole chip alone.
    int num_xcds = 8;
    bool whole_chip = false;
    uint64_t cache_bytes = 256ull << 20;
    std::string arch;
};

// The library is written for gfx950 only; any other device is refused, loudly.
const DeviceContext &context()
{
    static DeviceContext ctx = [] {
        DeviceContext c;
        int n = 0;
        if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
            g_hip_error = "no HIP device visible";
            return c;
        }
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return c;
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return c;
        c.device = dev;
        c.num_cus = prop.multiProcessorCount;
        c.wave_size = prop.warpSize;
        c.arch = prop.gcnArchName;
        if (c.arch.rfind("gfx950", 0) != 0) {
            g_hip_error = "device is " + c.arch + ", this library is built for gfx950 only";
            return c;
        }
        if (c.num_cus > 0 && c.num_cus % 32 == 0 && c.num_cus / 32 <= 8) c.num_xcds = c.num_cus / 32;
        c.whole_chip = c.num_cus == 256;
        c.cache_bytes = (256ull << 20) * uint64_t(c.num_xcds) / 8u;
        c.status = CUTE_OK;
        return c;
    }();
    return ctx;
}

// Scratch for cute_spmm_run_static: the partial tiles of cut panels, for callers that cannot allocate.
// One copy per GPU, part of the loaded code object, held until the process ends.  In host code the name
// of the array is only a handle for hipGetSymbolAddress -- never a device address.
static __device__ __align__(256) unsigned char scratch[CUTE_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
void *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per device.
int static_scratch(void **out)
{
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return CUTE_ERR_ARG;
    std::lock_guard<std::mutex> g(g_scratch_lock);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return CUTE_OK;
}

void drop_idle_device_memory();

// hipMalloc; when there is no memory left, once more without the idle blocks of the pool below.
hipError_t device_malloc(void **out, uint64_t bytes)
{
    hipError_t e = hipMalloc(out, std::max<uint64_t>(bytes, 16));
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        drop_idle_device_memory();
        e = hipMalloc(out, std::max<uint64_t>(bytes, 16));
    }
    if (e != hipSuccess) *out = nullptr;
    return e;
}

template <class T>
int upload(T **dst, const T *src, uint64_t count)
{
    *dst = nullptr;
    HIP_TRY(device_malloc(reinterpret_cast<void **>(dst), count * sizeof(T)));
    if (count) HIP_TRY(hipMemcpy(*dst, src, count * sizeof(T), hipMemcpyHostToDevice));
    return CUTE_OK;
}

}  // namespace

struct cute_hrpb_dev {
    uint32_t M = 0, K = 0, nnz = 0, P = 0, nb = 0;
    uint64_t numVals = 0, bytes = 0;
    // Of the two MFMA layouts only the one the planner's default rules would pick for this matrix is built by
    // the upload (none if every panel would go to the row kernel); the other is built from the device copy of
    // the CSR arrays the first time a plan asks for it.  `lock` guards those late builds.
    std::mutex lock;
    bool haveBricks = false, haveQuads = false;
    // one allocation each: the CSR arrays, the brick tiles, the quad lists
    void *csrMemory = nullptr, *brickMemory = nullptr, *quadMemory = nullptr, *windowMemory = nullptr;
    uint32_t *dHdr = nullptr;           // brick tiles: one 128-byte header line per block
    float *dVals = nullptr;             // brick tiles: values in lane order, then 64 zeros
    uint32_t *dRowPtr = nullptr, *dCols = nullptr;
    float *dCsrVals = nullptr;
    uint32_t *dQRecs = nullptr;         // quad lists: one record per group (16 columns, slot mask, first value)
    float *dQVals = nullptr;            // quad lists: the occupied value slots in lane order, then 64 zeros
    uint64_t numQuadVals = 0;
    uint64_t numGroups = 0;
    std::vector<uint32_t> brp;          // host copy of blockedRowPtr
    std::vector<uint32_t> qgp;          // the quad lists' groupPtr (known from the census, before the lists are built)
    std::vector<uint32_t> stripPairs;   // length of the merged column list of every 4-row strip
    uint32_t quadRows = CUTE_TM;        // rows per list unit: 16 (lockstep lists per panel) or 4 (strips)
    uint64_t quadPairs = 0;             // occupied (row group, column) pairs
    std::vector<uint32_t> panelNnz;     // nonzeros per row panel
    std::vector<uint32_t> panelCols;    // active columns per row panel
    std::vector<uint32_t> panelMaxRow;  // longest row of each panel
    std::vector<uint32_t> panelSpan;    // width of each panel's column window (last column - first column + 1)
    uint32_t longestPanel = 0;          // the largest of panelNnz
    bool anyLarge = false;              // panels that the panel kernels do not take
    std::vector<uint2> tileWindow;      // columns [first, end) of every tile of csr_rows_window; a tile without entries: [~0, 0)
    uint32_t widestTile = 0;            // the widest of these
    // the entries as csr_rows_window reads them (which describes them), built for the first plan that uses that kernel
    bool haveWindow = false;
    uint4 *dSlices = nullptr;
    uint2 *dWindowSlots = nullptr, *dWindowTiles = nullptr;
    cute_dev::f32x4 *dWindowVals = nullptr;
    std::vector<uint32_t> longStrips;   // 4 panel + strip of every strip of more than kPanelList entries, ascending
    std::vector<uint32_t> panelStored;  // entries of each panel that are not zero (what the quad lists store)
};

namespace { void give_device_memory(void *p); void drop_idle_pinned_memory(); }

struct cute_spmm_plan {
    const cute_hrpb_dev *d = nullptr;
    cute_plan_info info{};
    int vec = 4, ng = 1;                // brick kernel shape
    int pipeline = 1;                   // 1: rolling variant, 2: pipelined variant
    int shape = 2;                      // MFMA kernel: 1 16x16x4 bricks, 2 4x4x1 quad lists
    bool halfLists = false;             // quad kernel on slabs of 32 columns
    bool bf16x3 = false;                // brick kernel on the bf16 matrix pipeline (three products of bf16 hi/lo parts)
    int rows_vec = 4, rows_logl = 6;    // row kernel shape
    uint32_t rows_slabs = 1;
    void *memory = nullptr;             // one allocation for the tables and the partial tiles below
    uint4 *dChunks = nullptr;           // brick kernels
    uint32_t *dHeads = nullptr;         // quad kernels: per chunk, the descriptor and the record of its first group
    // hub plans: the most referenced B rows are staged in LDS by persistent work-groups (hrpb_quad_hub_f32)
    uint32_t numHub = 0;
    uint32_t *dHubRows = nullptr;       // the hub rows' column ids, slot order
    uint32_t *dHubRecs = nullptr;       // the plan's copy of the quad records, hub columns replaced by their slots
    // panels (or 4-row strips) cut into several chunks: each chunk stores a partial tile, and they are added up by
    // reduce_partials, or by themselves (store_piece) where the launch has a CutPieces: one set for cute_spmm_run, one for cute_spmm_run_static, because
    // calls of the two may overlap; cute_spmm_run_scratch, of which any number may, has the reduce_partials launch
    uint4 *dFixups = nullptr;           // {panel or strip, first piece, pieces, -}
    cute_dev::CutPieces *dCut = nullptr, *dCutStatic = nullptr;
    uint32_t numFixups = 0;
    uint32_t reduceBlocksY = 1;         // blocks of reduce_partials along a tile: enough for the tile with the most pieces
    uint32_t unitRows = CUTE_TM;        // rows of one panel / strip / piece
    float *dPartials = nullptr;         // pieces x unitRows rows of N floats; owned by the plan, so a plan runs on one stream at a time
    uint64_t partialBytes = 0;
    void *staticScratch = nullptr;      // device address of the library's static scratch array on the plan's device
    uint4 *dRowList = nullptr;          // rows of the sparse path with their row pointers: {row, first entry, end, 0}
    uint32_t numRows = 0;
    cute_dev::XcdRanges rowRanges{};   // row-kernel blocks of each XCD, balanced by nonzeros
    // slabs of the MFMA part and of the row part when an XCD owns columns instead of rows (cute_dev::xcd_share), else 0
    uint32_t columnSlabs = 0, rowColumnSlabs = 0;
    uint32_t rowBlocksPerXcd = 0;       // longest of those ranges
    // rows through csr_rows_split: lane groups that share a row (1: not used), a power of two
    uint32_t rowParts = 1;
    // rows through csr_rows_window: columns of B in its ring (0: not used) and the chains of tiles
    uint32_t windowColumns = 0, windowChains = 0, windowChainTiles = 0;
    bool windowWarm = false;
};

namespace {

// Work items of a plan: every one is written before it is read, so making room for them writes nothing.
template <class T> struct Unset : std::allocator<T> {
    template <class U> struct rebind { using other = Unset<U>; };
    template <class U, class... A> void construct(U *at, A &&...a)
    {
        if constexpr (sizeof...(A) == 0) ::new (static_cast<void *>(at)) U;
        else ::new (static_cast<void *>(at)) U(std::forward<A>(a)...);
    }
};
using WorkItems = std::vector<uint4, Unset<uint4>>;

// Deals the MFMA work items to the SIMDs by length.  When a launch fits on the device at once, nothing balances
// it afterwards: every wavefront is placed when the launch starts, and a SIMD that was handed three long panels
// keeps the whole launch waiting.  Where the work-groups land is regular (observed with the hardware id
// registers; nothing but speed depends on it): work-group g goes to XCD g % 8; the s-th work-group an XCD
// receives (x fastest, then the slabs) runs on its CU s % (CUs per XCD); and wavefront w of that work-group
// shares a SIMD with wavefront (w + 1) % 4 of the work-group the same CU received one round earlier.  So
// position (k, w) of an XCD's part of the list, in slab y, counts on SIMD lane (w + s / CUs) % 4 of CU s % CUs
// with s = y * groups_per_xcd + k.  Longest first, every item takes the free position that keeps the fullest
// SIMD it touches lowest (ties: the earliest position, so equal items stay in panel order and keep sharing B
// rows in the L1).  The new order is used only if the model says it shortens the fullest SIMD by 3 % or more.
// An item costs its length plus a fixed two units (descriptor, first operands, the store).
// The positions that meet the same SIMDs in every slab (cus_per_xcd work-groups apart, one wavefront further) are a class, one for every
// SIMD of the first slab, and a class is as loaded as any of its positions: a heap holds the classes by load and first free
// position, not the positions.  Nothing is dealt where even a perfect order would not gain the 3 %.  (The host threads take longer to wake than
// this takes.  One heap of all positions: 400 us of the 510 that a new 9-point matrix of 300 x 300 points took from format to product, N = 64.)
bool deal_chunks(WorkItems &chunks, uint32_t num_slabs, uint32_t cus_per_xcd, uint32_t waves_per_simd, bool force)
{
    constexpr uint32_t wpg = cute_dev::kWavesPerGroup, xcds = cute_dev::kNumXcd;
    if (cus_per_xcd == 0 || wpg != 4) return false;
    const uint64_t resident = uint64_t(cus_per_xcd) * xcds * 4u * waves_per_simd;
    if (uint64_t(chunks.size()) * num_slabs > resident) return false;      // later work-groups go wherever one retires
    const uint32_t count = uint32_t(chunks.size()), groups = (count + wpg - 1) / wpg;
    const uint32_t per_xcd = (groups + xcds - 1) / xcds, span = per_xcd * wpg, simds = cus_per_xcd * 4u;
    std::vector<uint32_t> lane(size_t(simds) * num_slabs);   // the SIMDs a class meets, slab by slab
    for (uint32_t k = 0; k < simds; ++k)
        for (uint32_t y = 0; y < num_slabs; ++y) {
            const uint32_t s = y * per_xcd + k / 4u;
            lane[size_t(k) * num_slabs + y] = (s % cus_per_xcd) * 4u + (k % 4u + s / cus_per_xcd) % 4u;
        }
    auto cost = [&](uint32_t i) { return uint64_t(chunks[i].y - chunks[i].x) + 2u; };
    auto begin_of = [&](uint32_t x) { return std::min(count, x * span); };
    std::vector<uint64_t> load(size_t(simds) * xcds);
    uint64_t before = 0, bound = 0, longest = 0;
    for (uint32_t x = 0; x < xcds; ++x) {
        const uint32_t b = begin_of(x), n = begin_of(x + 1u) - b;
        uint64_t *const of = load.data() + size_t(x) * simds, total = 0, shortest = ~0ull;
        for (uint32_t k = 0, cu = 0, turn = 0; k * wpg < n; ++k) {
            for (uint32_t w = 0; w < std::min(wpg, n - k * wpg); ++w) {
                const uint64_t c = cost(b + k * wpg + w);
                const uint32_t *const to = lane.data() + size_t(cu * 4u + (w + turn) % 4u) * num_slabs;
                for (uint32_t y = 0; y < num_slabs; ++y) of[to[y]] += c;
                total += c;
                shortest = std::min(shortest, c);
                longest = std::max(longest, c);
            }
            if (++cu == cus_per_xcd) { cu = 0; ++turn; }
        }
        before = std::max(before, *std::max_element(of, of + simds));
        if (n) bound = std::max({bound, (total * num_slabs + simds - 1u) / simds, (uint64_t(n) * num_slabs + simds - 1u) / simds * shortest});
    }
    bound = std::max(bound, longest);
    if (!force && bound * 100u > before * 97u) return false;

    std::vector<uint32_t> order(count);                      // of every XCD: longest first, then by position
    if (longest <= 4096u) {
        std::vector<uint32_t> place(longest + 1u);
        for (uint32_t x = 0; x < xcds; ++x) {
            const uint32_t b = begin_of(x), e = begin_of(x + 1u);
            std::fill(place.begin(), place.end(), 0u);
            for (uint32_t i = b; i < e; ++i) ++place[cost(i)];
            uint32_t at = b;
            for (size_t k = place.size(); k-- > 0;) { const uint32_t here = place[k]; place[k] = at; at += here; }
            for (uint32_t i = b; i < e; ++i) order[place[cost(i)]++] = i;
        }
    } else {
        for (uint32_t i = 0; i < count; ++i) order[i] = i;
        for (uint32_t x = 0; x < xcds; ++x)
            std::stable_sort(order.begin() + begin_of(x), order.begin() + begin_of(x + 1u), [&](uint32_t i, uint32_t k) { return cost(i) > cost(k); });
    }
    struct Class {
        uint64_t load;                                       // of its fullest SIMD, or what that was
        uint32_t pos, k;                                     // its first free position; its number
        bool operator<(const Class &o) const { return load != o.load ? load < o.load : pos < o.pos; }
    };
    std::vector<Class> heaps(size_t(simds) * xcds);
    WorkItems dealt(count);
    std::fill(load.begin(), load.end(), 0);
    for (uint32_t x = 0; x < xcds; ++x) {
        const uint32_t b = begin_of(x), e = begin_of(x + 1u), n = e - b;
        uint64_t *const of = load.data() + size_t(x) * simds;
        Class *const heap = heaps.data() + size_t(x) * simds;
        uint32_t size = std::min(simds, n);
        for (uint32_t k = 0; k < size; ++k) heap[k] = {0u, k, k};
        auto peak = [&](uint32_t k) {
            uint64_t most = 0;
            for (uint32_t y = 0; y < num_slabs; ++y) most = std::max(most, of[lane[size_t(k) * num_slabs + y]]);
            return most;
        };
        auto sink = [&](const Class c) {                 // c in the place of the first
            uint32_t at = 0;
            for (uint32_t child; (child = 2u * at + 1u) < size; at = child) {
                if (child + 1u < size && heap[child + 1u] < heap[child]) ++child;
                if (!(heap[child] < c)) break;
                heap[at] = heap[child];
            }
            heap[at] = c;
        };
        for (uint32_t o = b; o < e; ++o) {
            // loads only grow: one that another class has raised goes back with its new load
            for (uint64_t now; num_slabs > 1u && (now = peak(heap[0].k)) != heap[0].load;) sink({now, heap[0].pos, heap[0].k});
            Class c = heap[0];
            dealt[b + c.pos] = chunks[order[o]];
            for (uint32_t y = 0; y < num_slabs; ++y) of[lane[size_t(c.k) * num_slabs + y]] += cost(order[o]);
            c.load = peak(c.k);
            c.pos = (c.pos / 4u + cus_per_xcd) * 4u + (c.pos + 3u) % 4u;
            if (c.pos < n) sink(c);
            else if (--size) sink(heap[size]);
        }
    }
    if (!force && *std::max_element(load.begin(), load.end()) * 100u > before * 97u) return false;
    chunks.swap(dealt);
    return true;
}

}  // namespace

extern "C" {

const char *cute_last_hip_error(void) { return g_hip_error.c_str(); }

int cute_device_info(int *num_cus, int *wave_size, char *arch_name, size_t arch_cap)
{
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    if (num_cus) *num_cus = c.num_cus;
    if (wave_size) *wave_size = c.wave_size;
    if (arch_name && arch_cap) std::snprintf(arch_name, arch_cap, "%s", c.arch.c_str());
    return CUTE_OK;
}

void cute_release_idle_memory(void)
{
    drop_idle_device_memory();
    drop_idle_pinned_memory();
}

int cute_device_layout(int *num_xcds, int *cus_per_xcd, uint64_t *cache_bytes, int *whole_chip)
{
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    if (num_xcds) *num_xcds = c.num_xcds;
    if (cus_per_xcd) *cus_per_xcd = c.num_cus / c.num_xcds;
    if (cache_bytes) *cache_bytes = c.cache_bytes;
    if (whole_chip) *whole_chip = c.whole_chip ? 1 : 0;
    return CUTE_OK;
}

void cute_hrpb_dev_free(cute_hrpb_dev *d)
{
    if (!d) return;
    give_device_memory(d->csrMemory);
    give_device_memory(d->brickMemory);
    give_device_memory(d->quadMemory);
    give_device_memory(d->windowMemory);
    delete d;
}

uint64_t cute_hrpb_dev_bytes(const cute_hrpb_dev *d) { return d ? d->bytes : 0; }

int cute_hrpb_upload(const cute_hrpb_host *h, cute_hrpb_dev **out) { return cute_hrpb_upload_layout(h, 0, out); }

}  // extern "C"

namespace {

// ---- building the layouts on the device (kernels: build_kernels.hip.hpp) ----

// Waits for every stream of the device as hipFree does, by freeing a page (1.2 us).  Not hipDeviceSynchronize, which breaks a
// capture under way on any stream; hipFree is allowed beside a capture in relaxed mode, and a handle may be collected in the
// middle of one.
bool wait_for_device()
{
    void *page = nullptr;
    if (hipMalloc(&page, 4096) == hipSuccess) return hipFree(page) == hipSuccess;
    (void)hipGetLastError();
    return false;
}

// Device memory of handles, plans and their set-up.  hipMalloc and hipFree of a megabyte or more cost 25 to 50 us each (a new
// graph's product, 65 536 nodes: 300 us of 900 went there), so released blocks wait here for the next caller.  Bounded: at
// most kIdleBytes in kIdleBlocks blocks, none that the last kIdleUses releases have not touched; the rest goes back to the
// driver, and all of it does when an allocation fails.  Like hipFree, a release waits for the device first, so no kernel of
// any stream still uses a block that another thread is given; a block stays with its device.
constexpr uint64_t kIdleBytes = 512ull << 20, kPooledBlock = 1ull << 20, kLargestIdle = kIdleBytes / 4u, kIdleUses = 64;
constexpr size_t kIdleBlocks = 32;

class DevicePool {
    struct Block { void *p; uint64_t bytes; int device; uint64_t used; };
    std::mutex lock_;
    std::vector<Block> idle_;
    std::unordered_map<void *, std::pair<uint64_t, int>> out_;
    uint64_t idleBytes_ = 0, clock_ = 0;

    void drop(size_t i)
    {
        idleBytes_ -= idle_[i].bytes;
        (void)hipFree(idle_[i].p);
        idle_.erase(idle_.begin() + std::ptrdiff_t(i));
    }

public:
    int take(void **out, uint64_t bytes)
    {
        *out = nullptr;
        // (a block that will not be kept is as large as it was asked for)
        if (bytes < kPooledBlock || bytes > kLargestIdle) { HIP_TRY(device_malloc(out, bytes)); return CUTE_OK; }
        // eight sizes to an octave: matrices of nearly the same size meet in one
        const uint64_t step = 1ull << (60 - __builtin_clzll(bytes));
        bytes = (bytes + step - 1) / step * step;
        int device = 0;
        HIP_TRY(hipGetDevice(&device));
        {
            std::lock_guard<std::mutex> g(lock_);
            for (size_t i = idle_.size(); i-- > 0;)
                if (idle_[i].bytes == bytes && idle_[i].device == device) {
                    *out = idle_[i].p;
                    idleBytes_ -= bytes;
                    idle_.erase(idle_.begin() + std::ptrdiff_t(i));
                    break;
                }
        }
        if (!*out) HIP_TRY(device_malloc(out, bytes));
        std::lock_guard<std::mutex> g(lock_);
        out_[*out] = {bytes, device};
        return CUTE_OK;
    }
    void give(void *p)
    {
        if (!p) return;
        int device = -1;
        const bool known = hipGetDevice(&device) == hipSuccess;
        uint64_t bytes = 0;
        {
            std::lock_guard<std::mutex> g(lock_);
            const auto it = out_.find(p);
            if (it != out_.end()) {
                if (known && it->second.second == device) bytes = it->second.first;
                out_.erase(it);
            }
        }
        if (!bytes || !wait_for_device()) { (void)hipFree(p); return; }
        std::lock_guard<std::mutex> g(lock_);
        ++clock_;
        idle_.push_back({p, bytes, device, clock_});
        idleBytes_ += bytes;
        while (idle_.size() > kIdleBlocks || idleBytes_ > kIdleBytes || idle_.front().used + kIdleUses < clock_) drop(0);
    }
    void drop_all()
    {
        std::lock_guard<std::mutex> g(lock_);
        while (!idle_.empty()) drop(idle_.size() - 1);
    }
};

DevicePool &pool()
{
    static DevicePool *p = new DevicePool;   // never destroyed: the driver may be gone when a process ends
    return *p;
}

void give_device_memory(void *p) { pool().give(p); }
void drop_idle_device_memory() { pool().drop_all(); }

struct DevBuf {                       // device memory that lives as long as a scope
    void *p = nullptr;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { pool().give(p); }
    int alloc(uint64_t bytes) { return pool().take(&p, bytes); }
    void *release() { void *q = p; p = nullptr; return q; }
    template <class T> T *as() const { return static_cast<T *>(p); }
};

// Several arrays in one allocation: sizes first, then the pointers.
struct Layout {
    uint64_t bytes = 0;
    uint64_t add(uint64_t count, uint64_t size)
    {
        const uint64_t at = bytes;
        bytes += (count * size + 255u) & ~uint64_t(255);
        return at;
    }
    template <class T> static T *at(void *base, uint64_t offset) { return reinterpret_cast<T *>(static_cast<char *>(base) + offset); }
};

// Pinned host memory through which set-up exchanges its tables with the device: kernels read and write it directly.  A copy
// call moves up to 16 KB in about 13 us but 64 KB and more in 130 us (the copy engine's start); a kernel reads 64 KB of
// pinned memory in 3 us and 12 MB in 250.  Allocating and freeing a buffer costs 40 us, so released buffers wait here for the
// next caller: at most kPinnedBuffers of them and kPinnedBytes in all, anything beyond is freed at once.  A buffer belongs to
// one caller at a time and comes back only when no kernel uses it any more.
constexpr size_t kPinnedBuffers = 4;
constexpr uint64_t kPinnedBytes = 32ull << 20;
std::mutex g_pinned_lock;
std::vector<std::pair<void *, uint64_t>> g_pinned;

struct PinnedBuf {
    void *p = nullptr;
    uint64_t cap = 0;
    bool pending = false;             // a kernel that uses it may still run
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf &) = delete;
    PinnedBuf &operator=(const PinnedBuf &) = delete;
    ~PinnedBuf()
    {
        if (!p) return;
        if (pending) (void)hipStreamSynchronize(nullptr);
        {
            std::lock_guard<std::mutex> g(g_pinned_lock);
            uint64_t held = cap;
            for (const auto &b : g_pinned) held += b.second;
            if (g_pinned.size() < kPinnedBuffers && held <= kPinnedBytes) {
                g_pinned.emplace_back(p, cap);
                return;
            }
        }
        (void)hipHostFree(p);
    }
    int alloc(uint64_t bytes)
    {
        bytes = std::max<uint64_t>(bytes, 64u << 10);
        {
            std::lock_guard<std::mutex> g(g_pinned_lock);
            size_t best = g_pinned.size();
            for (size_t i = 0; i < g_pinned.size(); ++i)
                if (g_pinned[i].second >= bytes && (best == g_pinned.size() || g_pinned[i].second < g_pinned[best].second)) best = i;
            if (best < g_pinned.size()) {
                p = g_pinned[best].first;
                cap = g_pinned[best].second;
                g_pinned.erase(g_pinned.begin() + std::ptrdiff_t(best));
                return CUTE_OK;
            }
        }
        bytes = (bytes + 0xffffu) & ~uint64_t(0xffff);
        HIP_TRY(hipHostMalloc(&p, bytes, hipHostMallocPortable | hipHostMallocMapped));
        cap = bytes;
        return CUTE_OK;
    }
    int wait()
    {
        HIP_TRY(hipStreamSynchronize(nullptr));
        pending = false;
        return CUTE_OK;
    }
    template <class T> T *as(uint64_t offset = 0) const { return Layout::at<T>(p, offset); }
};

void drop_idle_pinned_memory()
{
    std::vector<std::pair<void *, uint64_t>> idle;
    {
        std::lock_guard<std::mutex> g(g_pinned_lock);
        idle.swap(g_pinned);
    }
    for (const auto &b : idle) (void)hipHostFree(b.first);
}

// A stream beside the default one for set-up kernels that need nothing from those on the default stream: one per device and process, non-blocking
// (what its kernels read is complete when they are launched), at the default priority.  Whoever has launched on it waits for it before it returns.
class SideStream {
    hipStream_t used_ = nullptr;

public:
    SideStream() = default;
    SideStream(const SideStream &) = delete;
    SideStream &operator=(const SideStream &) = delete;
    ~SideStream() { (void)wait(); }
    // the default stream where there is none
    hipStream_t get()
    {
        static std::mutex lock;
        static hipStream_t streams[kMaxDevices];
        int dev = -1;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
        std::lock_guard<std::mutex> g(lock);
        if (!streams[dev] && hipStreamCreateWithFlags(&streams[dev], hipStreamNonBlocking) != hipSuccess) {
            (void)hipGetLastError();
            streams[dev] = nullptr;
        }
        return used_ = streams[dev];
    }
    int wait()
    {
        const hipError_t e = used_ ? hipStreamSynchronize(used_) : hipSuccess;
        used_ = nullptr;
        return e == hipSuccess ? int(CUTE_OK) : hip_fail(e, "waiting for the side stream", __LINE__);
    }
};

inline dim3 panel_grid(uint32_t n) { return dim3(std::min(n, cute_build::kPanelRow), (n + cute_build::kPanelRow - 1u) / cute_build::kPanelRow); }
inline dim3 grid_of(uint64_t n) { return dim3(uint32_t(std::max<uint64_t>((n + cute_build::kThreads - 1) / cute_build::kThreads, 1))); }
// for kernels that walk their range with a stride
inline dim3 grid_capped(uint64_t n) { return dim3(std::min<uint32_t>(grid_of(n).x, 4096u)); }

int check_launch(const char *what);

#define CUTE_BUILD(kernel, grid, ...) CUTE_BUILD_LDS(kernel, grid, 0, __VA_ARGS__)
#define CUTE_BUILD_LDS(kernel, grid, lds, ...) hipLaunchKernelGGL(kernel, grid, dim3(cute_build::kThreads), lds, nullptr, __VA_ARGS__)
// a panel kernel of the given capacity over `count` panels: all of them, or a list
#define CUTE_PANELS(kernel, CAP, count, lds, stream, ...) \
    hipLaunchKernelGGL(kernel, panel_grid(count), dim3(cute_build::panel_threads(CAP)), lds, stream, __VA_ARGS__)

// The widest column window the panel kernels take on this matrix, and the LDS its bitmap and running counts need.
inline uint32_t max_span(const cute_hrpb_dev *d) { return std::min(d->K, cute_build::kPanelSpan); }
inline uint32_t window_lds(uint32_t span, uint32_t at_least) { return std::max(cute_build::window_room(span) / 2u * 9u, at_least); }
// No panel that the panel kernels take has a wider window: the widest of a tile of panels, which the census loop knows.
inline uint32_t widest_span(const cute_hrpb_dev *d) { return std::max(1u, std::min(max_span(d), d->widestTile)); }
constexpr const uint32_t *kAllPanels = nullptr;
inline bool panel_is_large(const cute_hrpb_dev *d, uint32_t p) { return d->panelNnz[p] > cute_build::kPanelCap || d->panelSpan[p] > max_span(d); }

// Words of scratch device_scan needs for an array of n values: the block sums of every level.
inline uint64_t scan_scratch_words(uint64_t n)
{
    uint64_t words = 0;
    while (n > cute_build::kScanBlock) { n = (n + cute_build::kScanBlock - 1) / cute_build::kScanBlock; words += n; }
    return words + 1;
}

// Inclusive prefix sums of n uint32 values, in place, on the default stream, for `arrays` arrays that stand `pitch` words apart
// (their scratch `scratch_pitch`).
void device_scan(uint32_t *data, uint64_t n, uint32_t *scratch, uint32_t arrays = 1, uint64_t pitch = 0, uint64_t scratch_pitch = 0)
{
    if (!n) return;
    const uint64_t nb = (n + cute_build::kScanBlock - 1) / cute_build::kScanBlock;
    const dim3 grid(uint32_t(nb), arrays);
    const uint32_t *sums = nullptr;
    if (nb > 1) {
        CUTE_BUILD(cute_build::scan_block_sums, grid, data, n, pitch, scratch, scratch_pitch);
        device_scan(scratch, nb, scratch + nb, arrays, scratch_pitch, scratch_pitch);
        sums = scratch;
    }
    CUTE_BUILD(cute_build::scan_block_apply, grid, data, n, pitch, sums, scratch_pitch);
}

// The panels that a launch over all panels leaves out because they hold more than `cap` entries, though a panel kernel takes them.
std::vector<uint32_t> panels_between(const cute_hrpb_dev *d, uint32_t cap)
{
    std::vector<uint32_t> list;
    for (uint32_t p = 0; d->longestPanel > cap && p < d->P; ++p)
        if (d->panelNnz[p] > cap && !panel_is_large(d, p)) list.push_back(p);
    return list;
}

// The panels that the panel kernels do not take and what their entry-parallel path keeps between its kernels.
struct LargeWork {
    std::vector<uint32_t> panel, prefix;
    DevBuf memory;
    cute_build::LargePanels L{};
    uint32_t *posP = nullptr, *posS = nullptr, *DP = nullptr, *DS = nullptr, *scratch = nullptr;
    cute_build::PanelCensus *res = nullptr;
};

// Lists the large panels (panelNnz and panelSpan are known).
void list_large_panels(const cute_hrpb_dev *d, LargeWork &w)
{
    if (!w.prefix.empty()) return;
    w.prefix.assign(1, 0u);
    if (!d->anyLarge) return;
    for (uint32_t p = 0; p < d->P; ++p)
        if (panel_is_large(d, p)) {
            w.panel.push_back(p);
            w.prefix.push_back(w.prefix.back() + d->panelNnz[p]);
        }
}

// The LDS that big_quads asks for beside its static part (a kilobyte at most) is a compute unit's whatever the matrix: a byte a column of a
// strip and three words for every 64 columns.
constexpr uint32_t kBigWindow = cute_build::big_window_words(cute_build::panel_window_words(cute_build::kPanelSpan));
static_assert((kBigWindow + cute_build::kBigEntries / 4u + cute_build::kBigEntries / 64u * 3u) * 4u + 1024u <= 160u << 10, "big_quads");

// Does big_quads take every large panel?  One panel beyond kBigEntries or kPanelSpan sends all large panels of the matrix to the entry-parallel path.
bool big_takes_all(const cute_hrpb_dev *d, const LargeWork &w)
{
    for (uint32_t p : w.panel)
        if (d->panelNnz[p] > cute_build::kBigEntries || d->panelSpan[p] > max_span(d)) return false;
    return true;
}

// The strips that panel_quads<true> takes beside whole panels (of up to kPanelList entries) and the longer ones, for big_quads: those of
// every panel of more than kPanelList entries, but of large panels only where big_quads takes them all.
struct StripLists {
    std::vector<uint32_t> strips, big;        // 4 panel + strip, cute_build::kHasZeros where the panel has entries of value zero
    uint32_t bigRows = 0, bigSteps = 0;       // LDS words of big_quads: a byte a column of the longest strip, and its steps of 64 columns
};

StripLists list_strips(const cute_hrpb_dev *d, bool with_large)
{
    StripLists l;
    auto next = d->longStrips.begin();
    for (uint32_t p = 0; d->longestPanel > cute_build::kPanelList && p < d->P; ++p) {
        if (d->panelNnz[p] <= cute_build::kPanelList || (!with_large && panel_is_large(d, p))) continue;
        const uint32_t zeros = d->panelStored[p] != d->panelNnz[p] ? cute_build::kHasZeros : 0u;
        for (uint32_t u = 4u * p; u < 4u * p + 4u; ++u) {
            if (!d->stripPairs[u]) continue;
            while (next != d->longStrips.end() && *next < u) ++next;
            if (next == d->longStrips.end() || *next != u) { l.strips.push_back(u | zeros); continue; }
            l.big.push_back(u | zeros);
            l.bigRows = std::max(l.bigRows, (d->stripPairs[u] + 3u) / 4u);
            l.bigSteps = std::max(l.bigSteps, (d->stripPairs[u] + 63u) / 64u * 3u);
        }
    }
    return l;
}

// Numbers the entries of the large panels.  With `out` given also counts for the planner, into the panels' census records.
int number_large_panels(const cute_hrpb_dev *d, LargeWork &w, cute_build::PanelCensus *out)
{
    list_large_panels(d, w);
    const uint32_t count = uint32_t(w.panel.size()), total = w.prefix.back();
    if (!count || w.posP) return CUTE_OK;
    Layout lay;
    const uint64_t oPanel = lay.add(count, 4), oPrefix = lay.add(count + 1u, 4), oRes = lay.add(count, sizeof(cute_build::PanelCensus));
    const uint64_t staged = lay.bytes;
    const uint64_t oPosP = lay.add(total, 4), oPosS = lay.add(total, 4), oDP = lay.add(total, 4), oDS = lay.add(total, 4),
                   oScratch = lay.add(2u * scan_scratch_words(total), 4);
    int rc = w.memory.alloc(lay.bytes);
    PinnedBuf pin;
    if (rc == CUTE_OK) rc = pin.alloc(staged);
    if (rc != CUTE_OK) return rc;
    std::memset(pin.p, 0, staged);
    std::memcpy(pin.as<char>(oPanel), w.panel.data(), count * 4u);
    std::memcpy(pin.as<char>(oPrefix), w.prefix.data(), (count + 1u) * 4u);
    void *m = w.memory.p;
    w.L = {Layout::at<uint32_t>(m, oPanel), Layout::at<uint32_t>(m, oPrefix), count, total};
    w.posP = Layout::at<uint32_t>(m, oPosP); w.posS = Layout::at<uint32_t>(m, oPosS);
    w.DP = Layout::at<uint32_t>(m, oDP); w.DS = Layout::at<uint32_t>(m, oDS);
    w.scratch = Layout::at<uint32_t>(m, oScratch);
    w.res = Layout::at<cute_build::PanelCensus>(m, oRes);
    pin.pending = true;
    CUTE_BUILD(cute_build::copy_words, grid_capped(staged / 4u), pin.as<const uint32_t>(), w.memory.as<uint32_t>(), staged / 4u);
    CUTE_BUILD(cute_build::large_positions, grid_of(total), w.L, d->dRowPtr, d->dCols, d->dCsrVals, d->K, w.posP, w.posS, w.DP, w.DS,
               out ? w.res : static_cast<cute_build::PanelCensus *>(nullptr));
    device_scan(w.DP, total, w.scratch, 2, (oDS - oDP) / 4u, scan_scratch_words(total));
    if (out) CUTE_BUILD(cute_build::large_counts, grid_of(count), w.L, d->dRowPtr, w.DP, w.DS, w.res, out);
    rc = check_launch("large panels");
    return rc == CUTE_OK ? pin.wait() : rc;
}

// Up to this many panels the layout builders read their tables where the host wrote them: no copy_words launch in front of them (4 us and the
// gap behind it), for a read of 1.5 us a work-group that waits for nothing until the panel's columns are numbered.  Format to product, copied / in
// place: 9-point stencils of 64 x 64 points 77.6 / 75.7, 300 x 300 (5 625 panels) 217 / 215, 500 x 500 (15 625 panels, whose reads
// add up) 486 / 492 us.  Nothing stands between the launches then, and those for longer panels go to the side stream.
constexpr uint32_t kTablesInPlace = 8192;

// Brick tiles from the device CSR copy: the arrays cute_hrpb_retile makes on the host, word for word.
int build_bricks_on_device(cute_hrpb_dev *d, LargeWork &w)
{
    int rc = number_large_panels(d, w, nullptr);
    if (rc != CUTE_OK) return rc;
    const uint64_t hdr_words = uint64_t(d->nb) * CUTE_TILED_HDR_WORDS, num_vals = uint64_t(d->nnz) + 64u;
    const uint32_t count = uint32_t(w.panel.size()), span = widest_span(d);
    Layout lay, tab;
    const uint64_t oBrp = tab.add(uint64_t(d->P) + 1u, 4), oUnit = tab.add(count, 4), oPrefix = tab.add(count + 1u, 4), oCols = tab.add(count, 4);
    const std::vector<uint32_t> medium = panels_between(d, cute_build::kPanelFirst);
    const uint64_t oMedium = tab.add(medium.size(), 4);
    const uint64_t oHdr = lay.add(hdr_words, 4), oVals = lay.add(num_vals, 4), oTab = lay.add(tab.bytes, 1);
    DevBuf mem;
    PinnedBuf pin;
    rc = mem.alloc(lay.bytes);
    if (rc == CUTE_OK) rc = pin.alloc(tab.bytes);
    if (rc != CUTE_OK) return rc;
    const bool in_place = !count && d->P <= kTablesInPlace;
    auto table = [&](uint64_t o) { return in_place ? pin.as<const uint32_t>(o) : Layout::at<const uint32_t>(mem.p, oTab + o); };
    SideStream side;
    uint32_t *hdr = Layout::at<uint32_t>(mem.p, oHdr);
    float *vals = Layout::at<float>(mem.p, oVals);
    std::memcpy(pin.p, d->brp.data(), d->brp.size() * 4u);
    if (!medium.empty()) std::memcpy(pin.as<char>(oMedium), medium.data(), medium.size() * 4u);
    uint32_t *unit = pin.as<uint32_t>(oUnit), *prefix = pin.as<uint32_t>(oPrefix), *cols = pin.as<uint32_t>(oCols);
    prefix[0] = 0;
    for (uint32_t k = 0; k < count; ++k) {
        const uint32_t p = w.panel[k];
        unit[k] = d->brp[p];
        prefix[k + 1] = prefix[k] + (d->brp[p + 1] - d->brp[p]);
        cols[k] = d->panelCols[p];
    }
    pin.pending = true;
    if (!in_place)
        CUTE_BUILD(cute_build::copy_words, grid_capped(tab.bytes / 4u), pin.as<const uint32_t>(), Layout::at<uint32_t>(mem.p, oTab), tab.bytes / 4u);
#define CUTE_PANEL_BRICKS(CAP, COUNT, STREAM, LIST)                                                                                    \
    CUTE_PANELS(cute_build::panel_bricks<CAP>, CAP, COUNT, window_lds(span, (CAP + 1u) * 2u), STREAM, d->dRowPtr, d->dCols, d->dCsrVals, d->P, d->nnz,  \
                span, LIST, table(oBrp), hdr, vals)
    if (d->longestPanel <= cute_build::kPanelShort) CUTE_PANEL_BRICKS(cute_build::kPanelShort, d->P, nullptr, kAllPanels);
    else CUTE_PANEL_BRICKS(cute_build::kPanelFirst, d->P, nullptr, kAllPanels);
    if (!medium.empty()) CUTE_PANEL_BRICKS(cute_build::kPanelCap, uint32_t(medium.size()), in_place ? side.get() : nullptr, table(oMedium));
#undef CUTE_PANEL_BRICKS
    if (count) {
        const uint32_t blocks = prefix[count];
        CUTE_BUILD(cute_build::large_clear, grid_of(uint64_t(blocks) * CUTE_TILED_HDR_WORDS), table(oUnit), table(oPrefix), count, uint32_t(CUTE_TILED_HDR_WORDS), hdr);
        CUTE_BUILD(cute_build::large_bricks, grid_of(w.L.total), w.L, d->dRowPtr, d->dCols, d->dCsrVals, w.posP, w.DP, table(oUnit), hdr, vals);
        CUTE_BUILD(cute_build::large_brick_ends, grid_of(blocks), w.L, d->dRowPtr, table(oUnit), table(oPrefix), table(oCols), hdr);
    }
    rc = check_launch("brick tiles");
    if (rc == CUTE_OK) rc = pin.wait();
    if (rc == CUTE_OK) rc = side.wait();
    if (rc != CUTE_OK) return rc;
    d->dHdr = hdr;
    d->dVals = vals;
    d->brickMemory = mem.release();
    d->bytes += hdr_words * 4u + num_vals * 4u;
    d->haveBricks = true;
    return CUTE_OK;
}

// Quad lists (in the layout the census chose) from the device CSR copy: the arrays cute_quad_pack makes.
int build_quads_on_device(cute_hrpb_dev *d, LargeWork &w)
{
    const uint64_t G = d->numGroups, stored = d->numQuadVals;
    const bool strips = d->quadRows == 4;
    list_large_panels(d, w);
    const bool with_large = strips && big_takes_all(d, w);
    const StripLists lists = strips ? list_strips(d, with_large) : StripLists();
    int rc = with_large ? int(CUTE_OK) : number_large_panels(d, w, nullptr);
    if (rc != CUTE_OK) return rc;
    const uint32_t count = with_large ? 0u : uint32_t(w.panel.size()), per = strips ? 4u : 1u, span = widest_span(d);
    Layout lay, tab;
    const uint64_t oGroup = tab.add(d->qgp.size(), 4), oBase = tab.add(uint64_t(d->P) + 1u, 4), oUnit = tab.add(count, 4),
                   oPrefix = tab.add(count + 1u, 4), oFirst = tab.add(uint64_t(count) * per, 4), oPairs = tab.add(uint64_t(count) * 4u, 4),
                   oLargeBase = tab.add(count, 4);
    const std::vector<uint32_t> medium = strips ? lists.strips : panels_between(d, cute_build::kPanelList);
    const uint64_t oMedium = tab.add(medium.size(), 4), oBig = tab.add(lists.big.size(), 4);
    const uint64_t oRecs = lay.add(G * CUTE_QUAD_RECORD_WORDS, 4), oVals = lay.add(stored + 64u, 4), oTab = lay.add(tab.bytes, 1);
    DevBuf mem, counts;
    PinnedBuf pin;
    rc = mem.alloc(lay.bytes);
    if (rc == CUTE_OK) rc = pin.alloc(tab.bytes);
    if (rc != CUTE_OK) return rc;
    const bool in_place = !count && d->P <= kTablesInPlace;
    auto table = [&](uint64_t o) { return in_place ? pin.as<const uint32_t>(o) : Layout::at<const uint32_t>(mem.p, oTab + o); };
    SideStream side;
    uint32_t *recs = Layout::at<uint32_t>(mem.p, oRecs);
    float *packed = Layout::at<float>(mem.p, oVals);
    std::memcpy(pin.as<char>(oGroup), d->qgp.data(), d->qgp.size() * 4u);
    if (!medium.empty()) std::memcpy(pin.as<char>(oMedium), medium.data(), medium.size() * 4u);
    if (!lists.big.empty()) std::memcpy(pin.as<char>(oBig), lists.big.data(), lists.big.size() * 4u);
    uint32_t *base = pin.as<uint32_t>(oBase), *unit = pin.as<uint32_t>(oUnit), *prefix = pin.as<uint32_t>(oPrefix), *first = pin.as<uint32_t>(oFirst),
             *pairs = pin.as<uint32_t>(oPairs), *large_base = pin.as<uint32_t>(oLargeBase);
    base[0] = 0;
    for (uint32_t p = 0; p < d->P; ++p) base[p + 1] = base[p] + d->panelStored[p];
    prefix[0] = 0;
    for (uint32_t k = 0; k < count; ++k) {
        const uint32_t p = w.panel[k];
        unit[k] = d->qgp[p * per];
        prefix[k + 1] = prefix[k] + (d->qgp[(p + 1) * per] - d->qgp[p * per]);
        for (uint32_t s = 0; s < per; ++s) first[k * per + s] = d->qgp[p * per + s];
        for (uint32_t s = 0; s < 4u; ++s) pairs[k * 4u + s] = d->stripPairs[p * 4u + s];
        large_base[k] = base[p];
    }
    const uint32_t groups = prefix[count];
    if (groups) rc = counts.alloc((uint64_t(groups) + scan_scratch_words(groups)) * 4u);
    if (rc != CUTE_OK) return rc;
    pin.pending = true;
    if (!in_place)
        CUTE_BUILD(cute_build::copy_words, grid_capped(tab.bytes / 4u), pin.as<const uint32_t>(), Layout::at<uint32_t>(mem.p, oTab), tab.bytes / 4u);
    uint32_t *sums = counts.as<uint32_t>();
    const uint32_t listed = uint32_t(medium.size());
#define CUTE_PANEL_QUADS(S, CAP, COUNT, LIST, LISTED, STREAM)                                                                         \
    CUTE_PANELS((cute_build::panel_quads<S, CAP>), CAP, COUNT, window_lds(span, CAP * 8u), STREAM, d->dRowPtr, d->dCols, d->dCsrVals, d->P, d->nnz,  \
                span, LIST, LISTED, table(oGroup), table(oBase), uint32_t(stored), recs, packed)
#define CUTE_BUILD_QUADS(S)                                                                                                           \
    if (d->longestPanel <= cute_build::kPanelShort) CUTE_PANEL_QUADS(S, cute_build::kPanelShort, d->P, kAllPanels, 0u, nullptr);            \
    else CUTE_PANEL_QUADS(S, cute_build::kPanelList, (S) ? d->P + listed : d->P, (S) ? table(oMedium) : kAllPanels, (S) ? listed : 0u, nullptr); \
    if constexpr (!(S))                                                                                                               \
        if (listed) CUTE_PANEL_QUADS(S, cute_build::kPanelCap, listed, table(oMedium), listed, in_place ? side.get() : nullptr);        \
    if (count) {                                                                                                                      \
        CUTE_BUILD(cute_build::large_clear, grid_of(uint64_t(groups) * CUTE_QUAD_RECORD_WORDS), table(oUnit), table(oPrefix), count,    \
                   uint32_t(CUTE_QUAD_RECORD_WORDS), recs);                                                                           \
        CUTE_BUILD((cute_build::large_quads<S, false>), grid_of(w.L.total), w.L, d->dRowPtr, d->dCols, d->dCsrVals, w.posS, w.DS,       \
                   table(oFirst), recs, packed);                                                                                      \
        CUTE_BUILD(cute_build::large_groups<S>, grid_of(groups), w.L, d->dRowPtr, d->dCols, table(oFirst), table(oPrefix), table(oPairs), recs, sums); \
        device_scan(sums, groups, sums + groups);                                                                                     \
        CUTE_BUILD(cute_build::large_first_values, grid_of(groups), table(oUnit), table(oPrefix), table(oLargeBase), count, sums, recs); \
        CUTE_BUILD((cute_build::large_quads<S, true>), grid_of(w.L.total), w.L, d->dRowPtr, d->dCols, d->dCsrVals, w.posS, w.DS,        \
                   table(oFirst), recs, packed);                                                                                      \
    }
    // (the strips that take longest go first)
    if (!lists.big.empty()) {
        const uint32_t words = cute_build::panel_window_words(span);
        hipLaunchKernelGGL(cute_build::big_quads, dim3(uint32_t(lists.big.size())), dim3(cute_build::kBigThreads),
                           (cute_build::big_window_words(words) + lists.bigRows + lists.bigSteps) * 4u, in_place ? side.get() : nullptr, d->dRowPtr, d->dCols, d->dCsrVals,
                           table(oBig), words, lists.bigRows, table(oGroup), table(oBase), recs, packed);
    }
    if (strips) { CUTE_BUILD_QUADS(true) } else { CUTE_BUILD_QUADS(false) }
#undef CUTE_BUILD_QUADS
#undef CUTE_PANEL_QUADS
    rc = check_launch("quad lists");
    if (rc == CUTE_OK) rc = pin.wait();
    if (rc == CUTE_OK) rc = side.wait();
    if (rc != CUTE_OK) return rc;
    d->dQRecs = recs;
    d->dQVals = packed;
    d->quadMemory = mem.release();
    d->bytes += G * CUTE_QUAD_RECORD_WORDS * 4u + (stored + 64u) * 4u;
    d->haveQuads = true;
    return CUTE_OK;
}

// A layout the upload did not build: made on the device from the device copy of the CSR arrays (the host
// arrays the format borrowed may be gone by now).  which: 1 brick tiles, 2 quad lists.
int ensure_layout(cute_hrpb_dev *d, int which)
{
    std::lock_guard<std::mutex> guard(d->lock);
    if (which == 1 ? d->haveBricks : d->haveQuads) return CUTE_OK;
    LargeWork w;
    return which == 1 ? build_bricks_on_device(d, w) : build_quads_on_device(d, w);
}

// What csr_rows_window wants to know of a matrix: of every slice of 64 rows, where its quads begin and how many its longest row takes
// (one at least), and the column window of every tile, widened so that neither end moves back from one tile to the next.
struct WindowShape {
    std::vector<uint4> slices;            // {first quad, -, quads, -}
    std::vector<uint2> tiles;             // {first column, column behind the last}
    uint64_t quads = 0;
    uint32_t longest = 0, widest = 0;
};

// false: rows or windows that the kernel does not take
bool window_shape(const cute_hrpb_dev *d, WindowShape &w)
{
    constexpr uint32_t per_slice = 64u / CUTE_TM;
    w.slices.resize((size_t(d->P) + per_slice - 1) / per_slice);
    w.tiles = d->tileWindow;
    for (uint32_t p = 0; p < d->P;) {
        uint4 &slice = w.slices[p / per_slice];
        uint32_t longest = 1;
        for (const uint32_t upto = std::min<uint32_t>(d->P, p + per_slice); p < upto; ++p) longest = std::max(longest, d->panelMaxRow[p]);
        if (longest > 64u) return false;
        w.longest = std::max(w.longest, longest);
        slice = make_uint4(uint32_t(w.quads), 0u, (longest + 3u) / 4u, 0u);
        w.quads += (longest + 3u) / 4u;
    }
    uint32_t first = d->K, end = 0;
    for (uint2 &tile : w.tiles) tile.y = end = std::max(end, tile.y);
    for (size_t t = w.tiles.size(); t-- > 0;) {
        first = std::min(first, w.tiles[t].x);
        w.tiles[t].x = std::min(first, w.tiles[t].y);
        w.widest = std::max(w.widest, w.tiles[t].y - w.tiles[t].x);
    }
    return w.widest <= cute_dev::kWindowRows<8> && w.quads <= 0xffffffffull;
}

// The entries csr_rows_window reads, for a ring of `ring_rows` rows (which follows from the widest window, so a handle has one such form).
// CUTE_ERR_NOMEM: there is no memory for them.
int ensure_window(cute_hrpb_dev *d, const WindowShape &w, uint32_t ring_rows)
{
    std::lock_guard<std::mutex> guard(d->lock);
    if (d->haveWindow) return CUTE_OK;
    Layout lay;
    const uint64_t oSlices = lay.add(w.slices.size(), sizeof(uint4)), oTiles = lay.add(w.tiles.size(), sizeof(uint2)), staged = lay.bytes;
    const uint64_t oSlots = lay.add(w.quads * 64u, sizeof(uint2)), oVals = lay.add(w.quads * 64u, 16u);
    DevBuf mem;
    PinnedBuf pin;
    int rc = mem.alloc(lay.bytes);
    if (rc == CUTE_OK) rc = pin.alloc(staged);
    if (rc != CUTE_OK) return g_hip_status == hipErrorOutOfMemory ? int(CUTE_ERR_NOMEM) : rc;
    std::memcpy(pin.as<char>(oSlices), w.slices.data(), w.slices.size() * sizeof(uint4));
    std::memcpy(pin.as<char>(oTiles), w.tiles.data(), w.tiles.size() * sizeof(uint2));
    pin.pending = true;
    const uint32_t longest = (w.longest + 3u) & ~3u;
    const cute_build::WindowTables T = {pin.as<const uint4>(oSlices), pin.as<const uint2>(oTiles), uint32_t(w.tiles.size()),
                                        Layout::at<uint4>(mem.p, oSlices), Layout::at<uint2>(mem.p, oTiles)};
    CUTE_BUILD_LDS(cute_build::window_entries, dim3(uint32_t(w.slices.size())), cute_build::window_entries_lds(longest), d->dRowPtr, d->dCols,
                   d->dCsrVals, d->M, ring_rows, T, longest, Layout::at<uint2>(mem.p, oSlots), Layout::at<cute_dev::f32x4>(mem.p, oVals));
    rc = check_launch("window entries");
    if (rc == CUTE_OK) rc = pin.wait();
    if (rc != CUTE_OK) return rc;
    d->dSlices = Layout::at<uint4>(mem.p, oSlices);
    d->dWindowTiles = Layout::at<uint2>(mem.p, oTiles);
    d->dWindowSlots = Layout::at<uint2>(mem.p, oSlots);
    d->dWindowVals = Layout::at<cute_dev::f32x4>(mem.p, oVals);
    d->windowMemory = mem.release();
    d->bytes += lay.bytes;
    d->haveWindow = true;
    return CUTE_OK;
}

// Group counts of the quad lists from the list length of every strip; picks lockstep lists unless they would
// be mostly padding (a few very long rows stretch the lists of their panel neighbours): then one list per strip.
int finish_quad_census(cute_hrpb_dev *d, int quad_layout)
{
    const uint32_t *const pairs_of = d->stripPairs.data(), P = d->P;
    uint64_t pairs = 0, lock_groups = 0, strip_groups = 0;
    for (uint32_t p = 0; p < P; ++p) {
        const uint32_t a = pairs_of[4 * p], b = pairs_of[4 * p + 1], c = pairs_of[4 * p + 2], e = pairs_of[4 * p + 3];
        pairs += uint64_t(a) + b + c + e;
        lock_groups += (std::max(std::max(a, b), std::max(c, e)) + 3) / 4;
        strip_groups += uint64_t((a + 15) / 16) + (b + 15) / 16 + (c + 15) / 16 + (e + 15) / 16;
    }
    if (quad_layout == 0) quad_layout = (lock_groups && double(pairs) < 0.6 * 16.0 * double(lock_groups)) ? 2 : 1;
    const bool strips = quad_layout == 2;
    d->quadRows = strips ? 4u : CUTE_TM;
    d->quadPairs = pairs;
    d->numGroups = strips ? strip_groups : lock_groups;
    if (d->numGroups > 0xffffffffull / 64) return CUTE_ERR_SHAPE;
    d->qgp.resize((strips ? size_t(P) * 4u : size_t(P)) + 1);
    uint32_t *const qgp = d->qgp.data(), groups = 0;
    qgp[0] = 0;
    for (uint32_t p = 0; p < P; ++p) {
        const uint32_t *const of = pairs_of + 4 * size_t(p);
        if (!strips) qgp[p + 1] = groups += (std::max(std::max(of[0], of[1]), std::max(of[2], of[3])) + 3) / 4;
        else
            for (uint32_t l = 0; l < 4u; ++l) qgp[4 * size_t(p) + l + 1] = groups += (of[l] + 15) / 16;
    }
    return CUTE_OK;
}

// Which MFMA layout would the planner's default rules use for this matrix (see cute_spmm_plan_create)?
// 0: none (every panel would go to the row kernel), 1 brick tiles, 2 quad lists.
int default_layout(const cute_hrpb_dev *d, uint64_t cache_bytes)
{
    const uint32_t lists = d->quadRows == 4 ? 4u : 1u;
    uint64_t slots = 0, bricks = 0, blocks = 0, entries = 0;
    for (uint32_t q = 0; q < d->P; ++q) {
        if (d->brp[q + 1] == d->brp[q]) continue;
        const uint32_t list_slots = (d->qgp[(q + 1) * lists] - d->qgp[q * lists]) * 16u;
        const uint32_t fetches = std::max(d->panelCols[q], list_slots);
        if (float(d->panelNnz[q]) < kMinReuse * float(fetches) && d->panelMaxRow[q] <= kMaxRowForRows) continue;   // row kernel
        slots += list_slots;
        entries += d->panelNnz[q];
        bricks += (d->panelCols[q] + 3u) / 4u;
        blocks += d->brp[q + 1] - d->brp[q];
    }
    if (!bricks) return 0;
    // (the width is not known yet: 128 columns stand in for it)
    return choose_mfma_shape(slots, bricks, blocks, entries, uint64_t(d->K) + d->M, d->nnz, 128u, 0u, cache_bytes);
}

int alloc_csr(cute_hrpb_dev *d)
{
    Layout lay;
    const uint64_t oRow = lay.add(uint64_t(d->M) + 1u, 4), oCols = lay.add(uint64_t(d->nnz) + kRowBatch, 4),
                   oVals = lay.add(uint64_t(d->nnz) + kRowBatch, 4);     // the row kernel reads whole batches
    const int rc = pool().take(&d->csrMemory, lay.bytes);
    if (rc != CUTE_OK) return rc;
    d->dRowPtr = Layout::at<uint32_t>(d->csrMemory, oRow);
    d->dCols = Layout::at<uint32_t>(d->csrMemory, oCols);
    d->dCsrVals = Layout::at<float>(d->csrMemory, oVals);
    d->bytes = (uint64_t(d->M) + 1) * 4 + uint64_t(d->nnz) * 8;
    return CUTE_OK;
}

// Host arrays to the device through pinned memory, piece by piece: the host threads fill a piece while a kernel reads
// the one before.  When the buffer is full the stream is waited for and the buffer used again.
struct HostToDevice {
    static constexpr uint64_t kPiece = 2ull << 20;
    PinnedBuf pin;
    uint64_t used = 0;
    int begin(uint64_t bytes) { return pin.alloc(std::min<uint64_t>((bytes + kPiece - 1) / kPiece * kPiece + kPiece, 16ull << 20)); }
    int copy(void *dst, const void *src, uint64_t bytes)
    {
        for (uint64_t at = 0; at < bytes;) {
            if (used + kPiece > pin.cap) {
                const int rc = pin.wait();
                if (rc != CUTE_OK) return rc;
                used = 0;
            }
            const uint64_t n = std::min(kPiece, bytes - at);
            parallel_ranges(n, 256u << 10, [&](uint64_t b, uint64_t e, unsigned) { std::memcpy(pin.as<char>(used + b), static_cast<const char *>(src) + at + b, e - b); });
            pin.pending = true;
            CUTE_BUILD(cute_build::copy_words, grid_capped(n / 4u), pin.as<const uint32_t>(used), Layout::at<uint32_t>(dst, at), n / 4u);
            used += (n + 255u) & ~uint64_t(255);
            at += n;
        }
        return CUTE_OK;
    }
};

// The census of every panel into `records`; a caller's arrays are copied to d's own.
void launch_census(const cute_hrpb_dev *d, const uint32_t *rowPtr, const uint32_t *cols, const float *vals, cute_build::PanelCensus *records)
{
    const uint32_t P = d->P;
    const cute_build::CsrCopy to = {d->dRowPtr, d->dCols, d->dCsrVals};
    const bool copy = rowPtr != d->dRowPtr;
    if (uint64_t(d->nnz) <= uint64_t(P) * cute_build::kWaveMean) {
        const uint32_t quarter = (P + 3u) / 4u, skew = uint32_t(uint64_t(quarter) * 3u / 10u),
                       front = P <= cute_build::kWaveFront ? P : quarter;
        const uint32_t lds_words = cute_build::wave_census_words(max_span(d));
        if (copy)
            CUTE_BUILD_LDS(cute_build::panel_census_waves<true>, panel_grid(front + quarter), lds_words * 4u, rowPtr, cols, vals, P, d->K, d->nnz, max_span(d), lds_words,
                           quarter, skew, front, to, records);
        else
            CUTE_BUILD_LDS(cute_build::panel_census_waves<false>, panel_grid(front + quarter), lds_words * 4u, rowPtr, cols, vals, P, d->K, d->nnz, max_span(d), lds_words,
                           quarter, skew, front, to, records);
    } else {
        const uint32_t lds_words = cute_build::census_words(max_span(d)), share = uint32_t((uint64_t(d->nnz) + P - 1u) / P);
        if (copy)
            CUTE_BUILD_LDS(cute_build::panel_census<true>, panel_grid(P), lds_words * 4u, rowPtr, cols, vals, P, d->K, d->nnz, max_span(d), lds_words, share, to, records);
        else
            CUTE_BUILD_LDS(cute_build::panel_census<false>, panel_grid(P), lds_words * 4u, rowPtr, cols, vals, P, d->K, d->nnz, max_span(d), lds_words, share, to, records);
    }
}

// The common tail of both uploads.  The CSR arrays are on their way to the device (default stream): to d's own, or they are the caller's and
// the census copies them.  Checks them, counts what
// the planner wants to know about every panel, and builds the one MFMA layout the planner's default rules would use for
// this matrix (none when every panel would go to the row kernel).
int finish_upload(cute_hrpb_dev *d, int quad_layout, const DeviceContext &c, const uint32_t *rowPtr, const uint32_t *cols, const float *vals)
{
    const uint32_t P = d->P;
    LargeWork large;
    {
        PinnedBuf pin;
        int rc = pin.alloc((uint64_t(P) + kTilePanels) * sizeof(cute_build::PanelCensus));      // (the loop below asks for records ahead of it)
        if (rc != CUTE_OK) return rc;
        pin.pending = true;
        launch_census(d, rowPtr, cols, vals, pin.as<cute_build::PanelCensus>());
        rc = check_launch("panel census");
        if (rc == CUTE_OK) rc = pin.wait();
        if (rc != CUTE_OK) return rc;
        const cute_build::PanelCensus *r = pin.as<const cute_build::PanelCensus>();
        uint32_t error = 0;
        bool any_large = false, any_left = false;      // panels for the lists' entry-parallel or long kernels; panels the census leaves to number_large_panels
        uint32_t longest = 0;
        d->panelNnz.resize(P);
        d->panelSpan.resize(P);
        // (a pair for 64 panels, not a word a panel: that cost a small new matrix 1 to 3 % of its way from format to product, 23 616 rows
        // of 5, N = 8, 63.5 -> 65.3 us)
        d->tileWindow.resize((size_t(P) + kTilePanels - 1) / kTilePanels);
        for (uint32_t p = 0; p < P;) {
            uint2 tile = make_uint2(~0u, 0u), &into = d->tileWindow[p / kTilePanels];
            for (const uint32_t last = std::min(P, p + kTilePanels); p < last; ++p) {
                __builtin_prefetch(r + p + kTilePanels);
                const uint32_t flags = r[p].error;
                error |= flags & cute_build::kAnyError;
                if (flags >= cute_build::kLongStrip)
                    for (uint32_t s = 0; s < 4u; ++s)
                        if (flags & (cute_build::kLongStrip << s)) d->longStrips.push_back(4u * p + s);
                d->panelNnz[p] = r[p].nnz;
                d->panelSpan[p] = r[p].span;
                longest = std::max(longest, r[p].nnz);
                tile.x = std::min(tile.x, r[p].first);
                tile.y = std::max(tile.y, r[p].end);
                if (panel_is_large(d, p)) {
                    any_large = true;
                    any_left = any_left || r[p].nnz > cute_build::kBigEntries || r[p].span > max_span(d);
                }
            }
            into = tile;
            if (tile.y) d->widestTile = std::max(d->widestTile, tile.y - tile.x);
        }
        d->longestPanel = longest;
        d->anyLarge = any_large;
        if (!error && any_left) {
            rc = number_large_panels(d, large, pin.as<cute_build::PanelCensus>());
            if (rc != CUTE_OK) return rc;
            for (uint32_t p : large.panel) error |= r[p].error & cute_build::kAnyError;
        }
        if (error & cute_build::kErrRange) return CUTE_ERR_RANGE;
        if (error & cute_build::kErrUnsorted) return CUTE_ERR_UNSORTED;
        d->brp.resize(size_t(P) + 1);
        d->panelCols.resize(P);
        d->panelMaxRow.resize(P);
        d->panelStored.resize(P);
        d->stripPairs.resize(size_t(P) * 4u);
        uint64_t blocks = 0;
        d->brp[0] = 0;
        d->numQuadVals = 0;
        for (uint32_t p = 0; p < P; ++p) {
            d->panelCols[p] = r[p].cols;
            d->panelMaxRow[p] = r[p].maxRow;
            d->panelStored[p] = r[p].stored;
            d->numQuadVals += r[p].stored;
            for (uint32_t s = 0; s < 4u; ++s) d->stripPairs[4u * p + s] = r[p].pairs[s];
            blocks += (r[p].cols + CUTE_TK - 1) / CUTE_TK;
            if (blocks > 0xffffffffull / CUTE_TILED_HDR_WORDS) return CUTE_ERR_SHAPE;
            d->brp[p + 1] = uint32_t(blocks);
        }
        d->nb = uint32_t(blocks);
    }
    int rc = finish_quad_census(d, quad_layout);
    if (rc != CUTE_OK) return rc;
    const int which = default_layout(d, c.cache_bytes);
    if (which == 2) rc = build_quads_on_device(d, large);
    else if (which == 1) rc = build_bricks_on_device(d, large);
    return rc;
}

// Tables of a hub plan: the hub_rows most referenced columns of the quad records (ties: the lower column) get
// the slots 0.. of the LDS table; the plan keeps their column ids in slot order and its own copy of the records
// in which those columns name their slot.
int make_hub_tables(cute_spmm_plan *p, const cute_hrpb_dev *d, uint32_t hub_rows)
{
    const uint64_t G = d->numGroups;
    DevBuf counts, slots;
    int rc = counts.alloc(uint64_t(d->K) * 4u);
    if (rc == CUTE_OK) rc = slots.alloc(uint64_t(d->K) * 4u);
    if (rc != CUTE_OK) return rc;
    HIP_TRY(hipMemset(counts.p, 0, uint64_t(d->K) * 4u));
    hipLaunchKernelGGL(cute_build::count_record_columns, grid_of(G * 16u), dim3(cute_build::kThreads), 0, nullptr, d->dQRecs, G,
                       counts.as<uint32_t>());
    std::vector<uint32_t> cnt(d->K), order(d->K), slot_of(d->K, ~0u);
    HIP_TRY(hipMemcpy(cnt.data(), counts.p, uint64_t(d->K) * 4u, hipMemcpyDeviceToHost));
    for (uint32_t k = 0; k < d->K; ++k) order[k] = k;
    std::partial_sort(order.begin(), order.begin() + hub_rows, order.end(),
                      [&](uint32_t a, uint32_t b) { return cnt[a] != cnt[b] ? cnt[a] > cnt[b] : a < b; });
    uint32_t used = 0;
    while (used < hub_rows && cnt[order[used]] > 1u) ++used;            // a row fetched once gains nothing from LDS
    if (!used) return CUTE_OK;
    for (uint32_t h = 0; h < used; ++h) slot_of[order[h]] = h;
    HIP_TRY(hipMemcpy(slots.p, slot_of.data(), uint64_t(d->K) * 4u, hipMemcpyHostToDevice));
    rc = upload(&p->dHubRows, order.data(), used);
    if (rc != CUTE_OK) return rc;
    HIP_TRY(device_malloc(reinterpret_cast<void **>(&p->dHubRecs), G * CUTE_QUAD_RECORD_WORDS * 4u));
    hipLaunchKernelGGL(cute_build::mark_hub_columns, grid_of(G * CUTE_QUAD_RECORD_WORDS), dim3(cute_build::kThreads), 0, nullptr,
                       d->dQRecs, G, slots.as<const uint32_t>(), uint32_t(cute_dev::kHubFlag), p->dHubRecs);
    rc = check_launch("hub records");
    if (rc != CUTE_OK) return rc;
    HIP_TRY(hipDeviceSynchronize());
    p->numHub = used;
    return CUTE_OK;
}

// How many lane groups share a row in csr_rows_split; 1: another kernel takes the rows.  Up to 8 columns, for rows of 24 entries or more on average, a
// lane group for three and a half to seven entries each: the four a lane has on their way are then nearly all used.  One row kernel or brick kernel / 4, 8,
// 16, 32 groups, us from a replayed graph: finite elements (rows of 60), 1 200 rows, N = 1 11.6 / 4.5, 3.2, 2.7, 2.7, 12 000 rows, N = 1 12.9 / 5.0, 3.8, 3.6, 3.6,
// N = 8 7.1 / 6.1, 4.6, 4.4, 5.1; rows of 32 in a band, 5 120 rows, N = 1 5.3 / 2.8, 2.6, 2.5, 2.7, 102 400 rows, N = 1 8.3 / 7.2, 5.9, 7.7, 10.8, N = 8
// 11.4 / 10.1, 9.7, 14.9, 26.7, N = 16 15.9 / 15.4, 16.5, 27.4.  Shorter rows gain little or lose: 20 000 rows of 16, N = 3 3.46 / 3.51; 100 000 rows of 8,
// N = 1 5.1 / 5.4; 9-point stencil of 500 x 500 points, N = 8 6.6 / 9.3.  Nor where one row is much longer than the others, for which the brick kernel cuts its
// panel: R-MAT graph of 32 768 nodes, N = 1 13.3 / 84, 43, 24, 14.  And the brick kernel, which fetches a row of B once for all rows of a panel, is ahead
// from three columns on where rows share columns and the launch no longer fits the device at once: finite elements, 48 000 rows, brick kernel / 16
// groups: N = 1 9.3 / 6.2, N = 3 9.3 / 9.9, N = 8 9.3 / 10.3; 500 000 rows of 32 in a band, N = 8 64.5 / 61.8.
// Nor, up to 55 entries a row, between launches that leave wavefront slots free (190 000 lanes) and matrices so large that the row kernel is slow, where a group
// more a row is more wavefronts and loads for the same entries: rows in a wide band, which share few columns, with two lanes a group (3 and 5 to 8 columns) or short
// rows and N = 4; bands of any width with two lanes where the groups' last turn leaves a lane in seven or more idle; columns at random, none shared, for N = 1 alone.
// Row kernel / groups: two lanes, N = 8, band of 400, 64 000 rows of 24 5.25 / 5.91, of 48 8.55 / 9.59, of 32 (every lane busy) 6.60 / 6.44, 128 000 of 24 8.51 / 10.05; band of
// 2 048, N = 5, 64 000 of 48 9.61 / 12.08, 32 000 of 32, N = 7 5.38 / 6.13; N = 4, 128 000 of 24 8.27 / 9.45, band of 800, 72 000 of 30 7.93 / 5.26; random, 64 000 of 32,
// N = 1 8.72 / 9.83, N = 5 13.2 / 12.2.  Beyond: band of 400, N = 8, 256 000 rows of 32 30.1 / 24.2.
uint32_t row_parts(const cute_hrpb_dev *d, uint32_t N)
{
    const uint64_t nnz = d->nnz, M = d->M;
    if (N > 8u || nnz < 24u * M) return 1u;
    uint32_t longest = 0, parts = 4;
    uint64_t active = 0;
    for (uint32_t q = 0; q < d->P; ++q) {
        longest = std::max(longest, d->panelMaxRow[q]);
        active += d->panelCols[q];
    }
    while (parts < 16u && nnz >= 7u * parts * M) parts *= 2u;
    const bool two = N > 4u || N == 3u;
    const uint64_t lanes = M * parts * (two ? 2u : 1u);
    if (N > 2u && nnz >= 2u * active && lanes > 524288u) return 1u;
    if (parts < 16u && lanes > 190000u) {
        const uint64_t turn = 4u * parts * M, turns = (nnz + turn - 1u) / turn;
        const bool idle = 20u * nnz < 17u * turns * turn;
        const bool random = 50u * nnz < 51u * active, wide = !random && 10u * nnz < 11u * active;
        if (two ? !random && (wide || (idle && (parts == 4u || lanes > 524288u))) && (parts == 4u || lanes < 2000000u)
                : N == 4u ? wide && parts == 4u && nnz < 4000000u : N == 1u && random && nnz < 2300000u) return 1u;
    }
    // (a launch has at most 2^32 threads, of which a row takes parts, twice as many from two lanes a group on)
    return longest * M > 4u * nnz || M * parts * 2u > 0x7fffffffu ? 1u : parts;
}

// Rows of a plan without MFMA panels through csr_rows_window where that is ahead.  Needs the widest window of a tile to fit the ring,
// rows of up to 64 entries (the LDS of window_entries) and little padding: a lane waits for the longest of 64 rows.  Then both kernels'
// times are estimated, in us, and the ring has to be ahead by 15 %.  Fitted on 400 banded matrices drawn
// over 4 096 ... 640 000 rows, 8 ... 48 entries a row, bands of 64 ... 2 048 and N = 16 ... 600 (rms 18 and 14 % for rings of 8
// and 16 columns, 15 % for the row kernel): with a lead of 15 % and 12 us none was more than 2.5 % slower, and over all of them the
// products take 0.895 of the row kernel's time where the better of the two would take 0.869.  65 536 rows of 32, band of 2 048, us row
// kernel / ring: N = 32 12.4 / 14.8, N = 256 82.6 / 58.6; 16 rows N = 128 24.4 / 26.2; 262 144 rows of 12, band of 700, N = 128
// 72.7 / 76.3; 32 768 rows of 24, band of 1 500, N = 128 17.0 / 19.1; band of 200, 65 536 rows of 32, N = 101 39.0 / 25.1; 1 048 576
// rows of 32, band of 2 048, N = 256 1 714 / 1 005.
//
// A plan may be made for one product (a matrix that is new to every step), so the lead has to pay for the second form of the
// entries as well: plan creation with it takes, in us, 25 longer for 65 536 rows of 32 entries, 32 for 200 000 of 12, 33 for 131 072
// of 32, 42 for 262 144, 46 for 524 288, 186 for 1 048 576 (format, plan and one product of 65 536 rows, N = 256: 202 / 223; 80 000
// rows of 30, N = 101: 191 / 212).  Nearest to the line of 40 drawn matrices, 73 840 rows of 25, N = 423: 316 / 309, and 357 / 379 on
// buffers used for the first time.  A caller that says its product runs in a loop (operand_residency 2) gets the ring without that.
int plan_window(cute_spmm_plan *p, cute_hrpb_dev *d, uint32_t N, const DeviceContext &c, bool loop)
{
    // (beyond 32 768 columns the 1 024 threads of every slab of up to 512 chains could pass the 2^32 a launch may have)
    if (N < 16u || N > 32768u || d->P == 0) return CUTE_OK;
    const double bytes = 8.0 * d->M * N + 8.0 * d->nnz, gathers = 4e-6 * double(d->nnz) * N;
    const bool beyond = uint64_t(d->K + uint64_t(d->M)) * N * sizeof(float) > c.cache_bytes;
    const uint32_t walk = uint32_t(p->rows_vec) << p->rows_logl;       // columns a lane group covers, used or not
    const double covered = double((N + walk - 1u) / walk * walk) / N;
    const double rows = 3.1 + gathers / 20.0 * (0.29 + 0.40 * covered + (N % 32u ? 0.10 : 0.0)) + bytes * 1e-6 * (0.04 + (beyond ? 0.09 : 0.0));
    const double lead = loop ? 12.0 : 15.0 + 2e-3 * d->P + 3e-6 * double(d->nnz);
    const uint32_t n = (d->P + kTilePanels - 1u) / kTilePanels, cus = uint32_t(c.num_cus) / cute_dev::kNumXcd;
    // a CU holds one work-group at a time: `rounds` of them after each other, each a first window and then its tiles
    auto ring_time = [&](uint32_t W, double row) {
        const uint32_t slabs = (N + W - 1u) / W;
        const double first = W == 16u ? 0.8 : 2.0, tile = (W == 16u ? 3.8 + 0.245 * row : 2.6 + 0.143 * row) + (beyond ? (W == 16u ? 2.4 : 1.7) : 0.0);
        double ring = 0.0;
        for (uint32_t per_xcd = 1;; ++per_xcd) {
            const uint32_t chains = per_xcd * cute_dev::kNumXcd, length = (n + chains - 1u) / chains, rounds = (slabs * per_xcd + cus - 1u) / cus;
            const double time = rounds * (first + length * tile);
            if (per_xcd == 1 || time < ring) {
                ring = time;
                p->windowChains = chains;
                p->windowChainTiles = length;
            }
            if (length <= 1u || per_xcd == 64u) return ring;
        }
    };
    auto ahead = [&](double ring) { return ring * 1.15 <= rows && rows - ring >= lead; };
    // (what the widest tile and the mean row allow at best, before the panels are looked at)
    const double mean = double(d->nnz) / double(d->M);
    if (d->widestTile > cute_dev::kWindowRows<8> || rows < lead ||
        !(ahead(ring_time(8, mean)) || (d->widestTile <= cute_dev::kWindowRows<16> && ahead(ring_time(16, mean))))) return CUTE_OK;
    WindowShape w;
    if (!window_shape(d, w) || w.quads * 256u > uint64_t(d->nnz) + d->nnz / 4u + 4096u) return CUTE_OK;
    const uint32_t W = w.widest <= cute_dev::kWindowRows<16> ? 16u : 8u;
    if (!ahead(ring_time(W, double(w.quads) * 256.0 / double(d->M)))) return CUTE_OK;
    const int rc = ensure_window(d, w, W == 16u ? cute_dev::kWindowRows<16> : cute_dev::kWindowRows<8>);
    if (rc == CUTE_ERR_NOMEM) return CUTE_OK;       // the row kernel takes the rows, whose sums are then added in the order of the entries
    if (rc != CUTE_OK) return rc;
    p->windowColumns = W;
    p->windowWarm = beyond;
    return CUTE_OK;
}

}  // namespace

extern "C" {

int cute_hrpb_upload_layout(const cute_hrpb_host *h, int quad_layout, cute_hrpb_dev **out)
{
    if (!h || !out || !h->rowPtr || quad_layout < 0 || quad_layout > 2) return CUTE_ERR_ARG;
    *out = nullptr;
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    if (h->M == 0 || h->M % CUTE_TM || h->K % CUTE_TK) return CUTE_ERR_SHAPE;
    cute_hrpb_dev *d = new cute_hrpb_dev;
    d->M = h->M;
    d->K = h->K;
    d->nnz = h->nnz;
    d->P = h->numRowPanels;
    d->numVals = h->nnz;                     // the brick tiles store every entry of the matrix once
    int rc = alloc_csr(d);
    {
        HostToDevice up;
        if (rc == CUTE_OK) rc = up.begin(d->bytes);
        if (rc == CUTE_OK) rc = up.copy(d->dRowPtr, h->rowPtr, (uint64_t(h->M) + 1) * 4u);
        if (rc == CUTE_OK) rc = up.copy(d->dCols, h->cols, uint64_t(h->nnz) * 4u);
        if (rc == CUTE_OK) rc = up.copy(d->dCsrVals, h->vals, uint64_t(h->nnz) * 4u);
        if (rc == CUTE_OK) rc = finish_upload(d, quad_layout, c, d->dRowPtr, d->dCols, d->dCsrVals);
    }
    // the device counted the active columns itself: it must have found the blocks the canonical format has
    if (rc == CUTE_OK && (d->nb != h->numBlocks || std::memcmp(d->brp.data(), h->blockedRowPtr, d->brp.size() * sizeof(uint32_t)) != 0))
        rc = CUTE_ERR_FORMAT;
    if (rc != CUTE_OK) { cute_hrpb_dev_free(d); return rc; }
    *out = d;
    return CUTE_OK;
}

// The device-side counterpart of HRPB::HRPB + DATASTRUCT (data.cu:80-335, timed at run.cu:17-20) for a CSR
// matrix that already lives on the device: the handle keeps its own copy of the three arrays (device to
// device), the layouts are built by kernels, and only one 48-byte record per panel travels to the host.
int cute_hrpb_upload_device_csr(uint32_t M, uint32_t K, uint32_t nnz, const uint32_t *dRowPtr, const uint32_t *dCols,
                                const float *dVals, int quad_layout, cute_hrpb_dev **out)
{
    if (!out || !dRowPtr || (nnz && (!dCols || !dVals)) || quad_layout < 0 || quad_layout > 2) return CUTE_ERR_ARG;
    *out = nullptr;
    if (M == 0 || K == 0 || M % CUTE_TM || K % CUTE_TK) return CUTE_ERR_SHAPE;
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    cute_hrpb_dev *d = new cute_hrpb_dev;
    d->M = M; d->K = K; d->nnz = nnz; d->P = M / CUTE_TM;
    d->numVals = nnz;
    int rc = alloc_csr(d);
    if (rc == CUTE_OK) rc = finish_upload(d, quad_layout, c, dRowPtr, dCols, dVals);
    // (set-up itself waits for the default stream only; the interface promises the device)
    if (rc == CUTE_OK && !wait_for_device()) {
        const hipError_t e = hipDeviceSynchronize();     // (not a page left to free)
        if (e != hipSuccess) rc = hip_fail(e, "waiting for the device", __LINE__);
    }
    if (rc != CUTE_OK) { cute_hrpb_dev_free(d); return rc; }
    *out = d;
    return CUTE_OK;
}

// Sizes and host copies of what a device handle holds, for inspection and tests.  Layouts that were not built
// have size 0; pass nullptr for arrays that are not wanted.
int cute_hrpb_dev_layout_sizes(const cute_hrpb_dev *d, uint32_t *numBlocks, uint64_t *numTileVals, uint64_t *numGroups,
                               uint64_t *numQuadVals, uint32_t *rowsPerList)
{
    if (!d) return CUTE_ERR_ARG;
    if (numBlocks) *numBlocks = d->haveBricks ? d->nb : 0u;
    if (numTileVals) *numTileVals = d->haveBricks ? d->numVals : 0u;
    if (numGroups) *numGroups = d->haveQuads ? d->numGroups : 0u;
    if (numQuadVals) *numQuadVals = d->haveQuads ? d->numQuadVals : 0u;
    if (rowsPerList) *rowsPerList = d->quadRows;
    return CUTE_OK;
}

int cute_hrpb_dev_read_layouts(const cute_hrpb_dev *d, uint32_t *blockedRowPtr, uint32_t *hdr, float *tileVals, uint32_t *groupPtr,
                               uint32_t *recs, float *quadVals)
{
    if (!d) return CUTE_ERR_ARG;
    if (blockedRowPtr) std::memcpy(blockedRowPtr, d->brp.data(), d->brp.size() * sizeof(uint32_t));
    if (groupPtr) std::memcpy(groupPtr, d->qgp.data(), d->qgp.size() * sizeof(uint32_t));
    if (d->haveBricks) {
        if (hdr && d->nb) HIP_TRY(hipMemcpy(hdr, d->dHdr, uint64_t(d->nb) * CUTE_TILED_HDR_WORDS * 4u, hipMemcpyDeviceToHost));
        if (tileVals && d->numVals) HIP_TRY(hipMemcpy(tileVals, d->dVals, d->numVals * 4u, hipMemcpyDeviceToHost));
    }
    if (d->haveQuads) {
        if (recs && d->numGroups) HIP_TRY(hipMemcpy(recs, d->dQRecs, d->numGroups * CUTE_QUAD_RECORD_WORDS * 4u, hipMemcpyDeviceToHost));
        if (quadVals && d->numQuadVals) HIP_TRY(hipMemcpy(quadVals, d->dQVals, d->numQuadVals * 4u, hipMemcpyDeviceToHost));
    }
    return CUTE_OK;
}

int cute_hrpb_dev_csr(const cute_hrpb_dev *d, const uint32_t **dRowPtr, const uint32_t **dCols, const float **dVals)
{
    if (!d) return CUTE_ERR_ARG;
    if (dRowPtr) *dRowPtr = d->dRowPtr;
    if (dCols) *dCols = d->dCols;
    if (dVals) *dVals = d->dCsrVals;
    return CUTE_OK;
}

void cute_spmm_plan_free(cute_spmm_plan *p)
{
    if (!p) return;
    give_device_memory(p->memory);
    (void)hipFree(p->dHubRows);
    (void)hipFree(p->dHubRecs);
    delete p;
}

int cute_spmm_plan_info(const cute_spmm_plan *p, cute_plan_info *out)
{
    if (!p || !out) return CUTE_ERR_ARG;
    *out = p->info;
    return CUTE_OK;
}

int cute_spmm_plan_column_slabs(const cute_spmm_plan *p, uint32_t *mfma, uint32_t *rows)
{
    if (!p) return CUTE_ERR_ARG;
    if (mfma) *mfma = p->info.numChunks ? p->columnSlabs : 0u;
    if (rows) *rows = p->numRows ? p->rowColumnSlabs : 0u;
    return CUTE_OK;
}

int cute_spmm_plan_row_parts(const cute_spmm_plan *p, uint32_t *parts)
{
    if (!p) return CUTE_ERR_ARG;
    if (parts) *parts = p->rowParts;
    return CUTE_OK;
}

int cute_spmm_plan_window(const cute_spmm_plan *p, uint32_t *columns)
{
    if (!p) return CUTE_ERR_ARG;
    if (columns) *columns = p->windowColumns;
    return CUTE_OK;
}

// Replaces SPMM_TC's constructor chain (spmm.cu:276-822).  The per-N launch shapes of
// spmm.cu:11-101 and the occupancy table of spmm.cu:290-690 describe NVIDIA parts; here
// the shape follows from wave64 MFMA tiles (16 lanes x VEC columns per group) and the slot
// count from the CU count of the device.
int cute_spmm_plan_create(cute_hrpb_dev *d, uint32_t N, const cute_tunables *tn, cute_spmm_plan **out)
{
    if (!d || !out) return CUTE_ERR_ARG;
    *out = nullptr;
    if (N == 0) return CUTE_ERR_SHAPE;
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    cute_tunables t{};
    if (tn) t = *tn;
    if (t.path < CUTE_PATH_AUTO || t.path > CUTE_PATH_ROWS) return CUTE_ERR_ARG;
    if (t.precision != CUTE_PREC_FP32 && t.precision != CUTE_PREC_BF16X3) return CUTE_ERR_ARG;
    const float min_reuse = t.min_reuse > 0.0f ? t.min_reuse : kMinReuse;
    const uint32_t max_row_for_rows = t.max_row_nnz ? t.max_row_nnz : kMaxRowForRows;
    // An MFMA work item always spans 64 output columns; when N is narrower the row kernel wastes
    // less, so the reuse a panel must offer to earn the MFMA kernel grows (measured on N = 8..32).
    const float reuse_bar = N <= 32 ? std::min(3.0f, min_reuse * 48.0f / float(N)) : min_reuse;
    // Wide products of large matrices: the row kernel walks three dependent round trips per row (row pointers,
    // entries, B rows), the quad kernel streams its lists two groups ahead, and with 256 columns or more and a launch
    // several times the size of the device that depth counts for more than reuse: on 262 144 rows of 8 entries at
    // random columns, N = 256, the quad kernel takes 326 us against 339 (smaller windows: see `narrow` below);
    // ncvxbqp1, mk12-b3, delaunay_n16 of the reference's matrices gained 10-20 % the same way.  There the bar drops to "the lists need no more fetches than the
    // panel has entries" (matrices whose short lists would be mostly padding -- cat_ears_4_4, Wordnet3 -- stay with
    // the row kernel, which is 20 % ahead on them).
    // ... provided the panel's B rows cannot come out of an L2 anyway: a banded matrix, whose panels read a window of B
    // that the L2s hold (the banded benchmark matrix: 4 112 columns), is bound by the L2-to-L1 gather rate, where the row
    // kernel's 16 bytes per lane beat the quad kernel's 4 (1 736 against 2 046 us), and keeps the usual bar.
    const bool wide_and_large = t.min_reuse <= 0.0f && N >= 256u &&
                                uint64_t(d->M) * ((N + 255u) / 256u) >= 4ull * uint64_t(c.num_cus) * 32u;

    cute_spmm_plan *p = new cute_spmm_plan;
    p->d = d;
    // (in locals: what is stored to a byte array could be a member of d)
    const uint32_t P = d->P, *const brp = d->brp.data(), *const qgp = d->qgp.data(), *const panelCols = d->panelCols.data(), *const panelNnz = d->panelNnz.data(),
                   *const panelMaxRow = d->panelMaxRow.data(), *const panelSpan = d->panelSpan.data();
    // classify panels
    std::vector<uint8_t> to_rows(P, 0);
    // panels that go to the MFMA kernel for another reason than their reuse (below); the choice of the MFMA shape is
    // made on the panels that earned it
    std::vector<uint8_t> joined(P, 0);
    // The row kernel gives a row N / VEC lanes; up to N = 128 several rows share a wavefront, which then takes as long
    // as its longest row.  A panel whose longest row is more than twice its mean row (and longer than two batches of
    // eight entries) keeps its wavefronts waiting for that one row, and the MFMA kernel, which walks the panel's
    // columns whatever row they belong to, is ahead although the reuse is low: on the reference's matrices with
    // long-tailed rows (jan99jac*, de2010, ri2010, Wordnet3, bayer04, ted_B: 99th percentile of the row lengths 3-6 times
    // the mean) 25-35 % at N = 16 and 32, geomean over the 43 matrices against the best single kernel 1.18 -> 1.10
    // (N = 16), 1.10 -> 1.04 (N = 32), 1.07 -> 1.03 (N = 128).  With one row per wavefront (N >= 256) the same move
    // loses (HEP-th-new, N = 512: 60 -> 68 us), so it is not made there.
    const bool rows_share_a_wavefront = t.max_row_nnz == 0 && (N + uint32_t(lane_floats(N)) - 1u) / uint32_t(lane_floats(N)) < 64u;
    // Scattered panels (kScatteredBytes).  Where their rows share columns (graphs), a large product leaves only the panels with
    // twice as many entries as fetches to the lists and takes rows of up to 96 entries to the row kernel, uneven or not: its
    // sixteen lanes a row ask for 256 bytes of B with one instruction, a list slot for the same with 64 lanes.  R-MAT graph
    // of 131 072 nodes and 2.5 million entries: N = 128 126 -> 92 us, N = 256 236 -> 228, N = 310 377 -> 320; below 2^24
    // elements of C the launch no longer fills the device and the long rows show (32 768 nodes, N = 128: 26 -> 33).
    // Much of that comes from the columns an XCD owns: where the lists stay in row order (below 256 columns, off the grid of 64), graphs of 24
    // entries a row lose (131 072 nodes, N = 208 235 -> 261, N = 240 263 -> 292; 20 entries a row 208 -> 203, 12 142 -> 134).
    const bool default_bars = t.path == CUTE_PATH_AUTO && t.min_reuse <= 0.0f && t.max_row_nnz == 0;
    auto scattered = [&](uint32_t q) { return uint64_t(panelSpan[q]) * std::min(N, 256u) * sizeof(float) > kScatteredBytes; };
    const bool graph_bars = default_bars && t.precision == CUTE_PREC_FP32 && N >= 128u && uint64_t(d->M) * N >= kGraphProduct &&
                            (N % 64u == 0 || N >= 256u || N % 4u != 0 || uint64_t(d->nnz) < 22ull * d->M);
    auto fetches_of = [&](uint32_t q) {
        // what the MFMA side would fetch for this panel: one B row per list slot of the quad
        // lists (pairs plus padding), which is at least one per active column
        const uint32_t lists = d->quadRows == 4 ? 4u : 1u;
        return std::max(panelCols[q], (qgp[(q + 1) * lists] - qgp[q * lists]) * 16u);
    };
    const uint32_t parts = default_bars && t.precision == CUTE_PREC_FP32 && !t.slots && !t.mfma_shape && !t.hub_rows && !t.max_chunk_blocks &&
                                   !t.brick_groups && !t.pipeline && !t.chunk_order ? row_parts(d, N) : 1u;
    uint64_t reused = 0;                          // entries of panels that go to the MFMA side by the usual bars: reuse, long or uneven rows
    uint32_t n_brick = 0, n_rows = 0, n_empty = 0;
    for (uint32_t q = 0; q < P; ++q) {
        const uint32_t nblk = brp[q + 1] - brp[q];
        bool rows;
        if (nblk == 0) { rows = true; n_empty++; }
        else if (t.path == CUTE_PATH_BRICK) rows = false;
        else if (t.path == CUTE_PATH_ROWS || parts > 1u) rows = true;
        else {
            // Row kernel when a B row fetched by the MFMA side serves hardly more than one nonzero of the
            // panel (the matrix cores then buy nothing) -- unless a row is so long that one lane group
            // would serialise it: the brick kernel cuts long panels into balanced chunks.
            const uint32_t fetches = fetches_of(q);
            const bool graph = graph_bars && scattered(q);
            const float bar = graph ? kGraphReuse
                              : (wide_and_large && uint64_t(panelSpan[q]) * N * sizeof(float) > kWideWindowBytes) ? kWideReuse : reuse_bar;
            rows = float(panelNnz[q]) < bar * float(fetches) && panelMaxRow[q] <= (graph ? kGraphMaxRow : max_row_for_rows);
            const bool uneven = rows_share_a_wavefront && panelMaxRow[q] > kUnevenRowFloor &&
                                uint64_t(panelMaxRow[q]) * CUTE_TM > uint64_t(kUnevenRowRatio) * panelNnz[q];
            if (uneven || panelMaxRow[q] > max_row_for_rows || float(panelNnz[q]) >= reuse_bar * float(fetches)) reused += panelNnz[q];
            if (rows && uneven && !graph) {
                rows = false;
                joined[q] = 1;
            }
        }
        to_rows[q] = rows;
        if (nblk) (rows ? n_rows : n_brick)++;
    }
    // An XCD per column slab.  Row panels over a scattered window gather from behind the L2s as long as every XCD reads whole
    // rows of B; when an XCD owns 32 columns instead, the piece of B it reads is (window) x 128 bytes and may fit its 4 MB.
    // `narrow` gives the width of such a slab, 0 where it does not pay: rows of B a multiple of 128 bytes apart are cut into
    // whole cache lines, a multiple of 64 bytes costs a line more per piece, any other pitch needs pieces of 64 columns.
    // Random columns, 8 entries a row, us in row order / by columns: 16 384 rows N = 256 18.1 / 7.9, N = 512 35.4 / 18.3;
    // 32 768 rows N = 128 18.2 / 11.3; 65 536 rows N = 256 82.8 / 64.5; 131 072 rows 167 / 159; 262 144 rows 339 / 356;
    // N = 400: 16 384 rows 29.1 / 19.1, 32 768 rows 63.5 / 53.8, 65 536 rows 133 / 153; N = 301: 16 384 rows 26.5 / 21.0,
    // 32 768 rows 55.7 / 57.3.  Longer rows share an L2 less well than lists, whose wavefronts walk the columns in step:
    // lists / by columns, 16 entries a row, 32 768 rows N = 256 45.2 / 39.7, 50 000 rows 88.9 / 115; 31 entries a row,
    // 16 384 rows N = 256 29.0 / 26.6, 32 768 rows 75.2 / 80.8.
    auto narrow = [&](uint64_t window, uint64_t mean_row) -> uint32_t {
        if (N % 32u == 0 && N >= 64u) return window <= (mean_row < 16u ? 131072u : mean_row < 24u ? 32768u : 16384u) ? 32u : 0u;
        if (N < 256u) return 0u;
        if (N % 16u == 0) return window <= (mean_row < 16u ? 32768u : 8192u) ? 32u : 0u;
        return window <= (mean_row < 16u ? 16384u : 8192u) ? 64u : 0u;
    };
    // The row kernel walks 256 columns at a time, and the last walk costs nearly a whole one however few columns are left; lists
    // pay for pieces of 64.  Off the 128-byte grid of B, lists / row kernel in row order, us, 4 and 10 entries a row:
    // 20 000 rows N = 264 16.4 / 18.7, 30.1 / 35.8, N = 301 37.1 / 40.3 (10), N = 600 equal; 30 000 rows N = 301 31.5 / 30.1;
    // 40 000 rows N = 272 32.3 / 37.3, 64.6 / 78.0, N = 301 rows 7 % ahead, N = 432 rows 5 % ahead and 100 / 105, N = 528 60.3 / 64.4,
    // 124 / 137, N = 600 159 / 147 (10); 65 536 rows N = 272 55.4 / 61.7, 117 / 129, N = 264 3 %, N = 280 equal, N = 528 222 / 233;
    // 131 072 rows N = 272 116 / 124, N = 264 rows 3 % ahead, N = 528 3 %.
    auto short_last_slab = [&](uint64_t window, uint64_t mean_row) {
        const uint32_t last = N % 256u;
        if (window <= 24576u) return last < 64u;
        if (window <= 49152u) return (N % 8u == 0 && last <= 48u) || (N % 16u == 0 && mean_row >= 8u);
        if (window <= 65536u) return N % 8u == 0 && last <= 16u;
        return N % 16u == 0 && last <= 16u && N < 512u;
    };
    bool half_window = false;
    // A matrix without reuse or hubs (less than a tenth of its entries in panels for the MFMA side): its scattered panels go to
    // the lists only where these are ahead of the row kernel in whichever order suits it.  24 entries a row, us row kernel /
    // lists: 65 536 rows N = 64 46.8 / 37.0, N = 128 106 / 81; 131 072 rows N = 256 457 / 408; rows of B off the 128-byte
    // grid: 32 768 rows N = 301 151 / 126, 65 536 rows N = 400 363 / 354, 98 304 rows 558 / 589.  8 entries a row off that
    // grid: 50 000 rows N = 301 87.7 / 95.2, 131 072 rows N = 400 274 / 305.  Products of 512 columns or more over windows
    // that do not fit an L2 in slabs of 32 columns stay with the lists (the planner's tests hold them to it; 50 000 rows of 7:
    // 32-column lists 80.6, the row kernel by columns 73.5).
    if (default_bars && t.precision == CUTE_PREC_FP32 && reused * 10u < uint64_t(d->nnz) &&
        uint64_t(d->M) * ((N + 255u) / 256u) >= 4ull * uint64_t(c.num_cus) * 32u) {
        auto concerned = [&](uint32_t q) { return brp[q + 1] != brp[q] && panelMaxRow[q] <= max_row_for_rows && scattered(q); };
        uint64_t windows = 0, entries = 0, panels = 0;
        for (uint32_t q = 0; q < P; ++q)
            if (concerned(q)) { windows += panelSpan[q]; entries += panelNnz[q]; ++panels; }
        if (panels) {
            const uint64_t window = windows / panels, mean_row = entries / (panels * CUTE_TM);
            // 32-column lists where a 64-column slab of the window outgrows the L2 by more than they do; us 64 / 32 columns:
            // 16 entries a row, 50 000 rows N = 64 21.2 / 17.9, N = 256 88.9 / 78.0, N = 512 181 / 145; 65 536 rows
            // N = 128 58.9 / 52.5; 31 entries a row, 32 768 rows N = 256 75.2 / 78.4, N = 512 155 / 135, 65 536 rows
            // N = 256 205 / 213, 98 304 rows N = 64 82.7 / 76.8; 131 072 rows of 16, N = 256 287 / 301.
            half_window = N % 32u == 0 && (window > 32768u || N >= 512u) && window <= (N <= 128u ? 98304u : N < 512u ? 57344u : 65536u);
            const bool on_grid = N % 32u == 0, wide = N >= 512u && window > 32768u;
            const bool lists_ahead = on_grid ? (wide || (narrow(window, mean_row) == 0 && (mean_row >= 16u || N >= 256u)))
                                             : (narrow(window, mean_row) == 0 && N >= 256u &&
                                                ((mean_row >= 16u && window <= 65536u) || short_last_slab(window, mean_row)));
            for (uint32_t q = 0; q < P; ++q) {
                if (!concerned(q)) continue;
                const uint8_t rows = !(lists_ahead && N >= 64u && float(panelNnz[q]) >= kWideReuse * float(fetches_of(q)));
                if (rows == to_rows[q]) continue;
                to_rows[q] = rows;
                joined[q] = 0;
                if (rows) { ++n_rows; --n_brick; } else { --n_rows; ++n_brick; }
            }
        }
    }
    // A handful of MFMA panels among row-kernel panels (the boundary panels of a stencil at N = 32: 64 of 16 384) would
    // turn the launch into the fused kernel for their sake, which costs the row blocks more than those panels gain
    // (9-point stencil of 512 x 512 points, N = 32: 29.0 us against 24.4 with every panel on the row kernel): when
    // the MFMA panels hold less than 2 % of the entries and none of them has a row too long for a lane group,
    // they go to the row kernel as well.
    // The same the other way round: a few row-kernel panels among MFMA panels cost a second launch or the fused
    // kernel (FEM benchmark matrix, 53 of 3 000 panels: N = 8 21.2 us against 11.0 with every panel on the brick
    // kernel, N = 16 12.3 against 10.7, N = 24 16.7 against 14.0); below 2 % of the entries they join the others.
    if (t.path == CUTE_PATH_AUTO && n_brick && n_rows) {
        uint64_t nnz_mfma = 0;
        bool movable = true;
        for (uint32_t q = 0; q < P; ++q)
            if (!to_rows[q]) {
                nnz_mfma += panelNnz[q];
                movable = movable && panelMaxRow[q] <= max_row_for_rows;
            }
        if (movable && nnz_mfma * 50u < uint64_t(d->nnz)) {
            std::fill(to_rows.begin(), to_rows.end(), uint8_t(1));
            n_rows += n_brick;
            n_brick = 0;
        } else if ((uint64_t(d->nnz) - nnz_mfma) * 50u < uint64_t(d->nnz)) {
            for (uint32_t q = 0; q < P; ++q)
                if (to_rows[q] && brp[q + 1] != brp[q]) { to_rows[q] = 0; joined[q] = 1; }   // (empty panels stay: the row kernel zeroes their rows)
            n_brick += n_rows;
            n_rows = 0;
        }
    }

    // brick kernel shape
    p->vec = lane_floats(N);
    p->rows_vec = p->vec;
    // a brick work item spans 16*VEC columns: for narrow N take the narrowest tile that still covers N
    while (p->vec > 1 && 8u * uint32_t(p->vec) >= N) p->vec /= 2;
    p->ng = (p->vec == 4 && N >= 128) ? 2 : 1;   // two column groups per lane pay off from 128 columns on (measured)
    // row kernel shape: lanes per row = smallest power of two covering N/VEC, at most 64
    {
        uint32_t need = (N + p->rows_vec - 1) / p->rows_vec, logl = 0;
        while ((1u << logl) < need && logl < 6) ++logl;
        p->rows_logl = int(logl);
        const uint32_t w = (1u << logl) * p->rows_vec;
        p->rows_slabs = (N + w - 1) / w;
    }
    // A mixed plan is one launch, and the two-group brick kernel holds only four wavefronts per SIMD: when its
    // work-groups and the row blocks together exceed that, the row blocks queue behind each other and the launch
    // takes as long as the two parts one after the other (bcsstk18, N = 128: 11.8 us against 5.1 + 6.5).  One
    // column group per lane halves the registers and doubles the resident wavefronts; the same when the row blocks
    // are the larger part of the launch anyway (ted_B, N = 128).
    bool ng_for_mixed = false;
    // (not when B and C come from HBM: there the wider row pieces of two column groups count for more)
    if (t.operand_residency > 2) { delete p; return CUTE_ERR_ARG; }
    const bool beyond_cache = t.operand_residency ? t.operand_residency == 1
                                                  : (uint64_t(d->K) + d->M) * N * sizeof(float) > c.cache_bytes;
    if (p->ng == 2 && t.brick_groups == 0 && n_brick && n_rows && !beyond_cache) {
        const uint64_t row_blocks = (uint64_t(n_rows) * CUTE_TM * p->rows_slabs + (256u >> p->rows_logl) - 1) / (256u >> p->rows_logl);
        const uint64_t groups = (uint64_t(n_brick) * ((N + 127u) / 128u) + cute_dev::kWavesPerGroup - 1) / cute_dev::kWavesPerGroup;
        if (row_blocks + groups > uint64_t(c.num_cus) * 4u || row_blocks >= groups) { p->ng = 1; ng_for_mixed = true; }
    }
    if (t.brick_groups == 1 || (t.brick_groups == 2 && p->vec == 4)) p->ng = int(t.brick_groups);
    if (t.pipeline > 2) { delete p; return CUTE_ERR_ARG; }
    // the rolling variant addresses B and the values with 32-bit byte offsets (24 x 24-bit product)
    const bool offsets_fit = cute_offsets_fit(d->M, d->K, N, d->numVals, 0) == 1;
    p->pipeline = t.pipeline ? int(t.pipeline) : 1;
    if (p->pipeline == 1 && !offsets_fit) p->pipeline = 2;
    if (t.mfma_shape > 2) { delete p; return CUTE_ERR_ARG; }
    if (t.mfma_shape) p->shape = int(t.mfma_shape);
    else if (t.precision == CUTE_PREC_BF16X3) p->shape = 1;      // the reduced-precision kernel works on the brick tiles
    else {
        // A 16x4 brick costs the same matrix time however few nonzeros it holds; the quad lists
        // only pay for occupied (4-row group, column) pairs but fetch a B row once per row group
        // instead of once per panel, and pad their lists.  Measured break-even on the benchmark
        // matrices and on the reference's 43: about 8 list slots (pairs plus padding) per brick.
        const uint32_t lists = d->quadRows == 4 ? 4u : 1u;     // list units per panel
        uint64_t slots = 0, bricks = 0, blocks = 0, entries = 0;
        for (uint32_t q = 0; q < P; ++q)
            if (!to_rows[q] && !joined[q]) {
                entries += panelNnz[q];
                slots += uint64_t(qgp[(q + 1) * lists] - qgp[q * lists]) * 16u;
                bricks += (panelCols[q] + 3u) / 4u;
                blocks += brp[q + 1] - brp[q];
            }
        p->shape = choose_mfma_shape(slots, bricks, blocks, entries, uint64_t(d->K) + d->M, d->nnz, N, t.operand_residency, c.cache_bytes);
    }
    if (p->shape == 2 && !(offsets_fit && (d->numQuadVals + 64u) * 4u <= 0xffffffffull)) p->shape = 1;
    // bf16x3 exists for the rolling brick kernel with four columns per lane, and is asked for with N a multiple of four;
    // any other shape computes in fp32
    p->bf16x3 = t.precision == CUTE_PREC_BF16X3 && p->shape == 1 && p->pipeline == 1 && p->vec == 4 && N % 4u == 0;
    // The brick kernel's slab follows the number of work items as well.  A wavefront walks its panel alone, 32 matrix cycles per
    // brick and 16 columns, so a launch that leaves SIMDs without a wavefront, or gives some of them one more than the others,
    // takes (fullest SIMD's wavefronts) x (slab): with T(w) = ceil(items / SIMDs) x w for slabs of 16 w columns, the narrower
    // slab is taken where T falls.  Narrower pieces of a B row cost more requests per byte, which shows once two or three
    // wavefronts a SIMD are running: the limits.  Finite-element matrices, us at the slab named, 128 / 64 / 32 / 16 columns:
    // 24 000 rows N = 128 20.1 / 15.7 / 23.8 / 32.8, N = 256 26.3 / 26.4 (equal T), N = 301 47.0 / 36.4; 2 400 rows N = 128
    // 19.0 / 13.2 / 10.6 / 10.5, N = 301 19.4 / 13.6 / 13.6 / 11.4; 4 800 rows N = 64 - / 10.7 / 8.1 / 8.5, N = 200
    // 16.7 / 13.9 / 15.9 / 14.9.  (Odd N gains from single columns a little longer: no other piece of its rows is aligned.)
    // bf16x3 spends a third of the matrix time, and beside row panels the SIMDs are not idle: where its operands come from HBM
    // the wide pieces count for more, as above.  131 072-node graph, 10 edges a node, us at 128 / 64 columns: N = 300 225 / 310, 384 227 / 310.
    if (p->shape == 1 && p->pipeline == 1 && t.brick_groups == 0 && n_brick) {
        const uint64_t simds = uint64_t(c.num_cus) * 4u;
        auto items = [&](uint32_t w) { return uint64_t(n_brick) * ((N + 16u * w - 1u) / (16u * w)); };
        auto T = [&](uint32_t w) { return (items(w) + simds - 1u) / simds * w; };
        if (p->ng == 2 && items(4) <= 8u * simds && ((T(4) < T(8) && !(p->bf16x3 && n_rows && beyond_cache)) || items(8) <= simds)) {
            p->ng = 1;
            ng_for_mixed = true;                  // (the fused launch has this shape)
        }
        const bool alone = n_rows == 0 && n_empty == 0 && t.precision == CUTE_PREC_FP32;    // no fused launch, no bf16 kernel for less than four
        if (p->ng == 1 && alone)
            for (uint32_t w = uint32_t(p->vec) / 2u; w; w /= 2u)
                if (items(w) <= (w == 1 && N % 2u ? 3u : 2u) * simds && T(w) < T(uint32_t(p->vec))) p->vec = int(w);
    }
    // Which parts of the launch go by columns (cute_dev::xcd_share).  A plan of rows alone takes the slab that `narrow` gives for
    // its mean window.  MFMA panels that share columns find a graph's hub rows in their XCD's slab whatever the window: R-MAT
    // graph of 32 768 nodes, N = 512 156 -> 104 us, 16 384 nodes, N = 256 33.5 -> 26.7, 131 072 nodes, N = 310 463 -> 413;
    // lists without reuse gain while the window fits two L2s (16 384 rows of 24, N = 512 46.4 -> 41.8; 65 536 rows 349 -> 367).
    // Off the 64-column grid the last slab is a remainder that unbalances few slabs (N = 101: 137 -> 147): 256 columns or more.
    // The brick kernels' slabs are up to 128 columns wide, a row kernel's beside them 256, and a remainder unbalances few of those at any
    // N: at least four times the width, or no remainder.  32 768 rows of 24 at random columns, us in row order / by columns: N = 300 109 / 120
    // (bf16x3 111 / 122), N = 320 86.2 / 94.5 (83.5 / 96.2); 131 072-node graph, bf16x3, N = 300 337 / 355, and with the rows
    // beside it in row order, 65 536 nodes, 185 / 189.  In fp32 a graph gains more than that costs (131 072 nodes, N = 257, 472 / 349).
    // Lists without reuse take a remainder of any size while the window is small (20 000 rows of 20, N = 264: 5 % ahead by columns), and up
    // to two L2s one that leaves no more than a tenth idle (30 000 rows of 10, us in row order / by columns, N = 257 55.1 / 59.4,
    // N = 280 26.1 / 27.5 at 4 entries; 24 000 rows of 4, N = 264 19.5 / 20.8; N = 301 equal).
    auto balanced = [&](uint32_t width) { return N % width == 0 || N >= 4u * width; };
    uint32_t rows_columns = 0;
    bool mfma_by_columns = false;
    {
        uint64_t scattered_nnz = 0, window[2] = {}, in[2] = {}, cols = 0;
        uint32_t row_panels = 0;
        for (uint32_t q = 0; q < P; ++q) {
            const uint32_t side = to_rows[q] ? 1u : 0u;
            if (scattered(q)) scattered_nnz += panelNnz[q];
            window[side] += uint64_t(panelSpan[q]) * panelNnz[q];
            in[side] += panelNnz[q];
            if (side == 0) cols += panelCols[q];
            else if (panelNnz[q]) ++row_panels;
        }
        if (scattered_nnz * 2u > uint64_t(d->nnz)) {
            const uint64_t mean_window[2] = {in[0] ? window[0] / in[0] : 0, in[1] ? window[1] / in[1] : 0};
            const bool sharing = in[0] * 5u >= cols * 6u;
            const uint32_t mfma_width = p->shape == 2 ? 64u : 16u * uint32_t(p->vec * p->ng);
            if (n_brick == 0)
                rows_columns = narrow(mean_window[1], in[1] / (uint64_t(row_panels) * CUTE_TM));
            else if (half_window && p->shape == 2 && !t.hub_rows && n_rows == 0 && n_empty == 0 && (N + 31u) / 32u <= 65535u)
                mfma_by_columns = p->halfLists = true;
            else if (((N % 64u == 0 && N >= 128u) || N >= 256u) &&
                     (sharing || mean_window[0] <= 32768u) && ((sharing && !p->bf16x3) || balanced(mfma_width)) &&
                     (sharing || mean_window[0] <= 20480u || (N + mfma_width - 1u) / mfma_width * mfma_width * 10u <= N * 11u)) {
                mfma_by_columns = true;
                // rows of uneven length share a wavefront: sixteen lanes a row (the brick kernel has no launch with fewer than its own)
                const uint32_t width = p->shape == 2 && p->rows_vec == 4 ? 64u : uint32_t(p->rows_vec << p->rows_logl);
                rows_columns = p->bf16x3 && !balanced(width) ? 0u : width;
            }
        }
        // (slabs are the y dimension of the launch)
        if (p->rows_vec == 4 && rows_columns && rows_columns < (4u << p->rows_logl) && (N + rows_columns - 1u) / rows_columns <= 65535u) {
            p->rows_logl = rows_columns == 32u ? 3 : 4;
            p->rows_slabs = (N + rows_columns - 1u) / rows_columns;
        }
        p->rowColumnSlabs = rows_columns ? p->rows_slabs : 0u;
    }
    if (n_brick == 0 && default_bars) {
        const int rc = plan_window(p, d, N, c, t.operand_residency == 2);
        if (rc != CUTE_OK) { delete p; return rc; }
    }
    // The chunk list depends on the MFMA kernel (its work units are blocks or list groups).  It is built, once more with fewer
    // cuts if these need more scratch than there is, and if the partial tiles of the cut panels then turn out to be more rows than the fast kernels'
    // 24-bit row operand can address, built once more for the pipelined brick kernel, whose stores use
    // 64-bit offsets.
    uint32_t slab = 0, num_slabs = 0, upp_log = 0, slots = 0, n_pieces = 0;
    WorkItems chunks;
    std::vector<uint4> fixups;
    uint64_t total_units = 0;          // of all work items, and of the longest
    uint32_t longest_item = 0;
    for (int attempt = 0;; ++attempt) {
        slab = p->shape == 2 ? (p->halfLists ? 32u : 64u) : 16u * p->vec * p->ng;   // the quad kernel: one column per lane (or half of them)
        num_slabs = (N + slab - 1) / slab;
        if (num_slabs > 65535u) { delete p; return CUTE_ERR_ARG; }   // slabs are the y dimension of the launch

        // chunk list for the brick kernel.  With t.slots set, the reference arithmetic
        // (spmm.cu:776-812) decides which panels are cut; its default there would cut every panel
        // that is one block above the (floored) mean as soon as the device holds all work items
        // at once, which is the normal case on 256 CUs.  The default policy therefore cuts only
        // outliers: a panel is split when it is more than twice as long as the per-item share
        // of the whole job (and at least 8 blocks), into pieces of about that share.
        // work units along a panel: 16-column blocks for the brick kernel, groups for the quad kernel
        const uint32_t *const unit = p->shape == 2 ? qgp : brp;
        // units per panel (its logarithm): 4 when the quad lists are kept per 4-row strip
        upp_log = (p->shape == 2 && d->quadRows == 4) ? 2u : 0u;
        const uint32_t num_units = P << upp_log;
        const uint32_t resident = uint32_t(c.num_cus) * 4u * 8u;   // 4 SIMDs x 8 wavefronts per CU
        slots = t.slots ? t.slots : resident;
        // A chunk of a cut panel carries the 1-based number of its partial tile; the pieces of one panel are
        // consecutive (panels ascend through the list), and one fixup entry per cut panel adds them up afterwards.
        chunks.clear();
        fixups.clear();
        n_pieces = longest_item = 0;
        total_units = 0;
        chunks.reserve((size_t(n_brick) << upp_log) + 64u);
        auto emit = [&](uint32_t s, uint32_t e, uint32_t pan, bool cut) {
            const uint32_t len = e - s, cap = t.max_chunk_blocks ? t.max_chunk_blocks : len, step = std::min(cap, len);
            cut = cut || len > cap;                    // cut further than the partition asked for
            for (uint32_t cs = s; cs < e; cs += step) {
                if (cut) {
                    if (fixups.empty() || fixups.back().x != pan) fixups.push_back(make_uint4(pan, n_pieces, 0u, 0u));
                    fixups.back().z++;
                    ++n_pieces;
                }
                chunks.push_back(make_uint4(cs, std::min(e, cs + step), pan, cut ? n_pieces : 0u));
            }
            total_units += len;
            longest_item = std::max(longest_item, step);
        };
        if (t.slots) {
            const int64_t n = cute_partition(num_units, unit, num_slabs, slots, nullptr, 0);
            if (n < 0) { delete p; return int(n); }
            std::vector<uint32_t> quads(uint64_t(n) * 4);
            cute_partition(num_units, unit, num_slabs, slots, quads.data(), uint64_t(n));
            for (size_t i = 0; i + 3 < quads.size(); i += 4)
                if (!to_rows[quads[i + 2] >> upp_log]) emit(quads[i], quads[i + 1], quads[i + 2], quads[i + 3] != 0);
        } else if (n_brick) {
            uint64_t work = 0;
            uint64_t busy = 0;
            for (uint32_t q = 0; q < P; ++q) {
                if (to_rows[q]) continue;
                work += unit[(q + 1) << upp_log] - unit[q << upp_log];
                for (uint32_t u = q << upp_log; u < (q + 1) << upp_log; ++u) busy += unit[u + 1] != unit[u];
            }
            const uint64_t mean = busy ? (work + busy - 1) / busy : 1;
            const uint64_t share = (work * num_slabs + resident - 1) / resident;
            // the mean only counts while it is short: a matrix whose few MFMA panels are all very long
            // (a handful of dense rows) must still be cut, or one wavefront walks a whole panel alone
            const uint32_t target = uint32_t(std::max<uint64_t>(std::max<uint64_t>(share, std::min<uint64_t>(mean, 16)), 8));
            // A launch that keeps every wavefront slot busy runs at the rate the memory system gathers B rows, and a
            // work item then advances about five times slower than one that runs alone (measured on the R-MAT
            // benchmark matrix: 0.39 us per list group alone, 1.7 us per group and slot under load).  So an item of several
            // shares still ends with the launch, and cutting it finer only adds partial tiles: lists are cut at four shares, into
            // pieces of two.  R-MAT graphs, nodes (log 2) / edges / N, us cut at six shares into fours, at four into twos, at three into twos,
            // at two into ones: 17/10/64 45.3, 43.2, 44.3, 46.7; 16/10/47 23.9, 21.6, 21.4, 22.9; 15/10/64 18.3, 17.2, 18.7, 18.5;
            // 15/6/100 26.6, 19.4, 18.9, 18.5; 16/6/128 35.4, 29.4, 29.3, 34.3; 14/10/200 29.3, 23.4, 23.5, 24.7; 16/12/256 115, 95.6, 95.7,
            // 95.2; 17/10/128 90.1, 89.8, 89.9, 94.0.  (Before the pieces added themselves up, six and four were the best.)
            // A graph's bricks, which it has below 32 columns, are bound by their matrix work and are cut like a launch that does not fill the device
            // and is bound by its longest item: at twice the target, into pieces of one (17/10/16 51.0, 39.2, 39.2, 30.3; 16/8/16 19.7, 18.2,
            // 18.1, 18.1).  Wider bricks keep six shares and four: bf16x3 loses (16/10/128 85.4, 88.0, 88.2, 102), in fp32 they are
            // those of even panels.  So do plans whose finer cut's tiles would not fit cute_spmm_run_static's scratch.  Who adds the pieces up does not
            // turn the rule round: run_scratch, hub and pipelined plans, with a second launch, at six into fours / four into twos: 16/10/47 26.3, 24.2 and
            // 17/10/64 45.9, 45.3 by run_scratch, 16/10/47 61.5, 42.9 and 17/10/64 91.5, 91.9 with 128 hub rows, 17/10/16 60.9, 36.7 pipelined.
            // Lists of two column slabs: most strips to be cut are the few lengths of a graph's hub panels, and where two shares make four pieces of one
            // (a work-group each) a launch of strips of more than 12 groups a share took up to 1.18 times the time of the coarser cut; twos of three shares do not, nor five fourths.
            // us at six into fours, four into twos, now: 16/12/128 64.0, 75.7, 55.2; 16/9/101 53.1, 61.2, 47.0; 16/8/128 41.6, 43.0, 35.2; 15/12/128 28.0, 27.4,
            // 23.2; 17/8/112 105, 88.0, 80.6; 17/8/128 78.3, 79.5, 78.7; 16/7/80 34.9, 28.9, 30.2.  With three slabs and more it gains and loses alike (16/12/144 91.6, 72.9, 76.6;
            // 16/9/160 57.6 to 63.0; 16/6/200 0.77 times), and nothing was slower than with the coarser cut.
            const bool finer = attempt == 0 && (p->shape == 2 || N < 32u);
            const bool two_slabs = finer && p->shape == 2 && num_slabs == 2u && share > 8u;
            const uint64_t least_cut = two_slabs ? 3u : finer ? (p->shape == 2 ? 4u : 0u) : 6u;
            const uint32_t limit = uint32_t(std::max<uint64_t>(2u * uint64_t(target), least_cut * share));
            const uint32_t piece = limit <= 2u * target ? target : uint32_t(two_slabs && share > 12u ? share * 5u / 4u : (finer ? 2u : 4u) * share);
            chunks.resize(std::max<size_t>(chunks.capacity(), 64u));
            size_t at = 0;
            for (uint32_t q = 0; q < num_units; ++q) {
                if (to_rows[q >> upp_log]) { q |= (1u << upp_log) - 1u; continue; }
                const uint32_t s = unit[q], e = unit[q + 1], nblk = e - s;
                if (nblk == 0) continue;
                if (nblk <= limit && !t.max_chunk_blocks) {
                    if (at == chunks.size()) chunks.resize(at + at / 2u);
                    chunks[at++] = make_uint4(s, e, q, 0u);
                    longest_item = std::max(longest_item, nblk);
                    total_units += nblk;
                    continue;
                }
                chunks.resize(at);
                if (nblk <= limit) emit(s, e, q, false);
                else {
                    const uint32_t pieces = (nblk + piece - 1) / piece, step = (nblk + pieces - 1) / pieces;
                    for (uint32_t cs = s; cs < e; cs += step) emit(cs, std::min(e, cs + step), q, true);
                }
                at = chunks.size();
                chunks.resize(std::max(chunks.capacity(), at + 64u));
            }
            chunks.resize(at);
        }
        // a strip without pairs inside an MFMA-routed panel still has to be written (as zeros): an empty chunk
        if (upp_log && n_brick)
            for (uint32_t q = 0; q < num_units; ++q)
                if (unit[q] == unit[q + 1] && !to_rows[q >> upp_log]) chunks.push_back(make_uint4(unit[q], unit[q], q, 0u));
        const bool lean = p->shape == 2 || p->pipeline == 1;
        const uint64_t tile_rows = uint64_t(n_pieces) * (CUTE_TM >> upp_log);
        const bool fits = !lean || !n_pieces || cute_offsets_fit(d->M, d->K, N, 0, tile_rows) == 1;
        // (with the default cut there are at most as many pieces as wavefronts, 32 MiB of tiles; max_chunk_blocks can add to them)
        if (attempt == 0 && !t.slots && (p->shape == 2 || N < 32u) && (!fits || tile_rows * N * sizeof(float) > uint64_t(CUTE_STATIC_SCRATCH_BYTES))) continue;
        if (fits) break;
        if (attempt == 2 || t.mfma_shape == 2 || t.pipeline == 1) { delete p; return CUTE_ERR_SHAPE; }   // the caller forced a fast kernel
        attempt = 1;
        p->shape = 1;
        p->pipeline = 2;
        p->bf16x3 = p->halfLists = false;
    }
    uint32_t num_row_panels = 0;
    for (uint32_t q = 0; q < P; ++q) num_row_panels += to_rows[q];
    // Every row on the row kernel: no row list needed, which takes one dependent load out of each row's chain.
    const bool every_row = num_row_panels == P;
    std::vector<uint32_t> row_panels;              // panels of the row kernel, unless it has them all
    if (!every_row && num_row_panels) {
        row_panels.reserve(num_row_panels);
        for (uint32_t q = 0; q < P; ++q)
            if (to_rows[q]) row_panels.push_back(q);
    }

    // Row-kernel blocks per XCD: contiguous ranges of rows (neighbouring rows share B rows, which then stay
    // in one L2), cut where the running work -- nonzeros plus a fixed cost per row -- passes each eighth.
    {
        const uint32_t items_per_block = 256u >> p->rows_logl;             // rows of one 256-thread block (per slab)
        const uint64_t total_items = uint64_t(num_row_panels) * CUTE_TM;
        const uint32_t total_blocks = uint32_t((total_items + items_per_block - 1) / items_per_block);
        uint64_t total_work = 0;
        for (uint32_t q = 0; q < P; ++q) total_work += to_rows[q] ? panelNnz[q] + uint64_t(4u * CUTE_TM) : 0u;
        uint64_t work = 0, items = 0;
        uint32_t x = 1;
        p->rowRanges.first[0] = 0;
        auto share = [&] { return (total_work * x + cute_dev::kNumXcd - 1u) / cute_dev::kNumXcd; };      // where range x begins
        uint64_t next = share();
        for (uint32_t q = 0; q < P && num_row_panels && x < cute_dev::kNumXcd; ++q) {
            if (!to_rows[q]) continue;
            work += panelNnz[q] + uint64_t(4u * CUTE_TM);
            items += uint64_t(CUTE_TM);
            for (; x < cute_dev::kNumXcd && work >= next; next = share())
                p->rowRanges.first[x++] = uint32_t(std::min<uint64_t>(total_blocks, (items + items_per_block - 1) / items_per_block));
        }
        while (x <= cute_dev::kNumXcd) p->rowRanges.first[x++] = total_blocks;
        p->rowBlocksPerXcd = 0;
        for (uint32_t k = 0; k < cute_dev::kNumXcd; ++k)
            p->rowBlocksPerXcd = std::max(p->rowBlocksPerXcd, p->rowRanges.first[k + 1] - p->rowRanges.first[k]);
    }
    if (t.chunk_order > 3) { delete p; return CUTE_ERR_ARG; }
    p->info.dealtChunks = 0;
    // A launch larger than the device starts its work-groups in list order as slots come free, and every XCD walks
    // its own eighth of the list.  In panel order that goes wrong in two ways: long items that start late keep the
    // launch waiting, and a matrix whose heavy panels sit together (the hub vertices of an R-MAT graph are its first
    // rows) gives one XCD most of the work.  So if the items differ widely in length (the longest at least four times
    // the mean), or the eighths of the list differ by more than a tenth in work, the long items go first and the list
    // is dealt round-robin to the XCDs: items are ordered by the power of two of their length only, so neighbours of
    // similar length stay neighbours and keep sharing B rows in the L2.
    // Hub plans: the strips of a graph with hub vertices through persistent work-groups that keep the most
    // referenced B rows in LDS.  Opt-in (cute_tunables.hub_rows); needs the quad kernel on strip lists.
    const uint32_t hub_rows = (t.hub_rows && p->shape == 2 && d->quadRows == 4 && !chunks.empty())
                                  ? std::min<uint32_t>(std::min<uint32_t>(t.hub_rows, kMaxHubRows), d->K) : 0u;
    if (hub_rows) {
        // work items are dealt to the wavefronts of the resident work-groups in list order: longest first
        std::stable_sort(chunks.begin(), chunks.end(), [](const uint4 &a, const uint4 &b) { return a.y - a.x > b.y - b.x; });
        p->info.dealtChunks = 2;
    }
    bool longest_first = t.chunk_order == 3 && !hub_rows;
    if (t.chunk_order == 0 && !chunks.empty() && !hub_rows) {
        const uint64_t resident = uint64_t(c.num_cus) * 4u * ((p->shape == 2 || p->ng == 1) ? 8u : 4u);
        longest_first = uint64_t(chunks.size()) * num_slabs > resident;
        if (longest_first && uint64_t(longest_item) * chunks.size() < 4u * total_units) {
            const uint32_t groups = (uint32_t(chunks.size()) + cute_dev::kWavesPerGroup - 1) / cute_dev::kWavesPerGroup;
            const size_t span = size_t((groups + cute_dev::kNumXcd - 1) / cute_dev::kNumXcd) * cute_dev::kWavesPerGroup;
            uint64_t fullest = 0;
            for (uint32_t x = 0; x < cute_dev::kNumXcd; ++x) {
                uint64_t work = 0;
                for (size_t i = std::min(chunks.size(), x * span); i < std::min(chunks.size(), (x + 1) * span); ++i) work += chunks[i].y - chunks[i].x + 2u;
                fullest = std::max(fullest, work);
            }
            const uint64_t even = (total_units + 2u * chunks.size() + cute_dev::kNumXcd - 1) / cute_dev::kNumXcd;
            longest_first = fullest * 10u > even * 11u;
        }
    }
    if (longest_first && !chunks.empty()) {
        size_t place[33] = {};                 // a counting sort by the power of two of the length, longest first, stable
        auto bucket = [](const uint4 &ck) { return size_t(__builtin_clz((ck.y - ck.x) | 1u)); };
        for (const uint4 &ck : chunks) ++place[bucket(ck) + 1];
        for (size_t k = 0; k < 32; ++k) place[k + 1] += place[k];
        // work-group g runs on XCD g % 8 and takes the list positions the kernels' XCD mapping gives it: XCD x walks
        // the groups [x * per_xcd, (x + 1) * per_xcd).  The sorted groups go round-robin into those ranges.
        const uint32_t wpg = cute_dev::kWavesPerGroup;
        const uint32_t groups = (uint32_t(chunks.size()) + wpg - 1) / wpg;
        const uint32_t per_xcd = (groups + cute_dev::kNumXcd - 1) / cute_dev::kNumXcd;
        uint32_t fill[cute_dev::kNumXcd] = {}, cap[cute_dev::kNumXcd];
        for (uint32_t x = 0; x < cute_dev::kNumXcd; ++x)
            cap[x] = uint32_t(std::min<uint64_t>(per_xcd, groups > x * per_xcd ? groups - x * per_xcd : 0));
        // the last group may be short: it must stay the last one of the list
        const bool ragged = chunks.size() % wpg != 0;
        uint32_t last_xcd = 0;
        for (uint32_t x = 0; x < cute_dev::kNumXcd; ++x) if (cap[x]) last_xcd = x;
        if (ragged) cap[last_xcd]--;
        std::vector<uint32_t> to(groups);      // where the sorted groups go
        for (uint32_t k = 0; k < groups - (ragged ? 1u : 0u); ++k) {
            uint32_t x = k % cute_dev::kNumXcd;
            while (fill[x] == cap[x]) x = (x + 1) % cute_dev::kNumXcd;
            to[k] = x * per_xcd + fill[x]++;
        }
        if (ragged) to[groups - 1u] = last_xcd * per_xcd + cap[last_xcd];
        WorkItems dealt(chunks.size());
        for (const uint4 &ck : chunks) {
            const size_t i = place[bucket(ck)]++;
            dealt[size_t(to[i / wpg]) * wpg + i % wpg] = ck;
        }
        chunks.swap(dealt);
        p->info.dealtChunks = 2;
    } else
    if (t.chunk_order != 1 && !hub_rows && c.whole_chip && (p->shape == 2 || p->pipeline == 1) && !chunks.empty())
        p->info.dealtChunks = deal_chunks(chunks, num_slabs, uint32_t(c.num_cus) / cute_dev::kNumXcd,
                                          p->shape == 2 || p->ng == 1 ? 8u : 4u, t.chunk_order == 2) ? 1u : 0u;
    // the layout this plan's MFMA kernel reads, if the upload has not built it
    int rc = chunks.empty() ? int(CUTE_OK) : ensure_layout(d, p->shape);
    if (rc == CUTE_OK && hub_rows) rc = make_hub_tables(p, d, hub_rows);
    p->unitRows = CUTE_TM >> upp_log;
    // reduce_partials walks a tile along grid.y, a block of sixteen wavefronts taking 16 / G segments of 64 elements, G = 1..16
    // wavefronts to a segment by the number of pieces (see the kernel): the launch gets the blocks its tile with the most
    // pieces needs (the others leave theirs early), not one per segment -- with thousands of cut panels of two or three
    // pieces each the blocks that only start and exit otherwise cost more than the sums
    if (rc == CUTE_OK && n_pieces && (uint64_t(CUTE_TM >> upp_log) * N + 63u) / 64u > 65535u) rc = CUTE_ERR_SHAPE;
    {
        uint32_t most = 1;
        for (const uint4 &fx : fixups) most = std::max(most, fx.z);
        const uint32_t G = cute_dev::reduce_waves(most);
        const uint32_t segments = ((CUTE_TM >> upp_log) * N + 63u) / 64u, per_block = uint32_t(cute_dev::kReduceWaves) / G;
        p->reduceBlocksY = std::max(1u, (segments + per_block - 1u) / per_block);
    }
    // (the fast kernels address the partial tiles like C, with 32-bit byte offsets: checked where the chunks were made)
    p->partialBytes = uint64_t(n_pieces) * p->unitRows * N * sizeof(float);
    if (rc == CUTE_OK && (!chunks.empty() || !every_row)) {
        // The quad kernels get one 128-byte head per work item, its descriptor and a copy of its first group's record, so that
        // a wavefront can ask for its first B rows after one scalar fetch instead of two dependent ones; heads and row
        // list are gathered on the device, where the records and the row pointers are.
        const uint32_t listed = every_row ? 0u : uint32_t(row_panels.size());
        const bool heads = p->shape == 2;
        uint64_t counters = 0;                     // a unit's eights and the unit, for every slab
        for (const uint4 &fx : fixups) counters += (fx.z + cute_dev::kPiecesAtOnce - 1u) / cute_dev::kPiecesAtOnce + 1u;
        const uint64_t counter_words = counters * num_slabs * 2u;
        Layout stage, lay;
        const uint64_t sChunks = stage.add(chunks.size(), sizeof(uint4)), sFixups = stage.add(fixups.size(), sizeof(uint4)), sRows = stage.add(listed, 4),
                       sCut = stage.add(n_pieces ? 2u : 0u, sizeof(cute_dev::CutPieces)), sPieces = stage.add(n_pieces, sizeof(uint4));
        const uint64_t oChunks = lay.add(chunks.size(), heads ? cute_dev::kQuadHeadWords * 4u : sizeof(uint4)), oFixups = lay.add(fixups.size(), sizeof(uint4)),
                       oRows = lay.add(uint64_t(listed) * CUTE_TM, sizeof(uint4)), oCut = lay.add(n_pieces ? 2u : 0u, sizeof(cute_dev::CutPieces)), oPieces = lay.add(n_pieces, sizeof(uint4)),
                       oCounters = lay.add(counter_words, 4), oPartials = lay.add(p->partialBytes, 1);
        PinnedBuf pin;
        rc = pin.alloc(stage.bytes);
        if (rc == CUTE_OK && pool().take(&p->memory, lay.bytes) != CUTE_OK) rc = CUTE_ERR_NOMEM;
        if (rc == CUTE_OK) {
            std::memcpy(pin.as<char>(sChunks), chunks.data(), chunks.size() * sizeof(uint4));
            std::memcpy(pin.as<char>(sFixups), fixups.data(), fixups.size() * sizeof(uint4));
            if (listed) std::memcpy(pin.as<char>(sRows), row_panels.data(), listed * sizeof(uint32_t));
            if (heads) p->dHeads = Layout::at<uint32_t>(p->memory, oChunks);
            else p->dChunks = Layout::at<uint4>(p->memory, oChunks);
            p->dFixups = Layout::at<uint4>(p->memory, oFixups);
            p->dRowList = listed ? Layout::at<uint4>(p->memory, oRows) : nullptr;
            p->dPartials = n_pieces ? Layout::at<float>(p->memory, oPartials) : nullptr;
            if (n_pieces) {
                uint4 *of_piece = pin.as<uint4>(sPieces);
                uint32_t counter = 0;
                for (const uint4 &fx : fixups) {
                    for (uint32_t k = 0; k < fx.z; ++k) of_piece[fx.y + k] = make_uint4(fx.y, fx.z, counter, fx.x);
                    counter += (fx.z + cute_dev::kPiecesAtOnce - 1u) / cute_dev::kPiecesAtOnce + 1u;
                }
                p->dCut = Layout::at<cute_dev::CutPieces>(p->memory, oCut);
                p->dCutStatic = p->dCut + 1;
                uint4 *const dPieces = Layout::at<uint4>(p->memory, oPieces);
                uint32_t *const dCounters = Layout::at<uint32_t>(p->memory, oCounters);
                cute_dev::CutPieces *cut = pin.as<cute_dev::CutPieces>(sCut);
                cut[0] = {dPieces, dCounters, num_slabs};
                cut[1] = {dPieces, dCounters + counters * num_slabs, num_slabs};
            }
            // (the two records, the pieces behind them and the counters behind these are staged and laid out alike)
            const uint64_t cut_items = n_pieces ? (oCounters - oCut) / sizeof(uint4) : 0u;
            const cute_build::PlanTables T = {pin.as<const uint4>(sChunks), pin.as<const uint4>(sFixups), pin.as<const uint32_t>(sRows),
                                              uint32_t(chunks.size()), uint32_t(fixups.size()), listed, p->dChunks, p->dHeads, p->dFixups, p->dRowList,
                                              pin.as<const uint4>(sCut), Layout::at<uint4>(p->memory, oCut), cut_items, counter_words};
            const uint64_t items = uint64_t(chunks.size()) * (heads ? cute_dev::kQuadHeadWords : 1) + fixups.size() + uint64_t(listed) * CUTE_TM + cut_items +
                                   (counter_words + 3u) / 4u;
            pin.pending = true;
            CUTE_BUILD(cute_build::plan_tables, grid_of(items), T, heads ? (p->dHubRecs ? p->dHubRecs : d->dQRecs) : static_cast<const uint32_t *>(nullptr),
                       uint32_t(cute_dev::kQuadHeadWords), d->dRowPtr);
            rc = check_launch("plan tables");
            if (rc == CUTE_OK) rc = pin.wait();
        }
    }
    if (rc == CUTE_OK) {
        // cute_spmm_run_static's scratch: its address on this device is looked up here, at set-up, so that the
        // run call itself is nothing but kernel launches
        rc = static_scratch(&p->staticScratch);
    }
    if (rc != CUTE_OK) { cute_spmm_plan_free(p); return rc; }
    p->numFixups = uint32_t(fixups.size());
    p->numRows = num_row_panels * CUTE_TM;
    p->info.N = N;
    p->info.slabWidth = slab;
    p->info.numSlabs = num_slabs;
    p->info.numChunks = uint32_t(chunks.size());
    p->info.numAtomicChunks = n_pieces;      // chunks of cut panels (the field keeps its name from the atomics they once used)
    p->info.numBrickPanels = n_brick;
    p->info.numRowPanelsSparse = n_rows;
    p->info.numEmptyPanels = n_empty;
    p->info.slots = slots;
    p->info.precision = p->bf16x3 ? uint32_t(CUTE_PREC_BF16X3) : uint32_t(CUTE_PREC_FP32);
    p->info.path = uint32_t(t.path);
    p->columnSlabs = mfma_by_columns ? num_slabs : 0u;
    p->rowParts = num_row_panels == P && !p->windowColumns ? parts : 1u;
    p->info.mfmaShape = uint32_t(p->shape);
    p->info.hubRows = p->numHub;
    p->info.pipeline = uint32_t(p->pipeline);
    // one launch for a mixed plan: the quad kernel with any row shape of 4-float lanes, the rolling brick
    // kernel in the shapes the planner itself picks for N (forced column groups fall back to two launches)
    const bool rows_fusable = !chunks.empty() && num_row_panels && p->rows_vec == 4;
    const bool brick_default_shape = ng_for_mixed || p->ng == ((p->vec == 4 && N >= 128) ? 2 : 1);
    p->info.partialTileKiB = uint32_t((p->partialBytes + 1023u) / 1024u);
    p->info.fusedLaunch = (rows_fusable && !p->bf16x3 && !p->numHub && (p->shape == 2 || (p->pipeline == 1 && brick_default_shape))) ? 1u : 0u;
    *out = p;
    return CUTE_OK;
}

}  // extern "C"

namespace {

template <int VEC, int NG, bool FULL, bool COLUMNS, bool CUT>
void launch_brick_full(const cute_spmm_plan *p, const float *dB, float *dC, float *partials, const cute_dev::CutPieces *cut, hipStream_t s)
{
    const uint32_t groups = (p->info.numChunks + cute_dev::kWavesPerGroup - 1) / cute_dev::kWavesPerGroup;
    const uint32_t per_xcd = (groups + cute_dev::kNumXcd - 1) / cute_dev::kNumXcd;
    const dim3 grid(per_xcd * cute_dev::kNumXcd, p->info.numSlabs), block(cute_dev::kWaveSize * cute_dev::kWavesPerGroup);
    if (p->bf16x3) {
        if constexpr (VEC == 4)
            hipLaunchKernelGGL((cute_dev::hrpb_brick_bf16x3<NG, FULL, COLUMNS, CUT>), grid, block, 0, s, p->dChunks, p->info.numChunks, per_xcd,
                               p->d->dHdr, p->d->dVals, uint32_t(p->d->numVals), dB, dC, partials, p->info.N, p->columnSlabs, cut);
    } else if (p->pipeline == 1) {
#define CUTE_ROLLING_LAUNCH(TOGETHER) \
    hipLaunchKernelGGL((cute_dev::hrpb_brick_f32_rolling<VEC, NG, FULL, COLUMNS, TOGETHER, CUT>), grid, block, 0, s, p->dChunks, p->info.numChunks, per_xcd, \
                       p->d->dHdr, p->d->dVals, uint32_t(p->d->numVals), dB, dC, partials, p->info.N, p->columnSlabs, cut)
        // An item's first two header lines together where B is small, one after the other where the launch is long and memory is the bound.  9-point stencils, us
        // together / after: 300 x 300 points, N = 64 (B of 23 MB) 9.5 / 9.7, 256 x 256, N = 128 (34) 13.30 / 13.43; 396 x 396, N = 256 (160) 68.8 / 66.5, 300 x 300, N = 512
        // (184) 80.3 / 78.0, 352 x 352 111.0 / 107.2, 508 x 508 238.0 / 235.3; 600 x 600, N = 100 (144) 75.5 both, finite elements level.
        if (uint64_t(p->d->K) * p->info.N * sizeof(float) * 8u <= context().cache_bytes * 3u) CUTE_ROLLING_LAUNCH(true);
        else CUTE_ROLLING_LAUNCH(false);
#undef CUTE_ROLLING_LAUNCH
    } else
        hipLaunchKernelGGL((cute_dev::hrpb_brick_f32<VEC, NG, FULL>), grid, block, 0, s, p->dChunks, p->info.numChunks,
                           per_xcd, p->d->dHdr, p->d->dVals, dB, dC, partials, p->info.N, p->columnSlabs);
}

template <int VEC, int NG, bool CUT>
void launch_brick_as(const cute_spmm_plan *p, const float *dB, float *dC, float *partials, const cute_dev::CutPieces *cut, hipStream_t s)
{
    const bool full = p->info.N % p->info.slabWidth == 0;
    if (p->columnSlabs && full) launch_brick_full<VEC, NG, true, true, CUT>(p, dB, dC, partials, cut, s);
    else if (p->columnSlabs) launch_brick_full<VEC, NG, false, true, CUT>(p, dB, dC, partials, cut, s);
    else if (full) launch_brick_full<VEC, NG, true, false, CUT>(p, dB, dC, partials, cut, s);
    else launch_brick_full<VEC, NG, false, false, CUT>(p, dB, dC, partials, cut, s);
}

template <int VEC, int NG>
void launch_brick(const cute_spmm_plan *p, const float *dB, float *dC, float *partials, const cute_dev::CutPieces *cut, hipStream_t s)
{
    if (p->numFixups) launch_brick_as<VEC, NG, true>(p, dB, dC, partials, cut, s);
    else launch_brick_as<VEC, NG, false>(p, dB, dC, partials, cut, s);
}

template <int VEC, bool BATCHED>
void launch_rows_vec(int logl, const uint4 *row_list, uint32_t num_rows, uint32_t slabs, const uint32_t *rp,
                     const uint32_t *cl, const float *vl, const float *dB, float *dC, uint32_t N, hipStream_t s,
                     const cute_dev::XcdRanges *ranges, uint32_t blocks_per_xcd, uint32_t column_slabs)
{
    const uint64_t lanes = (uint64_t(num_rows) * slabs) << logl;
    // the batched kernel deals its blocks to the XCDs in contiguous ranges (all as long as the longest)
    const uint32_t blocks = uint32_t((lanes + 255) / 256);
    // the batched kernel walks the slabs in the grid's y dimension; the plain one folds them into x
    const dim3 grid(BATCHED ? blocks_per_xcd * cute_dev::kNumXcd : blocks, BATCHED ? slabs : 1u), block(256);
    const cute_dev::XcdRanges rg = ranges ? *ranges : cute_dev::XcdRanges{};
#define CUTE_ROWS_CASE(LL)                                                                                        \
    case LL:                                                                                                      \
        if (BATCHED && VEC == 4 && LL >= 3 && column_slabs)   /* by columns: 64 columns or more */                \
            hipLaunchKernelGGL((cute_dev::csr_rows_batched<VEC, LL, kRowBatch, VEC == 4 && LL >= 3>), grid, block, 0, s, row_list, \
                               num_rows, rp, cl, vl, dB, dC, N, rg, column_slabs);                                \
        else if (BATCHED)                                                                                         \
            hipLaunchKernelGGL((cute_dev::csr_rows_batched<VEC, LL, kRowBatch, false>), grid, block, 0, s, row_list, num_rows, \
                               rp, cl, vl, dB, dC, N, rg, 0u);                                                    \
        else                                                                                                      \
            hipLaunchKernelGGL((cute_dev::csr_rows<VEC, LL>), grid, block, 0, s, static_cast<const uint32_t *>(nullptr), num_rows, slabs, rp, \
                               cl, vl, dB, dC, N);                                                                \
        break;
    switch (logl) {
        CUTE_ROWS_CASE(0) CUTE_ROWS_CASE(1) CUTE_ROWS_CASE(2) CUTE_ROWS_CASE(3)
        CUTE_ROWS_CASE(4) CUTE_ROWS_CASE(5) CUTE_ROWS_CASE(6)
    }
#undef CUTE_ROWS_CASE
}

// batched: the library's sparse-panel kernel; otherwise the plain comparison kernel
template <bool BATCHED>
void launch_rows(int vec, int logl, const uint4 *row_list, uint32_t num_rows, uint32_t slabs, const uint32_t *rp,
                 const uint32_t *cl, const float *vl, const float *dB, float *dC, uint32_t N, hipStream_t s,
                 const cute_dev::XcdRanges *ranges = nullptr, uint32_t blocks_per_xcd = 0, uint32_t column_slabs = 0)
{
    if (vec == 4) launch_rows_vec<4, BATCHED>(logl, row_list, num_rows, slabs, rp, cl, vl, dB, dC, N, s, ranges, blocks_per_xcd, column_slabs);
    else if (vec == 2) launch_rows_vec<2, BATCHED>(logl, row_list, num_rows, slabs, rp, cl, vl, dB, dC, N, s, ranges, blocks_per_xcd, column_slabs);
    else launch_rows_vec<1, BATCHED>(logl, row_list, num_rows, slabs, rp, cl, vl, dB, dC, N, s, ranges, blocks_per_xcd, column_slabs);
}

int check_launch(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, what, __LINE__);
    return CUTE_OK;
}

int csr_launch(int alg, const uint32_t *rp, const uint32_t *cl, const float *vl, const float *dB, float *dC, uint32_t M,
               uint32_t N, hipStream_t s)
{
    if (M == 0 || N == 0) return CUTE_ERR_SHAPE;
    switch (alg) {
        case 0:
            hipLaunchKernelGGL(cute_dev::csr_thread_per_element, dim3((N + 63) / 64, (M + 3) / 4), dim3(64, 4), 0, s, rp,
                               cl, vl, dB, dC, M, N);
            break;
        case 1:
            hipLaunchKernelGGL(cute_dev::csr_wave_scalar, dim3(uint32_t((uint64_t(M) * 64 + 255) / 256)), dim3(256), 0,
                               s, rp, cl, vl, dB, dC, M, N);
            break;
        case 2: {
            const int vec = lane_floats(N);
            uint32_t need = (N + vec - 1) / vec, logl = 0;
            while ((1u << logl) < need && logl < 6) ++logl;
            const uint32_t w = (1u << logl) * vec;
            launch_rows<false>(vec, int(logl), nullptr, M, (N + w - 1) / w, rp, cl, vl, dB, dC, N, s);
            break;
        }
        default: return CUTE_ERR_ARG;
    }
    return check_launch("csr kernel launch");
}

}  // namespace

namespace {
template <class Launch>
int time_launches(hipStream_t s, int warmup, int iters, float *ms_out, Launch launch)
{
    if (iters < 1 || !ms_out) return CUTE_ERR_ARG;
    std::vector<hipEvent_t> ev(size_t(iters) * 2, nullptr);
    int rc = CUTE_OK;
    for (auto &e : ev)
        if (rc == CUTE_OK && hipEventCreate(&e) != hipSuccess) rc = CUTE_ERR_HIP;
    for (int i = 0; i < warmup && rc == CUTE_OK; ++i) rc = launch();
    for (int i = 0; i < iters && rc == CUTE_OK; ++i) {
        (void)hipEventRecord(ev[2 * i], s);
        rc = launch();
        (void)hipEventRecord(ev[2 * i + 1], s);
    }
    if (rc == CUTE_OK && hipStreamSynchronize(s) != hipSuccess) rc = CUTE_ERR_HIP;
    for (int i = 0; i < iters && rc == CUTE_OK; ++i)
        if (hipEventElapsedTime(&ms_out[i], ev[2 * i], ev[2 * i + 1]) != hipSuccess) rc = CUTE_ERR_HIP;
    for (auto &e : ev)
        if (e) (void)hipEventDestroy(e);
    return rc;
}
}  // namespace

struct cute_blocked_ell_dev {
    int32_t blockSize = 0, height = 0, width = 0;
    int32_t *dColIdx = nullptr;
    float *dValues = nullptr;
};

struct cute_hybrid {
    cute_hybrid_info info{};
    uint32_t rows = 0;
    cute_blocked_ell_dev *ell = nullptr;    // heavy tiles (absent when no tile is heavy)
    uint32_t *dRowPtr = nullptr, *dCols = nullptr;
    float *dVals = nullptr;                 // the remainder as CSR
};

namespace {
template <int VEC, bool ACC>
void launch_blocked_ell(const cute_blocked_ell_dev *d, const float *dB, float *dC, uint32_t N, hipStream_t s)
{
    const uint32_t rows = uint32_t(d->height) * uint32_t(d->blockSize), strips = rows / 16u;
    // x extent a multiple of the XCD count: the kernel maps x so that each XCD owns a contiguous range of strips
    const uint32_t groups = (((strips + 3u) / 4u + 7u) / 8u) * 8u;
    const dim3 grid(groups, (N + 16u * VEC - 1u) / (16u * VEC)), block(256);
    if (N % (16u * VEC) == 0)
        hipLaunchKernelGGL((cute_dev::blocked_ell_f32<VEC, true, ACC>), grid, block, 0, s, d->dColIdx, d->dValues,
                           uint32_t(d->blockSize), uint32_t(d->width), strips, rows, dB, dC, N);
    else
        hipLaunchKernelGGL((cute_dev::blocked_ell_f32<VEC, false, ACC>), grid, block, 0, s, d->dColIdx, d->dValues,
                           uint32_t(d->blockSize), uint32_t(d->width), strips, rows, dB, dC, N);
}
}  // namespace

namespace {
// Brick chunks and sparse rows in one launch.  (VEC, NG, lanes per row) follow from N the way the planner
// picks them; returns false for a combination that is not instantiated (the caller then launches twice).
template <int VEC, int NG, int LOG_L>
void launch_brick_rows_as(const cute_spmm_plan *p, const float *dB, float *dC, float *partials, const cute_dev::CutPieces *cut, hipStream_t s, const dim3 &grid,
                          uint32_t per_xcd)
{
    const uint32_t N = p->info.N;
    const uint32_t rows_per_slab = p->rowBlocksPerXcd * cute_dev::kNumXcd;
    const uint64_t brick_blocks = uint64_t(grid.x) * grid.y, row_blocks = uint64_t(rows_per_slab) * p->rows_slabs;
    const dim3 flat(uint32_t(brick_blocks + row_blocks)), block(cute_dev::kWaveSize * cute_dev::kWavesPerGroup);
#define CUTE_BRICK_ROWS_AS(F, COLUMNS, CUT)                                                                               \
    hipLaunchKernelGGL((cute_dev::hrpb_brick_rows_f32<VEC, NG, F, LOG_L, COLUMNS, CUT>), flat, block, 0, s, grid.x, uint32_t(brick_blocks),  \
                       p->dChunks, p->info.numChunks, per_xcd, p->d->dHdr, p->d->dVals, uint32_t(p->d->numVals), p->dRowList, \
                       p->numRows, rows_per_slab, p->rowRanges, p->columnSlabs, p->rowColumnSlabs, p->d->dRowPtr, p->d->dCols, p->d->dCsrVals,                    \
                       dB, dC, partials, N, cut)
#define CUTE_BRICK_ROWS(F, COLUMNS)                               \
    {                                                             \
        if (p->numFixups) CUTE_BRICK_ROWS_AS(F, COLUMNS, true);   \
        else CUTE_BRICK_ROWS_AS(F, COLUMNS, false);               \
    }
    constexpr bool wide = LOG_L >= 5;            // a launch by columns has 128 columns or more
    const bool full = N % (16u * VEC * NG) == 0;
    if (wide && p->columnSlabs && full) CUTE_BRICK_ROWS(true, wide)
    else if (wide && p->columnSlabs) CUTE_BRICK_ROWS(false, wide)
    else if (full) CUTE_BRICK_ROWS(true, false)
    else CUTE_BRICK_ROWS(false, false)
#undef CUTE_BRICK_ROWS
#undef CUTE_BRICK_ROWS_AS
}

bool launch_brick_rows(const cute_spmm_plan *p, const float *dB, float *dC, float *partials, const cute_dev::CutPieces *cut, hipStream_t s)
{
    const uint32_t groups = (p->info.numChunks + cute_dev::kWavesPerGroup - 1) / cute_dev::kWavesPerGroup;
    const uint32_t per_xcd = (groups + cute_dev::kNumXcd - 1) / cute_dev::kNumXcd;
    const dim3 grid(per_xcd * cute_dev::kNumXcd, p->info.numSlabs);
    if (uint64_t(grid.x) * grid.y + uint64_t(p->rowBlocksPerXcd) * cute_dev::kNumXcd * p->rows_slabs >= 0x7fffffffull) return false;
    const int v = p->vec, g = p->ng, l = p->rows_logl;
    if (v == 1 && g == 1 && l == 0) launch_brick_rows_as<1, 1, 0>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 1 && g == 1 && l == 1) launch_brick_rows_as<1, 1, 1>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 1 && g == 1 && l == 2) launch_brick_rows_as<1, 1, 2>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 2 && g == 1 && l == 3) launch_brick_rows_as<2, 1, 3>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 4 && g == 1 && l == 4) launch_brick_rows_as<4, 1, 4>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 4 && g == 1 && l == 5) launch_brick_rows_as<4, 1, 5>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 4 && g == 1 && l == 6) launch_brick_rows_as<4, 1, 6>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 4 && g == 2 && l == 5) launch_brick_rows_as<4, 2, 5>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else if (v == 4 && g == 2 && l == 6) launch_brick_rows_as<4, 2, 6>(p, dB, dC, partials, cut, s, grid, per_xcd);
    else return false;
    return true;
}
}  // namespace

namespace {
// The launches of one product; `partials` is where the pieces of cut panels store their tiles, `cut` how they add themselves up
// (nullptr: reduce_partials does).
int run_with(const cute_spmm_plan *p, const float *dB, float *dC, void *stream, float *partials, const cute_dev::CutPieces *cut)
{
    if (!p || !dB || !dC) return CUTE_ERR_ARG;
    if ((reinterpret_cast<uintptr_t>(dB) | reinterpret_cast<uintptr_t>(dC)) & 15u) return CUTE_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t N = p->info.N;
    if (p->numHub || (p->shape == 1 && p->pipeline != 1)) cut = nullptr;      // (these kernels leave the tiles to reduce_partials)
    bool rows_launched = false;        // the sparse rows went out together with the MFMA chunks
    if (p->info.numChunks && p->shape == 2 && p->numHub) {
        // persistent work-groups of sixteen wavefronts, two per compute unit, each with the hub rows of its slab in LDS
        const uint32_t wgs = std::min<uint32_t>(2u * uint32_t(context().num_cus), (p->info.numChunks + cute_dev::kHubWaves - 1) / cute_dev::kHubWaves);
        const dim3 grid(wgs, p->info.numSlabs), block(cute_dev::kWaveSize * cute_dev::kHubWaves);
        const size_t lds = size_t(p->numHub) * cute_dev::kWaveSize * sizeof(float);
        if (N % 64u == 0)
            hipLaunchKernelGGL((cute_dev::hrpb_quad_hub_f32<true>), grid, block, lds, s, p->dHeads, p->info.numChunks, p->dHubRecs,
                               p->d->dQVals, uint32_t(p->d->numQuadVals), p->dHubRows, p->numHub, dB, dC, partials, N);
        else
            hipLaunchKernelGGL((cute_dev::hrpb_quad_hub_f32<false>), grid, block, lds, s, p->dHeads, p->info.numChunks, p->dHubRecs,
                               p->d->dQVals, uint32_t(p->d->numQuadVals), p->dHubRows, p->numHub, dB, dC, partials, N);
    } else if (p->info.numChunks && p->shape == 2) {
        const uint32_t groups = (p->info.numChunks + cute_dev::kWavesPerGroup - 1) / cute_dev::kWavesPerGroup;
        const uint32_t per_xcd = (groups + cute_dev::kNumXcd - 1) / cute_dev::kNumXcd;
        const dim3 grid(per_xcd * cute_dev::kNumXcd, p->info.numSlabs), block(cute_dev::kWaveSize * cute_dev::kWavesPerGroup);
        const bool full = N % 64u == 0, strips = p->d->quadRows == 4, pieces = p->numFixups != 0;
        // mixed plan: quad chunks and sparse rows in one launch (instantiated for 4-float lanes and 4..64 lanes per row)
        const uint32_t rows_per_slab = p->rowBlocksPerXcd * cute_dev::kNumXcd;
        const uint64_t row_blocks = uint64_t(rows_per_slab) * p->rows_slabs, quad_blocks = uint64_t(grid.x) * grid.y;
        if (p->info.fusedLaunch && quad_blocks + row_blocks < 0x7fffffffull) {
#define CUTE_FUSED_LAUNCH_AS(F, S, LL, COLUMNS, CUT)                                                                      \
    hipLaunchKernelGGL((cute_dev::hrpb_quad_rows_f32<F, S, LL, COLUMNS, CUT>), dim3(uint32_t(quad_blocks + row_blocks)), block, 0, s,     \
                       grid.x, uint32_t(quad_blocks), p->dHeads, p->info.numChunks, per_xcd, p->d->dQRecs, p->d->dQVals,   \
                       uint32_t(p->d->numQuadVals),                                                                  \
                       p->dRowList, p->numRows, rows_per_slab, p->rowRanges, p->columnSlabs, p->rowColumnSlabs, p->d->dRowPtr, p->d->dCols, p->d->dCsrVals, dB, dC,    \
                       partials, N, cut)
#define CUTE_FUSED_LAUNCH(F, S, LL, COLUMNS)                                    \
    {                                                                           \
        if (pieces) CUTE_FUSED_LAUNCH_AS(F, S, LL, COLUMNS, true);              \
        else CUTE_FUSED_LAUNCH_AS(F, S, LL, COLUMNS, false);                    \
    }
#define CUTE_FUSED_LL(F, S)                                                     \
    switch (p->rows_logl) {                                                     \
        case 0: CUTE_FUSED_LAUNCH(F, S, 0, false) break;                        \
        case 1: CUTE_FUSED_LAUNCH(F, S, 1, false) break;                        \
        case 2: CUTE_FUSED_LAUNCH(F, S, 2, false) break;                        \
        case 3: CUTE_FUSED_LAUNCH(F, S, 3, false) break;                        \
        case 4:   /* by columns: sixteen lanes a row */                         \
            if (p->columnSlabs) CUTE_FUSED_LAUNCH(F, S, 4, true)                \
            else CUTE_FUSED_LAUNCH(F, S, 4, false)                              \
            break;                                                              \
        case 5: CUTE_FUSED_LAUNCH(F, S, 5, false) break;                        \
        default: CUTE_FUSED_LAUNCH(F, S, 6, false) break;                       \
    }
            if (full && strips) { CUTE_FUSED_LL(true, true) }
            else if (full) { CUTE_FUSED_LL(true, false) }
            else if (strips) { CUTE_FUSED_LL(false, true) }
            else { CUTE_FUSED_LL(false, false) }
#undef CUTE_FUSED_LL
#undef CUTE_FUSED_LAUNCH
#undef CUTE_FUSED_LAUNCH_AS
            rows_launched = true;
        } else if (p->halfLists) {
#define CUTE_HALF_LAUNCH(S, CUT)                                                                                         \
    hipLaunchKernelGGL((cute_dev::hrpb_quad_half_f32<S, CUT>), grid, block, 0, s, p->dHeads, p->info.numChunks, per_xcd, p->d->dQRecs, \
                       p->d->dQVals, uint32_t(p->d->numQuadVals), dB, dC, partials, N, p->columnSlabs, cut)
            if (strips && pieces) CUTE_HALF_LAUNCH(true, true);
            else if (strips) CUTE_HALF_LAUNCH(true, false);
            else if (pieces) CUTE_HALF_LAUNCH(false, true);
            else CUTE_HALF_LAUNCH(false, false);
#undef CUTE_HALF_LAUNCH
        } else {
#define CUTE_QUAD_LAUNCH_AS(F, S, COLUMNS, CUT)                                                                          \
    hipLaunchKernelGGL((cute_dev::hrpb_quad_f32<F, S, COLUMNS, CUT>), grid, block, 0, s, p->dHeads, p->info.numChunks, per_xcd, \
                       p->d->dQRecs, p->d->dQVals, uint32_t(p->d->numQuadVals), dB, dC, partials, N, p->columnSlabs, cut)
#define CUTE_QUAD_LAUNCH(F, S)                                                  \
    if (p->columnSlabs && pieces) CUTE_QUAD_LAUNCH_AS(F, S, true, true);        \
    else if (p->columnSlabs) CUTE_QUAD_LAUNCH_AS(F, S, true, false);            \
    else if (pieces) CUTE_QUAD_LAUNCH_AS(F, S, false, true);                    \
    else CUTE_QUAD_LAUNCH_AS(F, S, false, false)
            if (full && strips) { CUTE_QUAD_LAUNCH(true, true); }
            else if (full) { CUTE_QUAD_LAUNCH(true, false); }
            else if (strips) { CUTE_QUAD_LAUNCH(false, true); }
            else { CUTE_QUAD_LAUNCH(false, false); }
#undef CUTE_QUAD_LAUNCH_AS
#undef CUTE_QUAD_LAUNCH
        }
    } else if (p->info.numChunks) {
        if (p->info.fusedLaunch && launch_brick_rows(p, dB, dC, partials, cut, s)) rows_launched = true;
        else if (p->vec == 4 && p->ng == 2) launch_brick<4, 2>(p, dB, dC, partials, cut, s);
        else if (p->vec == 4) launch_brick<4, 1>(p, dB, dC, partials, cut, s);
        else if (p->vec == 2) launch_brick<2, 1>(p, dB, dC, partials, cut, s);
        else launch_brick<1, 1>(p, dB, dC, partials, cut, s);
    }
    if (p->windowColumns) {
        const uint32_t slabs = (N + p->windowColumns - 1u) / p->windowColumns;
        const dim3 grid(p->windowChains * slabs), block(1024);
#define CUTE_WINDOW_LAUNCH(W, WARM)                                                                                              \
    hipLaunchKernelGGL((cute_dev::csr_rows_window<W, WARM>), grid, block, 0, s, p->d->dSlices, p->d->dWindowSlots, p->d->dWindowVals, \
                       p->d->dWindowTiles, (p->d->M + cute_dev::kWindowTile - 1u) / cute_dev::kWindowTile, p->windowChainTiles,   \
                       p->windowChains, slabs, dB, dC, p->d->M, N)
        if (p->windowColumns == 16u) { if (p->windowWarm) CUTE_WINDOW_LAUNCH(16, true); else CUTE_WINDOW_LAUNCH(16, false); }
        else { if (p->windowWarm) CUTE_WINDOW_LAUNCH(8, true); else CUTE_WINDOW_LAUNCH(8, false); }
#undef CUTE_WINDOW_LAUNCH
    } else if (p->rowParts > 1u) {
        uint32_t log_lanes = 0;
        while (uint32_t(p->rows_vec) << log_lanes < N) ++log_lanes;
        const uint32_t log_parts = uint32_t(__builtin_ctz(p->rowParts));
        const uint64_t threads = uint64_t(p->d->M) << (log_lanes + log_parts);
        const uint32_t per_xcd = uint32_t((threads + 256u * cute_dev::kNumXcd - 1u) / (256u * cute_dev::kNumXcd));
#define CUTE_SPLIT_LAUNCH(VEC)                                                                                                    \
    hipLaunchKernelGGL(cute_dev::csr_rows_split<VEC>, dim3(per_xcd * cute_dev::kNumXcd), dim3(256), 0, s, p->d->dRowPtr, p->d->dCols, p->d->dCsrVals, dB, dC, \
                       p->d->M, N, log_lanes, log_parts, per_xcd)
        if (p->rows_vec == 4) CUTE_SPLIT_LAUNCH(4);
        else if (p->rows_vec == 2) CUTE_SPLIT_LAUNCH(2);
        else CUTE_SPLIT_LAUNCH(1);
#undef CUTE_SPLIT_LAUNCH
    } else if (p->numRows && !rows_launched) {
        launch_rows<true>(p->rows_vec, p->rows_logl, p->dRowList, p->numRows, p->rows_slabs, p->d->dRowPtr, p->d->dCols,
                    p->d->dCsrVals, dB, dC, N, s, &p->rowRanges, p->rowBlocksPerXcd, p->rowColumnSlabs);
    }
    if (p->numFixups && !cut)
        hipLaunchKernelGGL(cute_dev::reduce_partials, dim3(p->numFixups, p->reduceBlocksY),
                           dim3(cute_dev::kWaveSize * cute_dev::kReduceWaves), 0, s, p->dFixups, p->numFixups, p->unitRows,
                           partials, dC, N);
    return check_launch("spmm launch");
}
}  // namespace

extern "C" {

// Replaces SPMM_TC::run (spmm.cu:823-839): picks the kernel instantiation from N and
// launches asynchronously on `stream`.
int cute_spmm_run(cute_spmm_plan *p, const float *dB, float *dC, void *stream)
{
    if (!p) return CUTE_ERR_ARG;
    return run_with(p, dB, dC, stream, p->dPartials, p->dCut);
}

// The same launches with the partial tiles in the library's static device array instead of the plan's
// buffer: no allocation, no copy, no memset, no synchronisation -- kernel launches only.
int cute_spmm_run_static(cute_spmm_plan *p, const float *dB, float *dC, void *stream)
{
    if (!p) return CUTE_ERR_ARG;
    if (p->partialBytes > uint64_t(CUTE_STATIC_SCRATCH_BYTES)) {
        g_hip_error = "plan needs " + std::to_string(p->partialBytes) + " bytes of partial tiles, the static scratch holds " +
                      std::to_string(uint64_t(CUTE_STATIC_SCRATCH_BYTES));
        return CUTE_ERR_SCRATCH;
    }
    return run_with(p, dB, dC, stream, static_cast<float *>(p->staticScratch), p->dCutStatic);   // the address was fetched when the plan was made
}

uint64_t cute_spmm_plan_scratch_bytes(const cute_spmm_plan *p) { return p ? p->partialBytes : 0; }

// The same launches with the partial tiles in memory the caller brings: one plan can then run on several
// streams at once, each call with a buffer of its own.
int cute_spmm_run_scratch(cute_spmm_plan *p, const float *dB, float *dC, void *stream, void *scratch, uint64_t scratch_bytes)
{
    if (!p) return CUTE_ERR_ARG;
    if (p->partialBytes) {
        if (!scratch || (reinterpret_cast<uintptr_t>(scratch) & 15u)) return CUTE_ERR_ARG;
        if (scratch_bytes < p->partialBytes) {
            g_hip_error = "plan needs " + std::to_string(p->partialBytes) + " bytes of partial tiles, the caller's scratch holds " +
                          std::to_string(scratch_bytes);
            return CUTE_ERR_SCRATCH;
        }
    }
    return run_with(p, dB, dC, stream, static_cast<float *>(scratch), nullptr);
}

int cute_csr_spmm_dev(int alg, const uint32_t *dRowPtr, const uint32_t *dCols, const float *dVals, const float *dB,
                      float *dC, uint32_t M, uint32_t N, void *stream)
{
    if (!dRowPtr || !dB || !dC) return CUTE_ERR_ARG;
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    return csr_launch(alg, dRowPtr, dCols, dVals, dB, dC, M, N, static_cast<hipStream_t>(stream));
}


void cute_blocked_ell_dev_free(cute_blocked_ell_dev *d)
{
    if (!d) return;
    (void)hipFree(d->dColIdx);
    (void)hipFree(d->dValues);
    delete d;
}

int cute_blocked_ell_upload(const cute_blocked_ell *e, cute_blocked_ell_dev **out)
{
    if (!e || !out || e->blockSize <= 0 || e->height < 0 || e->width < 0) return CUTE_ERR_ARG;
    *out = nullptr;
    if (e->blockSize % 16) return CUTE_ERR_SHAPE;        // the kernel walks 16 x 16 tiles
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    cute_blocked_ell_dev *d = new cute_blocked_ell_dev;
    d->blockSize = e->blockSize; d->height = e->height; d->width = e->width;
    const uint64_t cells = uint64_t(e->height) * uint64_t(e->width);
    int rc = upload(&d->dColIdx, e->ellColIdx, cells);
    if (rc == CUTE_OK) rc = upload(&d->dValues, e->ellValues, cells * uint64_t(e->blockSize) * uint64_t(e->blockSize));
    if (rc != CUTE_OK) { cute_blocked_ell_dev_free(d); return rc; }
    *out = d;
    return CUTE_OK;
}


// C[height*blockSize x N] (+)= ELL . B[ncols x N], device pointers, asynchronous on `stream`.
int cute_blocked_ell_spmm(const cute_blocked_ell_dev *d, const float *dB, float *dC, uint32_t N, int accumulate, void *stream)
{
    if (!d || !dB || !dC) return CUTE_ERR_ARG;
    if (N == 0) return CUTE_ERR_SHAPE;
    if ((reinterpret_cast<uintptr_t>(dB) | reinterpret_cast<uintptr_t>(dC)) & 15u) return CUTE_ERR_ARG;
    if (d->height == 0) return CUTE_OK;
    if ((N + 15u) / 16u > 65535u) return CUTE_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int vec = (N % 4 == 0) ? 4 : (N % 2 == 0) ? 2 : 1;
    if (accumulate) {
        if (vec == 4) launch_blocked_ell<4, true>(d, dB, dC, N, s);
        else if (vec == 2) launch_blocked_ell<2, true>(d, dB, dC, N, s);
        else launch_blocked_ell<1, true>(d, dB, dC, N, s);
    } else {
        if (vec == 4) launch_blocked_ell<4, false>(d, dB, dC, N, s);
        else if (vec == 2) launch_blocked_ell<2, false>(d, dB, dC, N, s);
        else launch_blocked_ell<1, false>(d, dB, dC, N, s);
    }
    return check_launch("blocked-ELL launch");
}

// ------------------------------------------------------------------------------------------------
// The hybrid the reference's earlier prototypes model (inc/SPMM.cuh:2528-2933 GPU_Compute_Multi_Kernel*,
// the 2-D variant at :2898: tiles with more than THRESHOLD entries go to the tensor cores as dense tiles,
// the rest to a plain kernel; inc/splitter.hpp and inc/preprocess.hpp:172-193 are its two split rules):
// heavy tiles as a Blocked-ELL matrix through blocked_ell_f32 (fp32 MFMA), the remainder through the CSR
// row kernel, both into one C.
// ------------------------------------------------------------------------------------------------
void cute_hybrid_free(cute_hybrid *h)
{
    if (!h) return;
    cute_blocked_ell_dev_free(h->ell);
    (void)hipFree(h->dRowPtr);
    (void)hipFree(h->dCols);
    (void)hipFree(h->dVals);
    delete h;
}

int cute_hybrid_create(const cute_csr_i32 *csr, int32_t tile_size, int32_t nnz_threshold, int32_t mode, float deviation_threshold,
                       float underload_dominance, cute_hybrid **out)
{
    if (!csr || !out || !csr->rowPtr || (mode != CUTE_HYBRID_SPLITTER && mode != CUTE_HYBRID_CLASSIFIER)) return CUTE_ERR_ARG;
    *out = nullptr;
    if (tile_size <= 0 || tile_size % 16 || csr->nrows <= 0 || csr->nrows % tile_size || csr->ncols % tile_size) return CUTE_ERR_SHAPE;
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return c.status;
    cute_hybrid *h = new cute_hybrid;
    h->info.tileSize = tile_size;
    h->info.mode = mode;
    h->rows = uint32_t(csr->nrows);
    int rc = cute_block_stats(csr, tile_size, h->info.stats);
    cute_split sp{};
    if (rc == CUTE_OK) {
        if (mode == CUTE_HYBRID_SPLITTER) {
            // Threshold 0: the fill from which a tile pays for itself on the matrix cores, measured on gfx950 with this
            // library's two kernels (16 384^2 matrices, a sparse background plus 20 000 tiles of a given fill, N = 128):
            // tiles 10 % full lose 10 us by moving to the Blocked-ELL part (37.6 against 27.9 us), tiles 20 % full win 9 us
            // (36.2 against 45.6), tiles 30 % full 28 us -- the break-even is near 15 % of the tile's cells.  And a heavy
            // part that would hold less than 2 % of the entries is not worth its own launch (14 tiles of the FEM
            // benchmark matrix: +9 us): everything then stays with the row kernel.
            const bool automatic = nnz_threshold <= 0;
            if (automatic) nnz_threshold = std::max(1, int32_t(std::ceil(kHybridFill * float(tile_size) * float(tile_size))));
            rc = cute_splitter_split(csr, tile_size, nnz_threshold, &sp);
            if (rc == CUTE_OK && automatic && sp.numHeavyElems && int64_t(sp.numHeavyElems) * 50 < int64_t(csr->nnz)) {
                cute_split_release(&sp);
                nnz_threshold = tile_size * tile_size + 1;
                rc = cute_splitter_split(csr, tile_size, nnz_threshold, &sp);
            }
        } else {
            rc = cute_split_by_class(csr, tile_size, deviation_threshold, underload_dominance, &sp);
            nnz_threshold = 0;
        }
    }
    h->info.threshold = nnz_threshold;
    cute_csr_i32 heavy{}, light{};
    cute_blocked_ell ell{};
    if (rc == CUTE_OK) {
        h->info.totalTiles = sp.totalTiles;
        h->info.heavyTiles = sp.numHeavyTiles; h->info.heavyElems = sp.numHeavyElems;
        h->info.lightTiles = sp.numLightTiles; h->info.lightElems = sp.numLightElems;
        rc = cute_coo_to_csr(&sp.light, &light);
    }
    if (rc == CUTE_OK && sp.numHeavyElems) rc = cute_coo_to_csr(&sp.heavy, &heavy);
    if (rc == CUTE_OK && sp.numHeavyElems) rc = cute_blocked_ell_build(&heavy, tile_size, &ell);
    if (rc == CUTE_OK && sp.numHeavyElems) {
        h->info.ellHeight = ell.height;
        h->info.ellWidth = ell.width;
        rc = cute_blocked_ell_upload(&ell, &h->ell);
    }
    if (rc == CUTE_OK) rc = upload(&h->dRowPtr, reinterpret_cast<const uint32_t *>(light.rowPtr), uint64_t(csr->nrows) + 1);
    if (rc == CUTE_OK) rc = upload(&h->dCols, reinterpret_cast<const uint32_t *>(light.cols), uint64_t(light.nnz));
    if (rc == CUTE_OK) rc = upload(&h->dVals, light.values, uint64_t(light.nnz));
    cute_blocked_ell_release(&ell);
    cute_csr_i32_release(&heavy);
    cute_csr_i32_release(&light);
    cute_split_release(&sp);
    if (rc != CUTE_OK) { cute_hybrid_free(h); return rc; }
    *out = h;
    return CUTE_OK;
}

int cute_hybrid_get_info(const cute_hybrid *h, cute_hybrid_info *out)
{
    if (!h || !out) return CUTE_ERR_ARG;
    *out = h->info;
    return CUTE_OK;
}

// C[nrows x N] = A . B: the remainder through the row kernel (which writes every row of C), then the heavy tiles
// added on top by the Blocked-ELL kernel; both asynchronous on `stream`, in that order.
int cute_hybrid_spmm(const cute_hybrid *h, const float *dB, float *dC, uint32_t N, void *stream)
{
    if (!h || !dB || !dC) return CUTE_ERR_ARG;
    if (N == 0) return CUTE_ERR_SHAPE;
    if ((reinterpret_cast<uintptr_t>(dB) | reinterpret_cast<uintptr_t>(dC)) & 15u) return CUTE_ERR_ARG;
    int rc = csr_launch(2, h->dRowPtr, h->dCols, h->dVals, dB, dC, h->rows, N, static_cast<hipStream_t>(stream));
    if (rc == CUTE_OK && h->ell) rc = cute_blocked_ell_spmm(h->ell, dB, dC, N, 1, stream);
    return rc;
}

// Shape of GPU_CSR_cuSPARSE_NEW (spmm.cu:860-960): host arrays in, host C out, one warm-up
// launch then `iters` timed launches between two events; returns ms per launch.
float cute_gpu_csr_spmm(const uint32_t *rowPtr, const uint32_t *cols, const float *vals, uint32_t nnz, const float *hB,
                        float *hC, uint32_t m, uint32_t k, uint32_t n, int iters, int alg)
{
    if (!rowPtr || !hB || !hC || iters < 1) return float(CUTE_ERR_ARG);
    const DeviceContext &c = context();
    if (c.status != CUTE_OK) return float(c.status);
    uint32_t *dR = nullptr, *dCl = nullptr;
    float *dV = nullptr, *dB = nullptr, *dC = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float ms = 0.0f;
    int rc = upload(&dR, rowPtr, uint64_t(m) + 1);
    if (rc == CUTE_OK) rc = upload(&dCl, cols, nnz);
    if (rc == CUTE_OK) rc = upload(&dV, vals, nnz);
    if (rc == CUTE_OK) rc = upload(&dB, hB, uint64_t(k) * n);
    if (rc == CUTE_OK && device_malloc(reinterpret_cast<void **>(&dC), uint64_t(m) * n * sizeof(float)) != hipSuccess)
        rc = CUTE_ERR_HIP;
    if (rc == CUTE_OK) rc = csr_launch(alg, dR, dCl, dV, dB, dC, m, n, nullptr);
    if (rc == CUTE_OK && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)) rc = CUTE_ERR_HIP;
    if (rc == CUTE_OK) {
        (void)hipEventRecord(e0, nullptr);
        for (int i = 0; i < iters && rc == CUTE_OK; ++i) rc = csr_launch(alg, dR, dCl, dV, dB, dC, m, n, nullptr);
        (void)hipEventRecord(e1, nullptr);
        if (hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = CUTE_ERR_HIP;
    }
    if (rc == CUTE_OK && hipMemcpy(hC, dC, uint64_t(m) * n * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
        rc = CUTE_ERR_HIP;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(dR); (void)hipFree(dCl); (void)hipFree(dV); (void)hipFree(dB); (void)hipFree(dC);
    return rc == CUTE_OK ? ms / float(iters) : float(rc);
}

int cute_spmm_time(cute_spmm_plan *p, const float *dB, float *dC, void *stream, int warmup, int iters, float *ms_out)
{
    if (!p) return CUTE_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return time_launches(s, warmup, iters, ms_out, [&] { return cute_spmm_run(p, dB, dC, stream); });
}

int cute_csr_spmm_time(int alg, const cute_hrpb_dev *d, const float *dB, float *dC, uint32_t N, void *stream, int warmup,
                       int iters, float *ms_out)
{
    if (!d) return CUTE_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return time_launches(s, warmup, iters, ms_out,
                         [&] { return csr_launch(alg, d->dRowPtr, d->dCols, d->dCsrVals, dB, dC, d->M, N, s); });
}

}  // extern "C"
