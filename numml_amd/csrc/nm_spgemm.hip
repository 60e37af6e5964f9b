// Hash-based CSR x CSR product (SpGEMM) and its backward for gfx950.
//
// Forward, two phases around the caller's allocation of C:
//   symbolic: rows of A are binned by an upper bound on their products
//             (sum of the lengths of the B rows they touch).  A group of lanes
//             (8 or 16, by bin) or a workgroup (longer rows) inserts the row's
//             column indices into a hash set in LDS and counts the distinct
//             ones; an exclusive scan of the counts is C_indptr.
//   numeric : rows are re-binned by their exact length.  The group accumulates
//             (column, value) pairs in an LDS hash table, walking A's row
//             entry by entry and B's row across the lanes (a workgroup deals
//             the products of a longer row to its threads and lets those that
//             meet in an entry take turns), so every output
//             entry receives its products in the order of A's row -- the
//             order of the serial SMMP loop (cpp/sparse_csr_cpu.cpp:182-212) --
//             and then writes the table out ranked by column, so C's rows are
//             ascending like the reference's.
// Rows too long for an LDS table spill to a dense accumulator in global memory
// (one slice of B_cols entries per spill workgroup).
// Short rows take a merge path instead of hashing: when a row of A and every row
// of B it names have at most 8 entries (stencil and aggregation operators), eight
// lanes each hold one B row, sorted as stored, and the group repeatedly emits the
// smallest head column; the lanes whose head equals it contribute their product,
// summed in lane order = the order of A's row.  These rows never enter the bins.
//
// Backward: eight lanes per row i of A; for each entry (i,k) the lanes share row
// k of B, find its columns in row i of C (staged in LDS) by bisection, and form
// grad_A (a sum in ascending column order, as the reference's merge,
// cpp/sparse_csr_cpu.cpp:246-278) and grad_B (atomic adds, one cache line per
// entry of A) in one pass.
//
// Algorithmic HBM bytes of the forward (s = sizeof(value)):
//   nnzA*(s+8) + rowsA*8 + products*(s+8) [upper; nnzB*(s+8) compulsory]
//   + nnzC*(s+8) + rowsA*8
#include "nm_common.hpp"
#include "nm_scan.hpp"
#include "nm_spgemm_plan.hpp"

namespace {

using nm::kWave;

constexpr int32_t kEmpty = -1;
constexpr int kBlock = 256;
constexpr int kBins = 10;
constexpr int kBinStart = 10, kBinCursor = 21, kBinInts = 32;   // layout of the bins array, see Work
// Workgroups (and dense accumulator slices of B_cols entries each) of the spill path: as many as
// fit a fixed budget of scratch, between 8 and 64.
constexpr int64_t kSpillBudgetBytes = int64_t(192) << 20;
inline int spill_groups(int64_t B_cols) {
    const int64_t g = kSpillBudgetBytes / (12 * (B_cols + 1));
    return (int)(g < 8 ? 8 : (g > 64 ? 64 : g));
}
constexpr int kSpillBlock = 1024;
constexpr int kTablePad = 4;         // entries between the hash tables of neighbouring groups (16 bytes)
constexpr int kAhead = 8;            // B rows whose first columns a group requests before inserting any
#ifndef NM_HASH_BATCH
#define NM_HASH_BATCH 8
#endif

// bin upper limits (inclusive); the last bin takes the rest and spills
// on the product bound (the symbolic phase has a bin less than the numeric one: the eighth takes no row)
constexpr int32_t kSymLimit[kBins - 1] = {64, 128, 256, 512, 1024, 2048, 8192, 24576, 24576};
// on the exact row length; the last one is what a whole CU's LDS holds (kRowLimitMost below)
constexpr int32_t kNumLimit[kBins - 2] = {32, 64, 128, 256, 512, 1024, 2048, 4096};
// lanes per row and table sizes per bin.  The kernels wait on memory (A's row, the bounds of its B
// rows, the B rows: a chain of round trips per row) and LDS decides how many rows a CU has in
// flight, so rows get the smallest table that holds them at half load.
// (Bins 0 to 2; longer rows get a workgroup each, see SetShape and RowShape.)
constexpr int kGroup0 = 8, kGroup1 = 16, kGroup2 = 16;
constexpr int kSymTable0 = 128, kSymTable1 = 256, kSymTable2 = 512;
constexpr int kNumTable0 = 64, kNumTable1 = 128, kNumTable2 = 256;

constexpr int kMergeCap = 8;                  // longest A row and B row of the merge path
constexpr int32_t kColEnd = 0x7fffffff;       // past-the-end column of a staged B row
constexpr int32_t kMergedKey = -1;            // binning key of a row the merge path has taken

struct Work {
    int32_t *key;      // [rows] binning key of the symbolic phase (product bound)
    int32_t *perm;     // [rows] rows grouped by bin
    int32_t *bins;     // [kBinInts]: rows per bin [0, kBins), first row of bin b at kBinStart + b (end at + b + 1), cursor at kBinCursor + b
    int32_t *count;    // [rows + 1] entries per row of C: the row pointer is made of them, the numeric phase bins by them
    int64_t *scan;     // [tiles + 1] sums of the counts by tile of the row pointer's scan
    int32_t *mark;     // [spill_groups(B_cols) * B_cols]
    double *acc;       // [spill_groups(B_cols) * B_cols]
    int64_t *summary;  // [2]: nnz(C) and the number of rows on the hash path, for the host
};

inline size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

size_t work_layout(int64_t rows, int64_t B_cols, void *base, Work *w) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void *p = base ? static_cast<char *>(base) + off : nullptr;
        off += align_up(bytes);
        return p;
    };
    int32_t *key = (int32_t *)take((rows + 1) * 4);
    int32_t *perm = (int32_t *)take((rows + 1) * 4);
    int32_t *bins = (int32_t *)take(kBinInts * 4);
    int32_t *count = (int32_t *)take((size_t)(rows + 1) * 4);
    int64_t *scan = (int64_t *)take(nm::scan_scratch_bytes(rows + 1));
    int64_t *summary = (int64_t *)take(2 * 8);
    int32_t *mark = (int32_t *)take((size_t)spill_groups(B_cols) * (B_cols + 1) * 4);
    double *acc = (double *)take((size_t)spill_groups(B_cols) * (B_cols + 1) * 8);
    if (w) *w = Work{key, perm, bins, count, scan, mark, acc, summary};
    return off;
}

// First slot of a key in a table of TABLE slots (a power of two): the HIGH bits of a
// multiplicative hash.  The low bits of key * odd depend on the low bits of the key alone,
// so columns a multiple of the table size apart -- the neighbours of a grid point in the
// next row or plane -- would all start their probes in the same slot.
template <int TABLE> __device__ __forceinline__ uint32_t first_slot(int32_t key) {
    static_assert(TABLE >= 2 && (TABLE & (TABLE - 1)) == 0, "table size");
    return ((uint32_t)key * 0x9E3779B1u) >> (32 - __builtin_ctz(TABLE));
}

// Lanes of a wavefront see each other's LDS accesses from before this point.  The fences keep a lane's
// accesses in order; the wave barrier (no instruction) keeps the lanes together: without it the
// compiler may let the lanes that skip a branch run on past the fence before it stores what the
// others store inside the branch.
template <int G> __device__ __forceinline__ void group_sync() {
    static_assert(G <= kWave, "a group is part of a wavefront");
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- binning ---------------------------------------------------------------

// ---- merge path (short rows) ---------------------------------------------------
//
// Lane layout: a merge group is the 8 lanes of equal parity in a 16-lane DPP row,
// so a wavefront holds 8 groups.  Neighbours inside a group are two lanes apart:
// rotations by 2, 4 and 8 inside the DPP row reduce over the group, and a shift by
// 2 feeds lane k the value of lane k-1 of its group with a hardware zero for k = 0.

__device__ __forceinline__ int merge_lane() { return (threadIdx.x & 15) >> 1; }
__device__ __forceinline__ int merge_group() { return ((threadIdx.x & 63) >> 4) * 2 + (threadIdx.x & 1); }

__device__ __forceinline__ int32_t merge_min(int32_t v) {
    v = min(v, nm::dpp_move<0x122>(v));   // row_ror 2
    v = min(v, nm::dpp_move<0x124>(v));   // row_ror 4
    v = min(v, nm::dpp_move<0x128>(v));   // row_ror 8
    return v;
}
__device__ __forceinline__ int32_t merge_max(int32_t v) {
    v = max(v, nm::dpp_move<0x122>(v));
    v = max(v, nm::dpp_move<0x124>(v));
    v = max(v, nm::dpp_move<0x128>(v));
    return v;
}
__device__ __forceinline__ int32_t merge_sum(int32_t v) {
    v += nm::dpp_move<0x122>(v);
    v += nm::dpp_move<0x124>(v);
    v += nm::dpp_move<0x128>(v);
    return v;
}

constexpr int kMergeRows = kBlock / 8;   // rows of A per workgroup pass
constexpr int kMergeStride = kBlock + 1; // slot stride of the staged B rows (odd: slots of one lane fall in different banks)

// Staging of the B rows of a wavefront into LDS.  Every lane owns one B row
// (start `bb`, `len` <= kMergeCap entries, 0 when it has none).  Loading them
// lane by lane would touch ~30 cache lines per instruction and use 8 bytes of
// each; instead the wavefront loads one LEG at a time: in pass u the eight lanes
// of sub-wavefront g read the eight entries of the row owned by lane u of group
// g, so an instruction reads eight contiguous 64-byte pieces -- and for banded
// matrices, where neighbouring rows of A name neighbouring rows of B, one
// contiguous span.  Entry k of the row owned by thread t lands in slot
// [k * kMergeStride + t]; slot kMergeCap is the end marker.
//
// The loads are unconditional: a lane with nothing to fetch reads `safe` (8 valid
// bytes) and discards the result.  Predicated loads would sit in their own
// branches, each followed by the wait for its data, i.e. one memory round trip
// per leg instead of one for all of them.
template <typename T, bool VALUES>
__device__ __forceinline__ void merge_stage(int64_t bb, int len, const int64_t *__restrict__ B_indices,
                                            const T *__restrict__ B_data, const int64_t *__restrict__ safe,
                                            int64_t *s_bb, int32_t *s_len, int32_t *s_col, T *s_val) {
    s_bb[threadIdx.x] = bb;
    s_len[threadIdx.x] = len;
    s_col[kMergeCap * kMergeStride + threadIdx.x] = kColEnd;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int lane = threadIdx.x & 63, g = lane >> 3, k = lane & 7;
    const int first = (threadIdx.x & ~63) + (g >> 1) * 16 + (g & 1);   // lane 0 of merge group g
    int64_t col[kMergeCap];
    T val[kMergeCap];
    bool have[kMergeCap];
#pragma unroll
    for (int u = 0; u < kMergeCap; ++u) {
        const int owner = first + 2 * u;
        const int64_t obb = s_bb[owner];
        have[u] = k < s_len[owner];
        col[u] = *(have[u] ? B_indices + obb + k : safe);
        if (VALUES) val[u] = *(have[u] ? B_data + obb + k : reinterpret_cast<const T *>(safe));
    }
#pragma unroll
    for (int u = 0; u < kMergeCap; ++u) {
        const int owner = first + 2 * u;
        s_col[k * kMergeStride + owner] = have[u] ? (int32_t)col[u] : kColEnd;
        if (VALUES) s_val[k * kMergeStride + owner] = have[u] ? val[u] : T(0);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// First kernel of the symbolic phase, over all rows in their natural order.  Eight
// lanes per row gather the lengths of the B rows it names.  Rows that qualify for
// the merge path are counted here (key = kMergedKey); for the others key[i] is the
// product bound min(sum of B row lengths, 2^31 - 8) that the hash path bins on.
__global__ __launch_bounds__(kBlock) void symbolic_front_kernel(
    int64_t rows, int64_t nbatch_padded, const int64_t *__restrict__ A_indices,
    const int64_t *__restrict__ A_indptr, const int64_t *__restrict__ B_indices,
    const int64_t *__restrict__ B_indptr, int32_t *__restrict__ key, int32_t *__restrict__ C_count,
    unsigned long long *__restrict__ hash_rows, unsigned long long token, uint64_t *__restrict__ dest,
    int32_t *__restrict__ bstart) {
    __shared__ int32_t s_col[(kMergeCap + 1) * kMergeStride];
    __shared__ int64_t s_bb[kBlock];
    __shared__ int32_t s_len[kBlock];
    const int gl = merge_lane();
    if (blockIdx.x == 0 && threadIdx.x == 0) C_count[rows] = 0;   // the scan's last entry: nnz(C)
    const int64_t batch = nm::xcd_tile(blockIdx.x, nbatch_padded);
    const int64_t row = batch * kMergeRows + (threadIdx.x >> 6) * 8 + merge_group();
    const bool live = row < rows;
    const int64_t ab = live ? A_indptr[row] : 0, ae = live ? A_indptr[row + 1] : 0;
    int64_t ub = 0, my_bb = 0;
    int32_t mx = 0, my_len = 0;
    for (int64_t a = ab + gl; a < ae; a += 8) {
        const int64_t j = A_indices[a];
        const int64_t bb = B_indptr[j], len = B_indptr[j + 1] - bb;
        ub += len;
        const int32_t l32 = (int32_t)(len > kMergeCap + 1 ? kMergeCap + 1 : len);
        mx = max(mx, l32);
        if (a - ab < 8) {
            my_bb = bb;
            my_len = l32;
        }
    }
    const int32_t ubc = merge_sum((int32_t)(ub > 0x0fffffff ? 0x0fffffff : ub));
    const bool merge = live && (ae - ab) <= kMergeCap && merge_max(mx) <= kMergeCap;
    if (live && !merge && gl == 0) key[row] = ubc;
    // A row left to the hash path raises a flag (a plain store of the same value by whoever finds one:
    // a counter that every wavefront of a product of long rows adds to would be a quarter of a
    // million atomics on one address); the exact count comes from the binning, if it runs.  The flag
    // is raised by writing the call's token, so that nobody need lower it first: whatever the word
    // held before is not this call's token, or at worst makes the hash path run over no rows.
    if (live && !merge && gl == 0) *hash_rows = token;
    merge_stage<float, false>(my_bb, merge ? my_len : 0, B_indices, nullptr, A_indptr, s_bb, s_len, s_col, nullptr);
    int32_t *pc = s_col + threadIdx.x;
    int32_t cur = *pc;
    int it = 0, last = -1;
    // The merge also leaves behind WHERE every product goes: the pass in which the k-th entry of a
    // lane's B row is taken is the position of that entry's column in the row of C.  A column that
    // has been taken is not needed again, so the pass is written over it in LDS -- one store, where
    // shifting it into a 64-bit word cost five vector instructions in a loop that is bound by what
    // it issues -- and the words the numeric phase adds the products up on (byte k = the pass of
    // entry k, 0xFF: no such entry; also what a product plan is made of) are put together after the
    // loop: the low byte of a place never taken is the past-the-end column's, 0xFF.
    static_assert((kColEnd & 0xFF) == 0xFF, "an entry never taken reads as no entry");
    for (;;) {
        const int32_t m = merge_min(cur);
        const bool open = m != kColEnd;
        if (__ballot(open) == 0) break;
        if (cur == m && open) {
            last = it;
            *pc = it;
            pc += kMergeStride;
            cur = *pc;
        }
        ++it;
    }
    const int cnt = merge_max(last) + 1;   // an open group emits one column per pass
    if (merge && gl == 0) {
        C_count[row] = cnt;
        key[row] = kMergedKey;
    }
    if (dest && merge && ab + gl < ae) {   // (read once, by another kernel: nontemporal)
        const int32_t *mine = s_col + threadIdx.x;
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo |= ((uint32_t)mine[j * kMergeStride] & 0xFFu) << (8 * j);
            hi |= ((uint32_t)mine[(4 + j) * kMergeStride] & 0xFFu) << (8 * j);
        }
        const uint64_t where = ((uint64_t)hi << 32) | lo;
        __builtin_nontemporal_store(where, dest + ab + gl);
        __builtin_nontemporal_store((int32_t)my_bb, bstart + ab + gl);
    }
}

// Numeric counterpart: rows marked kMergedKey are produced here, in natural order.
// The B rows are staged in LDS (columns and values); each pass emits the smallest head column and the sum of the
// matching products, accumulated from +0.0 in lane order, which is the order in
// which the serial loop adds them (cpp/sparse_csr_cpu.cpp:193-200).
template <typename T>
__global__ __launch_bounds__(kBlock) void numeric_front_kernel(
    int64_t rows, int64_t nbatch_padded, const int32_t *__restrict__ key, const T *__restrict__ A_data,
    const int64_t *__restrict__ A_indices, const int64_t *__restrict__ A_indptr, const T *__restrict__ B_data,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr,
    const int64_t *__restrict__ C_indptr, int64_t *__restrict__ C_indices, T *__restrict__ C_data) {
    __shared__ int32_t s_col[(kMergeCap + 1) * kMergeStride];
    __shared__ T s_val[kMergeCap * kMergeStride];
    __shared__ int64_t s_bb[kBlock];
    __shared__ int32_t s_len[kBlock];
    const int gl = merge_lane();
    const int64_t batch = nm::xcd_tile(blockIdx.x, nbatch_padded);
    const int64_t row = batch * kMergeRows + (threadIdx.x >> 6) * 8 + merge_group();
    // the row's bounds are requested together with its key: one memory round trip instead of two
    const bool live = row < rows;
    const int32_t my_key = live ? key[row] : 0;
    const int64_t ab0 = live ? A_indptr[row] : 0, ae0 = live ? A_indptr[row + 1] : 0;
    const int64_t out0 = live ? C_indptr[row] : 0;
    const bool merge = live && my_key == kMergedKey;
    if (__ballot(merge) == 0) return;   // wavefront-uniform; no workgroup barrier below
    const int64_t ab = merge ? ab0 : 0, ae = merge ? ae0 : 0;
    const bool mine = ab + gl < ae;
    const T av_raw = *(mine ? A_data + ab + gl : reinterpret_cast<const T *>(A_indptr));
    const int64_t j = mine ? *(A_indices + ab + gl) : 0;
    const T av = mine ? av_raw : T(0);
    const int64_t *bp = mine ? B_indptr + j : A_indptr;   // A_indptr: any two readable entries
    const int64_t bb = bp[0];
    const int my_len = mine ? (int)(bp[1] - bb) : 0;
    merge_stage<T, true>(bb, my_len, B_indices, B_data, A_indptr, s_bb, s_len, s_col, s_val);
    // lanes that take part in the ordered sum: the longest row of A in this wavefront
    int steps = 1;
#pragma unroll
    for (int q = kMergeCap; q > 1; --q)
        if (steps == 1 && __ballot((ae - ab) >= q) != 0) steps = q;
    // Emitted entries pass through a ring of 8 per group so that the group writes
    // them 8 at a time (one 64-byte piece per array) instead of lane by lane.
    // The ring reuses the exchange arrays of merge_stage, which are dead by now FOR THIS
    // WAVEFRONT: its ring entries and its exchange entries must be the same 64 slots, because
    // another wavefront of the workgroup may still be reading its own exchange entries (there
    // is no workgroup barrier).  A value therefore takes a whole 8-byte slot of s_bb whatever
    // T is (packed floats would put the ring of wavefront w over the exchange entries of
    // wavefront w / 2, which then read a wrong row start).
    static_assert(sizeof(T) <= sizeof(s_bb[0]), "a ring value must fit one exchange slot of s_bb");
    static_assert(sizeof(s_bb) / sizeof(s_bb[0]) == kBlock && sizeof(s_len) / sizeof(s_len[0]) == kBlock,
                  "one exchange slot per lane: wavefront w owns slots [64 w, 64 w + 64)");
    static_assert(8 /* groups per wavefront */ * 8 /* ring entries per group */ == nm::kWave,
                  "the ring of a wavefront must cover exactly that wavefront's own exchange slots");
    int32_t *s_oc = s_len;
    auto s_ov = [&](int slot) -> T & { return *reinterpret_cast<T *>(s_bb + slot); };
    const int ring = ((threadIdx.x >> 6) * 8 + merge_group()) * 8;
    int emitted = 0;   // entries of this row produced so far
    auto flush = [&](int base) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int e = base + gl;
        if (e < emitted) {
            C_indices[out0 + e] = (int64_t)s_oc[ring + gl];
            C_data[out0 + e] = s_ov(ring + gl);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    };
    const int32_t *pc = s_col + threadIdx.x;   // this lane's head column / value slots
    const T *pv = s_val + threadIdx.x;
    int32_t cur = *pc;
    T curv = av * *pv;
    int it = 0;
    for (;;) {
        const int32_t m = merge_min(cur);
        const bool open = m != kColEnd;
        if (__ballot(open) == 0) break;
        const bool hit = cur == m && open;
        const T x = hit ? curv : T(0);
        T t;
        if (__ballot(merge_sum(hit ? 1 : 0) > 2) == 0) {
            // at most two products per entry anywhere in the wavefront: a sum of two
            // terms (and exact zeros) does not depend on the order of the additions
            t = x + nm::dpp_move_zero<0x122>(x);
            t += nm::dpp_move_zero<0x124>(t);
            t += nm::dpp_move_zero<0x128>(t);
        } else {
            t = T(0);
#pragma unroll
            for (int q = 0; q < kMergeCap; ++q) {
                if (q >= steps) break;
                t = x + nm::dpp_move_zero<0x112>(t);   // row_shr 2: previous lane of the group, 0 for the first
            }
        }
        // every group that is still open has emitted exactly `it` entries so far
        if (gl == steps - 1 && open) {
            s_oc[ring + (it & 7)] = m;
            s_ov(ring + (it & 7)) = t;
        }
        ++it;
        if (open) emitted = it;
        if ((it & 7) == 0) flush(it - 8);
        if (hit) {
            pc += kMergeStride;
            pv += kMergeStride;
            cur = *pc;
            curv = av * (cur != kColEnd ? *pv : T(0));   // no value slot behind the end marker
        }
    }
    if (it & 7) flush(it & ~7);
}

// What the rows are binned by: their key (the symbolic phase), or the length of their row of C, which the
// symbolic phase has left in `count` (the numeric phase).  Negative keys (rows taken by the merge
// path) belong to no bin.
struct RowKeys {
    const int32_t *key, *count;   // count: null where the key itself is meant
    __device__ __forceinline__ int32_t operator[](int64_t i) const {
        const int32_t k = key[i], n = count ? count[i] : k;
        return k < 0 ? k : n;
    }
};
struct BinLimits { int32_t l[kBins - 1]; };
__device__ __forceinline__ int bin_of(int32_t k, const BinLimits &lim) {
    if (k < 0) return -1;
    int b = 0;
#pragma unroll
    for (int q = 0; q < kBins - 1; ++q) b += k > lim.l[q];
    return b;
}

__global__ void bin_clear_kernel(int32_t *bins) {
    if (threadIdx.x < kBinInts) bins[threadIdx.x] = 0;
}

// Rows per bin.  Each wavefront counts with ballots (one population count per
// bin) instead of 64 colliding LDS atomics.
__global__ __launch_bounds__(kBlock) void bin_count_kernel(int64_t rows, RowKeys key,
                                                           BinLimits lim, int32_t *bins) {
    __shared__ int s_cnt[kBins];
    if (threadIdx.x < kBins) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    int mine[kBins] = {};
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i0 = (int64_t)blockIdx.x * blockDim.x; i0 < rows; i0 += stride) {
        const int64_t i = i0 + threadIdx.x;
        const int b = i < rows ? bin_of(key[i], lim) : -1;
#pragma unroll
        for (int q = 0; q < kBins; ++q) mine[q] += __popcll(__ballot(b == q));
    }
    if (lane == 0)
        for (int q = 0; q < kBins; ++q)
            if (mine[q]) atomicAdd(&s_cnt[q], mine[q]);
    __syncthreads();
    if (threadIdx.x < kBins && s_cnt[threadIdx.x]) atomicAdd(bins + threadIdx.x, s_cnt[threadIdx.x]);
}

__global__ void bin_offsets_kernel(int32_t *bins) {
    if (threadIdx.x == 0) {
        int32_t run = 0;
        for (int b = 0; b < kBins; ++b) {
            bins[kBinStart + b] = run;
            bins[kBinCursor + b] = run;
            run += bins[b];
        }
        bins[kBinStart + kBins] = run;
    }
}

// Rows are placed a workgroup at a time, wavefront by wavefront and lane by lane, so that each
// bin keeps them in ascending order inside a workgroup's slice (neighbouring rows share B rows
// and C lines).  A workgroup takes ONE contiguous slice of the rows, counts it, claims its room
// in every bin with one atomic per bin, and then places the rows: thousands of workgroups claiming
// room 256 rows at a time queued up on the eight cursors (96 us for 2.1 M rows).
__global__ __launch_bounds__(kBlock) void bin_scatter_kernel(int64_t rows, RowKeys key,
                                                             BinLimits lim, int32_t *bins,
                                                             int32_t *__restrict__ perm) {
    constexpr int kWaves = kBlock / kWave;
    __shared__ int s_wave[kWaves][kBins];   // rows of bin q in wavefront w (of the slice, then of a step)
    __shared__ int s_base[kBins];           // where the workgroup's next rows of bin q go
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t per = ((rows + gridDim.x - 1) / gridDim.x + kBlock - 1) / kBlock * kBlock;   // whole steps
    const int64_t r0 = (int64_t)blockIdx.x * per, r1 = r0 + per < rows ? r0 + per : rows;
    if (r0 >= rows) return;
    // (where the rows of a wavefront are all of one bin, as a stencil's are, one ballot does for ten: 1 M rows
    // 21 -> 17 us)
    {   // count the slice
        int mine[kBins] = {};
        if (lane == 0)
            for (int q = 0; q < kBins; ++q) s_wave[wave][q] = 0;
        for (int64_t i0 = r0; i0 < r1; i0 += kBlock) {
            const int64_t i = i0 + threadIdx.x;
            const int b = i < r1 ? bin_of(key[i], lim) : -1;
            const int b0 = __builtin_amdgcn_readfirstlane(b);
            if (__ballot(b == b0) == ~0ull) {
                if (lane == 0 && b0 >= 0) s_wave[wave][b0] += kWave;
                continue;
            }
#pragma unroll
            for (int q = 0; q < kBins; ++q) mine[q] += __popcll(__ballot(b == q));
        }
        if (lane == 0)
            for (int q = 0; q < kBins; ++q) s_wave[wave][q] += mine[q];
        __syncthreads();
        if (threadIdx.x < kBins) {
            int total = 0;
            for (int w = 0; w < kWaves; ++w) total += s_wave[w][threadIdx.x];
            s_base[threadIdx.x] = total ? atomicAdd(bins + kBinCursor + threadIdx.x, total) : 0;
        }
        __syncthreads();
    }
    for (int64_t i0 = r0; i0 < r1; i0 += kBlock) {
        const int64_t i = i0 + threadIdx.x;
        const int b = i < r1 ? bin_of(key[i], lim) : -1;
        int before = 0;   // rows of my bin in lower lanes of my wavefront
        const int b0 = __builtin_amdgcn_readfirstlane(b);
        if (__ballot(b == b0) == ~0ull) {
            before = lane;
            if (lane < kBins) s_wave[wave][lane] = lane == b0 ? kWave : 0;
        } else {
#pragma unroll
            for (int q = 0; q < kBins; ++q) {
                const unsigned long long m = __ballot(b == q);
                if (b == q) before = __popcll(m & ((1ull << lane) - 1ull));
                if (lane == 0) s_wave[wave][q] = __popcll(m);
            }
        }
        __syncthreads();
        if (b >= 0) {
            int off = s_base[b] + before;
            for (int w = 0; w < wave; ++w) off += s_wave[w][b];
            perm[off] = (int32_t)i;
        }
        __syncthreads();
        if (threadIdx.x < kBins) {   // this step's rows are placed: the next step's go behind them
            int total = 0;
            for (int w = 0; w < kWaves; ++w) total += s_wave[w][threadIdx.x];
            s_base[threadIdx.x] += total;
        }
        __syncthreads();
    }
}

// Sums of the rows' counts by tile of kScanTile rows: the first pass of the row pointer's scan.
typedef int32_t I32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bool count_tile_whole(const int32_t *a, int64_t n) {
    static_assert(nm::kScanItems % 4 == 0, "counts are loaded four at a time");
    return ((int64_t)blockIdx.x + 1) * nm::kScanTile <= n && (reinterpret_cast<uintptr_t>(a) & 15) == 0;
}
__global__ __launch_bounds__(nm::kScanBlock) void count_tile_sums_kernel(const int32_t *__restrict__ count, int64_t n,
                                                                       int64_t *__restrict__ sums) {
    __shared__ int64_t s_wave[nm::kScanBlock / kWave];
    const int64_t base = (int64_t)blockIdx.x * nm::kScanTile + (int64_t)threadIdx.x * nm::kScanItems;
    int64_t v = 0;
    if (count_tile_whole(count, n)) {
        const I32x4 *p = reinterpret_cast<const I32x4 *>(count + base);
#pragma unroll
        for (int i = 0; i < nm::kScanItems / 4; ++i) {
            const I32x4 w = p[i];
            v += (int64_t)w[0] + w[1] + w[2] + w[3];
        }
    } else {
#pragma unroll
        for (int i = 0; i < nm::kScanItems; ++i)
            if (base + i < n) v += count[base + i];
    }
    int64_t total;
    nm::block_exclusive_scan(v, s_wave, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Row pointer of C from the rows' counts, and what the host needs between the phases: nnz(C) and
// the rows the hash path took.  count[0, n) with count[n - 1] == 0 -> C_indptr[0, n) (its exclusive
// scan, not in place: the counts of the merge path's rows survive a pass made before the hash
// path's rows are counted).  `sums` holds the sum of every tile of kScanTile counts; with
// `scanned` == 0 a workgroup adds up the sums before its own (a few thousand numbers out of L2
// against one more launch), otherwise they have been scanned already (their total behind them).
// The first workgroup, with nothing before it, adds up all tiles instead: nnz(C), which it leaves
// in summary[0], with the number of hash-path rows in summary[1] (from `bins`; where bins is null,
// 1 if the first kernel has left `token` there).  With `host_pinned` it also drops both into the
// host's landing place, followed by the ticket the host polls for: the host needs the numbers,
// not the row pointer, so it is told first and sizes C while the row pointer is being written.
constexpr int kInlineTiles = 4096;
__global__ __launch_bounds__(nm::kScanBlock) void row_pointer_kernel(
    const int32_t *__restrict__ count, int64_t n, const int64_t *__restrict__ sums, int scanned,
    int64_t *__restrict__ C_indptr, const int32_t *__restrict__ bins, int64_t *__restrict__ summary,
    int64_t token, volatile int64_t *host_pinned, int64_t ticket) {
    using nm::kScanItems;
    __shared__ int64_t s_wave[nm::kScanBlock / kWave];
    const int64_t base = (int64_t)blockIdx.x * nm::kScanTile + (int64_t)threadIdx.x * kScanItems;
    int32_t item[kScanItems];
    int64_t v = 0;
    const bool whole = count_tile_whole(count, n) && (reinterpret_cast<uintptr_t>(C_indptr) & 15) == 0;
    if (whole) {
        const I32x4 *p = reinterpret_cast<const I32x4 *>(count + base);
#pragma unroll
        for (int i = 0; i < kScanItems / 4; ++i) {
            const I32x4 w = p[i];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                item[4 * i + u] = w[u];
                v += w[u];
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < kScanItems; ++i) {
            item[i] = base + i < n ? count[base + i] : 0;
            v += item[i];
        }
    }
    // (the first workgroup, which has nothing before it, adds up all tiles instead: nnz(C), for the host)
    int64_t before;
    if (scanned) {
        before = sums[blockIdx.x == 0 ? gridDim.x : blockIdx.x];
    } else {
        const int upto = blockIdx.x == 0 ? (int)gridDim.x : (int)blockIdx.x;
        int64_t part = 0;
        for (int t = threadIdx.x; t < upto; t += nm::kScanBlock) part += sums[t];
        nm::block_exclusive_scan(part, s_wave, before);
    }
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) {
            const int64_t nnz = before;
            const int64_t hashed = bins ? (int64_t)bins[kBinStart + kBins] : (summary[1] == token ? 1 : 0);
            summary[0] = nnz;
            summary[1] = hashed;
            if (host_pinned) {
                host_pinned[0] = nnz;
                host_pinned[1] = hashed;
                __threadfence_system();
                host_pinned[2] = ticket;
            }
        }
        before = 0;
    }
    int64_t total;
    int64_t run = before + nm::block_exclusive_scan(v, s_wave, total);
    if (whole) {
        nm::I64x2 *p = reinterpret_cast<nm::I64x2 *>(C_indptr + base);
#pragma unroll
        for (int i = 0; i < kScanItems / 2; ++i) {
            nm::I64x2 w;
            w[0] = run;
            w[1] = run + item[2 * i];
            run = w[1] + item[2 * i + 1];
            p[i] = w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < kScanItems; ++i) {
            if (base + i < n) C_indptr[base + i] = run;
            run += item[i];
        }
    }
}

// host_pinned[0..1] = summary, then host_pinned[2] = ticket: the host polls the ticket.
__global__ void summary_out_kernel(const int64_t *__restrict__ summary, volatile int64_t *host_pinned,
                                   int64_t ticket) {
    if (threadIdx.x == 0) {
        host_pinned[0] = summary[0];
        host_pinned[1] = summary[1];
        __threadfence_system();
        host_pinned[2] = ticket;
    }
}

// The four binning steps by one workgroup, for so few rows that the launches cost more than the
// work: count, offsets, then rows placed in ascending order inside each bin (ballots, as in the
// grid-wide kernels).
constexpr int kBinSmallRows = 4096;
__global__ __launch_bounds__(1024) void bin_small_kernel(int64_t rows, RowKeys key,
                                                         BinLimits lim, int32_t *bins,
                                                         int32_t *__restrict__ perm) {
    constexpr int kWaves = 1024 / kWave;
    __shared__ int s_cnt[kWaves][kBins];
    __shared__ int s_start[kBins + 1], s_run[kBins];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // rows per bin
    int mine[kBins] = {};
    for (int64_t i0 = 0; i0 < rows; i0 += 1024) {
        const int64_t i = i0 + threadIdx.x;
        const int b = i < rows ? bin_of(key[i], lim) : -1;
#pragma unroll
        for (int q = 0; q < kBins; ++q) mine[q] += __popcll(__ballot(b == q));
    }
    if (lane == 0)
        for (int q = 0; q < kBins; ++q) s_cnt[wave][q] = mine[q];
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int q = 0; q < kBins; ++q) {
            s_start[q] = run;
            s_run[q] = run;
            for (int w = 0; w < kWaves; ++w) run += s_cnt[w][q];
        }
        s_start[kBins] = run;
    }
    __syncthreads();
    // rows placed chunk by chunk, wavefront by wavefront, lane by lane: ascending inside each bin
    for (int64_t i0 = 0; i0 < rows; i0 += 1024) {
        const int64_t i = i0 + threadIdx.x;
        const int b = i < rows ? bin_of(key[i], lim) : -1;
        int before = 0;
#pragma unroll
        for (int q = 0; q < kBins; ++q) {
            const unsigned long long m = __ballot(b == q);
            if (b == q) before = __popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) s_cnt[wave][q] = __popcll(m);
        }
        __syncthreads();
        if (b >= 0) {
            int off = s_run[b] + before;
            for (int w = 0; w < wave; ++w) off += s_cnt[w][b];
            perm[off] = (int32_t)i;
        }
        __syncthreads();
        if (threadIdx.x < kBins) {
            int t = 0;
            for (int w = 0; w < kWaves; ++w) t += s_cnt[w][threadIdx.x];
            s_run[threadIdx.x] += t;
        }
        __syncthreads();
    }
    if (threadIdx.x <= kBins) bins[kBinStart + threadIdx.x] = s_start[threadIdx.x];
    if (threadIdx.x < kBins) bins[threadIdx.x] = s_start[threadIdx.x + 1] - s_start[threadIdx.x];
}

int bin_rows(int64_t rows, RowKeys key, const int32_t limit[kBins - 1], const Work &w, hipStream_t s) {
    BinLimits lim;
    for (int q = 0; q < kBins - 1; ++q) lim.l[q] = limit[q];
    if (rows <= kBinSmallRows) {
        hipLaunchKernelGGL(bin_small_kernel, dim3(1), dim3(1024), 0, s, rows, key, lim, w.bins, w.perm);
        NM_LAUNCH_CHECK("bin_small_kernel");
        return NM_OK;
    }
    // (few enough workgroups that their atomics on the eight counters and cursors do not queue up)
    int64_t grid = nm::ceil_div(rows, kBlock);
    if (grid > 512) grid = 512;
    if (grid < 1) grid = 1;
    hipLaunchKernelGGL(bin_clear_kernel, dim3(1), dim3(64), 0, s, w.bins);
    hipLaunchKernelGGL(bin_count_kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, rows, key, lim, w.bins);
    hipLaunchKernelGGL(bin_offsets_kernel, dim3(1), dim3(64), 0, s, w.bins);
    hipLaunchKernelGGL(bin_scatter_kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, rows, key, lim, w.bins,
                       w.perm);
    NM_LAUNCH_CHECK("bin kernels");
    return NM_OK;
}

// ---- symbolic ----------------------------------------------------------------

template <int G, int TABLE>
__global__ __launch_bounds__(kBlock) void symbolic_hash_kernel(
    int bin, const int32_t *__restrict__ bins, const int32_t *__restrict__ perm,
    const int64_t *__restrict__ A_indices, const int64_t *__restrict__ A_indptr,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr,
    int32_t *__restrict__ C_count) {
    constexpr int GPB = kBlock / G;
    // the tables of the groups that share a wavefront start kTablePad entries apart in
    // bank space; without the pad they would all map slot t to the same LDS bank
    constexpr int STRIDE = TABLE + (GPB > 1 ? kTablePad : 0);
    __shared__ __align__(16) int32_t s_keys[GPB * STRIDE];
    const int gl = threadIdx.x % G, gi = threadIdx.x / G;
    int32_t *tab = s_keys + gi * STRIDE;
    const int32_t b0 = bins[kBinStart + bin], b1 = bins[kBinStart + bin + 1];
    for (int32_t idx0 = b0 + blockIdx.x * GPB; idx0 < b1; idx0 += gridDim.x * GPB) {
        const int32_t idx = idx0 + gi;
        const bool live = idx < b1;
        for (int t = gl; t < TABLE; t += G) tab[t] = kEmpty;
        group_sync<G>();
        int cnt = 0;
        int64_t row = 0;
        auto insert = [&](int32_t key) {
            uint32_t h = first_slot<TABLE>(key);
            int32_t old = atomicCAS(&tab[h], kEmpty, key);
            while (old != kEmpty && old != key) {   // one exit test: the common case probes once
                h = (h + 1) & (TABLE - 1);
                old = atomicCAS(&tab[h], kEmpty, key);
            }
            cnt += old == kEmpty;
        };
        {
            // Latency-lean walk: each lane fetches one entry of A's row together with the
            // bounds of the B row it names; the first G columns of up to kAhead B rows are
            // then requested back to back before any of them is inserted.
            // A group of 16 lanes takes TWO rows of B per step, eight lanes each: the rows these bins
            // see are mostly shorter than eight entries (stencil powers), and insertion into a set
            // has no order to keep, so the second half of the group need not idle.
            constexpr int W = G == 16 ? 8 : G, NSUB = G / W;
            const int hl = gl & (W - 1), half = gl / W;
            const int gbase = (threadIdx.x & (kWave - 1)) & ~(G - 1);
            row = live ? perm[idx] : 0;
            const int64_t ab = live ? A_indptr[row] : 0, ae = live ? A_indptr[row + 1] : 0;
            for (int64_t a0 = ab; a0 < ae; a0 += G) {
                const int64_t my_ai = a0 + gl;
                const bool mine = my_ai < ae;
                const int64_t my_j = mine ? A_indices[my_ai] : 0;
                const int64_t my_bb = mine ? B_indptr[my_j] : 0, my_be = mine ? B_indptr[my_j + 1] : 0;
                const int nb = (int)(ae - a0 < G ? ae - a0 : G);
                if constexpr (G == 16) {
                    // the group is one DPP row: entries 2 u and 2 u + 1 of A's row reach the two halves
                    // by row broadcasts instead of shuffles through the LDS crossbar, and the bounds of a
                    // row of B longer than eight entries are fetched again where its rest is walked
                    static_assert(kAhead * NSUB == G && W == 8, "one batch of pairs covers the group");
                    const int my_len = (int)(my_be - my_bb);
                    int32_t qk[kAhead];
                    nm::static_for<kAhead>([&](auto uc) {
                        constexpr int U = decltype(uc)::value;
                        // (broadcasts first, with all sixteen lanes active; then the lane's own tests)
                        const int64_t kk = nm::row_lane_halves<2 * U, 2 * U + 1>(my_bb) + hl;
                        const int len = nm::row_lane_halves<2 * U, 2 * U + 1>(my_len);
                        const bool ok = (2 * U + half < nb) & (hl < len);
                        qk[U] = ok ? (int32_t)B_indices[kk] : kEmpty;
                    });
                    nm::static_for<kAhead>([&](auto uc) {
                        constexpr int U = decltype(uc)::value;
                        if (2 * U >= nb) return;
                        if (qk[U] != kEmpty) insert(qk[U]);
                        // (the test is the same in all sixteen lanes, so that the broadcasts behind it
                        // find their source lanes active)
                        const int len_lo = nm::row_lane<2 * U>(my_len), len_hi = nm::row_lane<2 * U + 1>(my_len);
                        if ((len_lo > W) | (len_hi > W)) {   // (lanes past the row's end hold a length of 0)
                            const int64_t bb = nm::row_lane_halves<2 * U, 2 * U + 1>(my_bb);
                            const int64_t be_row = nm::row_lane_halves<2 * U, 2 * U + 1>(my_be);
                            const int64_t be = 2 * U + half < nb ? be_row : bb;
                            for (int64_t kk = bb + W + hl; kk < be; kk += W) insert((int32_t)B_indices[kk]);
                        }
                    });
                } else
                for (int e0 = 0; e0 < nb; e0 += kAhead * NSUB) {
                    int32_t pk[kAhead];
                    int64_t bbs[kAhead], bes[kAhead];
                    bool has[kAhead];
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) {
                        const int e = e0 + u * NSUB + half;
                        has[u] = e < nb;
                        const int src = gbase + (has[u] ? e : e0);
                        bbs[u] = __shfl(my_bb, src, kWave);
                        bes[u] = __shfl(my_be, src, kWave);
                        const int64_t kk = bbs[u] + hl;
                        pk[u] = (has[u] && kk < bes[u]) ? (int32_t)B_indices[kk] : kEmpty;
                    }
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) {
                        if (e0 + u * NSUB >= nb) break;
                        if (pk[u] != kEmpty) insert(pk[u]);
                        if (has[u])
                            for (int64_t kk = bbs[u] + W + hl; kk < bes[u]; kk += W) insert((int32_t)B_indices[kk]);
                    }
                }
            }
        }
        cnt = nm::group_sum<G>(cnt);
        if (live && gl == 0) C_count[row] = cnt;
        group_sync<G>();
    }
}

// Exclusive sum over the workgroup's threads; `total` gets the sum.  s_wave: one word per wavefront.
template <int TPB, typename V> __device__ __forceinline__ V row_scan(V v, V *s_wave, V &total) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    V incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const V up = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += up;
    }
    if constexpr (TPB == kWave) {
        total = __shfl(incl, kWave - 1, kWave);
        return incl - v;
    } else {
        __syncthreads();   // (the words may still be read from the last use)
        if (lane == kWave - 1) s_wave[wave] = incl;
        __syncthreads();
        V before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < TPB / kWave; ++w) {
            const V t = s_wave[w];
            if (w < wave) before += t;
            all += t;
        }
        total = all;
        return before + incl - v;
    }
}

// Spill path: distinct columns counted with a stamped dense marker per workgroup (of the first `groups`).
__device__ __forceinline__ void symbolic_spill(
    const int32_t *__restrict__ bins, const int32_t *__restrict__ perm, int64_t B_cols, int groups,
    const int64_t *__restrict__ A_indices, const int64_t *__restrict__ A_indptr,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr, int32_t *mark_all,
    int32_t *__restrict__ C_count) {
    __shared__ int s_red[kSpillBlock / kWave];
    const int32_t b0 = bins[kBinStart + kBins - 1], b1 = bins[kBinStart + kBins];
    if ((int)blockIdx.x >= groups || b0 + (int32_t)blockIdx.x >= b1) return;
    int32_t *mark = mark_all + (size_t)blockIdx.x * (B_cols + 1);
    for (int64_t c = threadIdx.x; c < B_cols; c += kSpillBlock) mark[c] = 0;
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    for (int32_t idx = b0 + blockIdx.x; idx < b1; idx += groups) {
        const int64_t row = perm[idx];
        const int32_t stamp = (int32_t)row + 1;
        int cnt = 0;
        const int64_t je = A_indptr[row + 1];
        for (int64_t jj = A_indptr[row] + wave; jj < je; jj += kSpillBlock / kWave) {
            const int64_t j = A_indices[jj];
            const int64_t ke = B_indptr[j + 1];
            for (int64_t kk = B_indptr[j] + lane; kk < ke; kk += kWave)
                if (atomicExch(mark + B_indices[kk], stamp) != stamp) ++cnt;
        }
        cnt = nm::wave_sum(cnt);
        if (lane == 0) s_red[wave] = cnt;
        __syncthreads();
        if (threadIdx.x == 0) {
            int t = 0;
            for (int w = 0; w < kSpillBlock / kWave; ++w) t += s_red[w];
            C_count[row] = t;
        }
        __syncthreads();
    }
}

// Rows of many products: one row per workgroup, its products numbered through and dealt to the
// threads by number (see numeric_row_kernel); a set has no order to keep, so there are no turns.
// Bound by the row's chain of round trips (A's row, the bounds of B's rows, their columns).  A
// 150 000-row power-law graph squared (mean 8, rows up to 1000, 10 M products), by product bound, against
// groups of 64 and 256 lanes that took B's rows one by one: 257-512 43 -> 22 us, 513-1024 70 -> 29,
// 1025-2048 51 -> 20, 2049-8192 106 -> 44, more (a marker per column in global memory) 94 -> 17.  Groups
// of 16 lanes with their tables side by side stay ahead below 256 products (46 us for 129-256).
// The launch for the longest rows takes those that spill as well.
template <int TPB_, int SLOTS_, bool SPILL_ = false> struct SetShape {
    static constexpr bool SPILL = SPILL_;
    static constexpr int TPB = TPB_, SLOTS = SLOTS_, BATCH = TPB < 512 ? TPB : 512, UNROLL = 4;
    static constexpr size_t at_row = 8 * (BATCH + 2), at_wave = at_row + 8 * BATCH, at_key = at_wave + 8 * (TPB / kWave) + 16;
    static constexpr size_t lds = at_key + 4 * SLOTS;
    static_assert(lds <= 160 * 1024, "a CU's LDS");
};
template <typename S>
__global__ __launch_bounds__(S::TPB) void symbolic_row_kernel(
    int bin, const int32_t *__restrict__ bins, const int32_t *__restrict__ perm,
    const int64_t *__restrict__ A_indices, const int64_t *__restrict__ A_indptr,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr, int32_t *__restrict__ C_count,
    int64_t B_cols, int32_t *mark, int spill_groups) {
    constexpr int TPB = S::TPB, SLOTS = S::SLOTS, BATCH = S::BATCH, U = S::UNROLL;
    extern __shared__ __align__(16) unsigned char s_raw[];
    int64_t *s_off = reinterpret_cast<int64_t *>(s_raw);               // number of an entry's first product
    int64_t *s_row = reinterpret_cast<int64_t *>(s_raw + S::at_row);   // start of its row of B, less that number
    int64_t *s_wave = reinterpret_cast<int64_t *>(s_raw + S::at_wave);
    int32_t *tab = reinterpret_cast<int32_t *>(s_raw + S::at_key);
    const int tid = threadIdx.x;
    const int32_t b0 = bins[kBinStart + bin], b1 = bins[kBinStart + bin + 1];
    for (int32_t idx = b0 + (int32_t)blockIdx.x; idx < b1; idx += (int32_t)gridDim.x) {
        const int64_t row = perm[idx];
        const int64_t ab = A_indptr[row], ae = A_indptr[row + 1];
        for (int t = tid; t < SLOTS; t += TPB) tab[t] = kEmpty;
        int cnt = 0;
        for (int64_t a0 = ab; a0 < ae; a0 += BATCH) {
            const bool mine = tid < BATCH && a0 + tid < ae;
            const int64_t j = mine ? A_indices[a0 + tid] : 0;
            const int64_t bb = mine ? B_indptr[j] : 0, be = mine ? B_indptr[j + 1] : 0;
            int64_t total;
            const int64_t off = row_scan<TPB, int64_t>(be - bb, s_wave, total);
            __syncthreads();   // the last batch's products are done with the lists
            if (tid < BATCH) {
                s_off[tid] = off;   // (threads past the row's end: the total)
                s_row[tid] = bb - off;
            }
            __syncthreads();
            for (int64_t p0 = 0; p0 < total; p0 += TPB * U) {
                int32_t key[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t p = p0 + u * TPB + tid;
                    const bool have = p < total;
                    const int64_t at = have ? p : 0;
                    int e = 0;   // the last entry whose first product is not behind this one
#pragma unroll
                    for (int step = BATCH / 2; step > 0; step >>= 1)
                        if (s_off[e + step] <= at) e += step;
                    key[u] = (int32_t)B_indices[s_row[e] + at];
                    if (!have) key[u] = kEmpty;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (key[u] == kEmpty) continue;
                    uint32_t h = __umulhi((uint32_t)key[u] * 0x9E3779B1u, (uint32_t)SLOTS);
                    int32_t old = atomicCAS(&tab[h], kEmpty, key[u]);
                    while (old != kEmpty && old != key[u]) {
                        h = h + 1 == SLOTS ? 0 : h + 1;
                        old = atomicCAS(&tab[h], kEmpty, key[u]);
                    }
                    cnt += old == kEmpty;
                }
            }
        }
        int all;
        row_scan<TPB, int>(cnt, reinterpret_cast<int *>(s_wave), all);
        if (tid == 0) C_count[row] = all;
        __syncthreads();
    }
    if constexpr (S::SPILL) {
        static_assert(TPB == kSpillBlock && S::lds + 256 <= 160 * 1024, "the spill path's workgroup and LDS");
        symbolic_spill(bins, perm, B_cols, spill_groups, A_indices, A_indptr, B_indices, B_indptr, mark, C_count);
    }
}
using SetShape3 = SetShape<64, 768>;      // up to 512 products
using SetShape4 = SetShape<64, 1536>;     // up to 1024
using SetShape5 = SetShape<256, 3072>;    // up to 2048
using SetShape6 = SetShape<512, 10240>;   // up to 8192
using SetShape7 = SetShape<1024, 32768, true>;   // up to 24576, and the rest

// ---- numeric -------------------------------------------------------------------

template <typename T, int G, int TABLE>
__global__ __launch_bounds__(kBlock) void numeric_hash_kernel(
    int bin, const int32_t *__restrict__ bins, const int32_t *__restrict__ perm,
    const T *__restrict__ A_data, const int64_t *__restrict__ A_indices,
    const int64_t *__restrict__ A_indptr, const T *__restrict__ B_data,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr,
    const int64_t *__restrict__ C_indptr, int64_t *__restrict__ C_indices, T *__restrict__ C_data) {
    constexpr int GPB = kBlock / G;
    constexpr int STRIDE = TABLE + (GPB > 1 ? kTablePad : 0);   // see symbolic_hash_kernel
    extern __shared__ __align__(16) unsigned char s_raw[];
    T *s_vals = reinterpret_cast<T *>(s_raw);
    int32_t *s_keys = reinterpret_cast<int32_t *>(s_raw + sizeof(T) * GPB * STRIDE);
    const int gl = threadIdx.x % G, gi = threadIdx.x / G;
    int32_t *tab = s_keys + gi * STRIDE;
    T *val = s_vals + gi * STRIDE;
    // compacted (column, slot) lists used to order the row on the way out.  The groups that share
    // a wavefront keep them where the key table was (its keys are in registers by then): LDS per
    // row is what decides how many rows a CU has in flight.
    constexpr int CSTRIDE = TABLE / 2 + 4;
    static_assert(CSTRIDE + TABLE / 4 <= TABLE && TABLE <= 65536, "the lists fit the key table");
    int32_t *ck = tab;
    uint16_t *cs16 = reinterpret_cast<uint16_t *>(ck + CSTRIDE);
    const int32_t b0 = bins[kBinStart + bin], b1 = bins[kBinStart + bin + 1];
    for (int32_t idx0 = b0 + blockIdx.x * GPB; idx0 < b1; idx0 += gridDim.x * GPB) {
        const int32_t idx = idx0 + gi;
        const bool live = idx < b1;
        for (int t = gl; t < TABLE; t += G) tab[t] = kEmpty;   // values are written by the first insert
        group_sync<G>();
        int64_t row = 0;
        auto add = [&](int32_t key, T prod) {
            uint32_t h = first_slot<TABLE>(key);
            int32_t old = atomicCAS(&tab[h], kEmpty, key);
            while (old != kEmpty && old != key) {   // one exit test: the common case probes once
                h = (h + 1) & (TABLE - 1);
                old = atomicCAS(&tab[h], kEmpty, key);
            }
            // The columns of one B row are distinct, so no other lane holds slot h now.  A slot
            // claimed just now holds no value yet: its first product is stored as it is
            // (0 + prod), the read of the slot is dropped by the select.
            const T cur = val[h];
            val[h] = old == kEmpty ? prod : cur + prod;
        };
        {
            // Same latency-lean walk as the symbolic phase; entries of A's row are still
            // applied one after the other, so every output entry gets its products in
            // the order of A's row.
            const int gbase = (threadIdx.x & (kWave - 1)) & ~(G - 1);
            row = live ? perm[idx] : 0;
            const int64_t ab = live ? A_indptr[row] : 0, ae = live ? A_indptr[row + 1] : 0;
            for (int64_t a0 = ab; a0 < ae; a0 += G) {
                const int64_t my_ai = a0 + gl;
                const bool mine = my_ai < ae;
                const int64_t my_j = mine ? A_indices[my_ai] : 0;
                const T my_a = mine ? A_data[my_ai] : T(0);
                const int64_t my_bb = mine ? B_indptr[my_j] : 0, my_be = mine ? B_indptr[my_j + 1] : 0;
                const int nb = (int)(ae - a0 < G ? ae - a0 : G);
                int32_t pk[kAhead];
                T pv[kAhead], as[kAhead];
                int64_t bbs[kAhead], bes[kAhead];
                // the entries of A's row held by lanes e0 .. e0 + kAhead - 1 of the group, applied in turn
                auto apply = [&](int e0) {
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) {
                        if (e0 + u >= nb) break;
                        if (pk[u] != kEmpty) add(pk[u], as[u] * pv[u]);
                        for (int64_t kk = bbs[u] + G + gl; kk < bes[u]; kk += G)
                            add((int32_t)B_indices[kk], as[u] * B_data[kk]);
                        group_sync<G>();  // the next entry of A's row adds after this one
                    }
                };
                if constexpr (G == 16) {
                    // A group is one 16-lane DPP row: what lane e of the group holds reaches the others
                    // by a row broadcast (one vector move per 32 bits) instead of a shuffle by lane
                    // number through the LDS crossbar.  That is cheap enough to fetch an entry's value
                    // and the bounds of its row of B again when they are used, so only the columns and
                    // values requested ahead stay in registers (116 -> fewer registers: more wavefronts).
                    constexpr int BATCH = NM_HASH_BATCH;   // rows of B requested ahead: 8 or 16
                    static_assert(G % BATCH == 0, "whole batches cover the group");
                    const int my_len = (int)(my_be - my_bb);
                    int32_t qk[BATCH];
                    T qv[BATCH];
                    auto batch = [&](auto first) {
                        constexpr int E0 = decltype(first)::value;
                        nm::static_for<BATCH>([&](auto uc) {
                            constexpr int U = decltype(uc)::value;
                            const int64_t kk = nm::row_lane<E0 + U>(my_bb) + gl;
                            const int len = nm::row_lane<E0 + U>(my_len);
                            const bool ok = (E0 + U < nb) & (gl < len);
                            qk[U] = ok ? (int32_t)B_indices[kk] : kEmpty;
                            qv[U] = ok ? B_data[kk] : T(0);
                        });
                        nm::static_for<BATCH>([&](auto uc) {
                            constexpr int U = decltype(uc)::value;
                            if (E0 + U >= nb) return;
                            const T a = nm::row_lane<E0 + U>(my_a);
                            if (qk[U] != kEmpty) add(qk[U], a * qv[U]);
                            if (nm::row_lane<E0 + U>(my_len) > G) {   // the rest of a row of B longer than the group
                                const int64_t bb = nm::row_lane<E0 + U>(my_bb), be = nm::row_lane<E0 + U>(my_be);
                                for (int64_t kk = bb + G + gl; kk < be; kk += G) add((int32_t)B_indices[kk], a * B_data[kk]);
                            }
                            group_sync<G>();  // the next entry of A's row adds after this one
                        });
                    };
                    batch(std::integral_constant<int, 0>{});
                    if constexpr (BATCH < G)
                        if (nb > BATCH) batch(std::integral_constant<int, BATCH < G ? BATCH : 0>{});
                } else {
                    for (int e0 = 0; e0 < nb; e0 += kAhead) {
#pragma unroll
                        for (int u = 0; u < kAhead; ++u) {
                            const int src = gbase + (e0 + u < nb ? e0 + u : e0);
                            bbs[u] = __shfl(my_bb, src, kWave);
                            bes[u] = __shfl(my_be, src, kWave);
                            as[u] = __shfl(my_a, src, kWave);
                            const int64_t kk = bbs[u] + gl;
                            const bool ok = e0 + u < nb && kk < bes[u];
                            pk[u] = ok ? (int32_t)B_indices[kk] : kEmpty;
                            pv[u] = ok ? B_data[kk] : T(0);
                        }
                        apply(e0);
                    }
                }
            }
        }
        // Output in ascending column order.
        {
            // The occupied slots are compacted into a dense list, then every entry is ranked
            // against that list only (its rank is its position in the row).  Rows fill at most
            // half of their table, so this is a fraction of the compares a rank over the whole
            // table would take.
            const int gbase = (threadIdx.x & (kWave - 1)) & ~(G - 1);
            constexpr int K = TABLE / G;
            int32_t keys[K];
            int mine = 0;
#pragma unroll
            for (int q = 0; q < K; ++q) {
                keys[q] = tab[gl + q * G];
                mine += keys[q] != kEmpty;
            }
            int incl = mine;
#pragma unroll
            for (int off = 1; off < G; off <<= 1) {
                const int up = __shfl_up(incl, off, kWave);
                if (gl >= off) incl += up;
            }
            const int c = __shfl(incl, gbase + G - 1, kWave);
            int pos = incl - mine;
            group_sync<G>();   // every lane holds its part of the table: the lists may take its place
#pragma unroll
            for (int q = 0; q < K; ++q)
                if (keys[q] != kEmpty) {
                    ck[pos] = keys[q];
                    cs16[pos] = (uint16_t)(gl + q * G);
                    ++pos;
                }
            if (gl < 4) ck[c + gl] = kEmpty;   // pad the list to a multiple of four keys
            group_sync<G>();
            if (live) {
                const int64_t base = C_indptr[row];
                const uint4 *ck4 = reinterpret_cast<const uint4 *>(ck);
                const int quads = (c + 3) >> 2;
                for (int e = gl; e < c; e += G) {
                    const uint32_t key = (uint32_t)ck[e];
                    int rank = 0;
                    for (int u = 0; u < quads; ++u) {   // four keys per LDS read; the pad never counts
                        const uint4 q = ck4[u];
                        rank += (q.x < key) + (q.y < key) + (q.z < key) + (q.w < key);
                    }
                    C_indices[base + rank] = (int64_t)key;
                    C_data[base + rank] = val[cs16[e]];
                }
            }
        }
        group_sync<G>();
    }
}

// Spill path: dense accumulator slice per workgroup (of the first `groups`), emitted by a scan of the
// touched column range (ascending by construction).
template <typename T>
__device__ __forceinline__ void numeric_spill(
    const int32_t *__restrict__ bins, const int32_t *__restrict__ perm, int64_t B_cols, int groups,
    const T *__restrict__ A_data, const int64_t *__restrict__ A_indices,
    const int64_t *__restrict__ A_indptr, const T *__restrict__ B_data,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr,
    const int64_t *__restrict__ C_indptr, int64_t *__restrict__ C_indices, T *__restrict__ C_data,
    int32_t *mark_all, double *acc_all) {
    __shared__ int64_t s_wave[kSpillBlock / kWave];
    __shared__ unsigned long long s_lo, s_hi;
    const int32_t b0 = bins[kBinStart + kBins - 1], b1 = bins[kBinStart + kBins];
    if ((int)blockIdx.x >= groups || b0 + (int32_t)blockIdx.x >= b1) return;
    int32_t *mark = mark_all + (size_t)blockIdx.x * (B_cols + 1);
    T *acc = reinterpret_cast<T *>(acc_all + (size_t)blockIdx.x * (B_cols + 1));
    for (int64_t c = threadIdx.x; c < B_cols; c += kSpillBlock) { mark[c] = 0; acc[c] = T(0); }
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    for (int32_t idx = b0 + blockIdx.x; idx < b1; idx += groups) {
        const int64_t row = perm[idx];
        const int32_t stamp = -((int32_t)row + 1);
        if (threadIdx.x == 0) { s_lo = ~0ull; s_hi = 0ull; }
        __syncthreads();
        unsigned long long lo = ~0ull, hi = 0ull;
        const int64_t je = A_indptr[row + 1];
        for (int64_t jj = A_indptr[row] + wave; jj < je; jj += kSpillBlock / kWave) {
            const int64_t j = A_indices[jj];
            const T a = A_data[jj];
            const int64_t ke = B_indptr[j + 1];
            for (int64_t kk = B_indptr[j] + lane; kk < ke; kk += kWave) {
                const unsigned long long c = (unsigned long long)B_indices[kk];
                nm::atomic_add(acc + c, a * B_data[kk]);
                mark[c] = stamp;
                lo = c < lo ? c : lo;
                hi = c > hi ? c : hi;
            }
        }
        if (lo != ~0ull) { atomicMin(&s_lo, lo); atomicMax(&s_hi, hi); }
        __syncthreads();
        const int64_t c_lo = (int64_t)s_lo, c_hi = (int64_t)s_hi;
        int64_t out = C_indptr[row];
        if (s_lo != ~0ull) {
            // Every wavefront takes a contiguous segment of the touched column range: it counts its
            // hits, the counts are summed over the wavefronts before it, and it then emits its
            // segment in order.  (A workgroup-wide scan per 1024 columns cost two barriers each.)
            constexpr int kWaves = kSpillBlock / kWave;
            const int64_t span = c_hi - c_lo + 1;
            const int64_t seg = ((span + kWaves - 1) / kWaves + kWave - 1) / kWave * kWave;
            const int64_t sb = c_lo + wave * seg;
            const int64_t se = sb + seg < c_hi + 1 ? sb + seg : c_hi + 1;
            int64_t cnt = 0;
            for (int64_t c0 = sb; c0 < se; c0 += kWave) {
                const int64_t c = c0 + lane;
                cnt += __popcll(__ballot(c < se && mark[c] == stamp));
            }
            if (lane == 0) s_wave[wave] = cnt;
            __syncthreads();
            for (int w = 0; w < wave; ++w) out += s_wave[w];
            const unsigned long long below = (1ull << lane) - 1ull;
            for (int64_t c0 = sb; c0 < se; c0 += kWave) {
                const int64_t c = c0 + lane;
                const bool hit = c < se && mark[c] == stamp;
                const unsigned long long m = __ballot(hit);
                if (hit) {
                    const int64_t at = out + __popcll(m & below);
                    C_indices[at] = c;
                    C_data[at] = acc[c];
                    acc[c] = T(0);
                }
                out += __popcll(m);
            }
        }
        __syncthreads();
    }
}

// ---- numeric, rows of more than 128 entries -------------------------------------------
//
// One row of C per workgroup.  The row's products are numbered in the order of A's row (and of
// B's rows inside it) and dealt to the threads by number, so the lanes are busy whatever the
// lengths of B's rows are; applied entry by entry of A's row, a row of B of eight entries kept
// eight of 256 lanes busy behind a barrier and a memory round trip each.  A product finds or
// claims its column's slot of the table in LDS; products of one chunk that meet in a slot take
// turns in the order of their numbers (every round the lowest one in each slot adds), so an entry
// of C still receives its products in the order of A's row, from +0.0.  After eight rounds with everybody
// the wavefronts go on one after the other, without barriers for every turn: 300 rows of 4000 entries whose every
// second product meets in one column, fp64, whole product 4.36 -> 0.86 ms, 1800 entries 1014 -> 345 us,
// every third product, fp32, 9000 entries 2.87 -> 1.32 ms.
// The row is then ordered by counting its columns into buckets of equal width between its first
// and last column and ranking each against its bucket, out of registers.  Where a bucket is
// crowded (columns packed together and one of them far away) that would be a
// compare for every pair of its columns, and the columns are sorted by a bitonic network instead.  300
// rows of a run of columns and one column 20 M away, fp32, whole product, ranked / sorted: 400
// entries 307 / 119 us, 1800 637 / 142, 4000 2519 / 228, 16000 14.8 / 0.67 ms.
// Bound by the row's chain of round trips and the barriers of the turns.  A 150 000-row power-law
// graph squared (mean 8, rows up to 1000, fp32), by length of C's row, against groups of 64 and 256
// lanes that applied A's entries one by one and ordered the row by ranks or a bitonic network:
// 129-256 60 -> 34 us, 257-512 127 -> 40, 513-1024 136 -> 43, 1025-4096 806 -> 108, more (dense
// accumulators in global memory) 854 -> 78.
// The launch for the longest rows takes those that spill as well.
template <typename T_, int TPB_, int SLOTS_, int LIMIT_, int UNROLL_, bool SPILL_ = false> struct RowShape {
    using T = T_;
    static constexpr bool SPILL = SPILL_;
    static constexpr int TPB = TPB_, SLOTS = SLOTS_, LIMIT = LIMIT_, UNROLL = UNROLL_;
    static constexpr int BATCH = TPB < 512 ? TPB : 512;                      // entries of A's row at a time
    static constexpr int TURNS = TPB < 1024 ? (TPB == kWave ? 512 : 1024) : 1024;   // turn words, by slot
    static constexpr int BUCKETS = TPB == kWave ? 256 : SLOTS < 4096 ? 1024 : 4096;
    static constexpr int PER = (SLOTS + TPB - 1) / TPB;                      // slots a thread reads out
    static constexpr int CROWD = TPB == kWave ? 64 : 128;                    // most columns of a bucket that are ranked
    static constexpr size_t at_off = sizeof(T) * SLOTS, at_row = at_off + 8 * (BATCH + 2), at_a = at_row + 8 * BATCH,
                            at_key = at_a + sizeof(T) * BATCH, at_turn = at_key + 4 * SLOTS,
                            end_sum = at_turn + 4 * TURNS;
    static constexpr size_t at_count = sizeof(T) * LIMIT, at_list = at_count + 4 * (BUCKETS + 2),
                            end_sort = at_list + 4 * LIMIT;
    static constexpr size_t at_red = ((end_sum > end_sort ? end_sum : end_sort) + 15) / 16 * 16;
    static constexpr size_t lds = at_red + 8 * (TPB / kWave) + 4 * 8;
    static_assert(lds <= 160 * 1024, "a CU's LDS");
    static constexpr int MOST = LIMIT & (LIMIT - 1) ? 2 << (31 - __builtin_clz(LIMIT)) : LIMIT;
    static_assert(4 * (size_t)MOST <= at_count, "a row padded to a power of two fits below the counts");
    static_assert(LIMIT < SLOTS && (TURNS & (TURNS - 1)) == 0 && SLOTS % 2 == 0 && LIMIT % 2 == 0, "tables");
};

// Rounds in which everybody asks for a turn before the wavefronts go one by one: of 1024 threads a round
// takes 0.5 us, all sixteen wavefronts in turn about 4 us.
constexpr uint32_t kTurnsTogether = 8;

template <typename S>
__global__ __launch_bounds__(S::TPB) void numeric_row_kernel(
    int bin, const int32_t *__restrict__ bins, const int32_t *__restrict__ perm,
    const typename S::T *__restrict__ A_data, const int64_t *__restrict__ A_indices,
    const int64_t *__restrict__ A_indptr, const typename S::T *__restrict__ B_data,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr,
    const int64_t *__restrict__ C_indptr, int64_t *__restrict__ C_indices, typename S::T *__restrict__ C_data,
    int64_t B_cols, int32_t *mark, double *acc, int spill_groups) {
    using T = typename S::T;
    constexpr int TPB = S::TPB, SLOTS = S::SLOTS, BATCH = S::BATCH, U = S::UNROLL, PER = S::PER;
    extern __shared__ __align__(16) unsigned char s_raw[];
    T *val = reinterpret_cast<T *>(s_raw);
    int64_t *s_off = reinterpret_cast<int64_t *>(s_raw + S::at_off);   // number of an entry's first product
    int64_t *s_row = reinterpret_cast<int64_t *>(s_raw + S::at_row);   // start of its row of B, less that number
    T *s_a = reinterpret_cast<T *>(s_raw + S::at_a);
    int32_t *tab = reinterpret_cast<int32_t *>(s_raw + S::at_key);
    uint32_t *turn = reinterpret_cast<uint32_t *>(s_raw + S::at_turn);
    int32_t *count = reinterpret_cast<int32_t *>(s_raw + S::at_count);
    int32_t *list = reinterpret_cast<int32_t *>(s_raw + S::at_list);
    int64_t *s_wave = reinterpret_cast<int64_t *>(s_raw + S::at_red);
    int32_t *s_flag = reinterpret_cast<int32_t *>(s_raw + S::at_red + 8 * (TPB / kWave));   // [0, 3) more, [3] first, [4] last column, [5] crowded
    const int tid = threadIdx.x;
    const int32_t b0 = bins[kBinStart + bin], b1 = bins[kBinStart + bin + 1];
    for (int32_t idx = b0 + (int32_t)blockIdx.x; idx < b1; idx += (int32_t)gridDim.x) {
        const int64_t row = perm[idx];
        const int64_t ab = A_indptr[row], ae = A_indptr[row + 1];
        for (int t = tid; t < SLOTS; t += TPB) {
            tab[t] = kEmpty;
            val[t] = T(0);
        }
        for (int t = tid; t < S::TURNS; t += TPB) turn[t] = 0;
        if (tid < 3) s_flag[tid] = 0;
        if (tid == 3) s_flag[3] = 0x7fffffff;
        if (tid == 4) s_flag[4] = -1;
        if (tid == 5) s_flag[5] = 0;
        uint32_t round = 0;
        int32_t first = 0x7fffffff, last = -1;
        for (int64_t a0 = ab; a0 < ae; a0 += BATCH) {
            const bool mine = tid < BATCH && a0 + tid < ae;
            const int64_t j = mine ? A_indices[a0 + tid] : 0;
            const T a = mine ? A_data[a0 + tid] : T(0);
            const int64_t bb = mine ? B_indptr[j] : 0, be = mine ? B_indptr[j + 1] : 0;
            int64_t total;
            const int64_t off = row_scan<TPB, int64_t>(be - bb, s_wave, total);
            __syncthreads();   // the last batch's products are done with the lists
            if (tid < BATCH) {
                s_off[tid] = off;   // (threads past the row's end: the total)
                s_row[tid] = bb - off;
                s_a[tid] = a;
            }
            __syncthreads();
            for (int64_t p0 = 0; p0 < total; p0 += TPB * U) {
                int32_t key[U];
                T prod[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t p = p0 + u * TPB + tid;
                    const bool have = p < total;
                    const int64_t at = have ? p : 0;
                    int e = 0;   // the last entry whose first product is not behind this one
#pragma unroll
                    for (int step = BATCH / 2; step > 0; step >>= 1)
                        if (s_off[e + step] <= at) e += step;
                    const int64_t kk = s_row[e] + at;
                    key[u] = (int32_t)B_indices[kk];
                    prod[u] = s_a[e] * B_data[kk];
                    if (!have) key[u] = kEmpty;
                }
                int slot[U] = {};
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (key[u] == kEmpty) continue;
                    first = min(first, key[u]);
                    last = max(last, key[u]);
                    uint32_t h = __umulhi((uint32_t)key[u] * 0x9E3779B1u, (uint32_t)SLOTS);
                    int32_t old = atomicCAS(&tab[h], kEmpty, key[u]);
                    while (old != kEmpty && old != key[u]) {
                        h = h + 1 == SLOTS ? 0 : h + 1;
                        old = atomicCAS(&tab[h], kEmpty, key[u]);
                    }
                    slot[u] = (int)h;
                }
                // Turns.  A word of `turn` holds the latest round it was asked for and, of the threads
                // that asked, the lowest: a later round's words are larger than an earlier one's, so
                // nothing is reset in between.  (Slots that share a word only wait for each other.)
                if (round >= (1u << 22) - 64 * U) {   // 10 bits below hold the thread
                    __syncthreads();
                    for (int t = tid; t < S::TURNS; t += TPB) turn[t] = 0;
                    if (tid < 3) s_flag[tid] = 0;
                    round = 0;
                    __syncthreads();
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (p0 + u * TPB >= total) break;
                    uint32_t *word = turn + (slot[u] & (S::TURNS - 1));
                    bool waits = key[u] != kEmpty;
                    bool more;
                    const uint32_t together = round + kTurnsTogether;
                    do {
                        ++round;
                        const int now = round % 3, next = (round + 1) % 3;
                        const uint32_t asked = round << 10 | (uint32_t)(TPB - 1 - tid);
                        if (waits) atomicMax(word, asked);
                        if (TPB > kWave && tid == 0) s_flag[next] = 0;
                        __syncthreads();
                        if (waits && *word == asked) {
                            val[slot[u]] += prod[u];
                            waits = false;
                        }
                        if constexpr (TPB > kWave) {
                            if (waits) s_flag[now] = 1;
                            __syncthreads();
                            more = s_flag[now] != 0;
                        } else {
                            more = __ballot(waits) != 0;
                        }
                    } while (more && round != together);
                    if (__builtin_expect(!more, 1)) continue;
                    // Many products for one slot (a column of B that is full, or nearly): the wavefronts go on
                    // one after the other, each with two turns among its own lanes and then slot by slot, a
                    // slot's products added up in the order of the lanes.
                    const int wave = tid / kWave;
                    for (int w = 0; w < TPB / kWave; ++w) {
                        if (wave == w) {
#pragma unroll
                            for (int t = 1; t <= 2; ++t) {
                                const uint32_t asked = (round + 2 * w + t) << 10 | (uint32_t)(TPB - 1 - tid);
                                if (waits) atomicMax(word, asked);
                                group_sync<kWave>();
                                if (waits && *word == asked) {
                                    val[slot[u]] += prod[u];
                                    waits = false;
                                }
                                group_sync<kWave>();
                            }
                            uint64_t left = __ballot(waits);
                            while (left) {
                                const int s0 = nm::read_lane(slot[u], __builtin_ctzll(left));
                                const uint64_t same = left & __ballot(slot[u] == s0);
                                T acc = val[s0];
                                for (uint64_t m = same; m; m &= m - 1) acc += nm::read_lane(prod[u], __builtin_ctzll(m));
                                val[s0] = acc;
                                left &= ~same;
                            }
                        }
                        if (TPB > kWave) __syncthreads();
                        else group_sync<kWave>();
                    }
                    round += 2 * (TPB / kWave);
                    if constexpr (TPB > kWave) {
                        if (tid < 3) s_flag[tid] = 0;
                        __syncthreads();
                    }
                }
            }
        }
        // ---- the row in ascending order of its columns ----
        if (last >= 0) {
            atomicMin(&s_flag[3], first);
            atomicMax(&s_flag[4], last);
        }
        int32_t key[PER], rank[PER];
        T sum[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int t = tid + q * TPB;
            key[q] = t < SLOTS ? tab[t] : kEmpty;
            sum[q] = t < SLOTS ? val[t] : T(0);
        }
        __syncthreads();   // the table's memory is free from here on
        const int32_t low = s_flag[3];
        const uint32_t width = s_flag[4] >= low ? (uint32_t)(s_flag[4] - low) : 0;
        constexpr int BITS = __builtin_ctz(S::BUCKETS);
        const int need = 32 - __clz(width | 1), shift = need > BITS ? need - BITS : 0;
        for (int t = tid; t < S::BUCKETS; t += TPB) count[t] = 0;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < PER; ++q)
            rank[q] = key[q] != kEmpty ? atomicAdd(&count[(uint32_t)(key[q] - low) >> shift], 1) : 0;
        __syncthreads();
        {
            constexpr int RUN = S::BUCKETS / TPB;
            int c[RUN], mine = 0, all;
#pragma unroll
            for (int q = 0; q < RUN; ++q) {
                c[q] = count[tid * RUN + q];
                mine += c[q];
                if (c[q] > S::CROWD) s_flag[5] = 1;
            }
            int run = row_scan<TPB, int>(mine, reinterpret_cast<int *>(s_wave), all);
#pragma unroll
            for (int q = 0; q < RUN; ++q) {
                count[tid * RUN + q] = run;
                run += c[q];
            }
            if (tid == 0) count[S::BUCKETS] = all;
        }
        __syncthreads();
        const int n = count[S::BUCKETS];
        const bool crowded = s_flag[5] != 0;
        int32_t *sorted = reinterpret_cast<int32_t *>(s_raw);
        int32_t *place = crowded ? sorted : list;
#pragma unroll
        for (int q = 0; q < PER; ++q)
            if (key[q] != kEmpty) place[count[(uint32_t)(key[q] - low) >> shift] + rank[q]] = key[q];
        if (!crowded) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                if (key[q] == kEmpty) continue;
                const uint32_t b = (uint32_t)(key[q] - low) >> shift;
                const int lo = count[b], hi = count[b + 1];
                int r = lo;
                for (int t = lo; t < hi; ++t) r += list[t] < key[q];
                rank[q] = r;
                sorted[r] = key[q];
            }
        } else {
            int P = 2 * kWave;
            while (P < n) P <<= 1;
            for (int t = n + tid; t < P; t += TPB) sorted[t] = kColEnd;
            __syncthreads();
            for (int k = 2; k <= P; k <<= 1) {
                for (int j = k >> 1; j > 0; j >>= 1) {
                    for (int t = tid; t < P / 2; t += TPB) {
                        const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), l = i | j;
                        const int32_t x = sorted[i], y = sorted[l];
                        if ((x > y) == ((i & k) == 0)) { sorted[i] = y; sorted[l] = x; }
                    }
                    // a wavefront's pairs stay inside its own 128 words while j <= 64
                    if (j > kWave) __syncthreads(); else group_sync<kWave>();
                }
                if (k >= 2 * kWave) __syncthreads();
            }
            // a column's place is the number of columns below it
#pragma unroll
            for (int q = 0; q < PER; ++q) rank[q] = 0;
            for (int step = P / 2; step > 0; step >>= 1)
#pragma unroll
                for (int q = 0; q < PER; ++q)
                    if (sorted[rank[q] + step - 1] < key[q]) rank[q] += step;
        }
        __syncthreads();
        const int64_t base = C_indptr[row];
        for (int t = tid; t < n; t += TPB) C_indices[base + t] = (int64_t)sorted[t];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < PER; ++q)
            if (key[q] != kEmpty) val[rank[q]] = sum[q];
        __syncthreads();
        for (int t = tid; t < n; t += TPB) C_data[base + t] = val[t];
        __syncthreads();
    }
    if constexpr (S::SPILL) {
        static_assert(TPB == kSpillBlock && S::lds + 256 <= 160 * 1024, "the spill path's workgroup and LDS");
        numeric_spill<T>(bins, perm, B_cols, spill_groups, A_data, A_indices, A_indptr, B_data, B_indices, B_indptr,
                         C_indptr, C_indices, C_data, mark, acc);
    }
}

// The shapes: LDS decides how many rows a CU has in flight, so a row gets the smallest table that
// holds its bin at three quarters load; the last one takes the LDS of a whole CU, at nine tenths, and
// keeps ten registers (fp64: eleven) of a thread's share of the table in scratch memory.
template <typename T> using RowShape3 = RowShape<T, 64, 384, 256, 2>;
template <typename T> using RowShape4 = RowShape<T, 64, 704, 512, 2>;
template <typename T> using RowShape5 = RowShape<T, 256, 1408, 1024, 2>;
template <typename T> using RowShape6 = RowShape<T, 512, 2816, 2048, 4>;
template <typename T> using RowShape7 = RowShape<T, 1024, 5632, 4096, 4>;
constexpr int32_t kRowLimitMost32 = 16384, kRowLimitMost64 = 10880;
template <typename T>
using RowShape8 = RowShape<T, 1024, sizeof(T) == 4 ? 18176 : 12224, sizeof(T) == 4 ? kRowLimitMost32 : kRowLimitMost64, 4, true>;

// ---- backward --------------------------------------------------------------------

// Backward.  A group of 8 lanes owns one row i of A.  Row i of C (column
// indices and upstream gradient, at most kBwdStage entries) is staged in LDS,
// so the per-product lookups are LDS bisections.  The group takes the row's entries
// (i,k) one at a time and spreads row k of B over its lanes, so the eight
// atomic updates of grad_B it issues land in one cache line (the L2 atomic
// units are bound by lines touched, not by lanes).  The products
// gC[i,c] * B[k,c] are then added lane by lane in ascending column order --
// the order of the reference's merge -- which keeps grad_A bit-identical.
//
// Rows of C longer than kBwdStage get a wavefront (up to 512 entries) or a workgroup each, of 256 (up
// to 2048) or 1024 threads.  The row's products are numbered through in the order of A's row and
// dealt to the threads by number (as in numeric_row_kernel), each looks its column up in the row of
// C in LDS, and the thread of an entry of A adds the entry's products from LDS in order.  Of a row
// longer than LDS holds, every stride-th column is staged: the last steps of the search then read
// global memory.
// Bound by the row's chain of round trips, the searches in LDS and the atomic adds of the gradient of B.  A
// 150 000-row power-law graph squared (mean 8, rows up to 1000, fp32), kernels of the rows of 65-2048 and of
// more entries, against one workgroup of 256 threads whose groups of eight lanes took A's entries
// one by one: 617 -> 208 us, 679 -> 223 us.
constexpr int kBwdG = 8;
constexpr int kBwdStage = 64;

// What lane E of every eight consecutive lanes holds, handed to all eight (ds_swizzle in bit mode:
// lane = (lane & 0x18) | E inside each half of the wavefront; no address to compute).
template <int E> __device__ __forceinline__ int group_lane(int v) {
    static_assert(E >= 0 && E < 8, "a lane of the group");
    return __builtin_amdgcn_ds_swizzle(v, (E << 5) | 0x18);
}
template <int E> __device__ __forceinline__ float group_lane(float v) {
    return __int_as_float(group_lane<E>(__float_as_int(v)));
}
template <int E> __device__ __forceinline__ int64_t group_lane(int64_t v) {
    const int lo = group_lane<E>((int)(v & 0xffffffffll)), hi = group_lane<E>((int)(v >> 32));
    return ((int64_t)hi << 32) | (uint32_t)lo;
}
template <int E> __device__ __forceinline__ double group_lane(double v) {
    return __longlong_as_double(group_lane<E>((int64_t)__double_as_longlong(v)));
}

template <typename T>
__global__ __launch_bounds__(kBlock) void spgemm_bwd_kernel(
    int64_t A_rows, const T *__restrict__ gC, const int64_t *__restrict__ C_indices,
    const int64_t *__restrict__ C_indptr, const T *__restrict__ A_data,
    const int64_t *__restrict__ A_indices, const int64_t *__restrict__ A_indptr,
    const T *__restrict__ B_data, const int64_t *__restrict__ B_indices,
    const int64_t *__restrict__ B_indptr, T *__restrict__ grad_A, T *__restrict__ grad_B) {
    constexpr int G = kBwdG, GPB = kBlock / G;
    static_assert(G == 8 && kBwdStage == 64, "group_lane and the six-step search are written for these");
    // (a group's row starts one bank further on than its neighbour's: the groups of a wavefront
    // probe the same place of their rows at the same step of the search)
    constexpr int kStride = kBwdStage + 1;
    __shared__ int32_t s_ci[GPB * kStride];
    __shared__ T s_g[GPB * kStride];
    const int gl = threadIdx.x % G, gi = G >= kWave ? __builtin_amdgcn_readfirstlane(threadIdx.x / G) : threadIdx.x / G;
    const int gbase = (threadIdx.x & (kWave - 1)) & ~(G - 1);   // first lane of the group inside its wavefront
    int32_t *ci = s_ci + gi * kStride;
    T *cg = s_g + gi * kStride;
    for (int64_t i0 = (int64_t)blockIdx.x * GPB; i0 < A_rows; i0 += (int64_t)gridDim.x * GPB) {
        const int64_t i = i0 + gi;
        const bool live = i < A_rows;
        const int64_t cb = live ? C_indptr[i] : 0, ce = live ? C_indptr[i + 1] : 0;
        const int clen = (int)(ce - cb < 0x7fffffff ? ce - cb : 0x7fffffff);
        const bool here = live && clen <= kBwdStage;   // longer rows are left to spgemm_bwd_long_kernel
        // (places past the row's end hold a column no entry has: the search below takes six steps
        // whatever the row's length and needs no bound)
        if (here)
            for (int t = gl; t < kBwdStage; t += G) {
                ci[t] = t < clen ? (int32_t)C_indices[cb + t] : 0x7fffffff;
                if (t < clen) cg[t] = gC[cb + t];
            }
        group_sync<G>();
        const int64_t ab = here ? A_indptr[i] : 0, ae = here ? A_indptr[i + 1] : 0;
        for (int64_t a0 = ab; a0 < ae; a0 += G) {
            // each lane fetches one entry of A's row and the bounds of the B row it names
            const int64_t my_ai = a0 + gl;
            const bool mine = my_ai < ae;
            const int64_t my_k = mine ? A_indices[my_ai] : 0;
            const T my_a = (mine && grad_B) ? A_data[my_ai] : T(0);
            const int64_t my_bb = mine ? B_indptr[my_k] : 0, my_be = mine ? B_indptr[my_k + 1] : 0;
            const int nb = (int)(ae - a0 < G ? ae - a0 : G);
            const int my_len = (int)(my_be - my_bb);
            T my_acc = 0;
            // (unrolled: the lane whose entry is applied is then a constant of the instruction that
            // hands its row start, length and value to the group, with no address to compute)
            nm::static_for<G>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                if (e >= nb) return;
                const int64_t bb = group_lane<e>(my_bb), be = bb + group_lane<e>(my_len);
                const T a = grad_B ? group_lane<e>(my_a) : T(0);
                T acc = 0;
                for (int64_t kk0 = bb; kk0 < be; kk0 += G) {
                    const int64_t kk = kk0 + gl;
                    const bool have = kk < be;
                    const int32_t c = have ? (int32_t)B_indices[kk] : -1;
                    const T bval = have && grad_A ? B_data[kk] : T(0);
                    // the number of staged columns below c (at most 63), in six steps without a branch
                    int l = 0;
#pragma unroll
                    for (int step = kBwdStage / 2; step > 0; step >>= 1)
                        if (ci[l + step - 1] < c) l += step;
                    const bool hit = have && ci[l] == c;
                    const T g = hit ? cg[l] : T(0);
                    if (hit && grad_B) nm::atomic_add(grad_B + kk, a * g);
                    if (!grad_A) continue;
                    // Ordered sum over the group's lanes = ascending column: the running sum walks up
                    // the lanes, one DPP shift and one addition a step (every lane adds what its lower
                    // neighbour held a step ago to its own product; lane s is right after step s and
                    // is read at step s + 1, what the others hold meanwhile is never used).  A lane
                    // without a product adds +0.0, which changes no sum that began at +0.0.
                    const T prod = g * bval;   // (g is +0.0 without a hit, bval finite or the lane's own)
                    T run = acc + (hit ? prod : T(0));
#pragma unroll
                    for (int step = 1; step < G; ++step) run = nm::dpp_move<0x111>(run) + (hit ? prod : T(0));
                    acc = group_lane<G - 1>(run);
                }
                if (gl == e) my_acc = acc;
            });
            if (mine && grad_A) grad_A[my_ai] = my_acc;
        }
        group_sync<G>();
    }
}

// Threads that work on a row: a wavefront or a workgroup.
template <int TPB> __device__ __forceinline__ void row_sync() {
    if constexpr (TPB == kWave) group_sync<kWave>();
    else __syncthreads();
}

template <typename T> struct BackArgs {
    int64_t A_rows;
    int piece;   // rows a workgroup looks at side by side, see back_row
    const T *gC;
    const int64_t *C_indices, *C_indptr;
    const T *A_data;
    const int64_t *A_indices, *A_indptr;
    const T *B_data;
    const int64_t *B_indices, *B_indptr;
    T *grad_A, *grad_B;
};

template <typename T_, int TPB_, int CAP_, int UNROLL_> struct BackShape {
    using T = T_;
    static constexpr int TPB = TPB_, CAP = CAP_, UNROLL = UNROLL_, BATCH = TPB < 512 ? TPB : 512;
    static constexpr int STEP = TPB * UNROLL;                                  // products at a time
    static constexpr size_t at_prod = sizeof(T) * CAP, at_off = at_prod + sizeof(T) * STEP,
                            at_row = at_off + 8 * (BATCH + 2), at_a = at_row + 8 * BATCH,
                            at_wave = at_a + 8 * BATCH, at_col = at_wave + 8 * (TPB / kWave) + 16;
    static constexpr size_t lds = (at_col + 4 * CAP + 15) / 16 * 16;
    static_assert((CAP * sizeof(T)) % 8 == 0 && (STEP * sizeof(T)) % 8 == 0, "64-bit words behind the values");
};

// Row i by the threads of shape S, the first of them `tid` 0, in the S::lds bytes at s_raw.
template <typename S>
__device__ __forceinline__ void back_one_row(const BackArgs<typename S::T> &g, int64_t i, int tid, unsigned char *s_raw) {
    using T = typename S::T;
    constexpr int TPB = S::TPB, CAP = S::CAP, BATCH = S::BATCH, U = S::UNROLL, STEP = S::STEP;
    const T *__restrict__ gC = g.gC, *__restrict__ A_data = g.A_data, *__restrict__ B_data = g.B_data;
    const int64_t *__restrict__ C_indices = g.C_indices, *__restrict__ C_indptr = g.C_indptr;
    const int64_t *__restrict__ A_indices = g.A_indices, *__restrict__ A_indptr = g.A_indptr;
    const int64_t *__restrict__ B_indices = g.B_indices, *__restrict__ B_indptr = g.B_indptr;
    T *__restrict__ grad_A = g.grad_A, *__restrict__ grad_B = g.grad_B;
    T *cg = reinterpret_cast<T *>(s_raw);
    T *s_prod = reinterpret_cast<T *>(s_raw + S::at_prod);
    int64_t *s_off = reinterpret_cast<int64_t *>(s_raw + S::at_off);   // number of an entry's first product
    int64_t *s_row = reinterpret_cast<int64_t *>(s_raw + S::at_row);   // start of its row of B, less that number
    T *s_a = reinterpret_cast<T *>(s_raw + S::at_a);
    int64_t *s_wave = reinterpret_cast<int64_t *>(s_raw + S::at_wave);
    int32_t *ci = reinterpret_cast<int32_t *>(s_raw + S::at_col);
    const int64_t cb = C_indptr[i], clen = C_indptr[i + 1] - cb;
    const int64_t stride = (clen + CAP - 1) / CAP;
    const int ns = (int)((clen + stride - 1) / stride);
    const bool whole = stride == 1;
    for (int t = tid; t < ns; t += TPB) {
        ci[t] = (int32_t)C_indices[cb + t * stride];
        if (whole) cg[t] = gC[cb + t];
    }
    const int top = 1 << (31 - __clz(ns));   // the first step of a search through ns columns
    const int64_t ab = A_indptr[i], ae = A_indptr[i + 1];
    for (int64_t a0 = ab; a0 < ae; a0 += BATCH) {
        const bool mine = tid < BATCH && a0 + tid < ae;
        const int64_t j = mine ? A_indices[a0 + tid] : 0;
        const T a = mine && grad_B ? A_data[a0 + tid] : T(0);
        const int64_t bb = mine ? B_indptr[j] : 0, be = mine ? B_indptr[j + 1] : 0;
        int64_t total;
        const int64_t off = row_scan<TPB, int64_t>(be - bb, s_wave, total), end = off + (be - bb);
        if (tid < BATCH) {
            s_off[tid] = off;   // (threads past the row's end: the total)
            s_row[tid] = bb - off;
            s_a[tid] = a;
        }
        row_sync<TPB>();
        T acc = 0;
        for (int64_t p0 = 0; p0 < total; p0 += STEP) {
            int64_t kk[U], c[U];
            T b[U], av[U];
            int l[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t p = p0 + u * TPB + tid;
                const bool have = p < total;
                const int64_t at = have ? p : 0;
                int e = 0;   // the last entry whose first product is not behind this one
#pragma unroll
                for (int step = BATCH / 2; step > 0; step >>= 1)
                    if (s_off[e + step] <= at) e += step;
                kk[u] = s_row[e] + at;
                av[u] = s_a[e];
                c[u] = B_indices[kk[u]];
                b[u] = grad_A ? B_data[kk[u]] : T(0);
                if (!have) c[u] = -1;
                l[u] = 0;
            }
            // the number of staged columns below c
            for (int step = top; step > 0; step >>= 1)
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (l[u] + step <= ns && (int64_t)ci[l[u] + step - 1] < c[u]) l[u] += step;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                bool hit;
                T g = 0;
                if (whole) {
                    hit = l[u] < ns && (int64_t)ci[l[u]] == c[u];
                    if (hit) g = cg[l[u]];
                } else {
                    // sample l is the first one not below c: the column, if present, sits
                    // after sample l - 1 and no later than sample l
                    int64_t lo = l[u] == 0 ? 0 : (int64_t)(l[u] - 1) * stride + 1;
                    int64_t hi = (int64_t)l[u] * stride < clen ? (int64_t)l[u] * stride : clen;
                    if (c[u] < 0) hi = lo;
                    while (lo < hi) {
                        const int64_t mid = (lo + hi) >> 1;
                        if (C_indices[cb + mid] < c[u]) lo = mid + 1; else hi = mid;
                    }
                    hit = c[u] >= 0 && lo < clen && C_indices[cb + lo] == c[u];
                    if (hit) g = gC[cb + lo];
                }
                if (hit && grad_B) nm::atomic_add(grad_B + kk[u], av[u] * g);
                s_prod[u * TPB + tid] = hit ? g * b[u] : T(0);
            }
            if (!grad_A) continue;
            row_sync<TPB>();
            // an entry's thread adds its products in ascending column (a product that is missing
            // is +0.0, which changes no sum that began at +0.0)
            if (off < p0 + STEP && end > p0) {
                int t = off > p0 ? (int)(off - p0) : 0;
                const int t1 = end - p0 < STEP ? (int)(end - p0) : STEP;
                // (eight are on their way while eight are added: one after the other, a row of B of
                // a thousand entries was a thousand trips to LDS)
                constexpr int W = 8;
                if (t + W <= t1) {
                    T x[W];
#pragma unroll
                    for (int w = 0; w < W; ++w) x[w] = s_prod[t + w];
                    for (t += W; t + W <= t1; t += W) {
                        T y[W];
#pragma unroll
                        for (int w = 0; w < W; ++w) y[w] = s_prod[t + w];
#pragma unroll
                        for (int w = 0; w < W; ++w) {
                            acc += x[w];
                            x[w] = y[w];
                        }
                    }
#pragma unroll
                    for (int w = 0; w < W; ++w) acc += x[w];
                }
                for (; t < t1; ++t) acc += s_prod[t];
            }
            row_sync<TPB>();
        }
        if (mine && grad_A) grad_A[a0 + tid] = acc;
        row_sync<TPB>();   // (the lists are this batch's until here)
    }
    row_sync<TPB>();
}

// A workgroup looks through its rows for the long ones, a thread a row.  Rows next to each other are often alike,
// so they are dealt in pieces of up to eight (a cache line of the row pointer) in turn: the row of thread t in the
// workgroup's `turn`-th look, or past the last one.
__device__ __forceinline__ int64_t back_row(int64_t turn, int t, int threads, int piece) {
    return ((turn * (threads / piece) + t / piece) * (int64_t)gridDim.x + blockIdx.x) * piece + t % piece;
}

// Rows of C of kBwdStage + 1 to 512 entries, a wavefront each, and of up to 2048, the workgroup's.
constexpr int kBackMid = 256;
constexpr int64_t kBackWave = 512, kBackGroup = 2048;
template <typename T> using BackMidRow = BackShape<T, kBackMid, kBackGroup, 4>;
template <typename T> using BackWaveRow = BackShape<T, kWave, kBackWave, 4>;
template <typename T>
constexpr size_t kBackMidLds = BackMidRow<T>::lds > kBackMid / kWave * BackWaveRow<T>::lds ? BackMidRow<T>::lds
                                                                                          : kBackMid / kWave * BackWaveRow<T>::lds;

template <typename T> __global__ __launch_bounds__(kBackMid) void spgemm_bwd_mid_kernel(BackArgs<T> g) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    __shared__ uint8_t s_of_wave[kBackMid], s_of_group[kBackMid];
    __shared__ int s_n[3];   // rows in the two lists, next of the first
    static_assert(kBackMid <= 256, "a thread's number fits a byte");
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    for (int64_t turn = 0; back_row(turn, 0, kBackMid, g.piece) < g.A_rows; ++turn) {
        const int64_t r = back_row(turn, tid, kBackMid, g.piece);
        const int64_t len = r < g.A_rows ? g.C_indptr[r + 1] - g.C_indptr[r] : 0;
        const bool of_wave = len > kBwdStage && len <= kBackWave, of_group = len > kBackWave && len <= kBackGroup;
        if (!__syncthreads_or(of_wave || of_group)) continue;
        if (tid < 3) s_n[tid] = 0;
        __syncthreads();
        if (of_wave) s_of_wave[atomicAdd(&s_n[0], 1)] = (uint8_t)tid;
        if (of_group) s_of_group[atomicAdd(&s_n[1], 1)] = (uint8_t)tid;
        __syncthreads();
        const int waves = s_n[0], groups = s_n[1];
        for (int q = 0; q < groups; ++q)
            back_one_row<BackMidRow<T>>(g, back_row(turn, s_of_group[q], kBackMid, g.piece), tid, s_raw);
        while (true) {
            int q = 0;
            if (lane == 0) q = atomicAdd(&s_n[2], 1);
            q = __builtin_amdgcn_readfirstlane(q);
            if (q >= waves) break;
            back_one_row<BackWaveRow<T>>(g, back_row(turn, s_of_wave[q], kBackMid, g.piece), lane,
                                         s_raw + wave * BackWaveRow<T>::lds);
        }
        __syncthreads();
    }
}

// Longer rows, one at a time by a workgroup that takes a CU's LDS.
template <typename T> using BackLongRow = BackShape<T, 1024, sizeof(T) == 4 ? 14336 : 8192, 4>;
template <typename T> __global__ __launch_bounds__(1024) void spgemm_bwd_long_kernel(BackArgs<T> g) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    __shared__ uint16_t s_long[1024];
    __shared__ int s_n;
    static_assert(BackLongRow<T>::lds + sizeof(s_long) + 16 <= 160 * 1024, "a CU's LDS");
    const int tid = threadIdx.x;
    for (int64_t turn = 0; back_row(turn, 0, 1024, g.piece) < g.A_rows; ++turn) {
        const int64_t r = back_row(turn, tid, 1024, g.piece);
        const bool is_long = r < g.A_rows && g.C_indptr[r + 1] - g.C_indptr[r] > kBackGroup;
        if (!__syncthreads_or(is_long)) continue;
        if (tid == 0) s_n = 0;
        __syncthreads();
        if (is_long) s_long[atomicAdd(&s_n, 1)] = (uint16_t)tid;
        __syncthreads();
        const int n = s_n;
        for (int q = 0; q < n; ++q)
            back_one_row<BackLongRow<T>>(g, back_row(turn, s_long[q], 1024, g.piece), tid, s_raw);
        __syncthreads();
    }
}

int check_common(int64_t A_rows, int64_t B_cols) {
    NM_REQUIRE(A_rows >= 0 && B_cols >= 0, "negative size");
    if (A_rows >= 0x7ffffffe || B_cols >= 0x7ffffffe)
        return nm::fail(NM_ERR_UNSUPPORTED, "spgemm indexes rows and columns with 32 bits inside its tables");
    return NM_OK;
}

constexpr unsigned kPersistGrid = 4096;

template <typename T>
int launch_numeric(const Work &w, int64_t B_cols, const void *A_data, const int64_t *A_indices,
                   const int64_t *A_indptr, const void *B_data, const int64_t *B_indices,
                   const int64_t *B_indptr, const int64_t *C_indptr, int64_t *C_indices, void *C_data,
                   hipStream_t s) {
    const T *Ad = (const T *)A_data, *Bd = (const T *)B_data;
    T *Cd = (T *)C_data;
    constexpr size_t per = sizeof(T) + sizeof(int32_t);
    auto hashed = [&](auto group, auto table, int bin, unsigned grid) -> int {
        constexpr int G = decltype(group)::value, TABLE = decltype(table)::value;
        auto k = numeric_hash_kernel<T, G, TABLE>;
        const size_t lds = (kBlock / G) * per * (TABLE + kTablePad);   // tables (values + keys), padded apart
        static_assert((kBlock / G) * per * (TABLE + kTablePad) <= 64 * 1024, "no attribute asked for");
        hipLaunchKernelGGL(k, dim3(grid), dim3(kBlock), lds, s, bin, w.bins, w.perm, Ad, A_indices, A_indptr, Bd,
                           B_indices, B_indptr, C_indptr, C_indices, Cd);
        NM_LAUNCH_CHECK("numeric_hash_kernel");
        return NM_OK;
    };
    using std::integral_constant;
    if (int rc = hashed(integral_constant<int, kGroup0>{}, integral_constant<int, kNumTable0>{}, 0, kPersistGrid)) return rc;
    if (int rc = hashed(integral_constant<int, kGroup1>{}, integral_constant<int, kNumTable1>{}, 1, kPersistGrid)) return rc;
    if (int rc = hashed(integral_constant<int, kGroup2>{}, integral_constant<int, kNumTable2>{}, 2, kPersistGrid)) return rc;
    auto rows = [&](auto shape, int bin, unsigned grid) -> int {
        using S = decltype(shape);
        auto k = numeric_row_kernel<S>;
        if (S::lds > 64 * 1024)
            NM_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds));
        hipLaunchKernelGGL(k, dim3(grid), dim3(S::TPB), S::lds, s, bin, w.bins, w.perm, Ad, A_indices, A_indptr, Bd,
                           B_indices, B_indptr, C_indptr, C_indices, Cd, B_cols, w.mark, w.acc, spill_groups(B_cols));
        NM_LAUNCH_CHECK("numeric_row_kernel");
        return NM_OK;
    };
    if (int rc = rows(RowShape3<T>{}, 3, kPersistGrid)) return rc;
    if (int rc = rows(RowShape4<T>{}, 4, kPersistGrid)) return rc;
    if (int rc = rows(RowShape5<T>{}, 5, kPersistGrid)) return rc;
    if (int rc = rows(RowShape6<T>{}, 6, 2048)) return rc;
    if (int rc = rows(RowShape7<T>{}, 7, 1024)) return rc;
    if (int rc = rows(RowShape8<T>{}, 8, 512)) return rc;
    return NM_OK;
}

}  // namespace

extern "C" int nm_spgemm_workspace_bytes(int64_t A_rows, int64_t B_cols, size_t *bytes) {
    NM_REQUIRE(bytes != nullptr, "bytes is null");
    if (int rc = check_common(A_rows, B_cols)) return rc;
    *bytes = work_layout(A_rows, B_cols, nullptr, nullptr);
    return NM_OK;
}

namespace {

// The symbolic phase; with `map` its first kernel also records where every product of a
// merge-path row goes (the destination bytes and B row starts of a product plan).
int symbolic_phase(int64_t A_rows, int64_t A_cols, int64_t B_cols, const int64_t *A_indices,
                   const int64_t *A_indptr, const int64_t *B_indices, const int64_t *B_indptr, int64_t *C_indptr,
                   void *workspace, size_t workspace_bytes, void *host_landing, const nm::PPlan *map,
                   nm_stream stream) {
    if (int rc = check_common(A_rows, B_cols)) return rc;
    NM_REQUIRE(A_cols >= 0, "negative size");
    NM_REQUIRE(A_indptr && B_indptr && C_indptr && workspace, "null pointer argument");
    Work w;
    const size_t need = work_layout(A_rows, B_cols, workspace, &w);
    if (workspace_bytes < need)
        return nm::fail(NM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, need);
    hipStream_t s = nm::as_stream(stream);
    if (A_rows == 0) return nm::fill_async(C_indptr, 1, (int64_t)0, s);

    const int64_t tiles = nm::ceil_div(A_rows + 1, nm::kScanTile);
    if (tiles > nm::kMaxGrid) return nm::fail(NM_ERR_UNSUPPORTED, "%lld rows are too many", (long long)A_rows);
    // What the first kernel writes over summary[1] where it leaves a row to the hash path: not a
    // count of rows (the word's content at the end of every call) and not an earlier call's token.
    volatile int64_t *both = (volatile int64_t *)host_landing;
    const int64_t ticket = both ? both[2] + 1 : 1;
    const int64_t token = ticket | ((int64_t)1 << 62);
    const int64_t nbatch = nm::xcd_padded(nm::ceil_div(A_rows, kMergeRows));
    hipLaunchKernelGGL(symbolic_front_kernel, dim3((unsigned)nbatch), dim3(kBlock), 0, s, A_rows, nbatch,
                       A_indices, A_indptr, B_indices, B_indptr, w.key, w.count,
                       reinterpret_cast<unsigned long long *>(w.summary + 1), (unsigned long long)token,
                       map ? reinterpret_cast<uint64_t *>(map->dest) : (uint64_t *)nullptr,
                       map ? map->bstart : (int32_t *)nullptr);
    NM_LAUNCH_CHECK("symbolic_front_kernel");
    // The row pointer from the counts: their sums by tile, then the pass that writes it.
    auto row_pointer = [&](const int32_t *bins, volatile int64_t *landing) -> int {
        hipLaunchKernelGGL(count_tile_sums_kernel, dim3((unsigned)tiles), dim3(nm::kScanBlock), 0, s, w.count,
                           A_rows + 1, w.scan);
        NM_LAUNCH_CHECK("count_tile_sums_kernel");
        const bool scanned = tiles > kInlineTiles;
        if (scanned) {
            hipLaunchKernelGGL(nm::scan_sums_kernel, dim3(1), dim3(1024), 0, s, w.scan, tiles);
            NM_LAUNCH_CHECK("scan_sums_kernel");
        }
        hipLaunchKernelGGL(row_pointer_kernel, dim3((unsigned)tiles), dim3(nm::kScanBlock), 0, s, w.count, A_rows + 1,
                           w.scan, scanned ? 1 : 0, C_indptr, bins, w.summary, token, landing, ticket);
        NM_LAUNCH_CHECK("row_pointer_kernel");
        return NM_OK;
    };
    // With a landing place in pinned host memory the row pointer is made at once, as if the first
    // kernel had taken every row (it has, for a product of stencil or aggregation matrices), and its
    // first workgroup tells the host nnz(C) and whether a row was left to the hash path.  If none was,
    // that was the symbolic phase: the binning and the nine launches of the hash path, which would
    // find nothing to do, are left out, and nm_spgemm_symbolic_result finds its answer landed (the
    // workspace's address in the landing place's fourth word says so).  Otherwise the pass was for
    // nothing (30 us against the milliseconds of a hash path) and is made again below.
    if (both) {
        both[3] = 0;
        if (int rc = row_pointer(nullptr, both)) return rc;
        bool arrived = false;
        for (int spin = 0; spin < (1 << 22) && !arrived; ++spin) arrived = both[2] == ticket;
        if (!arrived) {
            NM_HIP_TRY(hipStreamSynchronize(s));
            NM_REQUIRE(both[2] == ticket, "the count of hash-path rows did not arrive");
        }
        if (both[1] == 0) {
            both[3] = (int64_t)reinterpret_cast<intptr_t>(workspace);
            return NM_OK;
        }
    }
    {
    if (int rc = bin_rows(A_rows, RowKeys{w.key, nullptr}, kSymLimit, w, s)) return rc;

    hipLaunchKernelGGL((symbolic_hash_kernel<kGroup0, kSymTable0>), dim3(kPersistGrid), dim3(kBlock), 0, s, 0, w.bins,
                       w.perm, A_indices, A_indptr, B_indices, B_indptr, w.count);
    hipLaunchKernelGGL((symbolic_hash_kernel<kGroup1, kSymTable1>), dim3(kPersistGrid), dim3(kBlock), 0, s, 1, w.bins,
                       w.perm, A_indices, A_indptr, B_indices, B_indptr, w.count);
    hipLaunchKernelGGL((symbolic_hash_kernel<kGroup2, kSymTable2>), dim3(kPersistGrid), dim3(kBlock), 0, s, 2, w.bins,
                       w.perm, A_indices, A_indptr, B_indices, B_indptr, w.count);
    NM_LAUNCH_CHECK("symbolic_hash_kernel");
    auto sets = [&](auto shape, int bin, unsigned grid) -> int {
        using S = decltype(shape);
        auto k = symbolic_row_kernel<S>;
        if (S::lds > 64 * 1024)
            NM_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds));
        hipLaunchKernelGGL(k, dim3(grid), dim3(S::TPB), S::lds, s, bin, w.bins, w.perm, A_indices, A_indptr,
                           B_indices, B_indptr, w.count, B_cols, w.mark, spill_groups(B_cols));
        NM_LAUNCH_CHECK("symbolic_row_kernel");
        return NM_OK;
    };
    if (int rc = sets(SetShape3{}, 3, kPersistGrid)) return rc;
    if (int rc = sets(SetShape4{}, 4, kPersistGrid)) return rc;
    if (int rc = sets(SetShape5{}, 5, kPersistGrid)) return rc;
    if (int rc = sets(SetShape6{}, 6, 1024)) return rc;
    if (int rc = sets(SetShape7{}, 7, 512)) return rc;
    }
    return row_pointer(w.bins, nullptr);
}

}  // namespace

extern "C" int nm_spgemm_symbolic(int64_t A_rows, int64_t A_cols, int64_t B_cols, const int64_t *A_indices,
                                  const int64_t *A_indptr, const int64_t *B_indices, const int64_t *B_indptr,
                                  int64_t *C_indptr, void *workspace, size_t workspace_bytes,
                                  void *host_landing, nm_stream stream) {
    return symbolic_phase(A_rows, A_cols, B_cols, A_indices, A_indptr, B_indices, B_indptr, C_indptr, workspace,
                          workspace_bytes, host_landing, nullptr, stream);
}

extern "C" int nm_spgemm_symbolic_mapped(int64_t A_rows, int64_t A_cols, int64_t B_cols, int64_t A_nnz,
                                         int64_t B_nnz, const int64_t *A_indices, const int64_t *A_indptr,
                                         const int64_t *B_indices, const int64_t *B_indptr, int64_t *C_indptr,
                                         void *workspace, size_t workspace_bytes, void *plan_mem,
                                         size_t plan_bytes, void *host_landing, nm_stream stream) {
    NM_REQUIRE(A_nnz >= 0 && B_nnz >= 0 && plan_mem, "bad arguments");
    NM_REQUIRE(A_nnz < ((int64_t)1 << 31) && B_nnz < ((int64_t)1 << 31), "the plan keeps positions in 31 bits");
    const size_t need = nm::pplan_layout(A_nnz, nullptr, nullptr);
    if (plan_bytes < need) return nm::fail(NM_ERR_WORKSPACE, "plan of %zu bytes, %zu needed", plan_bytes, need);
    nm::PPlan map;
    nm::pplan_layout(A_nnz, plan_mem, &map);
    return symbolic_phase(A_rows, A_cols, B_cols, A_indices, A_indptr, B_indices, B_indptr, C_indptr, workspace,
                          workspace_bytes, host_landing, &map, stream);
}

extern "C" int nm_spgemm_symbolic_result(int64_t A_rows, int64_t B_cols, const void *workspace,
                                         size_t workspace_bytes, int64_t *nnz_C, int64_t *hash_rows,
                                         void *host_landing, nm_stream stream) {
    if (int rc = check_common(A_rows, B_cols)) return rc;
    NM_REQUIRE(workspace && nnz_C && hash_rows, "null pointer argument");
    Work w;
    const size_t need = work_layout(A_rows, B_cols, const_cast<void *>(workspace), &w);
    if (workspace_bytes < need)
        return nm::fail(NM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, need);
    *nnz_C = 0;
    *hash_rows = 0;
    if (A_rows == 0) return NM_OK;
    hipStream_t s = nm::as_stream(stream);
    if (!host_landing) {
        // no landing place from the caller: an ordinary copy and a wait for the stream
        int64_t both[2] = {0, 0};
        NM_HIP_TRY(hipMemcpyAsync(both, w.summary, sizeof(both), hipMemcpyDeviceToHost, s));
        NM_HIP_TRY(hipStreamSynchronize(s));
        *nnz_C = both[0];
        *hash_rows = both[1];
        return NM_OK;
    }
    // The two numbers are written straight into the caller's pinned host memory by a one-lane
    // kernel, followed by a ticket the host polls for: waking up from hipStreamSynchronize, or a
    // copy-engine transfer of 16 bytes, takes ~30 us, several times what the kernels of a small
    // product take together.  The ticket is one more than the last one this landing place saw.
    volatile int64_t *both = (volatile int64_t *)host_landing;
    if (both[3] != 0 && both[3] == (int64_t)reinterpret_cast<intptr_t>(workspace)) {
        // nm_spgemm_symbolic on this workspace has had the numbers dropped here already
        both[3] = 0;
        *nnz_C = both[0];
        *hash_rows = both[1];
        return NM_OK;
    }
    const int64_t ticket = both[2] + 1;
    hipLaunchKernelGGL(summary_out_kernel, dim3(1), dim3(64), 0, s, w.summary, both, ticket);
    NM_LAUNCH_CHECK("summary_out_kernel");
    bool arrived = false;
    for (int spin = 0; spin < (1 << 22) && !arrived; ++spin) arrived = both[2] == ticket;
    if (!arrived) {   // a long queue ahead of the kernel, or memory the host sees late: wait the ordinary way
        NM_HIP_TRY(hipStreamSynchronize(s));
        NM_REQUIRE(both[2] == ticket, "the symbolic phase's result did not arrive");
    }
    *nnz_C = both[0];
    *hash_rows = both[1];
    return NM_OK;
}

extern "C" int nm_spgemm_numeric(nm_dtype dt, int64_t A_rows, int64_t A_cols, int64_t B_cols,
                                 const void *A_data, const int64_t *A_indices, const int64_t *A_indptr,
                                 const void *B_data, const int64_t *B_indices, const int64_t *B_indptr,
                                 const int64_t *C_indptr, int64_t *C_indices, void *C_data, void *workspace,
                                 size_t workspace_bytes, int64_t hash_rows, nm_stream stream) {
    if (int rc = check_common(A_rows, B_cols)) return rc;
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(A_indptr && B_indptr && C_indptr && workspace, "null pointer argument");
    Work w;
    const size_t need = work_layout(A_rows, B_cols, workspace, &w);
    if (workspace_bytes < need)
        return nm::fail(NM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, need);
    if (A_rows == 0) return NM_OK;
    hipStream_t s = nm::as_stream(stream);
    // hash_rows == 0 (from nm_spgemm_symbolic_result): every row is one of the merge path's and
    // the binning and the hash launches, a dozen launches that would find nothing to do, are left out
    const bool hashed = hash_rows != 0;
    if (hashed) {
        int32_t limit[kBins - 1];
        for (int q = 0; q < kBins - 2; ++q) limit[q] = kNumLimit[q];
        limit[kBins - 2] = dt == NM_F32 ? kRowLimitMost32 : kRowLimitMost64;
        if (int rc = bin_rows(A_rows, RowKeys{w.key, w.count}, limit, w, s)) return rc;
    }
    const int64_t nbatch = nm::xcd_padded(nm::ceil_div(A_rows, kMergeRows));
    // (every row on the hash path: the merge kernel would look at each row's key and leave)
    if (hash_rows == A_rows) {
    } else if (dt == NM_F32)
        hipLaunchKernelGGL(numeric_front_kernel<float>, dim3((unsigned)nbatch), dim3(kBlock), 0, s, A_rows, nbatch,
                           w.key, (const float *)A_data, A_indices, A_indptr, (const float *)B_data, B_indices,
                           B_indptr, C_indptr, C_indices, (float *)C_data);
    else
        hipLaunchKernelGGL(numeric_front_kernel<double>, dim3((unsigned)nbatch), dim3(kBlock), 0, s, A_rows, nbatch,
                           w.key, (const double *)A_data, A_indices, A_indptr, (const double *)B_data, B_indices,
                           B_indptr, C_indptr, C_indices, (double *)C_data);
    NM_LAUNCH_CHECK("numeric_front_kernel");
    if (!hashed) return NM_OK;
    if (dt == NM_F32)
        return launch_numeric<float>(w, B_cols, A_data, A_indices, A_indptr, B_data, B_indices, B_indptr,
                                     C_indptr, C_indices, C_data, s);
    return launch_numeric<double>(w, B_cols, A_data, A_indices, A_indptr, B_data, B_indices, B_indptr, C_indptr,
                                  C_indices, C_data, s);
}

extern "C" int nm_spgemm_numeric_mapped(nm_dtype dt, int64_t A_rows, int64_t A_cols, int64_t B_cols, int64_t A_nnz,
                                        int64_t C_nnz, const void *A_data, const int64_t *A_indices,
                                        const int64_t *A_indptr, const void *B_data, const int64_t *B_indices,
                                        const int64_t *B_indptr, const int64_t *C_indptr, int64_t *C_indices,
                                        void *C_data, void *workspace, size_t workspace_bytes, int64_t hash_rows,
                                        void *plan_mem, size_t plan_bytes, int keep_plan, nm_stream stream) {
    // rows on the hash path (or an unknown number of them), or positions beyond 31 bits: the map
    // the symbolic phase left is incomplete or unusable, the ordinary numeric phase runs
    if (hash_rows != 0 || !plan_mem || A_nnz <= 0 || C_nnz <= 0 || C_nnz >= ((int64_t)1 << 31))
        return nm_spgemm_numeric(dt, A_rows, A_cols, B_cols, A_data, A_indices, A_indptr, B_data, B_indices, B_indptr,
                                 C_indptr, C_indices, C_data, workspace, workspace_bytes, hash_rows, stream);
    if (int rc = check_common(A_rows, B_cols)) return rc;
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(A_data && A_indptr && B_data && B_indices && C_indptr && C_indices && C_data, "null pointer argument");
    const size_t need = nm::pplan_layout(A_nnz, nullptr, nullptr);
    if (plan_bytes < need) return nm::fail(NM_ERR_WORKSPACE, "plan of %zu bytes, %zu needed", plan_bytes, need);
    nm::PPlan map;
    nm::pplan_layout(A_nnz, plan_mem, &map);
    return nm::spgemm_numeric_on_map(dt, A_rows, A_nnz, A_data, A_indptr, B_data, B_indices, map, C_indptr, C_indices,
                                     C_data, keep_plan != 0, nm::as_stream(stream));
}

extern "C" int nm_spgemm_backward(nm_dtype dt, int64_t A_rows, int64_t A_nnz, int64_t B_nnz, const void *gC,
                                  const int64_t *C_indices, const int64_t *C_indptr, const void *A_data,
                                  const int64_t *A_indices, const int64_t *A_indptr, const void *B_data,
                                  const int64_t *B_indices, const int64_t *B_indptr, void *grad_A,
                                  void *grad_B, nm_stream stream) {
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(A_rows >= 0 && A_nnz >= 0 && B_nnz >= 0, "negative size");
    hipStream_t s = nm::as_stream(stream);
    if (grad_B) {
        int rc = dt == NM_F32 ? nm::fill_async((float *)grad_B, B_nnz, 0.0f, s)
                              : nm::fill_async((double *)grad_B, B_nnz, 0.0, s);
        if (rc) return rc;
    }
    if (A_nnz == 0 || A_rows == 0 || (!grad_A && !grad_B)) return NM_OK;
    NM_REQUIRE(C_indptr && A_indices && A_indptr && B_indptr && A_data, "null pointer argument");
    int64_t grid = nm::ceil_div(A_rows, kBlock / kBwdG);
    if (grid > 1 << 20) grid = 1 << 20;
    if (dt == NM_F32)
        hipLaunchKernelGGL(spgemm_bwd_kernel<float>, dim3((unsigned)grid), dim3(kBlock), 0, s, A_rows,
                           (const float *)gC, C_indices, C_indptr, (const float *)A_data, A_indices, A_indptr,
                           (const float *)B_data, B_indices, B_indptr, (float *)grad_A, (float *)grad_B);
    else
        hipLaunchKernelGGL(spgemm_bwd_kernel<double>, dim3((unsigned)grid), dim3(kBlock), 0, s, A_rows,
                           (const double *)gC, C_indices, C_indptr, (const double *)A_data, A_indices, A_indptr,
                           (const double *)B_data, B_indices, B_indptr, (double *)grad_A, (double *)grad_B);
    NM_LAUNCH_CHECK("spgemm_bwd_kernel");
    // Two launches whether or not there are long rows, which the host does not know: so few workgroups
    // that finding none is short (a launch of 1024-thread workgroups that take a CU's LDS each: 17 us with
    // 2800 of them, 4 with 256), so many that long rows find the chip (150 000-row graph: both gradients
    // 497 us with 1024 workgroups for the longest rows, 546 with 512; 20 000 rows of 600 entries: 685 us
    // with 4096 of the others, 732 with 2500, 886 with 512).  Both gradients of 5-point 300^2 A A, fp32: 36
    // us (61 with four launches, one for each shape, of 2800 to 22500 workgroups), 7-point 20^3, fp64: 18 (35).
    auto groups = [&](int64_t rows_each, int64_t least, int64_t most) {
        const int64_t n = A_rows / rows_each;
        return n < least ? least : n > most ? most : n;
    };
    auto longer = [&](auto value) -> int {
        using T = decltype(value);
        BackArgs<T> g{A_rows, 8, (const T *)gC, C_indices, C_indptr, (const T *)A_data, A_indices, A_indptr,
                      (const T *)B_data, B_indices, B_indptr, (T *)grad_A, (T *)grad_B};
        auto launch = [&](auto kernel, int threads, size_t lds, int64_t groups) -> int {
            for (g.piece = 8; g.piece > 1 && A_rows < groups * g.piece;) g.piece /= 2;
            const int64_t most = nm::ceil_div(A_rows, g.piece);
            if (lds > 64 * 1024)
                NM_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            hipLaunchKernelGGL(kernel, dim3((unsigned)(most < groups ? most : groups)), dim3(threads), lds, s, g);
            return NM_OK;
        };
        if (int rc = launch(spgemm_bwd_mid_kernel<T>, kBackMid, kBackMidLds<T>, groups(4, 512, 4096))) return rc;
        NM_LAUNCH_CHECK("spgemm_bwd_mid_kernel");
        if (int rc = launch(spgemm_bwd_long_kernel<T>, 1024, BackLongRow<T>::lds, groups(128, 256, 1024))) return rc;
        NM_LAUNCH_CHECK("spgemm_bwd_long_kernel");
        return NM_OK;
    };
    return dt == NM_F32 ? longer(0.0f) : longer(0.0);
}
