// Sparse LU without pivoting: symbolic phase (pattern of M = L + U with fill).
// Stands in for the first half of splu (cpp/sparse_csr_cpu.cpp:777-954).
//
// The pattern of row i is found, as in the reference, by the fill2 traversal of
// Rose and Tarjan: stored neighbours of i are kept; then the pivots t < i that
// have been reached are expanded in ascending order by a breadth-first walk that
// continues through vertices <= t and keeps (without expanding) every newly
// reached vertex > t.  Rows are independent, so one wavefront takes one row at a
// time (rows w, w + W, w + 2W, ... for wavefront w of W): the queue is popped
// serially, the edges of the popped vertex are handled by the lanes, and the scan
// for the next pivot and the emission of the kept columns go 64 vertices at a time.
// Each wavefront owns three arrays of `rows` entries in the caller's scratch
// (visit stamps, queue, keep flags); they are accessed with volatile operations
// because lanes of the wavefront communicate through them.
//
// The work per row is that of the serial algorithm (the reference spends O(rows)
// per row as well): this is meant for the moderate sizes a direct solve is used at.
//
// Numeric phase (cpp/sparse_csr_cpu.cpp:956-1000): left-looking column LU on the rows of
// M^T (= columns of M).  For the entries (i, k), i < k, of column k in ascending i, every
// later entry (j, k) takes  M_jk -= M_ji * M_ik  where column i stores row j; then the
// entries below the diagonal are divided by it.  Per entry the operations come in the
// serial order, so the factors equal the reference's bit for bit.
// Column k needs the finished columns i of its entries above the diagonal, and nothing
// else: workgroups take batches of consecutive columns in ascending order from a ticket
// counter, one column per wavefront, keep the columns in LDS, and before using column i wait
// for its flag -- a flag and values in LDS when column i belongs to the same batch, in global
// memory otherwise.  A wavefront only ever waits for a column with a smaller number, which a
// running wavefront holds, so the grid always makes progress whatever part of it is resident;
// a bounded number of polls backs that up, after which every wavefront leaves and the call
// reports an error.  Early pivots of a column
// overlap with the tail of the columns before it, which is where a banded factor, whose
// columns form one long dependency chain, gets its parallelism from.  Factors that stay within a
// narrow band have a kernel of their own (lu_band_kernel, below): one workgroup, whose wavefronts wait
// for each other in LDS.  Those waits have no bound: the wavefronts of a workgroup run or none does.
#include "nm_common.hpp"
#include "nm_scan.hpp"

namespace {

constexpr int kBlock = 256;
constexpr int kLuWaves = 4096;   // wavefronts that share the rows

struct LuScratch {
    int32_t *stamp, *queue;   // [waves][rows]
    uint8_t *keep;            // [waves][rows]
    int64_t *scan;            // scan scratch for the row pointer
};

inline size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

// Wavefronts that share the rows: at most kLuWaves, at most one per row, and few enough that
// their scratch (9 bytes per row each) stays within kLuScratchBytes.
constexpr int64_t kLuScratchBytes = int64_t(1) << 30;
inline int lu_waves(int64_t rows) {
    if (rows < 1) return 1;
    int64_t w = rows < kLuWaves ? rows : kLuWaves;
    const int64_t fit = kLuScratchBytes / (9 * rows);
    // (a launch is whole workgroups of four wavefronts: fewer wavefronts than rows must be a
    //  multiple of four, or the last workgroup's extra wavefronts would take rows without scratch)
    if (w > fit) w = (fit < 64 ? 64 : fit) / 4 * 4;
    return (int)w;
}

size_t lu_layout(int64_t rows, void *base, LuScratch *S) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void *q = base ? static_cast<char *>(base) + off : nullptr;
        off += align_up(bytes);
        return q;
    };
    const size_t w = (size_t)lu_waves(rows), n = (size_t)(rows > 0 ? rows : 1);
    LuScratch s;
    s.stamp = (int32_t *)take(w * n * 4);
    s.queue = (int32_t *)take(w * n * 4);
    s.keep = (uint8_t *)take(w * n);
    s.scan = (int64_t *)take(nm::scan_scratch_bytes(rows + 1));
    if (S) *S = s;
    return off;
}

__global__ void lu_init_kernel(int64_t total, int32_t *__restrict__ stamp, uint8_t *__restrict__ keep) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        stamp[i] = -1;
        keep[i] = 0;
    }
}

// FILL == false: As_indptr[i] = number of kept columns of row i.
// FILL == true : As_indices / As_data of row i are written at As_indptr[i]: the value of A where A
//                stores the column, 0 at the fill (cpp/sparse_csr_cpu.cpp:908-954).
template <typename T, bool FILL>
__global__ __launch_bounds__(kBlock) void lu_rows_kernel(int64_t rows, const T *__restrict__ A_data,
                                                         const int64_t *__restrict__ A_indices,
                                                         const int64_t *__restrict__ A_indptr,
                                                         int64_t *__restrict__ As_indptr,
                                                         int64_t *__restrict__ As_indices, T *__restrict__ As_data,
                                                         int32_t *stamp_all, int32_t *queue_all, uint8_t *keep_all) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    volatile int32_t *stamp = stamp_all + wave * rows;
    volatile int32_t *queue = queue_all + wave * rows;
    volatile uint8_t *keep = keep_all + wave * rows;
    const unsigned long long lower_lanes = (1ull << lane) - 1ull;

    for (int64_t i = wave; i < rows; i += nwaves) {
        const int32_t mark = (int32_t)i;   // rows come in ascending order per wavefront: a stamp names one row
        if (lane == 0) stamp[i] = mark;
        for (int64_t k = A_indptr[i] + lane; k < A_indptr[i + 1]; k += 64) {
            const int64_t u = A_indices[k];
            if (u < 0 || u >= rows) continue;   // not a column of a square matrix: ignored rather than written
            stamp[u] = mark;
            keep[u] = 1;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        // pivots t < i that have been reached, in ascending order; a walk may reach later pivots
        for (int64_t t0 = 0; t0 < i; t0 += 64) {
            int64_t done = t0 - 1;
            for (;;) {
                const int64_t tc = t0 + lane;
                const bool cand = tc < i && tc > done && stamp[tc] == mark;
                const unsigned long long m = __ballot(cand);
                if (m == 0) break;
                const int64_t t = t0 + (__ffsll((long long)m) - 1);
                done = t;
                // breadth-first walk from t through vertices <= t
                int64_t head = 0, tail = 1;
                if (lane == 0) queue[0] = (int32_t)t;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                while (head < tail) {
                    const int64_t u = queue[head++];
                    const int64_t kb = A_indptr[u], ke = A_indptr[u + 1];
                    for (int64_t k0 = kb; k0 < ke; k0 += 64) {
                        const int64_t k = k0 + lane;
                        int64_t w = -1;
                        bool fresh = false;
                        if (k < ke) {
                            w = A_indices[k];
                            fresh = w >= 0 && w < rows && stamp[w] != mark;   // columns of a row are distinct: no two lanes share w
                        }
                        if (fresh) {
                            stamp[w] = mark;
                            if (w > t) keep[w] = 1;
                        }
                        const bool push = fresh && w <= t;
                        const unsigned long long pm = __ballot(push);
                        if (push) queue[tail + __popcll(pm & lower_lanes)] = (int32_t)w;
                        tail += __popcll(pm);
                        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    }
                }
            }
        }
        // kept columns in ascending order
        int64_t out = FILL ? As_indptr[i] : 0;
        const int64_t ab = A_indptr[i], ae = A_indptr[i + 1];
        for (int64_t j0 = 0; j0 < rows; j0 += 64) {
            const int64_t j = j0 + lane;
            const bool kept = j < rows && keep[j] != 0;
            const unsigned long long m = __ballot(kept);
            if (kept) {
                keep[j] = 0;
                if (FILL) {
                    const int64_t pos = out + __popcll(m & lower_lanes);
                    int64_t lo = ab, hi = ae;   // A's value at column j, if stored
                    while (lo < hi) {
                        const int64_t mid = (lo + hi) >> 1;
                        if (A_indices[mid] < j) lo = mid + 1; else hi = mid;
                    }
                    As_indices[pos] = j;
                    As_data[pos] = (lo < ae && A_indices[lo] == j) ? A_data[lo] : T(0);
                }
            }
            out += __popcll(m);
        }
        if (!FILL && lane == 0) As_indptr[i] = out;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
}

// Values on a known filled pattern: one wavefront per row, a lane per entry of the row.
template <typename T>
__global__ __launch_bounds__(kBlock) void lu_values_kernel(int64_t rows, const T *__restrict__ A_data,
                                                           const int64_t *__restrict__ A_indices,
                                                           const int64_t *__restrict__ A_indptr,
                                                           const int64_t *__restrict__ As_indptr,
                                                           const int64_t *__restrict__ As_indices,
                                                           T *__restrict__ As_data) {
    const int lane = threadIdx.x & 63;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t i = (int64_t)blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
         i < rows; i += nwaves) {
        const int64_t ab = A_indptr[i], ae = A_indptr[i + 1], pe = As_indptr[i + 1];
        for (int64_t p = As_indptr[i] + lane; p < pe; p += 64) {
            const int64_t j = As_indices[p];
            int64_t lo = ab, hi = ae;
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                if (A_indices[mid] < j) lo = mid + 1; else hi = mid;
            }
            As_data[p] = (lo < ae && A_indices[lo] == j) ? A_data[lo] : T(0);
        }
    }
}

#ifndef NM_LU_WAVES
#define NM_LU_WAVES 8
#endif
constexpr int kLuCap = 1024;              // entries of a column kept in LDS, per wavefront
constexpr int kLuWavesPerBlock = NM_LU_WAVES;   // columns of a batch = wavefronts of a workgroup of the numeric phase
constexpr int kLuFlowBlock = kLuWavesPerBlock * 64;
constexpr int64_t kLuSpinLimit = 1 << 24;  // polls of one dependency flag, without any column finishing, before giving up

struct LuFlow {
    int64_t *below;  // [cols] position of the column's first entry below the diagonal
    int32_t *done;   // [cols] 0 = pending, 1 = the column holds its final values
    int32_t *ctl;    // [0] next ticket, [1] failure, [2] columns finished,
                     // [4] reach above the diagonal, [5] below it, [6] columns that do not name their predecessor
};

size_t flow_layout(int64_t cols, void *base, LuFlow *F) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void *q = base ? static_cast<char *>(base) + off : nullptr;
        off += align_up(bytes);
        return q;
    };
    LuFlow f;
    f.ctl = (int32_t *)take(64);
    f.done = (int32_t *)take((size_t)(cols > 0 ? cols : 1) * 4);
    f.below = (int64_t *)take((size_t)(cols > 0 ? cols : 1) * 8);
    if (F) *F = f;
    return off;
}

// The column of a wavefront: in LDS (rows as 32-bit, values) or, when it is too long, in
// place in global memory, where the lanes hand values on through volatile accesses.
template <typename T, bool IN_LDS>
struct OwnColumn {
    int32_t *s_rows;
    T *s_vals;
    const int64_t *g_rows;
    volatile T *g_vals;
    __device__ __forceinline__ int64_t row(int64_t e) const { return IN_LDS ? (int64_t)s_rows[e] : g_rows[e]; }
    __device__ __forceinline__ T val(int64_t e) const { return IN_LDS ? s_vals[e] : g_vals[e]; }
    __device__ __forceinline__ void set(int64_t e, T v) const {
        if (IN_LDS) s_vals[e] = v; else g_vals[e] = v;
    }
};

// below[k] = position of the first entry of column k with a row index > k; no column is done.  Also what the choice of
// the numeric kernel depends on: ctl[4] / ctl[5] = entries the widest column reaches above / below its
// diagonal, ctl[6] = columns that do not name the column before them, ctl[9] = whether a value is -0.
template <typename T>
__global__ __launch_bounds__(kBlock) void lu_below_kernel(int64_t cols, const int64_t *__restrict__ indices,
                                                          const int64_t *__restrict__ indptr, const T *__restrict__ values,
                                                          int64_t *__restrict__ below, int32_t *__restrict__ done, int32_t *ctl) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nnz = indptr[cols];
    bool negative = false;
    for (int64_t e = first; e < nnz; e += 8 * stride) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = values[e + u * stride < nnz ? e + u * stride : nnz - 1];
#pragma unroll
        for (int u = 0; u < 8; ++u) negative = negative || (v[u] == T(0) && __builtin_signbit(v[u]));
    }
    if (__any(negative) && (threadIdx.x & 63) == 0) __hip_atomic_store(ctl + 9, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int32_t up = 0, down = 0, breaks = 0;
    for (int64_t k = first; k < cols; k += stride) {
        const int64_t pb = indptr[k], pe = indptr[k + 1];
        int64_t lo = pb, hi = pe;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (indices[mid] <= k) lo = mid + 1; else hi = mid;
        }
        below[k] = lo;
        done[k] = 0;
        if (pe > pb) {
            const int64_t first = indices[pb], last = indices[pe - 1];
            if (first < k) up = max(up, (int32_t)(k - first));
            if (last > k) down = max(down, (int32_t)(last - k));
        }
        int64_t q = lo - 1;                        // last entry on or above the diagonal
        if (q >= pb && indices[q] == k) --q;
        if (k > 0 && !(q >= pb && indices[q] == k - 1)) ++breaks;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        up = max(up, __shfl_xor(up, off, nm::kWave));
        down = max(down, __shfl_xor(down, off, nm::kWave));
        breaks += __shfl_xor(breaks, off, nm::kWave);
    }
    if ((threadIdx.x & 63) == 0) {
        if (up) atomicMax(ctl + 4, up);
        if (down) atomicMax(ctl + 5, down);
        if (breaks) atomicAdd(ctl + 6, breaks);
    }
}

// Returns false when a dependency did not arrive within the poll limit (or another wavefront failed).
// Everything about a pivot that the structure alone decides -- which entries of column i lie below
// its diagonal and where their rows sit in this column -- is looked up before the wait for column i,
// so that what follows the arrival of the flag is one load, one multiply and one subtraction.
// The columns of one batch [base, base + kLuWavesPerBlock) are worked on by the wavefronts of one
// workgroup: a column of the batch that sits in LDS is read there, behind an LDS flag, by the
// later columns of the batch, which spares them the round trip through global memory that the
// flag and the values of a column of another workgroup cost.
template <typename T>
struct LuBatch {
    int64_t base;                 // first column of the batch
    const int64_t *pb;            // [kLuWavesPerBlock] LDS: start of each column in the CSR arrays
    T (*vals)[kLuCap];            // LDS values of the batch's columns
    volatile int32_t *ready;      // [kLuWavesPerBlock] LDS: 0 pending, 1 final values in LDS, 2 final values in global memory only
};

// RESUME: the rows before `base` of the column are final (lu_band_kernel wrote them), so that pivots there only update
// the rows from `base` on.
template <typename T, bool IN_LDS, bool RESUME>
__device__ bool lu_column(int64_t base, int64_t k, int64_t pb, int64_t len, const OwnColumn<T, IN_LDS> &own,
                          const LuBatch<T> &batch,
                          const int64_t *__restrict__ indices, const int64_t *__restrict__ indptr,
                          const int64_t *__restrict__ below_of, T *values, int32_t *done, int32_t *ctl,
                          int64_t spin_limit, int lane) {
    if (IN_LDS) {
        for (int64_t e = lane; e < len; e += 64) {
            own.s_rows[e] = (int32_t)indices[pb + e];
            own.s_vals[e] = values[pb + e];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // position in this column of row j, searched among the entries after e; -1 when not stored
    auto find = [&](int64_t e, int64_t j) {
        int64_t lo = e + 1, hi = len;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (own.row(mid) < j) lo = mid + 1; else hi = mid;
        }
        return (lo < len && own.row(lo) == j) ? lo : (int64_t)-1;
    };
    // What the structure alone says about pivot e: the column i it names, where the entries of
    // column i below its diagonal start and end, this lane's entry of them and the place of
    // that entry's row in this column.  Looked up one pivot ahead: the two dependent loads it
    // takes would otherwise stand between the arrival of a flag and the update it allows.
    struct Look {
        int64_t i, ls, ie, t_first, at_first;
    };
    auto look = [&](int64_t e) {
        Look L{-1, 0, 0, 0, -1};
        if (e >= len) return L;
        const int64_t i = own.row(e);
        if (i >= k) return L;
        L.i = i;
        L.ls = below_of[i];
        L.ie = indptr[i + 1];
        L.t_first = L.ls + lane;
        L.at_first = L.t_first < L.ie ? find(e, indices[L.t_first]) : (int64_t)-1;
        return L;
    };
    int64_t e = 0;
    Look next = look(0);
    for (; next.i >= 0; ++e) {
        const Look cur = next;
        next = look(e + 1);
        const int64_t i = cur.i, ls = cur.ls, ie = cur.ie, t_first = cur.t_first, at_first = cur.at_first;
        // The limit bounds polls WITHOUT PROGRESS: every 256 polls the wavefront looks at the failure
        // word and at the count of finished columns, and starts counting afresh when that count has
        // moved.  A wavefront that legitimately waits behind a chain of thousands of slow columns
        // is thus never cut off, while a grid in which nothing finishes any more is.
        int64_t polls = 0;
        int32_t seen_done = -1;
        auto still_hopeful = [&]() -> bool {   // false: give up
            if (++polls > spin_limit) return false;
            if ((polls & 255) == 0) {
                if (__hip_atomic_load(ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
                const int32_t now = __hip_atomic_load(ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (now != seen_done) {
                    seen_done = now;
                    polls = 0;
                }
            }
            return true;
        };
        bool in_lds = false;   // column i is one of this batch's and its final values are in LDS
        if (i >= batch.base) {
            const int wi = (int)(i - batch.base);
            int32_t state;
            while ((state = batch.ready[wi]) == 0) {
                if (!still_hopeful()) return false;
                __builtin_amdgcn_s_sleep(1);
            }
            in_lds = state == 1;
        } else {
            while (__hip_atomic_load(done + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
                if (!still_hopeful()) return false;
                __builtin_amdgcn_s_sleep(1);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");   // the value loads below stay after the flag
        const T m_ik = own.val(e);
        // entry t of the CSR arrays, which belongs to column i
        auto other = [&](int64_t t) -> T {
            if (in_lds) {
                const int wi = (int)(i - batch.base);
                return batch.vals[wi][t - batch.pb[wi]];
            }
            return __hip_atomic_load(values + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        if (at_first >= 0 && !(RESUME && own.row(at_first) < base)) {
            const T prod = other(t_first) * m_ik;
            own.set(at_first, own.val(at_first) - prod);
        }
        for (int64_t t0 = ls + 64; t0 < ie; t0 += 64) {          // columns with more than 64 entries below
            const int64_t t = t0 + lane;
            const int64_t at = t < ie ? find(e, indices[t]) : (int64_t)-1;
            if (at >= 0 && !(RESUME && own.row(at) < base)) {
                const T prod = other(t) * m_ik;
                own.set(at, own.val(at) - prod);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (e < len && own.row(e) == k) {
        const T d = own.val(e);
        for (int64_t q = e + 1 + lane; q < len; q += 64) own.set(q, own.val(q) / d);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // the later columns of the batch first: they read this one in LDS
    if (IN_LDS) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0) batch.ready[k - batch.base] = 1;
        for (int64_t q = lane; q < len; q += 64) values[pb + q] = own.s_vals[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if (lane == 0) {
        __hip_atomic_store(done + k, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        atomicAdd(ctl + 2, 1);   // columns finished so far: what a waiting wavefront watches for progress
        if (!IN_LDS) batch.ready[k - batch.base] = 2;
    }
    return true;
}

// Columns are drawn from ctl[0]; RESUME: from ctl[8], where lu_band_kernel has left some.
template <typename T, bool RESUME>
__device__ __forceinline__ void lu_flow(int64_t cols, const int64_t *__restrict__ indices, const int64_t *__restrict__ indptr,
                                        const int64_t *__restrict__ below, T *values, int32_t *done, int32_t *ctl,
                                        int64_t spin_limit) {
    // dynamic LDS: the batch's columns, values first (8-byte aligned), then rows
    extern __shared__ __align__(16) unsigned char s_columns[];
    T (*s_vals)[kLuCap] = reinterpret_cast<T (*)[kLuCap]>(s_columns);
    int32_t (*s_rows)[kLuCap] =
        reinterpret_cast<int32_t (*)[kLuCap]>(s_columns + sizeof(T) * kLuWavesPerBlock * kLuCap);
    __shared__ int64_t s_pb[kLuWavesPerBlock];
    __shared__ int32_t s_ready[kLuWavesPerBlock];
    __shared__ int32_t s_ticket, s_abort;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t resume = RESUME ? (int64_t)ctl[7] : 0;
    for (;;) {
        // one ticket per workgroup and batch of consecutive columns, one column per wavefront
        if (threadIdx.x == 0) {
            s_ticket = atomicAdd(ctl + (RESUME ? 8 : 0), kLuWavesPerBlock);
            s_abort = __hip_atomic_load(ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (threadIdx.x < kLuWavesPerBlock) s_ready[threadIdx.x] = 0;
        __syncthreads();
        const int64_t base = s_ticket;
        if (base >= cols || s_abort != 0) break;   // the same decision in every wavefront
        const int64_t k = base + w;
        if (k < cols) {
            const int64_t pb = indptr[k], len = indptr[k + 1] - pb;
            if (lane == 0) s_pb[w] = pb;
            const LuBatch<T> batch{base, s_pb, s_vals, s_ready};
            bool ok;
            if (len <= kLuCap) {
                const OwnColumn<T, true> own{s_rows[w], s_vals[w], nullptr, nullptr};
                ok = lu_column<T, true, RESUME>(resume, k, pb, len, own, batch, indices, indptr, below, values, done, ctl, spin_limit,
                                        lane);
            } else {
                const OwnColumn<T, false> own{nullptr, nullptr, indices + pb, values + pb};
                ok = lu_column<T, false, RESUME>(resume, k, pb, len, own, batch, indices, indptr, below, values, done, ctl, spin_limit,
                                         lane);
            }
            if (!ok && lane == 0) atomicExch(ctl + 1, 1);
        }
        __syncthreads();   // the batch's columns in LDS have no readers left
    }
}

template <typename T>
__global__ __launch_bounds__(kLuFlowBlock) void lu_flow_kernel(int64_t cols, const int64_t *__restrict__ indices,
                                                         const int64_t *__restrict__ indptr,
                                                         const int64_t *__restrict__ below, T *values,
                                                         int32_t *done, int32_t *ctl, int64_t spin_limit) {
    if (ctl[7] == 0) lu_flow<T, false>(cols, indices, indptr, below, values, done, ctl, spin_limit);
    else lu_flow<T, true>(cols, indices, indptr, below, values, done, ctl, spin_limit);
}

// ---- banded factors --------------------------------------------------------------
//
// A factor whose entries stay near the diagonal is ONE chain of columns: column k + 1 needs column k,
// and lu_flow_kernel pays a hand-over between wavefronts, workgroups or compute units (1.4 us) for
// every link of it whatever the width of the band.  Here one workgroup keeps the window of the matrix that
// is being worked on in LDS and eliminates it panel by panel of eight columns.  Every entry receives the
// same products in the same ascending order of pivots, so the factors are the serial ones bit for
// bit.  The wavefronts have tasks of their own and wait for counts in LDS, never at a barrier:
//   * wavefronts 0 and 1 factor the panels in turn, rows in lanes, columns in registers: while one divides and
//     updates inside its panel, the other applies the panel before that one to the next and then each pivot as it comes
//     out;
//   * wavefronts 2 and 3 (lanes are columns) finish the panel's eight rows to the right of it, pivot by pivot;
//   * six wavefronts apply the panel to the rest of the window, eight columns of all its rows at a time;
//   * wavefronts 14 and 15 bring columns in, 8 and 9 rows, as far ahead as the rings allow, and wavefront 4 writes
//     what is finished.
// What bounds it: the chain inside a panel, a division, the broadcast of the row and the update of the next column a
// pivot (380 cycles), and the last pivot's way to the panel that waits for it (1700 cycles a panel of eight); at a
// reach of 64 and more the update of the window takes over.  us for 4096 columns with everything around it (a kernel
// that kept the window in registers and handed every column round by itself took the figure in brackets):
//   reach      1            8            28           56           64           76           92
//   fp64  1116 (1166)  1120 (1169)  1121 (1164)  1170 (2070)  1328 (2491)  2191 (2559)  2501 (2942)
//   fp32  1052 (1162)  1055 (1160)  1052 (1178)  1090 (1780)  1182 (2187)  1490 (2231)  1918 (2375)
// with a -0 among the inputs (SIGNED, below; ending the launch there and going on column by column took 3100 at a
// reach of 1, 5600 at 64, 9300 at 92)
//   fp64  1508         1508         1515         1663         1866         3589         4192
//   fp32  1390         1382         1371         1401         1482         2198         2422
// A 100 x 100 grid in fp32, which did not fit the registers, takes 4.9 ms instead of 25.
// Entries that the pattern does not have are zeros when they are handed on, whatever a product has left in
// their places, and a zero takes no part in a sum of finite numbers (no input is -0, a difference is
// -0 only where one operand was).  Where an input IS -0 (a masked or negated matrix with explicit zeros), it must keep its
// sign until a product of two stored entries comes: there such entries are handed on as NaN, and a product that is NaN
// counts as +0, which leaves every operand as it is (SIGNED).  An infinity or a NaN among the factors ends
// the launch before they are written or used further: lu_flow_kernel goes on at that panel.
#define NM_INLINE __attribute__((always_inline))   // (lambdas over register arrays)
constexpr int kBandWaves = 16;
constexpr int kBandTrailing = 6;     // wavefronts of the update
constexpr int kPanel = 8;
static_assert(kPanel == kLuWavesPerBlock, "lu_flow_kernel goes on at a batch of its own");
constexpr size_t kBandLds = 160 * 1024;
// More breaks in the chain (columns that do not name their predecessor) than this and the matrix may
// be made of three independent blocks or more, which lu_flow_kernel works on side by side.
constexpr int kBandMaxBreaks = 1;

enum BandCount : int {
    kPivots,                     // pivots whose multipliers are there
    kRows0, kRows1,              // rows of U that are there, of the first 64 columns right of the panel and of the rest
    kColumns0, kColumns1, kIn0, kIn1,   // panels whose new columns / rows are in the window (kLoaded: all four)
    kWritten,                    // panels written
    kGoodPanel0, kGoodPanel1,    // panels found finite, by the wavefront that factors them
    kGoodRows0, kGoodRows1,
    kStop,                       // somebody found one that is not
    kTrailing0 = 16,             // per wavefront: panels applied to the rest of the window
    kBandCounts = kTrailing0 + kBandTrailing
};
constexpr int32_t kBandNever = 0x40000000;
constexpr int kLoaded = kColumns0, kLoaders = 4;

template <typename T> struct Band {
    int32_t n, panels, blb, bub;   // columns; blocks of eight rows below, columns right of a panel's own
    int32_t rb, cb, pitch;         // blocks of the window (rings), entries from column to column (odd)
    int32_t slack, kept;           // panels that the rings hold beyond the window; panels whose multipliers and rows are kept
    T *win, *F, *U;                // F, U: the kept panels' multipliers [pivot][row - panel's first], rows [pivot][column - panel's end]
    int32_t fr, fp, uc;            // rows of a panel, the same rounded up to whole registers, columns right of it
    uint8_t *has;                  // [block of rows][column]: which of the eight are stored
    int64_t *base;                 // by column of the window: where it starts in the arrays, its length, entries brought in, written
    int32_t *len, *in, *out;
    int32_t *count;
    const int64_t *indices;
    T *values;
    const int64_t *indptr;
    __device__ __forceinline__ T *column(int32_t slot) const { return win + slot * pitch; }
    __device__ __forceinline__ T *multipliers(int32_t K) const { return F + (K & (kept - 1)) * (kPanel * fp); }
    __device__ __forceinline__ T *rows(int32_t K) const { return U + (K & (kept - 1)) * (kPanel * uc); }
};
// Waits until the count of every lane's number is at least the lane's `least`; false: the launch ends.
template <bool SLEEP> __device__ __forceinline__ bool band_wait(int32_t *count, int32_t least) {
    const int lane = threadIdx.x & 63;
    while (true) {
        const int32_t now = nm::lds_get(count + min(lane, (int)kBandCounts - 1));
        if (!__any(now < least)) return true;
        if (__any(lane == kStop && now != 0)) return false;
        if (SLEEP) __builtin_amdgcn_s_sleep(1);
    }
}
// `least` with the counts [first, first + number) to be v at least
__device__ __forceinline__ int32_t band_need(int32_t least, int first, int number, int32_t v) {
    const int lane = threadIdx.x & 63;
    return lane >= first && lane < first + number ? v : least;
}
constexpr int32_t kBandAny = -0x7fffffff;
// (all lanes write the one word: less to issue than choosing one of them)
__device__ __forceinline__ void band_tell(int32_t *count, int which, int32_t v) { nm::lds_put(count + which, v); }
__device__ __forceinline__ int32_t ring(int32_t at, int32_t size) { return at >= size ? at - size : at; }

// Eight values that are the same for all lanes.
template <typename T> struct alignas(16) Eight { T v[kPanel]; };

template <bool SIGNED, typename T> __device__ __forceinline__ T absent() { return SIGNED ? (T)__builtin_nanf("") : T(0); }
template <bool SIGNED, typename T> __device__ __forceinline__ T product(T l, T u) {
    const T p = l * u;
    return SIGNED && p != p ? T(0) : p;
}

// Wavefronts 0 and 1: panels K = v, v + 2, ...  RL registers of 64 rows hold the panel's rows, the first RA of them
// the rows that the panel before reaches.
template <bool SIGNED, typename T, int RL, int RA> __device__ __forceinline__ void band_panels(const Band<T> &B, int v) {
    const int lane = threadIdx.x & 63;
    const int32_t cbs = B.cb * kPanel;
    int32_t row_slot = lane / kPanel % B.rb, col_slot = 0;   // of panel 0
    auto forward = [&](int32_t by) NM_INLINE {
        row_slot = ring(row_slot + by, B.rb);
        col_slot = ring(col_slot + by, B.cb);
    };
    if (v) forward(1);
    __builtin_amdgcn_s_setprio(3);
    for (int32_t K = v; K < B.panels; K += 2) {
        int32_t least = band_need(kBandAny, kLoaded, kLoaders, K + 1);
        least = band_need(least, kTrailing0 + K % kBandTrailing, 1, K - 2);   // (whose columns these are)
        if (!band_wait<false>(B.count, least)) return;
        T W[kPanel][RL];
        uint32_t has_lo[RL], has_hi[RL];   // bit 8 (c & 3): stored in column c
#pragma unroll
        for (int q = 0; q < RL; ++q) {
            const bool mine = lane / kPanel + 8 * q <= B.blb;
            const int32_t slot = mine ? (row_slot + 8 * q) % B.rb : row_slot;
            const uint64_t m = *reinterpret_cast<const uint64_t *>(B.has + slot * cbs + col_slot * kPanel);
            has_lo[q] = mine ? (uint32_t)m >> (lane & 7) : 0u;
            has_hi[q] = mine ? (uint32_t)(m >> 32) >> (lane & 7) : 0u;
#pragma unroll
            for (int c = 0; c < kPanel; ++c) W[c][q] = B.column(col_slot * kPanel + c)[slot * kPanel + (lane & 7)];
        }
        // row t of the panel `back` before, whose rows are in W from the row 8 back - 8 of that panel's rest on
        auto apply = [&](int back, int t) NM_INLINE {
            const T *const F = B.multipliers(K - back) + t * B.fp;
            const Eight<T> u = *reinterpret_cast<const Eight<T> *>(B.rows(K - back) + t * B.uc + (back - 1) * kPanel);
            T l[RA];
#pragma unroll
            for (int q = 0; q < RA; ++q) {
                const int32_t at = back * kPanel + lane + 64 * q;
                const T x = F[min(at, B.fp - 1)];
                l[q] = at < B.fp ? x : absent<SIGNED, T>();
            }
#pragma unroll
            for (int c = 0; c < kPanel; ++c)
#pragma unroll
                for (int q = 0; q < RA; ++q) {
                    const T p = product<SIGNED>(l[q], u.v[c]);
                    W[c][q] = W[c][q] - p;
                }
        };
        if (K > 1 && B.bub > 1) {
            if (!band_wait<false>(B.count, band_need(kBandAny, kRows0, 1, (K - 1) * kPanel))) return;
#pragma unroll 1
            for (int t = 0; t < kPanel; ++t) apply(2, t);
        }
        if (K > 0) {
#pragma unroll 1   // (registers: unrolled, 370 of them are spilled)
            for (int t = 0; t < kPanel; ++t) {
                if (!band_wait<false>(B.count, band_need(kBandAny, kPivots, 2, (K - 1) * kPanel + t + 1))) return;
                apply(1, t);
            }
        }
        // (the panel whose place this one takes is written, and applied to the rest and to the rows of the next)
        least = band_need(kBandAny, kWritten, 1, K + 1 - B.kept);
        least = band_need(least, kTrailing0, kBandTrailing, K + 1 - B.kept);
        if (!band_wait<false>(B.count, band_need(least, kRows0, 2, (K + 2 - B.kept) * kPanel))) return;
        T *const F = B.multipliers(K);
        T finite = T(0);
        nm::static_for<kPanel>([&](auto pivot) NM_INLINE {
            constexpr int t = decltype(pivot)::value;
            const uint32_t row_lo = (uint32_t)__builtin_amdgcn_readlane((int)has_lo[0], t);
            const uint32_t row_hi = (uint32_t)__builtin_amdgcn_readlane((int)has_hi[0], t);
            const T d = nm::read_lane(W[t][0], t);
            const bool divide = ((t < 4 ? row_lo : row_hi) >> 8 * (t & 3) & 1) != 0;   // (the diagonal is stored)
            T l[RL];
#pragma unroll
            for (int q = 0; q < RL; ++q) {
                const bool stored = ((t < 4 ? has_lo[q] : has_hi[q]) >> 8 * (t & 3) & 1) != 0;
                const bool below = q > 0 || lane > t;
                const T quotient = W[t][q] / d;
                T x = divide && below ? quotient : W[t][q];
                x = stored ? x : T(0);
                finite = __builtin_fma(x, T(0), finite);
                if (SIGNED) x = stored ? x : absent<SIGNED, T>();
                F[t * B.fp + lane + 64 * q] = x;   // (nothing is stored in the rows past the panel's)
                l[q] = below ? x : absent<SIGNED, T>();
            }
            band_tell(B.count, kPivots, K * kPanel + t + 1);
#pragma unroll
            for (int c = t + 1; c < kPanel; ++c) {
                const bool stored = ((c < 4 ? row_lo : row_hi) >> 8 * (c & 3) & 1) != 0;
                const T there = nm::read_lane(W[c][0], t);
                const T u = stored ? there : absent<SIGNED, T>();
#pragma unroll
                for (int q = 0; q < RL; ++q) {
                    const T p = product<SIGNED>(l[q], u);
                    W[c][q] = W[c][q] - p;
                }
            }
        });
        if (__any(finite != T(0))) {
            band_tell(B.count, kStop, 1);
            return;
        }
        band_tell(B.count, kGoodPanel0 + v, K + 1);
        forward(2);
    }
}

// Wavefronts 2 and 3: the panel's rows, columns 64 w .. right of it, a lane each.  They apply the panel before to these rows
// themselves, so that they wait for the update of the one before that only.
template <bool SIGNED, typename T> __device__ __forceinline__ void band_rows(const Band<T> &B, int w) {
    const int lane = threadIdx.x & 63, at = 64 * w + lane;
    const int32_t width = B.bub * kPanel, cbs = B.cb * kPanel;
    if (64 * w >= width) return;
    const bool mine = at < width;
    int32_t row_slot = 0, col_slot = (1 + at / kPanel) % B.cb;
    __builtin_amdgcn_s_setprio(2);
    for (int32_t K = 0; K < B.panels; ++K) {
        int32_t least = band_need(kBandAny, kLoaded, kLoaders, K + 1);
        least = band_need(least, kTrailing0, kBandTrailing, K - 1);
        least = band_need(least, kPivots, 3, K * kPanel);
        least = band_need(least, kWritten, 1, K + 1 - B.kept);
        if (!band_wait<false>(B.count, least)) return;
        const int32_t slot = mine ? col_slot * kPanel + (lane & 7) : 0;
        const T *const column = B.column(slot) + row_slot * kPanel;
        const uint32_t stored = mine && (K + 1) * kPanel + at < B.n ? B.has[row_slot * cbs + slot] : 0u;
        T X[kPanel];
#pragma unroll
        for (int s = 0; s < kPanel; ++s) X[s] = column[s];
        if (K > 0) {
            const T *const F = B.multipliers(K - 1), *const U = B.rows(K - 1);
            const bool reached = at + kPanel < width;
            T u[kPanel];
#pragma unroll
            for (int t = 0; t < kPanel; ++t) u[t] = reached ? U[t * B.uc + at + kPanel] : absent<SIGNED, T>();
#pragma unroll
            for (int t = 0; t < kPanel; ++t) {
                const Eight<T> l = *reinterpret_cast<const Eight<T> *>(F + t * B.fp + kPanel);
#pragma unroll
                for (int s = 0; s < kPanel; ++s) {
                    const T p = product<SIGNED>(l.v[s], u[t]);
                    X[s] = X[s] - p;
                }
            }
        }
        const T *const F = B.multipliers(K);
        T *const U = B.rows(K);
        T finite = T(0);
        bool going = true;
        nm::static_for<kPanel>([&](auto pivot) NM_INLINE {
            constexpr int t = decltype(pivot)::value;
            X[t] = stored >> t & 1u ? X[t] : T(0);
            finite = __builtin_fma(X[t], T(0), finite);
            if (SIGNED) X[t] = stored >> t & 1u ? X[t] : absent<SIGNED, T>();
            if constexpr (t == 0)   // (panel K has taken the rows that these replace)
                going = B.kept > 2 || band_wait<false>(B.count, band_need(kBandAny, kPivots, 1, K * kPanel + 1));
            if (mine) U[t * B.uc + at] = X[t];
            band_tell(B.count, kRows0 + w, K * kPanel + t + 1);
            if constexpr (t + 1 < kPanel) {
                going = going && band_wait<false>(B.count, band_need(kBandAny, kPivots, 1, K * kPanel + t + 1));
                const Eight<T> l = *reinterpret_cast<const Eight<T> *>(F + t * B.fp);
#pragma unroll
                for (int s = t + 1; s < kPanel; ++s) {
                    const T p = product<SIGNED>(l.v[s], X[t]);
                    X[s] = X[s] - p;
                }
            }
        });
        if (!going) return;
        if (__any(finite != T(0))) {
            band_tell(B.count, kStop, 1);
            return;
        }
        band_tell(B.count, kGoodRows0 + w, K + 1);
        row_slot = ring(row_slot + 1, B.rb);
        col_slot = ring(col_slot + 1, B.cb);
    }
}

// Six wavefronts: the panel applied to the columns from the third block right of it on and the rows from the second
// block below it on, a block of columns at a time.
template <bool SIGNED, typename T, int RL> __device__ __forceinline__ void band_trailing(const Band<T> &B, int w) {
    const int lane = threadIdx.x & 63;
    if (B.bub < 3 || B.blb < 2) return;
    // (a block of columns stays with the wavefront of its number modulo six, so nobody waits for another's update)
    int32_t row_slot = (2 + lane / kPanel) % B.rb, col_slot = 3 % B.cb, first = w < 3 ? w + kBandTrailing - 3 : w - 3;
    for (int32_t K = 0; K < B.panels; ++K, first = first == 0 ? kBandTrailing - 1 : first - 1) {
        int32_t least = band_need(kBandAny, kPivots, 3, (K + 1) * kPanel);
        least = band_need(least, kLoaded, kLoaders, K + 1);
        if (!band_wait<true>(B.count, least)) return;
        const T *const F = B.multipliers(K) + 2 * kPanel, *const U = B.rows(K);
        for (int32_t b = 3 + first; b <= B.bub && K + b < B.panels; b += kBandTrailing) {
            T *const block = B.column(ring(col_slot + (b - 3), B.cb) * kPanel);
            int32_t at[RL];
            bool mine[RL];
            T W[RL][kPanel];
#pragma unroll
            for (int q = 0; q < RL; ++q) {
                mine[q] = lane / kPanel + 8 * q + 1 < B.blb;
                at[q] = (mine[q] ? (row_slot + 8 * q) % B.rb : 0) * kPanel + (lane & 7);
#pragma unroll
                for (int c = 0; c < kPanel; ++c) W[q][c] = block[c * B.pitch + at[q]];
            }
#pragma unroll 2
            for (int t = 0; t < kPanel; ++t) {
                const Eight<T> u = *reinterpret_cast<const Eight<T> *>(U + t * B.uc + (b - 1) * kPanel);
#pragma unroll
                for (int q = 0; q < RL; ++q) {
                    const T l = F[t * B.fp + (mine[q] ? lane + 64 * q : 0)];
#pragma unroll
                    for (int c = 0; c < kPanel; ++c) {
                        const T p = product<SIGNED>(l, u.v[c]);
                        W[q][c] = W[q][c] - p;
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < RL; ++q)
                if (mine[q]) {
#pragma unroll
                    for (int c = 0; c < kPanel; ++c) block[c * B.pitch + at[q]] = W[q][c];
                }
        }
        asm volatile("" ::: "memory");
        band_tell(B.count, kTrailing0 + w, K + 1);
        row_slot = ring(row_slot + 1, B.rb);
        col_slot = ring(col_slot + 1, B.cb);
    }
}

// Wavefronts 14 and 15: the blocks of columns in turn, block n + bub coming into the window with panel n (the first ones with
// panel 0), down to the window's last row then.  A block is requested before the one before it is placed.
template <typename T> struct BandColumns {
    int64_t ptr;                  // lane c: where column c starts
    int32_t row[kPanel][2];
    T value[kPanel][2];
    __device__ __forceinline__ int64_t start(int c) const {
        return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(ptr >> 32), c) << 32 |
                         (uint32_t)__builtin_amdgcn_readlane((int)ptr, c));
    }
};
template <typename T> __device__ __forceinline__ void band_load_columns(const Band<T> &B, int w) {
    const int lane = threadIdx.x & 63;
    const int32_t cbs = B.cb * kPanel;
    auto pointers = [&](int32_t block) NM_INLINE { return B.indptr[min(block * kPanel + min(lane, kPanel), B.n)]; };
    auto fetch = [&](BandColumns<T> &C, int64_t ptr) NM_INLINE {
        C.ptr = ptr;
#pragma unroll
        for (int c = 0; c < kPanel; ++c) {
            const int64_t b = C.start(c);
            const int32_t length = (int32_t)(C.start(c + 1) - b);
            // (an empty column: the entry before it, or the first of all)
            const int64_t from = length > 0 ? b : max(b - 1, (int64_t)0);
            const T *const values = B.values + from;
            const int32_t *const rows = reinterpret_cast<const int32_t *>(B.indices + from);   // (low halves: rows fit 31 bits)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (q > 0 && length <= 64) continue;
                const uint32_t at = min(lane + 64 * q, max(length - 1, 0));
                C.row[c][q] = rows[2 * at];
                C.value[c][q] = values[at];
            }
        }
    };
    auto place = [&](const BandColumns<T> &C, int32_t block) NM_INLINE {
        const int32_t n = max(block - B.bub, 0), slot = block % B.cb * kPanel;
        int32_t least = band_need(kBandAny, kPivots, 3, (n + 1 - B.slack) * kPanel);
        least = band_need(least, kWritten, 1, n + 1 - B.slack);
        if (!band_wait<true>(B.count, least)) return false;
        const int32_t limit = (n + B.blb + 1) * kPanel, row_slot = n % B.rb;
#pragma unroll
        for (int c = 0; c < kPanel; ++c)
            for (int32_t r = lane; r < B.rb * kPanel; r += 64) B.column(slot + c)[r] = T(0);
        if (lane < B.rb) *reinterpret_cast<uint64_t *>(B.has + lane * cbs + slot) = 0ull;
        asm volatile("" ::: "memory");
#pragma unroll
        for (int c = 0; c < kPanel; ++c) {
            const int64_t begin = C.start(c);
            const int32_t length = (int32_t)(C.start(c + 1) - begin);
            int32_t in = 0;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (q > 0 && length <= 64) continue;
                const bool there = lane + 64 * q < length && C.row[c][q] < limit;
                const uint64_t all = __ballot(there);
                in += __popcll(all);
                if (all != 0 && there) {
                    const int32_t at = ring(row_slot + (C.row[c][q] / kPanel - n), B.rb), s = C.row[c][q] & 7;
                    B.column(slot + c)[at * kPanel + s] = C.value[c][q];
                    atomicOr(reinterpret_cast<uint32_t *>(B.has + at * cbs + slot) + c / 4, 1u << (8 * (c & 3) + s));
                }
            }
            if (lane == 0) {
                B.base[slot + c] = begin;
                B.len[slot + c] = length;
                B.in[slot + c] = in;
                B.out[slot + c] = 0;
            }
        }
        asm volatile("" ::: "memory");
        // (the next block is the other wavefront's)
        band_tell(B.count, kColumns0 + w, max(block + 2 - B.bub, 0));
        return true;
    };
    // (two sets by name: a copy would wait for the loads; a block past the last one is nobody's, its columns are empty)
    BandColumns<T> C, D;
    int64_t next = pointers(w + 2);
    fetch(C, pointers(w));
    for (int32_t block = w; block < B.panels; block += 4) {
        fetch(D, next);
        next = pointers(block + 4);
        if (!place(C, block)) return;
        if (block + 2 >= B.panels) break;
        fetch(C, next);
        next = pointers(block + 6);
        if (!place(D, block + 2)) return;
    }
    band_tell(B.count, kColumns0 + w, kBandNever);
}

// Wavefronts 8 and 9: the rows that come into the window with panel n.  A lane keeps to one place for a column, whose
// entries it takes in their order, requested before the rows' place is free.
template <typename T> __device__ __forceinline__ void band_load_rows(const Band<T> &B, int w) {
    const int lane = threadIdx.x & 63, slot = 64 * w + lane;
    const int32_t cbs = B.cb * kPanel;
    if (64 * w >= cbs) return;
    band_tell(B.count, kIn0 + w, 1);   // (panel 0 has nothing but new columns)
    int32_t row_slot = (1 + B.blb) % B.rb, ahead = slot / kPanel;   // blocks from panel n's own to the lane's
    int32_t left = 0;
    int64_t from = 0;
    for (int32_t n = 1; n < B.panels; ++n) {
        ahead = ahead == 0 ? B.cb - 1 : ahead - 1;
        const bool active = slot < cbs && ahead < B.bub && (n + ahead) * kPanel + (lane & 7) < B.n;
        if (!band_wait<true>(B.count, band_need(kBandAny, kColumns0, 2, n))) return;
        if (active && (n == 1 || ahead == B.bub - 1)) {
            left = B.len[slot] - B.in[slot];
            from = B.base[slot] + B.in[slot];
        }
        int32_t row[kPanel];
        T value[kPanel];
#pragma unroll
        for (int s = 0; s < kPanel; ++s) {
            const int64_t e = active ? max(from + min(s, left - 1), (int64_t)0) : 0;
            row[s] = reinterpret_cast<const int32_t *>(B.indices)[2 * e];
            value[s] = B.values[e];
        }
        int32_t least = band_need(kBandAny, kPivots, 3, (n + 1 - B.slack) * kPanel);
        least = band_need(least, kWritten, 1, n + 1 - B.slack);
        if (!band_wait<true>(B.count, least)) return;
        if (active) {
            const int32_t limit = (n + B.blb + 1) * kPanel;
            T *const column = B.column(slot) + row_slot * kPanel;
#pragma unroll
            for (int s = 0; s < kPanel; ++s) column[s] = T(0);
            asm volatile("" ::: "memory");
            uint32_t has = 0;
            int32_t taken = 0;
#pragma unroll
            for (int s = 0; s < kPanel; ++s)
                if (s < left && row[s] < limit) {
                    column[row[s] & 7] = value[s];
                    has |= 1u << (row[s] & 7);
                    ++taken;
                }
            B.has[row_slot * cbs + slot] = (uint8_t)has;
            left -= taken;
            from += taken;
        }
        asm volatile("" ::: "memory");
        band_tell(B.count, kIn0 + w, n + 1);
        row_slot = ring(row_slot + 1, B.rb);
    }
}

// Wavefront 4: a panel's rows and columns into the arrays, once all of them are known to be finite.
template <typename T> __device__ __forceinline__ void band_write(const Band<T> &B) {
    const int lane = threadIdx.x & 63;
    const int32_t width = B.bub * kPanel, cbs = B.cb * kPanel;
    int32_t row_slot = 0, col_slot = 0;
    for (int32_t K = 0; K < B.panels; ++K) {
        int32_t least = band_need(kBandAny, kGoodPanel0 + (K & 1), 1, K + 1);
        least = band_need(least, kGoodRows0, 2, K + 1);
        if (!band_wait<true>(B.count, least)) return;
        const T *const F = B.multipliers(K), *const U = B.rows(K);
        const int32_t own = col_slot * kPanel + (lane & 7);
        const int64_t start = B.base[own] + B.out[own];   // of column lane % 8
        int64_t at[kPanel];
#pragma unroll
        for (int c = 0; c < kPanel; ++c)
            at[c] = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(start >> 32), c) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)start, c));
        for (int32_t r0 = 0; r0 < B.fr; r0 += 64) {
            const int32_t r = r0 + lane;
            const uint64_t m = r < B.fr ? *reinterpret_cast<const uint64_t *>(B.has + ring(row_slot + r / kPanel, B.rb) * cbs + col_slot * kPanel) >> (r & 7) : 0;
            T x[kPanel];
#pragma unroll
            for (int c = 0; c < kPanel; ++c) x[c] = F[c * B.fp + r];
#pragma unroll
            for (int c = 0; c < kPanel; ++c) {
                const bool stored = (m >> 8 * c & 1) != 0;
                const uint64_t all = __ballot(stored);
                if (stored) B.values[at[c] + __popcll(all & ((1ull << lane) - 1ull))] = x[c];
                at[c] += __popcll(all);
            }
        }
        for (int32_t at0 = 0; at0 < width; at0 += 64) {
            const int32_t at = at0 + lane;
            if (at < width && (K + 1) * kPanel + at < B.n) {
                const int32_t slot = ring(col_slot + 1 + at / kPanel, B.cb) * kPanel + (lane & 7);
                const uint32_t has = B.has[row_slot * cbs + slot];
                const int32_t before = B.out[slot];
                T *const out = B.values + B.base[slot] + before;
                T x[kPanel];
#pragma unroll
                for (int s = 0; s < kPanel; ++s) x[s] = U[s * B.uc + at];
#pragma unroll
                for (int s = 0; s < kPanel; ++s)
                    if (has >> s & 1u) out[__popc(has & ((1u << s) - 1u))] = x[s];
                B.out[slot] = before + __popc(has);
            }
        }
        asm volatile("" ::: "memory");
        band_tell(B.count, kWritten, K + 1);
        row_slot = ring(row_slot + 1, B.rb);
        col_slot = ring(col_slot + 1, B.cb);
    }
}

template <bool SIGNED, typename T>
__device__ __forceinline__ void lu_band(int32_t n, const int64_t *__restrict__ indices, const int64_t *__restrict__ indptr, T *values, int32_t *ctl,
                                        int32_t *done, unsigned char *s_band) {
    const int bu = ctl[4], bl = ctl[5];
    if (ctl[6] > kBandMaxBreaks || n >= 1 << 30 || indptr[n] == 0) return;   // lu_flow_kernel's
    Band<T> B;
    B.n = n;
    B.panels = (n + kPanel - 1) / kPanel;
    B.blb = max(1, (bl + kPanel - 1) / kPanel);
    B.bub = max(1, (bu + kPanel - 1) / kPanel);
    if (B.blb > 15 || B.bub > 13) return;
    B.fr = (B.blb + 1) * kPanel;
    B.fp = (B.fr + 63) / 64 * 64;
    B.uc = B.bub * kPanel;
    // room for the loads and the writes to lag behind, as much as LDS has
    size_t used = 0;
    for (B.slack = 5, B.kept = 4; ; B.slack = 3, B.kept = 2) {
        B.rb = B.blb + B.slack;
        B.cb = B.bub + B.slack;
        B.pitch = B.rb * kPanel + 1;
        used = 0;
        auto take = [&](size_t bytes) {
            unsigned char *p = s_band + used;
            used += (bytes + 15) & ~size_t(15);
            return p;
        };
        const int32_t columns = B.cb * kPanel;
        B.count = reinterpret_cast<int32_t *>(take(kBandCounts * 4));
        B.base = reinterpret_cast<int64_t *>(take(columns * 8));
        B.len = reinterpret_cast<int32_t *>(take(columns * 4));
        B.in = reinterpret_cast<int32_t *>(take(columns * 4));
        B.out = reinterpret_cast<int32_t *>(take(columns * 4));
        B.has = take(B.rb * columns);
        B.F = reinterpret_cast<T *>(take((size_t)B.kept * kPanel * B.fp * sizeof(T)));
        B.U = reinterpret_cast<T *>(take((size_t)B.kept * kPanel * B.uc * sizeof(T)));
        B.win = reinterpret_cast<T *>(take((size_t)columns * B.pitch * sizeof(T)));
        if ((used <= kBandLds && B.cb <= 16) || B.slack == 3) break;   // (128 places for columns: band_load_rows)
    }
    if (used > kBandLds || B.cb > 16 || B.rb > 64) return;   // (the same in every thread, as are the other ways out above)
    B.indices = indices;
    B.indptr = indptr;
    B.values = values;
    const int v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x < kBandCounts) {
        // wavefronts with nothing to do keep nobody waiting
        const int i = threadIdx.x;
        const bool idle = (B.bub <= 8 && (i == kRows1 || i == kGoodRows1)) || (B.cb <= 8 && i == kIn1) ||
                          (i >= kTrailing0 && (B.bub < 3 || B.blb < 2));
        B.count[i] = idle ? kBandNever : 0;
    }
    __syncthreads();
    // (a SIMD takes every fourth wavefront: the panels' have the least company)
    if (v < 2) {
        if (B.fr <= 64) band_panels<SIGNED, T, 1, 1>(B, v);
        else if (B.fr <= 72) band_panels<SIGNED, T, 2, 1>(B, v);
        else band_panels<SIGNED, T, 2, 2>(B, v);
    } else if (v < 4) {
        band_rows<SIGNED, T>(B, v - 2);
    } else if (v == 4) {
        __builtin_amdgcn_s_setprio(1);
        band_write<T>(B);
    } else if (v == 8 || v == 9) {
        __builtin_amdgcn_s_setprio(1);
        band_load_rows<T>(B, v - 8);
    } else if (v == 14 || v == 15) {
        __builtin_amdgcn_s_setprio(1);
        band_load_columns<T>(B, v - 14);
    } else if (v != 12) {
        const int w = v == 6 ? 0 : v == 7 ? 1 : v == 10 ? 2 : v == 11 ? 3 : v == 5 ? 4 : 5;
        if (B.blb <= 9) band_trailing<SIGNED, T, 1>(B, w);
        else band_trailing<SIGNED, T, 2>(B, w);
    }
    __syncthreads();
    // lu_flow_kernel finds no column left to draw, or goes on behind the last panel that is written (ctl[7]).
    const int32_t written = min(B.count[kWritten] * kPanel, n);
    if (written < n) {
        for (int32_t k = threadIdx.x; k < written; k += kBandWaves * 64) done[k] = 1;
        if (written == 0) return;   // (from the start)
    }
    if (threadIdx.x == 0) {
        ctl[0] = n;
        ctl[7] = written < n ? written : 0;
        ctl[8] = written < n ? written : n;
    }
}

template <typename T>
__global__ __launch_bounds__(kBandWaves * 64) void lu_band_kernel(int32_t n, const int64_t *__restrict__ indices,
                                                                  const int64_t *__restrict__ indptr, T *values,
                                                                  int32_t *ctl, int32_t *done) {
    __shared__ __align__(16) unsigned char s_band[kBandLds];
    if (ctl[9] == 0) lu_band<false>(n, indices, indptr, values, ctl, done, s_band);
    else lu_band<true>(n, indices, indptr, values, ctl, done, s_band);
}

int check_rows(int64_t rows) {
    NM_REQUIRE(rows >= 0, "negative size");
    if (rows >= (int64_t(1) << 31) - 2)
        return nm::fail(NM_ERR_UNSUPPORTED, "splu indexes rows with 32 bits");
    return NM_OK;
}

}  // namespace

extern "C" int nm_splu_symbolic_bytes(int64_t rows, size_t *bytes) {
    NM_REQUIRE(bytes != nullptr, "bytes is null");
    if (int rc = check_rows(rows)) return rc;
    *bytes = lu_layout(rows, nullptr, nullptr);
    return NM_OK;
}

extern "C" int nm_splu_symbolic(int64_t rows, const int64_t *A_indices, const int64_t *A_indptr,
                                int64_t *As_indptr, void *workspace, size_t workspace_bytes, nm_stream stream) {
    if (int rc = check_rows(rows)) return rc;
    NM_REQUIRE(A_indptr && As_indptr && workspace, "null pointer argument");
    LuScratch S;
    const size_t need = lu_layout(rows, workspace, &S);
    if (workspace_bytes < need)
        return nm::fail(NM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, need);
    hipStream_t s = nm::as_stream(stream);
    if (int rc = nm::fill_async(As_indptr + rows, 1, (int64_t)0, s)) return rc;
    if (rows == 0) return NM_OK;
    const int waves = lu_waves(rows);
    hipLaunchKernelGGL(lu_init_kernel, dim3(1024), dim3(kBlock), 0, s, (int64_t)waves * rows, S.stamp, S.keep);
    NM_LAUNCH_CHECK("lu_init_kernel");
    const unsigned grid = (unsigned)nm::ceil_div((int64_t)waves * 64, kBlock);
    hipLaunchKernelGGL((lu_rows_kernel<float, false>), dim3(grid), dim3(kBlock), 0, s, rows, (const float *)nullptr,
                       A_indices, A_indptr, As_indptr, (int64_t *)nullptr, (float *)nullptr, S.stamp, S.queue,
                       S.keep);
    NM_LAUNCH_CHECK("lu_rows_kernel<count>");
    return nm::scan_exclusive_i64(As_indptr, rows + 1, S.scan, s);
}

extern "C" int nm_splu_fill(nm_dtype dt, int64_t rows, const void *A_data, const int64_t *A_indices,
                            const int64_t *A_indptr, const int64_t *As_indptr, int64_t *As_indices, void *As_data,
                            void *workspace, size_t workspace_bytes, nm_stream stream) {
    if (int rc = check_rows(rows)) return rc;
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    if (rows == 0) return NM_OK;
    NM_REQUIRE(A_indptr && As_indptr && workspace, "null pointer argument");
    LuScratch S;
    const size_t need = lu_layout(rows, workspace, &S);
    if (workspace_bytes < need)
        return nm::fail(NM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, need);
    hipStream_t s = nm::as_stream(stream);
    const int waves = lu_waves(rows);
    hipLaunchKernelGGL(lu_init_kernel, dim3(1024), dim3(kBlock), 0, s, (int64_t)waves * rows, S.stamp, S.keep);
    NM_LAUNCH_CHECK("lu_init_kernel");
    const unsigned grid = (unsigned)nm::ceil_div((int64_t)waves * 64, kBlock);
    if (dt == NM_F32)
        hipLaunchKernelGGL((lu_rows_kernel<float, true>), dim3(grid), dim3(kBlock), 0, s, rows, (const float *)A_data,
                           A_indices, A_indptr, const_cast<int64_t *>(As_indptr), As_indices, (float *)As_data,
                           S.stamp, S.queue, S.keep);
    else
        hipLaunchKernelGGL((lu_rows_kernel<double, true>), dim3(grid), dim3(kBlock), 0, s, rows,
                           (const double *)A_data, A_indices, A_indptr, const_cast<int64_t *>(As_indptr), As_indices,
                           (double *)As_data, S.stamp, S.queue, S.keep);
    NM_LAUNCH_CHECK("lu_rows_kernel<fill>");
    return NM_OK;
}

extern "C" int nm_splu_values(nm_dtype dt, int64_t rows, const void *A_data, const int64_t *A_indices,
                              const int64_t *A_indptr, const int64_t *As_indptr, const int64_t *As_indices,
                              void *As_data, nm_stream stream) {
    if (int rc = check_rows(rows)) return rc;
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    if (rows == 0) return NM_OK;
    NM_REQUIRE(A_indptr && As_indptr, "null pointer argument");
    hipStream_t s = nm::as_stream(stream);
    int64_t grid = nm::ceil_div(rows * 64, kBlock);
    if (grid > 65536) grid = 65536;
    if (dt == NM_F32)
        hipLaunchKernelGGL(lu_values_kernel<float>, dim3((unsigned)grid), dim3(kBlock), 0, s, rows,
                           (const float *)A_data, A_indices, A_indptr, As_indptr, As_indices, (float *)As_data);
    else
        hipLaunchKernelGGL(lu_values_kernel<double>, dim3((unsigned)grid), dim3(kBlock), 0, s, rows,
                           (const double *)A_data, A_indices, A_indptr, As_indptr, As_indices, (double *)As_data);
    NM_LAUNCH_CHECK("lu_values_kernel");
    return NM_OK;
}

extern "C" int nm_splu_numeric_bytes(int64_t cols, size_t *bytes) {
    NM_REQUIRE(bytes != nullptr, "bytes is null");
    if (int rc = check_rows(cols)) return rc;
    *bytes = flow_layout(cols, nullptr, nullptr);
    return NM_OK;
}

extern "C" int nm_splu_numeric(nm_dtype dt, int64_t cols, void *Mt_data, const int64_t *Mt_indices,
                               const int64_t *Mt_indptr, void *workspace, size_t workspace_bytes,
                               int64_t poll_limit, nm_stream stream) {
    if (int rc = check_rows(cols)) return rc;
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    if (cols == 0) return NM_OK;
    NM_REQUIRE(Mt_indptr && workspace, "null pointer argument");
    LuFlow F;
    const size_t need = flow_layout(cols, workspace, &F);
    if (workspace_bytes < need)
        return nm::fail(NM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, need);
    hipStream_t s = nm::as_stream(stream);
    if (int rc = nm::fill_async(F.ctl, 16, (int32_t)0, s)) return rc;
    {
        // (a workgroup for 8 columns, since it looks at their values as well)
        const int64_t g = nm::ceil_div(cols, 8);
        const dim3 grid((unsigned)(g > 65536 ? 65536 : g));
        if (dt == NM_F32)
            hipLaunchKernelGGL(lu_below_kernel<float>, grid, dim3(kBlock), 0, s, cols, Mt_indices, Mt_indptr,
                               (const float *)Mt_data, F.below, F.done, F.ctl);
        else
            hipLaunchKernelGGL(lu_below_kernel<double>, grid, dim3(kBlock), 0, s, cols, Mt_indices, Mt_indptr,
                               (const double *)Mt_data, F.below, F.done, F.ctl);
        NM_LAUNCH_CHECK("lu_below_kernel");
    }
    // Whether the factors are a band is known on the device only: the band kernel leaves at once
    // where they are not, lu_flow_kernel where the band kernel has made them.  (A caller that bounds
    // the polls asks for the kernel that polls.)
    if (poll_limit <= 0) {
        if (dt == NM_F32)
            hipLaunchKernelGGL(lu_band_kernel<float>, dim3(1), dim3(kBandWaves * 64), 0, s, (int32_t)cols, Mt_indices,
                               Mt_indptr, (float *)Mt_data, F.ctl, F.done);
        else
            hipLaunchKernelGGL(lu_band_kernel<double>, dim3(1), dim3(kBandWaves * 64), 0, s, (int32_t)cols, Mt_indices,
                               Mt_indptr, (double *)Mt_data, F.ctl, F.done);
        NM_LAUNCH_CHECK("lu_band_kernel");
    }
    int64_t grid = nm::ceil_div(cols, kLuWavesPerBlock);
    if (grid > 1024) grid = 1024;
    const int64_t limit = poll_limit > 0 ? poll_limit : kLuSpinLimit;
    const size_t lds = (size_t)kLuWavesPerBlock * kLuCap * ((dt == NM_F32 ? 4 : 8) + 4);
    auto flow = [&](auto value) -> int {
        using T = decltype(value);
        if (lds > 64 * 1024)
            NM_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(lu_flow_kernel<T>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(lu_flow_kernel<T>, dim3((unsigned)grid), dim3(kLuFlowBlock), lds, s, cols, Mt_indices,
                           Mt_indptr, F.below, (T *)Mt_data, F.done, F.ctl, limit);
        NM_LAUNCH_CHECK("lu_flow_kernel");
        return NM_OK;
    };
    if (int rc = dt == NM_F32 ? flow(0.f) : flow(0.)) return rc;
    int32_t ctl_h[2] = {0, 0};
    if (hipMemcpyAsync(ctl_h, F.ctl, sizeof(ctl_h), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return nm::fail(NM_ERR_HIP, "reading the factorisation status back failed: %s",
                        hipGetErrorString(hipGetLastError()));
    if (ctl_h[1] != 0)
        return nm::fail(NM_ERR_HIP, "a column waited more than %lld polls for one it depends on",
                        (long long)limit);
    return NM_OK;
}
