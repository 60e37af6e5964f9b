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

// below[k] = position of the first entry of column k with a row index > k.  Also what the choice of
// the numeric kernel depends on: ctl[4] / ctl[5] = entries the widest column reaches above / below its
// diagonal, ctl[6] = columns that do not name the column before them.
__global__ __launch_bounds__(kBlock) void lu_below_kernel(int64_t cols, const int64_t *__restrict__ indices,
                                                          const int64_t *__restrict__ indptr,
                                                          int64_t *__restrict__ below, int32_t *ctl) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int32_t up = 0, down = 0, breaks = 0;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < cols; k += stride) {
        const int64_t pb = indptr[k], pe = indptr[k + 1];
        int64_t lo = pb, hi = pe;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (indices[mid] <= k) lo = mid + 1; else hi = mid;
        }
        below[k] = lo;
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

template <typename T, bool IN_LDS>
__device__ bool lu_column(int64_t k, int64_t pb, int64_t len, const OwnColumn<T, IN_LDS> &own,
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
        if (at_first >= 0) {
            const T prod = other(t_first) * m_ik;
            own.set(at_first, own.val(at_first) - prod);
        }
        for (int64_t t0 = ls + 64; t0 < ie; t0 += 64) {          // columns with more than 64 entries below
            const int64_t t = t0 + lane;
            const int64_t at = t < ie ? find(e, indices[t]) : (int64_t)-1;
            if (at >= 0) {
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

template <typename T>
__global__ __launch_bounds__(kLuFlowBlock) void lu_flow_kernel(int64_t cols, const int64_t *__restrict__ indices,
                                                         const int64_t *__restrict__ indptr,
                                                         const int64_t *__restrict__ below, T *values,
                                                         int32_t *done, int32_t *ctl, int64_t spin_limit) {
    // dynamic LDS: the batch's columns, values first (8-byte aligned), then rows
    extern __shared__ __align__(16) unsigned char s_columns[];
    T (*s_vals)[kLuCap] = reinterpret_cast<T (*)[kLuCap]>(s_columns);
    int32_t (*s_rows)[kLuCap] =
        reinterpret_cast<int32_t (*)[kLuCap]>(s_columns + sizeof(T) * kLuWavesPerBlock * kLuCap);
    __shared__ int64_t s_pb[kLuWavesPerBlock];
    __shared__ int32_t s_ready[kLuWavesPerBlock];
    __shared__ int32_t s_ticket, s_abort;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (;;) {
        // one ticket per workgroup and batch of consecutive columns, one column per wavefront
        if (threadIdx.x == 0) {
            s_ticket = atomicAdd(ctl, kLuWavesPerBlock);
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
                ok = lu_column<T, true>(k, pb, len, own, batch, indices, indptr, below, values, done, ctl, spin_limit,
                                        lane);
            } else {
                const OwnColumn<T, false> own{nullptr, nullptr, indices + pb, values + pb};
                ok = lu_column<T, false>(k, pb, len, own, batch, indices, indptr, below, values, done, ctl, spin_limit,
                                         lane);
            }
            if (!ok && lane == 0) atomicExch(ctl + 1, 1);
        }
        __syncthreads();   // the batch's columns in LDS have no readers left
    }
}

// ---- banded factors --------------------------------------------------------------
//
// A factor whose entries stay near the diagonal is ONE chain of columns: column k + 1 needs column k,
// and lu_flow_kernel pays a hand-over between wavefronts, workgroups or compute units (1.4 us) for
// every link of it whatever the width of the band.  Here one workgroup keeps the part of the matrix
// that is still to be updated in registers and eliminates column by column (right-looking): every
// entry receives the same products in the same ascending order of pivots, so the factors are the
// serial ones bit for bit.
//   * Wavefront v owns the columns j = v mod 16, CS of them at a time; its lanes are rows: row i sits
//     in lane i mod 64 of register i / 64 mod RL, a ring of 64 RL rows.  At step k the last row of any
//     column at hand is below k + 16 CS + bl <= k + 64 RL, so a place of the ring means one row.
//   * Step k: the multipliers of column k come through LDS; the pivot row's entries are in the
//     wavefront's own registers (one lane of each column) and become scalars.  The owner of column
//     k + 1 updates that column first, divides it and hands its multipliers on before it turns to
//     its other columns; the others wait for the column's number in LDS, not for a barrier.
//   * Only products of two STORED entries are subtracted (a bit per row and column, read with the
//     pivot row; a ballot per column of multipliers): a zero or infinite pivot spreads exactly as far
//     as in the serial loop.
//   * A finished column is written out, and the wavefront's next one, requested a round of sixteen
//     steps earlier, takes its place, in the two steps after, when nobody waits for this wavefront.
// 64 x 64 five-point grid in fp64 (4096 columns, reach 64 either way): 5.57 -> 2.41 ms, 0.59 us a column.
// Bound by what the SIMDs issue: 240 vector instructions per step and SIMD, three quarters of the
// time; the chain alone (LDS trip, update, division, LDS trip) would be 0.34 us.  Eight wavefronts of
// nine columns: 2.84 ms; a barrier a step instead of the numbers in LDS: 4.6 ms; without the raised
// priority of the wavefronts whose turn is near: 2.75 ms; the owner putting off the update before its
// turn as well: 2.65 ms.
#define NM_INLINE __attribute__((always_inline))   // (lambdas over register arrays)
constexpr int kBandWaves = 16;
constexpr int kBandMaxRl = 3;
// More breaks in the chain (columns that do not name their predecessor) than this and the matrix may
// be made of three independent blocks or more, which lu_flow_kernel works on side by side: it takes
// 0.75 us a column of ONE block where the reach is 1 and 1.3 us where it is 60, this kernel 0.27 and
// 0.50 us whatever the blocks.
constexpr int kBandMaxBreaks = 1;

// Multipliers are kept for as many columns as there are wavefronts: who publishes column c has seen
// every other wavefront publish one of the fifteen columns before it, and each read the multipliers
// of column c - 16 before it did.
constexpr int kBandDepth = kBandWaves;

struct BandShared {
    double l[kBandDepth][64 * kBandMaxRl];              // multipliers of a column, by ring position (T at the front)
    uint64_t head[kBandDepth][kBandMaxRl + 1];          // which of them are stored entries, whose they are (written last)
    double value[kBandWaves][64 * kBandMaxRl];          // columns on their way into the registers
    int32_t entry[kBandWaves][64 * kBandMaxRl];
};

// w -= l * u on the active lanes for every place S of a register whose bit of `stored` is set; products and
// differences are rounded on their own.  In assembler because the compiler turned the choice per
// column into selects, branches or copies of every column (a step 1.5 to 4 times as long).  The
// inner places are mostly all stored and then go without a choice; the first (finished for a step
// out of eight) and the last (mostly outside the band) are chosen by the execution mask.
#define NM_BAND_M64(i, t) "v_mul_f64 %[t" #t "], %[l], %[u" #i "]\n\t"
#define NM_BAND_M32(i, t) "v_mul_f32 %[t" #t "], %[u" #i "], %[l]\n\t"
#define NM_BAND_D64(i, t) "v_add_f64 %[w" #i "], %[w" #i "], -%[t" #t "]\n\t"
#define NM_BAND_D32(i, t) "v_sub_f32 %[w" #i "], %[w" #i "], %[t" #t "]\n\t"
#define NM_BAND_IF(i) "s_bitcmp1_b32 %[stored], %[S]+" #i "\n\ts_cselect_b64 exec, %[sv], 0\n\t"
#define NM_BAND_P64(i, t) NM_BAND_IF(i) NM_BAND_D64(i, t)
#define NM_BAND_P32(i, t) NM_BAND_IF(i) NM_BAND_D32(i, t)
#define NM_BAND_SEQ2(M, D) M(0, 0) M(1, 1) D(0, 0) D(1, 1)
#define NM_BAND_SEQ3(M, D) M(0, 0) M(1, 1) M(2, 2) D(0, 0) D(1, 1) D(2, 2)
#define NM_BAND_SEQ4(M, D) M(0, 0) M(1, 1) M(2, 2) M(3, 3) D(0, 0) D(1, 1) D(2, 2) D(3, 3)
#define NM_BAND_ALL_LANES "s_mov_b64 exec, %[sv]\n\t"
#define NM_BAND_TEXT(SEQ, M, D, P)                                                                                   \
    "s_bfe_u32 %[bits], %[stored], %[field]\n\ts_cmp_eq_u32 %[bits], %[whole]\n\ts_cbranch_scc0 .Lpick_%=\n\t" SEQ(M, D)    \
    "s_branch .Ldone_%=\n.Lpick_%=:\n\ts_mov_b64 %[sv], exec\n\t" SEQ(M, P) NM_BAND_ALL_LANES ".Ldone_%=:"
#define NM_BAND_W(i) [w##i] "+v"(W[S + i][q])
#define NM_BAND_U(i) [u##i] "s"(u[S + i])
#define NM_BAND_LIST2(X) X(0), X(1)
#define NM_BAND_LIST3(X) NM_BAND_LIST2(X), X(2)
#define NM_BAND_LIST4(X) NM_BAND_LIST3(X), X(3)
#define NM_BAND_CASE(N)                                                                                              \
    if constexpr (CS - 2 == N) {                                                                                     \
        if constexpr (sizeof(T) == 8)                                                                                \
            NM_BAND_ASM_(NM_BAND_TEXT(NM_BAND_SEQ##N, NM_BAND_M64, NM_BAND_D64, NM_BAND_P64), N);                    \
        else                                                                                                         \
            NM_BAND_ASM_(NM_BAND_TEXT(NM_BAND_SEQ##N, NM_BAND_M32, NM_BAND_D32, NM_BAND_P32), N);                    \
    }
#define NM_BAND_ASM_(TEXT, N)                                                                                        \
    asm volatile(TEXT : NM_BAND_LIST##N(NM_BAND_W), [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3),  \
                 [sv] "=&s"(sv), [bits] "=&s"(bits) : [l] "v"(l), [stored] "s"(stored), [S] "n"(S),                  \
                 [field] "n"(S | N << 16), [whole] "n"((1 << N) - 1), NM_BAND_LIST##N(NM_BAND_U) : "scc")
// the places 1 .. CS - 2
template <int CS, typename T, int RL>
__device__ __forceinline__ void band_inner(T l, uint32_t stored, const T (&u)[CS], T (&W)[CS][RL], int q) {
    constexpr int S = 1;
    uint64_t sv;
    uint32_t bits;
    T t0, t1, t2, t3;
    NM_BAND_CASE(2)
    NM_BAND_CASE(3)
    NM_BAND_CASE(4)
}
// the two outer places, bits 0 and 1 of `stored`
template <typename T>
__device__ __forceinline__ void band_outer(T l, uint32_t stored, T u0, T u1, T &w0, T &w1) {
    uint64_t sv;
    T t0, t1;
    constexpr int S = 0;
    if constexpr (sizeof(T) == 8)
        asm volatile("s_mov_b64 %[sv], exec\n\t" NM_BAND_SEQ2(NM_BAND_M64, NM_BAND_P64) "s_mov_b64 exec, %[sv]"
                     : [w0] "+v"(w0), [w1] "+v"(w1), [t0] "=&v"(t0), [t1] "=&v"(t1), [sv] "=&s"(sv)
                     : [l] "v"(l), [stored] "s"(stored), [S] "n"(S), [u0] "s"(u0), [u1] "s"(u1) : "scc");
    else
        asm volatile("s_mov_b64 %[sv], exec\n\t" NM_BAND_SEQ2(NM_BAND_M32, NM_BAND_P32) "s_mov_b64 exec, %[sv]"
                     : [w0] "+v"(w0), [w1] "+v"(w1), [t0] "=&v"(t0), [t1] "=&v"(t1), [sv] "=&s"(sv)
                     : [l] "v"(l), [stored] "s"(stored), [S] "n"(S), [u0] "s"(u0), [u1] "s"(u1) : "scc");
}

// LDS accesses that stay in program order (no waits between them).
template <typename V> __device__ __forceinline__ V lds_get(V *p) {
    asm volatile("" ::: "memory");
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename V> __device__ __forceinline__ void lds_put(V *p, V v) {
    asm volatile("" ::: "memory");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename T, int RL, int CS>
__device__ __forceinline__ void lu_band(int32_t n, int bl, const int64_t *__restrict__ indices,
                                        const int64_t *__restrict__ indptr, T *values, BandShared &sh) {
    constexpr int R = 64 * RL;
    const int lane = threadIdx.x & 63, v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    T W[CS][RL];              // the wavefront's columns
    uint32_t pos[CS];         // entry number inside the column of each of this lane's rows, a byte each; 0xff: not stored
    uint32_t has[RL];         // bit S: this lane's row of the register is stored in column S and not finished
    T fetched[RL];            // the next column: entry e = lane + 64 q
    int32_t fetched_row[RL];
    int32_t fetched_len = 0;
    int64_t base[CS], fetched_b = 0, staged_b = 0;   // where a column starts in the arrays: of the columns, of the
                                                     // one requested, of the one in LDS
    int64_t next_b, next_e;   // place of the column after that in the arrays
    int32_t next_col = 0;

    // (vector loads: a scalar load would be waited for with the next access to LDS, microseconds later)
    int32_t zero = 0;
    asm volatile("" : "+v"(zero));
    auto pointers = [&](int32_t col) NM_INLINE {
        const int32_t at = min(col, n - 1) + zero;
        next_b = indptr[at];
        next_e = indptr[at + 1];
        next_col = col;
    };
    // Requests the column that `pointers` looked up last: unconditional loads (clamped to an entry
    // that exists), so that nothing waits for them before `stage` does.
    auto fetch = [&]() NM_INLINE {
        fetched_len = next_col < n ? (int32_t)(next_e - next_b) : 0;
        fetched_b = next_b;
#pragma unroll
        for (int q = 0; q < RL; ++q) {
            const int64_t t = max(min(next_b + q * 64 + lane, next_e - 1), (int64_t)0);
            fetched_row[q] = reinterpret_cast<const int32_t *>(indices)[2 * t];   // (low half: rows fit 31 bits)
            fetched[q] = values[t];
        }
    };
    T *s_value = reinterpret_cast<T *>(sh.value[v]);
    int32_t *s_entry = sh.entry[v];
    auto stage = [&]() NM_INLINE {
        staged_b = fetched_b;
#pragma unroll
        for (int q = 0; q < RL; ++q) s_entry[q * 64 + lane] = -1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int q = 0; q < RL; ++q)
            if (q * 64 + lane < fetched_len) {
                const uint32_t at = (uint32_t)fetched_row[q] % (uint32_t)R;
                s_value[at] = fetched[q];
                s_entry[at] = q * 64 + lane;
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    // the column in LDS takes the last place
    auto unstage = [&]() NM_INLINE {
        constexpr int S = CS - 1;
        base[S] = staged_b;
        pos[S] = 0;
#pragma unroll
        for (int q = 0; q < RL; ++q) {
            const int32_t e = s_entry[q * 64 + lane];
            W[S][q] = e >= 0 ? s_value[q * 64 + lane] : T(0);
            pos[S] |= (uint32_t)(e >= 0 ? e : 0xff) << (8 * q);
            has[q] |= e >= 0 ? 1u << S : 0u;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    // the columns move up, so that the next one to finish is always in place 0
    auto shift = [&]() NM_INLINE {
#pragma unroll
        for (int S = 0; S + 1 < CS; ++S) {
            pos[S] = pos[S + 1];
            base[S] = base[S + 1];
#pragma unroll
            for (int q = 0; q < RL; ++q) W[S][q] = W[S + 1][q];
        }
#pragma unroll
        for (int q = 0; q < RL; ++q) has[q] >>= 1;
    };
    // f(constant q) for the register that holds ring position p
    auto by_ring = [&](int p, auto f) NM_INLINE {
        if (RL == 1 || p < 64)
            f(std::integral_constant<int, 0>{});
        else if (RL == 2 || p < 128)
            f(std::integral_constant<int, RL < 2 ? 0 : 1>{});
        else
            f(std::integral_constant<int, RL - 1>{});
    };
    // which of this lane's rows are stored below the diagonal (ring position p) of the column in place 0
    bool below[RL];
    uint64_t below_mask[RL];
    bool has_diagonal = false;
    auto look_below = [&](int p) NM_INLINE {
#pragma unroll
        for (int q = 0; q < RL; ++q) {
            int delta = q * 64 + lane - p;
            if (delta < 0) delta += R;
            below[q] = delta >= 1 && delta <= bl && (has[q] & 1u) != 0;
            below_mask[q] = __ballot(below[q]);
        }
        by_ring(p, [&](auto q) NM_INLINE { has_diagonal = (nm::read_lane((int)has[q], p & 63) & 1) != 0; });
    };
    // Divides column c, in place 0 (diagonal at ring position p), and leaves its multipliers for everybody.
    // A wavefront's LDS accesses are carried out in order: who sees the column's number sees them.
    auto finish = [&](int32_t c, int p) NM_INLINE {
        const int buffer = c % kBandDepth;
        T *s_l = reinterpret_cast<T *>(sh.l[buffer]);
        if (has_diagonal) {
            T d = T(0);
            by_ring(p, [&](auto q) NM_INLINE { d = nm::read_lane(W[0][q], p & 63); });
#pragma unroll
            for (int q = 0; q < RL; ++q) {
                const T quot = W[0][q] / d;
                W[0][q] = below[q] ? quot : W[0][q];
            }
        }
#pragma unroll
        for (int q = 0; q < RL; ++q) lds_put(s_l + q * 64 + lane, W[0][q]);
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < RL; ++q) lds_put(&sh.head[buffer][q], below_mask[q]);
            lds_put(reinterpret_cast<int32_t *>(&sh.head[buffer][kBandMaxRl]), c);
        }
#pragma unroll
        for (int q = 0; q < RL; ++q) has[q] &= ~1u;
    };
    auto write_out = [&]() NM_INLINE {
#pragma unroll
        for (int q = 0; q < RL; ++q) {
            const uint32_t e = pos[0] >> (8 * q) & 0xffu;
            if (e != 0xffu) values[base[0] + e] = W[0][q];
        }
    };

#pragma unroll
    for (int q = 0; q < RL; ++q) has[q] = 0;
#pragma unroll
    for (int S = 0; S < CS; ++S) {
        pos[S] = ~0u;
        base[S] = 0;
#pragma unroll
        for (int q = 0; q < RL; ++q) W[S][q] = T(0);
    }
    pointers(v);
#pragma unroll 1
    for (int S = 0; S < CS; ++S) {
        fetch();
        pointers(v + kBandWaves * (S + 1));
        stage();
        shift();
        unstage();
    }
    int32_t ahead = v + kBandWaves * CS;        // column `next_b` belongs to
    if (threadIdx.x < kBandDepth) sh.head[threadIdx.x][kBandMaxRl] = ~0ull;
    __syncthreads();
    int p = 0;                                  // ring position of row k
    auto next = [&](int p) NM_INLINE { return p + 1 == R ? 0 : p + 1; };
    // the multipliers of column k into l, their mask into m; HURRY: asks for everything every time
    auto receive = [&](int32_t k, T (&l)[RL], uint64_t (&m)[RL], auto HURRY) NM_INLINE {
        const int buffer = k & (kBandDepth - 1);
        T *s_l = reinterpret_cast<T *>(sh.l[buffer]);
        int32_t *s_column = reinterpret_cast<int32_t *>(&sh.head[buffer][kBandMaxRl]);
        auto read = [&]() NM_INLINE {
            const int32_t there = lds_get(s_column);
            uint64_t w[RL];
#pragma unroll
            for (int q = 0; q < RL; ++q) w[q] = lds_get(&sh.head[buffer][q]);
#pragma unroll
            for (int q = 0; q < RL; ++q) l[q] = lds_get(s_l + q * 64 + lane);
#pragma unroll
            for (int q = 0; q < RL; ++q)
                m[q] = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w[q] >> 32)) << 32 |
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)w[q]);
            return __builtin_amdgcn_readfirstlane(there) == k;
        };
        if constexpr (HURRY) {
            while (!read()) {}
        } else if (__builtin_expect(!read(), 0)) {
            while (__builtin_amdgcn_readfirstlane(lds_get(s_column)) != k) __builtin_amdgcn_s_sleep(1);
            read();
        }
    };
    // the column whose multipliers are l applied to the columns of this wavefront; OWN: but not to place 0
    auto apply = [&](const T (&l)[RL], const uint64_t (&m)[RL], const T (&u)[CS], uint32_t stored, auto OWN) NM_INLINE {
        stored = (uint32_t)__builtin_amdgcn_readfirstlane((int)stored);
        const uint32_t first = OWN ? 0u : stored & 1u;
        const uint32_t outer = (uint32_t)__builtin_amdgcn_readfirstlane((int)(first | stored >> (CS - 1) << 1));
#pragma unroll
        for (int q = 0; q < RL; ++q)
            if (__builtin_amdgcn_inverse_ballot_w64(m[q])) {
                band_inner<CS>(l[q], stored, u, W, q);
                band_outer(l[q], outer, u[0], u[CS - 1], W[0][q], W[CS - 1][q]);
            }
    };
    // the entries of the row at ring position p in this wavefront's columns, and which of them are stored
    auto row = [&](int p, T (&u)[CS]) NM_INLINE {
        uint32_t stored = 0;
        by_ring(p, [&](auto q) NM_INLINE {
            stored = (uint32_t)nm::read_lane((int)has[q], p & 63);
            nm::static_for<CS>([&](auto S) NM_INLINE { u[S] = nm::read_lane(W[S][q], p & 63); });
        });
        return stored;
    };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    auto step = [&](int32_t k) NM_INLINE {
        T l[RL], u[CS];
        uint64_t m[RL];
        const uint32_t stored = row(p, u);
        receive(k, l, m, no);
        apply(l, m, u, stored, no);
        p = next(p);
    };
    auto update_first = [&](const T (&l)[RL], const uint64_t (&m)[RL], T u0, uint32_t stored) NM_INLINE {
        if ((uint32_t)__builtin_amdgcn_readfirstlane((int)stored) & 1u) {
#pragma unroll
            for (int q = 0; q < RL; ++q)
                if (__builtin_amdgcn_inverse_ballot_w64(m[q])) {
                    const T prod = l[q] * u0;
                    W[0][q] = W[0][q] - prod;
                }
        }
    };
    // Step c - 1: column c is finished and handed on before the wavefront turns to its other columns.
    auto own = [&](int32_t c) NM_INLINE {
        T l[RL], u[CS];
        uint64_t m[RL];
        uint32_t stored = 0;
        const int p1 = c >= 1 ? next(p) : p;    // row c
        look_below(p1);
        if (c >= 1) {
            stored = row(p, u);
            receive(c - 1, l, m, yes);
            __builtin_amdgcn_s_setprio(3);
            update_first(l, m, u[0], stored);
        }
        finish(c, p1);
        __builtin_amdgcn_s_setprio(0);
        if (c >= 1) apply(l, m, u, stored, yes);
        p = p1;
    };
    // Sixteen steps a round: the wavefront finishes its column c, writes it out at step c, puts the column
    // that waits in LDS in its place at step c + 1 and requests the next one, which has the rest of the
    // round to arrive.
#pragma unroll 1
    for (int32_t c = v - kBandWaves; c < n; c += kBandWaves) {
        int32_t k = 0;
        if (c >= 0) {
            own(c);
#pragma unroll 1
            for (k = c; k < min(c + 2, n); ++k) {
                step(k);
                if (k == c) {
                    write_out();
                    shift();
                } else {
                    unstage();
                }
            }
        }
        fetch();
        ahead += kBandWaves;
        pointers(ahead);
        // a wavefront goes before the others of its SIMD as the step at which everybody waits for it comes up
#pragma unroll 1
        for (; k < min(c + kBandWaves - 1, n); ++k) {
            if (k == c + kBandWaves - 8) __builtin_amdgcn_s_setprio(1);
            if (k == c + kBandWaves - 4) __builtin_amdgcn_s_setprio(2);
            step(k);
        }
        stage();
    }
}

template <typename T>
__global__ __launch_bounds__(kBandWaves * 64) void lu_band_kernel(int32_t n, const int64_t *__restrict__ indices,
                                                                  const int64_t *__restrict__ indptr, T *values,
                                                                  int32_t *ctl) {
    __shared__ BandShared sh;
    const int bu = ctl[4], bl = ctl[5];
    if (ctl[6] > kBandMaxBreaks || n >= 1 << 30 || indptr[n] == 0) return;   // lu_flow_kernel's
    // The smallest set of registers that holds the band: the ring (above), and room for bu + 4 columns, as
    // a column is in place two steps after its predecessor is done.  us a column, fp64, this kernel
    // and lu_flow_kernel: reach 28 0.27 and 1.24, reach 60 0.50 and 1.30, reach 76 0.61 and 2.2, reach
    // 92 0.70 and 2.2.
    auto fits = [&](int rl, int cs) { return bu + 4 <= kBandWaves * cs && bl + kBandWaves * cs <= 64 * rl; };
    if (fits(1, 2)) lu_band<T, 1, 2>(n, bl, indices, indptr, values, sh);
    else if (fits(2, 4)) lu_band<T, 2, 4>(n, bl, indices, indptr, values, sh);
    else if (fits(3, 5)) lu_band<T, 3, 5>(n, bl, indices, indptr, values, sh);
    else if (fits(3, 6)) lu_band<T, 3, 6>(n, bl, indices, indptr, values, sh);
    else return;
    // lu_flow_kernel finds no column left to draw.  (A flag that it looks at first is 8 us less of 2.5 ms
    // here, and 50 us of 1.32 ms there for an arrowhead of 1000 columns: the test costs its loop over a column.)
    if (threadIdx.x == 0) ctl[0] = n;
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
    if (int rc = nm::fill_async(F.done, cols, (int32_t)0, s)) return rc;
    {
        int64_t g = nm::ceil_div(cols, kBlock);
        hipLaunchKernelGGL(lu_below_kernel, dim3((unsigned)(g > 65536 ? 65536 : g)), dim3(kBlock), 0, s, cols,
                           Mt_indices, Mt_indptr, F.below, F.ctl);
        NM_LAUNCH_CHECK("lu_below_kernel");
    }
    // Whether the factors are a band is known on the device only: the band kernel leaves at once
    // where they are not, lu_flow_kernel where the band kernel has made them.  (A caller that bounds
    // the polls asks for the kernel that polls.)
    if (poll_limit <= 0) {
        if (dt == NM_F32)
            hipLaunchKernelGGL(lu_band_kernel<float>, dim3(1), dim3(kBandWaves * 64), 0, s, (int32_t)cols, Mt_indices,
                               Mt_indptr, (float *)Mt_data, F.ctl);
        else
            hipLaunchKernelGGL(lu_band_kernel<double>, dim3(1), dim3(kBandWaves * 64), 0, s, (int32_t)cols, Mt_indices,
                               Mt_indptr, (double *)Mt_data, F.ctl);
        NM_LAUNCH_CHECK("lu_band_kernel");
    }
    int64_t grid = nm::ceil_div(cols, kLuWavesPerBlock);
    if (grid > 1024) grid = 1024;
    const int64_t limit = poll_limit > 0 ? poll_limit : kLuSpinLimit;
    const size_t lds = (size_t)kLuWavesPerBlock * kLuCap * ((dt == NM_F32 ? 4 : 8) + 4);
    if (lds > 64 * 1024) {
        const void *fn = dt == NM_F32 ? reinterpret_cast<const void *>(lu_flow_kernel<float>)
                                      : reinterpret_cast<const void *>(lu_flow_kernel<double>);
        NM_HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    }
    if (dt == NM_F32)
        hipLaunchKernelGGL(lu_flow_kernel<float>, dim3((unsigned)grid), dim3(kLuFlowBlock), lds, s, cols, Mt_indices,
                           Mt_indptr, F.below, (float *)Mt_data, F.done, F.ctl, limit);
    else
        hipLaunchKernelGGL(lu_flow_kernel<double>, dim3((unsigned)grid), dim3(kLuFlowBlock), lds, s, cols, Mt_indices,
                           Mt_indptr, F.below, (double *)Mt_data, F.done, F.ctl, limit);
    NM_LAUNCH_CHECK("lu_flow_kernel");
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
