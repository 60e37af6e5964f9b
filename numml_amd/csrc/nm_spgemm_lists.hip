// Product plan of C = A B by lists: for products beyond the records of nm_spgemm_plan.hip (long rows of B
// or of C).  Every product a_e b_f that C receives is written down three times, in the order in which the
// three passes add it up:
//
//   forward   C[c]      = sum of a[u] * b[v]   products of entry c of C in the order of A's row
//                                              (cpp/sparse_csr_cpu.cpp:193-200)
//   grad_A    gA[e]     = sum of gC[u] * b[v]  products of entry e of A in the order of B's row
//                                              (cpp/sparse_csr_cpu.cpp:261-274)
//   grad_B    gB[f]     = sum of a[u] * gC[v]  products of entry f of B, rows of A ascending
//                                              (cpp/sparse_csr_cpu.cpp:291-303)
//
// so that each pass is one kernel without a merge, a hash table, a search or an atomic, and the serial loops'
// bits.  24 bytes a product; the pattern of C is the caller's.  What bounds them: the requests for the factors that lie
// scattered, one line each from beyond L2 for gC in grad_B.  Power-law graph of 150 000 rows squared (10.1 M
// products, fp32): forward 781 -> 56 us (the hash path and its symbolic phase before), with gradients 1326 -> 230;
// 50 000 rows, 5 entries a row, fp64: 445 -> 17, 600 -> 62.  Making the plan takes 2 ms of the former, 0.4 of the latter.
//
// A workgroup takes its products a tile at a time and a lane adds up a segment alone, so a workgroup with very many
// products makes everybody wait.  Counted before any list is made: the plan is refused where a workgroup would have more
// than kBusiest products; where one of a gradient's would have more than kBusiestBack the gradients are
// left to the kernels without a plan.  Measured in microseconds, this plan against none (fp32, forward + gradients):
//   a workgroup of C:    48 x 48 from 48 x 256 (65 536)       137 + 33 -> 278 + 563
//                        one entry of 32 768 products         301 + 12 -> 9923 + 19564
//   of both gradients:   256 x 1 times 1 x 64 (16 384)          7 + 49 ->  89 + 40
//                        256 x 1 times 1 x 128 (32 768)         8 + 98 -> 108 + 25
//                        256 x 1 times 1 x 256 (65 536)        7 + 242 -> 105 + 28
#include "nm_common.hpp"
#include "nm_scan.hpp"
#include "nm_transpose.hpp"

#include <algorithm>

namespace {

using nm::kWave;
constexpr int kBlock = 256;
constexpr int kTile = 2048;                // products in LDS at a time
constexpr int kPerLane = kTile / kBlock;
constexpr int kBusiest = 65536, kBusiestBack = 16384;   // most products of a workgroup, and of one of a gradient's

struct Lists {          // out[s] = sum over p in [ptr[s], ptr[s + 1]) of U[u[p]] * V[v[p]]
    int32_t *ptr, *u, *v;
};
struct Plan {
    Lists c, a, b;
    int32_t *flags;     // products of the busiest workgroup [0] of C, [1] of a gradient, where they are many
};

size_t plan_layout(int64_t nnzA, int64_t nnzB, int64_t nnzC, int64_t products, void *base, Plan *plan) {
    size_t off = 0;
    auto take = [&](int64_t n) {
        int32_t *q = base ? (int32_t *)((char *)base + off) : nullptr;
        off += nm::align256((size_t)n * 4);
        return q;
    };
    Plan p;
    p.flags = take(64);
    for (auto [list, n] : {std::pair<Lists *, int64_t>{&p.c, nnzC}, {&p.a, nnzA}, {&p.b, nnzB}}) {
        list->ptr = take(n + 1);
        list->u = take(products);
        list->v = take(products);
    }
    if (plan) *plan = p;
    return off;
}

struct Work {
    int64_t *count;     // lengths, scanned in place (the longest of the three)
    int64_t *scan;
    int32_t *entry;     // entry of A of every product, in the order of A
    int32_t *raw;       // products of C's entries in any order
    int32_t *cursor;
};
size_t work_layout(int64_t rowsB, int64_t nnzA, int64_t nnzB, int64_t nnzC, int64_t products, void *base, Work *work) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void *q = base ? (char *)base + off : nullptr;
        off += nm::align256(bytes);
        return q;
    };
    const int64_t most = std::max(std::max(nnzA, nnzB), std::max(nnzC, rowsB)) + 1;
    Work w;
    w.count = (int64_t *)take((size_t)most * 8);
    w.scan = (int64_t *)take(nm::scan_scratch_bytes(most));
    w.entry = (int32_t *)take((size_t)products * 4);
    w.raw = (int32_t *)take((size_t)products * 4);
    w.cursor = (int32_t *)take((size_t)nnzC * 4);
    if (work) *work = w;
    return off;
}

// count[e] = entries of the row of B that entry e of A names (count[nnzA] = 0)
__global__ __launch_bounds__(kBlock) void lengths_kernel(int64_t nnzA, const int64_t *__restrict__ A_indices,
                                                         const int64_t *__restrict__ B_indptr, int64_t *__restrict__ count) {
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e > nnzA) return;
    count[e] = e < nnzA ? B_indptr[A_indices[e] + 1] - B_indptr[A_indices[e]] : 0;
}

__global__ void narrow_kernel(int64_t n, const int64_t *__restrict__ wide, int32_t *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (int32_t)wide[i];
}

// The last index in [lo, hi) whose pointer is at or before p (ptr[lo] <= p): past empty ones, the one that p lies in.
template <typename P> __device__ __forceinline__ int64_t last_at(const P *__restrict__ ptr, int64_t lo, int64_t hi, int64_t p) {
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) >> 1;
        if (ptr[mid] <= p) lo = mid; else hi = mid;
    }
    return lo;
}

// Where a product lies: the entry in whose list it is and that entry's row.  Product by product, so that neither a row
// nor an entry with millions of products keeps one wavefront busy; a workgroup's products are consecutive, and
// its two ends bound what its lanes look through.
struct Place {
    int64_t entry, row;
};
__device__ __forceinline__ Place place_of(int64_t p, int64_t products, const int32_t *__restrict__ ptr, int64_t entries,
                                          const int64_t *__restrict__ indptr, int64_t rows) {
    __shared__ Place s_end[2];
    if (threadIdx.x < 2) {
        const int64_t end = (int64_t)(blockIdx.x + threadIdx.x) * kBlock - threadIdx.x;
        const int64_t e = last_at(ptr, 0, entries, end < products ? end : products - 1);
        s_end[threadIdx.x] = Place{e, last_at(indptr, 0, rows, e)};
    }
    __syncthreads();
    const int64_t e = last_at(ptr, s_end[0].entry, s_end[1].entry + 1, p);
    return Place{e, last_at(indptr, s_end[0].row, s_end[1].row + 1, e)};
}

// Place in C, entry of A and entry of B of every product; counts the products of C's entries.
__global__ __launch_bounds__(kBlock) void products_kernel(
    int64_t products, int64_t rows, int64_t nnzA, const int64_t *__restrict__ A_indices, const int64_t *__restrict__ A_indptr,
    const int64_t *__restrict__ B_indices, const int64_t *__restrict__ B_indptr, const int64_t *__restrict__ C_indices,
    const int64_t *__restrict__ C_indptr, Lists a, int32_t *__restrict__ entry, unsigned long long *__restrict__ count) {
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const Place at = place_of(p < products ? p : products - 1, products, a.ptr, nnzA, A_indptr, rows);
    if (p >= products) return;
    const int64_t f = B_indptr[A_indices[at.entry]] + (p - a.ptr[at.entry]);
    const int64_t column = B_indices[f];
    int64_t l = C_indptr[at.row], h = C_indptr[at.row + 1];
    while (l < h) {
        const int64_t mid = (l + h) >> 1;
        if (C_indices[mid] < column) l = mid + 1; else h = mid;
    }
    a.u[p] = (int32_t)l;
    a.v[p] = (int32_t)f;
    entry[p] = (int32_t)at.entry;
    atomicAdd(&count[l], 1ull);
}

__global__ __launch_bounds__(kBlock) void place_kernel(int64_t products, const int32_t *__restrict__ dest, int32_t *__restrict__ cursor,
                                                       int32_t *__restrict__ raw) {
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p < products) raw[atomicAdd(&cursor[dest[p]], 1)] = (int32_t)p;
}

// The factors of C's products, whose numbers lie in `raw` entry by entry, ascending
__global__ __launch_bounds__(kBlock) void c_lists_kernel(int64_t products, const int32_t *__restrict__ raw, const int32_t *__restrict__ entry,
                                                         const int32_t *__restrict__ f, Lists c) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= products) return;
    const int32_t p = raw[i];
    c.u[i] = entry[p];
    c.v[i] = f[p];
}

// count[j] = products of row j of B: its entries times the entries of A's column j
__global__ void row_products_kernel(int64_t rowsB, const int64_t *__restrict__ B_indptr, const int32_t *__restrict__ t_indptr,
                                    int64_t *__restrict__ count) {
    const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (j <= rowsB) count[j] = j < rowsB ? (B_indptr[j + 1] - B_indptr[j]) * (t_indptr[j + 1] - t_indptr[j]) : 0;
}

// Where the lists of B's entries begin: an entry of row j has a product with every entry of A's column j (a wavefront a
// row of B in turn).
__global__ __launch_bounds__(kBlock) void b_ptr_kernel(int64_t rowsB, int64_t products, const int64_t *__restrict__ B_indptr,
                                                       const int32_t *__restrict__ t_indptr, const int64_t *__restrict__ start, Lists b) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t waves = (int64_t)gridDim.x * (kBlock / kWave);
    for (int64_t j = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; j < rowsB; j += waves) {
        const int64_t fb = B_indptr[j], len = B_indptr[j + 1] - fb, col = t_indptr[j + 1] - t_indptr[j], p0 = start[j];
        for (int64_t k = lane; k < len; k += kWave) b.ptr[fb + k] = (int32_t)(p0 + k * col);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) b.ptr[B_indptr[rowsB]] = (int32_t)products;
}

__global__ __launch_bounds__(kBlock) void b_lists_kernel(int64_t products, int64_t rowsB, int64_t nnzB, const int64_t *__restrict__ B_indptr,
                                                         const int32_t *__restrict__ t_indptr, const int32_t *__restrict__ t_perm,
                                                         Lists a, Lists b) {
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const Place at = place_of(p < products ? p : products - 1, products, b.ptr, nnzB, B_indptr, rowsB);
    if (p >= products) return;
    const int32_t e = t_perm[t_indptr[at.row] + (p - b.ptr[at.entry])];
    b.u[p] = e;
    b.v[p] = a.u[a.ptr[e] + (at.entry - B_indptr[at.row])];
}

// Products of the busiest workgroup of segments_kernel, where they are more than kBusiestBack
__global__ __launch_bounds__(kBlock) void busiest_kernel(int64_t segments, int per_block, const int32_t *__restrict__ ptr, int32_t *flag) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x, s = i * per_block;
    int n = 0;
    if (s < segments) n = ptr[s + per_block < segments ? s + per_block : segments] - ptr[s];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) n = max(n, __shfl_xor(n, off, kWave));
    if ((threadIdx.x & (kWave - 1)) == 0 && n > kBusiestBack) atomicMax(flag, n);
}

// out[s] = sum over p of U[u[p]] * V[v[p]], terms in the order of p from +0.0: a workgroup has kBlock * L
// consecutive segments, makes their products a tile at a time (coalesced over the lists, eight products a
// lane in flight) and leaves them in LDS, where a lane adds up its L segments.
template <typename T, int L>
__global__ __launch_bounds__(kBlock) void segments_kernel(int64_t segments, Lists x, const T *__restrict__ U, const T *__restrict__ V,
                                                          T *__restrict__ out) {
    __shared__ T s_p[kTile];
    const int64_t s0 = (int64_t)blockIdx.x * (kBlock * L);
    const int64_t s1 = s0 + kBlock * L < segments ? s0 + kBlock * L : segments;
    const int t = threadIdx.x;
    const int begin = x.ptr[s0], end = x.ptr[s1];
    int b[L], e[L];
    T acc[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int64_t s = s0 + i * kBlock + t;
        b[i] = s < s1 ? x.ptr[s] : end;
        e[i] = s < s1 ? x.ptr[s + 1] : end;
        acc[i] = T(0);
    }
    for (int base = begin; base < end; base += kTile) {
        const int n = end - base < kTile ? end - base : kTile;
        int u[kPerLane], v[kPerLane];
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
            const int p = base + (t + k * kBlock < n ? t + k * kBlock : n - 1);
            u[k] = nm::stream_load(x.u + p);
            v[k] = nm::stream_load(x.v + p);
        }
        T fu[kPerLane], fv[kPerLane];
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
            fu[k] = U[u[k]];
            fv[k] = V[v[k]];
        }
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) s_p[t + k * kBlock] = fu[k] * fv[k];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int stop = (e[i] < base + n ? e[i] : base + n) - base;
            int p = (b[i] > base ? b[i] : base) - base;
            // (eight reads under way at a time: a wavefront's lanes wait for the longest segment among theirs; 145 ->
            // 59 us for grad_A of the power-law graph)
            for (; p + 8 <= stop; p += 8) {
                T term[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) term[k] = s_p[p + k];
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[i] += term[k];
            }
            for (; p < stop; ++p) acc[i] += s_p[p];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int64_t s = s0 + i * kBlock + t;
        if (s < s1) out[s] = acc[i];
    }
}

// Segments a lane has: as many as make a tile of products where segments are short
int per_lane(int64_t segments, int64_t products) { return products < 2 * segments ? 8 : 1; }

unsigned grid_of(int64_t n, int64_t per_block) { return (unsigned)nm::ceil_div(n, per_block); }

template <typename T>
int add_up(int64_t segments, int64_t products, const Lists &x, const void *U, const void *V, void *out, hipStream_t s) {
    if (segments == 0) return NM_OK;
    if (per_lane(segments, products) == 8)
        hipLaunchKernelGGL((segments_kernel<T, 8>), dim3(grid_of(segments, kBlock * 8)), dim3(kBlock), 0, s, segments, x, (const T *)U,
                           (const T *)V, (T *)out);
    else
        hipLaunchKernelGGL((segments_kernel<T, 1>), dim3(grid_of(segments, kBlock)), dim3(kBlock), 0, s, segments, x, (const T *)U,
                           (const T *)V, (T *)out);
    NM_LAUNCH_CHECK("segments_kernel");
    return NM_OK;
}

bool fits(int64_t n) { return n >= 0 && n < 0x7ffffffe; }

}  // namespace

extern "C" int nm_spgemm_lists_products(int64_t A_nnz, const int64_t *A_indices, const int64_t *B_indptr, void *work,
                                        size_t work_bytes, int64_t *products, nm_stream stream) {
    NM_REQUIRE(A_nnz >= 0 && products, "negative size or null output");
    *products = 0;
    if (A_nnz == 0) return NM_OK;
    NM_REQUIRE(A_indices && B_indptr && work, "null pointer argument");
    const size_t counts = nm::align256((size_t)(A_nnz + 1) * 8);
    NM_REQUIRE(work_bytes >= counts + nm::scan_scratch_bytes(A_nnz + 1), "work memory too small");
    hipStream_t s = nm::as_stream(stream);
    int64_t *const count = (int64_t *)work;
    hipLaunchKernelGGL(lengths_kernel, dim3(grid_of(A_nnz + 1, kBlock)), dim3(kBlock), 0, s, A_nnz, A_indices, B_indptr, count);
    NM_LAUNCH_CHECK("lengths_kernel");
    if (int rc = nm::scan_exclusive_i64(count, A_nnz + 1, (int64_t *)((char *)work + counts), s)) return rc;
    NM_HIP_TRY(hipMemcpyAsync(products, count + A_nnz, 8, hipMemcpyDeviceToHost, s));
    NM_HIP_TRY(hipStreamSynchronize(s));
    return NM_OK;
}

extern "C" int nm_spgemm_lists_bytes(int64_t B_rows, int64_t A_nnz, int64_t B_nnz, int64_t C_nnz, int64_t products,
                                     size_t *plan_bytes, size_t *work_bytes) {
    NM_REQUIRE(plan_bytes && work_bytes, "null output");
    if (!fits(B_rows) || !fits(A_nnz) || !fits(B_nnz) || !fits(C_nnz) || !fits(products))
        return nm::fail(NM_ERR_UNSUPPORTED, "lists of products index with 32 bits");
    *plan_bytes = plan_layout(A_nnz, B_nnz, C_nnz, products, nullptr, nullptr);
    *work_bytes = work_layout(B_rows, A_nnz, B_nnz, C_nnz, products, nullptr, nullptr);
    return NM_OK;
}

extern "C" int nm_spgemm_lists_build(int64_t A_rows, int64_t B_rows, int64_t A_nnz, int64_t B_nnz, int64_t C_nnz,
                                     int64_t products, const int64_t *A_indices, const int64_t *A_indptr,
                                     const int64_t *B_indices, const int64_t *B_indptr, const int64_t *C_indices,
                                     const int64_t *C_indptr, const void *A_plan_mem, void *plan_mem, size_t plan_bytes,
                                     void *work, size_t work_bytes, int *usable, nm_stream stream) {
    size_t pneed = 0, wneed = 0;
    if (int rc = nm_spgemm_lists_bytes(B_rows, A_nnz, B_nnz, C_nnz, products, &pneed, &wneed)) return rc;
    NM_REQUIRE(A_rows > 0 && A_rows < 0x7ffffffe && A_nnz > 0 && B_nnz > 0 && C_nnz > 0 && products > 0, "an empty product");
    NM_REQUIRE(A_indices && A_indptr && B_indices && B_indptr && C_indices && C_indptr && A_plan_mem && plan_mem && work && usable,
               "null pointer argument");
    NM_REQUIRE(plan_bytes >= pneed && work_bytes >= wneed, "plan or work memory too small");
    *usable = 0;
    hipStream_t s = nm::as_stream(stream);
    Plan p;
    Work w;
    plan_layout(A_nnz, B_nnz, C_nnz, products, plan_mem, &p);
    work_layout(B_rows, A_nnz, B_nnz, C_nnz, products, work, &w);
    nm::TPlan t;
    nm::tplan_layout(A_rows, B_rows, A_nnz, const_cast<void *>(A_plan_mem), &t);
    // (a workgroup has these many at least: no need to look)
    for (int64_t n : {C_nnz, A_nnz, B_nnz})
        if (products > kBusiest * nm::ceil_div(n, (int64_t)kBlock * per_lane(n, products))) return NM_OK;
    if (int rc = nm::fill_async(p.flags, (int64_t)2, (int32_t)0, s)) return rc;
    auto look_at = [&](int64_t n, const Lists &list, int32_t *flag) {
        const int per_block = kBlock * per_lane(n, products);
        hipLaunchKernelGGL(busiest_kernel, dim3(grid_of(nm::ceil_div(n, per_block), kBlock)), dim3(kBlock), 0, s, n, per_block, list.ptr, flag);
    };
    // where the lists begin: A's entries
    hipLaunchKernelGGL(lengths_kernel, dim3(grid_of(A_nnz + 1, kBlock)), dim3(kBlock), 0, s, A_nnz, A_indices, B_indptr, w.count);
    NM_LAUNCH_CHECK("lengths_kernel");
    if (int rc = nm::scan_exclusive_i64(w.count, A_nnz + 1, w.scan, s)) return rc;
    hipLaunchKernelGGL(narrow_kernel, dim3(grid_of(A_nnz + 1, kBlock)), dim3(kBlock), 0, s, A_nnz + 1, w.count, p.a.ptr);
    NM_LAUNCH_CHECK("narrow_kernel");
    look_at(A_nnz, p.a, p.flags + 1);
    // B's entries
    hipLaunchKernelGGL(row_products_kernel, dim3(grid_of(B_rows + 1, kBlock)), dim3(kBlock), 0, s, B_rows, B_indptr, t.t_indptr, w.count);
    NM_LAUNCH_CHECK("row_products_kernel");
    if (int rc = nm::scan_exclusive_i64(w.count, B_rows + 1, w.scan, s)) return rc;
    const int64_t b_blocks = std::min<int64_t>(nm::ceil_div(B_rows, kBlock / kWave), 65536);
    hipLaunchKernelGGL(b_ptr_kernel, dim3((unsigned)b_blocks), dim3(kBlock), 0, s, B_rows, products, B_indptr, t.t_indptr, w.count, p.b);
    NM_LAUNCH_CHECK("b_ptr_kernel");
    look_at(B_nnz, p.b, p.flags + 1);
    // C's entries
    if (int rc = nm::fill_async(w.count, C_nnz + 1, (int64_t)0, s)) return rc;
    const dim3 each(grid_of(products, kBlock));
    hipLaunchKernelGGL(products_kernel, each, dim3(kBlock), 0, s, products, A_rows, A_nnz, A_indices, A_indptr, B_indices,
                       B_indptr, C_indices, C_indptr, p.a, w.entry, (unsigned long long *)w.count);
    NM_LAUNCH_CHECK("products_kernel");
    if (int rc = nm::scan_exclusive_i64(w.count, C_nnz + 1, w.scan, s)) return rc;
    hipLaunchKernelGGL(narrow_kernel, dim3(grid_of(C_nnz + 1, kBlock)), dim3(kBlock), 0, s, C_nnz + 1, w.count, p.c.ptr);
    hipLaunchKernelGGL(narrow_kernel, dim3(grid_of(C_nnz, kBlock)), dim3(kBlock), 0, s, C_nnz, w.count, w.cursor);
    NM_LAUNCH_CHECK("narrow_kernel");
    look_at(C_nnz, p.c, p.flags);
    NM_LAUNCH_CHECK("busiest_kernel");
    int32_t most[2] = {0, 0};
    NM_HIP_TRY(hipMemcpyAsync(most, p.flags, sizeof(most), hipMemcpyDeviceToHost, s));
    NM_HIP_TRY(hipStreamSynchronize(s));
    if (most[0] > kBusiest || most[1] > kBusiest) return NM_OK;
    // the lists; C's products are put into ascending order entry by entry (in the meantime c.u is scratch)
    hipLaunchKernelGGL(place_kernel, each, dim3(kBlock), 0, s, products, p.a.u, w.cursor, w.raw);
    NM_LAUNCH_CHECK("place_kernel");
    if (int rc = nm::segments_sort_i32(nullptr, C_nnz, products, p.c.ptr, w.raw, p.c.u, s)) return rc;
    hipLaunchKernelGGL(c_lists_kernel, each, dim3(kBlock), 0, s, products, w.raw, w.entry, p.a.v, p.c);
    NM_LAUNCH_CHECK("c_lists_kernel");
    *usable = most[1] > kBusiestBack ? 2 : 1;
    if (*usable == 2) return NM_OK;
    hipLaunchKernelGGL(b_lists_kernel, each, dim3(kBlock), 0, s, products, B_rows, B_nnz, B_indptr, t.t_indptr, t.t_perm, p.a, p.b);
    NM_LAUNCH_CHECK("b_lists_kernel");
    return NM_OK;
}

extern "C" int nm_spgemm_numeric_lists(nm_dtype dt, int64_t A_nnz, int64_t B_nnz, int64_t C_nnz, int64_t products,
                                       const void *A_data, const void *B_data, const void *plan_mem, void *C_data,
                                       nm_stream stream) {
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(fits(A_nnz) && fits(B_nnz) && fits(C_nnz) && fits(products) && products > 0, "size outside a plan's range");
    NM_REQUIRE(A_data && B_data && plan_mem && C_data, "null pointer argument");
    Plan p;
    plan_layout(A_nnz, B_nnz, C_nnz, products, const_cast<void *>(plan_mem), &p);
    hipStream_t s = nm::as_stream(stream);
    return dt == NM_F32 ? add_up<float>(C_nnz, products, p.c, A_data, B_data, C_data, s)
                        : add_up<double>(C_nnz, products, p.c, A_data, B_data, C_data, s);
}

extern "C" int nm_spgemm_backward_lists(nm_dtype dt, int64_t A_nnz, int64_t B_nnz, int64_t C_nnz, int64_t products,
                                        const void *grad_C, const void *A_data, const void *B_data, const void *plan_mem,
                                        void *grad_A, void *grad_B, nm_stream stream) {
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(fits(A_nnz) && fits(B_nnz) && fits(C_nnz) && fits(products) && products > 0, "size outside a plan's range");
    NM_REQUIRE(grad_C && A_data && B_data && plan_mem, "null pointer argument");
    Plan p;
    plan_layout(A_nnz, B_nnz, C_nnz, products, const_cast<void *>(plan_mem), &p);
    hipStream_t s = nm::as_stream(stream);
    if (grad_A) {
        if (int rc = dt == NM_F32 ? add_up<float>(A_nnz, products, p.a, grad_C, B_data, grad_A, s)
                                  : add_up<double>(A_nnz, products, p.a, grad_C, B_data, grad_A, s))
            return rc;
    }
    if (!grad_B) return NM_OK;
    return dt == NM_F32 ? add_up<float>(B_nnz, products, p.b, A_data, grad_C, grad_B, s)
                        : add_up<double>(B_nnz, products, p.b, A_data, grad_C, grad_B, s);
}
