// Values between A's row-major order and column-major order where columns are scattered.
//
// A walk by column on the transposed structure reads the value of every entry and writes its gradient through
// t_perm.  Where A's columns are scattered each of these is a cache line of its own from beyond L2, 4 or 8
// bytes of it used: at 64 fp32 columns the backward of a sparse times dense product asks for four lines
// an entry, two of them for this, at up to 32 columns for three.  Values brought into column-major order
// beforehand, and gradients taken back from it afterwards, cost two passes each whose requests are coalesced:
//
//   row-major  <->  staged       inside a bin of consecutive row-major positions (a workgroup, through LDS)
//   staged     <->  column-major inside a tile of consecutive column-major positions (the same)
//
// Staged order keeps, inside a bin, the order of the column-major positions, so that the entries that a tile has in
// a bin are consecutive there.  Bins and tiles have as many entries as give such runs about 16 of them
// (tile_of).
//
// The plan (built once per pattern, from its transposed-structure plan):
//   local[q]   row-major position of staged position q, relative to its bin                  (nnz uint16)
//   run[i]     staged positions of a tile's entries, ascending                               (nnz int32)
//   from[i]    column-major position of that entry, relative to its tile                     (nnz uint16)
//
// Not kept: the walk itself reading and writing in staged order (one pass a direction instead of two; the
// lines it has open, 2 MB a die, are in L2 for reading but written out by small pieces, 14.5 M write requests
// for 15.6 M entries: graph of 15.6 M entries, 64 columns, 1533 us a step against 1373).
#include "nm_common.hpp"
#include "nm_permute.hpp"
#include "nm_transpose.hpp"

namespace {

constexpr int kThreads = 1024;

__global__ void invert_kernel(int64_t nnz, const int32_t *__restrict__ perm, int32_t *__restrict__ inverse) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < nnz) inverse[perm[p]] = (int32_t)p;
}

// Ascending order of N keys in LDS (bitonic)
template <int N> __device__ __forceinline__ void sort_keys(int32_t *s) {
    __syncthreads();
    for (int size = 2; size <= N; size *= 2)
        for (int step = size / 2; step > 0; step /= 2) {
#pragma unroll
            for (int k = 0; k < N / 2 / kThreads; ++k) {
                const int t = threadIdx.x + k * kThreads;
                const int lo = 2 * t - (t & (step - 1)), hi = lo + step;
                const int32_t a = s[lo], b = s[hi];
                if ((a > b) == ((lo & size) == 0)) {
                    s[lo] = b;
                    s[hi] = a;
                }
            }
            __syncthreads();
        }
}

// A bin: column-major positions of its entries into ascending order.  inverse[k] is the column-major
// position of row-major entry k going in, that of staged position k coming out.
template <int N>
__global__ __launch_bounds__(kThreads) void bin_kernel(int64_t nnz, const int32_t *__restrict__ perm, int32_t *__restrict__ inverse,
                                                       int32_t *__restrict__ place, uint16_t *__restrict__ local) {
    __shared__ int32_t s_p[N];
    const int64_t base = (int64_t)blockIdx.x * N;
    const int cnt = (int)(nnz - base < N ? nnz - base : N);
    for (int i = threadIdx.x; i < N; i += kThreads) s_p[i] = i < cnt ? inverse[base + i] : 0x7fffffff;
    sort_keys<N>(s_p);
    for (int i = threadIdx.x; i < cnt; i += kThreads) {
        const int32_t p = s_p[i];
        inverse[base + i] = p;
        place[p] = (int32_t)(base + i);
        local[base + i] = (uint16_t)(perm[p] - base);
    }
}

// A tile: staged positions of its entries into ascending order, in place.
template <int N>
__global__ __launch_bounds__(kThreads) void tile_kernel(int64_t nnz, const int32_t *__restrict__ column_major,
                                                        int32_t *__restrict__ run, uint16_t *__restrict__ from) {
    __shared__ int32_t s_q[N];
    const int64_t base = (int64_t)blockIdx.x * N;
    const int cnt = (int)(nnz - base < N ? nnz - base : N);
    for (int i = threadIdx.x; i < N; i += kThreads) s_q[i] = i < cnt ? run[base + i] : 0x7fffffff;
    sort_keys<N>(s_q);
    for (int i = threadIdx.x; i < cnt; i += kThreads) {
        const int32_t q = s_q[i];
        run[base + i] = q;
        from[base + i] = (uint16_t)(column_major[q] - base);
    }
}

// A block's N values through LDS: out[PUT(i)] = LDS[GIVE(i)] after LDS[KEEP(i)] = in[TAKE(i)], where an
// index is i itself or comes from one of the plan's arrays.
//   bin to staged      LDS[i] = in[i]             out[i] = LDS[local[i]]
//   staged to tile     LDS[from[i]] = in[run[i]]  out[i] = LDS[i]
//   tile to staged     LDS[i] = in[i]             out[run[i]] = LDS[from[i]]
//   staged to bin      LDS[local[i]] = in[i]      out[i] = LDS[i]
enum Move { kBinToStaged, kStagedToTile, kTileToStaged, kStagedToBin };
template <typename T, int N, Move MOVE>
__global__ __launch_bounds__(kThreads) void move_kernel(int64_t nnz, const uint16_t *__restrict__ at, const int32_t *__restrict__ run,
                                                        const T *__restrict__ in, T *__restrict__ out) {
    constexpr int kEach = N / kThreads;
    constexpr bool kScatterIn = MOVE == kStagedToTile || MOVE == kStagedToBin;   // LDS[at] = v, else out = LDS[at]
    constexpr bool kRun = MOVE == kStagedToTile || MOVE == kTileToStaged;
    __shared__ T s_v[N];
    const int64_t base = (int64_t)blockIdx.x * N;
    const int cnt = (int)(nnz - base < N ? nnz - base : N);
    int where[kEach], q[kEach];
    T v[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int i = threadIdx.x + k * kThreads;
        const int64_t j = base + (i < cnt ? i : cnt - 1);
        where[k] = nm::stream_load(at + j);
        if constexpr (kRun) q[k] = nm::stream_load(run + j);
        if constexpr (MOVE != kStagedToTile) v[k] = nm::stream_load(in + j);
    }
    if constexpr (MOVE == kStagedToTile) {
#pragma unroll
        for (int k = 0; k < kEach; ++k) v[k] = in[q[k]];
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int i = threadIdx.x + k * kThreads;
        if (i < cnt) s_v[kScatterIn ? where[k] : i] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int i = threadIdx.x + k * kThreads;
        if (i < cnt) out[MOVE == kTileToStaged ? (int64_t)q[k] : base + i] = s_v[kScatterIn ? i : where[k]];
    }
}

// Entries of a bin and of a tile: nnz / N bins meet a tile of N, N * N / nnz entries at a time.
int tile_of(int64_t nnz) { return nnz <= (2 << 20) ? 4096 : nnz <= (8 << 20) ? 8192 : 16384; }

template <typename F> int by_tile(int64_t nnz, F f) {
    const unsigned blocks = (unsigned)nm::ceil_div(nnz, (int64_t)tile_of(nnz));
    switch (tile_of(nnz)) {
        case 4096: return f(std::integral_constant<int, 4096>{}, blocks);
        case 8192: return f(std::integral_constant<int, 8192>{}, blocks);
        default: return f(std::integral_constant<int, 16384>{}, blocks);
    }
}

template <typename T, Move MOVE>
int move(int64_t nnz, const uint16_t *at, const int32_t *run, const T *in, T *out, hipStream_t s) {
    return by_tile(nnz, [&](auto n, unsigned blocks) {
        hipLaunchKernelGGL((move_kernel<T, n(), MOVE>), dim3(blocks), dim3(kThreads), 0, s, nnz, at, run, in, out);
        NM_LAUNCH_CHECK("move_kernel");
        return (int)NM_OK;
    });
}

}  // namespace

namespace nm {

template <typename T> int to_columns(const PermutePlan &p, int64_t nnz, const T *rows, T *staged, T *columns, hipStream_t s) {
    if (nnz == 0) return NM_OK;
    if (int rc = move<T, kBinToStaged>(nnz, p.local, nullptr, rows, staged, s)) return rc;
    return move<T, kStagedToTile>(nnz, p.from, p.run, staged, columns, s);
}
template <typename T> int to_rows(const PermutePlan &p, int64_t nnz, const T *columns, T *staged, T *rows, hipStream_t s) {
    if (nnz == 0) return NM_OK;
    if (int rc = move<T, kTileToStaged>(nnz, p.from, p.run, columns, staged, s)) return rc;
    return move<T, kStagedToBin>(nnz, p.local, nullptr, staged, rows, s);
}
template int to_columns<float>(const PermutePlan &, int64_t, const float *, float *, float *, hipStream_t);
template int to_columns<double>(const PermutePlan &, int64_t, const double *, double *, double *, hipStream_t);
template int to_rows<float>(const PermutePlan &, int64_t, const float *, float *, float *, hipStream_t);
template int to_rows<double>(const PermutePlan &, int64_t, const double *, double *, double *, hipStream_t);

}  // namespace nm

extern "C" int nm_permute_plan_bytes(int64_t nnz, size_t *plan_bytes, size_t *work_bytes) {
    NM_REQUIRE(nnz >= 0 && nnz < 0x7ffffffe, "nnz outside a plan's range");
    NM_REQUIRE(plan_bytes && work_bytes, "null output");
    *plan_bytes = nm::permute_layout(nnz, nullptr, nullptr);
    *work_bytes = nm::align256((size_t)nnz * 4);
    return NM_OK;
}

extern "C" int nm_permute_plan_build(int64_t rows, int64_t cols, int64_t nnz, const void *transpose_plan, void *plan,
                                     size_t plan_bytes, void *work, size_t work_bytes, nm_stream stream) {
    NM_REQUIRE(rows >= 0 && cols >= 0 && nnz >= 0 && nnz < 0x7ffffffe, "size outside a plan's range");
    if (nnz == 0) return NM_OK;
    NM_REQUIRE(transpose_plan && plan && work, "null memory");
    NM_REQUIRE(plan_bytes >= nm::permute_layout(nnz, nullptr, nullptr) && work_bytes >= (size_t)nnz * 4, "memory too small");
    nm::TPlan t;
    nm::tplan_layout(rows, cols, nnz, const_cast<void *>(transpose_plan), &t);
    nm::PermutePlan p;
    nm::permute_layout(nnz, plan, &p);
    hipStream_t s = nm::as_stream(stream);
    int32_t *const inverse = (int32_t *)work;
    hipLaunchKernelGGL(invert_kernel, dim3((unsigned)nm::ceil_div(nnz, 256)), dim3(256), 0, s, nnz, t.t_perm, inverse);
    NM_LAUNCH_CHECK("invert_kernel");
    return by_tile(nnz, [&](auto n, unsigned blocks) {
        hipLaunchKernelGGL((bin_kernel<n()>), dim3(blocks), dim3(kThreads), 0, s, nnz, t.t_perm, inverse, p.run, p.local);
        NM_LAUNCH_CHECK("bin_kernel");
        hipLaunchKernelGGL((tile_kernel<n()>), dim3(blocks), dim3(kThreads), 0, s, nnz, inverse, p.run, p.from);
        NM_LAUNCH_CHECK("tile_kernel");
        return (int)NM_OK;
    });
}
