// CSR SpMV forward and its fused backward for gfx950.
//
// Work mapping ("row-block streaming"): one 256-lane workgroup owns R
// consecutive rows.  It stages the rows' offsets in LDS and, when the block's
// stored entries fit the LDS tile, walks them with fully coalesced loads of
// `data` and `indices`, leaving the per-entry results in LDS; blocks whose
// entries do not fit take runs of rows that do, one after the other.  One lane
// per row then adds its row's slice in storage order, which is the summation
// order of the serial CPU loop (cpp/sparse_csr_cpu.cpp:29-35), so rows of fewer
// than kLongRow entries reproduce it bit for bit.  Longer rows are added by a
// wavefront each, entry k by lane k % 64, in every tile and kernel of this file.
//
// Algorithmic HBM bytes, s = sizeof(value):
//   forward : nnz*(s+8) + (rows+1)*8 + cols*s + rows*s
//   backward: nnz*(s+8) + (rows+1)*8 + rows*s + cols*s + nnz*s + cols*s
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <type_traits>

#include "nm_common.hpp"
#include "nm_permute.hpp"
#include "nm_transpose.hpp"

namespace {

using nm::kWave;

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
// Rows of at least this many entries are added in the order of a wavefront (slice_sum).
constexpr int kLongRow = 32;
// A wavefront that has at least so many rows of kLongRow to 2 * kWave entries gives each to its lane.
constexpr int kManyRows = 6;

template <typename T> struct Tile;
template <> struct Tile<float>  { static constexpr int R = 512; static constexpr int CAP = 4096; };
template <> struct Tile<double> { static constexpr int R = 512; static constexpr int CAP = 4096; };
// forward: lanes per workgroup, rows per workgroup, LDS products
#ifndef NM_FWD_BLOCK
#define NM_FWD_BLOCK 256
#endif
#ifndef NM_FWD_R
#define NM_FWD_R 512
#define NM_FWD_CAP 4096
#endif
constexpr int kFwdBlock = NM_FWD_BLOCK, kFwdR = NM_FWD_R;
// LDS products per workgroup: 4096 of fp32 (16 KB), 3072 of fp64 (24 KB instead of 32: six
// workgroups per CU instead of four; 2048 x 2048 Poisson matrix in fp64 73 -> 64 us, row sums of a
// 25-per-row pattern 0.090 -> 0.080 ms, the 7-point pattern 0.058 -> 0.060 ms)
template <typename T> constexpr int kFwdCap = sizeof(T) == 4 ? NM_FWD_CAP : NM_FWD_CAP * 3 / 4;
// entries a lane of the forward keeps in flight when it reads 32-bit structure
#ifndef NM_FWD32_K
#define NM_FWD32_K 5
#endif
// 1: the forward on 32-bit structure loads 4 consecutive entries per lane and request
// (2048 x 2048 Poisson matrix, fp32: 47.6 -> 44.3 us; the same change in the planned backward made
// it slower, 83 -> 87 us and more, so NM_BWD_VEC stays 0)
#ifndef NM_FWD32_VEC
#define NM_FWD32_VEC 1
#endif
// 1: the planned backward loads 4 consecutive entries per lane and request, NM_BWD_VEC_U requests in flight
#ifndef NM_BWD_VEC
#define NM_BWD_VEC 0
#endif
#ifndef NM_BWD_VEC_U
#define NM_BWD_VEC_U 2
#endif
// 1: that forward requests a tile's entries before its row pointers have arrived (2048 x 2048
// Poisson matrix, fp32: 43.2 -> 41.7 us; requesting the planned backward's first entries before
// its own factors are spread made that one slower, 75 -> 78.5 us)
#ifndef NM_FWD_EARLY
#define NM_FWD_EARLY 1
#endif
#ifndef NM_FWD32_VEC_U
#define NM_FWD32_VEC_U 2
#endif
// entries a lane of the planned backward keeps in flight
#ifndef NM_BWD_K
#define NM_BWD_K 6
#endif
// columns per workgroup / LDS entries of the planned backward (measured best at cfg2: 96 vs 101 us)
#ifndef NM_PLANNED_R
#define NM_PLANNED_R 256
#define NM_PLANNED_CAP 2048
#endif
constexpr int kPlannedR = NM_PLANNED_R, kPlannedCap = NM_PLANNED_CAP;

// A block of rows with this many entries or more is walked straight from global memory.
constexpr int32_t kHuge = 1 << 30;

// Loads the block's row offsets relative to `base` into LDS, clamped to kHuge
// so that they fit 32 bits whatever the block holds.
template <int R, int CAP, int BLOCK, typename IDX = int64_t>
__device__ __forceinline__ void stage_offsets(const IDX *__restrict__ indptr, int64_t r0, int nr,
                                              int64_t base, int32_t *s_off) {
    for (int t = threadIdx.x; t <= nr; t += BLOCK) {
        const int64_t d = (int64_t)indptr[r0 + t] - base;
        s_off[t] = (int32_t)(d > kHuge ? kHuge : d);
    }
}

// Rows (or columns) a workgroup takes at a time: the compiled maximum `most` where rows are
// short, fewer where they are long, so that a block holds about `cap` entries -- a matrix with
// few, long rows would otherwise be cut into fewer blocks than the chip has CUs.
inline int block_rows(int64_t rows, int64_t nnz, int most, int cap) {
    const int64_t mean = rows > 0 ? (nnz + rows - 1) / rows : 1;
    const int64_t r = cap / (mean > 0 ? mean : 1);
    return (int)(r > most ? most : (r < 8 ? 8 : r));
}

// The same for the kernels whose work is done when a tile's entries have come: tiles of long_cap entries where rows are long,
// and at least 1024 of them where there are rows enough.  (The tail of a power-law graph is the
// tile with the most entries; a wave that is nearly empty costs as much as a full one.)  Gradient of A,
// fp32, tiles of up to 4096 entries -> 1024: 100 000 rows of 12 on average 15.7 -> 10.5 us, 50 000 12.7 -> 7.4, 200 000 of
// 20 48 -> 36; rows of 7 in 31 500 5.5 -> 5.1; 512 or 2048 tiles at least: 60 x 55 x 50 fp32 5.3 -> 6.3 and 6.9.
// Matrices whose rows are all of one length, and large graphs, want more: row sums of 1 M rows of 20, fp64, with 1024 / 2048 / 4096
// entries 44.6 / 33.9 / 31.4 us, of a graph of 400 000 rows of 20 42.3 / 40.5 / 41.2; gradients of A, rows of 35, 400 000,
// 89 / 52 / 44, the graph 81.8 / 75.8 / 77.4.  With sums that are added to memory 1024 up to 48 entries a row (1 M rows of 20
// 316 / 351 / 393), beyond that all that LDS holds (100 000 rows of 150 227 / 194 / 158).
inline int small_block_rows(int64_t rows, int64_t nnz, int most, int cap, int long_cap) {
    int r = block_rows(rows, nnz, most, nnz > 8 * rows ? std::min(long_cap, cap) : cap);
    while (r > 16 && rows < (int64_t)r * 1024) r /= 2;
    return r;
}

// End of the run of rows that starts at row s0 of the block and fits the LDS tile: the
// largest e in [s0, nr] with at most cap entries in rows [s0, e); e == s0 when row s0
// alone is longer.
__device__ __forceinline__ int run_end(const int32_t *s_off, int s0, int nr, int cap) {
    const int64_t limit = (int64_t)s_off[s0] + cap;
    if (s_off[nr] <= limit) return nr;
    int lo = s0, hi = nr;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (s_off[mid] <= limit) lo = mid; else hi = mid;
    }
    return lo;
}

// The products [b, e) of a row in LDS, added one after the other by one lane.  A row read one product after the
// other is a trip to LDS each (~100 cycles): four are under way at a time (sixteen or eight: the same within 2 %, rows
// of kLongRow being shared).
template <typename T> __device__ __forceinline__ T serial_sum(const T *s_prod, int b, int e) {
    T acc = 0;
    auto add = [&](auto count) {
        constexpr int U = count();
        for (; b + U <= e; b += U) {
            T term[U];
#pragma unroll
            for (int u = 0; u < U; ++u) term[u] = s_prod[b + u];
#pragma unroll
            for (int u = 0; u < U; ++u) acc += term[u];
        }
    };
    add(std::integral_constant<int, 4>{});
    add(std::integral_constant<int, 1>{});
    return acc;
}

// The order of long rows: term l, l + 64, ... to part l, and the 64 parts pairwise (nm::wave_sum).  Here one lane does that for
// its slice [b, e) of kLongRow to 2 * kWave products, eight terms at a time; the others of the wavefront do the same for
// theirs.
template <typename T> __device__ __forceinline__ T lane_sum_long(const T *s_prod, int b, int e, bool on) {
    constexpr int C = 8;
    const int n = on ? e - b : 0;
    const bool twice = __any(n > kWave);
    auto eight = [&](int c0) {      // parts c0 .. c0 + 7, pairwise
        T v[C];
        if (!__any(n > c0)) return T(0);
#pragma unroll
        for (int u = 0; u < C; ++u) v[u] = s_prod[c0 + u < n ? b + c0 + u : 0];
#pragma unroll
        for (int u = 0; u < C; ++u) v[u] = T(0) + (c0 + u < n ? v[u] : T(0));
        if (twice) {
#pragma unroll
            for (int u = 0; u < C; ++u) {
                const T w = s_prod[c0 + u + kWave < n ? b + c0 + u + kWave : 0];
                v[u] += c0 + u + kWave < n ? w : T(0);
            }
        }
        return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    };
    auto quarter = [&](int c0) { const T lo = eight(c0); return lo + eight(c0 + C); };
    auto half = [&](int c0) { const T lo = quarter(c0); return lo + quarter(c0 + 2 * C); };
    const T lo = half(0);
    return lo + half(4 * C);
}

// Sum of a lane's slice [b, e) of the products in LDS (all lanes of a wavefront call it; empty where b == e): in storage
// order, and slices of kLongRow products in the order above, by the wavefront one after the other or (ALONE), where it has
// many of up to 2 * kWave products, each by its lane: the same bits.  So a row's bits do not depend on the tile it is in.
// What bounds it: a workgroup waits for the longest row of its tile, and the wavefront's sum of one row takes as many
// instructions as 64 lanes' sums of their own.  Forward, graphs in fp32, a lane for every row and a trip to LDS for every
// product -> the wavefront, with small tiles (launch_fwd): 100 000 rows, 1.2 M entries 53 -> 15.7 us; 20 000 rows of up to 5000
// entries 63 -> 5.5; 400 000 rows, 7.6 M entries 122 -> 68.  Rows of 35 throughout, a band of 100 000, fp32 / fp64: the wavefront 20
// / 31 us, a lane each 12 / 16.  (The error of a long row's sum against 64 bits is smaller in this order: 6.13e-8 -> 5.98e-8 over
// 30 000 rows of 26.)
template <bool ALONE = true, typename T> __device__ __forceinline__ T slice_sum(const T *s_prod, int b, int e) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool wide = e - b >= kLongRow, alone = wide && e - b <= 2 * kWave;
    T total = 0;
    if (!wide) total = serial_sum(s_prod, b, e);
    unsigned long long todo = __ballot(wide);
    if constexpr (ALONE) {
        const unsigned long long many = __ballot(alone);
        if (__popcll(many) >= kManyRows) {
            const T sum = lane_sum_long(s_prod, b, e, alone);
            if (alone) total = sum;
            todo &= ~many;
        }
    }
    for (; todo; todo &= todo - 1) {
        const int src = __builtin_ctzll(todo);
        const int wb = ALONE ? nm::read_lane(b, src) : __shfl(b, src, kWave), we = ALONE ? nm::read_lane(e, src) : __shfl(e, src, kWave);
        T acc = 0;
        for (int j = wb + lane; j < we; j += kWave) acc += s_prod[j];
        acc = nm::wave_sum(acc);
        if (lane == src) total = acc;
    }
    return total;
}

// The same, left at out[t] where `on` (a slice is empty where it is not on).
template <bool STREAM, bool ALONE = true, typename T>
__device__ __forceinline__ void slice_sums(const T *s_prod, int b, int e, bool on, T *__restrict__ out, int t) {
    const T total = slice_sum<ALONE>(s_prod, b, e);
    if (!on) return;
    if constexpr (STREAM) nm::stream_store(out + t, total);
    else out[t] = total;
}

// Which of n rows of a tile thread t takes first: its own number, or where there are only a few, and so long ones, a share of
// them for every wavefront (rows of 150, fp64: 55 -> 49 us, of 96 48 -> 33; with 64 or 128 rows shared rows of 20 take
// 65 instead of 61).
template <int BLOCK> __device__ __forceinline__ int row_of_thread(int n) {
    const int t = threadIdx.x;
    return n > 16 ? t : (t & (kWave - 1)) * (BLOCK / kWave) + t / kWave;
}

// Rows [s0, e0) of a tile whose products lie in LDS from s_off[s0] - o0 on.
template <typename T, int BLOCK, bool ALONE>
__device__ __forceinline__ void row_sums(const T *s_prod, const int32_t *s_off, int s0, int e0, int o0, T *__restrict__ y) {
    for (int tb = s0; tb < e0; tb += BLOCK) {
        const int t = tb + (ALONE ? row_of_thread<BLOCK>(e0 - s0) : (int)threadIdx.x);
        slice_sums<true, ALONE>(s_prod, t < e0 ? s_off[t] - o0 : 0, t < e0 ? s_off[t + 1] - o0 : 0, t < e0, y, t);
    }
}

// One value for the places [b, e) of a wavefront's slices of LDS, one slice a lane; long ones by the wavefront, unless it has
// many of up to 2 * kWave places.
template <typename T> __device__ __forceinline__ void slice_fill(T *s_v, int b, int e, T v) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool alone = e - b <= 2 * kWave && __popcll(__ballot(e - b >= kLongRow && e - b <= 2 * kWave)) >= kManyRows;
    const bool wide = e - b >= kLongRow && !alone;
    if (!wide)
        for (int j = b; j < e; ++j) s_v[j] = v;
    for (unsigned long long todo = __ballot(wide); todo; todo &= todo - 1) {
        const int src = __builtin_ctzll(todo);
        const int wb = nm::read_lane(b, src), we = nm::read_lane(e, src);
        const T wv = nm::read_lane(v, src);
        for (int j = wb + lane; j < we; j += kWave) s_v[j] = wv;
    }
}

// Element idx of an array.  O32: the array is smaller than 4 GiB, so the address is the base (in
// scalar registers) plus a 32-bit byte offset (one vector register instead of two per access).
template <bool O32, typename X>
__device__ __forceinline__ X *at(X *base, int32_t idx) {
    if (O32) {
        using C = std::conditional_t<std::is_const<X>::value, const char, char>;
        return reinterpret_cast<X *>(reinterpret_cast<C *>(base) + (uint32_t)idx * (uint32_t)sizeof(X));
    }
    return base + idx;
}

// 1: kernels that find a staging list in the plan load the listed segments of x (and, in the
// backward, of g) into LDS with coalesced requests and look the factors of the entries up there,
// instead of one gather instruction per entry and operand.  A gather of 64 scattered words keeps
// the address unit of a compute unit busy for as long as a 1 KB coalesced request, and it was these
// instructions, not bytes, that the kernels waited for (2048 x 2048 Poisson matrix, fp32: forward
// 37.9 -> 31 us in a lab kernel).
#ifndef NM_STAGE_FWD
#define NM_STAGE_FWD 1
#endif
#ifndef NM_STAGE_BWD
#define NM_STAGE_BWD 1
#endif

// quads of staged x per lane of the forward
template <int BLOCK> constexpr int kFwdXQ = nm::kStageFwd * nm::kStageSeg / (4 * BLOCK);

// One tile of the forward whose block of rows has a staging list (see nm_transpose.hpp): n entries,
// 4 <= n <= NQ * 4 * BLOCK <= CAP, starting at `base`.  Written to issue
// as few vector memory instructions as the tile's bytes allow, all of them before the first wait:
// the list arrives in scalar registers with the tile's ends, x comes a quad per lane, a lane owns two
// neighbouring rows and fetches their three pointers with one request, their sums leave as a pair.
template <typename T, int BLOCK, int R, int CAP, int NQ>
__device__ __forceinline__ void fwd_tile_staged(const int64_t r0, const int nr, const int32_t base, const int n,
                                                const T *__restrict__ data, const int16_t *__restrict__ off16,
                                                const int32_t *__restrict__ indptr, const int32_t lo0,
                                                const int32_t hi0, const int32_t lo1, const int32_t hi1,
                                                const T *__restrict__ x,
                                                T *__restrict__ y, T *s_prod, T *s_x) {
    typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef T T2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    typedef uint32_t SV __attribute__((ext_vector_type(2), aligned(2)));    // four 16-bit places
    typedef int32_t I3 __attribute__((ext_vector_type(3), aligned(4)));
    constexpr int XQ = kFwdXQ<BLOCK>;                                       // quads of x per lane
    static_assert(NQ * 4 * BLOCK <= CAP && XQ * 4 * BLOCK == nm::kStageFwd * nm::kStageSeg, "whole quads per lane");
    static_assert(R == 2 * BLOCK && nm::kStageSeg == 128, "two rows per lane, two segments per wavefront and request");
    const int tid = threadIdx.x;
    // The wavefront's two segments per request (lo/hi = places 2 * wave + 8 u and the next one of
    // the list, in scalar registers); an unused place loads segment 0.
    TV xs[XQ];
#pragma unroll
    for (int u = 0; u < XQ; ++u) {
        int32_t seg = u == 0 ? ((tid & 32) ? hi0 : lo0) : ((tid & 32) ? hi1 : lo1);
        seg = seg < 0 ? 0 : seg;
        xs[u] = *reinterpret_cast<const TV *>(x + (int64_t)seg * nm::kStageSeg + 4 * (tid & 31));
    }
    // pointers of rows 2 tid, 2 tid + 1 and the end of the second one
    int32_t p0, p1, p2;
    if (nr == R) {
        const I3 pp = *reinterpret_cast<const I3 *>(indptr + r0 + 2 * tid);
        p0 = pp[0], p1 = pp[1], p2 = pp[2];
    } else {
        const int t = 2 * tid;
        p0 = indptr[r0 + (t < nr ? t : nr)];
        p1 = indptr[r0 + (t + 1 < nr ? t + 1 : nr)];
        p2 = indptr[r0 + (t + 2 < nr ? t + 2 : nr)];
    }
    // the entries: values and places in the staged segments, every quad of the tile at once; the
    // last quad is moved back to end with the tile and overlaps the one before it
    const T *__restrict__ d = data + base;
    const int16_t *__restrict__ co = off16 + base;
    TV aa[NQ];
    SV oo[NQ];
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
        int kc = tid * 4 + u * 4 * BLOCK;
        kc = kc < n - 4 ? kc : n - 4;
        aa[u] = __builtin_nontemporal_load(reinterpret_cast<const TV *>(d + kc));
        oo[u] = __builtin_nontemporal_load(reinterpret_cast<const SV *>(co + kc));
    }
#pragma unroll
    for (int u = 0; u < XQ; ++u) *reinterpret_cast<TV *>(s_x + 4 * (tid + u * BLOCK)) = xs[u];
    __syncthreads();
    // (the entries are pinned here: left alone, the compiler moves the requests of a quad that only
    // some lanes use down into the branch that uses it, behind the barrier)
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
#pragma unroll
        for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(aa[u][q]));
        asm volatile("" : "+v"(oo[u][0]), "+v"(oo[u][1]));
    }
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
        int k = tid * 4 + u * 4 * BLOCK;
        if (k < n) {
            k = k < n - 4 ? k : n - 4;
            TV p;
            p[0] = aa[u][0] * s_x[oo[u][0] & 0xffffu];
            p[1] = aa[u][1] * s_x[oo[u][0] >> 16];
            p[2] = aa[u][2] * s_x[oo[u][1] & 0xffffu];
            p[3] = aa[u][3] * s_x[oo[u][1] >> 16];
            *reinterpret_cast<TV *>(s_prod + k) = p;
        }
    }
    __syncthreads();
    // (a tile with a list has eight entries a row at most: few long ones)
    const T acc0 = slice_sum<false>(s_prod, p0 - base, p1 - base), acc1 = slice_sum<false>(s_prod, p1 - base, p2 - base);
    if (2 * tid + 1 < nr) {
        T2 out;
        out[0] = acc0, out[1] = acc1;
        __builtin_nontemporal_store(out, reinterpret_cast<T2 *>(y + r0 + 2 * tid));
    } else if (2 * tid < nr) {
        nm::stream_store(y + r0 + 2 * tid, acc0);
    }
}

// UNIT: x is taken as all ones and not read, which makes y the row sums
// (cpp/sparse_csr_cpu.cpp:1121-1127); a * 1 == a exactly, so the summation is
// the same storage-order sum.
//
// IDX: int64_t for the structure arrays as the interface delivers them, int32_t for the
// 32-bit copies a transposed-structure plan of the same pattern holds.
//
// LISTS: the instantiation that takes the tiles with a staging list through fwd_tile_staged.  It
// keeps LDS for the staged segments of x, which costs resident workgroups on patterns without
// lists (fp64: 43 instead of 26 KB), so it is a separate instantiation that the caller asks for;
// without it a tile with a list is read through the plan's 32-bit columns (its 16-bit words hold
// places in the list, not offsets).
template <typename T, int BLOCK, int R, int CAP, bool UNIT = false, typename IDX = int64_t, bool LISTS = false>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_num_sgpr(72))) void spmv_fwd_kernel(
    int64_t rows, int rt, const T *__restrict__ data, const IDX *__restrict__ indices,
    const IDX *__restrict__ indptr, const T *__restrict__ x, T *__restrict__ y,
    const int16_t *__restrict__ off16 = nullptr, const int32_t *__restrict__ flags = nullptr,
    const int32_t *__restrict__ f_desc = nullptr) {
    // rt <= R: rows per block of this launch (block_rows); the build for plans without lists finds in its high half those
    // that a plan without packed columns is walked in
    if constexpr (sizeof(IDX) == 4 && !UNIT && !LISTS) rt = flags[2] != 0 ? rt & 0xffff : rt >> 16;
    constexpr bool STAGE = LISTS && NM_STAGE_FWD && NM_FWD32_VEC && sizeof(IDX) == 4 && !UNIT && R == nm::kPackRows;
    constexpr bool HAS_LISTS = NM_STAGE_FWD && sizeof(IDX) == 4 && !UNIT && R == nm::kPackRows;
    // 64-bit structure, fp64: a lane takes 2 consecutive entries per request (16 bytes of values and of columns, aligned
    // to 8), three requests in flight, and the row pointers wait in registers as below.  Requests bound it, not
    // bytes: 127 x 113 x 101 seven-point 41.4 -> 36.7 us (two and four in flight 37.7, 38.8), 27-point on 60^3 24.1 ->
    // 21.5, 1024^2 five-point 21.4 -> 20.9, 20 random entries a row the same.  Not in fp32, whose 8-byte value
    // requests gain nothing there (29.3 -> 29.2) and lose on 1024^2 (16.5 -> 18.7).
    constexpr bool PAIRS = sizeof(IDX) == 8 && sizeof(T) == 8 && !UNIT;
    __shared__ int32_t s_off[R + 1];
    __shared__ __align__(16) T s_prod[CAP];
    __shared__ __align__(16) T s_x[STAGE ? nm::kStageFwd * nm::kStageSeg : 4];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // off16: columns as 16-bit offsets from the first row of a block of nm::kPackRows rows (a plan's
    // c_off16, valid when its flags[2] is set); read when a workgroup's rows are exactly such a block
    const bool packed = sizeof(IDX) == 4 && !UNIT && off16 != nullptr && rt == nm::kPackRows && flags[2] != 0;

    const int64_t ntiles = (rows + rt - 1) / rt, npad = nm::xcd_padded(ntiles);
    for (int64_t id = blockIdx.x; id < npad; id += gridDim.x) {
        const int64_t tile = nm::xcd_tile(id, npad);
        if (tile >= ntiles) continue;
        const int64_t r0 = tile * rt;
        int nr = (int)(rows - r0 < rt ? rows - r0 : rt);
        nr = nr < R ? nr : R;   // rt <= R
        const int64_t base = indptr[r0];
        bool packed_here = packed;
        if constexpr (HAS_LISTS && !STAGE) {
            if (packed && f_desc != nullptr && f_desc[tile * nm::kStageDesc] >= 0) packed_here = false;
        }
        if constexpr (STAGE) if (f_desc != nullptr && rt == nm::kPackRows) {
            // A block of rows with a staging list keeps places in that list where other blocks
            // keep column offsets.  The tile's end, the head of its list and the wavefront's
            // four places of the list are requested together (scalar loads, one round trip);
            // `live` is always true and only keeps those requests in front of the branch.
            const int32_t *__restrict__ desc = f_desc + tile * nm::kStageDesc;
            const int64_t span = (int64_t)indptr[r0 + nr] - base;
            const int32_t d0 = desc[0];
            static_assert(kFwdXQ<BLOCK> == 2, "two requests per lane cover the list");
            const int32_t lo0 = desc[2 * wave], hi0 = desc[2 * wave + 1];
            const int32_t lo1 = desc[BLOCK / 32 + 2 * wave], hi1 = desc[BLOCK / 32 + 2 * wave + 1];
            const bool live = (lo0 & hi0 & lo1 & hi1) != INT32_MIN;
            if ((span >= 4) & (d0 >= 0) & live) {
                if (span <= CAP) {
                    // as many quads per lane as the tile has (a 5-point row block: three of four)
                    constexpr int NQ = CAP / (4 * BLOCK);
                    const int32_t *__restrict__ ip = reinterpret_cast<const int32_t *>(indptr);
                    if (span <= (NQ - 1) * 4 * BLOCK)
                        fwd_tile_staged<T, BLOCK, R, CAP, NQ - 1>(r0, nr, (int32_t)base, (int)span, data, off16, ip,
                                                                  lo0, hi0, lo1, hi1, x, y, s_prod, s_x);
                    else
                        fwd_tile_staged<T, BLOCK, R, CAP, NQ>(r0, nr, (int32_t)base, (int)span, data, off16, ip, lo0, hi0,
                                                              lo1, hi1, x, y, s_prod, s_x);
                    __syncthreads();
                    continue;
                }
                packed_here = false;
            }
        }
        // Both ends of the tile are the same for every lane (scalar loads), so the entry streams
        // can be requested without waiting for the row pointers to pass through LDS: those stay
        // in registers until the products are on their way.
        constexpr int Q = (R + BLOCK) / BLOCK;
        int32_t po[Q];
        bool early = false;
        int n_early = 0;
        if (NM_FWD_EARLY && NM_FWD32_VEC && !UNIT && (sizeof(IDX) == 4 || PAIRS)) {
            const int64_t span = (int64_t)indptr[r0 + nr] - base;
            early = span <= CAP;
            n_early = (int)span;
        }
        if (early) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int t = (int)threadIdx.x + q * BLOCK;
                po[q] = (int32_t)((int64_t)indptr[r0 + (t <= nr ? t : nr)] - base);
            }
        } else {
            stage_offsets<R, CAP, BLOCK, IDX>(indptr, r0, nr, base, s_off);
            __syncthreads();
        }
        const int n = early ? n_early : s_off[nr];
        if (NM_FWD32_VEC && sizeof(IDX) == 4 && !UNIT && n <= CAP) {
            // 32-bit structure: a lane takes 4 consecutive entries per request (16-byte loads of
            // values and columns, aligned to 4 bytes only: a tile starts wherever its first row
            // does), two requests in flight
            typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
            typedef IDX IV __attribute__((ext_vector_type(4), aligned(sizeof(IDX))));
            typedef int16_t SV __attribute__((ext_vector_type(4), aligned(2)));
            const T *__restrict__ d = data + base;
            const IDX *__restrict__ ci = indices + base;
            const int16_t *__restrict__ co = off16 ? off16 + base : nullptr;
            const int n4 = n & ~3;
            constexpr int U = NM_FWD32_VEC_U;
            auto walk = [&](auto pk) {
                constexpr bool PACKED = decltype(pk)::value;
                for (int k0 = threadIdx.x * 4; k0 < n4; k0 += U * 4 * BLOCK) {
                    TV aa[U];
                    IV cc[U];
                    T xx[U][4];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int kc = k0 + u * 4 * BLOCK < n4 ? k0 + u * 4 * BLOCK : n4 - 4;
                        aa[u] = __builtin_nontemporal_load(reinterpret_cast<const TV *>(d + kc));
                        if (PACKED) {
                            const SV o = __builtin_nontemporal_load(reinterpret_cast<const SV *>(co + kc));
#pragma unroll
                            for (int q = 0; q < 4; ++q) cc[u][q] = (IDX)r0 + o[q];
                        } else {
                            cc[u] = __builtin_nontemporal_load(reinterpret_cast<const IV *>(ci + kc));
                        }
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int q = 0; q < 4; ++q) xx[u][q] = x[cc[u][q]];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (k0 + u * 4 * BLOCK < n4) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) s_prod[k0 + u * 4 * BLOCK + q] = aa[u][q] * xx[u][q];
                        }
                }
            };
            if (packed_here) walk(std::true_type{}); else walk(std::false_type{});
            for (int k = n4 + threadIdx.x; k < n; k += BLOCK) s_prod[k] = d[k] * x[ci[k]];
            if (early) {
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const int t = (int)threadIdx.x + q * BLOCK;
                    if (t <= nr) s_off[t] = po[q];
                }
            }
            __syncthreads();
            row_sums<T, BLOCK, !LISTS>(s_prod, s_off, 0, nr, 0, y + r0);
        } else if (n <= CAP) {
            const T *__restrict__ d = data + base;
            const IDX *__restrict__ ci = indices + base;
            if constexpr (PAIRS) {
                typedef T TV __attribute__((ext_vector_type(2), aligned(sizeof(T))));
                typedef IDX IV __attribute__((ext_vector_type(2), aligned(sizeof(IDX))));
                const int n2 = n & ~1;
                constexpr int U = 3;
                for (int k0 = threadIdx.x * 2; k0 < n2; k0 += U * 2 * BLOCK) {
                    TV aa[U];
                    IV cc[U];
                    T xx[U][2];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int kc = k0 + u * 2 * BLOCK < n2 ? k0 + u * 2 * BLOCK : n2 - 2;
                        aa[u] = __builtin_nontemporal_load(reinterpret_cast<const TV *>(d + kc));
                        cc[u] = __builtin_nontemporal_load(reinterpret_cast<const IV *>(ci + kc));
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int q = 0; q < 2; ++q) xx[u][q] = x[cc[u][q]];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (k0 + u * 2 * BLOCK < n2) {
#pragma unroll
                            for (int q = 0; q < 2; ++q) s_prod[k0 + u * 2 * BLOCK + q] = aa[u][q] * xx[u][q];
                        }
                }
                if (n2 < n && threadIdx.x == 0) s_prod[n2] = d[n2] * x[ci[n2]];
            } else {
                // K entries in flight per lane: all their streams, then all their gathers of x.
                // Loads are unconditional on a clamped position (a predicated load would sit in
                // its own branch with its own wait).
                constexpr int K = sizeof(IDX) == 4 ? NM_FWD32_K : 5;   // int64: 4, 5 and 10 measure the same on the 2048 x 2048 Poisson matrix
                for (int k0 = threadIdx.x; k0 < n; k0 += K * BLOCK) {
                    T aa[K], xx[K];
                    IDX cc[K];
#pragma unroll
                    for (int u = 0; u < K; ++u) {
                        const int kc = k0 + u * BLOCK < n ? k0 + u * BLOCK : n - 1;
                        aa[u] = nm::stream_load(d + kc);
                        if (!UNIT) cc[u] = nm::stream_load(ci + kc);
                    }
#pragma unroll
                    for (int u = 0; u < K; ++u) xx[u] = UNIT ? T(1) : x[cc[u]];
                    if (k0 + (K - 1) * BLOCK < n) {
#pragma unroll
                        for (int u = 0; u < K; ++u) s_prod[k0 + u * BLOCK] = aa[u] * xx[u];
                    } else {
#pragma unroll
                        for (int u = 0; u < K; ++u)
                            if (k0 + u * BLOCK < n) s_prod[k0 + u * BLOCK] = aa[u] * xx[u];
                    }
                }
            }
            if (early) {
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const int t = (int)threadIdx.x + q * BLOCK;
                    if (t <= nr) s_off[t] = po[q];
                }
            }
            __syncthreads();
            row_sums<T, BLOCK, !LISTS>(s_prod, s_off, 0, nr, 0, y + r0);
        } else if (n < kHuge) {
            // The block's entries do not fit the tile: runs of consecutive rows that do are taken
            // one after the other.
            auto products = [&](int64_t first, int cnt) {   // s_prod[j] = data * x of entry first + j
                const T *__restrict__ d = data + first;
                const IDX *__restrict__ ci = indices + first;
                constexpr int K = 5;
                for (int k0 = threadIdx.x; k0 < cnt; k0 += K * BLOCK) {
                    T aa[K], xx[K];
                    IDX cc[K];
#pragma unroll
                    for (int u = 0; u < K; ++u) {
                        const int kc = k0 + u * BLOCK < cnt ? k0 + u * BLOCK : cnt - 1;
                        aa[u] = nm::stream_load(d + kc);
                        if (!UNIT) cc[u] = nm::stream_load(ci + kc);
                    }
#pragma unroll
                    for (int u = 0; u < K; ++u) xx[u] = UNIT ? T(1) : x[cc[u]];
#pragma unroll
                    for (int u = 0; u < K; ++u)
                        if (k0 + u * BLOCK < cnt) s_prod[k0 + u * BLOCK] = aa[u] * xx[u];
                }
            };
            for (int s0 = 0; s0 < nr;) {
                const int e0 = run_end(s_off, s0, nr, CAP);
                if (e0 == s0) {
                    // a row longer than the tile, CAP entries at a time; wavefront 0 keeps the
                    // lanes' partial sums (CAP is a multiple of 64: entry k stays with lane k % 64)
                    const int64_t first = base + s_off[s0];
                    const int len = s_off[s0 + 1] - s_off[s0];
                    T acc = 0;
                    for (int c0 = 0; c0 < len; c0 += CAP) {
                        const int cnt = len - c0 < CAP ? len - c0 : CAP;
                        products(first + c0, cnt);
                        __syncthreads();
                        if (wave == 0)
                            for (int j = lane; j < cnt; j += kWave) acc += s_prod[j];
                        __syncthreads();
                    }
                    if (wave == 0) {
                        acc = nm::wave_sum(acc);
                        if (lane == 0) y[r0 + s0] = acc;
                    }
                    s0 += 1;
                    continue;
                }
                const int o0 = s_off[s0];
                products(base + o0, s_off[e0] - o0);
                __syncthreads();
                row_sums<T, BLOCK, !LISTS>(s_prod, s_off, s0, e0, o0, y + r0);
                __syncthreads();
                s0 = e0;
            }
        } else {
            // short rows: one lane each, straight from global memory
            for (int t = threadIdx.x; t < nr; t += BLOCK) {
                const int64_t b = indptr[r0 + t], e = indptr[r0 + t + 1];
                if (e - b >= kLongRow) continue;
                T acc = 0;
                for (int64_t k = b; k < e; ++k) acc += data[k] * (UNIT ? T(1) : x[indices[k]]);
                y[r0 + t] = acc;
            }
            // long rows: one wavefront each
            for (int t = wave; t < nr; t += (BLOCK / kWave)) {
                const int64_t b = indptr[r0 + t], e = indptr[r0 + t + 1];
                if (e - b < kLongRow) continue;
                T acc = 0;
                for (int64_t k = b + lane; k < e; k += kWave) acc += data[k] * (UNIT ? T(1) : x[indices[k]]);
                acc = nm::wave_sum(acc);
                if (lane == 0) y[r0 + t] = acc;
            }
        }
        __syncthreads();
    }
}

// Fused backward by rows, without a plan: out_A[k] = alpha * (a[row] * b[col]); ADD: grad_x[col] += a[row] * data[k] (a build of
// its own: with the rest in one, 2048^2 five-point fp32 191 -> 216 us).  Without ADD this is the masked outer
// product (cpp/sparse_csr_cpu.cpp:60-65 and :750-755).
template <typename T, int R, int CAP, bool ADD>
__global__ __launch_bounds__(kBlock) void spmv_bwd_kernel(
    int64_t rows, int rt, const T *__restrict__ data, const int64_t *__restrict__ indices,
    const int64_t *__restrict__ indptr, const T *__restrict__ a, const T *__restrict__ b, T alpha,
    T *__restrict__ out_A, T *__restrict__ grad_x) {
    typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef int64_t IV __attribute__((ext_vector_type(4), aligned(8)));
    __shared__ int32_t s_off[R + 1];
    __shared__ T s_a[CAP];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

    const int64_t ntiles = (rows + rt - 1) / rt, npad = nm::xcd_padded(ntiles);
    for (int64_t id = blockIdx.x; id < npad; id += gridDim.x) {
        const int64_t tile = nm::xcd_tile(id, npad);
        if (tile >= ntiles) continue;
        const int64_t r0 = tile * rt;
        int nr = (int)(rows - r0 < rt ? rows - r0 : rt);
        nr = nr < R ? nr : R;   // rt <= R
        const int64_t base = indptr[r0];
        stage_offsets<R, CAP, kBlock>(indptr, r0, nr, base, s_off);
        __syncthreads();
        const int n = s_off[nr];
        // entry k, whose row's factor is av
        auto entry = [&](int64_t k, T av) {
            if constexpr (ADD) {
                const int64_t c = indices[k];
                if (out_A) out_A[k] = alpha * (av * b[c]);
                nm::atomic_add(grad_x + c, av * data[k]);
            } else {
                out_A[k] = alpha * (av * b[indices[k]]);
            }
        };
        // a[row] to the entries of rows [s0, e0) in s_a, which begins at entry o0 of the block: one lane per short
        // row, a wavefront per row of kLongRow entries or more
        auto spread = [&](int s0, int e0, int o0) {
            for (int tb = s0; tb < e0; tb += kBlock) {
                const int t = tb + row_of_thread<kBlock>(e0 - s0);
                const int jb = t < e0 ? s_off[t] - o0 : 0, je = t < e0 ? s_off[t + 1] - o0 : 0;
                const T av = t < e0 ? a[r0 + t] : T(0);
                slice_fill(s_a, jb, je, av);
            }
        };
        // `cnt` entries from `first` on, whose factors are s_a[0, cnt): four consecutive entries a lane, unless their
        // sums are added to memory (neighbouring lanes' additions to neighbouring columns go together)
        auto entries = [&](int64_t first, int cnt) {
            if constexpr (ADD) {
                for (int k = threadIdx.x; k < cnt; k += kBlock) entry(first + k, s_a[k]);
                return;
            }
            const int n4 = cnt & ~3;
            for (int k = 4 * threadIdx.x; k < n4; k += 4 * kBlock) {
                const IV c = *(const IV *)(indices + first + k);
                TV o;
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = b[c[v]];
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = alpha * (s_a[k + v] * o[v]);
                *(TV *)(out_A + first + k) = o;
            }
            if (threadIdx.x < (cnt & 3)) entry(first + n4 + threadIdx.x, s_a[n4 + threadIdx.x]);
        };
        if (n <= CAP) {
            spread(0, nr, 0);
            __syncthreads();
            entries(base, n);
        } else if (n < kHuge) {
            // runs of consecutive rows that fit the tile, one after the other
            for (int s0 = 0; s0 < nr;) {
                const int e0 = run_end(s_off, s0, nr, CAP);
                if (e0 == s0) {
                    // a row longer than the tile: lane = entry, straight from global memory
                    const int64_t rb = base + s_off[s0];
                    const int len = s_off[s0 + 1] - s_off[s0];
                    const T av = a[r0 + s0];
                    for (int k = threadIdx.x; k < len; k += kBlock) entry(rb + k, av);
                    s0 += 1;
                    continue;
                }
                const int o0 = s_off[s0];
                spread(s0, e0, o0);
                __syncthreads();
                entries(base + o0, s_off[e0] - o0);
                __syncthreads();
                s0 = e0;
            }
        } else {
            for (int t = threadIdx.x; t < nr; t += kBlock) {
                const int64_t rb = indptr[r0 + t], re = indptr[r0 + t + 1];
                if (re - rb >= kLongRow) continue;
                const T av = a[r0 + t];
                for (int64_t k = rb; k < re; ++k) entry(k, av);
            }
            for (int t = wave; t < nr; t += kWavesPerBlock) {
                const int64_t rb = indptr[r0 + t], re = indptr[r0 + t + 1];
                if (re - rb < kLongRow) continue;
                const T av = a[r0 + t];
                for (int64_t k = rb + lane; k < re; k += kWave) entry(k, av);
            }
        }
        __syncthreads();
    }
}

// The same on a transposed-structure plan: out_A[k] = a[row] * b[col] and / or prod[k] = a[row] * data[k].  A workgroup has
// `tile` consecutive entries (a multiple of 64, at most CAP), whatever rows they are of: chunk_row tells the first one's.  (With
// tiles of rows one workgroup has all of a long row and of long rows side by side: 20 rows of 100 000 1210 -> 9 us, power-law
// rows in descending order, 100 000 rows, 2 M entries 403 -> 12.5.)
//
// It reads b once an entry and everything else in order, so that a grid moves its bytes (127 x 113 x 101 fp32: 81 MB in
// 20 us) and a graph waits for its gathers from L2.  The gradient of A alone is made here too: a walk by column writes it
// entry by entry where columns are scattered (7.6 M entries fp32 243 -> 50 us) and gathers positions where they are not
// (the grid 46 -> 20).
template <typename T, int R, int CAP>
__global__ __launch_bounds__(kBlock) void spmv_bwd_entries_kernel(
    int64_t rows, int64_t nnz, int tile, const T *__restrict__ data, const int32_t *__restrict__ idx32,
    const int32_t *__restrict__ ptr32, const int32_t *__restrict__ chunk_row, const T *__restrict__ a, const T *__restrict__ b,
    T *__restrict__ out_A, T *__restrict__ prod) {
    typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef int32_t IV __attribute__((ext_vector_type(4), aligned(4)));
    __shared__ int32_t s_off[R + 1];
    __shared__ T s_a[CAP];
    const int64_t ntiles = (nnz + tile - 1) / tile, npad = nm::xcd_padded(ntiles);
    for (int64_t id = blockIdx.x; id < npad; id += gridDim.x) {
        const int64_t at = nm::xcd_tile(id, npad);
        if (at >= ntiles) continue;
        const int64_t base = at * tile, next = base + tile;
        const int n = (int)(nnz - base < tile ? nnz - base : tile);
        const int32_t r0 = chunk_row[base / kWave], r1 = next < nnz ? chunk_row[next / kWave] : (int32_t)(rows - 1);
        // a[row] to the rows' entries: rows r0 .. r1 with their entries among these n
        if (r1 - r0 < 4 * R) {
            for (int32_t s0 = r0; s0 <= r1; s0 += R) {
                const int nr = r1 - s0 + 1 < R ? r1 - s0 + 1 : R;
                if (s0 > r0) __syncthreads();
                for (int t = threadIdx.x; t <= nr; t += kBlock) {
                    const int64_t d = (int64_t)ptr32[s0 + t] - base;
                    s_off[t] = (int)(d < 0 ? 0 : d < n ? d : n);
                }
                __syncthreads();
                for (int tb = 0; tb < nr; tb += kBlock) {
                    const int t = tb + row_of_thread<kBlock>(nr);
                    const int jb = t < nr ? s_off[t] : 0, je = t < nr ? s_off[t + 1] : 0;
                    slice_fill(s_a, jb, je, je > jb ? a[s0 + t] : T(0));
                }
            }
        } else {
            // (nearly all of these rows are empty: every entry looks for its own)
            for (int k = threadIdx.x; k < n; k += kBlock) {
                int32_t lo = r0, hi = r1 + 1;
                while (hi - lo > 1) {
                    const int32_t mid = lo + (hi - lo) / 2;
                    if (ptr32[mid] <= base + k) lo = mid; else hi = mid;
                }
                s_a[k] = a[lo];
            }
        }
        __syncthreads();
        const int n4 = n & ~3;
        for (int k = 4 * threadIdx.x; k < n4; k += 4 * kBlock) {
            IV c;
            TV d, o;
            if (out_A) c = *(const IV *)(idx32 + base + k);
            if (prod) d = *(const TV *)(data + base + k);
            if (out_A) {
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = b[c[v]];
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = s_a[k + v] * o[v];
                *(TV *)(out_A + base + k) = o;
            }
            if (prod) {
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = s_a[k + v] * d[v];
                *(TV *)(prod + base + k) = o;
            }
        }
        if (const int k = n4 + threadIdx.x; k < n) {
            if (out_A) out_A[base + k] = s_a[k] * b[idx32[base + k]];
            if (prod) prod[base + k] = s_a[k] * data[base + k];
        }
        __syncthreads();
    }
}

// quads of staged g (and x) per lane of the planned backward
template <int BLOCK> constexpr int kBwdXQ = (nm::kStageBwd * nm::kStageSeg / 4 + BLOCK - 1) / BLOCK;

// One tile of the planned backward, both gradients of a symmetric pattern, for a block of columns
// with a staging list and valid packed words: n entries, 1 <= n <= CAP, the first one at position
// `base` of the plan.  Like fwd_tile_staged it issues every request of the tile before its first
// wait, unconditionally (a request inside a branch makes the compiler's wait counts pessimistic:
// it then waits for nearly everything in flight), in the order in which the answers are needed
// (requests are answered in order), and as few vector memory instructions as the bytes allow: the
// listed segments of g and x a quad per lane, a column's two bounds with one request, the packed
// words of the first 1024 entries four consecutive entries per lane (QUAD; grad_A then leaves 16
// bytes per lane as well) and the rest in ER rounds of one entry per lane; only the values of A
// are gathered entry by entry.
template <typename T, int R, int CAP, bool O32, bool QUAD, int ER>
__device__ __forceinline__ void bwd_tile_staged(const int64_t c0, const int nc, const int32_t base, const int n,
                                                const int32_t lo0, const int32_t hi0, const int32_t lo1,
                                                const int32_t hi1, const bool seg2, const T *__restrict__ data,
                                                const int32_t *__restrict__ t_indptr,
                                                const int32_t *__restrict__ t_pack, const T *__restrict__ x,
                                                const T *__restrict__ g, T *__restrict__ grad_A,
                                                T *__restrict__ grad_x, T *s_v, T *s_g, T *s_x) {
    typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef int32_t I4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef int32_t I2 __attribute__((ext_vector_type(2), aligned(4)));
    constexpr int kQuads = QUAD ? 4 * kBlock : 0;       // entries of the quad phase
    static_assert(R == kBlock && nm::kStageSeg == 128, "lane = column, two segments per wavefront and request");
    static_assert(kBwdXQ<kBlock> == 2, "a list of at most sixteen places");
    const int tid = threadIdx.x;
    // Places eight and up of the list (seg2: the list has that many): the one request of the tile
    // that is not made every time.  It goes first: a request that may or may not have been made
    // only spoils the compiler's count of what is still in flight for the requests BEHIND it.
    TV gs1, xs1;
    const bool second = seg2 && 4 * (tid + kBlock) < nm::kStageBwd * nm::kStageSeg;
    if (seg2) {
        int32_t seg = (tid & 32) ? hi1 : lo1;
        seg = seg < 0 ? 0 : seg;
        const int64_t at0 = (int64_t)seg * nm::kStageSeg + 4 * (tid & 31);
        gs1 = *reinterpret_cast<const TV *>(g + at0);
        xs1 = *reinterpret_cast<const TV *>(x + at0);
    }
    // packed words
    I4 wq;
    if (QUAD) wq = __builtin_nontemporal_load(reinterpret_cast<const I4 *>(at<O32>(t_pack, base + tid * 4)));
    int32_t we[ER > 0 ? ER : 1];
#pragma unroll
    for (int r = 0; r < ER; ++r) {
        const int k = kQuads + r * kBlock + tid;
        we[r] = nm::stream_load(at<O32>(t_pack, base + (k < n ? k : n - 1)));
    }
    // the wavefront's two segments of places 0-7 (an unused place of the list loads segment 0)
    TV gs0, xs0;
    {
        // (separate scalars, not an array: the compiler turns a choice between array elements into
        // an indexed read of a copy of the array in scratch memory)
        int32_t seg = (tid & 32) ? hi0 : lo0;
        seg = seg < 0 ? 0 : seg;
        const int64_t at0 = (int64_t)seg * nm::kStageSeg + 4 * (tid & 31);
        gs0 = *reinterpret_cast<const TV *>(g + at0);
        xs0 = *reinterpret_cast<const TV *>(x + at0);
    }
    // bounds of column c0 + tid and the factor its entries share (the lane writes the mirror entry)
    int32_t pa, pb;
    if (nc == R) {
        const I2 pp = *reinterpret_cast<const I2 *>(t_indptr + c0 + tid);
        pa = pp[0], pb = pp[1];
    } else {
        pa = t_indptr[c0 + (tid < nc ? tid : nc)];
        pb = t_indptr[c0 + (tid + 1 < nc ? tid + 1 : nc)];
    }
    T own = g[c0 + (tid < nc ? tid : nc - 1)];
    // the values of A at the positions the packed words name
    T dq[4], de[ER > 0 ? ER : 1];
    if (QUAD) {
#pragma unroll
        for (int q = 0; q < 4; ++q) dq[q] = *at<O32>(data, base + tid * 4 + q + (wq[q] >> nm::kStagePlaceBits));
    }
#pragma unroll
    for (int r = 0; r < ER; ++r) {
        const int k = kQuads + r * kBlock + tid;
        const int kc = k < n ? k : n - 1;
        de[r] = *at<O32>(data, base + kc + (we[r] >> nm::kStagePlaceBits));
    }
    *reinterpret_cast<TV *>(s_g + 4 * tid) = gs0;
    *reinterpret_cast<TV *>(s_x + 4 * tid) = xs0;
    if (second) {       // (the list's last places: half a workgroup)
        *reinterpret_cast<TV *>(s_g + 4 * (tid + kBlock)) = gs1;
        *reinterpret_cast<TV *>(s_x + 4 * (tid + kBlock)) = xs1;
    }
    // (pinned: left alone, the compiler moves the request for `own` down into the branch that
    // uses it, behind the gathers)
    asm volatile("" : "+v"(own));
    if (tid < nc)
        for (int j = pa - base; j < pb - base; ++j) s_v[j] = own;
    __syncthreads();
    if (QUAD) {
        const int k = tid * 4;
        const TV sv = *reinterpret_cast<const TV *>(s_v + k);
        TV out, nv;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int li = wq[q] & ((1 << nm::kStagePlaceBits) - 1);
            out[q] = sv[q] * s_x[li];
            nv[q] = s_g[li] * dq[q];
        }
        *reinterpret_cast<TV *>(s_v + k) = nv;
        *reinterpret_cast<TV *>(at<O32>(grad_A, base + k)) = out;
    }
#pragma unroll
    for (int r = 0; r < ER; ++r) {
        const int k = kQuads + r * kBlock + tid;
        if (k < n) {
            const int li = we[r] & ((1 << nm::kStagePlaceBits) - 1);
            *at<O32>(grad_A, base + k) = s_v[k] * s_x[li];
            s_v[k] = s_g[li] * de[r];
        }
    }
    __syncthreads();
    // grad_x[column] = sum of the column's slice in ascending row order
    slice_sums<false, false>(s_v, pa - base, pb - base, tid < nc, grad_x + c0, tid);
}

// Backward over the transposed-structure plan (columns of A as rows of A^T):
// no atomics and no clearing of grad_x.  A workgroup owns R consecutive
// columns; lane p of the entry-parallel phase reads (row, position) of the
// p-th entry in column-major order and leaves g[row] * data[position] in LDS;
// one lane per column then adds its slice in ascending row order, the order in
// which the serial CPU loop accumulates grad_x (cpp/sparse_csr_cpu.cpp:68-73),
// so grad_x matches it bit for bit and is the same on every run.
//
// grad_A: in general entry p = (row r, column c) sits at `position` in A's
// arrays and grad_A[position] = g[r] * x[c] is a scattered store.  When the
// pattern is symmetric (plan flag) the column-major entry p is the mirror of the
// row-major entry p = (row c, column r), so the lane writes
// grad_A[p] = g[c] * x[r] instead: a coalesced store, every entry once.
// LISTS: the build for plans most of whose column blocks have a staging list (it keeps the listed
// segments of g and x in LDS).  The other build takes a block with a list through the plan's
// unpacked arrays (t_row, t_perm), which every plan holds, and needs no LDS for segments.
// (The resident wavefronts asked for are what each build reaches anyway; stating them changes the
// schedule the compiler picks, measured 4 M-row tridiagonal fp32 47.6 -> 40.8 us, 2048^2 five-point
// 61.4 -> 59.9 us.)
template <typename T, int R, int CAP, bool O32, bool LISTS>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? (LISTS ? 6 : 8) : (LISTS ? 3 : 7)))) void spmv_bwd_planned_kernel(
    int64_t cols, const T *__restrict__ data, const int32_t *__restrict__ t_indptr,
    const int32_t *__restrict__ t_row, const int32_t *__restrict__ t_perm, const int32_t *__restrict__ t_pack,
    const int32_t *__restrict__ flags, const T *__restrict__ x, const T *__restrict__ g,
    T *__restrict__ grad_A, T *__restrict__ grad_x, const int32_t *__restrict__ b_desc, int width) {
    static_assert(R == nm::kPackCols, "t_pack holds rows relative to the first column of a workgroup's block");
    static_assert(nm::kStageBwdCap <= CAP, "a block with a staging list fits the tile");
    constexpr bool STAGE = LISTS && NM_STAGE_BWD != 0;
    constexpr int kStaged = nm::kStageBwd * nm::kStageSeg;
    __shared__ int32_t s_off[R + 1];
    __shared__ __align__(16) T s_v[CAP];
    // the segments of g and of x that a block with a staging list names
    __shared__ __align__(16) T s_g[STAGE ? kStaged : 4];
    __shared__ __align__(16) T s_x[STAGE ? kStaged : 4];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool mirror = flags[0] != 0;
    // one packed word per entry in place of (t_row, t_perm): patterns near the diagonal
    const bool packed_plan = flags[1] != 0;
    static_assert(R == kBlock, "lane t of a workgroup stages column t of its block");
    const int rt = LISTS ? R : width;   // divides R
    const int64_t ntiles = (cols + rt - 1) / rt, npad = nm::xcd_padded(ntiles);
    const bool fused = mirror && grad_A;
    // the factor a column's entries share: g[column] (symmetric pattern: the lane writes the mirror
    // entry) or x[column]
    const T *__restrict__ own_of = grad_A ? (mirror ? g : x) : nullptr;
    const int tid = threadIdx.x;
    for (int64_t id = blockIdx.x; id < npad; id += gridDim.x) {
        const int64_t tile = nm::xcd_tile_reversed(id, npad);
        if (tile >= ntiles) continue;
        const int64_t c0 = tile * rt;
        const int nc = (int)(cols - c0 < rt ? cols - c0 : rt);
        const int32_t block0 = (int32_t)c0 & ~(R - 1);     // what packed rows are relative to
        bool packed = packed_plan;
        // (the low half of a packed word of a block with a list is a place in the listed segments)
        if constexpr (!STAGE) if (packed_plan && b_desc != nullptr) packed = b_desc[c0 / R * nm::kStageDesc] < 0;
        if constexpr (STAGE) if (fused && packed && b_desc != nullptr) {
            // a block of columns with a staging list, both gradients: the tile's ends, the head of
            // its list and the wavefront's four places of the list come together (scalar loads);
            // `live` is always true and only keeps those requests in front of the branch
            const int32_t *__restrict__ desc = b_desc + tile * nm::kStageDesc;
            const int32_t first = t_indptr[c0], n_all = t_indptr[c0 + nc] - first, d0 = desc[0];
            static_assert(kBwdXQ<kBlock> == 2, "two requests per lane cover the list");
            const int32_t lo0 = desc[2 * wave], hi0 = desc[2 * wave + 1];
            const int32_t lo1 = desc[kBlock / 32 + 2 * wave], hi1 = desc[kBlock / 32 + 2 * wave + 1];
            const bool live = (lo0 & hi0 & lo1 & hi1) != INT32_MIN;
            if ((d0 >= 0) & (n_all >= 4 * kBlock) & (n_all <= CAP) & live) {
                const bool seg2 = desc[8] >= 0;
#define NM_BWD_TILE(QUAD, ER)                                                                                       \
    bwd_tile_staged<T, R, CAP, O32, QUAD, ER>(c0, nc, first, n_all, lo0, hi0, lo1, hi1, seg2, data, t_indptr, t_pack, \
                                              x, g, grad_A, grad_x, s_v, s_g, s_x)
                // the first 1024 entries in quads where there are as many, the rest in rounds of 256
                // (the five-point block: quads and one round)
                static_assert(CAP == 8 * kBlock, "up to four rounds behind the quads");
                static_assert(nm::kStageBwdMin == 4 * kBlock, "a block with a list fills the quads");
                switch ((n_all - 4 * kBlock + kBlock - 1) / kBlock) {
                    case 0: NM_BWD_TILE(true, 0); break;
                    case 1: NM_BWD_TILE(true, 1); break;
                    case 2: NM_BWD_TILE(true, 2); break;
                    case 3: NM_BWD_TILE(true, 3); break;
                    default: NM_BWD_TILE(true, 4); break;
                }
#undef NM_BWD_TILE
                __syncthreads();
                continue;
            }
            // (a block with a list always has the entries that test asks for; were it ever not so,
            // its words must not be read as row offsets)
            if (d0 >= 0) packed = false;
        }
        // Lane t holds the bounds of column c0 + t and its own factor; all three loads leave
        // together (one memory round trip before the tile's entries can be read).
        const int32_t my_a = *at<O32>(t_indptr, (int32_t)c0 + (tid < nc ? tid : nc));
        const int32_t my_b = *at<O32>(t_indptr, (int32_t)c0 + (tid + 1 < nc ? tid + 1 : nc));
        const T my_own = own_of ? *at<O32>(own_of, (int32_t)c0 + (tid < nc ? tid : nc - 1)) : T(0);
        // A block of columns with a staging list (only made where the packed words are valid) keeps
        // in the low half of a packed word the place of the entry's row in the listed segments:
        // those segments of g (and of x, where the mirror entry is written) go to LDS, a quad per
        // lane and request.
        bool staged = false;
        if constexpr (STAGE) {
            typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
            constexpr int XQ = (kStaged / 4 + kBlock - 1) / kBlock;
            const int32_t *__restrict__ desc = b_desc + tile * nm::kStageDesc;
            // (both gradients of such a block were taken by bwd_tile_staged above)
            staged = !fused && packed && b_desc != nullptr && desc[0] >= 0;
            if (staged) {
                const bool want_x = mirror && grad_A != nullptr;
                TV gs[XQ], xs[XQ];
#pragma unroll
                for (int u = 0; u < XQ; ++u) {
                    const int f = tid + u * kBlock;
                    int32_t seg = desc[f < kStaged / 4 ? f / (nm::kStageSeg / 4) : 0];
                    seg = seg < 0 ? 0 : seg;
                    const int64_t at0 = (int64_t)seg * nm::kStageSeg + 4 * (f % (nm::kStageSeg / 4));
                    gs[u] = *reinterpret_cast<const TV *>(g + at0);
                    xs[u] = *reinterpret_cast<const TV *>((want_x ? x : g) + at0);
                }
#pragma unroll
                for (int u = 0; u < XQ; ++u) {
                    const int f = tid + u * kBlock;
                    if (f < kStaged / 4) {
                        *reinterpret_cast<TV *>(s_g + 4 * f) = gs[u];
                        *reinterpret_cast<TV *>(s_x + 4 * f) = xs[u];
                    }
                }
            }
        }
        // s_off[t] = first entry of column c0 + t in the plan (an absolute position), t = 0 .. nc
        s_off[tid] = my_a;
        if (tid == nc - 1) s_off[nc] = my_b;
        __syncthreads();
        const int32_t base = s_off[0];
        const int n = s_off[nc] - base;

        // s_v[j] = own[column] for the entries j of columns [s0, e0); o0 = offset of column s0.
        auto spread = [&](auto whole, const T *__restrict__ own, const int s0, const int e0, const int32_t o0) {
            constexpr bool WHOLE = decltype(whole)::value;
            for (int tb = s0; tb < e0; tb += kBlock) {
                const int t = tb + threadIdx.x;
                int jb, je;
                T v;
                if (WHOLE) {    // s0 == 0, e0 == nc <= kBlock: one pass, lane = column, all in registers
                    jb = t < e0 ? my_a - o0 : 0;
                    je = t < e0 ? my_b - o0 : 0;
                    v = my_own;
                } else {
                    jb = t < e0 ? s_off[t] - o0 : 0;
                    je = t < e0 ? s_off[t + 1] - o0 : 0;
                    v = t < e0 ? own[c0 + t] : T(0);
                }
                slice_fill(s_v, jb, je, v);
            }
        };
        // grad_x[column] = sum of the column's slice of s_v
        auto sums = [&](auto whole, const int s0, const int e0, const int32_t o0) {
            constexpr bool WHOLE = decltype(whole)::value;
            for (int tb = s0; tb < e0; tb += kBlock) {
                const int t = tb + threadIdx.x;
                const int jb = t < e0 ? (WHOLE ? my_a : s_off[t]) - o0 : 0;
                const int je = t < e0 ? (WHOLE ? my_b : s_off[t + 1]) - o0 : 0;
                slice_sums<false, !LISTS>(s_v, jb, je, t < e0, grad_x + c0, t);
            }
        };
        // Entries first .. first + cnt of the plan, lane = entry, s_v holding the own factor of
        // each: both gradients of a symmetric pattern -> every global access but the gathers of
        // g, x and data is a coalesced stream.
        auto entries_fused = [&](const int32_t first, const int cnt) {
            const int32_t *__restrict__ tr = t_row + first;
            const int32_t *__restrict__ tp = t_perm + first;
            T *__restrict__ ga = grad_A + first;
            // K entries in flight per lane: all their plan loads, then all their gathers, then
            // the stores -- two memory round trips per K entries.  Loads are unconditional on a
            // clamped position (a predicated load would sit in its own branch with its own wait).
            // Measured on the 2048 x 2048 Poisson matrix (5 entries per lane and tile), kernel time:
            // K = 2: 103 us, 4: 95 us, 5: 90 us, 6: 86 us, 8: 91 us.
            if (NM_BWD_VEC) {
                // a lane takes 4 consecutive entries per request: 16-byte loads of the two plan
                // streams and one 16-byte store of grad_A (aligned to 4 bytes only), U requests in flight
                typedef int32_t I4 __attribute__((ext_vector_type(4), aligned(4)));
                typedef T T4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
                constexpr int U = NM_BWD_VEC_U;
                const int c4 = cnt & ~3;
                for (int p0 = threadIdx.x * 4; p0 < c4; p0 += U * 4 * kBlock) {
                    I4 kk[U], rr[U];
                    T gg[U][4], xx[U][4], dd[U][4];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int pc = p0 + u * 4 * kBlock < c4 ? p0 + u * 4 * kBlock : c4 - 4;
                        kk[u] = __builtin_nontemporal_load(reinterpret_cast<const I4 *>(tp + pc));
                        rr[u] = __builtin_nontemporal_load(reinterpret_cast<const I4 *>(tr + pc));
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            gg[u][q] = g[rr[u][q]];
                            xx[u][q] = x[rr[u][q]];
                            dd[u][q] = data[kk[u][q]];
                        }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int p = p0 + u * 4 * kBlock;
                        if (p < c4) {
                            T4 out;
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                out[q] = s_v[p + q] * xx[u][q];
                                s_v[p + q] = gg[u][q] * dd[u][q];
                            }
                            *reinterpret_cast<T4 *>(ga + p) = out;
                        }
                    }
                }
                for (int p = c4 + threadIdx.x; p < cnt; p += kBlock) {
                    const int32_t k = tp[p], r = tr[p];
                    ga[p] = s_v[p] * x[r];
                    s_v[p] = g[r] * data[k];
                }
                return;
            }
            // (one entry fewer where every address takes a register pair, or the lanes spill)
            constexpr int K = O32 ? NM_BWD_K : NM_BWD_K - 1;
            for (int p0 = threadIdx.x; p0 < cnt; p0 += K * kBlock) {
                int32_t kk[K], rr[K];
                T gg[K], xx[K], dd[K];
                if (packed) {
#pragma unroll
                    for (int u = 0; u < K; ++u) {
                        const int pc = p0 + u * kBlock < cnt ? p0 + u * kBlock : cnt - 1;
                        const int32_t w = nm::stream_load(at<O32>(t_pack, first + pc));
                        kk[u] = first + pc + (w >> 16);
                        rr[u] = block0 + (int16_t)w;
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < K; ++u) {
                        const int pc = p0 + u * kBlock < cnt ? p0 + u * kBlock : cnt - 1;
                        kk[u] = nm::stream_load(at<O32>(t_perm, first + pc));
                        rr[u] = nm::stream_load(at<O32>(t_row, first + pc));
                    }
                }
#pragma unroll
                for (int u = 0; u < K; ++u) {
                    gg[u] = *at<O32>(g, rr[u]);
                    xx[u] = *at<O32>(x, rr[u]);
                    dd[u] = *at<O32>(data, kk[u]);
                }
                if (p0 + (K - 1) * kBlock < cnt) {
#pragma unroll
                    for (int u = 0; u < K; ++u) {
                        const int p = p0 + u * kBlock;
                        *at<O32>(grad_A, first + p) = s_v[p] * xx[u];
                        s_v[p] = gg[u] * dd[u];
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < K; ++u) {
                        const int p = p0 + u * kBlock;
                        if (p < cnt) {
                            *at<O32>(grad_A, first + p) = s_v[p] * xx[u];
                            s_v[p] = gg[u] * dd[u];
                        }
                    }
                }
            }
        };
        // The same for one gradient only or a pattern that is not symmetric; two entries a lane under way (one: 127 x
        // 113 x 101 seven-point, gradient of x, fp32 42.5 us, fp64 67.8; two 37.7 and 57.2; four 38.2 and 56.6, eight 41.5 and
        // 46.1; 2000 x 1980 five-point fp32 82, 78, 84 and 90).
        auto entries_any = [&](const int32_t first, const int cnt) {
            const int32_t *__restrict__ tr = t_row + first;
            const int32_t *__restrict__ tp = t_perm + first;
            constexpr int K = 2;
            for (int p0 = threadIdx.x; p0 < cnt; p0 += K * kBlock) {
                int32_t k[K], r[K];
                T gr[K], dd[K];
#pragma unroll
                for (int u = 0; u < K; ++u) {
                    const int p = p0 + u * kBlock < cnt ? p0 + u * kBlock : cnt - 1;
                    if (packed) {
                        const int32_t w = nm::stream_load(t_pack + first + p);
                        k[u] = first + p + ((STAGE && staged) ? w >> nm::kStagePlaceBits : w >> 16);
                        r[u] = (STAGE && staged) ? (w & ((1 << nm::kStagePlaceBits) - 1)) : block0 + (int16_t)w;
                    } else {
                        k[u] = nm::stream_load(tp + p);
                        r[u] = nm::stream_load(tr + p);
                    }
                }
#pragma unroll
                for (int u = 0; u < K; ++u) {
                    gr[u] = (STAGE && staged) ? s_g[r[u]] : g[r[u]];
                    dd[u] = data[k[u]];
                }
#pragma unroll
                for (int u = 0; u < K; ++u) {
                    const int p = p0 + u * kBlock;
                    if (p < cnt) {
                        if (grad_A) grad_A[k[u]] = gr[u] * s_v[p];
                        s_v[p] = gr[u] * dd[u];
                    }
                }
            }
        };
        // columns [s0, e0) through LDS
        auto run = [&](auto whole, const int s0, const int e0) {
            constexpr bool WHOLE = decltype(whole)::value;
            const int32_t o0 = WHOLE ? base : s_off[s0];
            const int cnt = s_off[e0] - o0;
            if (fused) {
                spread(whole, g, s0, e0, o0);
                __syncthreads();
                entries_fused(o0, cnt);
            } else {
                if (grad_A) {
                    spread(whole, own_of, s0, e0, o0);
                    __syncthreads();
                }
                entries_any(o0, cnt);
            }
            __syncthreads();
            sums(whole, s0, e0, o0);
        };

        if (n <= CAP) {
            run(std::true_type{}, 0, nc);
        } else if (n < kHuge) {
            for (int s0 = 0; s0 < nc;) {
                const int e0 = run_end(s_off, s0, nc, CAP);
                if (e0 > s0) {
                    run(std::false_type{}, s0, e0);
                    __syncthreads();
                    s0 = e0;
                    continue;
                }
                // a column longer than the tile, CAP entries at a time; wavefront 0 keeps the
                // lanes' partial sums (CAP is a multiple of 64: entry p stays with lane p % 64)
                const int32_t first = s_off[s0];
                const int len = s_off[s0 + 1] - s_off[s0];
                const T own = grad_A ? own_of[c0 + s0] : T(0);
                T acc = 0;
                for (int q0 = 0; q0 < len; q0 += CAP) {
                    const int cnt = len - q0 < CAP ? len - q0 : CAP;
                    if (grad_A) {
                        for (int j = threadIdx.x; j < cnt; j += kBlock) s_v[j] = own;
                        __syncthreads();
                    }
                    if (fused) entries_fused(first + q0, cnt); else entries_any(first + q0, cnt);
                    __syncthreads();
                    if (wave == 0)
                        for (int j = lane; j < cnt; j += kWave) acc += s_v[j];
                    __syncthreads();
                }
                if (wave == 0) {
                    acc = nm::wave_sum(acc);
                    if (lane == 0) grad_x[c0 + s0] = acc;
                }
                s0 += 1;
            }
        } else {
            for (int t = threadIdx.x; t < nc; t += kBlock) {
                const int32_t pb = t_indptr[c0 + t], pe = t_indptr[c0 + t + 1];
                if (pe - pb >= kLongRow) continue;
                const T xv = x[c0 + t];
                T acc = 0;
                for (int32_t p = pb; p < pe; ++p) {
                    const int32_t k = t_perm[p];
                    const T gr = g[t_row[p]];
                    if (grad_A) grad_A[k] = gr * xv;
                    acc += gr * data[k];
                }
                grad_x[c0 + t] = acc;
            }
            for (int t = wave; t < nc; t += kWavesPerBlock) {
                const int32_t pb = t_indptr[c0 + t], pe = t_indptr[c0 + t + 1];
                if (pe - pb < kLongRow) continue;
                const T xv = x[c0 + t];
                T acc = 0;
                for (int32_t p = pb + lane; p < pe; p += kWave) {
                    const int32_t k = t_perm[p];
                    const T gr = g[t_row[p]];
                    if (grad_A) grad_A[k] = gr * xv;
                    acc += gr * data[k];
                }
                acc = nm::wave_sum(acc);
                if (lane == 0) grad_x[c0 + t] = acc;
            }
        }
        __syncthreads();
    }
}

// set by nm_spgemv_configure: 64-bit offsets in the planned backward whatever the sizes (tests)
std::atomic<bool> g_wide_offsets{false};

int check_csr(int64_t rows, int64_t cols, int64_t nnz, const void *data, const int64_t *indices,
              const int64_t *indptr) {
    NM_REQUIRE(rows >= 0 && cols >= 0 && nnz >= 0, "negative size (rows=%lld cols=%lld nnz=%lld)",
               (long long)rows, (long long)cols, (long long)nnz);
    NM_REQUIRE(indptr != nullptr, "indptr is null");
    NM_REQUIRE(nnz == 0 || (data != nullptr && indices != nullptr), "data/indices null with nnz > 0");
    return NM_OK;
}

template <typename T, typename IDX, bool LISTS = false>
int launch_fwd(int64_t rows, int64_t nnz, const T *data, const IDX *indices, const IDX *indptr, const T *x,
               T *y, hipStream_t s, const int16_t *off16 = nullptr, const int32_t *flags = nullptr,
               const int32_t *f_desc = nullptr) {
    // (the build with lists reserves LDS for the listed segments anyway, which holds a CU to three
    // workgroups in fp64 whether the tile has 3072 or 4096 products: it takes the whole 4096, so
    // that blocks of 512 rows with seven entries a row stay blocks of 512 rows)
    constexpr int R = kFwdR, CAP = LISTS ? NM_FWD_CAP : kFwdCap<T>;
    // Long rows: tiles of about 1024 products (of 2048 or 4096, fp32 graphs of 200 000 rows, 20 entries each on average
    // 45 -> 56, 63 us; of 100 000 and 12, 15.6 -> 17.8, 22), without a plan and in fp64 1280 (1 M rows of 9, band 35.6 -> 32.1 us,
    // random the same; 1536: 29.7, but a graph of 400 000 rows of 10 38.0 -> 42.7).  Short ones: a tile of 512 rows reads the plan's packed
    // columns; without a plan at least 512 tiles (60 x 55 x 50 seven-point fp64 7.7 -> 5.9 us, with 1024 6.9; 30 x 35 x 30
    // 6.2 -> 4.4, with 1024 5.6).  On a plan whose columns are not packed, which only the device knows, at least 1024 (graphs, fp32,
    // of 512 rows a tile -> 512 -> 1024 tiles: 200 000 rows of 7 entries on average 26.2 -> 23.9 -> 19.4 us, 130 000 of 5 14.6 ->
    // 8.4 -> 8.1), and below 65 536 rows, where every column fits 16 bits, on any without lists (20 000 rows of 3 12.7 ->
    // 5.6, 10 000 of 7 10.8 -> 5.0; grids the same).
    // Long rows on a plan whose columns are packed (a band: neighbouring rows name the same part of x) want more a tile, from
    // 65 536 rows on, where packed means that: 1024 -> 3072 products, 400 000 rows of 35 fp64 54 -> 40 us, of 1 to 70 72 -> 55,
    // 1 M rows of 20 61 -> 53, fp32 41 -> 35 (2048: 43, 54, 55, 35); 100 000 rows of 16 fp64 7.2 -> 8.6.
    const bool long_rows = nnz > 8 * rows;
    constexpr bool kByPacking = sizeof(IDX) == 4 && !LISTS;
    auto at_least_512 = [&](int r) {
        while (r > 16 && rows < (int64_t)r * 512) r /= 2;
        return r;
    };
    int rt = block_rows(rows, nnz, R, long_rows ? (sizeof(T) == 8 && sizeof(IDX) == 8 ? 1280 : 1024) : CAP);
    if (long_rows || sizeof(IDX) == 8) rt = at_least_512(rt);
    int narrow = rt;
    if (kByPacking && long_rows) rt = at_least_512(block_rows(rows, nnz, R, 3072));
    if (kByPacking && !long_rows)
        while (narrow > 16 && rows < (int64_t)narrow * 1024) narrow /= 2;
    narrow = std::min(narrow, rt);
    int64_t grid = nm::xcd_padded(nm::ceil_div(rows, narrow));
    if (grid > nm::kMaxGrid) grid = nm::kMaxGrid;
    if (kByPacking) rt = (rows < (1 << 16) ? narrow : rt) | narrow << 16;
    hipLaunchKernelGGL((spmv_fwd_kernel<T, kFwdBlock, R, CAP, false, IDX, LISTS>), dim3((unsigned)grid), dim3(kFwdBlock), 0, s,
                       rows, rt, data, indices, indptr, x, y, off16, flags, f_desc);
    NM_LAUNCH_CHECK("spmv_fwd_kernel");
    return NM_OK;
}

template <typename T, typename IDX>
int launch_row_sum(int64_t rows, int64_t nnz, const T *data, const IDX *indptr, T *y, hipStream_t s) {
    constexpr int R = kFwdR, CAP = kFwdCap<T>;
    const int rt = small_block_rows(rows, nnz, R, CAP, 2048);
    int64_t grid = nm::xcd_padded(nm::ceil_div(rows, rt));
    if (grid > nm::kMaxGrid) grid = nm::kMaxGrid;
    hipLaunchKernelGGL((spmv_fwd_kernel<T, kFwdBlock, R, CAP, true, IDX>), dim3((unsigned)grid), dim3(kFwdBlock), 0, s, rows,
                       rt, data, (const IDX *)nullptr, indptr, (const T *)nullptr, y, (const int16_t *)nullptr,
                       (const int32_t *)nullptr, (const int32_t *)nullptr);
    NM_LAUNCH_CHECK("spmv_fwd_kernel<unit>");
    return NM_OK;
}

template <typename T>
int launch_bwd(int64_t rows, int64_t nnz, const T *data, const int64_t *indices, const int64_t *indptr, const T *a,
               const T *b, T alpha, T *out_A, T *grad_x, hipStream_t s) {
    constexpr int R = Tile<T>::R, CAP = Tile<T>::CAP;
    const int rt = small_block_rows(rows, nnz, R, CAP, !grad_x ? 2048 : nnz > 48 * rows ? CAP : 1024);
    int64_t grid = nm::xcd_padded(nm::ceil_div(rows, rt));
    if (grid > nm::kMaxGrid) grid = nm::kMaxGrid;
    if (grad_x)
        hipLaunchKernelGGL((spmv_bwd_kernel<T, R, CAP, true>), dim3((unsigned)grid), dim3(kBlock), 0, s, rows, rt,
                           data, indices, indptr, a, b, alpha, out_A, grad_x);
    else
        hipLaunchKernelGGL((spmv_bwd_kernel<T, R, CAP, false>), dim3((unsigned)grid), dim3(kBlock), 0, s, rows, rt, data,
                           indices, indptr, a, b, alpha, out_A, grad_x);
    NM_LAUNCH_CHECK("spmv_bwd_kernel");
    return NM_OK;
}

}  // namespace

extern "C" int nm_spgemv_forward(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                 const int64_t *indices, const int64_t *indptr, const void *x, void *y,
                                 nm_stream stream) {
    if (int rc = check_csr(rows, cols, nnz, data, indices, indptr)) return rc;
    if (rows == 0) return NM_OK;
    NM_REQUIRE(y != nullptr, "y is null");
    NM_REQUIRE(cols == 0 || x != nullptr, "x is null");
    hipStream_t s = nm::as_stream(stream);
    switch (dt) {
        case NM_F32:
            return launch_fwd<float, int64_t>(rows, nnz, (const float *)data, indices, indptr, (const float *)x,
                                              (float *)y, s);
        case NM_F64:
            return launch_fwd<double, int64_t>(rows, nnz, (const double *)data, indices, indptr, (const double *)x,
                                               (double *)y, s);
    }
    return nm::fail(NM_ERR_INVALID, "unknown dtype %d", (int)dt);
}

namespace {
int forward_planned(nm_dtype dt, bool lists, int64_t rows, int64_t cols, int64_t nnz, const void *data, const nm::TPlan &t,
                    const void *x, void *y, hipStream_t s) {
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(y != nullptr && (nnz == 0 || data != nullptr), "null pointer argument");
    NM_REQUIRE(cols == 0 || x != nullptr, "x is null");
    auto launch = [&](auto *one, auto with_lists) {
        using T = std::remove_pointer_t<decltype(one)>;
        return launch_fwd<T, int32_t, with_lists()>(rows, nnz, (const T *)data, t.c_idx32, t.c_ptr32, (const T *)x, (T *)y, s,
                                                    t.c_off16, t.flags, nnz > 0 ? t.f_desc : nullptr);
    };
    if (dt == NM_F32) return lists ? launch((float *)nullptr, std::true_type{}) : launch((float *)nullptr, std::false_type{});
    return lists ? launch((double *)nullptr, std::true_type{}) : launch((double *)nullptr, std::false_type{});
}

int forward_on_transpose_plan(nm_dtype dt, bool lists, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                              const void *plan_mem, const void *x, void *y, nm_stream stream) {
    NM_REQUIRE(rows >= 0 && cols >= 0 && nnz >= 0 && plan_mem != nullptr, "bad sizes or null plan");
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    if (rows == 0) return NM_OK;
    nm::TPlan t;
    nm::tplan_layout(rows, cols, nnz, const_cast<void *>(plan_mem), &t);
    return forward_planned(dt, lists, rows, cols, nnz, data, t, x, y, nm::as_stream(stream));
}

bool fits_rows_plan(int64_t rows, int64_t cols, int64_t nnz) {
    return rows >= 0 && cols >= 0 && nnz >= 0 && rows < 0x7ffffffe && cols < 0x7ffffffe && nnz < 0x7ffffffe;
}
}  // namespace

extern "C" int nm_spgemv_forward_planned(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                         const void *plan_mem, const void *x, void *y, nm_stream stream) {
    return forward_on_transpose_plan(dt, false, rows, cols, nnz, data, plan_mem, x, y, stream);
}

extern "C" int nm_spgemv_forward_planned_lists(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                               const void *plan_mem, const void *x, void *y, nm_stream stream) {
    return forward_on_transpose_plan(dt, true, rows, cols, nnz, data, plan_mem, x, y, stream);
}

extern "C" int nm_spgemv_rows_plan_bytes(int64_t rows, int64_t cols, int64_t nnz, size_t *plan_bytes) {
    NM_REQUIRE(plan_bytes != nullptr, "null output");
    if (!fits_rows_plan(rows, cols, nnz)) return nm::fail(NM_ERR_UNSUPPORTED, "plans index with 32 bits");
    *plan_bytes = nm::rows_plan_layout(rows, nnz, nullptr, nullptr);
    return NM_OK;
}

extern "C" int nm_spgemv_rows_plan_build(int64_t rows, int64_t cols, int64_t nnz, const int64_t *indices, const int64_t *indptr,
                                         void *plan_mem, size_t plan_bytes, int32_t info[16], nm_stream stream) {
    size_t need = 0;
    if (int rc = nm_spgemv_rows_plan_bytes(rows, cols, nnz, &need)) return rc;
    NM_REQUIRE(rows > 0 && nnz > 0, "an empty matrix");
    NM_REQUIRE(indices && indptr && plan_mem && info && plan_bytes >= need, "null pointer argument or plan memory too small");
    hipStream_t s = nm::as_stream(stream);
    nm::TPlan t;
    nm::rows_plan_layout(rows, nnz, plan_mem, &t);
    if (int rc = nm::rows_plan_build(rows, cols, nnz, indices, indptr, t, s)) return rc;
    NM_HIP_TRY(hipMemcpyAsync(info, t.flags, 16 * sizeof(int32_t), hipMemcpyDeviceToHost, s));
    NM_HIP_TRY(hipStreamSynchronize(s));
    return NM_OK;
}

extern "C" int nm_spgemv_forward_rows(nm_dtype dt, int lists, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                      const void *plan_mem, const void *x, void *y, nm_stream stream) {
    NM_REQUIRE(fits_rows_plan(rows, cols, nnz) && rows > 0 && nnz > 0 && plan_mem != nullptr, "bad sizes or null plan");
    nm::TPlan t;
    nm::rows_plan_layout(rows, nnz, const_cast<void *>(plan_mem), &t);
    return forward_planned(dt, lists != 0, rows, cols, nnz, data, t, x, y, nm::as_stream(stream));
}

extern "C" int nm_csr_row_sum_forward(nm_dtype dt, int64_t rows, int64_t nnz, const void *data,
                                      const int64_t *indptr, void *x, nm_stream stream) {
    NM_REQUIRE(rows >= 0 && nnz >= 0, "negative size");
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    if (rows == 0) return NM_OK;
    NM_REQUIRE(indptr && x && (nnz == 0 || data), "null pointer argument");
    hipStream_t s = nm::as_stream(stream);
    if (dt == NM_F32) return launch_row_sum<float, int64_t>(rows, nnz, (const float *)data, indptr, (float *)x, s);
    return launch_row_sum<double, int64_t>(rows, nnz, (const double *)data, indptr, (double *)x, s);
}

extern "C" int nm_spgemv_backward(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                  const int64_t *indices, const int64_t *indptr, const void *x,
                                  const void *g, void *grad_A, void *grad_x, nm_stream stream) {
    if (int rc = check_csr(rows, cols, nnz, data, indices, indptr)) return rc;
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    hipStream_t s = nm::as_stream(stream);
    if (grad_x) {
        int rc = dt == NM_F32 ? nm::fill_async((float *)grad_x, cols, 0.0f, s)
                              : nm::fill_async((double *)grad_x, cols, 0.0, s);
        if (rc) return rc;
    }
    if (rows == 0 || nnz == 0 || (!grad_A && !grad_x)) return NM_OK;
    NM_REQUIRE(g != nullptr && x != nullptr, "g or x is null");
    if (dt == NM_F32)
        return launch_bwd<float>(rows, nnz, (const float *)data, indices, indptr, (const float *)g,
                                 (const float *)x, 1.0f, (float *)grad_A, (float *)grad_x, s);
    return launch_bwd<double>(rows, nnz, (const double *)data, indices, indptr, (const double *)g,
                              (const double *)x, 1.0, (double *)grad_A, (double *)grad_x, s);
}

extern "C" int nm_masked_outer(nm_dtype dt, int64_t rows, int64_t nnz, const int64_t *indices,
                               const int64_t *indptr, double alpha, const void *a, const void *b, void *out,
                               nm_stream stream) {
    NM_REQUIRE(rows >= 0 && nnz >= 0 && indptr != nullptr, "bad sizes or null indptr");
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    if (rows == 0 || nnz == 0) return NM_OK;
    NM_REQUIRE(indices && a && b && out, "null pointer argument");
    hipStream_t s = nm::as_stream(stream);
    if (dt == NM_F32)
        return launch_bwd<float>(rows, nnz, nullptr, indices, indptr, (const float *)a, (const float *)b,
                                 (float)alpha, (float *)out, (float *)nullptr, s);
    return launch_bwd<double>(rows, nnz, nullptr, indices, indptr, (const double *)a, (const double *)b, alpha,
                              (double *)out, (double *)nullptr, s);
}

extern "C" int nm_spgemv_configure(int wide_offsets) {
    g_wide_offsets.store(wide_offsets != 0, std::memory_order_relaxed);
    return NM_OK;
}

namespace {
template <typename T, bool LISTS>
void launch_bwd_planned(int64_t cols, int64_t nnz, const nm::TPlan &t, bool o32, const void *data, const void *x,
                        const void *g, void *grad_A, void *grad_x, hipStream_t s) {
    constexpr int R = kPlannedR, CAP = kPlannedCap;
    // Columns of a tile: where they hold more than eight entries each and 256 at a time are fewer than 1024 tiles,
    // fewer (a power of two: a tile lies in one block of packed rows).  Graphs, both gradients, 256 -> this many:
    // 10 000 columns of 26 fp32 33.5 -> 8.0 us, fp64 37 -> 8.3; 30 000 of 18 23.4 -> 12.1 and 30.5 -> 17.0; 80 000 of 8 26.7
    // -> 18.2 (512 tiles: 20.7).  Columns of five: 30 x 35 x 30 the same.
    int width = R;
    if (!LISTS && nnz > 8 * cols)
        while (width > 16 && cols < (int64_t)width * 1024) width /= 2;
    int64_t grid = nm::xcd_padded(nm::ceil_div(cols, width));
    if (grid > nm::kMaxGrid) grid = nm::kMaxGrid;
    const int32_t *desc = nnz > 0 ? t.b_desc : nullptr;
    if (o32)
        hipLaunchKernelGGL((spmv_bwd_planned_kernel<T, R, CAP, true, LISTS>), dim3((unsigned)grid), dim3(kBlock), 0, s,
                           cols, (const T *)data, t.t_indptr, t.t_row, t.t_perm, t.t_pack, t.flags, (const T *)x,
                           (const T *)g, (T *)grad_A, (T *)grad_x, desc, width);
    else
        hipLaunchKernelGGL((spmv_bwd_planned_kernel<T, R, CAP, false, LISTS>), dim3((unsigned)grid), dim3(kBlock), 0, s,
                           cols, (const T *)data, t.t_indptr, t.t_row, t.t_perm, t.t_pack, t.flags, (const T *)x,
                           (const T *)g, (T *)grad_A, (T *)grad_x, desc, width);
}

// Tiles of 2048 entries (1 M rows of 12, band, fp32 / fp64, 1024 / 2048 / 4096 entries: 22.9, 19.7, 20.5 / 27.7, 27.0, 31.0
// us), of fewer where these were not 1024 tiles.
template <typename T>
int by_rows(int64_t rows, int64_t nnz, const nm::TPlan &t, const void *data, const void *x, const void *g, void *grad_A,
            void *prod, hipStream_t s) {
    constexpr int64_t kMost = 2048;
    const int64_t tile = std::min(kMost, std::max<int64_t>(256, (nnz / 1024 + 255) / 256 * 256));
    const int64_t grid = std::min<int64_t>(nm::xcd_padded(nm::ceil_div(nnz, tile)), nm::kMaxGrid);
    hipLaunchKernelGGL((spmv_bwd_entries_kernel<T, 1024, kMost>), dim3((unsigned)grid), dim3(kBlock), 0, s, rows, nnz, (int)tile, (const T *)data,
                       t.c_idx32, t.c_ptr32, t.chunk_row, (const T *)g, (const T *)x, (T *)grad_A, (T *)prod);
    NM_LAUNCH_CHECK("spmv_bwd_entries_kernel");
    return NM_OK;
}

// Scattered columns: the kernel on the plan alone gathers a value and writes a gradient per entry, each a cache line
// from beyond L2.  Here both stay in row-major order, and only the products are brought into column-major order, with
// coalesced requests: 400 000 rows, 7.6 M entries, fp32, 304 -> 121 us, of which 50 the walk by rows (it
// waits for x from L2), 48 the two passes of the permutation, 10 the sums.
template <typename T>
int backward_staged(int64_t rows, int64_t cols, int64_t nnz, const nm::TPlan &t, const nm::PermutePlan &p, void *work,
                    const void *data, const void *x, const void *g, void *grad_A, void *grad_x, hipStream_t s) {
    T *const one = (T *)work, *const two = (T *)((char *)work + nm::align256((size_t)nnz * sizeof(T)));
    if (int rc = by_rows<T>(rows, nnz, t, data, x, g, grad_A, one, s)) return rc;
    if (int rc = nm::to_columns<T>(p, nnz, one, two, one, s)) return rc;
    return launch_row_sum<T, int32_t>(cols, nnz, one, t.t_indptr, (T *)grad_x, s);
}

template <bool LISTS>
int backward_planned(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data, const void *plan_mem,
                     const void *x, const void *g, void *grad_A, void *grad_x, nm_stream stream) {
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(rows >= 0 && cols >= 0 && nnz >= 0 && plan_mem != nullptr, "bad sizes or null plan");
    if (cols == 0 || (!grad_A && !grad_x)) return NM_OK;
    NM_REQUIRE(nnz == 0 || (data && x && g), "null pointer argument");
    nm::TPlan t;
    nm::tplan_layout(rows, cols, nnz, const_cast<void *>(plan_mem), &t);
    hipStream_t s = nm::as_stream(stream);
    if (!grad_x) {
        if (rows == 0 || nnz == 0) return NM_OK;
        if (dt == NM_F32) return by_rows<float>(rows, nnz, t, data, x, g, grad_A, nullptr, s);
        return by_rows<double>(rows, nnz, t, data, x, g, grad_A, nullptr, s);
    }
    // every array the kernel indexes stays below 4 GiB: 32-bit byte offsets
    const int64_t longest = std::max(std::max(rows, cols) + 2, nnz + 1);
    const bool o32 = !g_wide_offsets.load(std::memory_order_relaxed) && longest * (dt == NM_F32 ? 4 : 8) < (int64_t(1) << 32);
    if (dt == NM_F32) launch_bwd_planned<float, LISTS>(cols, nnz, t, o32, data, x, g, grad_A, grad_x, s);
    else launch_bwd_planned<double, LISTS>(cols, nnz, t, o32, data, x, g, grad_A, grad_x, s);
    NM_LAUNCH_CHECK("spmv_bwd_planned_kernel");
    return NM_OK;
}
}  // namespace

extern "C" int nm_spgemv_backward_planned(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                          const void *plan_mem, const void *x, const void *g, void *grad_A,
                                          void *grad_x, nm_stream stream) {
    return backward_planned<false>(dt, rows, cols, nnz, data, plan_mem, x, g, grad_A, grad_x, stream);
}

extern "C" int nm_spgemv_backward_planned_lists(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz,
                                                const void *data, const void *plan_mem, const void *x,
                                                const void *g, void *grad_A, void *grad_x, nm_stream stream) {
    return backward_planned<true>(dt, rows, cols, nnz, data, plan_mem, x, g, grad_A, grad_x, stream);
}

extern "C" int nm_spgemv_staged_bytes(nm_dtype dt, int64_t nnz, size_t *bytes) {
    NM_REQUIRE(dt == NM_F32 || dt == NM_F64, "unknown dtype %d", (int)dt);
    NM_REQUIRE(nnz >= 0 && nnz < 0x7ffffffe && bytes, "nnz outside a plan's range or null output");
    *bytes = 2 * nm::align256((size_t)nnz * (dt == NM_F32 ? 4 : 8));
    return NM_OK;
}

extern "C" int nm_spgemv_backward_staged(nm_dtype dt, int64_t rows, int64_t cols, int64_t nnz, const void *data,
                                         const void *transpose_plan, const void *permute_plan, void *work, size_t work_bytes,
                                         const void *x, const void *g, void *grad_A, void *grad_x, nm_stream stream) {
    size_t need = 0;
    if (int rc = nm_spgemv_staged_bytes(dt, nnz, &need)) return rc;
    NM_REQUIRE(rows > 0 && cols > 0 && nnz > 0, "an empty matrix");
    NM_REQUIRE(rows < 0x7ffffffe && cols < 0x7ffffffe, "size outside a plan's range");
    NM_REQUIRE(data && transpose_plan && permute_plan && work && x && g && grad_x, "null pointer argument");
    NM_REQUIRE(work_bytes >= need, "work memory too small");
    nm::TPlan t;
    nm::tplan_layout(rows, cols, nnz, const_cast<void *>(transpose_plan), &t);
    nm::PermutePlan p;
    nm::permute_layout(nnz, const_cast<void *>(permute_plan), &p);
    hipStream_t s = nm::as_stream(stream);
    if (dt == NM_F32) return backward_staged<float>(rows, cols, nnz, t, p, work, data, x, g, grad_A, grad_x, s);
    return backward_staged<double>(rows, cols, nnz, t, p, work, data, x, g, grad_A, grad_x, s);
}
