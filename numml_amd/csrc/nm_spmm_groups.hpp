// CSR x dense with a dense operand of up to 1 KB a row: several entries of A per request.
//
// What bounds these products is the rows of the dense operand that the entries name.  With uniformly
// random columns every entry fetches its row from beyond L2, and this part delivers about 57 cache
// lines (128 bytes) a nanosecond from there, whether a line is wanted whole or by half: 15.6 M rows
// of 256 bytes take 535 us, of 128 bytes 287, of 64 bytes 275.  A kernel reaches that only if it
// asks for rows fast enough.  With lane = dense column (the kernels of nm_spmm.hip) an entry costs
// the compute unit one request of ~16 cycles and a wavefront some eight instructions however narrow
// the operand is: 520 us at 16 columns, where the lines would allow 275.
//
// Here a group of G lanes takes an entry, V = 16 bytes of its row a lane, so that a wavefront's
// request covers 64 / G entries.  Every group walks its own rows of A and adds each row's terms in
// storage order, like the serial loop (cpp/sparse_csr_cpu.cpp:586-598): same bits.  The groups of a
// workgroup draw rows from a counter in LDS, so one that has a longer row holds nobody up.  Rows of
// more than kShared entries are left to the workgroups at the head of the grid, which look for them and
// share each one among all their groups (or, where they find many, deal them to their groups): up to kSplit entries the
// products meet in LDS and are added in storage order, beyond that chunks of 16 entries are summed and the sums added in
// order (deterministic, the serial sum up to rounding).
//
// The walk gives out[r, :] = sum of value * dense[index, :] over the entries of row r and, with DOT,
// dots[position] = <dense[index, :], own[r, :]>: the backward by column needs the same row of gC for
// grad_B and for grad_A.  Dot products alone go by entry (dots_kernel).
//
// Measured on graphs with power-law rows and uniformly random columns, forward / backward with both gradients, against
// lane = column: 1 M rows, 15.6 M entries, fp32: 64 columns 637 -> 608 / 1007 -> 696 us (the rows' lines
// alone take 535, index, values and result 60 more), 16 columns 524 -> 321 / 747 -> 416; fp64, 16 columns 690 -> 355 / 975 -> 583.
// 100 000 rows of mean 15, 64 columns fp32 97 -> 73.  Lane = column is the better one for rows of one to three entries of
// 33 to 64 values (100 000 rows of one, fp64, 48 columns: 16 -> 22) and for fp64 rows of 48 to 64 values where a few
// rows have thousands of entries (0.5 M rows, 20 M entries, 48 columns: 1067 -> 1300, the backward 1450 -> 1310).
#pragma once

#include "nm_common.hpp"

namespace nm_groups {

using nm::kWave;
constexpr int kThreads = 256;
// Rows of more than kShared entries are shared by the groups of a workgroup, up to kSplit entries with
// their terms in storage order.  (Taken by one group each up to 512 entries, such rows kept the rest of
// their workgroup waiting: 957 against 650 us.  From 65 entries on: 655 us; from 33: 745.)
constexpr int kShared = 128, kSplit = 512;
// Where kAlone eighths of the rows that a workgroup looks through have kShared to kSplit entries, its groups take one each:
// there long rows are the rule and none keeps the others waiting, while sharing costs two barriers a turn and one group's addition.
// Rows of 140 to 500 entries throughout, fp32, us, lane = column / all shared / this: 100 000 rows of 140, 16 columns 334 / 446 /
// 126, 64 columns 449 / 956 / 262; 30 000 of 500, 64 columns 474 / 745 / 200; 3000 of 200, 64 columns 120 / 104 / 24.  (30 000
// rows, of 16: from 3 or 4 on power-law rows up to 1000 entries take 50 instead of 26 us at 16 columns; from 12 on rows of 0 to 280
// 236 instead of 157 at 64.  kShared at 192: power-law rows up to 1000 entries 15 % slower.)  Rows around kShared are
// the least gain: 30 000 of 90 +- 30, 64 columns, lane = column / this: fp32 111 / 103, fp64 169 / 195.
constexpr int kAlone = 3;
constexpr int kChunk = 16;         // entries of a row a group takes from memory at once
constexpr int kPass = 4;           // entries of a shared row a group takes at once where their order counts
// A matrix of few rows leaves compute units free while one workgroup after the other is at work on the
// longest rows: there a workgroup looks through fewer rows, and a shared row's result is cut into slices of
// 128 bytes (kSliceLanes lanes), a workgroup each, which has more of the row's entries in flight (60 000 rows,
// up to 10 000 entries, 64 columns: 205 -> 89 us).  Where the chip is full anyway slices only cost
// (1 M rows of 37 columns: 650 -> 785 us, the slices of a row share lines).
// (In the slices a group takes kSliceBatch rows of the operand at once.  With eight the walk of the other rows, which
// shares the kernel's registers, had five wavefronts a SIMD instead of seven: 100 000 rows of 5, 64 columns fp32 31 -> 27 us,
// of 35 120 -> 95.)
constexpr int kSliceLanes = 8, kSliceBatch = 4;
// Workgroups at the head of the grid, slices included, that look for long rows: a matrix without any has them for nothing,
// while few of them have one long row after the other.  2048 fill the chip once.  (2048 before slices, up to 12 500 with
// them: 100 000 rows of one, fp64, 48 columns 26 -> 22 us; 1024: 200 000 rows of 4 and 256 neighbours of 500, 64 columns fp32 57 -> 96.)
constexpr int64_t kFewBlocks = 2048, kFewRows = 64;
constexpr int kScan = kThreads;    // rows a workgroup at the head of the grid looks through,
// in kPlaces places far apart, so that neighbouring long rows (a sorted graph, a block of dense rows) get workgroups
// of their own: with 256 neighbours a workgroup one had them all.  fp32, 64 columns, rows of 4 entries and among them 256
// neighbours of 500: 1 M rows 4930 -> 255 us, 200 000 rows 1330 -> 57; power-law rows in descending order, 200 000: 4840 -> 330.
// (A row by itself each: a line of row pointers a row, 1 M rows of 12 entries 242 -> 248 us at 16 columns.)
constexpr int kPlaces = 32;
constexpr int kDrawRows = 4;       // rows of a workgroup per group: enough to draw from, few enough that the
                                   // rows of `own` (16 KB) leave room for eight workgroups a compute unit.
// Fewer, down to one, where a matrix has too few for kFewBlocks workgroups: four rows one after the other took 10 000 rows
// of 60, both gradients of 16 columns, fp32 84 us (157 workgroups on 256 compute units; lane = column 63) and take 25 side by side;
// 30 000 rows of 20, 33 columns 41 -> 33, 100 000 rows of 20, 16 columns 76 -> 68.

// V consecutive elements at an address that need only suit one of them
template <typename T, int V> struct Vec { typedef T type __attribute__((ext_vector_type(V), aligned(sizeof(T)))); };
template <typename T> struct Vec<T, 1> { typedef T type; };
template <typename T, int V> struct Held { typedef T type __attribute__((ext_vector_type(V))); };   // the same in LDS
template <typename T> struct Held<T, 1> { typedef T type; };
template <typename T, int V> __device__ __forceinline__ T part(const typename Vec<T, V>::type &v, int i) {
    if constexpr (V == 1) return v; else return v[i];
}

template <typename T, typename IDX> struct Args {
    int64_t rows;             // rows that are walked (columns of A on the transposed structure)
    const IDX *ptr, *idx;
    const int32_t *perm;      // PERM: where an entry's value is and its dot product goes
    const T *data;
    const T *dense;           // gathered rows
    int64_t ld;
    int n;
    T *out;
    int64_t ldo;
    const T *own;             // DOT: row r belongs to walked row r
    int64_t ldw;
    T *dots;
    int scan_rows;            // rows each of the workgroups that look for long rows looks through
    int stripe;               // neighbours among these, as a power of two
    int64_t scan_sets;        // parts the rows are dealt into for that
    unsigned scan_blocks;     // workgroups that look for long rows, a multiple of nm::kXcds
    unsigned tiles;           // workgroups that walk rows, the same
    int tile_rows;            // rows each of these walks
};

// Sum over the G lanes of a group, in every one of them and with the same bits in each (every step adds
// two lanes' sums that are added the other way round in the other lane).
template <int G, typename T> __device__ __forceinline__ T group_total(T v) {
    v += nm::dpp_move<0xB1>(v);                          // quad_perm [1,0,3,2]
    v += nm::dpp_move<0x4E>(v);                          // quad_perm [2,3,0,1]
    if constexpr (G >= 8) v += nm::dpp_move<0x141>(v);   // row_half_mirror: the other quad of the 8
    if constexpr (G >= 16) v += nm::dpp_move<0x140>(v);  // row_mirror: the other 8 of the 16
    if constexpr (G >= 32) v += __shfl_xor(v, 16, kWave);
    if constexpr (G == 64) v += __shfl_xor(v, 32, kWave);
    return v;
}

template <typename T, int V, int G, typename IDX, bool PERM, bool DOT, int BATCH = (G >= 32 ? 4 : 8)>
struct Walker {
    static constexpr int kGroups = kThreads / G, kRows = kGroups * kDrawRows;
    // rows of the dense operand in flight at once: with 16 too few wavefronts fit (936 against 650 us)
    static constexpr int kBatch = BATCH;
    static constexpr int kHeld = G < kChunk ? kChunk / G : 1;   // entries of a chunk a lane holds
    static constexpr int kWidth = V;
    static constexpr bool kDot = DOT;
    using value = T;
    using vec = typename Vec<T, V>::type;
    using held = typename Held<T, V>::type;

    const Args<T, IDX> &a;
    int l, first;          // lane of the group, the group's first lane
    int c0;                // first column of the lane (the last lane's are moved back to end at n)
    bool live;             // the lane has columns of its own
    int fresh;             // the lane's first column that the lane before has not
    const char *dense_c;
    uint32_t row_bytes;
    T dot[kHeld];          // dot products of the entries the lane holds

    // (slice: the columns from slice * G * V on)
    __device__ __forceinline__ Walker(const Args<T, IDX> &args, int slice = 0) : a(args) {
        const int lane = threadIdx.x & (kWave - 1);
        l = lane & (G - 1);
        first = lane & ~(G - 1);
        const int c = (slice * G + l) * V;
        live = c < a.n;
        c0 = c + V <= a.n ? c : a.n - V;
        fresh = c - c0;
        dense_c = reinterpret_cast<const char *>(a.dense + c0);
        row_bytes = (uint32_t)(a.ld * (int64_t)sizeof(T));
    }
    // entries [kc, kc + cnt) of the chunk, cnt >= 1; places beyond them hold the last one
    struct Chunk {
        uint32_t col[kHeld];
        T val[kHeld];
        int32_t pos[kHeld];
    };
    __device__ __forceinline__ void load(Chunk &c, int64_t kc, int cnt) const {
#pragma unroll
        for (int h = 0; h < kHeld; ++h) {
            const int e = h * G + l;
            const int64_t k = kc + (e < cnt ? e : cnt - 1);
            // (kept in the caches: the rows of other groups lie in the same lines.  Streamed past them: 30 000 rows of 140,
            // 16 columns fp32 48 instead of 32 us, 100 000 rows of 35, 24 columns 90 instead of 75)
            c.col[h] = (uint32_t)a.idx[k];
            if constexpr (PERM) c.pos[h] = a.perm[k];
            if constexpr (!PERM) c.val[h] = a.data[k];
        }
        if constexpr (PERM) {
#pragma unroll
            for (int h = 0; h < kHeld; ++h) c.val[h] = a.data[c.pos[h]];
        }
    }
    __device__ __forceinline__ vec gather(const Chunk &c, int e) const {
        const uint32_t col = (uint32_t)__shfl((int)c.col[e / G], first + e % G, kWave);
        return *reinterpret_cast<const vec *>(dense_c + (uint64_t)col * row_bytes);
    }
    __device__ __forceinline__ void add(const Chunk &c, int e, const vec &b, T (&acc)[V]) const {
        const T x = __shfl(c.val[e / G], first + e % G, kWave);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] += x * part<T, V>(b, v);
    }
    __device__ __forceinline__ vec product(const Chunk &c, int e, const vec &b) const {
        return __shfl(c.val[e / G], first + e % G, kWave) * b;
    }
    __device__ __forceinline__ T product_sum(const vec &b, const vec &mine) const {
        T p[V];
#pragma unroll
        for (int v = 0; v < V; ++v) p[v] = live && v >= fresh ? part<T, V>(b, v) * part<T, V>(mine, v) : T(0);
        T s = p[0];
        if constexpr (V == 2) s = p[0] + p[1];
        if constexpr (V == 4) s = (p[0] + p[1]) + (p[2] + p[3]);
        return group_total<G>(s);
    }
    __device__ __forceinline__ void multiply(int e, const vec &b, const vec &mine) {
        const T s = product_sum(b, mine);
        if (l == e % G) dot[e / G] = s;
    }
    __device__ __forceinline__ void store_dots(const Chunk &c, int64_t kc, int cnt) const {
#pragma unroll
        for (int h = 0; h < kHeld; ++h) {
            const int e = h * G + l;
            if (e < cnt && e < kChunk) a.dots[PERM ? (int64_t)c.pos[h] : kc + e] = dot[h];
        }
    }
    static __device__ __forceinline__ vec pack(const T (&acc)[V]) {
        vec o;
        if constexpr (V == 1) {
            o = acc[0];
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) o[v] = acc[v];
        }
        return o;
    }
    __device__ __forceinline__ void store_row(int64_t row, const T (&acc)[V]) const {
        // (past the caches, which the rows of `dense` need: 1 M rows of one, 64 columns fp64 213 -> 190 us, 2 M rows of 12, 48
        // columns 1652 -> 1611, 10 000 rows and more never slower)
        if (live) nm::stream_store(reinterpret_cast<vec *>(a.out + row * a.ldo + c0), pack(acc));
    }
    __device__ __forceinline__ vec own_row(int64_t row) const {
        return *reinterpret_cast<const vec *>(a.own + row * a.ldw + c0);
    }
};

// Places 0 .. nr - 1 of a workgroup's rows, each walked by one group in storage order.  The groups draw places from the
// counter `next`; the first one of each is its own number r.  open(r, row, kc, e, mine) tells whether the row at r is to be
// walked, and fills in the row, its entries and (DOT) its row of `own`.  A turn of the loop takes a chunk of every
// group's row, whatever the rows' lengths.
template <typename W, typename OPEN> __device__ __forceinline__ void walk_rows(W &w, int r, int nr, int *next, OPEN open) {
    using T = typename W::value;
    using vec = typename W::vec;
    constexpr int V = W::kWidth, kBatch = W::kBatch;
    constexpr bool DOT = W::kDot;
    typename W::Chunk c;
    int64_t row = 0, kc = 0, e = 0;
    T acc[V] = {};
    vec mine{};
    auto draw = [&]() {
        int drawn = 0;
        if (w.l == 0) drawn = atomicAdd(next, 1);
        r = __shfl(drawn, w.first, kWave);
    };
    auto begin = [&]() {
        for (; r < nr; draw()) {
            if (!open(r, row, kc, e, mine)) continue;
#pragma unroll
            for (int v = 0; v < V; ++v) acc[v] = T(0);
            return;
        }
    };
    begin();
    while (r < nr) {
        const int cnt = (int)(e - kc < kChunk ? e - kc : kChunk);
        w.load(c, kc, cnt);
#pragma unroll
        for (int j0 = 0; j0 < kChunk; j0 += kBatch) {
            if (j0 < cnt) {
                vec d[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) d[u] = w.gather(c, j0 + u);
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    if (j0 + u < cnt) {
                        w.add(c, j0 + u, d[u], acc);
                        if constexpr (DOT) w.multiply(j0 + u, d[u], mine);
                    }
                }
            }
        }
        if constexpr (DOT) w.store_dots(c, kc, cnt);
        kc += cnt;
        if (kc == e) {
            w.store_row(row, acc);
            draw();
            begin();
        }
    }
}

template <typename T, int V, int G, typename IDX, bool PERM, bool DOT, bool SLICED>
__global__ __launch_bounds__(kThreads, 5) void groups_kernel(const Args<T, IDX> a) {
    using W = Walker<T, V, G, IDX, PERM, DOT>;
    using vec = typename W::vec;
    constexpr int kGroups = W::kGroups, kRows = W::kRows;
    __shared__ int64_t s_ptr[kRows + 1];
    // the walked rows' rows of `own`; in the workgroups that share rows: products, partial sums
    __shared__ typename W::held s_mem[(DOT ? kRows * G : 1) > kThreads * kPass ? kRows * G : kThreads * kPass];
    typename W::held *const s_own = s_mem, *const s_pass = s_mem;
    __shared__ int s_list[kScan], s_found[2];
    __shared__ int s_next;
    const int t = threadIdx.x;

    if (blockIdx.x < a.scan_blocks) {
        // ---- rows of more than kShared entries, each shared by the groups of the workgroup ----
        // (sums alone: a workgroup takes 128 bytes of the row's result, so that wide operands have
        // more workgroups and more entries at once on a row; a dot product wants the whole row)
        constexpr int GS = SLICED ? kSliceLanes : G, kGroups = kThreads / GS;
        using WS = Walker<T, V, GS, IDX, PERM, DOT, SLICED ? kSliceBatch : W::kBatch>;
        using Chunk = typename WS::Chunk;
        constexpr int kBatch = WS::kBatch;
        const int slices = SLICED ? (a.n + GS * V - 1) / (GS * V) : 1;
        WS w(a, SLICED ? blockIdx.x % slices : 0);
        const int g = t / GS;
        const int64_t set = blockIdx.x / slices;
        auto row_of = [&](int place) { return (((place >> a.stripe) * a.scan_sets + set) << a.stripe) + (place & ((1 << a.stripe) - 1)); };
        // (listed from the front: up to kSplit entries; from the back: more)
        if (t == 0) {
            s_next = kGroups;
            s_found[0] = s_found[1] = 0;
        }
        __syncthreads();
        if (t < a.scan_rows && set < a.scan_sets) {
            const int64_t row = row_of(t);
            const int64_t n = row < a.rows ? (int64_t)(a.ptr[row + 1] - a.ptr[row]) : 0;
            if (n > kSplit) s_list[kScan - 1 - atomicAdd(&s_found[1], 1)] = t;
            else if (n > kShared) s_list[atomicAdd(&s_found[0], 1)] = t;
        }
        __syncthreads();
        int split = s_found[0];
        const int longer = s_found[1];
        if (split * 8 >= a.scan_rows * kAlone) {
            walk_rows(w, g, split, &s_next, [&](int r, int64_t &row, int64_t &kc, int64_t &e, vec &mine) {
                row = row_of(s_list[r]);
                kc = a.ptr[row];
                e = a.ptr[row + 1];
                if constexpr (DOT) mine = w.own_row(row);
                return true;
            });
            split = 0;
        }
        for (int i = 0; i < split + longer; ++i) {   // (the order of the list does not matter)
            const int64_t row = row_of(s_list[i < split ? i : kScan - 1 - (i - split)]), b = a.ptr[row], e = a.ptr[row + 1];
            T acc[V] = {};
            vec mine{};
            if constexpr (DOT) mine = w.own_row(row);
            Chunk c, later;
            if (e - b <= kSplit) {
                // every group takes four entries of a pass; their products meet in LDS, where one group
                // adds them up in storage order
                auto mine_of = [&](int64_t base) {   // entries of the pass at `base` that are this group's
                    const int64_t left = e - base - g * kPass;
                    return (int)(left < kPass ? left : kPass);
                };
                if (mine_of(b) > 0) w.load(c, b + g * kPass, mine_of(b));
                for (int64_t base = b; base < e; base += kGroups * kPass) {
                    const int cnt = mine_of(base), next = mine_of(base + kGroups * kPass);
                    if (next > 0) w.load(later, base + kGroups * kPass + g * kPass, next);
                    if (cnt > 0) {
                        vec d[kPass];
#pragma unroll
                        for (int u = 0; u < kPass; ++u) d[u] = w.gather(c, u);
#pragma unroll
                        for (int u = 0; u < kPass; ++u) {
                            if (u < cnt) {
                                s_pass[(g * kPass + u) * GS + w.l] = w.product(c, u, d[u]);
                                if constexpr (DOT) w.multiply(u, d[u], mine);
                            }
                        }
                        if constexpr (DOT) w.store_dots(c, base + g * kPass, cnt);
                    }
                    __syncthreads();
                    if (g == 0) {
                        const int all = (int)(e - base < kGroups * kPass ? e - base : kGroups * kPass);
#pragma unroll 4
                        for (int j = 0; j < all; ++j) {
                            const vec p = s_pass[j * GS + w.l];
#pragma unroll
                            for (int v = 0; v < V; ++v) acc[v] += part<T, V>(p, v);
                        }
                    }
                    __syncthreads();
                    c = later;
                }
                if (g == 0) w.store_row(row, acc);
                continue;
            }
            // longer ones: a chunk of entries a group and pass, whose sums are added in the order of the
            // chunks (so the bits do not depend on how many groups there are)
            constexpr int64_t kStep = (int64_t)kGroups * kChunk;
            auto count = [&](int64_t kc) { return (int)(e - kc < kChunk ? e - kc : kChunk); };
            int64_t kc = b + (int64_t)g * kChunk;
            if (kc < e) w.load(c, kc, count(kc));
            for (int64_t base = b; base < e; base += kStep, kc += kStep) {
                if (kc + kStep < e) w.load(later, kc + kStep, count(kc + kStep));
                if (kc < e) {
                    const int cnt = count(kc);
                    T sum[V] = {};
#pragma unroll
                    for (int j0 = 0; j0 < kChunk; j0 += kBatch) {
                        vec d[kBatch];
#pragma unroll
                        for (int u = 0; u < kBatch; ++u) d[u] = w.gather(c, j0 + u);
#pragma unroll
                        for (int u = 0; u < kBatch; ++u) {
                            if (j0 + u < cnt) {
                                w.add(c, j0 + u, d[u], sum);
                                if constexpr (DOT) w.multiply(j0 + u, d[u], mine);
                            }
                        }
                    }
                    if constexpr (DOT) w.store_dots(c, kc, cnt);
                    s_pass[t] = WS::pack(sum);
                }
                {
                    __syncthreads();
                    if (g == 0) {
                        const int64_t left = (e - base + kChunk - 1) / kChunk;
                        const int all = (int)(left < kGroups ? left : kGroups);
#pragma unroll 4
                        for (int j = 0; j < all; ++j) {
                            const vec p = s_pass[j * GS + w.l];
#pragma unroll
                            for (int v = 0; v < V; ++v) acc[v] += part<T, V>(p, v);
                        }
                    }
                    __syncthreads();
                }
                c = later;
            }
            if (g == 0) w.store_row(row, acc);
        }
        return;
    }

    // ---- all other rows, drawn by the groups one at a time ----
    W w(a);
    const int g = t / G;
    const int64_t r0 = nm::xcd_tile(blockIdx.x - a.scan_blocks, a.tiles) * a.tile_rows;
    if (r0 >= a.rows) return;
    const int nr = (int)(a.rows - r0 < a.tile_rows ? a.rows - r0 : a.tile_rows);
    for (int i = t; i <= nr; i += kThreads) s_ptr[i] = (int64_t)a.ptr[r0 + i];
    if constexpr (DOT) {
        for (int i = g; i < nr; i += kGroups) s_own[i * G + w.l] = w.own_row(r0 + i);
    }
    if (t == 0) s_next = kGroups;
    __syncthreads();
    walk_rows(w, g, nr, &s_next, [&](int r, int64_t &row, int64_t &kc, int64_t &e, vec &mine) {
        row = r0 + r;
        kc = s_ptr[r];
        e = s_ptr[r + 1];
        if (e == kc) {
            const T zero[V] = {};
            w.store_row(row, zero);
            return false;
        }
        if (e - kc > kShared) return false;
        if constexpr (DOT) mine = s_own[r * G + w.l];
        return true;
    });
}

// Dot products alone: dots[k] = <dense[idx[k], :], own[row of k, :]>, by entry and not by row, since nothing is
// added up over a row (one row may hold all entries).  A wavefront takes 64 consecutive entries, lane l entry
// l: it finds that entry's row among the ends of the next 64 rows; a group then takes its lanes' entries one
// after the other, a request a side, and every lane keeps its own entry's product (in the order of
// groups_kernel: same bits).  `chunk_row`, when given, holds the row of every 64th entry.
template <typename T, int V, int G>
__global__ __launch_bounds__(kThreads) void dots_kernel(const Args<T, int64_t> a, int64_t nnz, const int32_t *__restrict__ chunk_row) {
    using W = Walker<T, V, G, int64_t, false, true>;
    using vec = typename W::vec;
    constexpr int kFlight = G < 8 ? G : 8;
    const W w(a);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t chunk = (int64_t)blockIdx.x * (kThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t kb = chunk * kWave;
    if (kb >= nnz) return;
    const int64_t k = kb + lane < nnz ? kb + lane : nnz - 1;
    const uint32_t mycol = (uint32_t)nm::stream_load(a.idx + k);
    auto row_of = [&](int64_t entry, int64_t lo) {   // the last row r >= lo - 1 with ptr[r] <= entry
        int64_t hi = a.rows + 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (a.ptr[mid] <= entry) lo = mid + 1; else hi = mid;
        }
        return lo - 1;
    };
    const int64_t row0 = chunk_row ? (int64_t)chunk_row[chunk] : row_of(kb, 0);
    const int64_t end = row0 + 1 + lane;
    const int64_t my_end = a.ptr[end <= a.rows ? end : a.rows];
    int lo = 0, hi = kWave;
#pragma unroll
    for (int step = 0; step < 7; ++step) {   // 65 possible answers: seven halvings
        const int mid = (lo + hi) >> 1;      // == 64 only once lo == hi == 64: the read is ignored then
        const int64_t e = __shfl(my_end, mid & (kWave - 1), kWave);
        if (lo < hi) {
            if (e <= k) lo = mid + 1; else hi = mid;
        }
    }
    // (more than 64 rows that end inside the chunk: empty ones)
    const uint32_t myrow = (uint32_t)(lo == kWave ? row_of(k, row0 + lo) : row0 + lo);
    const char *const own_c = reinterpret_cast<const char *>(a.own + w.c0);
    const uint32_t own_bytes = (uint32_t)(a.ldw * (int64_t)sizeof(T));
    T dot = T(0);
#pragma unroll 1
    for (int s0 = 0; s0 < G; s0 += kFlight) {
        vec d[kFlight], o[kFlight];
#pragma unroll
        for (int u = 0; u < kFlight; ++u) {
            const uint32_t c = (uint32_t)__shfl((int)mycol, w.first + s0 + u, kWave), r = (uint32_t)__shfl((int)myrow, w.first + s0 + u, kWave);
            d[u] = *reinterpret_cast<const vec *>(w.dense_c + (uint64_t)c * w.row_bytes);
            o[u] = *reinterpret_cast<const vec *>(own_c + (uint64_t)r * own_bytes);
        }
#pragma unroll
        for (int u = 0; u < kFlight; ++u) {
            const T s = w.product_sum(d[u], o[u]);
            if (w.l == s0 + u) dot = s;
        }
    }
    if (kb + lane < nnz) a.dots[kb + lane] = dot;
}

// The widest dense operand these kernels take: 64 lanes of 16 bytes.
template <typename T> constexpr int64_t most_columns() { return kWave * (16 / (int64_t)sizeof(T)); }

// Whether a product may go this way: indices that fit 32 bits and row strides that fit them in bytes.
// (`own_rows`, `ldw`: of the operand the dot products are with)
template <typename T> bool takes(int64_t indexed, int64_t ld, int64_t n, int64_t own_rows = 0, int64_t ldw = 0) {
    return n >= 1 && n <= most_columns<T>() && indexed <= 0x7fffffff && own_rows <= 0x7fffffff &&
           ld * (int64_t)sizeof(T) <= 0xffffffffll && ldw * (int64_t)sizeof(T) <= 0xffffffffll;
}

template <typename T, int V, int G, typename IDX, bool PERM, bool DOT>
int launch_shape(Args<T, IDX> a, hipStream_t s) {
    constexpr int kGroups = kThreads / G;
    a.tile_rows = kGroups * kDrawRows;
    while (a.tile_rows > kGroups && nm::ceil_div(a.rows, a.tile_rows) < kFewBlocks) a.tile_rows /= 2;
    constexpr bool kMaySlice = !DOT && G > kSliceLanes;
    const bool sliced = kMaySlice && nm::ceil_div(a.rows, kFewRows) < kFewBlocks;
    const int64_t slices = sliced ? nm::ceil_div(a.n, kSliceLanes * V) : 1;
    // rows a workgroup at the head of the grid looks through: few where the matrix has few, since it takes
    // the long ones that it finds one after the other
    a.scan_rows = kScan;
    while (a.scan_rows > 16 && nm::ceil_div(a.rows, a.scan_rows) * slices < kFewBlocks) a.scan_rows /= 2;
    a.scan_sets = nm::ceil_div(a.rows, a.scan_rows);
    a.stripe = 0;
    while ((kPlaces << a.stripe) < a.scan_rows) ++a.stripe;
    const int64_t scan = nm::xcd_padded(a.scan_sets * slices), tiles = nm::xcd_padded(nm::ceil_div(a.rows, a.tile_rows));
    NM_REQUIRE(scan + tiles <= 0x7fffffff, "too many rows");
    a.scan_blocks = (unsigned)scan;
    a.tiles = (unsigned)tiles;
    const dim3 grid((unsigned)(scan + tiles));
    if constexpr (kMaySlice) {
        if (sliced) {
            hipLaunchKernelGGL((groups_kernel<T, V, G, IDX, PERM, DOT, true>), grid, dim3(kThreads), 0, s, a);
            NM_LAUNCH_CHECK("groups_kernel");
            return NM_OK;
        }
    }
    hipLaunchKernelGGL((groups_kernel<T, V, G, IDX, PERM, DOT, false>), grid, dim3(kThreads), 0, s, a);
    NM_LAUNCH_CHECK("groups_kernel");
    return NM_OK;
}

// f(std::integral_constant<int, V>, std::integral_constant<int, G>) for a dense operand of n columns
template <typename T, typename F> int by_width(int n, F f) {
    constexpr int V = 16 / (int)sizeof(T);
    using Wide = std::integral_constant<int, V>;
    if (n < V) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
    if (n <= 4 * V) return f(Wide{}, std::integral_constant<int, 4>{});
    if (n <= 8 * V) return f(Wide{}, std::integral_constant<int, 8>{});
    if (n <= 16 * V) return f(Wide{}, std::integral_constant<int, 16>{});
    if (n <= 32 * V) return f(Wide{}, std::integral_constant<int, 32>{});
    return f(Wide{}, std::integral_constant<int, 64>{});
}

// out = sums of rows of `dense`, with DOT dots as well
template <typename T, typename IDX, bool PERM, bool DOT> int launch(const Args<T, IDX> &a, hipStream_t s) {
    if (a.rows == 0) return NM_OK;
    return by_width<T>(a.n, [&](auto v, auto g) { return launch_shape<T, v(), g(), IDX, PERM, DOT>(a, s); });
}

template <typename T> int launch_dots(const Args<T, int64_t> &a, int64_t nnz, const int32_t *chunk_row, hipStream_t s) {
    const int64_t grid = nm::ceil_div(nnz, (int64_t)kThreads);
    NM_REQUIRE(grid <= 0x7fffffff, "too many entries");
    return by_width<T>(a.n, [&](auto v, auto g) {
        hipLaunchKernelGGL((dots_kernel<T, v(), g()>), dim3((unsigned)grid), dim3(kThreads), 0, s, a, nnz, chunk_row);
        NM_LAUNCH_CHECK("dots_kernel");
        return (int)NM_OK;
    });
}

}  // namespace nm_groups
