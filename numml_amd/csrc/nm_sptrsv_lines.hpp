// Triangular solves on a grid's lines.
//
// The triangle of a five-point or seven-point matrix in the grid's own order (and its transpose): a row
// depends on the row before it in each direction of the grid.  (An upper triangle is a lower one with
// the rows numbered from the end.)  Level by level such a solve pays a barrier or a hand-over between compute
// units per level, several times what a row's arithmetic takes.  Here a lane is a LINE of the grid: a
// wavefront takes a patch of up to 64 lines (64 of a plane; 8 x 8 of a volume) and lane (a, b) solves
// row t - 2 a - b of its line at step t, so that
//   * the row before in the line is the lane's own last result, in a register;
//   * the row before along b is what the lane to the left found a step ago (a DPP move), along a what the lane
//     eight to the left found two steps ago, a trip to LDS with a step to spare: no barrier;
//   * only a patch's first lanes wait for other workgroups.  These leave the rows of a patch's last lines in
//     an `edge`: one 64-bit word a row that holds kUnsolved until the row is solved (never torn, so there is
//     no flag and no fence).
// Patches are drawn from a counter in an order in which none waits for a later one: whatever part of
// the launch is on the chip gets on.  Waits are bounded all the same (NaN throughout, as elsewhere).
//
// A pass over the whole chip (28.5 us of 1 M rows, 92 MB: half the rate of a copy, since lanes next to each other read rows of
// different lines) first puts the call's values where the
// wavefronts read them: entry (p, lane) of a patch holds the row that the lane is at in the steps t = p (mod
// length), so the arrays are as long as the matrix has rows, and a step reads 40 or 48 bytes a lane, coalesced.
//
// The division is the hardware's own sequence (reciprocal, two refinements, quotient, remainder,
// quotient) with the first half, which knows the diagonal only, done in that pass.  The sequence is valid as it
// stands where nothing has to be scaled: the pass leaves NaN for a diagonal outside 2^-128 .. 2^128, and a quotient
// outside 2^-800 .. 2^800 (a zero, an infinity, NaN among them) is looked for once a block of eight steps.  (The
// remainder's last bit is then 2^-128-800-104 at least, so none of the sequence is rounded as a denormal.)
// The wavefront goes on with divisions in full at a block that has such a quotient, 90 ns a step instead of 68, and
// returns to the short ones after sixteen blocks that have none.  Zeros are what it meets in earnest: the
// rows ahead of the first right-hand side that is not zero.  us with a dense right-hand side, with zeros
// throughout, and that level by level (a wavefront that made such blocks again one by one and always
// tried the short division first: the figure in brackets): 1024 x 1024 fp64 209, 281 (684), 700;
// 97 x 89 x 101 120, 136 (284), 325; 300 x 70 38, 54 (119), 104; 64 x 64 18, 21 (44), 37.
//
// Sums run in double in the serial loop's order (cpp/sparse_csr_cpu.cpp:672-718: the farthest dependency
// first), a dependency that is not there adding a zero product to a sum that is never -0: the same bits.
//
// What bounds it: a step is ~24 instructions of one wavefront, 68 ns (the arithmetic's chain alone is 28 ns; three
// loads, the store to LDS and the DPP moves are the rest), and 2-3 us a hand-over between patches.  64 x 4096 rows
// 282 us, 68 ns a level where a workgroup with a barrier a level takes 270; fp64, ms before and now: 1024 x 1024
// 0.70 and 0.21, 60 x 60 0.036 and 0.018, 97 x 89 x 101 0.325 and 0.12, 16 x 16 x 16 0.031 and 0.021, 300^3
// 2.17 and 1.68.
#pragma once
#include "nm_common.hpp"

#include <type_traits>

namespace {
namespace lines {

constexpr int kAhead = 16;         // steps that operands are requested ahead
// Steps of a block, after which a wavefront looks at what the others have done (four: 64 x 4096 282 -> 330 us, and no
// more than 2 % off what hands over most, 97 x 89 x 101).
constexpr int kBlockSteps = 8;
constexpr int kFullBlocks = 16;    // blocks without a quotient that needs it for which the division in full is kept up
constexpr int kPatch = 8;          // lines of a patch in either direction of a volume
constexpr int kSkewPlane = 2;      // steps from a line to the one of the next plane
constexpr unsigned long long kUnsolved = ~0ull;   // a NaN; a result with these bits is handed on as the default NaN
constexpr unsigned kSafeDiag = 128, kSafeQuotient = 800;   // exponents

// A grid in the roles that its directions have here: lines run along one of them, a patch's lanes b (neighbours a step
// apart) and a (kSkewPlane steps apart) lie along the others.
struct Grid {
    int32_t length = 0;            // rows of a line; 0: the pattern is not a grid's
    int32_t width = 0, planes = 0; // lines along b, along a (1: two dimensions)
    int32_t along = 0, across = 0, apart = 0;   // distance between rows along a line, along b, along a
    int32_t role[3] = {};          // of the directions by ascending distance: 0 the line's, 1 b, 2 a
    int32_t ah = 0, bw = 0;        // a patch: lines along a, along b
    int32_t ni = 0, nj = 0;        // patches along a, along b
    __host__ __device__ int64_t edge_n() const { return (int64_t)(nj - 1) * planes * length; }
    __host__ __device__ int64_t edges() const { return edge_n() + (int64_t)(ni - 1) * width * length; }
    __host__ __device__ int32_t row(int32_t i, int32_t j, int32_t c) const { return i * apart + j * across + c * along; }
};

// The grid whose rows are `step` apart in its second direction and, `far` > 0, `far` in its third; false where these do
// not divide up the rows.  Lines go the way that is expected to take the least: 85 ns a step from the first row to the
// last, 2.3 us a hand-over between patches (96 x 16 x 16: lines of 16 rows 57 us, of 96 rows 29 us).  The sum of three
// products is the serial one as long as the nearest row's is added last (the first two may change places),
// so rows next to each other are a line's or b's.
inline bool make_grid(int64_t rows, int64_t step, int64_t far, Grid *out) {
    if (step < 2 || rows % step != 0 || (far > 0 && (far % step != 0 || rows % far != 0 || far <= step))) return false;
    const int64_t size[3] = {step, (far > 0 ? far : rows) / step, far > 0 ? rows / far : 1}, apart[3] = {1, step, far};
    static const int roles[4][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}};   // of the three directions
    double best = 1e300;
    for (int way = 0; way < (far > 0 ? 4 : 3); ++way) {
        if (far == 0 && way == 1) continue;
        Grid g;
        for (int d = 0; d < 3; ++d) {
            g.role[d] = roles[way][d];
            (g.role[d] == 0 ? g.length : g.role[d] == 1 ? g.width : g.planes) = (int32_t)size[d];
            (g.role[d] == 0 ? g.along : g.role[d] == 1 ? g.across : g.apart) = (int32_t)apart[d];
        }
        if (g.length < 2 || g.length >= 1 << 20) continue;   // (a patch's operands are addressed with 31 bits)
        auto cut = [](int32_t n, int32_t most, int32_t *each, int32_t *count) {
            *count = (n + most - 1) / most;
            *each = (n + *count - 1) / *count;
            *count = (n + *each - 1) / *each;
        };
        cut(g.planes, kPatch, &g.ah, &g.ni);
        cut(g.width, far > 0 ? kPatch : 64, &g.bw, &g.nj);
        const double ns = 85. * (g.length + (double)kSkewPlane * g.planes + g.width) + 2300. * (g.ni + g.nj);
        if (ns < best) {
            best = ns;
            *out = g;
        }
    }
    return best < 1e300;
}

// Steps that line (a, b) of a patch runs behind its first one.
__device__ __forceinline__ int32_t skew(int32_t a, int32_t b) { return kSkewPlane * a + b; }

struct Patch {
    int32_t I, J, i0, j0, na, nb;   // its place, its first plane and line, how many of either
    int32_t base;                   // its first entry in the arrays by (p, lane)
};
__device__ __forceinline__ Patch patch_of(const Grid &g, int32_t id) {
    Patch p;
    p.I = id / g.nj;
    p.J = id - p.I * g.nj;
    p.i0 = p.I * g.ah;
    p.j0 = p.J * g.bw;
    p.na = min(g.ah, g.planes - p.i0);
    p.nb = min(g.bw, g.width - p.j0);
    p.base = (p.i0 * g.width + p.na * p.j0) * g.length;
    return p;
}
// out[0]: the smallest distance of a dependency above 1, out[1]: the largest
__global__ __launch_bounds__(256) void reach_kernel(int32_t rows, const int32_t *__restrict__ order,
                                                    const int32_t *__restrict__ dptr,
                                                    const int32_t *__restrict__ dslot, int32_t *out) {
    int32_t least = 0x7fffffff, most = 0;
    for (int32_t q = blockIdx.x * 256 + threadIdx.x; q < rows; q += gridDim.x * 256)
        for (int32_t at = dptr[q]; at < dptr[q + 1]; ++at) {
            const int32_t d = abs(order[q] - order[dslot[at]]);
            if (d > 1) least = min(least, d);
            most = max(most, d);
        }
    for (int off = 32; off > 0; off >>= 1) {
        least = min(least, __shfl_xor(least, off, 64));
        most = max(most, __shfl_xor(most, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        if (least < out[0]) atomicMin(out, least);
        if (most > out[1]) atomicMax(out + 1, most);
    }
}

// Raises `bad` unless every row has exactly the dependencies of its place in the grid, farthest first.  src[r], r the row's
// number in the solve's direction: where the coefficients on the rows before along a, along b and of the line are stored,
// and the diagonal (-1: none).
__global__ __launch_bounds__(256) void plan_kernel(Grid g, int32_t rows, int mirrored, const int32_t *__restrict__ order,
                                                   const int32_t *__restrict__ dptr,
                                                   const int32_t *__restrict__ dslot,
                                                   const int32_t *__restrict__ dsrc, const int32_t *__restrict__ diag,
                                                   int4 *__restrict__ src, int32_t *bad) {
    bool wrong = false;
    for (int32_t q = blockIdx.x * 256 + threadIdx.x; q < rows; q += gridDim.x * 256) {
        const int32_t row = order[q], r = mirrored ? rows - 1 - row : row;
        int32_t at = dptr[q], rest = r, of[3] = {-1, -1, -1};   // by role
        const int32_t end = dptr[q + 1];
        for (int d = 2; d >= 0; --d) {
            const int32_t role = g.role[d], apart = role == 0 ? g.along : role == 1 ? g.across : g.apart;
            if (apart == 0 || rest < apart) continue;   // no such direction, or no row before
            rest %= apart;
            if (at < end && order[dslot[at]] == (mirrored ? row + apart : row - apart)) {
                const int32_t from = dsrc[at++];
                if (role == 0) of[0] = from;
                else if (role == 1) of[1] = from;
                else of[2] = from;
            } else {
                wrong = true;
            }
        }
        wrong = wrong || at != end;
        src[r] = int4{of[2], of[1], of[0], diag[q]};
    }
    if (__any(wrong) && (threadIdx.x & 63) == 0) *bad = 1;
}

template <typename T> struct Args {
    Grid g;
    int32_t rows, mirrored, unit;
    const int4 *src;
    const T *data, *b;
    T *x;
    double2 *near;      // by entry: coefficient on the line before, on the row before
    double2 *rd;        // right-hand side, diagonal
    double *y;          // two dimensions: refined reciprocal; three: (reciprocal, coefficient on the plane before)
    unsigned long long *edge;
    int32_t *status;    // [0]: somebody gave up waiting; [1]: patches drawn
    int64_t poll_limit;
};

template <typename T, bool THREE> __global__ __launch_bounds__(256) void gather_kernel(Args<T> k) {
    const int64_t first = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
    const int64_t all = (int64_t)gridDim.x * gridDim.y * 256;
    if (first < 2) k.status[first] = 0;
    for (int64_t e = first; e < k.g.edges(); e += all) k.edge[e] = kUnsolved;
    const int32_t patches = k.g.ni * k.g.nj, length = k.g.length;
    for (int32_t id = blockIdx.y; id < patches; id += gridDim.y) {
        const Patch P = patch_of(k.g, id);
        const int32_t w = P.na * P.nb;
        for (int32_t e = blockIdx.x * 256 + threadIdx.x; e < w * length; e += gridDim.x * 256) {
            const int32_t p = e / w, lane = e - p * w, a = THREE ? lane / P.nb : 0, b = lane - a * P.nb;
            int32_t c = p - skew(a, b) % length;
            if (c < 0) c += length;
            const int32_t r = k.g.row(P.i0 + a, P.j0 + b, c);
            const int64_t at = (int64_t)P.base + e;
            const int4 s = k.src[r];
            k.near[at] = double2{s.y >= 0 ? (double)k.data[s.y] : 0., s.z >= 0 ? (double)k.data[s.z] : 0.};
            const double d = k.unit ? 1. : s.w >= 0 ? (double)k.data[s.w] : 0.;
            k.rd[at] = double2{(double)k.b[k.mirrored ? k.rows - 1 - r : r], d};
            const unsigned exponent = (unsigned)__double2hiint(d) >> 20 & 0x7ffu;
            double y = __builtin_amdgcn_rcp(d);
            y = __builtin_fma(y, __builtin_fma(-d, y, 1.), y);
            y = __builtin_fma(y, __builtin_fma(-d, y, 1.), y);
            if (exponent - (1023u - kSafeDiag) > 2u * kSafeDiag) y = __longlong_as_double(0x7ff8000000000000ll);
            if (THREE) reinterpret_cast<double2 *>(k.y)[at] = double2{y, s.x >= 0 ? (double)k.data[s.x] : 0.};
            else k.y[at] = y;
        }
    }
}

// How far the wavefronts of a workgroup are, in steps.
struct Progress {
    int32_t imported;   // steps whose imports are in LDS
    int32_t exported;   // steps whose results are in the edges
    int32_t written;    // steps whose results are in x
    int32_t done;       // steps solved
};
constexpr int32_t kAll = 0x40000000;
constexpr int kKept = 64;       // steps whose results, and whose imports, stay in LDS (a power of two)
// x: by step and lane, ahead of the lanes in a row what the first plane's lines need in the step after the
// next, so that entry `lane` of a row is the line of the plane before's for every lane (73: a line's steps lie in banks
// of their own).
struct Shared {
    union { Progress now; int4 all; };
    int32_t patch;
    double x[kKept][kPatch + 64 + 1];
    double from_n[kKept][kPatch];   // by step and plane: what the planes' first lines need
};
__device__ __forceinline__ unsigned long long look(const unsigned long long *at) {
    return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void leave(unsigned long long *at, double v) {
    unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    if (bits == kUnsolved) bits = 0x7ff8000000000000ull;
    __hip_atomic_store(at, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wavefront 0: the steps.  It waits for memory on account of its operands only, which come in the order they are
// asked for; whatever takes another time to come or go is the other three wavefronts' business.  A step is
// bound by what one wavefront issues (8 cycles an instruction), so everything that does not change from
// step to step is kept out of it.
// LINE_LAST: the row before of the line is the nearest, whose product the serial sum adds last; else b's is.
template <typename T, bool THREE, bool LINE_LAST> __device__ __forceinline__ void solve_patch(const Args<T> &k, const Patch &P, Shared &sh) {
    struct Operands { double2 near, rd; double y, far; };
    const int lane = threadIdx.x & 63;
    const int32_t length = k.g.length, w = P.na * P.nb, deepest = skew(P.na - 1, P.nb - 1), steps = length + deepest;
    const int a0 = THREE ? lane / kPatch : 0, b0 = THREE ? lane % kPatch : lane;
    const bool valid = a0 < P.na && b0 < P.nb;
    const int32_t depth = valid ? skew(a0, b0) : 0x40000000;
    constexpr int kWidthY = THREE ? 16 : 8;
    const int32_t bytes = w * length * 16;
    auto resource = [&](const double *from, int width) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(from) + (int64_t)P.base * width), (short)0,
                                                 bytes / 16 * width, 0x00027000);
    };
    const auto near = resource(reinterpret_cast<const double *>(k.near), 16), rd = resource(reinterpret_cast<const double *>(k.rd), 16),
               y = resource(k.y, kWidthY);
    const int32_t mine = valid ? a0 * P.nb + b0 : 0;
    auto request_at = [&](Operands &o, int32_t place) __attribute__((always_inline)) {
        o.near = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(near, mine * 16, place, 0));
        o.rd = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rd, mine * 16, place, 0));
        if (THREE) {
            const double2 yf = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(y, mine * 16, place, 0));
            o.y = yf.x;
            o.far = yf.y;
        } else {
            o.y = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(y, mine * 8, place >> 1, 0));
            o.far = 0.;
        }
    };
    int32_t place = 0;
    auto request = [&](Operands &o) __attribute__((always_inline)) {
        request_at(o, place);
        place += w * 16;
        place = place == bytes ? 0 : place;
    };
    Operands o[kAhead];
    double x = 0.;
    uint32_t worst = 0;   // of the block's quotients: how far from the smallest exponent that is safe
    auto step = [&](Operands &v, double import_n, double xg, int32_t t, double *keep, auto ramp, auto in_full) __attribute__((always_inline)) {
        // (one wait for all of a step's operands)
        asm volatile("" : "+v"(v.near.x), "+v"(v.near.y), "+v"(v.rd.x), "+v"(v.rd.y), "+v"(v.y));
        if (THREE) asm volatile("" : "+v"(v.far));
        const long long xi = __double_as_longlong(x), in = __double_as_longlong(import_n);
        constexpr int left = THREE ? 0x111 : 0x138;   // row_shr:1, wave_shr:1: the lane to the left's
        const int lo = __builtin_amdgcn_update_dpp((int)in, (int)xi, left, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp((int)(in >> 32), (int)(xi >> 32), left, 0xf, 0xf, false);
        double xn = __longlong_as_double((long long)hi << 32 | (unsigned)lo);
        if (THREE) xn = b0 == 0 ? import_n : xn;
        // (a product and +0: the sum starts at +0 in the serial loop, which makes a -0 of the first product +0)
        double acc;
        if constexpr (!THREE) acc = __builtin_fma(v.near.x, xn, 0.) + v.near.y * x;
        else if constexpr (LINE_LAST) acc = __builtin_fma(v.far, xg, 0.) + v.near.x * xn + v.near.y * x;
        else acc = __builtin_fma(v.far, xg, 0.) + v.near.y * x + v.near.x * xn;
        const double n = v.rd.x - acc;
        bool live = true;
        if constexpr (ramp) live = (uint32_t)(t - depth) < (uint32_t)length;
        double q = in_full ? n / v.rd.y : n * v.y;
        int high = __double2hiint(q);
        asm volatile("" : "+v"(high));
        const uint32_t off = ((uint32_t)high << 1) - ((1023u - kSafeQuotient) << 21);
        worst = max(worst, live ? off : 0u);
        if constexpr (!in_full) q = __builtin_fma(__builtin_fma(-v.rd.y, q, n), v.y, q);
        x = live ? q : 0.;
        *keep = x;
        // The lane of the next plane reads this from its own `lane`, an address that the compiler can prove is never the
        // one stored to here: it must not move that load ahead of the store.  (97 x 89 x 101 119.0 -> 119.7 us, which
        // other ways of saying so cost as well: a wavefront release 120.0, an address it knows nothing of 119.9.)
        if constexpr (THREE) asm volatile("" ::: "memory");
    };
    constexpr int kSteps = kBlockSteps, kRow = kPatch + 64 + 1;
    int4 progress = int4{0, 0, 0, 0};
    double import_n[2][kSteps];   // of this block and of the next one, in turn
    // how far the others are, and then the imports of the block at t
    auto ask = [&](int32_t t, double (&n)[kSteps]) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        progress = sh.all;
        asm volatile("" ::: "memory");
#pragma unroll
        for (int s = 0; s < kSteps; ++s) n[s] = sh.from_n[(t & (kKept - 1)) + s][THREE ? a0 : 0];
    };
    // (the same in every lane)
    auto missing = [&](int32_t t) { return progress.x < t + kSteps || min(progress.y, progress.z) < t + kSteps - kKept; };
    auto await = [&](int32_t t, double (&n)[kSteps]) __attribute__((always_inline)) {
        while (__any(missing(t))) ask(t, n);
    };
    auto refused = [&]() __attribute__((always_inline)) { return valid && worst >= (2u * kSafeQuotient) << 21; };
    // The first block that has a quotient which is not the short division's (-1: none).  It is made again with divisions in
    // full; what comes after it in its round is nothing that anybody has been told of.
    int32_t bad = -1;
    auto block = [&](Operands *ops, double (&n)[kSteps], double (&next_n)[kSteps], int32_t t, auto ramp) __attribute__((always_inline)) {
        double *const row = sh.x[t & (kKept - 1)];
        worst = 0;
        // entry `lane` of the row two steps before, asked for a step ahead
        double xg = THREE ? sh.x[(t - 2) & (kKept - 1)][lane] : 0.;
        nm::static_for<kSteps>([&](auto at) __attribute__((always_inline)) {
            constexpr int s = decltype(at)::value;
            const double xg_now = xg;
            if constexpr (THREE && s == 0) xg = sh.x[(t - 1) & (kKept - 1)][lane];
            else if constexpr (THREE && s + 1 < kSteps) xg = row[(s - 1) * kRow + lane];
            step(ops[s], n[s], xg_now, t + s, row + s * kRow + kPatch + lane, ramp, std::false_type{});
            request(ops[s]);
            if constexpr (s == kSteps / 2) ask(t + kSteps, next_n);
        });
        // (one test for all that hardly ever is.  In a volume most blocks have to wait: 97 x 89 x 101 120.6 us with that test,
        // 119.5 without; 1024^2 446 and 462, both solves.)
        const bool again = refused();
        if (THREE || __builtin_expect(__any(again || missing(t + kSteps)) || bad >= 0, 0)) {
            if (bad < 0 && __any(again)) bad = t;
            if (bad < 0) nm::lds_put(&sh.now.done, t + kSteps);
            await(t + kSteps, next_n);
        } else {
            nm::lds_put(&sh.now.done, t + kSteps);
        }
    };
    int32_t t = 0;
    auto round = [&](auto ramp) __attribute__((always_inline)) {
        nm::static_for<kAhead / kSteps>([&](auto part) __attribute__((always_inline)) {
            constexpr int i = decltype(part)::value;
            block(o + i * kSteps, import_n[i % 2], import_n[(i + 1) % 2], t + i * kSteps, ramp);
        });
        t += kAhead;
    };
    // From step t on with divisions in full, until kFullBlocks blocks in a row could have done without.
    auto go_in_full = [&]() __attribute__((always_inline)) {
        Operands v[kSteps];
        double n[kSteps];
        place = t % length * w * 16;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            request(v[s]);
            asm volatile("" ::: "memory");
        }
        ask(t, n);
#pragma unroll 1
        for (int left = kFullBlocks; left > 0 && t < steps; t += kSteps) {
            double *const row = sh.x[t & (kKept - 1)];
            worst = 0;
            double xg = THREE ? sh.x[(t - 2) & (kKept - 1)][lane] : 0.;
            nm::static_for<kSteps>([&](auto at) __attribute__((always_inline)) {
                constexpr int s = decltype(at)::value;
                const double xg_now = xg;
                if constexpr (THREE && s == 0) xg = sh.x[(t - 1) & (kKept - 1)][lane];
                else if constexpr (THREE && s + 1 < kSteps) xg = row[(s - 1) * kRow + lane];
                step(v[s], n[s], xg_now, t + s, row + s * kRow + kPatch + lane, std::true_type{}, std::true_type{});
                request(v[s]);
            });
            left = __any(refused()) ? kFullBlocks : left - 1;
            nm::lds_put(&sh.now.done, t + kSteps);
            ask(t + kSteps, n);
            await(t + kSteps, n);
        }
    };
    while (true) {
        // (in the order of the steps, here too: else the first step of every round waits for all that is under way)
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            request(o[s]);
            asm volatile("" ::: "memory");
        }
        ask(t, import_n[0]);
        await(t, import_n[0]);
        bad = -1;
        // (a patch that a right-hand side reaches late, or never, starts with zeros)
        if (t == 0 && __any(lane == 0 && o[0].rd.x == 0. && import_n[0][0] == 0.)) bad = 0;
#pragma unroll 1
        while (t < deepest && bad < 0) round(std::true_type{});
#pragma unroll 1
        while (t + kAhead <= length && bad < 0) round(std::false_type{});
#pragma unroll 1
        while (t < steps && bad < 0) round(std::true_type{});
        if (bad < 0) break;
        t = bad;
        x = sh.x[(t - 1) & (kKept - 1)][kPatch + lane];
        go_in_full();
        place = t % length * w * 16;
        if (t >= steps) break;
    }
    // (nobody waits for more steps than there are, whatever multiple they count in)
    if (lane == 0) nm::lds_put(&sh.now.done, kAll);
}

// Wavefront 1: the rows of other patches that this one needs, from the edges into LDS.  False: it gave up.
template <typename T, bool THREE> __device__ __forceinline__ bool import_edges(const Args<T> &k, const Patch &P, Shared &sh) {
    const int lane = threadIdx.x & 63;
    const int32_t length = k.g.length;
    const bool in_n = P.J > 0, in_g = THREE && P.I > 0;
    if (!in_n && !in_g) return true;
    const unsigned long long *edge_n = k.edge + ((int64_t)(P.J - 1) * k.g.planes + P.i0) * length;
    const unsigned long long *edge_g = k.edge + k.g.edge_n() + ((int64_t)(P.I - 1) * k.g.width + P.j0) * length;
    const int32_t steps = length + skew(P.na - 1, P.nb - 1);
    // A poll: 64 rows of an edge, or eight steps of two.  (Polls for what is not there yet slow its coming: three of them under
    // way at a time 1024^2 208 -> 223 us, 97 x 89 x 101 118 -> 141 us; four after one that found all 118 -> 134.)
    const int e = THREE ? lane % kPatch : 0, ahead = THREE ? lane / kPatch : lane;
    int64_t waited = 0;
    for (int32_t t = 0; t < steps;) {
        if (k.poll_limit < 0 || waited > k.poll_limit) return false;
        const int32_t room = __builtin_amdgcn_readfirstlane(nm::lds_get(&sh.now.done)) + kKept - 2;
        const int32_t at = t + ahead, cn = at - skew(e, 0), cg = at - skew(0, e);
        const unsigned long long n = in_n && cn >= 0 && cn < length && e < P.na ? look(edge_n + (int64_t)cn * P.na + e) : 0ull;
        const unsigned long long g = in_g && cg >= 0 && cg < length && e < P.nb ? look(edge_g + (int64_t)cg * P.nb + e) : 0ull;
        const unsigned long long open = __ballot(n == kUnsolved || g == kUnsolved || at >= room);
        const int got = (open ? __builtin_ctzll(open) : 64) / (THREE ? kPatch : 1);
        if (ahead < got) {
            nm::lds_put(&sh.from_n[at & (kKept - 1)][e], __longlong_as_double((long long)n));
            if (THREE) nm::lds_put(&sh.x[(at - 2) & (kKept - 1)][e], __longlong_as_double((long long)g));
        }
        t += got;
        if (got > 0 && lane == 0) nm::lds_put(&sh.now.imported, t);
        waited = got > 0 || t + 1 >= room ? 0 : waited + 1;
    }
    return true;
}

// Waits until `upto` steps are solved.
__device__ __forceinline__ void await_steps(Shared &sh, int32_t upto) {
    while (__builtin_amdgcn_readfirstlane(nm::lds_get(&sh.now.done)) < upto) __builtin_amdgcn_s_sleep(1);
}

// Wavefront 2: the patch's last lines into the edges.
template <typename T, bool THREE> __device__ __forceinline__ void export_edges(const Args<T> &k, const Patch &P, Shared &sh) {
    const int lane = threadIdx.x & 63;
    const int32_t length = k.g.length, steps = length + skew(P.na - 1, P.nb - 1);
    const bool to_n = P.J + 1 < k.g.nj, to_g = THREE && P.I + 1 < k.g.ni;
    if (!to_n && !to_g) return;
    unsigned long long *edge_n = k.edge + ((int64_t)P.J * k.g.planes + P.i0) * length;
    unsigned long long *edge_g = k.edge + k.g.edge_n() + ((int64_t)P.I * k.g.width + P.j0) * length;
    // a block's steps, eight lines
    constexpr int kSteps = kBlockSteps;
    const int e = THREE ? lane % kPatch : 0, s = THREE ? lane / kPatch : lane;
    for (int32_t t = 0; t < steps; t += kSteps) {
        await_steps(sh, t + kSteps);
        const int32_t at = t + s, cn = at - skew(e, P.nb - 1), cg = at - skew(P.na - 1, e);
        const double *row = sh.x[at & (kKept - 1)] + kPatch;
        if (to_n && s < kSteps && e < P.na && cn >= 0 && cn < length)
            leave(edge_n + (int64_t)cn * P.na + e, nm::lds_get(row + (THREE ? e * kPatch : 0) + P.nb - 1));
        if (THREE && to_g && s < kSteps && e < P.nb && cg >= 0 && cg < length)
            leave(edge_g + (int64_t)cg * P.nb + e, nm::lds_get(row + (P.na - 1) * kPatch + e));
        if (lane == 0) nm::lds_put(&sh.now.exported, t + kSteps);
    }
}

// Wavefront 3: the results into x, sixteen steps at a time: sixteen rows of four lines with a store where a line's rows lie
// next to each other, else the eight rows along b with the same place in their lines, eight such places with a store.
template <typename T, bool THREE> __device__ __forceinline__ void write_rows(const Args<T> &k, const Patch &P, Shared &sh) {
    const int lane = threadIdx.x & 63;
    const int32_t length = k.g.length, steps = length + skew(P.na - 1, P.nb - 1);
    constexpr int kRows = 16;
    auto write = [&](auto lines_apart) __attribute__((always_inline)) {
        // store g: line `first(g)` + line0, step t + offset(g)
        constexpr bool kApart = decltype(lines_apart)::value;
        const int32_t line0 = kApart ? lane % 8 : lane / kRows;
        for (int32_t t = 0; t < steps; t += kRows) {
            await_steps(sh, t + kRows);
            double v[kRows];
            nm::static_for<kRows>([&](auto at) __attribute__((always_inline)) {
                constexpr int g = decltype(at)::value;
                const int32_t l = (kApart ? g / 2 * 8 : g * 4) + line0;
                const int32_t s = kApart ? (g % 2 * 8 + lane / 8 + lane % 8) % kRows : lane % kRows;
                v[g] = sh.x[(t & (kKept - 1)) + s][kPatch + l];
            });
            asm volatile("" ::: "memory");
            if (lane == 0) nm::lds_put(&sh.now.written, t + kRows);
            nm::static_for<kRows>([&](auto at) __attribute__((always_inline)) {
                constexpr int g = decltype(at)::value;
                constexpr int first = kApart ? g / 2 * 8 : g * 4, a = THREE ? first / kPatch : 0, b0 = THREE ? first % kPatch : first;
                const int32_t s = kApart ? (g % 2 * 8 + lane / 8 + lane % 8) % kRows : lane % kRows;
                const int32_t b = b0 + line0, c = t + s - skew(a, b);
                if (a < P.na && b < P.nb && (uint32_t)c < (uint32_t)length) {
                    const int32_t r = k.g.row(P.i0 + a, P.j0 + b, c);
                    k.x[k.mirrored ? k.rows - 1 - r : r] = (T)v[g];
                }
            });
        }
    };
    if (k.g.along == 1) write(std::false_type{});
    else write(std::true_type{});
}

template <typename T, bool THREE, bool LINE_LAST> __global__ __launch_bounds__(256) void solve_kernel(Args<T> k) {
    __shared__ Shared sh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    while (true) {
        if (threadIdx.x == 0) sh.patch = atomicAdd(k.status + 1, 1);
        __syncthreads();
        const int32_t id = __builtin_amdgcn_readfirstlane(sh.patch);
        if (id >= k.g.ni * k.g.nj) return;
        const Patch P = patch_of(k.g, id);
        // what is not imported is zero: no line before, no plane before, no row solved yet
        for (int e = threadIdx.x; e < kKept * (kPatch + 64); e += 256) sh.x[e / (kPatch + 64)][e % (kPatch + 64)] = 0.;
        for (int e = threadIdx.x; e < kKept * kPatch; e += 256) sh.from_n[e / kPatch][e % kPatch] = 0.;
        if (threadIdx.x == 0) {
            sh.now.imported = P.J > 0 || (THREE && P.I > 0) ? 0 : kAll;
            sh.now.exported = P.J + 1 < k.g.nj || (THREE && P.I + 1 < k.g.ni) ? 0 : kAll;
            sh.now.written = sh.now.done = 0;
        }
        __syncthreads();
        if (wave == 0) {
            solve_patch<T, THREE, LINE_LAST>(k, P, sh);
        } else if (wave == 1) {
            const bool ok = import_edges<T, THREE>(k, P, sh);
            if (!ok && (threadIdx.x & 63) == 0)
                __hip_atomic_store(k.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((threadIdx.x & 63) == 0) nm::lds_put(&sh.now.imported, kAll);
        } else if (wave == 2) {
            export_edges<T, THREE>(k, P, sh);
        } else {
            write_rows<T, THREE>(k, P, sh);
        }
        __syncthreads();
    }
}

// x = NaN throughout where somebody gave up waiting
template <typename T> __global__ __launch_bounds__(256) void failed_kernel(int32_t rows, const int32_t *__restrict__ status,
                                                                           T *__restrict__ x) {
    if (status[0] == 0) return;
    for (int32_t i = blockIdx.x * 256 + threadIdx.x; i < rows; i += gridDim.x * 256) x[i] = (T)__longlong_as_double(0x7ff8000000000000ll);
}

constexpr int kMaxGroups = 1024;   // workgroups, which draw patches until there are none

// Room in the per-call areas of doubles: `wide` takes four a row, `pairs` two, `edges` the edges.
template <typename T>
int solve(const Grid &g, int64_t rows, bool mirrored, const int32_t *src, const T *data, int unit, const T *b, T *x,
          double *wide, double *pairs, double *edges, int32_t *status, int64_t poll_limit, int most_groups, hipStream_t s) {
    Args<T> k;
    k.g = g;
    k.rows = (int32_t)rows;
    k.mirrored = mirrored;
    k.unit = unit;
    k.src = reinterpret_cast<const int4 *>(src);
    k.data = data;
    k.b = b;
    k.x = x;
    k.near = reinterpret_cast<double2 *>(wide);
    k.y = wide + 2 * rows;
    k.rd = reinterpret_cast<double2 *>(pairs);
    k.edge = reinterpret_cast<unsigned long long *>(edges);
    k.status = status;
    k.poll_limit = poll_limit;
    const int32_t patches = g.ni * g.nj;
    const int64_t entries = (int64_t)g.ah * g.bw * g.length;
    int64_t gx = nm::ceil_div(entries, (int64_t)256), gy = patches < 4096 ? patches : 4096;
    if (gx > 1024) gx = 1024;
    const dim3 grid((unsigned)gx, (unsigned)gy), groups((unsigned)(patches < most_groups ? patches : most_groups));
    if (g.planes > 1) {
        hipLaunchKernelGGL((gather_kernel<T, true>), grid, dim3(256), 0, s, k);
        if (g.along == 1) hipLaunchKernelGGL((solve_kernel<T, true, true>), groups, dim3(256), 0, s, k);
        else hipLaunchKernelGGL((solve_kernel<T, true, false>), groups, dim3(256), 0, s, k);
    } else {
        hipLaunchKernelGGL((gather_kernel<T, false>), grid, dim3(256), 0, s, k);
        hipLaunchKernelGGL((solve_kernel<T, false, true>), groups, dim3(256), 0, s, k);
    }
    NM_LAUNCH_CHECK("lines::solve_kernel");
    if (patches > 1) {
        hipLaunchKernelGGL(failed_kernel<T>, dim3(64), dim3(256), 0, s, (int32_t)rows, status, x);
        NM_LAUNCH_CHECK("lines::failed_kernel");
    }
    return NM_OK;
}

}  // namespace lines
}  // namespace
