// spmm.hip -- CSR SpMM C = alpha*A*B + beta*C for gfx950 (wave64).
//
// Replaces execute(::EmitterBackend, ::Op{:SpMM}, ...)
// (ext/KernelAbstractionsExt/ops/spmm.jl:397-423).  Per output the reference
// sums val[k]*B[col[k], c] sequentially over the row and writes
// alpha*acc + beta*C (spmm.jl:272-279 for the Tiled strategy used at k > 32).
//
// B and C are column-major (Julia layout).  Gathering a row B[j, :] straight
// from column-major B touches k cache lines 4*ldb bytes apart for k useful
// values, so the kernel first re-lays B out row-major (Bt, n x ldt) in the
// library's scratch buffer with an LDS-tiled transpose: one coalesced read
// and one coalesced write of B.  csr_spmm_rows_kernel then gathers whole rows
// of Bt for several rows of A at once, and writes its results column by column
// through LDS.  One column needs no copy (csr_spmm_group_kernel).
#include "common.hpp"

#include <cstdlib>
#include <memory>
#include <type_traits>
#include <vector>

namespace jlust {
namespace {

constexpr int SPMM_BLOCK = 256;

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }
constexpr int SPMM_ROWS = 32;

__device__ __forceinline__ int bcast_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

template <typename T, int VEC> struct Vec;
template <typename T> struct Vec<T, 1> { T v[1]; };
template <typename T> struct alignas(2 * sizeof(T)) Vec<T, 2> { T v[2]; };
template <typename T> struct alignas(4 * sizeof(T)) Vec<T, 4> { T v[4]; };

// Bt[j*ldt + c] = B[j + c*ldb] for j < n, c < k, in tiles of CT columns and
// 4096/CT rows through LDS: columns are read 64 rows at a time, rows written
// VEC columns at a time.  CT is the smallest of 16, 32 and 64 that holds the
// columns, so a narrow B's tile holds as many entries as a wide one's (262k
// rows, f64, 20 columns: 19.4 us with 64-column tiles and one column per
// write, 16.2 us).  Padding columns (ldt beyond k) take what the tile holds,
// and are never used; row n of Bt is zeroed for the lanes of the rows kernel
// that have no entry.
template <typename T, int VEC, int CT>
__global__ __launch_bounds__(256) void transpose_kernel(int64_t n, int64_t k, const T *__restrict__ B,
                                                        int64_t ldb, T *__restrict__ Bt, int64_t ldt)
{
    constexpr int JT = 4096 / CT;
    constexpr int UR = CT / VEC;               // writes per row of the tile
    __shared__ T tile[CT][JT + 1];
    const int64_t j0 = (int64_t)blockIdx.x * JT;
    const int64_t c0 = (int64_t)blockIdx.y * CT;
    const int ncol = (int)min((int64_t)CT, k - c0);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int i = threadIdx.x + 256 * s;
        const int cc = i / JT, jj = i % JT;
        if (j0 + jj < n && cc < ncol) tile[cc][jj] = B[j0 + jj + (c0 + cc) * ldb];
    }
    __syncthreads();
    const int nwr = (int)min((int64_t)CT, ldt - c0);
#pragma unroll
    for (int s = 0; s < 16 / VEC; ++s) {
        const int i = threadIdx.x + 256 * s;
        const int jj = i / UR, cc = i % UR * VEC;
        if (cc >= nwr || j0 + jj > n) continue;
        Vec<T, VEC> v;
#pragma unroll
        for (int e = 0; e < VEC; ++e) v.v[e] = j0 + jj < n ? tile[cc + e][jj] : T(0);
        *reinterpret_cast<Vec<T, VEC> *>(Bt + (j0 + jj) * ldt + c0 + cc) = v;
    }
}

// One column, and 2 to 4 columns of long rows: groups of KV lanes (KV the
// smallest power of two >= the columns), one nonzero per group per step, so a
// wave takes 64/KV nonzeros per step (64 at k = 1, where the kernel is a
// wave-per-row SpMV).  Each lane loads its group's col/val itself (the group's
// lanes read one address), gathers its column of the nonzero's Bt row, and
// keeps its group's sum in nonzero order; the groups' sums are added with
// xor-shuffles at the row's end.  U steps are loaded at once (indices clamped
// into the row, products of the clamped copies dropped by a select; U is
// chosen per call from the mean row length, so a short row issues no clamped
// copies), and the next row's pointers are loaded before the current row's
// nonzeros, so a wave's rows do not wait on each other's pointer loads.
template <typename T, int KV, int U>
__global__ __launch_bounds__(SPMM_BLOCK) void csr_spmm_group_kernel(
    int64_t m, int64_t k, int32_t origin, const int32_t *__restrict__ rowptr,
    const int32_t *__restrict__ colind, const T *__restrict__ val, const T *__restrict__ Bt,
    int64_t ldt, T alpha, T beta, int beta_zero, T *__restrict__ C, int64_t ldc,
    int skip_empty_rows, const int32_t *__restrict__ rowend, const uint8_t *__restrict__ row_skip)
{
    constexpr int G = 64 / KV;                 // nonzeros per step
    constexpr int NW = SPMM_BLOCK / 64;
    __shared__ T s_c[SPMM_ROWS][KV + 1];
    __shared__ int s_empty[SPMM_ROWS];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int grp = lane / KV;
    const int col = lane % KV;
    const int64_t row0 = (int64_t)blockIdx.x * SPMM_ROWS;
    const int nrows = (int)min((int64_t)SPMM_ROWS, m - row0);
    const int64_t cl = col < k ? col : 0;      // clamped, in-bounds column

    int32_t lo_n = 0, hi_n = 0;
    if (wave < nrows) {
        lo_n = rowptr[row0 + wave];
        hi_n = rowend ? rowend[row0 + wave] : rowptr[row0 + wave + 1];
    }
    for (int rr = wave; rr < nrows; rr += NW) {
        const int64_t lo = (int64_t)lo_n - origin;
        int64_t hi = (int64_t)hi_n - origin;
        if (rr + NW < nrows) {                 // the wave's next row
            lo_n = rowptr[row0 + rr + NW];
            hi_n = rowend ? rowend[row0 + rr + NW] : rowptr[row0 + rr + NW + 1];
        }
        const bool skip = row_skip && row_skip[row0 + rr];
        if (skip) hi = lo;                     // a split row: its segments compute it
        if (lane == 0) s_empty[rr] = skip ? 2 : hi <= lo;
        T acc = T(0);
        for (int64_t p0 = lo + grp; p0 < hi; p0 += (int64_t)G * U) {
            int32_t c[U];
            T a[U], b[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t p = min(p0 + (int64_t)u * G, hi - 1);
                c[u] = colind[p];
                a[u] = val[p];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) b[u] = Bt[(int64_t)(c[u] - origin) * ldt + cl];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const T s = acc + a[u] * b[u];
                acc = p0 + (int64_t)u * G < hi ? s : acc;
            }
        }
#pragma unroll
        for (int off = KV; off < 64; off <<= 1) acc += __shfl_xor(acc, off, 64);
        if (lane < KV) s_c[rr][col] = acc;
    }
    __syncthreads();
    const int ncols = (int)k;                  // k <= KV here
    for (int idx = tid; idx < SPMM_ROWS * ncols; idx += SPMM_BLOCK) {
        const int rr = idx % SPMM_ROWS;
        const int cc = idx / SPMM_ROWS;
        if (rr >= nrows) continue;
        if (s_empty[rr] == 2 || (skip_empty_rows && s_empty[rr])) continue;
        T *dst = C + (row0 + rr) + cc * ldc;
        const T s = alpha * s_c[rr][cc];
        *dst = beta_zero ? s : s + beta * *dst;
    }
}

// A set of rows for csr_spmm_rows_kernel: the matrix's rows (hi null: row r
// ends where r + 1 starts), or the segments of a plan's split rows.
template <typename T>
struct SpmmJob {
    int64_t rows = 0;
    const int32_t *lo = nullptr, *hi = nullptr;
    const uint8_t *skip = nullptr;       // rows left untouched
    T alpha = T(0), beta = T(0);
    T *C = nullptr;
    int64_t ldc = 0;
    int beta_zero = 1, skip_empty_rows = 0;
    int R = 1;                           // rows per block, at most 64
    unsigned blocks = 0;
    unsigned run = 1;                    // consecutive blocks per XCD
};

// Most entries of a block staged at once, and most slices of rows among them:
// a remainder per row, and one per 32 entries.
constexpr int SPMM_STAGE = 2040;
constexpr int SPMM_TASKS = 64 + SPMM_STAGE / 32 + 2;

// How the columns lie over a wave, and the block's buffers.
struct SpmmShape {
    int64_t k;                           // columns of the pass
    int64_t ldt;                         // row stride of Bt
    int64_t zero_row;                    // Bt's row of zeros
    int cols;                            // columns per blockIdx.y, a multiple of VEC
    int L;                               // lanes per entry: cols / VEC
    int slice_log2;                      // entries of a slice
    int cld;                             // row stride of the result tile
    int rmax;                            // rows of the result tile
    int ch;                              // entries staged at once, above a slice
    int xmax;                            // further slices of the staged rows
};

__device__ __forceinline__ int wave_min(int v)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v = min(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ int wave_max(int v) { return -wave_min(-v); }

// Row-split SpMM over the row-major copy of B.  A wave's 64 lanes form
// NG = 64 / L groups; a group takes a row, each lane VEC columns of B's row per
// entry, so one vector load of a wave serves NG entries of NG rows and no sum
// crosses lanes.  What bounds it is the gathers: L1 where rows share columns (the
// f64 mesh below: an access in 94 % of its cycles), the fabric behind the L2s
// where they do not (200k power-law rows below: L2 hits 14 %, 6.7 TB/s past it;
// 1M uniform rows, 64 columns: 4 %, 7.6 TB/s).
//   - The block's entries (colind turned into an offset into Bt, and val) are
//     staged in LDS with coalesced loads and read back by the groups: a load
//     of col and val by each group would take as many address cycles as the
//     gathers.  Groups past their row's end read a staged entry that points at
//     Bt's row of zeros, so no product needs a select.
//   - The unit of work is a slice of a row: 32 to 256 entries by the number of
//     columns, counted from the row's start, so most rows are one. A slice is
//     summed by one group, and a row's slices are added in order: a
//     row's sum depends on its own entries alone, not on the rows around it.
//     Slices are dealt to the groups longest first (whole slices, then what
//     remains of the rows in four classes of length), so that the groups of a
//     wave end together.
//   - The results pass through LDS and are written column by column.
//   - Blocks are numbered so that an XCD takes `run` consecutive ones: rows
//     that share columns then find B's rows in one L2 (the f64 mesh product
//     below: 65 us with one block at a time per XCD, 60 us).
// Measured against one row per wave (k > 32) and one entry per 2^i lanes
// (k <= 32), both loading col and val from memory for every entry, in us per
// product with B's copy: 27-point mesh of 262k rows, f64, k = 20: 297 -> 80,
// f32, k = 64: 224 -> 124; 200k power-law rows of 14, f32, k = 100: 1380 -> 274
// (segments of split rows included: 743 of the 1380); 8000 rows of 300, f32,
// k = 20: 107 -> 34; 200k uniform rows of 16 (bound by the fabric), f64, k = 8:
// 69 -> 63, k = 64: 291 -> 297.
// 5 waves per SIMD at least, as many as the LDS of 5 blocks leaves (the f64 mesh
// at k = 20: 71 us at 4); 4 where the sums and the entries in flight take more
// registers than that leaves (f64, 2 columns a lane, 12 of both: 9 to 24 spilled
// at 5; mesh below, k = 8: 50 -> 46 us with twice the sums, band of 30 a row, k =
// 16: 18.1 -> 15.9).
template <typename T, int VEC, int U, int ACC, bool BIG>
__global__ __launch_bounds__(SPMM_BLOCK, (ACC + U) * VEC * sizeof(T) > 160 ? 4 : 5) void csr_spmm_rows_kernel(
    SpmmJob<T> ja, SpmmJob<T> jb, SpmmShape sh, int32_t origin, const int32_t *__restrict__ colind,
    const T *__restrict__ val, const T *__restrict__ Bt0)
{
    constexpr int NW = SPMM_BLOCK / 64;
    using V = Vec<T, VEC>;
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    T *const s_val = reinterpret_cast<T *>(s_mem);                             // [ch + 1]
    T *const s_c = s_val + sh.ch + 2;                                          // [rmax][cld]
    T *const s_x = s_c + sh.rmax * sh.cld;                                     // [xmax][cld]
    uint32_t *const s_off = reinterpret_cast<uint32_t *>(s_x + sh.xmax * sh.cld);   // [ch + 1]
    __shared__ int s_task[SPMM_TASKS];

    const bool second = blockIdx.x >= ja.blocks;
    const SpmmJob<T> &j = second ? jb : ja;
    unsigned lb = blockIdx.x - (second ? ja.blocks : 0u);
    if (!second) {
        const unsigned x = lb % NUM_XCD, i = lb / NUM_XCD;
        lb = (i / j.run * NUM_XCD + x) * j.run + i % j.run;
    }
    const int64_t row0 = (int64_t)lb * j.R;
    if (row0 >= j.rows) return;
    const int nrows = (int)min((int64_t)j.R, j.rows - row0);
    const int c0 = (int)blockIdx.y * sh.cols;
    const int kk = (int)min((int64_t)sh.cols, sh.k - c0);
    const T *const Bt = Bt0 + c0;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int L = sh.L, NG = 64 / L, NGB = NG * NW;
    const int grp = lane / L, sub = lane - grp * L;
    // The lane's first column; the last lanes of the last columns stay in Bt's row.
    const int col = min(sub * VEC, (int)(sh.ldt - c0) - VEC);
    const uint32_t colb = (uint32_t)(col * (int)sizeof(T));

    int lo = 0, hi = 0;
    bool skip = false;
    if (lane < nrows) {
        lo = j.lo[row0 + lane] - origin;
        hi = (j.hi ? j.hi[row0 + lane] : j.lo[row0 + lane + 1]) - origin;
        skip = j.skip && j.skip[row0 + lane];
        if (skip) lo = hi;
    }
    const bool empty = hi <= lo;
    // A lane whose row is not followed by the next row's entries ends a run.
    const int next = __shfl_down(lo, 1, 64);
    const bool brk = lane == nrows - 1 || (lane < nrows && (next != hi || next < lo));
    const bool whole = __popcll(__ballot(brk)) == 1;     // the rows' entries are one run
    const int last = whole ? bcast_i(hi, nrows - 1) : wave_max(empty ? INT_MIN + 1 : hi);

    const int ss = sh.slice_log2, S = 1 << ss;

    // N steps of every group: entries p + s .. p + s + N - 1, those with s + u < n,
    // entry u into sum (FIRST + u) mod ACC of ACC sums per column.
    T acc[ACC][VEC];
    auto steps = [&](auto N, auto FIRST, int p, int s, int n) {
        constexpr int NS = decltype(N)::value, F = decltype(FIRST)::value;
        uint32_t off[NS];
        T a[NS];
        V b[NS];
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            const int i = s + u < n ? p + s + u : sh.ch;
            off[u] = s_off[i];
            a[u] = s_val[i];
        }
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            if (BIG)
                b[u] = *reinterpret_cast<const V *>(Bt + (uint64_t)off[u] * (uint64_t)sh.ldt + col);
            else
                b[u] = *reinterpret_cast<const V *>(reinterpret_cast<const char *>(Bt) + (off[u] + colb));
        }
#pragma unroll
        for (int u = 0; u < NS; ++u)
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[(F + u) % ACC][e] += a[u] * b[u].v[e];
    };
    using I0 = std::integral_constant<int, 0>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    auto row_sum = [&](int p, int n) {
        int s = 0;
        if constexpr (ACC == 8) {
            for (; __any(s + 6 < n); s += 8) {
                steps(I4(), I0(), p, s, n);
                steps(I4(), I4(), p, s + 4, n);
            }
            if (__any(s + 2 < n)) {
                steps(I4(), I0(), p, s, n);
                s += 4;
                if (__any(s < n)) steps(I2(), I4(), p, s, n);
                return;
            }
        } else {
            if constexpr (U == 8)
                for (; __any(s + 4 < n); s += 8) steps(std::integral_constant<int, 8>(), I0(), p, s, n);
            for (; __any(s + 2 < n); s += 4) steps(I4(), I0(), p, s, n);
        }
        if (__any(s < n)) steps(I2(), I0(), p, s, n);
    };

    int a = whole ? bcast_i(lo, 0) : wave_min(empty ? INT_MAX : lo);
    while (a < last) {
        // The next entries [a, b): from the first unfinished row on, no further
        // than its run, the end of the rows and the buffer.
        if (!whole) a = wave_min(!empty && hi > a ? max(lo, a) : INT_MAX);
        if (a >= last) break;
        int b = a + min(sh.ch, last - a);
        if (!whole) b = min(b, wave_min(brk && hi > a ? hi : INT_MAX));
        // The row that holds entry b is left before its start, or at the end of a slice.
        const uint64_t left = __ballot(lo < b && b < hi);
        if (left) {
            const int to = hi - lo > S ? lo + ((b - lo) >> ss << ss) : lo;
            b = max(bcast_i(max(to, max(lo, a)), __ffsll((unsigned long long)left) - 1), a + 1);
        }
        const int n = empty ? 0 : max(0, min(hi, b) - max(lo, a));
        const int st = min(max(max(lo, a) - a, 0), sh.ch);

        // The slices: full ones, the row's remainder, and those beyond the
        // row's first, which have sums of their own until all are done.
        const bool cont = lo < a;
        const int full = n >> ss, rem = n & (S - 1);
        const int more = n > 0 ? full + (rem > 0) - !cont : 0;
        const uint64_t xrows = __ballot(more > 0);
        int fbase = full, xbase = more, nfull = 0;
        if (xrows || __any(full > 0)) {
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int f = __shfl_up(fbase, off, 64), x = __shfl_up(xbase, off, 64);
                fbase += lane >= off ? f : 0;
                xbase += lane >= off ? x : 0;
            }
            nfull = bcast_i(fbase, 63);
        }
        fbase -= full;
        xbase -= more;
        int at = nfull, ntask = nfull;
#pragma unroll
        for (int c = 3; c >= 0; --c) {
            const uint64_t in = __ballot(rem > 0 && rem >> (ss - 2) == c);
            if (rem >> (ss - 2) == c) at = ntask + __popcll(in & ((1ull << lane) - 1));
            ntask += __popcll(in);
        }
        ntask = min(ntask, SPMM_TASKS);

        __syncthreads();                       // the last entries are done with
        // A slice is (first entry | entries | place of its sum: a row, or 64 + s_x's).
        auto task = [&](int q, int i, int cnt) {
            const int x = i - !cont;
            const int place = x < 0 ? lane : 64 + min(xbase + x, sh.xmax - 1);
            if (q < SPMM_TASKS) s_task[q] = (st + (i << ss)) | cnt << 11 | place << 20;
        };
        for (int i = wave; i < full; i += NW) task(fbase + i, i, S);
        if (wave == 0 && rem > 0) task(at, full, rem);
        for (int i = tid; i < b - a; i += SPMM_BLOCK) {
            const uint32_t c = (uint32_t)(colind[a + i] - origin);
            s_off[i] = BIG ? c : c * (uint32_t)(sh.ldt * sizeof(T));
            s_val[i] = val[a + i];
        }
        if (tid == 0) {
            s_off[sh.ch] = BIG ? (uint32_t)sh.zero_row : (uint32_t)(sh.zero_row * sh.ldt * sizeof(T));
            s_val[sh.ch] = T(0);
        }
        __syncthreads();

        int turn = 0;
        for (int q0 = 0; q0 < ntask; q0 += NGB, ++turn) {
            const int q = q0 + (turn & 1 ? NW - 1 - wave : wave) * NG + grp;
            const int t = grp < NG && q < ntask ? s_task[q] : 0;
            const int cnt = t >> 11 & 511;
#pragma unroll
            for (int h = 0; h < ACC; ++h)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[h][e] = T(0);
            row_sum(t & 2047, cnt);
            // s_x follows s_c, rmax rows on.
            const int place = t >> 20;
            T *const dst = s_c + (place < 64 ? place : place - 64 + sh.rmax) * sh.cld + sub * VEC;
            if (cnt > 0) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    T v = acc[0][e] + acc[1][e];
                    if constexpr (ACC >= 4) v += acc[2][e] + acc[3][e];
                    if constexpr (ACC == 8) v += (acc[4][e] + acc[5][e]) + (acc[6][e] + acc[7][e]);
                    dst[e] = v;
                }
            }
        }
        if (xrows) {
            __syncthreads();
            uint64_t left_rows = xrows;
            for (int i = 0; left_rows; ++i, left_rows &= left_rows - 1) {
                if ((i & (NW - 1)) != wave) continue;
                const int r = __ffsll((unsigned long long)left_rows) - 1;
                const int x0 = bcast_i(xbase, r), cnt = min(bcast_i(more, r), sh.xmax - x0);
                for (int c = lane; c < kk; c += 64) {
                    T v = s_c[r * sh.cld + c];
                    for (int h = 0; h < cnt; ++h) v += s_x[(x0 + h) * sh.cld + c];
                    s_c[r * sh.cld + c] = v;
                }
            }
        }
        a = b;
    }
    __syncthreads();
    if (lane >= nrows || skip || (j.skip_empty_rows && empty)) return;
    for (int c = wave; c < kk; c += NW) {
        T *const dst = j.C + (row0 + lane) + (c0 + c) * j.ldc;
        const T v = j.alpha * (empty ? T(0) : s_c[lane * sh.cld + c]);
        *dst = j.beta_zero ? v : v + j.beta * *dst;
    }
}

// Columns per pass: all of k while the row-major copy of B fits a budget of
// the 256 MB MALL, else the widest multiple of 16 columns that does (at least
// 16).  JLUST_HIP_SPMM_KCHUNK=c forces c columns per pass.
constexpr size_t SPMM_MALL_BUDGET = (size_t)256 << 20;

int64_t spmm_kchunk(int64_t n, int64_t k, size_t tsz)
{
    static const int64_t forced = [] {
        const char *e = getenv("JLUST_HIP_SPMM_KCHUNK");
        return e ? (int64_t)atoll(e) : (int64_t)0;
    }();
    if (forced > 0) return forced < k ? forced : k;
    const size_t row = (size_t)(n > 0 ? n : 1) * tsz;
    if ((size_t)k * row <= SPMM_MALL_BUDGET) return k;
    int64_t kc = (int64_t)(SPMM_MALL_BUDGET / row) / 16 * 16;
    if (kc < 16) kc = 16;
    return kc < k ? kc : k;
}

// Long rows of a prepared plan: a row with more than SPMM_LONG_ROW entries
// is cut into segments of SPMM_SEG entries, each a row of its own in the same
// launch (blocks after the rows') writing one partial row into the plan's
// workspace; spmm_long_reduce_kernel adds a row's partials in segment order.
// A block otherwise walks a whole row alone, so a 10^5-entry row of a power-law
// matrix would keep one block busy long after the others.
constexpr int64_t SPMM_LONG_ROW = 1024;
constexpr int64_t SPMM_SEG = 256;

// C[r, c] = alpha * sum_s part[s, c] + beta * C[r, c] for the long rows:
// one thread per (long row, column), partials of the row's segments
// [seg_first[l], seg_first[l+1]) added in segment order.
template <typename T>
__global__ void spmm_long_reduce_kernel(int64_t nlong, int64_t kk, const int32_t *__restrict__ long_rows,
                                        const int32_t *__restrict__ seg_first, const T *__restrict__ part,
                                        int64_t ldp, T alpha, T beta, int beta_zero, T *__restrict__ C,
                                        int64_t ldc)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nlong * kk) return;
    const int64_t l = t % nlong, c = t / nlong;
    const int32_t s0 = seg_first[l], s1 = seg_first[l + 1];
    T acc = part[s0 + c * ldp];
    for (int32_t q = s0 + 1; q < s1; ++q) acc += part[q + c * ldp];
    T *dst = C + long_rows[l] + c * ldc;
    const T v = alpha * acc;
    *dst = beta_zero ? v : v + beta * *dst;
}

// How one column chunk of kk columns is computed: VEC columns per lane of the
// rows kernel and the row stride of B's copy (whole vectors), or one column
// from B itself.
//   - 16 bytes per lane where L1 and L2 serve the gathers: half the loads of
//     8 bytes (27-point mesh, k = 64: f32 105 against 146 us, f64 249 against
//     321 us).
//   - Fewer columns per lane below 13 (f32) and 5 (f64) of them, so that the
//     block's groups do not outnumber the 64 rows its lanes hold (200k
//     power-law rows, f32, k = 8: 71 us, 87 with 4 columns per lane; f64, k = 4
//     likewise).
//   - 8 bytes per lane for wide f32 chunks of a copy past 128 MB, where random
//     rows come from the MALL: a wave's load then spans half as many rows
//     (1M uniform rows of 32, 64 columns: 1.135 against 1.160 ms; a mesh would
//     rather have 16).  f64 keeps 16: the mesh loses more than random rows
//     gain (262k rows, k = 128: 519 -> 680 us; 200k uniform rows of 16: 585 ->
//     567 us).
//   - The group kernel for one column, and for 2 to 4 (f64: 2) where rows hold
//     more than 48 entries on average: so few columns leave the rows kernel's
//     slices too few for its groups (100k rows of 200, band of +-150, f32:
//     k = 2 79.7 against 47.5 us, k = 4 92.4 against 72.3 us; f64: k = 2 92.3
//     against 65.2, k = 4 106 against 126; with 27 entries, f32, k = 4, 27.6
//     against 54.2 us).
struct SpmmChunk {
    bool group;                          // the group kernel
    bool direct;                         // B's own column, no copy
    int vec;
    int64_t ldt;
};

template <typename T>
SpmmChunk spmm_chunk_kind(int64_t n, int64_t kk, int64_t mean)
{
    constexpr int W16 = 16 / sizeof(T), W8 = 8 / sizeof(T);
    SpmmChunk c;
    c.direct = kk == 1;
    c.group = c.direct || (kk <= (sizeof(T) == 4 ? 4 : 2) && mean > 48);
    c.vec = W16;
    if (sizeof(T) == 4 && kk >= 48 && n * kk * 4 > (int64_t)128 << 20) c.vec = W8;
    if (kk <= 12 && sizeof(T) == 4) c.vec = W8;
    if (kk <= 4) c.vec = 1;
    c.ldt = (kk + c.vec - 1) / c.vec * c.vec;
    return c;
}

// Elements of the row-major copy of a pass of at most kc of k columns.
int64_t spmm_copy_elems(int64_t n, int64_t kc, int64_t k)
{
    return (n + 1) * ((min(kc, k > 0 ? k : 1) + 3) / 4 * 4);
}

// Row-major copy of kk columns of B into Bt, vec columns per write (ldt a
// multiple of vec).
template <typename T>
int spmm_copy_chunk(int64_t n, int64_t kk, const T *B, int64_t ldb, T *Bt, int64_t ldt, int vec, hipStream_t s)
{
    if (n == 0) return JLUST_STATUS_SUCCESS;
#define JLUST_TRANSPOSE(V, CT)                                                                             \
    hipLaunchKernelGGL((transpose_kernel<T, V, CT>),                                                       \
                       dim3((unsigned)(n / (4096 / CT) + 1), (unsigned)((kk + CT - 1) / CT)), dim3(256), 0, \
                       s, n, kk, B, ldb, Bt, ldt)
#define JLUST_TRANSPOSE_CT(V)                \
    do {                                     \
        if (kk <= 16) JLUST_TRANSPOSE(V, 16); \
        else if (kk <= 32) JLUST_TRANSPOSE(V, 32); \
        else JLUST_TRANSPOSE(V, 64);         \
    } while (0)
    if (vec == 1) JLUST_TRANSPOSE_CT(1);
    else if (vec == 2) JLUST_TRANSPOSE_CT(2);
    else JLUST_TRANSPOSE_CT((16 / (int)sizeof(T)));
#undef JLUST_TRANSPOSE_CT
#undef JLUST_TRANSPOSE
    return check_launch("transpose_kernel");
}

// Rows per block of the rows kernel for `rows` rows of `mean` entries.  A round
// gives each of the block's ngb groups one slice; as many rounds as 64 lanes
// hold rows, fewer where the result tile would pass 9 KB (8 blocks per CU want
// 20 KB each; columns of C still get whole 128-byte lines), where the staged
// entries would not fit and where the rows would not make 1024 blocks.
template <typename T>
int spmm_rows_per_block(int64_t rows, int64_t mean, int ngb, int slice_log2, int cld)
{
    const int64_t slices = ((mean - 1) >> slice_log2) + 1;
    const int64_t step = min(max(ngb / slices, (int64_t)1), (int64_t)64), line = 128 / sizeof(T);
    int64_t r = 64 / step * step;
    while (r > step && r - step >= line && r * cld * (int64_t)sizeof(T) > (9 << 10)) r -= step;
    while (r > step && (r * mean > 1800 || rows / r < 1024)) r -= step;
    return (int)r;
}

template <typename T, int VEC>
int spmm_rows_launch(int64_t n, int64_t kk, int64_t nnz_rows, int64_t nnz_seg, int32_t origin, SpmmJob<T> ja,
                     SpmmJob<T> jb, const int32_t *colind, const T *val, const T *Bt, int64_t ldt, hipStream_t s)
{
    const int64_t ny = (kk + 64 * VEC - 1) / (64 * VEC);
    SpmmShape sh;
    sh.k = kk;
    sh.ldt = ldt;
    sh.zero_row = n;
    sh.cols = (int)(((kk + ny - 1) / ny + VEC - 1) / VEC * VEC);
    sh.L = sh.cols / VEC;
    sh.cld = sh.cols | 1;
    const int ngb = 64 / sh.L * (SPMM_BLOCK / 64);
    sh.slice_log2 = sh.L <= 8 ? 5 : sh.L <= 16 ? 6 : sh.L <= 32 ? 7 : 8;
    const int64_t mean_a = ja.rows ? nnz_rows / ja.rows + 1 : 1, mean_b = jb.rows ? nnz_seg / jb.rows + 1 : 1;
    ja.R = spmm_rows_per_block<T>(ja.rows, mean_a, ngb, sh.slice_log2, sh.cld);
    jb.R = spmm_rows_per_block<T>(jb.rows, mean_b, ngb, sh.slice_log2, sh.cld);
    const int64_t nb = (ja.rows + ja.R - 1) / ja.R;
    ja.run = xcd_run(nb);
    ja.blocks = (unsigned)((nb + ja.run * NUM_XCD - 1) / (ja.run * NUM_XCD) * (ja.run * NUM_XCD));
    jb.blocks = (unsigned)((jb.rows + jb.R - 1) / jb.R);
    sh.rmax = max(ja.R, jb.rows ? jb.R : 1);
    const int64_t want = max(ja.R * mean_a * 9 / 8, jb.rows ? jb.R * mean_b : 0) + 32;
    sh.ch = (int)min(max(want, ((int64_t)1 << sh.slice_log2) + 32), (int64_t)SPMM_STAGE);
    sh.xmax = (sh.ch >> sh.slice_log2) + 2;
    const size_t lds = sizeof(T) * (size_t)(sh.ch + 2 + (sh.rmax + sh.xmax) * sh.cld) + 4 * (size_t)(sh.ch + 1);
    const dim3 grid(ja.blocks + jb.blocks, (unsigned)ny);
    // 8 entries in flight per group for long f64 rows (27-point mesh, k = 128:
    // 558 -> 523 us), else 4: short rows would load past their ends (1M
    // power-law rows of 5, f64, k = 64: 827 -> 752 us), and f32 gains nothing.
    // Eight sums per column up to 8 columns, four up to 16, else two: counted
    // over rows of 32 entries and fewer, no more error than the 64 / p sums of
    // a row split over a wave's lanes (p the power of two at the columns or
    // above; four sums for 8 columns made 1.09 times that).
#define JLUST_ROWS(U, ACC, BIG)                                                                               \
    hipLaunchKernelGGL((csr_spmm_rows_kernel<T, VEC, U, ACC, BIG>), grid, dim3(SPMM_BLOCK), lds, s, ja, jb, sh, \
                       origin, colind, val, Bt)
    // Only what spmm_chunk_kind's columns per lane leave to choose from.
    constexpr bool SOME8 = VEC <= 2, SOME4 = VEC >= 2;
    constexpr int DEEP = sizeof(T) == 8 ? 8 : 4;
    const bool big = (uint64_t)(n + 1) * (uint64_t)ldt * sizeof(T) > 0xffffff00ull;
    const bool deep = DEEP == 8 && mean_a > 20;
    if constexpr (SOME8) {
        if (!SOME4 || kk <= 8) {
            if (big) JLUST_ROWS(4, 8, true);
            else JLUST_ROWS(4, 8, false);
            return check_launch("csr_spmm_rows_kernel");
        }
    }
    if constexpr (SOME4) {
        if (big) JLUST_ROWS(4, 4, true);
        else if (kk <= 16 && deep) JLUST_ROWS(DEEP, 4, false);
        else if (kk <= 16) JLUST_ROWS(4, 4, false);
        else if (deep) JLUST_ROWS(DEEP, 2, false);
        else JLUST_ROWS(4, 2, false);
    }
#undef JLUST_ROWS
    return check_launch("csr_spmm_rows_kernel");
}

template <typename T>
int spmm_rows_pass(int64_t n, int64_t kk, int64_t nnz_rows, int64_t nnz_seg, int32_t origin, const SpmmJob<T> &ja,
                   const SpmmJob<T> &jb, const int32_t *colind, const T *val, const T *Bt, const SpmmChunk &ck,
                   hipStream_t s)
{
    auto run = [&](auto V) {
        return spmm_rows_launch<T, decltype(V)::value>(n, kk, nnz_rows, nnz_seg, origin, ja, jb, colind, val, Bt,
                                                       ck.ldt, s);
    };
    if (ck.vec == 1) return run(std::integral_constant<int, 1>());
    if (ck.vec == 2) return run(std::integral_constant<int, 2>());
    return run(std::integral_constant<int, 16 / sizeof(T)>());
}

// The product of one narrow chunk over m rows (rows of A, or segments when
// rowend is given) by the group kernel: C[:, 0:kk] (ldc) = alpha * A[rows, :] *
// Bsrc + beta * C, rows flagged in row_skip left untouched.  nnz_rows: the
// entries these rows hold (for the steps per load).
template <typename T>
int spmm_group_launch(int64_t m, int64_t kk, int64_t nnz_rows, int32_t origin, const SpmmJob<T> &j,
                      const int32_t *colind, const T *val, const T *Bsrc, int64_t ldt, hipStream_t s)
{
    if (m == 0) return JLUST_STATUS_SUCCESS;
    const dim3 grid((unsigned)((m + SPMM_ROWS - 1) / SPMM_ROWS));
#define JLUST_GROUP_U(KV, U)                                                                                \
    hipLaunchKernelGGL((csr_spmm_group_kernel<T, KV, U>), grid, dim3(SPMM_BLOCK), 0, s, m, kk, origin, j.lo, \
                       colind, val, Bsrc, ldt, j.alpha, j.beta, j.beta_zero, j.C, j.ldc, j.skip_empty_rows,  \
                       j.hi, j.skip)
#define JLUST_GROUP(KV)                                                                                \
    do {                                                                                               \
        const int64_t steps = (nnz_rows + m * (64 / KV) - 1) / (m * (64 / KV));  /* per row */          \
        if (steps <= 1) JLUST_GROUP_U(KV, 1);                                                          \
        else if (steps <= 2) JLUST_GROUP_U(KV, 2);                                                     \
        else if (steps <= 4) JLUST_GROUP_U(KV, 4);                                                     \
        else JLUST_GROUP_U(KV, 8);                                                                     \
    } while (0)
    if (kk == 1) {
        JLUST_GROUP(1);
    } else if (kk == 2) {
        JLUST_GROUP(2);
    } else {
        if constexpr (sizeof(T) == 4) JLUST_GROUP(4);   // f64: 2 columns at most (spmm_chunk_kind)
    }
#undef JLUST_GROUP
#undef JLUST_GROUP_U
    return check_launch("csr_spmm_group_kernel");
}

// One column chunk over the rows of ja and the segments of jb.
template <typename T>
int spmm_chunk(int64_t n, int64_t kk, int64_t nnz_rows, int64_t nnz_seg, int32_t origin, const SpmmJob<T> &ja,
               const SpmmJob<T> &jb, const int32_t *colind, const T *val, const T *B, int64_t ldb, T *Bt,
               hipStream_t s)
{
    // The mean over all entries, so that a plan and a plain call choose alike.
    const int64_t mean = ja.rows ? (nnz_rows + nnz_seg) / ja.rows : 0;
    const SpmmChunk ck = spmm_chunk_kind<T>(n, kk, mean);
    if (!ck.direct)
        if (int st = spmm_copy_chunk<T>(n, kk, B, ldb, Bt, ck.ldt, ck.vec, s)) return st;
    if (ck.group) {
        const T *Bsrc = ck.direct ? B : Bt;
        if (int st = spmm_group_launch<T>(ja.rows, kk, nnz_rows, origin, ja, colind, val, Bsrc, ck.ldt, s)) return st;
        return spmm_group_launch<T>(jb.rows, kk, nnz_seg, origin, jb, colind, val, Bsrc, ck.ldt, s);
    }
    return spmm_rows_pass<T>(n, kk, nnz_rows, nnz_seg, origin, ja, jb, colind, val, Bt, ck, s);
}

int check_spmm_args(const char *who, int64_t m, int64_t n, int64_t k, int64_t nnz, int32_t origin,
                    const void *rowptr, const void *colind, const void *val)
{
    if (m < 0 || n < 0 || k < 0 || nnz < 0) return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: negative extent", who);
    if (m > INT32_MAX - 1 || n > INT32_MAX || nnz > INT32_MAX)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: extents exceed the Int32 index range", who);
    if (int st = check_origin(origin)) return st;
    if ((m > 0 && !rowptr) || bad_ptr(colind, nnz) || bad_ptr(val, nnz))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: null device pointer", who);
    if (nnz > 0 && n == 0) return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: nnz > 0 with n == 0", who);
    return JLUST_STATUS_SUCCESS;
}

int check_dense_args(const char *who, int64_t m, int64_t n, int64_t k, int64_t nnz, const void *B, int64_t ldb,
                     const void *C, int64_t ldc)
{
    if (ldb < (n > 0 ? n : 1) || ldc < (m > 0 ? m : 1))
        return fail(JLUST_STATUS_INVALID_ARGUMENT,
                    "%s: leading dimensions too small (ldb=%lld < n=%lld or ldc=%lld < m=%lld)", who,
                    (long long)ldb, (long long)n, (long long)ldc, (long long)m);
    if (bad_ptr(B, (nnz > 0 && k > 0) ? n : 0) || bad_ptr(C, m * k))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: null device pointer", who);
    return JLUST_STATUS_SUCCESS;
}

template <typename T>
int csr_spmm(int64_t m, int64_t n, int64_t k, int64_t nnz, int32_t origin,
             const int32_t *rowptr, const int32_t *colind, const T *val, T alpha, const T *B,
             int64_t ldb, T beta, T *C, int64_t ldc, int skip_empty_rows, jlust_stream_t stream)
{
    clear_error();
    if (int st = check_spmm_args("csr_spmm", m, n, k, nnz, origin, rowptr, colind, val)) return st;
    if (int st = check_dense_args("csr_spmm", m, n, k, nnz, B, ldb, C, ldc)) return st;
    if (int st = require_device(nullptr)) return st;
    if (m == 0 || k == 0) return JLUST_STATUS_SUCCESS;
    hipStream_t s = (hipStream_t)stream;

    // Column chunks: every B row a nonzero gathers is a random row of the
    // row-major copy; when that copy is larger than the MALL budget the
    // gathers come from HBM, so B is processed in column chunks whose copy
    // fits (config 3: 2 chunks of 64 columns, 3.14 -> 2.56 ms).
    const int64_t kc = spmm_kchunk(n, k, sizeof(T));
    void *ws = nullptr;
    if (int st = scratch(stream, sizeof(T) * (size_t)spmm_copy_elems(n, kc, k), &ws)) return st;
    T *Bt = (T *)ws;
    SpmmJob<T> rows;
    rows.rows = m;
    rows.lo = rowptr;
    rows.alpha = alpha;
    rows.beta = beta;
    rows.beta_zero = beta == T(0);
    rows.ldc = ldc;
    rows.skip_empty_rows = skip_empty_rows;
    for (int64_t c0 = 0; c0 < k; c0 += kc) {
        rows.C = C + c0 * ldc;
        if (int st = spmm_chunk<T>(n, min(kc, k - c0), nnz, 0, origin, rows, SpmmJob<T>(), colind, val, B + c0 * ldb,
                                   ldb, Bt, s))
            return st;
    }
    return JLUST_STATUS_SUCCESS;
}

}  // namespace

int spmm_row_major_copy(int value_type, int64_t n, int64_t k, const void *B, int64_t ldb, void *Bt, int64_t ldt,
                        hipStream_t s)
{
    if (value_type == 0)
        return spmm_copy_chunk<double>(n, k, (const double *)B, ldb, (double *)Bt, ldt, ldt % 2 ? 1 : 2, s);
    return spmm_copy_chunk<float>(n, k, (const float *)B, ldb, (float *)Bt, ldt, ldt % 2 ? 1 : ldt % 4 ? 2 : 4, s);
}

}  // namespace jlust

using namespace jlust;

extern "C" int jlust_hip_csr_spmm_f64_i32(int64_t m, int64_t n, int64_t k, int64_t nnz,
                                          int32_t origin, const int32_t *rowptr,
                                          const int32_t *colind, const double *val, double alpha,
                                          const double *B, int64_t ldb, double beta, double *C,
                                          int64_t ldc, int skip_empty_rows, jlust_stream_t stream)
{
    return csr_spmm<double>(m, n, k, nnz, origin, rowptr, colind, val, alpha, B, ldb, beta, C,
                            ldc, skip_empty_rows, stream);
}

extern "C" int jlust_hip_csr_spmm_f32_i32(int64_t m, int64_t n, int64_t k, int64_t nnz,
                                          int32_t origin, const int32_t *rowptr,
                                          const int32_t *colind, const float *val, float alpha,
                                          const float *B, int64_t ldb, float beta, float *C,
                                          int64_t ldc, int skip_empty_rows, jlust_stream_t stream)
{
    return csr_spmm<float>(m, n, k, nnz, origin, rowptr, colind, val, alpha, B, ldb, beta, C,
                           ldc, skip_empty_rows, stream);
}

// ------------------------------------------------------------------- plans

// A prepared CSR SpMM (the cuSPARSE SpMM handle contract: analysis and
// workspace once, execute many times, update_values! for new values of the
// same pattern; ext/CUDAExt/ops/spmm.jl:8-70).  Analysis: the column chunk
// per pass for the plan's k; the rows longer than SPMM_LONG_ROW, cut into
// segments; the entries left to the row kernels (for their steps per load).
// Workspace: the row-major copy of one column chunk of B and the segments'
// partial rows, so an execute allocates nothing and can be captured.
struct jlust_spmm_plan {
    int64_t m = 0, n = 0, k = 0, nnz = 0;
    int32_t origin = 0;
    int value_type = 0;
    const int32_t *rowptr = nullptr;
    const int32_t *colind = nullptr;
    const void *val = nullptr;
    int device = 0;
    int64_t kc = 1;                 // columns per pass
    void *mem = nullptr;            // one allocation holds everything below
    void *Bt = nullptr;             // n x ldt row-major copy of one column chunk of B
    uint8_t *row_skip = nullptr;    // [m] 1 for a split row (null: none)
    int64_t nlong = 0, nseg = 0;
    int32_t *long_rows = nullptr;   // [nlong] the split rows
    int32_t *seg_first = nullptr;   // [nlong + 1] first segment of each split row
    int32_t *seg_lo = nullptr;      // [nseg] segment start (origin-based, like rowptr)
    int32_t *seg_hi = nullptr;      // [nseg] segment end
    void *part = nullptr;           // nseg x kc partial rows, column-major (ld nseg)
    int64_t nnz_rows = 0;           // entries of the rows that are not split
    // COO/CSC plans (coo_csc.hip): the row order the plan runs on is owned in
    // own_mem; perm (null when the source was already in row order) maps its
    // entries to the caller's, and val_copy holds the values in that order.
    void *own_mem = nullptr;
    const int32_t *perm = nullptr;
    void *val_copy = nullptr;
};

namespace jlust {
int spmm_plan_adopt_reorder(jlust_spmm_plan_t plan, void *mem, const int32_t *perm, void *val_copy)
{
    plan->own_mem = mem;
    plan->perm = perm;
    plan->val_copy = val_copy;
    return JLUST_STATUS_SUCCESS;
}
}  // namespace jlust

static int csr_spmm_plan_create_body(int64_t m, int64_t n, int64_t k, int64_t nnz, int32_t origin,
                                     int value_type, const int32_t *rowptr, const int32_t *colind,
                                     const void *val, jlust_stream_t stream,
                                     jlust_spmm_plan_t *plan_out)
{
    clear_error();
    if (!plan_out) return fail(JLUST_STATUS_INVALID_ARGUMENT, "spmm_plan_create: null plan_out");
    *plan_out = nullptr;
    if (value_type != 0 && value_type != 1)
        return fail(JLUST_STATUS_UNSUPPORTED_VALUE_TYPE,
                    "spmm_plan_create: value_type %d (0 = Float64, 1 = Float32)", value_type);
    if (int st = check_spmm_args("spmm_plan_create", m, n, k, nnz, origin, rowptr, colind, val)) return st;
    int dev = 0;
    if (int st = require_device(&dev)) return st;
    hipStream_t s = (hipStream_t)stream;
    const size_t tsz = value_type == 0 ? sizeof(double) : sizeof(float);
    std::unique_ptr<jlust_spmm_plan> p(new jlust_spmm_plan());
    p->m = m;
    p->n = n;
    p->k = k;
    p->nnz = nnz;
    p->origin = origin;
    p->value_type = value_type;
    p->rowptr = rowptr;
    p->colind = colind;
    p->val = val;
    p->device = dev;
    p->kc = k > 0 ? spmm_kchunk(n, k, tsz) : 1;
    p->nnz_rows = nnz;

    // Row analysis on the host copy of rowptr: which rows to split.
    std::vector<int32_t> rp((size_t)(m + 1));
    if (m > 0) {
        JLUST_HIP_TRY(hipMemcpyAsync(rp.data(), rowptr, sizeof(int32_t) * (size_t)(m + 1), hipMemcpyDeviceToHost, s));
        JLUST_HIP_TRY(hipStreamSynchronize(s));
        if ((int64_t)rp[0] != origin || (int64_t)rp[m] - origin != nnz)
            return fail(JLUST_STATUS_NONCANONICAL_STORAGE,
                        "spmm_plan_create: rowptr runs from %d to %d, expected %d to %lld", rp[0], rp[m], origin,
                        (long long)(nnz + origin));
    }
    std::vector<int32_t> long_rows, seg_first, seg_lo, seg_hi;
    for (int64_t i = 0; i < m; ++i) {
        const int64_t len = (int64_t)rp[i + 1] - rp[i];
        if (len < 0)
            return fail(JLUST_STATUS_NONCANONICAL_STORAGE, "spmm_plan_create: rowptr decreases at row %lld",
                        (long long)i);
        if (len <= SPMM_LONG_ROW) continue;
        long_rows.push_back((int32_t)i);
        seg_first.push_back((int32_t)seg_lo.size());
        for (int64_t a = rp[i]; a < rp[i + 1]; a += SPMM_SEG) {
            seg_lo.push_back((int32_t)a);
            seg_hi.push_back((int32_t)min(a + SPMM_SEG, (int64_t)rp[i + 1]));
        }
        p->nnz_rows -= len;
    }
    seg_first.push_back((int32_t)seg_lo.size());
    p->nlong = (int64_t)long_rows.size();
    p->nseg = (int64_t)seg_lo.size();
    std::vector<uint8_t> skip(p->nlong ? (size_t)m : 0, 0);   // host tables before the device allocation
    for (int32_t r : long_rows) skip[(size_t)r] = 1;

    // One allocation: B copy, row flags, segment tables, partial rows.
    const size_t sz_bt = align_up(tsz * (size_t)spmm_copy_elems(n, p->kc, k), 256);
    const size_t sz_skip = p->nlong ? align_up((size_t)m, 256) : 0;
    const size_t sz_lr = align_up(sizeof(int32_t) * (size_t)(p->nlong + 1), 256);
    const size_t sz_sg = align_up(sizeof(int32_t) * (size_t)(p->nseg > 0 ? p->nseg : 1), 256);
    const size_t sz_part = p->nseg ? align_up(tsz * (size_t)p->nseg * (size_t)p->kc, 256) : 0;
    JLUST_HIP_TRY(hipMalloc(&p->mem, sz_bt + sz_skip + 2 * sz_lr + 2 * sz_sg + sz_part));
    char *b = (char *)p->mem;
    p->Bt = b;                           b += sz_bt;
    if (p->nlong) { p->row_skip = (uint8_t *)b; b += sz_skip; }
    p->long_rows = (int32_t *)b;         b += sz_lr;
    p->seg_first = (int32_t *)b;         b += sz_lr;
    p->seg_lo = (int32_t *)b;            b += sz_sg;
    p->seg_hi = (int32_t *)b;            b += sz_sg;
    if (p->nseg) p->part = b;
    int st = JLUST_STATUS_SUCCESS;
    if (p->nlong) {
        hipError_t e = hipMemcpyAsync(p->row_skip, skip.data(), (size_t)m, hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(p->long_rows, long_rows.data(), sizeof(int32_t) * long_rows.size(),
                               hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(p->seg_first, seg_first.data(), sizeof(int32_t) * seg_first.size(),
                               hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(p->seg_lo, seg_lo.data(), sizeof(int32_t) * seg_lo.size(), hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(p->seg_hi, seg_hi.data(), sizeof(int32_t) * seg_hi.size(), hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);   // the host tables go out of scope
        if (e != hipSuccess) st = hip_fail(e, "spmm_plan_create: table upload");
    }
    if (st) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(p->mem);
        return st;
    }
    *plan_out = p.release();
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_csr_spmm_plan_create(int64_t m, int64_t n, int64_t k, int64_t nnz, int32_t origin,
                                              int value_type, const int32_t *rowptr, const int32_t *colind,
                                              const void *val, jlust_stream_t stream,
                                              jlust_spmm_plan_t *plan_out)
{
    return jlust::host_guard("csr_spmm_plan_create", [&] {
        return csr_spmm_plan_create_body(m, n, k, nnz, origin, value_type, rowptr, colind, val, stream,
                                         plan_out);
    });
}

extern "C" int jlust_hip_csr_spmm_plan_update_values(jlust_spmm_plan_t plan, const void *val,
                                                     jlust_stream_t stream)
{
    clear_error();
    if (!plan) return fail(JLUST_STATUS_INVALID_ARGUMENT, "spmm_plan_update_values: null plan");
    if (bad_ptr(val, plan->nnz)) return fail(JLUST_STATUS_INVALID_ARGUMENT, "spmm_plan_update_values: null values");
    if (!plan->perm) {
        plan->val = val;    // the kernels read the values in place: nothing to copy
        return JLUST_STATUS_SUCCESS;
    }
    // A reordered COO/CSC plan: the values into its row order, on the stream.
    int dev = 0;
    if (int st = require_device(&dev)) return st;
    if (dev != plan->device)
        return fail(JLUST_STATUS_INVALID_ARGUMENT,
                    "spmm_plan_update_values: plan belongs to device %d, current device is %d", plan->device, dev);
    return perm_gather(plan->value_type, plan->nnz, plan->perm, val, plan->val_copy, (hipStream_t)stream);
}

template <typename T>
static int spmm_plan_execute(jlust_spmm_plan_t p, int want_type, T alpha, const T *B, int64_t ldb, T beta, T *C,
                             int64_t ldc, int skip_empty_rows, jlust_stream_t stream)
{
    clear_error();
    if (!p) return fail(JLUST_STATUS_INVALID_ARGUMENT, "spmm_plan_execute: null plan");
    if (p->value_type != want_type)
        return fail(JLUST_STATUS_UNSUPPORTED_VALUE_TYPE, "spmm_plan_execute: plan was created for %s values",
                    p->value_type == 0 ? "Float64" : "Float32");
    if (int st = check_dense_args("spmm_plan_execute", p->m, p->n, p->k, p->nnz, B, ldb, C, ldc)) return st;
    int dev = 0;
    if (int st = require_device(&dev)) return st;
    if (dev != p->device)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "spmm_plan_execute: plan belongs to device %d, current device is %d",
                    p->device, dev);
    if (p->m == 0 || p->k == 0) return JLUST_STATUS_SUCCESS;
    hipStream_t s = (hipStream_t)stream;
    const T *val = (const T *)p->val;
    T *Bt = (T *)p->Bt;
    T *part = (T *)p->part;
    const int bz = beta == T(0);
    SpmmJob<T> rows, segs;
    rows.rows = p->m;
    rows.lo = p->rowptr;
    rows.skip = p->row_skip;
    rows.alpha = alpha;
    rows.beta = beta;
    rows.beta_zero = bz;
    rows.ldc = ldc;
    rows.skip_empty_rows = skip_empty_rows;
    segs.rows = p->nseg;
    segs.lo = p->seg_lo;
    segs.hi = p->seg_hi;
    segs.alpha = T(1);
    segs.C = part;
    segs.ldc = p->nseg;
    for (int64_t c0 = 0; c0 < p->k; c0 += p->kc) {
        const int64_t kk = min(p->kc, p->k - c0);
        rows.C = C + c0 * ldc;
        if (int st = spmm_chunk<T>(p->n, kk, p->nnz_rows, p->nnz - p->nnz_rows, p->origin, rows, segs, p->colind, val,
                                   B + c0 * ldb, ldb, Bt, s))
            return st;
        if (p->nseg == 0) continue;
        const int64_t t = p->nlong * kk;
        hipLaunchKernelGGL((spmm_long_reduce_kernel<T>), dim3((unsigned)((t + 255) / 256)), dim3(256), 0, s,
                           p->nlong, kk, p->long_rows, p->seg_first, part, p->nseg, alpha, beta, bz,
                           C + c0 * ldc, ldc);
        if (int st = check_launch("spmm_long_reduce_kernel")) return st;
    }
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_csr_spmm_plan_execute_f64(jlust_spmm_plan_t plan, double alpha, const double *B,
                                                   int64_t ldb, double beta, double *C, int64_t ldc,
                                                   int skip_empty_rows, jlust_stream_t stream)
{
    return spmm_plan_execute<double>(plan, 0, alpha, B, ldb, beta, C, ldc, skip_empty_rows, stream);
}

extern "C" int jlust_hip_csr_spmm_plan_execute_f32(jlust_spmm_plan_t plan, float alpha, const float *B,
                                                   int64_t ldb, float beta, float *C, int64_t ldc,
                                                   int skip_empty_rows, jlust_stream_t stream)
{
    return spmm_plan_execute<float>(plan, 1, alpha, B, ldb, beta, C, ldc, skip_empty_rows, stream);
}

extern "C" int jlust_hip_csr_spmm_plan_info(jlust_spmm_plan_t plan, int64_t *split_rows, int64_t *segments,
                                            int64_t *cols_per_pass, int32_t *reordered)
{
    clear_error();
    if (!plan) return fail(JLUST_STATUS_INVALID_ARGUMENT, "spmm_plan_info: null plan");
    if (split_rows) *split_rows = plan->nlong;
    if (segments) *segments = plan->nseg;
    if (cols_per_pass) *cols_per_pass = plan->kc;
    if (reordered) *reordered = plan->perm != nullptr;
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_csr_spmm_plan_destroy(jlust_spmm_plan_t plan)
{
    clear_error();
    if (!plan) return JLUST_STATUS_SUCCESS;
    // Work queued on any stream may still read the plan's buffers.
    hipError_t e = hipDeviceSynchronize();
    for (void *m : {plan->mem, plan->own_mem}) {
        if (!m) continue;
        const hipError_t e2 = hipFree(m);
        if (e == hipSuccess) e = e2;
    }
    delete plan;
    if (e != hipSuccess) return hip_fail(e, "spmm_plan_destroy");
    return JLUST_STATUS_SUCCESS;
}

namespace jlust {
int preload_spmm()
{
    JLUST_PRELOAD_KERNEL((transpose_kernel<float, 4, 64>));
    return JLUST_STATUS_SUCCESS;
}
}  // namespace jlust
