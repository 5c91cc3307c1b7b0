// convert.hip -- bit-exact sparse format conversions on the GPU.
//
// Restates JLUST's convert_format (src/convert.jl:302-388) for the hot-path
// formats CSR, CSC, COO, DCSR and BSR (src/named_formats.jl:24-27,106-128):
//   1. every stored entry is visited in storage order (TensorDecomposer,
//      convert.jl:5-122) and explicit zeros are dropped (convert.jl:316);
//   2. entries are keyed by their coordinates in the target's level order
//      (dim2lvl) and sorted stably unless the target is the identity
//      ordering and the source is ordered identity (convert.jl:331-349);
//   3. the target's buffers are composed (TensorComposer, convert.jl:124-299):
//      on a unique level, adjacent entries with equal coordinates form one
//      segment and only the first value of a segment is kept; Dense levels
//      of a block are zero-filled;
//   4. the result keeps the source's index origin (convert.jl:363-377).
// Pipeline on the device: per-entry coordinates (segment ids by scatter +
// max-scan), zero-drop compaction, stable LSD radix sort (rocPRIM) of packed
// level keys with source positions as values, adjacent-key dedup, then the
// target's pos/crd/val from the sorted keys.  CSR to CSC and CSC to CSR or COO
// move whole entries by coordinate instead (convert_direct), and CSR to small
// blocks goes by block-rows (convert_blocks).  Integer work only; values are
// moved as bits.
//
// Also: sparse_to_dense (ext/KernelAbstractionsExt/ops/conversion.jl:47-65)
// and the index shift of materialize's origin change (CUDAExt.jl:199-220).
#include <algorithm>
#include <cstring>

#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "common.hpp"
#include "wave.hpp"

namespace jlust {
namespace {

constexpr int CV_BLOCK = 256;

unsigned cv_grid(int64_t n) { return (unsigned)((n + CV_BLOCK - 1) / CV_BLOCK); }

int bits_for(int64_t n)             // bits to hold values in [0, n)
{
    int b = 0;
    while (b < 63 && ((int64_t)1 << b) < n) ++b;
    return b;
}

// Level layout of a target format: the key of an entry is
//   major << (minor_bits + inner_bits) | minor << inner_bits | inner,
// with (major, minor) = (row, col) for CSR/COO/DCSR, (col, row) for CSC and
// (block row, block col) for BSR, whose `inner` is the position inside the
// block in storage order (row-major: ii*b2 + jj, column-major: jj*b1 + ii).
struct KeyLayout {
    int fmt = 0;
    int b1 = 1, b2 = 1, row_major = 1;
    int minor_bits = 0, inner_bits = 0, total_bits = 0;
    int64_t major_dim = 0, minor_dim = 0;
};

__device__ __forceinline__ uint64_t make_key(const KeyLayout &L, int64_t row, int64_t col)
{
    uint64_t major, minor, inner = 0;
    if (L.fmt == JLUST_FORMAT_CSC) {
        major = (uint64_t)col;
        minor = (uint64_t)row;
    } else if (L.fmt == JLUST_FORMAT_BSR) {
        major = (uint64_t)(row / L.b1);
        minor = (uint64_t)(col / L.b2);
        const int64_t ii = row % L.b1, jj = col % L.b2;
        inner = (uint64_t)(L.row_major ? ii * L.b2 + jj : jj * L.b1 + ii);
    } else {
        major = (uint64_t)row;
        minor = (uint64_t)col;
    }
    return (major << (L.minor_bits + L.inner_bits)) | (minor << L.inner_bits) | inner;
}

__device__ __forceinline__ int64_t key_major(const KeyLayout &L, uint64_t k)
{
    return (int64_t)(k >> (L.minor_bits + L.inner_bits));
}
__device__ __forceinline__ int64_t key_minor(const KeyLayout &L, uint64_t k)
{
    return (int64_t)((k >> L.inner_bits) & ((1ull << L.minor_bits) - 1));
}
__device__ __forceinline__ int64_t key_inner(const KeyLayout &L, uint64_t k)
{
    return (int64_t)(k & ((1ull << L.inner_bits) - 1));
}
// Key without the inner part: identifies a BSR block.
__device__ __forceinline__ uint64_t key_block(const KeyLayout &L, uint64_t k)
{
    return k >> L.inner_bits;
}

// ------------------------------------------------------------- kernels

// mark[ptr[s] - origin] = s for every nonempty segment s < nseg (positions
// below len); with mark zero-initialised, an inclusive max-scan then gives the
// segment of every position.
__global__ void seg_mark_kernel(const int32_t *__restrict__ ptr, int64_t nseg, int32_t origin,
                                int64_t len, int32_t *__restrict__ mark)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    const int64_t a = (int64_t)ptr[s] - origin, b = (int64_t)ptr[s + 1] - origin;
    if (b > a && a >= 0 && a < len) mark[a] = (int32_t)s;
}

// Per stored value p: its (row, col), a keep flag (value != 0) and its key;
// *dropped (if given) counts the values not kept, one atomic per wave that
// drops any.
template <typename T>
__global__ void decompose_kernel(jlust_sparse src, const int32_t *__restrict__ seg, KeyLayout L,
                                 uint64_t *__restrict__ keys, int32_t *__restrict__ keep,
                                 int32_t *__restrict__ bad, int32_t *__restrict__ dropped)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= src.nnz) return;
    const int32_t o = src.origin;
    int64_t row = 0, col = 0;
    switch (src.format) {
    case JLUST_FORMAT_CSR: row = seg[p]; col = (int64_t)src.crd2[p] - o; break;
    case JLUST_FORMAT_CSC: col = seg[p]; row = (int64_t)src.crd2[p] - o; break;
    case JLUST_FORMAT_COO: row = (int64_t)src.crd1[p] - o; col = (int64_t)src.crd2[p] - o; break;
    case JLUST_FORMAT_DCSR: row = (int64_t)src.crd1[seg[p]] - o; col = (int64_t)src.crd2[p] - o; break;
    default: {                                   // BSR: seg holds the block row of each block
        const int64_t bs = (int64_t)src.b1 * src.b2;
        const int64_t q = p / bs, e = p % bs;
        const int64_t ii = src.row_major_blocks ? e / src.b2 : e % src.b1;
        const int64_t jj = src.row_major_blocks ? e % src.b2 : e / src.b1;
        row = (int64_t)seg[q] * src.b1 + ii;
        col = ((int64_t)src.crd2[q] - o) * src.b2 + jj;
    }
    }
    const bool inb = row >= 0 && row < src.m && col >= 0 && col < src.n;
    if (!inb) bad[0] = 1;
    const T v = static_cast<const T *>(src.val)[p];
    const bool kp = inb && v != T(0);           // -0.0 == 0 is dropped, NaN kept
    keep[p] = kp ? 1 : 0;
    keys[p] = inb ? make_key(L, row, col) : 0;
    if (dropped) {
        const uint64_t d = __ballot(!kp);
        if (d && __lane_id() == (int)__builtin_ctzll(__ballot(1))) atomicAdd(dropped, (int32_t)__popcll(d));
    }
}

__global__ void iota_kernel(int64_t n, int32_t *__restrict__ p)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int32_t)i;
}

// out[idx[i]] = in[i] for flagged i, idx = exclusive scan of the flags.
__global__ void compact_kernel(int64_t n, const int32_t *__restrict__ flag,
                               const int32_t *__restrict__ idx, const uint64_t *__restrict__ kin,
                               const int32_t *__restrict__ pin, uint64_t *__restrict__ kout,
                               int32_t *__restrict__ pout)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !flag[i]) return;
    kout[idx[i]] = kin[i];
    pout[idx[i]] = pin ? pin[i] : (int32_t)i;
}

// head[i] = 1 where key (or, with block_only, its block) differs from i-1;
// *repeats (if given) counts the others, one atomic per wave that has any.
__global__ void head_kernel(int64_t n, const uint64_t *__restrict__ k, KeyLayout L, int block_only,
                            int32_t *__restrict__ head, int32_t *__restrict__ repeats)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    bool h = i == 0;
    if (!h) h = block_only ? key_block(L, k[i]) != key_block(L, k[i - 1]) : k[i] != k[i - 1];
    head[i] = h ? 1 : 0;
    if (repeats) {
        const uint64_t r = __ballot(!h);
        if (r && __lane_id() == (int)__builtin_ctzll(__ballot(1))) atomicAdd(repeats, (int32_t)__popcll(r));
    }
}

// Sets bad[0] when the major coordinate decreases (an unsorted "ordered" source).
__global__ void major_order_kernel(int64_t n, const uint64_t *__restrict__ k, KeyLayout L,
                                   int32_t *__restrict__ bad)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0 || i >= n) return;
    if (key_major(L, k[i]) < key_major(L, k[i - 1])) bad[0] = 1;
}

// ptr[r] = origin + first i with major(key[i]) >= r, for r in [0, nmajor].
// `major` (if given) holds per-item majors instead of keys.
__global__ void lower_bound_ptr_kernel(int64_t n, const uint64_t *__restrict__ k,
                                       const int32_t *__restrict__ major, KeyLayout L,
                                       int64_t nmajor, int32_t origin, int32_t *__restrict__ ptr)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nmajor) return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        const int64_t mj = major ? (int64_t)major[mid] : key_major(L, k[mid]);
        if (mj < r) lo = mid + 1;
        else hi = mid;
    }
    ptr[r] = (int32_t)(lo + origin);
}

// Entry arrays of CSR/CSC/COO/DCSR targets (pos null: entry i is stored value i).
template <typename T>
__global__ void fill_entries_kernel(int64_t n, const uint64_t *__restrict__ k,
                                    const int32_t *__restrict__ pos, KeyLayout L, int32_t origin,
                                    const T *__restrict__ sval, int32_t *__restrict__ major_out,
                                    int32_t *__restrict__ minor_out, T *__restrict__ val_out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (major_out) major_out[i] = (int32_t)(key_major(L, k[i]) + origin);
    minor_out[i] = (int32_t)(key_minor(L, k[i]) + origin);
    val_out[i] = sval[pos ? pos[i] : i];
}

// DCSR: at run heads of the row, crd1[run] = row + origin and pos2[run] = i + origin.
__global__ void fill_runs_kernel(int64_t n, const uint64_t *__restrict__ k,
                                 const int32_t *__restrict__ head, const int32_t *__restrict__ run,
                                 KeyLayout L, int32_t origin, int64_t nruns,
                                 int32_t *__restrict__ crd1, int32_t *__restrict__ pos2,
                                 int32_t *__restrict__ pos1)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        pos2[nruns] = (int32_t)(n + origin);
        if (pos1) {
            pos1[0] = origin;
            pos1[1] = (int32_t)(nruns + origin);
        }
    }
    if (i >= n || !head[i]) return;
    crd1[run[i]] = (int32_t)(key_major(L, k[i]) + origin);
    pos2[run[i]] = (int32_t)(i + origin);
}

// BSR target: block b = run[i] of entry i; at block heads the block column
// and block row; every entry's value into its block slot (pos as above).
template <typename T>
__global__ void fill_bsr_kernel(int64_t n, const uint64_t *__restrict__ k,
                                const int32_t *__restrict__ pos, const int32_t *__restrict__ head,
                                const int32_t *__restrict__ run, KeyLayout L, int32_t origin,
                                const T *__restrict__ sval, int32_t *__restrict__ bcol,
                                int32_t *__restrict__ brow, T *__restrict__ val_out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t b = run[i];
    if (head[i]) {
        bcol[b] = (int32_t)(key_minor(L, k[i]) + origin);
        brow[b] = (int32_t)key_major(L, k[i]);
    }
    val_out[b * L.b1 * L.b2 + key_inner(L, k[i])] = sval[pos ? pos[i] : i];
}

template <typename T>
__global__ void zero_kernel(int64_t n, T *__restrict__ p)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = T(0);
}

__global__ void pair_kernel(int32_t *__restrict__ p, int32_t a, int32_t b)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        p[0] = a;
        p[1] = b;
    }
}

// dense[row + col*ld] = value of stored entry i (keys in CSR layout).
template <typename T>
__global__ void to_dense_kernel(int64_t n, const uint64_t *__restrict__ k, KeyLayout L,
                                const T *__restrict__ sval, T *__restrict__ dense, int64_t ld)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t row = key_major(L, k[i]), col = key_minor(L, k[i]);
    dense[row + col * ld] = sval[i];
}

__global__ void shift_kernel(int64_t n, int32_t *__restrict__ dst, const int32_t *__restrict__ src,
                             int32_t delta)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i] + delta;
}

// --------------------------------------------- CSR <-> CSC and CSC -> COO
//
// A conversion that orders the entries by the source's inner coordinate and
// keeps their order otherwise (sort_bits' major_only) is a stable sort of
// (coordinate, segment, value) by the coordinate.  The general path sorts
// 64-bit keys with positions and then fetches each value from where it was
// stored: 16M f64 entries take 480 us of sorting, 326 of random 8-byte reads
// and 250 of passes that make and check the keys.  Here an entry moves whole,
// 16 bytes, in passes of up to CS_BITS bits (two for up to 4M columns), the
// first of which reads the source and the last of which writes the target.
//
// What bounds it: memory, 32 bytes an entry and pass.  A workgroup takes
// CS_TILE consecutive entries, ranks them by digit (equal digits of a wave
// found by ballots, in order; waves by a table in LDS), puts them in digit
// order in LDS and writes each digit's stretch at its place, found by a scan
// of the tiles' digit counts.  The larger the tile, the longer the stretches:
// 8,192 entries leave 8 of each of 1,024 digits, 64 bytes of values.
// Consecutive tiles go to the same XCD, so that their stretches, which are
// neighbours, meet in one L2.
//
// 16M f64 entries of 1,000,003 columns (512 MB of traffic a pass): the first
// pass' count 28 us (67 when it read the values too, to drop zeros), the
// second's 20, each move 163 (3.1 TB/s; 16 entries a thread without spills, two
// tiles a CU; 1,024 threads of 8 in 64 registers took 195, with spills 285),
// scans 18, repeats 24, pointers 28: a whole conversion 508 us, 1,196 by the
// general path.  With 5 % of zeros, which cost a second run, 1,113 us against
// 3,992.  10,007 rows of 9: 126 us, 260 there, both mostly launches.
constexpr int CS_THREADS = 512, CS_WAVES = CS_THREADS / 64, CS_ITEMS = 16;
constexpr int CS_TILE = CS_THREADS * CS_ITEMS;
// A tile's workgroup walks up to this many segments; past it the entries search
// theirs (1.4M f64 entries, 20M empty segments among them: 12.3 ms -> 240 us; 33k
// of them: 183 us either way).
constexpr int CS_GAP = 4 * CS_TILE;
constexpr int CC_THREADS = 1024, CC_ITEMS = CS_TILE / CC_THREADS;      // the counting kernel
constexpr int CS_BITS = 11;
constexpr int CS_DIGITS = 1 << CS_BITS;
constexpr int CS_WPT = CS_DIGITS / 2 / CS_THREADS;       // pairs of digits a thread

struct SortPass {
    int shift, bits;                       // the digit
    int64_t ntiles;
};

__device__ __forceinline__ int64_t sort_tile(int64_t ntiles)
{
    const int64_t per = (ntiles + 7) / 8;
    return (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

enum { CS_BAD = 0, CS_POINTERS = 1, CS_REPEATS = 2, CS_COUNT = 3, CS_ZEROS = 4 };     // flags[]

// The source of a pass: the entries of the pass before, the source's, or the
// source's without its zeros.
enum SortFrom { CS_ENTRIES, CS_SOURCE, CS_NONZEROS };

// hist[digit * ntiles + tile]: how often the tile's entries hold the digit.
// The first pass reads the source and checks the coordinates and the segment
// pointers; the others read the keys of the pass before.
template <typename T, int FROM>
__global__ __launch_bounds__(CC_THREADS) void sort_count_kernel(jlust_sparse src, int64_t nseg, int64_t major_dim,
                                                                const uint32_t *__restrict__ keys, SortPass ps,
                                                                int32_t *__restrict__ hist,
                                                                int32_t *__restrict__ flags)
{
    constexpr bool FIRST = FROM != CS_ENTRIES;
    __shared__ uint32_t h[CS_DIGITS];
    const int64_t tile = sort_tile(ps.ntiles);
    if (tile >= ps.ntiles) return;
    const int nd = 1 << ps.bits, tid = threadIdx.x;
    const int64_t n = FIRST ? src.nnz : (int64_t)flags[CS_COUNT];
    for (int d = tid; d < nd; d += CC_THREADS) h[d] = 0;
    __syncthreads();
    bool bad = false;
    if (tile * CS_TILE < n) {
        // All loads first; threads past the end read the last entry.
        const int64_t p0 = tile * CS_TILE + tid;
        int64_t key[CC_ITEMS];
        bool valid[CC_ITEMS];
#pragma unroll
        for (int j = 0; j < CC_ITEMS; ++j) {
            const int64_t p = min(p0 + j * CC_THREADS, n - 1);
            valid[j] = p0 + j * CC_THREADS < n;
            if (FIRST) {
                key[j] = (int64_t)src.crd2[p] - src.origin;
                const bool inb = key[j] >= 0 && key[j] < major_dim;
                bad = bad || !inb;
                valid[j] = valid[j] && inb;
                if (FROM == CS_NONZEROS)                         // no -0.0; NaN kept
                    valid[j] = valid[j] && static_cast<const T *>(src.val)[p] != T(0);
            } else {
                key[j] = keys[p];
            }
        }
#pragma unroll
        for (int j = 0; j < CC_ITEMS; ++j)
            if (valid[j]) atomicAdd(&h[(uint32_t)key[j] >> ps.shift & (nd - 1)], 1u);
    }
    if (FIRST) {
        if (bad) flags[CS_BAD] = 1;
        const int64_t per = (nseg + ps.ntiles - 1) / ps.ntiles;
        bool off = tile == 0 && tid == 0 &&
                   (src.pos2[0] != src.origin || (int64_t)src.pos2[nseg] != src.nnz + src.origin);
        for (int64_t s = tile * per + tid; s < min((tile + 1) * per, nseg); s += CC_THREADS)
            off = off || src.pos2[s + 1] < src.pos2[s];
        if (off) flags[CS_POINTERS] = 1;
    }
    __syncthreads();
    for (int d = tid; d < nd; d += CC_THREADS) hist[(int64_t)d * ps.ntiles + tile] = (int32_t)h[d];
    if (tile == 0 && tid == 0) hist[(int64_t)nd * ps.ntiles] = 0;
}

// The last segment that starts at position p or before (0 if none), by a
// whole wave; ends for any pointer array.
__device__ __forceinline__ int32_t segment_of(const int32_t *__restrict__ ptr, int64_t nseg, int32_t origin, int64_t p)
{
    const int lane = threadIdx.x & 63;
    int64_t lo = 0, hi = nseg;
    while (hi - lo > 1) {
        const int64_t step = (hi - lo + 63) / 64, at = lo + lane * step;
        const bool le = lane == 0 || (at < hi && (int64_t)ptr[at] - origin <= p);
        lo += (63 - __builtin_clzll(__ballot(le))) * step;
        hi = min(hi, lo + step);
    }
    return (int32_t)lo;
}

// One pass: the entries of each tile to their places by digit, hist holding
// the exclusive scan of the counts.  okey gets the coordinate + kadd, ominor
// the segment + madd (the target's index origin in the last pass).
template <typename T, int FROM>
__global__ __launch_bounds__(CS_THREADS, 4) void sort_move_kernel(jlust_sparse src, int64_t nseg, int64_t major_dim,
                                                                  const uint32_t *__restrict__ ikey,
                                                                  const uint32_t *__restrict__ iminor,
                                                                  const T *__restrict__ ival, SortPass ps,
                                                                  const int32_t *__restrict__ hist,
                                                                  int32_t *__restrict__ flags,
                                                                  uint32_t *__restrict__ okey,
                                                                  uint32_t *__restrict__ ominor,
                                                                  T *__restrict__ oval, uint32_t kadd, uint32_t madd)
{
    constexpr bool FIRST = FROM != CS_ENTRIES;
    // In turn: segment marks, the waves' digit counts, the entries in order.
    __shared__ __align__(16) char lds[CS_TILE * 8];
    __shared__ int32_t delta[CS_DIGITS];
    __shared__ int32_t wsum[CS_WAVES];
    __shared__ int32_t seg01[2];
    const int64_t tile = sort_tile(ps.ntiles);
    if (tile >= ps.ntiles) return;
    const int nd = 1 << ps.bits, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t n = FIRST ? src.nnz : (int64_t)flags[CS_COUNT];
    const int64_t t0 = tile * CS_TILE, t1 = min(t0 + CS_TILE, n);
    if (t0 >= n) return;
    const int base = wave * (64 * CS_ITEMS) + lane;       // this thread's entries: base + 64 j
    // An entry's value stays in memory until its place is known, except where
    // zeros are dropped.
    const int last = (int)(t1 - t0) - 1;
    const T *value = (FIRST ? static_cast<const T *>(src.val) : ival) + t0;
    const uint32_t *keys = (FIRST ? reinterpret_cast<const uint32_t *>(src.crd2) : ikey) + t0;
    uint32_t key[CS_ITEMS], minor[CS_ITEMS], valid = 0;
    T val[CS_ITEMS];
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j) {
        const uint32_t i = (uint32_t)min(base + 64 * j, last) & (CS_TILE - 1);
        key[j] = keys[i];
        if (FROM == CS_NONZEROS) val[j] = value[i];
    }
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j) {
        if (FIRST) key[j] -= (uint32_t)src.origin;
        const bool in = base + 64 * j <= last,
                   ok = !FIRST | (((int64_t)key[j] < major_dim) & (FROM != CS_NONZEROS || val[j] != T(0)));
        valid |= (uint32_t)(in & ok) << j;
    }
    if (FIRST) {
        // The entries' segments: each segment marked at its first entry, then
        // a running maximum, unless the tile holds a long run of empty ones.
        int32_t *mark = reinterpret_cast<int32_t *>(lds);
        if (wave < 2) {
            const int32_t s = segment_of(src.pos2, nseg, src.origin, wave == 0 ? t0 : t1 - 1);
            if (lane == 0) seg01[wave] = s;
        }
        for (int i = tid; i < CS_TILE; i += CS_THREADS) mark[i] = 0;
        __syncthreads();
        const int32_t s0 = seg01[0], s1 = seg01[1];
        if (s1 - s0 > CS_GAP) {
            // Far more segments than entries, in one tile: each entry's by
            // binary search.
#pragma unroll
            for (int j = 0; j < CS_ITEMS; ++j) minor[j] = (uint32_t)s0;
            for (int32_t step = 1 << (31 - __builtin_clz((uint32_t)(s1 - s0))); step > 0; step >>= 1) {
#pragma unroll
                for (int j = 0; j < CS_ITEMS; ++j) {
                    const int64_t to = (int64_t)minor[j] + step;
                    if (to <= s1 && (int64_t)src.pos2[to] - src.origin <= t0 + min(base + 64 * j, last))
                        minor[j] = (uint32_t)to;
                }
            }
        } else {
            if (tid == 0) mark[0] = s0;
            for (int64_t s = (int64_t)s0 + 1 + tid; s <= s1; s += CS_THREADS) {
                const int64_t a = (int64_t)src.pos2[s] - src.origin, b = (int64_t)src.pos2[s + 1] - src.origin;
                if (b > a && a > t0 && a < t1) mark[a - t0] = (int32_t)s;
            }
            __syncthreads();
            int32_t m[CS_ITEMS];
#pragma unroll
            for (int j = 0; j < CS_ITEMS; ++j) {
                m[j] = mark[tid * CS_ITEMS + j];
                if (j) m[j] = max(m[j], m[j - 1]);
            }
            int32_t top = m[CS_ITEMS - 1];
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int32_t o = __shfl_up(top, d, 64);
                if (lane >= d) top = max(top, o);
            }
            if (lane == 63) wsum[wave] = top;
            int32_t before = __shfl_up(top, 1, 64);
            if (lane == 0) before = 0;
            __syncthreads();
            for (int w = 0; w < wave; ++w) before = max(before, wsum[w]);
#pragma unroll
            for (int j = 0; j < CS_ITEMS; ++j) mark[tid * CS_ITEMS + j] = max(m[j], before);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < CS_ITEMS; ++j) minor[j] = (uint32_t)mark[base + 64 * j];
            __syncthreads();
        }
    }
    // Ranks: in its wave, by the wave's own count of each digit so far.
    uint32_t *cnt2 = reinterpret_cast<uint32_t *>(lds);   // two digits a word
    uint16_t *cnt = reinterpret_cast<uint16_t *>(lds) + wave * nd;
    const int words = nd / 2;
    for (int i = tid; i < CS_WAVES * words; i += CS_THREADS) cnt2[i] = 0;
    int32_t place[CS_WPT][2];                             // of this thread's digits
#pragma unroll
    for (int q = 0; q < CS_WPT; ++q)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int d = 2 * (tid * CS_WPT + q) + e;
            place[q][e] = d < nd ? hist[(int64_t)d * ps.ntiles + tile] : 0;
        }
    __syncthreads();
    uint32_t at[CS_ITEMS];
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j) {
        const bool v = valid >> j & 1;
        const uint32_t d = key[j] >> ps.shift & (uint32_t)(nd - 1);
        const uint64_t all = __ballot(v);
        uint32_t lo = (uint32_t)all, hi = (uint32_t)(all >> 32);
        for (int b = 0; b < ps.bits; ++b) {
            const uint32_t on = (uint32_t)__builtin_amdgcn_sbfe((int)d, (uint32_t)b, 1u);   // 0 or all ones
            const uint64_t m = __ballot(on != 0);
            lo &= ~((uint32_t)m ^ on);
            hi &= ~((uint32_t)(m >> 32) ^ on);
        }
        if (v) {
            const uint32_t old = __hip_atomic_load(cnt + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            const uint32_t prior = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
            at[j] = old + prior;
            if (prior == 0)
                __hip_atomic_store(cnt + d, (uint16_t)(old + __builtin_popcount(lo) + __builtin_popcount(hi)),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // The tile's stretches, by each thread's digits.
    uint32_t c[CS_WAVES][CS_WPT], sum[CS_WPT];
    int32_t mine = 0;
#pragma unroll
    for (int q = 0; q < CS_WPT; ++q) {
        sum[q] = 0;
        if (tid * CS_WPT + q < words) {
#pragma unroll
            for (int w = 0; w < CS_WAVES; ++w) sum[q] += c[w][q] = cnt2[w * words + tid * CS_WPT + q];
        }
        mine += (int32_t)(sum[q] & 0xffff) + (int32_t)(sum[q] >> 16);
    }
    int32_t inc = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int32_t o = __shfl_up(inc, d, 64);
        if (lane >= d) inc += o;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int32_t first = inc - mine, total = 0;
#pragma unroll
    for (int w = 0; w < CS_WAVES; ++w) {
        const int32_t t = wsum[w];
        if (w < wave) first += t;
        total += t;
    }
#pragma unroll
    for (int q = 0; q < CS_WPT; ++q) {
        const int word = tid * CS_WPT + q;
        if (word >= words) break;
        const int32_t second = first + (int32_t)(sum[q] & 0xffff);
        uint32_t run = (uint32_t)first | (uint32_t)second << 16;
#pragma unroll
        for (int w = 0; w < CS_WAVES; ++w) {
            cnt2[w * words + word] = run;
            run += c[w][q];
        }
        delta[2 * word] = place[q][0] - first;
        delta[2 * word + 1] = place[q][1] - second;
        first = second + (int32_t)(sum[q] >> 16);
    }
    if (FIRST && tile == 0 && tid == 0) flags[CS_COUNT] = hist[(int64_t)nd * ps.ntiles];
    // (An index the compiler can't see through: loads moved up would spill.)
    uint32_t here = (uint32_t)base;
    asm volatile("" : "+v"(here));
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j) {
        const uint32_t i = min(here + 64 * j, (uint32_t)last) & (CS_TILE - 1);
        if (!FIRST) minor[j] = iminor[t0 + i];
        val[j] = value[i];
    }
    if (FROM == CS_SOURCE) {
        bool zero = false;
#pragma unroll
        for (int j = 0; j < CS_ITEMS; ++j) zero = zero || val[j] == T(0);
        if (zero) flags[CS_ZEROS] = 1;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j)
        if (valid >> j & 1) at[j] += cnt[key[j] >> ps.shift & (uint32_t)(nd - 1)];
    __syncthreads();
    // Out in digit order, one array after the other through the same LDS.
    uint32_t *box = reinterpret_cast<uint32_t *>(lds);
    T *vbox = reinterpret_cast<T *>(lds);
    uint32_t dst[CS_ITEMS];
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j)
        if (valid >> j & 1) box[at[j]] = key[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j) {
        const int i = tid + CS_THREADS * j;
        if (i >= total) continue;
        const uint32_t k = box[i];
        dst[j] = (uint32_t)(delta[k >> ps.shift & (uint32_t)(nd - 1)] + i);
        okey[dst[j]] = k + kadd;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j)
        if (valid >> j & 1) box[at[j]] = minor[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j)
        if (tid + CS_THREADS * j < total) ominor[dst[j]] = box[tid + CS_THREADS * j] + madd;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j)
        if (valid >> j & 1) vbox[at[j]] = val[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CS_ITEMS; ++j)
        if (tid + CS_THREADS * j < total) oval[dst[j]] = vbox[tid + CS_THREADS * j];
}

// Counts the sorted entries that repeat the coordinates before them, and
// (head given) marks the others.
__global__ __launch_bounds__(256) void sort_repeats_kernel(int64_t nmax, const uint32_t *__restrict__ key,
                                                           const uint32_t *__restrict__ minor,
                                                           int32_t *__restrict__ flags, int32_t *__restrict__ head)
{
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    const int64_t n = min(nmax, (int64_t)flags[CS_COUNT]);
    int repeats = 0;
    if (i + 4 <= n) {
        const uint4 k = *reinterpret_cast<const uint4 *>(key + i);
        uint4 m;                            // the caller's, of any alignment
        __builtin_memcpy(&m, minor + i, sizeof(m));
        const uint32_t kp = i > 0 ? key[i - 1] : ~k.x, mp = i > 0 ? minor[i - 1] : 0;
        const int r0 = kp == k.x && mp == m.x, r1 = k.x == k.y && m.x == m.y, r2 = k.y == k.z && m.y == m.z,
                  r3 = k.z == k.w && m.z == m.w;
        repeats = r0 + r1 + r2 + r3;
        if (head) *reinterpret_cast<int4 *>(head + i) = make_int4(1 - r0, 1 - r1, 1 - r2, 1 - r3);
    } else {
        for (int64_t t = i; t < n; ++t) {
            const int r = t > 0 && key[t] == key[t - 1] && minor[t] == minor[t - 1];
            repeats += r;
            if (head) head[t] = 1 - r;
        }
    }
    if (head) return;
    int sum = 0;                            // of the wave: each thread has 0 to 4
    for (int b = 0; b < 3; ++b) sum += __popcll(__ballot(repeats >> b & 1)) << b;
    if (sum > 0 && (threadIdx.x & 63) == 0) atomicAdd(&flags[CS_REPEATS], sum);
}

// The marked entries to their places (idx: the exclusive scan of the marks).
template <typename T>
__global__ __launch_bounds__(256) void sort_heads_kernel(int64_t n, const int32_t *__restrict__ head,
                                                         const int32_t *__restrict__ idx,
                                                         const uint32_t *__restrict__ key,
                                                         const uint32_t *__restrict__ minor,
                                                         const T *__restrict__ val, uint32_t *__restrict__ okey,
                                                         uint32_t *__restrict__ ominor, T *__restrict__ oval)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !head[i]) return;
    okey[idx[i]] = key[i];
    ominor[idx[i]] = minor[i];
    oval[idx[i]] = val[i];
}

// ptr[r] = origin + first i with key[i] >= r, r in [0, nmajor], of the first
// *count keys.
__global__ __launch_bounds__(256) void sort_ptr_kernel(const uint32_t *__restrict__ key,
                                                       const int32_t *__restrict__ count, int64_t nmajor,
                                                       int32_t origin, int32_t *__restrict__ ptr)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nmajor) return;
    int64_t lo = 0, hi = *count;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)key[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    ptr[r] = (int32_t)(lo + origin);
}

// ------------------------------------------------- CSR to BSR, small blocks
//
// A block-row's entries are one stretch of a CSR's, and where each row's
// columns increase its block columns are the union of a few sorted lists: no
// sort.  The general path sorts every entry by a 64-bit key and fetches its
// value by position.
//
// A wave takes a block-row.  bsr_heads_kernel finds each block's first stored
// entry (no nonzero before it in its row's part of the block, and none in the
// rows above, found by binary search), gathers their block columns in LDS,
// puts them in order by counting and leaves them at the block-row's place in
// heads.  bsr_blocks_kernel, after a scan of the counts, writes each entry to
// its block, found by binary search among them.  Explicit zeros are dropped:
// a block of nothing else is not stored.  Rows that do not increase, pointers
// that do not cover the entries, block-rows past BR_ENTRIES entries or
// BR_BLOCKS blocks go to the general path (a wave is too little for those).
//
// What bounds it: the searches and the serial loop of a wave in the first
// kernel, memory in the second (entries read, blocks written, twice where zeros
// fill them up).  Mesh of 59,200 nodes, 4 x 4 f64, 24M entries: 187 and 168 us, a
// whole conversion 419 (2,038 by the general path); 3 x 3 f32, 24,000 nodes: 132
// (762); 400k uniform rows of 8 to 8 x 8 blocks, mostly zeros: 623 (937).
// Past 2,048 entries a wave is the whole kernel's tail, and they are found before
// the others are read: 400k power-law rows of 16 into 4 x 4 blocks, which the
// general path takes, 1,263 us (1,195 there; 1,651 with 8,192 allowed).
constexpr int BR_WAVES = 4, BR_BLOCKS = 1024, BR_ENTRIES = 2048, BR_STAGE = 2048, BR_DIM = 8;

// The least i in [lo, hi) with a[i] >= x, hi if none.
__device__ __forceinline__ int br_lower(const int32_t *a, int lo, int hi, int x)
{
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// flags[0] = 1 where a block-row is too long or the pointers do not cover the
// entries: found before the others' entries are read.
__global__ __launch_bounds__(256) void bsr_long_kernel(jlust_sparse src, int64_t mb, int b1, int32_t *__restrict__ flags)
{
    const int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (R >= mb) return;
    const int64_t a = (int64_t)src.pos2[R * b1] - src.origin, b = (int64_t)src.pos2[(R + 1) * b1] - src.origin;
    if ((R == 0 && a != 0) || (R == mb - 1 && b != src.nnz) || b - a > BR_ENTRIES) flags[0] = 1;
}

// flags[0] = 1: not for this path.  full[R]: the block-row's entries fill its
// blocks.  count[mb] = 0.  stage: entries of a block-row that fit its LDS.
template <typename T, int B2>
__global__ __launch_bounds__(64 * BR_WAVES) void bsr_heads_kernel(jlust_sparse src, int64_t mb, int b1, int stage,
                                                                  int32_t *__restrict__ heads,
                                                                  int32_t *__restrict__ count,
                                                                  uint8_t *__restrict__ full,
                                                                  int32_t *__restrict__ flags)
{
    extern __shared__ int32_t br_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t R = (int64_t)blockIdx.x * BR_WAVES + wave;
    if (R >= mb) {
        if (R == mb && lane == 0) count[mb] = 0;
        return;
    }
    if (flags[0]) return;
    int32_t *h = br_lds + wave * (stage + BR_BLOCKS);
    uint32_t *staged = reinterpret_cast<uint32_t *>(h + BR_BLOCKS);
    const int32_t *ptr = src.pos2 + R * b1, *col = src.crd2;
    const T *val = static_cast<const T *>(src.val);
    const int32_t o = src.origin;
    const int32_t at = (int32_t)((int64_t)ptr[min(lane, b1)] - o), next = __shfl_down(at, 1, 64);
    const int32_t p0 = __builtin_amdgcn_readlane(at, 0), p1 = __builtin_amdgcn_readlane(at, b1);
    const bool off = at < 0 || at > src.nnz || (lane < b1 && next < at) || (lane == 0 && R == 0 && at != 0) ||
                     (lane == b1 && R == mb - 1 && at != src.nnz);
    if (__ballot(off) != 0 || p1 - p0 > BR_ENTRIES) {
        if (lane == 0) flags[0] = 1;
        return;
    }
    int nb = 0, nz = 0;
    bool bad = false;
    // entry(p): twice the column of entry p, plus one if it is a zero.
    auto find = [&](auto entry) {
        for (int q0 = p0; q0 < p1; q0 += 64) {
            const int p = q0 + lane;
            bool head = false;
            int bc = 0, r = 0, rs = p0;
            for (int i = 1; i < b1; ++i) {
                const int32_t s = __builtin_amdgcn_readlane(at, i);
                if (s <= p) {
                    r = i;
                    rs = s;
                }
            }
            if (p < p1) {
                const uint32_t e = entry(p), c = e >> 1;
                bad = bad || c >= (uint64_t)src.n || (p > rs && (entry(p - 1) >> 1) >= c);
                bc = (int)(c / B2);
                head = !(e & 1);
                nz += head;
                const uint32_t first = 2 * (uint32_t)(bc * B2), past = first + 2 * B2;
                // Nonzeros of the block before it: in its row, then in those above.
                for (int q = p - 1; head && q >= rs && q > p - B2; --q) {
                    const uint32_t f = entry(q);
                    if (f < first) break;
                    head = f & 1;
                }
                int s = p0;
                for (int i = 0; i < b1 - 1; ++i) {
                    const int end = __builtin_amdgcn_readlane(at, i + 1);
                    if (head && i < r) {
                        int lo = s, hi = end;
                        while (lo < hi) {
                            const int mid = (lo + hi) >> 1;
                            if (entry(mid) < first) lo = mid + 1;
                            else hi = mid;
                        }
                        for (; head && lo < end; ++lo) {
                            const uint32_t f = entry(lo);
                            if (f >= past) break;
                            head = f & 1;
                        }
                    }
                    s = end;
                }
            }
            const uint64_t m = __ballot(head);
            const int k =
                nb + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            if (head && k < BR_BLOCKS) h[k] = bc;
            nb += __popcll(m);
        }
    };
    auto load = [&](int p) {
        const int32_t c = col[p] - o;
        bad = bad || c < 0;                               // would look like another one once doubled
        return (uint32_t)c << 1 | (uint32_t)(val[p] == T(0));
    };
    if (p1 - p0 <= stage) {
        for (int q = p0 + lane; q < p1; q += 256) {
            uint32_t e[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) e[j] = load(min(q + 64 * j, p1 - 1));
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (q + 64 * j < p1) staged[q + 64 * j - p0] = e[j];
        }
        wave_sync();
        find([&](int p) { return staged[p - p0]; });
    } else {
        find(load);
    }
    if (__ballot(bad) != 0 || nb > BR_BLOCKS) {
        if (lane == 0) flags[0] = 1;
        return;
    }
    wave_sync();
    for (int i = lane; i < nb; i += 64) {
        const int x = h[i];
        int rank = 0;
#pragma unroll 4
        for (int j = 0; j < nb; ++j) rank += h[j] < x;
        heads[p0 + rank] = x;
    }
#pragma unroll
    for (int d = 32; d; d >>= 1) nz += __shfl_xor(nz, d, 64);
    if (lane == 0) {
        count[R] = nb;
        full[R] = nz == nb * b1 * B2;
    }
}

template <typename T, int B2>
__global__ __launch_bounds__(64 * BR_WAVES) void bsr_blocks_kernel(jlust_sparse src, int64_t mb, int b1, int row_major,
                                                                   const int32_t *__restrict__ heads,
                                                                   const uint8_t *__restrict__ full,
                                                                   const int32_t *__restrict__ browptr, int64_t nnzb,
                                                                   int32_t *__restrict__ bcol, T *__restrict__ out)
{
    __shared__ int32_t lds[BR_WAVES][BR_BLOCKS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t R = (int64_t)blockIdx.x * BR_WAVES + wave;
    if (R >= mb) return;
    int32_t *h = lds[wave];
    const int32_t o = src.origin;
    const int32_t *ptr = src.pos2 + R * b1, *col = src.crd2;
    const T *val = static_cast<const T *>(src.val);
    const int32_t at = ptr[min(lane, b1)] - o;
    const int32_t p0 = __builtin_amdgcn_readlane(at, 0), p1 = __builtin_amdgcn_readlane(at, b1);
    const int64_t base = (int64_t)browptr[R] - o, end = (int64_t)browptr[R + 1] - o;
    if (base < 0 || end > nnzb || end < base || end - base > min(p1 - p0, BR_BLOCKS)) return;
    const int nb = (int)(end - base), bb = b1 * B2;
    for (int i = lane; i < nb; i += 64) {
        const int x = heads[p0 + i];
        h[i] = x;
        bcol[base + i] = x + o;
    }
    T *blocks = out + base * bb;
    if (!full[R]) {
        for (int i = lane; i < nb * bb; i += 64) blocks[i] = T(0);
        __threadfence_block();                            // these stores, then the entries'
    }
    wave_sync();
    for (int q0 = p0; q0 < p1; q0 += 64) {
        const int p = q0 + lane;
        int r = 0;
        for (int i = 1; i < b1; ++i) r += __builtin_amdgcn_readlane(at, i) <= p;
        if (p >= p1) continue;
        const int c = col[p] - o, bc = c / B2, cc = c - bc * B2;
        const T v = val[p];
        if (v == T(0)) continue;
        const int k = br_lower(h, 0, nb, bc);
        if (k < nb) blocks[(int64_t)k * bb + (row_major ? r * B2 + cc : cc * b1 + r)] = v;
    }
}

// ----------------------------------------------------------------- host

int check_format(int fmt) { return fmt >= JLUST_FORMAT_CSR && fmt <= JLUST_FORMAT_BSR; }

bool src_ordered_identity(int fmt)
{
    return fmt == JLUST_FORMAT_CSR || fmt == JLUST_FORMAT_COO || fmt == JLUST_FORMAT_DCSR;
}
bool dst_identity(int fmt)
{
    return fmt == JLUST_FORMAT_CSR || fmt == JLUST_FORMAT_COO || fmt == JLUST_FORMAT_DCSR;
}

int check_sparse(const jlust_sparse *a, const char *what)
{
    if (!a) return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: null descriptor", what);
    if (!check_format(a->format))
        return fail(JLUST_STATUS_UNSUPPORTED_FORMAT, "%s: unknown format %d", what, a->format);
    if (int st = check_origin(a->origin)) return st;
    if (a->m < 0 || a->n < 0 || a->nnz < 0 || a->nouter < 0 || a->m > INT32_MAX ||
        a->n > INT32_MAX || a->nnz > INT32_MAX)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: extents outside the Int32 range", what);
    if (a->format == JLUST_FORMAT_BSR) {
        if (a->b1 <= 0 || a->b2 <= 0 || (int64_t)a->b1 * a->b2 > 65536 || a->m % a->b1 ||
            a->n % a->b2)
            return fail(JLUST_STATUS_INVALID_ARGUMENT, "%s: BSR block size %d x %d does not tile %lld x %lld",
                        what, a->b1, a->b2, (long long)a->m, (long long)a->n);
    }
    return JLUST_STATUS_SUCCESS;
}

KeyLayout layout_for(int fmt, int64_t m, int64_t n, int b1, int b2, int row_major)
{
    KeyLayout L;
    L.fmt = fmt;
    if (fmt == JLUST_FORMAT_CSC) {
        L.major_dim = n;
        L.minor_dim = m;
    } else if (fmt == JLUST_FORMAT_BSR) {
        L.b1 = b1;
        L.b2 = b2;
        L.row_major = row_major;
        L.major_dim = m / b1;
        L.minor_dim = n / b2;
        L.inner_bits = bits_for((int64_t)b1 * b2);
    } else {
        L.major_dim = m;
        L.minor_dim = n;
    }
    L.minor_bits = bits_for(L.minor_dim);
    L.total_bits = bits_for(L.major_dim) + L.minor_bits + L.inner_bits;
    return L;
}

int64_t segment_positions(const jlust_sparse *s)
{
    return s->format == JLUST_FORMAT_BSR ? s->nouter : s->nnz;
}

// The scans' and the sort's temporary storage over n items.
int scan_bytes(int64_t n, size_t *need)
{
    int32_t *v = nullptr;
    size_t a = 0, b = 0, c = 0;
    JLUST_HIP_TRY(rocprim::inclusive_scan(nullptr, a, v, v, (size_t)n, rocprim::maximum<int32_t>(), (hipStream_t)0));
    JLUST_HIP_TRY(rocprim::exclusive_scan(nullptr, b, v, v, 0, (size_t)n, rocprim::plus<int32_t>(), (hipStream_t)0));
    JLUST_HIP_TRY(rocprim::inclusive_scan(nullptr, c, v, v, (size_t)n, rocprim::plus<int32_t>(), (hipStream_t)0));
    *need = std::max(a, std::max(b, c));
    return JLUST_STATUS_SUCCESS;
}

int sort_bytes(int64_t n, int begin_bit, int end_bit, size_t *need)
{
    uint64_t *k = nullptr;
    int32_t *v = nullptr;
    JLUST_HIP_TRY(rocprim::radix_sort_pairs(nullptr, *need, k, k, v, v, (size_t)n, begin_bit, end_bit, (hipStream_t)0));
    return JLUST_STATUS_SUCCESS;
}

// Segment id per position for CSR/CSC/DCSR (per value) and BSR (per block);
// tmp: scan_bytes of the positions.
int segments(const jlust_sparse *s, int32_t *seg, int64_t &len, void *tmp, hipStream_t st)
{
    int64_t nseg = 0;
    len = s->nnz;
    switch (s->format) {
    case JLUST_FORMAT_CSR: nseg = s->m; break;
    case JLUST_FORMAT_CSC: nseg = s->n; break;
    case JLUST_FORMAT_DCSR: nseg = s->nouter; break;
    case JLUST_FORMAT_BSR:
        nseg = s->m / s->b1;
        len = s->nouter;
        break;
    default: return JLUST_STATUS_SUCCESS;
    }
    if (len == 0) return JLUST_STATUS_SUCCESS;
    JLUST_HIP_TRY(hipMemsetAsync(seg, 0, sizeof(int32_t) * (size_t)len, st));
    if (nseg > 0) {
        hipLaunchKernelGGL(seg_mark_kernel, dim3(cv_grid(nseg)), dim3(CV_BLOCK), 0, st, s->pos2, nseg,
                           s->origin, len, seg);
        if (int e = check_launch("seg_mark_kernel")) return e;
    }
    size_t need = 0;
    JLUST_HIP_TRY(rocprim::inclusive_scan(nullptr, need, seg, seg, (size_t)len,
                                          rocprim::maximum<int32_t>(), st));
    JLUST_HIP_TRY(rocprim::inclusive_scan(tmp, need, seg, seg, (size_t)len,
                                          rocprim::maximum<int32_t>(), st));
    return JLUST_STATUS_SUCCESS;
}

}  // namespace
}  // namespace jlust

using namespace jlust;

struct jlust_convert {
    KeyLayout L;
    int32_t dst_format = 0, origin = 0, value_type = 0;
    int64_t m = 0, n = 0;
    int64_t count = 0;          // entries after drop + dedup
    int64_t nruns = 0;          // DCSR rows / BSR blocks
    const void *src_val = nullptr;
    void *mem = nullptr;        // the analysis workspace if the handle owns it: keys, pos, head, run
                                // and spare point into it
    uint64_t *spare = nullptr;  // a buffer of as many words as there are stored values, free after analyse
    uint64_t *keys = nullptr;
    int32_t *pos = nullptr, *head = nullptr, *run = nullptr;   // pos null: the identity
};

namespace {

struct Workspace {
    void *p = nullptr;
    ~Workspace() { if (p) (void)hipFree(p); }
};

// The bits an entry's key is sorted by: [begin, end), empty where target and
// source share the identity ordering (convert.jl:331-349).  A source whose
// segments run in the order of the target's minor coordinate (CSR rows to a
// CSC target, CSC columns to a row-major one) holds equal majors in ascending
// minor order already, so the stable sort need only order the major bits.
bool sort_bits(const jlust_sparse *src, int dst_format, const KeyLayout &L, int *begin_bit, int *end_bit)
{
    if (dst_identity(dst_format) && src_ordered_identity(src->format)) return false;
    const bool major_only = (src->format == JLUST_FORMAT_CSR && dst_format == JLUST_FORMAT_CSC) ||
                            (src->format == JLUST_FORMAT_CSC && dst_identity(dst_format));
    *end_bit = L.total_bits > 0 ? L.total_bits : 1;
    *begin_bit = major_only && L.minor_bits + L.inner_bits < *end_bit ? L.minor_bits + L.inner_bits : 0;
    return true;
}

// The analysis workspace: keys x2, positions x2, flags and their scan per
// stored value, segments, two counters, and the library's temporary storage.
struct AnalyzeLayout {
    size_t tmp = 0, bytes = 0;
};

int analyze_layout(const jlust_sparse *src, int dst_format, const KeyLayout &L, AnalyzeLayout *out)
{
    const int64_t N = src->nnz;
    *out = AnalyzeLayout();
    if (N == 0) return JLUST_STATUS_SUCCESS;
    size_t scan = 0, sort = 0;
    if (int e = scan_bytes(std::max(N, segment_positions(src)), &scan)) return e;
    int begin_bit = 0, end_bit = 0;
    if (sort_bits(src, dst_format, L, &begin_bit, &end_bit))
        if (int e = sort_bytes(N, begin_bit, end_bit, &sort)) return e;
    out->tmp = (std::max(scan, sort) + 255) / 256 * 256;
    out->bytes = out->tmp + 8 * (size_t)N * 2 + 4 * (size_t)N * 4 + 4 * (size_t)segment_positions(src) + 256;
    return JLUST_STATUS_SUCCESS;
}

// ws: analyze_layout's bytes, the caller's (the handle keeps pointers into it).
template <typename T>
int analyze(const jlust_sparse *src, jlust_convert *h, void *ws, const AnalyzeLayout &al, hipStream_t st)
{
    const int64_t N = src->nnz;
    KeyLayout &L = h->L;
    if (N == 0) return JLUST_STATUS_SUCCESS;
    const size_t n = (size_t)N;
    char *b = (char *)ws;
    void *tmp = b;                    b += al.tmp;
    uint64_t *k0 = (uint64_t *)b;     b += 8 * n;
    uint64_t *k1 = (uint64_t *)b;     b += 8 * n;
    int32_t *p0 = (int32_t *)b;       b += 4 * n;
    int32_t *p1 = (int32_t *)b;       b += 4 * n;
    int32_t *flag = (int32_t *)b;     b += 4 * n;
    int32_t *idx = (int32_t *)b;      b += 4 * n;
    int32_t *bad = (int32_t *)b;      b += 64;   // bad[0]: a coordinate out of range; bad[1]: values dropped
    int32_t *seg = (int32_t *)b;
    JLUST_HIP_TRY(hipMemsetAsync(bad, 0, 2 * sizeof(int32_t), st));

    int64_t seglen = 0;
    if (int e = segments(src, seg, seglen, tmp, st)) return e;
    hipLaunchKernelGGL((decompose_kernel<T>), dim3(cv_grid(N)), dim3(CV_BLOCK), 0, st, *src, seg, L, k0,
                       flag, bad, bad + 1);
    if (int e = check_launch("decompose_kernel")) return e;

    // count of flagged items (exclusive scan + last flag), read back.
    auto count_flags = [&](int64_t len, int64_t *out) -> int {
        size_t need = 0;
        JLUST_HIP_TRY(rocprim::exclusive_scan(nullptr, need, flag, idx, 0, (size_t)len,
                                              rocprim::plus<int32_t>(), st));
        JLUST_HIP_TRY(rocprim::exclusive_scan(tmp, need, flag, idx, 0, (size_t)len,
                                              rocprim::plus<int32_t>(), st));
        int32_t last[2] = {0, 0};
        JLUST_HIP_TRY(hipMemcpyAsync(&last[0], idx + len - 1, 4, hipMemcpyDeviceToHost, st));
        JLUST_HIP_TRY(hipMemcpyAsync(&last[1], flag + len - 1, 4, hipMemcpyDeviceToHost, st));
        JLUST_HIP_TRY(hipStreamSynchronize(st));
        *out = (int64_t)last[0] + last[1];
        return JLUST_STATUS_SUCCESS;
    };

    // 1. drop explicit zeros (stable).  With none dropped the keys stay in
    // place and an entry's position is its index (pc null).
    int32_t flags_h[2] = {0, 0};
    JLUST_HIP_TRY(hipMemcpyAsync(flags_h, bad, sizeof(flags_h), hipMemcpyDeviceToHost, st));
    JLUST_HIP_TRY(hipStreamSynchronize(st));
    if (flags_h[0])
        return fail(JLUST_STATUS_INVALID_ARGUMENT,
                    "convert: a stored coordinate lies outside the %lld x %lld extents",
                    (long long)src->m, (long long)src->n);
    uint64_t *kc = k0;
    int32_t *pc = nullptr;
    int64_t K = N;
    if (flags_h[1] > 0) {
        if (int e = count_flags(N, &K)) return e;
        hipLaunchKernelGGL(compact_kernel, dim3(cv_grid(N)), dim3(CV_BLOCK), 0, st, N, flag, idx, k0,
                           (const int32_t *)nullptr, k1, p1);
        if (int e = check_launch("compact_kernel")) return e;
        kc = k1;
        pc = p1;
    }
    if (K == 0) return JLUST_STATUS_SUCCESS;

    // 2. sort by level coordinates.
    int begin_bit = 0, end_bit = 0;
    if (sort_bits(src, h->dst_format, L, &begin_bit, &end_bit)) {
        if (!pc) {                                  // the positions to carry: 0..K-1
            hipLaunchKernelGGL(iota_kernel, dim3(cv_grid(K)), dim3(CV_BLOCK), 0, st, K, p1);
            if (int e = check_launch("iota_kernel")) return e;
            pc = p1;
        }
        uint64_t *ko = kc == k0 ? k1 : k0;
        size_t need = 0;
        JLUST_HIP_TRY(rocprim::radix_sort_pairs(nullptr, need, kc, ko, pc, p0, (size_t)K, begin_bit, end_bit, st));
        Workspace more;                             // fewer entries than N may take another sort
        if (need > al.tmp) JLUST_HIP_TRY(hipMalloc(&more.p, need));
        JLUST_HIP_TRY(rocprim::radix_sort_pairs(more.p ? more.p : tmp, need, kc, ko, pc, p0, (size_t)K, begin_bit,
                                                end_bit, st));
        kc = ko;
        pc = p0;
    } else if (h->dst_format == JLUST_FORMAT_CSR) {
        // CSR's Dense row level needs non-decreasing rows; the reference
        // asserts it (convert.jl:254).  COO and DCSR targets keep any order.
        JLUST_HIP_TRY(hipMemsetAsync(bad, 0, sizeof(int32_t), st));
        hipLaunchKernelGGL(major_order_kernel, dim3(cv_grid(K)), dim3(CV_BLOCK), 0, st, K, kc, L, bad);
        if (int e = check_launch("major_order_kernel")) return e;
        int32_t badh = 0;
        JLUST_HIP_TRY(hipMemcpyAsync(&badh, bad, 4, hipMemcpyDeviceToHost, st));
        JLUST_HIP_TRY(hipStreamSynchronize(st));
        if (badh)
            return fail(JLUST_STATUS_NONCANONICAL_STORAGE,
                        "convert: the source's rows are not in non-decreasing order");
    }

    // 3. merge adjacent equal coordinates on unique levels (keep the first);
    // nothing to do when no key repeats.
    int64_t C = K;
    if (h->dst_format != JLUST_FORMAT_COO) {
        JLUST_HIP_TRY(hipMemsetAsync(bad + 1, 0, sizeof(int32_t), st));
        hipLaunchKernelGGL(head_kernel, dim3(cv_grid(K)), dim3(CV_BLOCK), 0, st, K, kc, L, 0, flag, bad + 1);
        if (int e = check_launch("head_kernel")) return e;
        int32_t repeats = 0;
        JLUST_HIP_TRY(hipMemcpyAsync(&repeats, bad + 1, sizeof(int32_t), hipMemcpyDeviceToHost, st));
        JLUST_HIP_TRY(hipStreamSynchronize(st));
        if (repeats > 0) {
            if (int e = count_flags(K, &C)) return e;
            uint64_t *ko = kc == k1 ? k0 : k1;
            int32_t *po = pc == p1 ? p0 : p1;       // pc null: positions are indices
            hipLaunchKernelGGL(compact_kernel, dim3(cv_grid(K)), dim3(CV_BLOCK), 0, st, K, flag, idx, kc, pc,
                               ko, po);
            if (int e = check_launch("compact_kernel")) return e;
            kc = ko;
            pc = po;
        }
    }

    // 4. the handle keeps the workspace: keys, positions, and (DCSR rows /
    // BSR blocks) run heads and ids in the flag and index arrays, free now.
    const size_t c = (size_t)C;
    h->keys = kc;
    h->spare = kc == k0 ? k1 : k0;
    h->pos = pc;
    h->head = flag;
    h->run = idx;
    h->count = C;
    if (h->dst_format == JLUST_FORMAT_DCSR || h->dst_format == JLUST_FORMAT_BSR) {
        KeyLayout Lr = L;
        if (h->dst_format == JLUST_FORMAT_DCSR) {   // runs of equal row: compare majors only
            Lr.inner_bits = L.minor_bits + L.inner_bits;
            Lr.minor_bits = 0;
        }
        hipLaunchKernelGGL(head_kernel, dim3(cv_grid(C)), dim3(CV_BLOCK), 0, st, C, h->keys, Lr, 1,
                           h->head, nullptr);
        if (int e = check_launch("head_kernel")) return e;
        size_t need = 0;
        JLUST_HIP_TRY(rocprim::inclusive_scan(nullptr, need, h->head, h->run, c, rocprim::plus<int32_t>(), st));
        JLUST_HIP_TRY(rocprim::inclusive_scan(tmp, need, h->head, h->run, c, rocprim::plus<int32_t>(), st));
        int32_t nr = 0;
        JLUST_HIP_TRY(hipMemcpyAsync(&nr, h->run + C - 1, 4, hipMemcpyDeviceToHost, st));
        JLUST_HIP_TRY(hipStreamSynchronize(st));
        h->nruns = nr;
        // run ids 0-based
        hipLaunchKernelGGL(shift_kernel, dim3(cv_grid(C)), dim3(CV_BLOCK), 0, st, C, h->run, h->run, -1);
        if (int e = check_launch("shift_kernel")) return e;
    }
    JLUST_HIP_TRY(hipStreamSynchronize(st));
    return JLUST_STATUS_SUCCESS;
}

// The passes and the workspace of a direct conversion; passes == 0: not one.
struct DirectLayout {
    int64_t nseg = 0, major_dim = 0, ntiles = 0;
    int passes = 0, bits = 0;
    size_t tmp = 0, hist = 0, bytes = 0;
};

int direct_layout(const jlust_sparse *src, int dst_format, size_t vsize, DirectLayout *out)
{
    *out = DirectLayout();
    const bool csr = src->format == JLUST_FORMAT_CSR;
    if (!(csr && dst_format == JLUST_FORMAT_CSC) &&
        !(src->format == JLUST_FORMAT_CSC && (dst_format == JLUST_FORMAT_CSR || dst_format == JLUST_FORMAT_COO)))
        return JLUST_STATUS_SUCCESS;
    out->nseg = csr ? src->m : src->n;
    out->major_dim = csr ? src->n : src->m;
    // The tiles look at every segment: where almost all are empty the general
    // path's scan over the entries is the better one.
    if (src->nnz == 0 || out->major_dim == 0 || out->nseg == 0 || out->nseg > 16 * src->nnz)
        return JLUST_STATUS_SUCCESS;
    const int bits = std::max(1, bits_for(out->major_dim));
    out->passes = (bits + CS_BITS - 1) / CS_BITS;
    out->bits = (bits + out->passes - 1) / out->passes;
    out->ntiles = (src->nnz + CS_TILE - 1) / CS_TILE;
    out->hist = ((size_t)1 << out->bits) * (size_t)out->ntiles + 1;
    int32_t *v = nullptr;
    size_t a = 0, b = 0;
    JLUST_HIP_TRY(rocprim::exclusive_scan(nullptr, a, v, v, 0, out->hist, rocprim::plus<int32_t>(), (hipStream_t)0));
    JLUST_HIP_TRY(rocprim::exclusive_scan(nullptr, b, v, v, 0, (size_t)src->nnz, rocprim::plus<int32_t>(),
                                          (hipStream_t)0));
    out->tmp = std::max(a, b);
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    const size_t n = (size_t)src->nnz, entry = up(vsize * n) + 2 * up(4 * n);
    // flags, counts, scan; the entries after the first pass; marks and their
    // scan, or the entries after the second of three; the target's majors.
    out->bytes = 256 + up(4 * out->hist) + up(out->tmp) + entry + (out->passes > 2 ? entry : 2 * up(4 * n)) + up(4 * n);
    return JLUST_STATUS_SUCCESS;
}

template <typename T>
int direct_run(const jlust_sparse *src, const jlust_sparse *dst, const DirectLayout &dl, void *ws, int64_t *count,
               hipStream_t st)
{
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    const int64_t N = src->nnz;
    const size_t n = (size_t)N;
    char *b = (char *)ws;
    auto take = [&](size_t bytes) { char *p = b; b += up(bytes); return p; };
    struct Entries { uint32_t *key, *minor; T *val; };
    auto entries = [&] { Entries e; e.val = (T *)take(sizeof(T) * n); e.key = (uint32_t *)take(4 * n);
                         e.minor = (uint32_t *)take(4 * n); return e; };
    int32_t *flags = (int32_t *)take(256);
    int32_t *hist = (int32_t *)take(4 * dl.hist);
    void *tmp = take(dl.tmp);
    const Entries e1 = entries();
    char *after = b;
    Entries e2 = {nullptr, nullptr, nullptr};
    int32_t *head = nullptr, *idx = nullptr;
    if (dl.passes > 2) e2 = entries();
    else b += 2 * up(4 * n);
    head = (int32_t *)after;
    idx = (int32_t *)(after + up(4 * n));
    uint32_t *major = (uint32_t *)take(4 * n);
    const bool coo = dst->format == JLUST_FORMAT_COO;
    const uint32_t o = (uint32_t)dst->origin;
    const Entries out = {coo ? (uint32_t *)dst->crd1 : major, (uint32_t *)dst->crd2, (T *)dst->val};
    const dim3 grid((unsigned)((dl.ntiles + 7) / 8 * 8)), block(CS_THREADS);
    // Zeros are to be dropped, and there are none as a rule: the first count
    // reads the coordinates alone, and where a pass meets a zero all is done
    // again without them.
    auto passes = [&](bool nonzeros) -> int {
        JLUST_HIP_TRY(hipMemsetAsync(flags, 0, 16 * sizeof(int32_t), st));
        Entries in = {nullptr, nullptr, nullptr};
        for (int p = 0; p < dl.passes; ++p) {
            const SortPass ps = {p * dl.bits, dl.bits, dl.ntiles};
            const bool last = p == dl.passes - 1;
            const Entries to = last ? out : p % 2 ? e2 : e1;
#define JLUST_COUNT(FROM)                                                                                         \
            hipLaunchKernelGGL((sort_count_kernel<T, FROM>), grid, dim3(CC_THREADS), 0, st, *src, dl.nseg, dl.major_dim, \
                               in.key, ps, hist, flags)
#define JLUST_MOVE(FROM)                                                                                          \
            hipLaunchKernelGGL((sort_move_kernel<T, FROM>), grid, block, 0, st, *src, dl.nseg, dl.major_dim, in.key,  \
                               in.minor, in.val, ps, hist, flags, to.key, to.minor, to.val, kadd, madd)
            if (p > 0) JLUST_COUNT(CS_ENTRIES);
            else if (nonzeros) JLUST_COUNT(CS_NONZEROS);
            else JLUST_COUNT(CS_SOURCE);
            if (int e = check_launch("sort_count_kernel")) return e;
            size_t need = dl.tmp;
            JLUST_HIP_TRY(rocprim::exclusive_scan(tmp, need, hist, hist, 0, dl.hist, rocprim::plus<int32_t>(), st));
            const uint32_t kadd = last && coo ? o : 0, madd = last ? o : 0;
            if (p > 0) JLUST_MOVE(CS_ENTRIES);
            else if (nonzeros) JLUST_MOVE(CS_NONZEROS);
            else JLUST_MOVE(CS_SOURCE);
#undef JLUST_COUNT
#undef JLUST_MOVE
            if (int e = check_launch("sort_move_kernel")) return e;
            in = to;
        }
        return JLUST_STATUS_SUCCESS;
    };
    auto pointers = [&]() -> int {
        hipLaunchKernelGGL(sort_ptr_kernel, dim3(cv_grid(dl.major_dim + 1)), dim3(256), 0, st, major, flags + CS_COUNT,
                           dl.major_dim, dst->origin, dst->pos2);
        return check_launch("sort_ptr_kernel");
    };
    int32_t got[5] = {0, 0, 0, 0, 0};
    for (int nonzeros = 0; nonzeros < 2; ++nonzeros) {
        if (int e = passes(nonzeros != 0)) return e;
        if (!coo) {
            hipLaunchKernelGGL(sort_repeats_kernel, dim3(cv_grid((N + 3) / 4)), dim3(256), 0, st, N, major,
                               (uint32_t *)dst->crd2, flags, (int32_t *)nullptr);
            if (int e = check_launch("sort_repeats_kernel")) return e;
            if (int e = pointers()) return e;
        }
        JLUST_HIP_TRY(hipMemcpyAsync(got, flags, sizeof(got), hipMemcpyDeviceToHost, st));
        JLUST_HIP_TRY(hipStreamSynchronize(st));
        if (got[CS_POINTERS]) return JLUST_STATUS_SUCCESS;      // *count stays -1
        if (got[CS_BAD])
            return fail(JLUST_STATUS_INVALID_ARGUMENT,
                        "convert: a stored coordinate lies outside the %lld x %lld extents", (long long)src->m,
                        (long long)src->n);
        if (!got[CS_ZEROS]) break;
    }
    int64_t C = got[CS_COUNT];
    if (coo && dst->pos1) {
        hipLaunchKernelGGL(pair_kernel, dim3(1), dim3(64), 0, st, dst->pos1, dst->origin, (int32_t)(C + dst->origin));
        if (int e = check_launch("pair_kernel")) return e;
    }
    if (got[CS_REPEATS] > 0) {                              // unique levels keep the first of equal coordinates
        hipLaunchKernelGGL(sort_repeats_kernel, dim3(cv_grid((C + 3) / 4)), dim3(256), 0, st, C, major,
                           (uint32_t *)dst->crd2, flags, head);
        if (int e = check_launch("sort_repeats_kernel")) return e;
        size_t need = dl.tmp;
        JLUST_HIP_TRY(rocprim::exclusive_scan(tmp, need, head, idx, 0, (size_t)C, rocprim::plus<int32_t>(), st));
        hipLaunchKernelGGL(sort_heads_kernel<T>, dim3(cv_grid(C)), dim3(256), 0, st, C, head, idx, major,
                           (uint32_t *)dst->crd2, (T *)dst->val, e1.key, e1.minor, e1.val);
        if (int e = check_launch("sort_heads_kernel")) return e;
        C -= got[CS_REPEATS];
        got[CS_COUNT] = (int32_t)C;
        JLUST_HIP_TRY(hipMemcpyAsync(major, e1.key, 4 * (size_t)C, hipMemcpyDeviceToDevice, st));
        JLUST_HIP_TRY(hipMemcpyAsync(dst->crd2, e1.minor, 4 * (size_t)C, hipMemcpyDeviceToDevice, st));
        JLUST_HIP_TRY(hipMemcpyAsync(dst->val, e1.val, sizeof(T) * (size_t)C, hipMemcpyDeviceToDevice, st));
        JLUST_HIP_TRY(hipMemcpyAsync(flags + CS_COUNT, &got[CS_COUNT], 4, hipMemcpyHostToDevice, st));
        if (int e = pointers()) return e;
        JLUST_HIP_TRY(hipStreamSynchronize(st));            // `got` is read until here
    }
    *count = C;
    return JLUST_STATUS_SUCCESS;
}

// CSR to BSR by block-rows: the workspace (bytes == 0: not a conversion of
// this kind).
struct BlocksLayout {
    int64_t mb = 0;
    size_t tmp = 0, bytes = 0;
};

int blocks_layout(const jlust_sparse *src, int b1, int b2, BlocksLayout *out)
{
    *out = BlocksLayout();
    if (src->format != JLUST_FORMAT_CSR || b1 > BR_DIM || b2 > BR_DIM || src->nnz == 0 || src->m == 0)
        return JLUST_STATUS_SUCCESS;
    out->mb = src->m / b1;
    // A wave to a block-row: where almost all are empty the general path's
    // passes over the entries are the better ones.
    if (out->mb > 16 * src->nnz) return JLUST_STATUS_SUCCESS;
    int32_t *v = nullptr;
    JLUST_HIP_TRY(rocprim::exclusive_scan(nullptr, out->tmp, v, v, 0, (size_t)out->mb + 1, rocprim::plus<int32_t>(),
                                          (hipStream_t)0));
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    // flags, heads, counts, full, the scan's
    out->bytes = 256 + up(4 * (size_t)src->nnz) + up(4 * ((size_t)out->mb + 1)) + up((size_t)out->mb) + up(out->tmp);
    return JLUST_STATUS_SUCCESS;
}

struct BlocksWs {
    int32_t *flags, *heads, *count;
    uint8_t *full;
    void *tmp;
};

BlocksWs blocks_ws(const jlust_sparse *src, const BlocksLayout &bl, void *ws)
{
    char *b = (char *)ws;
    auto take = [&](size_t bytes) { char *p = b; b += (bytes + 255) / 256 * 256; return p; };
    BlocksWs w;
    w.flags = (int32_t *)take(256);
    w.heads = (int32_t *)take(4 * (size_t)src->nnz);
    w.count = (int32_t *)take(4 * ((size_t)bl.mb + 1));
    w.full = (uint8_t *)take((size_t)bl.mb);
    w.tmp = take(bl.tmp);
    return w;
}

#define JLUST_BY_B2(b2, CALL)                                              \
    switch (b2) {                                                          \
    case 1: CALL(1); break;                                                \
    case 2: CALL(2); break;                                                \
    case 3: CALL(3); break;                                                \
    case 4: CALL(4); break;                                                \
    case 5: CALL(5); break;                                                \
    case 6: CALL(6); break;                                                \
    case 7: CALL(7); break;                                                \
    default: CALL(8);                                                      \
    }

template <typename T>
int blocks_count(const jlust_sparse *src, int b1, int b2, const BlocksLayout &bl, const BlocksWs &w, int32_t *browptr,
                 int64_t *nnzb, hipStream_t st)
{
    JLUST_HIP_TRY(hipMemsetAsync(w.flags, 0, 256, st));
    const dim3 grid((unsigned)(bl.mb / BR_WAVES + 1)), block(64 * BR_WAVES);
    hipLaunchKernelGGL(bsr_long_kernel, dim3(cv_grid(bl.mb)), dim3(256), 0, st, *src, bl.mb, b1, w.flags);
    if (int e = check_launch("bsr_long_kernel")) return e;
    // LDS for block-rows of up to twice the mean, in steps of 64 entries: the
    // searches read it instead of L1 (4 x 4 f64 mesh, 24M entries: 311 -> 187
    // us); the others search in memory.
    const int64_t mean = src->nnz / bl.mb + 1;
    const int stage = (int)std::min((2 * mean + 63) / 64 * 64, (int64_t)BR_STAGE);
    const size_t lds = 4 * BR_WAVES * (size_t)(stage + BR_BLOCKS);
#define JLUST_HEADS(B2)                                                                                           \
    hipLaunchKernelGGL((bsr_heads_kernel<T, B2>), grid, block, lds, st, *src, bl.mb, b1, stage, w.heads, w.count, \
                       w.full, w.flags)
    JLUST_BY_B2(b2, JLUST_HEADS)
#undef JLUST_HEADS
    if (int e = check_launch("bsr_heads_kernel")) return e;
    int32_t bad = 0, total = 0;
    JLUST_HIP_TRY(hipMemcpyAsync(&bad, w.flags, 4, hipMemcpyDeviceToHost, st));
    size_t need = bl.tmp;
    JLUST_HIP_TRY(rocprim::exclusive_scan(w.tmp, need, w.count, browptr, src->origin, (size_t)bl.mb + 1,
                                          rocprim::plus<int32_t>(), st));
    JLUST_HIP_TRY(hipMemcpyAsync(&total, browptr + bl.mb, 4, hipMemcpyDeviceToHost, st));
    JLUST_HIP_TRY(hipStreamSynchronize(st));
    if (!bad) *nnzb = (int64_t)total - src->origin;
    return JLUST_STATUS_SUCCESS;
}

template <typename T>
int blocks_fill(const jlust_sparse *src, const jlust_sparse *dst, const BlocksLayout &bl, const BlocksWs &w,
                hipStream_t st)
{
    const dim3 grid((unsigned)((bl.mb + BR_WAVES - 1) / BR_WAVES)), block(64 * BR_WAVES);
#define JLUST_BLOCKS(B2)                                                                                      \
    hipLaunchKernelGGL((bsr_blocks_kernel<T, B2>), grid, block, 0, st, *src, bl.mb, dst->b1,                  \
                       dst->row_major_blocks != 0, w.heads, w.full, dst->pos2, dst->nouter, dst->crd2, (T *)dst->val)
    JLUST_BY_B2(dst->b2, JLUST_BLOCKS)
#undef JLUST_BLOCKS
    return check_launch("bsr_blocks_kernel");
}

template <typename T>
int fill(const jlust_convert *h, const jlust_sparse *d, hipStream_t st)
{
    const KeyLayout &L = h->L;
    const int64_t C = h->count;
    const int32_t o = h->origin;
    const T *sval = (const T *)h->src_val;
    switch (h->dst_format) {
    case JLUST_FORMAT_CSR:
    case JLUST_FORMAT_CSC:
        hipLaunchKernelGGL(lower_bound_ptr_kernel, dim3(cv_grid(L.major_dim + 1)), dim3(CV_BLOCK), 0, st, C,
                           h->keys, (const int32_t *)nullptr, L, L.major_dim, o, d->pos2);
        if (int e = check_launch("lower_bound_ptr_kernel")) return e;
        if (C > 0) {
            hipLaunchKernelGGL((fill_entries_kernel<T>), dim3(cv_grid(C)), dim3(CV_BLOCK), 0, st, C, h->keys,
                               h->pos, L, o, sval, (int32_t *)nullptr, d->crd2, (T *)d->val);
            if (int e = check_launch("fill_entries_kernel")) return e;
        }
        break;
    case JLUST_FORMAT_COO:
        if (d->pos1) {
            hipLaunchKernelGGL(pair_kernel, dim3(1), dim3(64), 0, st, d->pos1, o, (int32_t)(C + o));
            if (int e = check_launch("pair_kernel")) return e;
        }
        if (C > 0) {
            hipLaunchKernelGGL((fill_entries_kernel<T>), dim3(cv_grid(C)), dim3(CV_BLOCK), 0, st, C, h->keys,
                               h->pos, L, o, sval, d->crd1, d->crd2, (T *)d->val);
            if (int e = check_launch("fill_entries_kernel")) return e;
        }
        break;
    case JLUST_FORMAT_DCSR:
        hipLaunchKernelGGL(fill_runs_kernel, dim3(cv_grid(C > 0 ? C : 1)), dim3(CV_BLOCK), 0, st, C, h->keys,
                           h->head, h->run, L, o, h->nruns, d->crd1, d->pos2, d->pos1);
        if (int e = check_launch("fill_runs_kernel")) return e;
        if (C > 0) {
            hipLaunchKernelGGL((fill_entries_kernel<T>), dim3(cv_grid(C)), dim3(CV_BLOCK), 0, st, C, h->keys,
                               h->pos, L, o, sval, (int32_t *)nullptr, d->crd2, (T *)d->val);
            if (int e = check_launch("fill_entries_kernel")) return e;
        }
        break;
    default: {                                       // BSR
        const int64_t nb = h->nruns;
        const int64_t nv = nb * L.b1 * L.b2;
        int32_t *brow = nullptr;
        if (nb > 0) {
            brow = (int32_t *)h->spare;              // nb blocks, of one stored value or more each
            hipLaunchKernelGGL((zero_kernel<T>), dim3(cv_grid(nv)), dim3(CV_BLOCK), 0, st, nv, (T *)d->val);
            if (int e = check_launch("zero_kernel")) return e;
            hipLaunchKernelGGL((fill_bsr_kernel<T>), dim3(cv_grid(C)), dim3(CV_BLOCK), 0, st, C, h->keys, h->pos,
                               h->head, h->run, L, o, sval, d->crd2, brow, (T *)d->val);
            if (int e = check_launch("fill_bsr_kernel")) return e;
        }
        hipLaunchKernelGGL(lower_bound_ptr_kernel, dim3(cv_grid(L.major_dim + 1)), dim3(CV_BLOCK), 0, st, nb,
                           (const uint64_t *)nullptr, brow, L, L.major_dim, o, d->pos2);
        if (int e = check_launch("lower_bound_ptr_kernel")) return e;
    }
    }
    return JLUST_STATUS_SUCCESS;
}

int dst_check(const jlust_convert *h, const jlust_sparse *d)
{
    if (!d) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_fill: null descriptor");
    const KeyLayout &L = h->L;
    if (d->format != h->dst_format || d->origin != h->origin || d->m != h->m || d->n != h->n)
        return fail(JLUST_STATUS_INVALID_ARGUMENT,
                    "convert_fill: descriptor does not match the analysed conversion");
    if (h->dst_format == JLUST_FORMAT_BSR &&
        (d->b1 != L.b1 || d->b2 != L.b2 || (d->row_major_blocks != 0) != (L.row_major != 0)))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_fill: BSR block layout differs from analyse");
    const int64_t want = h->dst_format == JLUST_FORMAT_BSR ? h->nruns * L.b1 * L.b2 : h->count;
    if (d->nnz != want)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_fill: nnz %lld, analyse reported %lld",
                    (long long)d->nnz, (long long)want);
    bool bad = bad_ptr(d->val, want);
    switch (h->dst_format) {
    case JLUST_FORMAT_CSR:
    case JLUST_FORMAT_CSC: bad = bad || !d->pos2 || bad_ptr(d->crd2, want); break;
    case JLUST_FORMAT_COO: bad = bad || bad_ptr(d->crd1, want) || bad_ptr(d->crd2, want); break;
    case JLUST_FORMAT_DCSR: bad = bad || !d->pos2 || bad_ptr(d->crd1, h->nruns) || bad_ptr(d->crd2, want); break;
    default: bad = bad || !d->pos2 || bad_ptr(d->crd2, h->nruns);
    }
    if (bad) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_fill: null device pointer");
    return JLUST_STATUS_SUCCESS;
}

bool src_ptrs_ok(const jlust_sparse *s)
{
    const int64_t nz = s->nnz;
    switch (s->format) {
    case JLUST_FORMAT_CSR: return (s->m == 0 || s->pos2) && !bad_ptr(s->crd2, nz) && !bad_ptr(s->val, nz);
    case JLUST_FORMAT_CSC: return (s->n == 0 || s->pos2) && !bad_ptr(s->crd2, nz) && !bad_ptr(s->val, nz);
    case JLUST_FORMAT_COO: return !bad_ptr(s->crd1, nz) && !bad_ptr(s->crd2, nz) && !bad_ptr(s->val, nz);
    case JLUST_FORMAT_DCSR:
        return (s->nouter == 0 || (s->pos2 && s->crd1)) && !bad_ptr(s->crd2, nz) && !bad_ptr(s->val, nz);
    default:
        return (s->m == 0 || s->pos2) && !bad_ptr(s->crd2, s->nouter) && !bad_ptr(s->val, nz) &&
               s->nnz == s->nouter * s->b1 * s->b2;
    }
}

}  // namespace

namespace {

// The checks and the key layout of an analysis.
int analyze_args(const jlust_sparse *src, int32_t dst_format, int32_t dst_b1, int32_t dst_b2,
                 int32_t dst_row_major_blocks, int value_type, KeyLayout *L)
{
    if (int st = check_sparse(src, "convert_analyze")) return st;
    if (!check_format(dst_format))
        return fail(JLUST_STATUS_UNSUPPORTED_FORMAT, "convert_analyze: unknown target format %d", dst_format);
    if (value_type != 0 && value_type != 1)
        return fail(JLUST_STATUS_UNSUPPORTED_VALUE_TYPE, "convert_analyze: value_type %d", value_type);
    if (!src_ptrs_ok(src)) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_analyze: null or inconsistent source buffers");
    if (dst_format == JLUST_FORMAT_BSR &&
        (dst_b1 <= 0 || dst_b2 <= 0 || (int64_t)dst_b1 * dst_b2 > 65536 || src->m % dst_b1 || src->n % dst_b2))
        return fail(JLUST_STATUS_INVALID_ARGUMENT,
                    "convert_analyze: BSR block size %d x %d does not tile %lld x %lld", dst_b1, dst_b2,
                    (long long)src->m, (long long)src->n);
    *L = layout_for(dst_format, src->m, src->n, dst_b1, dst_b2, dst_row_major_blocks);
    if (L->total_bits > 64)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_analyze: coordinates need more than 64 key bits");
    return JLUST_STATUS_SUCCESS;
}

// ws null: the handle allocates its workspace and frees it when destroyed.
int convert_analyze(const jlust_sparse *src, int32_t dst_format, int32_t dst_b1, int32_t dst_b2,
                    int32_t dst_row_major_blocks, int value_type, void *ws, size_t ws_bytes, hipStream_t stream,
                    jlust_convert_t *out, int64_t *dst_nnz, int64_t *dst_nouter)
{
    clear_error();
    if (!out || !dst_nnz || !dst_nouter)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_analyze: null output pointer");
    *out = nullptr;
    KeyLayout L;
    if (int st = analyze_args(src, dst_format, dst_b1, dst_b2, dst_row_major_blocks, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    AnalyzeLayout al;
    if (int st = analyze_layout(src, dst_format, L, &al)) return st;
    if (ws && ws_bytes < al.bytes)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_analyze: workspace of %zu bytes, %zu needed", ws_bytes,
                    al.bytes);
    auto *h = new jlust_convert();
    h->dst_format = dst_format;
    h->origin = src->origin;
    h->value_type = value_type;
    h->m = src->m;
    h->n = src->n;
    h->src_val = src->val;
    h->L = L;
    int st = JLUST_STATUS_SUCCESS;
    if (!ws && al.bytes) {
        const hipError_t e = hipMalloc(&h->mem, al.bytes);
        if (e != hipSuccess) st = hip_fail(e, "hipMalloc(convert workspace)");
        ws = h->mem;
    }
    if (!st)
        st = value_type == 0 ? analyze<double>(src, h, ws, al, stream) : analyze<float>(src, h, ws, al, stream);
    if (st) {
        if (h->mem) (void)hipFree(h->mem);
        delete h;
        return st;
    }
    *dst_nnz = dst_format == JLUST_FORMAT_BSR ? h->nruns * dst_b1 * dst_b2 : h->count;
    *dst_nouter = (dst_format == JLUST_FORMAT_DCSR || dst_format == JLUST_FORMAT_BSR) ? h->nruns : 0;
    *out = h;
    return JLUST_STATUS_SUCCESS;
}

}  // namespace

extern "C" int jlust_hip_convert_analyze(const jlust_sparse *src, int32_t dst_format, int32_t dst_b1,
                                         int32_t dst_b2, int32_t dst_row_major_blocks, int value_type,
                                         jlust_stream_t stream, jlust_convert_t *out, int64_t *dst_nnz,
                                         int64_t *dst_nouter)
{
    return convert_analyze(src, dst_format, dst_b1, dst_b2, dst_row_major_blocks, value_type, nullptr, 0,
                           (hipStream_t)stream, out, dst_nnz, dst_nouter);
}

extern "C" int jlust_hip_convert_workspace(const jlust_sparse *src, int32_t dst_format, int32_t dst_b1,
                                           int32_t dst_b2, int32_t dst_row_major_blocks, int value_type,
                                           int64_t *bytes)
{
    clear_error();
    if (!bytes) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_workspace: null output pointer");
    KeyLayout L;
    if (int st = analyze_args(src, dst_format, dst_b1, dst_b2, dst_row_major_blocks, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    AnalyzeLayout al;
    if (int st = analyze_layout(src, dst_format, L, &al)) return st;
    *bytes = (int64_t)al.bytes;
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_convert_analyze_ws(const jlust_sparse *src, int32_t dst_format, int32_t dst_b1,
                                            int32_t dst_b2, int32_t dst_row_major_blocks, int value_type,
                                            void *ws, int64_t ws_bytes, jlust_stream_t stream,
                                            jlust_convert_t *out, int64_t *dst_nnz, int64_t *dst_nouter)
{
    if (ws_bytes < 0 || (ws_bytes > 0 && !ws) || (uintptr_t)ws % 256)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_analyze: workspace null or not 256-byte aligned");
    return convert_analyze(src, dst_format, dst_b1, dst_b2, dst_row_major_blocks, value_type, ws, (size_t)ws_bytes,
                           (hipStream_t)stream, out, dst_nnz, dst_nouter);
}

extern "C" int jlust_hip_convert_direct_workspace(const jlust_sparse *src, int32_t dst_format, int value_type,
                                                  int64_t *bytes)
{
    clear_error();
    if (!bytes) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_direct: null output pointer");
    KeyLayout L;
    *bytes = 0;
    if (dst_format == JLUST_FORMAT_BSR) return JLUST_STATUS_SUCCESS;
    if (int st = analyze_args(src, dst_format, 1, 1, 1, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    DirectLayout dl;
    if (int st = direct_layout(src, dst_format, value_type == 0 ? 8 : 4, &dl)) return st;
    *bytes = (int64_t)dl.bytes;
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_convert_direct(const jlust_sparse *src, const jlust_sparse *dst, int value_type, void *ws,
                                        int64_t ws_bytes, jlust_stream_t stream, int64_t *count)
{
    clear_error();
    if (!count || !dst) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_direct: null argument");
    *count = -1;
    KeyLayout L;
    if (dst->format == JLUST_FORMAT_BSR) return JLUST_STATUS_SUCCESS;
    if (int st = analyze_args(src, dst->format, 1, 1, 1, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    DirectLayout dl;
    if (int st = direct_layout(src, dst->format, value_type == 0 ? 8 : 4, &dl)) return st;
    if (dl.passes == 0) return JLUST_STATUS_SUCCESS;
    if (!ws || (uintptr_t)ws % 256 || ws_bytes < (int64_t)dl.bytes)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_direct: workspace of %lld bytes, %zu needed at 256",
                    (long long)ws_bytes, dl.bytes);
    if (dst->origin != src->origin || dst->m != src->m || dst->n != src->n || dst->nnz != src->nnz)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_direct: target does not match the source");
    if (!dst->val || !dst->crd2 || (dst->format == JLUST_FORMAT_COO ? !dst->crd1 : !dst->pos2))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_direct: null device pointer");
    return value_type == 0 ? direct_run<double>(src, dst, dl, ws, count, (hipStream_t)stream)
                           : direct_run<float>(src, dst, dl, ws, count, (hipStream_t)stream);
}

extern "C" int jlust_hip_convert_blocks_workspace(const jlust_sparse *src, int32_t b1, int32_t b2, int value_type,
                                                  int64_t *bytes)
{
    clear_error();
    if (!bytes) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: null output pointer");
    *bytes = 0;
    KeyLayout L;
    if (int st = analyze_args(src, JLUST_FORMAT_BSR, b1, b2, 1, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    BlocksLayout bl;
    if (int st = blocks_layout(src, b1, b2, &bl)) return st;
    *bytes = (int64_t)bl.bytes;
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_convert_blocks_count(const jlust_sparse *src, int32_t b1, int32_t b2, int value_type, void *ws,
                                              int64_t ws_bytes, jlust_stream_t stream, int32_t *browptr, int64_t *nnzb)
{
    clear_error();
    if (!nnzb) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: null output pointer");
    *nnzb = -1;
    KeyLayout L;
    if (int st = analyze_args(src, JLUST_FORMAT_BSR, b1, b2, 1, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    BlocksLayout bl;
    if (int st = blocks_layout(src, b1, b2, &bl)) return st;
    if (bl.bytes == 0) return JLUST_STATUS_SUCCESS;
    if (!ws || (uintptr_t)ws % 256 || ws_bytes < (int64_t)bl.bytes || !browptr)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: workspace of %lld bytes, %zu needed at 256",
                    (long long)ws_bytes, bl.bytes);
    const BlocksWs w = blocks_ws(src, bl, ws);
    return value_type == 0 ? blocks_count<double>(src, b1, b2, bl, w, browptr, nnzb, (hipStream_t)stream)
                           : blocks_count<float>(src, b1, b2, bl, w, browptr, nnzb, (hipStream_t)stream);
}

extern "C" int jlust_hip_convert_blocks_fill(const jlust_sparse *src, const jlust_sparse *dst, int value_type,
                                             const void *ws, int64_t ws_bytes, jlust_stream_t stream)
{
    clear_error();
    if (!dst || dst->format != JLUST_FORMAT_BSR)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: null or other target");
    KeyLayout L;
    if (int st = analyze_args(src, JLUST_FORMAT_BSR, dst->b1, dst->b2, 1, value_type, &L)) return st;
    if (int st = require_device(nullptr)) return st;
    BlocksLayout bl;
    if (int st = blocks_layout(src, dst->b1, dst->b2, &bl)) return st;
    if (bl.bytes == 0 || !ws || (uintptr_t)ws % 256 || ws_bytes < (int64_t)bl.bytes)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: not this conversion, or its workspace");
    if (dst->origin != src->origin || dst->m != src->m || dst->n != src->n || dst->nouter < 0 ||
        dst->nnz != dst->nouter * dst->b1 * dst->b2)
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: target does not match the source");
    if (!dst->pos2 || bad_ptr(dst->crd2, dst->nouter) || bad_ptr(dst->val, dst->nnz))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_blocks: null device pointer");
    const BlocksWs w = blocks_ws(src, bl, const_cast<void *>(ws));
    return value_type == 0 ? blocks_fill<double>(src, dst, bl, w, (hipStream_t)stream)
                           : blocks_fill<float>(src, dst, bl, w, (hipStream_t)stream);
}

extern "C" int jlust_hip_convert_fill(jlust_convert_t h, const jlust_sparse *dst, jlust_stream_t stream)
{
    clear_error();
    if (!h) return fail(JLUST_STATUS_INVALID_ARGUMENT, "convert_fill: null handle");
    if (int st = dst_check(h, dst)) return st;
    if (int st = require_device(nullptr)) return st;
    return h->value_type == 0 ? fill<double>(h, dst, (hipStream_t)stream)
                              : fill<float>(h, dst, (hipStream_t)stream);
}

extern "C" int jlust_hip_convert_destroy(jlust_convert_t h)
{
    clear_error();
    if (!h) return JLUST_STATUS_SUCCESS;
    hipError_t e = h->mem ? hipFree(h->mem) : hipSuccess;
    delete h;
    if (e != hipSuccess) return hip_fail(e, "hipFree(convert)");
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_sparse_to_dense(const jlust_sparse *src, int value_type, void *dense, int64_t ld,
                                         jlust_stream_t stream)
{
    clear_error();
    if (int st = check_sparse(src, "sparse_to_dense")) return st;
    if (value_type != 0 && value_type != 1)
        return fail(JLUST_STATUS_UNSUPPORTED_VALUE_TYPE, "sparse_to_dense: value_type %d", value_type);
    if (ld < (src->m > 0 ? src->m : 1))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "sparse_to_dense: ld %lld < m %lld", (long long)ld,
                    (long long)src->m);
    if (!src_ptrs_ok(src) || bad_ptr(dense, src->m * src->n))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "sparse_to_dense: null device pointer");
    if (int st = require_device(nullptr)) return st;
    hipStream_t s = (hipStream_t)stream;
    const size_t tsz = value_type == 0 ? 8 : 4;
    if (src->m > 0 && src->n > 0)
        JLUST_HIP_TRY(hipMemset2DAsync(dense, (size_t)ld * tsz, 0, (size_t)src->m * tsz, (size_t)src->n, s));
    // Every stored entry is scattered (explicit zeros write 0; duplicates of
    // one coordinate are not defined, as in the reference).
    const int64_t N = src->nnz;
    if (N == 0) return JLUST_STATUS_SUCCESS;
    const KeyLayout L = layout_for(JLUST_FORMAT_CSR, src->m, src->n, 1, 1, 1);
    Workspace ws;
    size_t tmp_bytes = 0;
    if (int st = scan_bytes(segment_positions(src), &tmp_bytes)) return st;
    tmp_bytes = (tmp_bytes + 255) / 256 * 256;
    const size_t nseg_len = (size_t)(src->format == JLUST_FORMAT_BSR ? src->nouter : N) + 1;
    JLUST_HIP_TRY(hipMalloc(&ws.p, tmp_bytes + 8 * (size_t)N + 4 * (size_t)N + 4 * nseg_len + 64));
    char *b = (char *)ws.p;
    void *tmp = b;                      b += tmp_bytes;
    uint64_t *k = (uint64_t *)b;        b += 8 * (size_t)N;
    int32_t *keep = (int32_t *)b;       b += 4 * (size_t)N;
    int32_t *seg = (int32_t *)b;        b += 4 * nseg_len;
    int32_t *bad = (int32_t *)b;
    JLUST_HIP_TRY(hipMemsetAsync(bad, 0, 4, s));
    int64_t seglen = 0;
    if (int st = segments(src, seg, seglen, tmp, s)) return st;
    if (value_type == 0)
        hipLaunchKernelGGL((decompose_kernel<double>), dim3(cv_grid(N)), dim3(CV_BLOCK), 0, s, *src, seg, L, k,
                           keep, bad, nullptr);
    else
        hipLaunchKernelGGL((decompose_kernel<float>), dim3(cv_grid(N)), dim3(CV_BLOCK), 0, s, *src, seg, L, k,
                           keep, bad, nullptr);
    if (int st = check_launch("decompose_kernel")) return st;
    int32_t badh = 0;
    JLUST_HIP_TRY(hipMemcpyAsync(&badh, bad, 4, hipMemcpyDeviceToHost, s));
    JLUST_HIP_TRY(hipStreamSynchronize(s));
    if (badh)
        return fail(JLUST_STATUS_INVALID_ARGUMENT,
                    "sparse_to_dense: a stored coordinate lies outside the %lld x %lld extents",
                    (long long)src->m, (long long)src->n);
    if (value_type == 0)
        hipLaunchKernelGGL((to_dense_kernel<double>), dim3(cv_grid(N)), dim3(CV_BLOCK), 0, s, N, k, L,
                           (const double *)src->val, (double *)dense, ld);
    else
        hipLaunchKernelGGL((to_dense_kernel<float>), dim3(cv_grid(N)), dim3(CV_BLOCK), 0, s, N, k, L,
                           (const float *)src->val, (float *)dense, ld);
    if (int st = check_launch("to_dense_kernel")) return st;
    JLUST_HIP_TRY(hipStreamSynchronize(s));
    return JLUST_STATUS_SUCCESS;
}

extern "C" int jlust_hip_shift_index(int32_t *dst, const int32_t *src, int64_t len, int32_t delta,
                                     jlust_stream_t stream)
{
    clear_error();
    if (len < 0) return fail(JLUST_STATUS_INVALID_ARGUMENT, "shift_index: negative length");
    if (bad_ptr(dst, len) || bad_ptr(src, len))
        return fail(JLUST_STATUS_INVALID_ARGUMENT, "shift_index: null device pointer");
    if (int st = require_device(nullptr)) return st;
    if (len == 0) return JLUST_STATUS_SUCCESS;
    hipLaunchKernelGGL(shift_kernel, dim3(cv_grid(len)), dim3(CV_BLOCK), 0, (hipStream_t)stream, len, dst,
                       src, delta);
    return check_launch("shift_kernel");
}

namespace jlust {
// The unit's device code plus the rocPRIM instantiations a conversion runs
// (64-bit key sort, int32 scans), each launched once on 64 elements.
int preload_convert(hipStream_t s)
{
    JLUST_PRELOAD_KERNEL(compact_kernel);
    constexpr size_t n = 64;
    size_t need_sort = 0, need_max = 0, need_ex = 0, need_in = 0;
    uint64_t *kn = nullptr;
    int32_t *vn = nullptr;
    JLUST_HIP_TRY(rocprim::radix_sort_pairs(nullptr, need_sort, kn, kn, vn, vn, n, 0, 64, s));
    JLUST_HIP_TRY(rocprim::inclusive_scan(nullptr, need_max, vn, vn, n, rocprim::maximum<int32_t>(), s));
    JLUST_HIP_TRY(rocprim::exclusive_scan(nullptr, need_ex, vn, vn, 0, n, rocprim::plus<int32_t>(), s));
    JLUST_HIP_TRY(rocprim::inclusive_scan(nullptr, need_in, vn, vn, n, rocprim::plus<int32_t>(), s));
    const size_t need = std::max(std::max(need_sort, need_max), std::max(need_ex, need_in));
    void *buf = nullptr;
    JLUST_HIP_TRY(hipMalloc(&buf, 2 * n * 8 + 2 * n * 4 + (need + 255) / 256 * 256));
    char *b = (char *)buf;
    uint64_t *k0 = (uint64_t *)b, *k1 = (uint64_t *)(b + n * 8);
    int32_t *v0 = (int32_t *)(b + 2 * n * 8), *v1 = (int32_t *)(b + 2 * n * 8 + n * 4);
    void *tmp = b + 2 * n * 8 + 2 * n * 4;
    hipError_t e = hipMemsetAsync(buf, 0, 2 * n * 8 + 2 * n * 4, s);
    size_t t = need;
    if (e == hipSuccess) e = rocprim::radix_sort_pairs(tmp, t, k0, k1, v0, v1, n, 0, 64, s);
    t = need;
    if (e == hipSuccess) e = rocprim::inclusive_scan(tmp, t, v0, v1, n, rocprim::maximum<int32_t>(), s);
    t = need;
    if (e == hipSuccess) e = rocprim::exclusive_scan(tmp, t, v0, v1, 0, n, rocprim::plus<int32_t>(), s);
    t = need;
    if (e == hipSuccess) e = rocprim::inclusive_scan(tmp, t, v0, v1, n, rocprim::plus<int32_t>(), s);
    const hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(buf);
    if (e != hipSuccess) return hip_fail(e, "preload_convert");
    if (e2 != hipSuccess) return hip_fail(e2, "preload_convert");
    return JLUST_STATUS_SUCCESS;
}
}  // namespace jlust
