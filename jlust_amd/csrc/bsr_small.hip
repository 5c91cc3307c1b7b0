// bsr_small.hip -- BSR SpMM C = alpha*A*B + beta*C for square blocks of 2 to 8
// rows (gfx950, wave64), on the blocks as stored.
//
// Computes what bsr_spmm.hip computes for these shapes through a CSR
// expansion (ext/KernelAbstractionsExt/ops/spmm.jl:397-423 over the expanded
// rows), without the expansion: one column index per block instead of one per
// entry, and every gathered row of B used for all of the block's rows.
//
// B is re-laid row-major (spmm_row_major_copy), in passes of columns where the
// copy would be large (small_kchunk).  A wave's 64 lanes form NG =
// 64 / L groups; a group takes a block-row, each lane CPL columns of C for its
// B block-row rows in registers.  A group's next SB blocks are loaded by its
// own lanes, a stage ahead, and kept in LDS column by column, from where every
// lane of the group reads the same 16 bytes; waves share nothing, so nothing
// waits on a barrier.  Results pass through the wave's LDS and are written as
// runs of consecutive rows of C.
//
// What bounds it are the gathers behind L1, at four waves a SIMD (the mesh below:
// L1 serves an access in 47 % of its cycles and waits for L2 in 50 %, 38 % of its
// accesses missing); the LDS reads of a block's values serve NG block-rows at
// once.  Measured per product, with
// B's copy: 27-point mesh of 60,680 block-rows of 4 x 4 f64 blocks, k = 24:
// 955 us through the CSR expansion and the SpMM kernels before, 295 through
// the present ones, 134 here (2.2 TB/s of compulsory bytes); a plain call,
// which expanded A every time (440 us), saves that too.  8 x 8 f64, 30,690
// block-rows, k = 24: 1886 -> 235 us.
#include <algorithm>

#include "common.hpp"
#include "wave.hpp"

namespace jlust {
namespace {

constexpr int BS_BLOCK = 256;
constexpr int BS_WAVES = BS_BLOCK / 64;
constexpr int BS_STAGE = 8;              // values a lane loads per stage

template <typename T, int N>
struct alignas(sizeof(T) * N < 16 ? sizeof(T) * N : 16) Pack {
    T v[N];
};

struct SmallShape {
    int64_t mb;
    int64_t ldt;
    int k;
    int cols;                            // columns per blockIdx.y
    int L;                               // lanes per group: cols / CPL or more
    int sb;                              // blocks per stage
    int gs;                              // values of a group's stage in LDS
    int wave_vals;                       // values of a wave's stage or result tile in LDS
    int sums_at;                         // where a wave's further sums start
    int wave_stride;                     // values from one wave's LDS to the next
    int32_t origin;
    int row_major;
    unsigned run;                        // consecutive workgroups per XCD
};

// LV sums per row and column: a block's product goes into the first, in a
// register, which goes into the next, in LDS, after four blocks (LV = 2) or
// three, that one into a third after three of those (small_levels).  In
// registers they cost waves (8 x 8 f64, k = 2: 190 registers, 115 us against
// 66).
template <typename T, int B, int CPL, int LV>
__global__ __launch_bounds__(BS_BLOCK) void bsr_small_spmm_kernel(
    SmallShape sh, const int32_t *__restrict__ browptr, const int32_t *__restrict__ bcolind,
    const T *__restrict__ val, const T *__restrict__ Bt0, T alpha, T beta, int beta_zero, T *__restrict__ C,
    int64_t ldc)
{
    constexpr int V16 = 16 / sizeof(T);
    constexpr int W = CPL < V16 ? CPL : V16;               // columns per load of B
    constexpr int AW = B <= 2 ? 2 : V16 < 4 ? 2 : 4;       // values per read of A
    constexpr int BP = (B + AW - 1) / AW * AW;             // a block row in LDS
    constexpr int BB = B * B;
    constexpr int HALF = B < 5 || LV == 1 ? B : (B + 1) / 2;   // a block row's product in two halves
    extern __shared__ __attribute__((aligned(16))) char s_mem[];

    const unsigned x = blockIdx.x % NUM_XCD, i0 = blockIdx.x / NUM_XCD;
    const int64_t wg = (int64_t)(i0 / sh.run * NUM_XCD + x) * sh.run + i0 % sh.run;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int L = sh.L, NG = 64 / L;
    const int64_t R0 = (wg * BS_WAVES + wave) * NG;
    if (R0 >= sh.mb) return;
    const int grp = lane / L, sub = lane - grp * L;
    T *const s_a = reinterpret_cast<T *>(s_mem) + wave * sh.wave_stride;
    uint32_t *const s_off = reinterpret_cast<uint32_t *>(s_a + sh.wave_vals);
    T *const s_sum = s_a + sh.sums_at + lane;              // sum h, row r, column c: [((h - 1) * B + r) * CPL + c][lane]
    const int c0 = (int)blockIdx.y * sh.cols;
    const int kk = min(sh.cols, sh.k - c0);
    const uint32_t col = (uint32_t)(c0 + min(sub * CPL, (int)sh.ldt - c0 - CPL)) * (uint32_t)sizeof(T);
    const uint32_t row_bytes = (uint32_t)(sh.ldt * sizeof(T));

    const bool live = grp < NG && R0 + grp < sh.mb;
    int64_t q0 = 0;
    int n = 0;
    if (live) {
        q0 = (int64_t)browptr[R0 + grp] - sh.origin;
        n = max(browptr[R0 + grp + 1] - sh.origin - (int)q0, 0);
    }
    const T *const va = val + q0 * BB;
    T *const a_dst = s_a + grp * sh.gs;

    // A stage: blocks s0 .. s0 + sb - 1 of the group, element e = sub + t * L.
    T st[BS_STAGE];
    uint32_t oc = 0;
    auto load_stage = [&](int s0) {
        const int cnt = min(sh.sb, n - s0);
        const T *const p = va + (int64_t)s0 * BB;
#pragma unroll
        for (int t = 0; t < BS_STAGE; ++t)
            if (sub + t * L < cnt * BB) st[t] = p[sub + t * L];
        if (sub < cnt) oc = (uint32_t)(bcolind[q0 + s0 + sub] - sh.origin) * (uint32_t)B * row_bytes;
    };
    auto store_stage = [&](int s0) {
        const int cnt = min(sh.sb, n - s0);
#pragma unroll
        for (int t = 0; t < BS_STAGE; ++t) {
            const int e = sub + t * L;
            if (e < cnt * BB) {
                const int blk = e / BB, w = e % BB, r = w / B, c = w % B;
                const int ii = sh.row_major ? r : c, jj = sh.row_major ? c : r;
                a_dst[(blk * B + ii) * BP + jj] = st[t];
            }
        }
        if (sub < cnt) s_off[grp * sh.sb + sub] = oc;
    };

    T acc[B][CPL];
#pragma unroll
    for (int r = 0; r < B; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[r][c] = T(0);
#pragma unroll
    for (int i = 0; i < (LV - 1) * B * CPL; ++i) s_sum[i * 64] = T(0);
    auto carry = [&](int h) {                              // sum h into the next
#pragma unroll
        for (int r = 0; r < B; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                T *const up = s_sum + ((h * B + r) * CPL + c) * 64;
                if (h == 0) {
                    *up += acc[r][c];
                    acc[r][c] = T(0);
                } else {
                    *up += *(up - B * CPL * 64);
                    *(up - B * CPL * 64) = T(0);
                }
            }
    };
    int filled0 = 0, filled1 = 0;

    load_stage(0);
    for (int s0 = 0; __any(s0 < n); s0 += sh.sb) {
        wave_sync();
        store_stage(s0);
        wave_sync();
        load_stage(s0 + sh.sb);
        const int top = min(sh.sb, n - s0);
        for (int u = 0; __any(u < top); ++u) {
            if (u < top) {
                const char *const bp = reinterpret_cast<const char *>(Bt0);
                const uint32_t off = s_off[grp * sh.sb + u] + col;
                Pack<T, W> b[B][CPL / W];
#pragma unroll
                for (int jj = 0; jj < B; ++jj)
#pragma unroll
                    for (int v = 0; v < CPL / W; ++v)
                        b[jj][v] = *reinterpret_cast<const Pack<T, W> *>(
                            bp + (off + (uint32_t)jj * row_bytes + (uint32_t)(v * W * sizeof(T))));
                // A row of the block's own product first, then into the row's sum.
#pragma unroll
                for (int r = 0; r < B; ++r) {
                    T a[BP];
#pragma unroll
                    for (int v = 0; v < BP / AW; ++v) {
                        const Pack<T, AW> p = *reinterpret_cast<const Pack<T, AW> *>(a_dst + (u * B + r) * BP + v * AW);
#pragma unroll
                        for (int e = 0; e < AW; ++e) a[v * AW + e] = p.v[e];
                    }
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        T t = a[0] * b[0][c / W].v[c % W];
#pragma unroll
                        for (int jj = 1; jj < HALF; ++jj) t += a[jj] * b[jj][c / W].v[c % W];
                        if constexpr (HALF < B) {
                            T t2 = a[HALF] * b[HALF][c / W].v[c % W];
#pragma unroll
                            for (int jj = HALF + 1; jj < B; ++jj) t2 += a[jj] * b[jj][c / W].v[c % W];
                            t += t2;
                        }
                        acc[r][c] += t;
                    }
                }
            }
            // All groups together: a sum of a finished row stays what it is, now
            // or below.
            if constexpr (LV > 1) {
                if (++filled0 == (LV == 2 ? 4 : 3)) {
                    filled0 = 0;
                    carry(0);
                    if constexpr (LV > 2) {
                        if (++filled1 == 3) {
                            filled1 = 0;
                            carry(1);
                        }
                    }
                }
            }
        }
    }
    if constexpr (LV > 1) {
#pragma unroll
        for (int r = 0; r < B; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                T *const up = s_sum + (r * CPL + c) * 64;
                acc[r][c] += *up;
                if constexpr (LV > 2) acc[r][c] += up[B * CPL * 64];
            }
    }

    // Column c of every lane: the wave's rows, one run per column of C.
    const int nr = (int)min((int64_t)NG, sh.mb - R0) * B, ts = NG * B + 1;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        wave_sync();
        if (grp < NG) {
#pragma unroll
            for (int r = 0; r < B; ++r) s_a[sub * ts + grp * B + r] = acc[r][c];
        }
        wave_sync();
        for (int s = 0; s < L; ++s) {
            if (s * CPL + c >= kk) break;
            T *const dst = C + R0 * B + (int64_t)(c0 + s * CPL + c) * ldc;
            for (int r = lane; r < nr; r += 64) {
                const T v = alpha * s_a[s * ts + r];
                dst[r] = beta_zero ? v : v + beta * dst[r];
            }
        }
    }
}

// out[0] = the longest block-row, out[1] set where browptr decreases, out[2] and
// out[3] its ends: one copy to the host, which costs a plain call more than the
// kernel does.
__global__ void block_row_longest_kernel(int64_t mb, const int32_t *__restrict__ browptr, int32_t *__restrict__ out)
{
    int32_t len = 0;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < mb; r += (int64_t)gridDim.x * blockDim.x) {
        const int64_t d = (int64_t)browptr[r + 1] - browptr[r];
        if (d < 0) out[1] = 1;
        len = max(len, (int32_t)min(d, (int64_t)INT32_MAX));
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) len = max(len, __shfl_xor(len, off, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(out, len);
    if (blockIdx.x == 0 && threadIdx.x < 2) out[2 + threadIdx.x] = browptr[threadIdx.x * mb];
}

__global__ void clear_pair_kernel(int32_t *p)
{
    if (threadIdx.x < 2) p[threadIdx.x] = 0;
}

template <typename T>
constexpr int MAX_COLS = 16 / (int)sizeof(T);

// Columns per lane: 16 bytes, fewer while a group has less than 4 lanes.
template <typename T>
int small_cpl(int64_t k)
{
    int c = MAX_COLS<T>;
    while (c > 1 && (k + c - 1) / c < 4) c /= 2;
    return c;
}

// Sums per row and column.  The expansion's kernels hold S = 64 / p sums of a
// column's products for k <= 32 columns (p the power of two at k or above), one
// beyond.  One chain of the blocks' products rounds as little as those below S =
// b, two levels below 3b, three from there: counted over rows of 3 to 32 blocks,
// 0.53-1.02 times the error of the S sums, where one chain made up to 1.34.
// Measured, f32, 27 blocks a row: 2 x 2, k = 2, 1.01 (one chain 1.53); 3 x 3, k =
// 12, 0.83 (1.14).
inline int small_levels(int64_t b, int64_t k)
{
    int64_t p = 1;
    while (p < k) p *= 2;
    const int64_t S = p <= 32 ? 64 / p : 1;
    return S >= 3 * b ? 3 : S >= b ? 2 : 1;
}

template <typename T, int B, int CPL, int LV>
int launch(const SmallShape &base, const int32_t *browptr, const int32_t *bcolind, const T *val, const T *Bt, T alpha,
           T beta, T *C, int64_t ldc, hipStream_t s)
{
    SmallShape sh = base;
    const int64_t ny = (sh.k + 64 * CPL - 1) / (64 * CPL);
    sh.cols = (int)(((sh.k + ny - 1) / ny + CPL - 1) / CPL * CPL);
    // Lanes beyond the columns where a stage would not hold a block otherwise; for
    // blocks up to 4 x 4, four values a lane: with eight, two lanes hold a block and
    // 32 block-rows' blocks, a line or more apart, make up each load.  Mesh of 27
    // blocks a row, 38^3, k = 2, against eight: 4 x 4 f32 70 -> 34 us, f64 57 -> 45;
    // 3 x 3 f32 50 -> 36, f64 52 -> 37; against the expansion 52, 94, 43, 59.
    // Larger blocks fill their loads with eight (8 x 8 f64: 74 us, 98 with four).
    sh.L = max(sh.cols / CPL, (B * B + (B <= 4 ? 4 : BS_STAGE) - 1) / (B <= 4 ? 4 : BS_STAGE));
    const int NG = 64 / sh.L;
    constexpr int V16 = 16 / (int)sizeof(T), AW = B <= 2 ? 2 : V16 < 4 ? 2 : 4, BP = (B + AW - 1) / AW * AW;
    sh.sb = max(1, min(min(8, sh.L), BS_STAGE * sh.L / (B * B)));
    // A group's stage starts an odd number of 16-byte units after the last one's.
    sh.gs = (sh.sb * B * BP + V16 - 1) / V16 * V16;
    if (sh.gs / V16 % 2 == 0) sh.gs += V16;
    sh.wave_vals = (max(NG * sh.gs, sh.L * (NG * B + 1)) + V16 - 1) / V16 * V16;
    sh.sums_at = (sh.wave_vals + NG * sh.sb * 4 / (int)sizeof(T) + V16) / V16 * V16;
    sh.wave_stride = sh.sums_at + (LV - 1) * B * CPL * 64;
    const size_t per_wave = sizeof(T) * (size_t)sh.wave_stride;
    const int64_t wgs = (sh.mb + (int64_t)BS_WAVES * NG - 1) / (BS_WAVES * NG);
    sh.run = xcd_run(wgs);
    const dim3 grid((unsigned)((wgs + (int64_t)sh.run * NUM_XCD - 1) / ((int64_t)sh.run * NUM_XCD) * sh.run * NUM_XCD),
                    (unsigned)ny);
    hipLaunchKernelGGL((bsr_small_spmm_kernel<T, B, CPL, LV>), grid, dim3(BS_BLOCK), per_wave * BS_WAVES, s, sh, browptr,
                       bcolind, val, Bt, alpha, beta, beta == T(0), C, ldc);
    return check_launch("bsr_small_spmm_kernel");
}

template <typename T, int B>
int launch_cpl(int cpl, const SmallShape &sh, const int32_t *browptr, const int32_t *bcolind, const T *val,
               const T *Bt, T alpha, T beta, T *C, int64_t ldc, hipStream_t s)
{
    constexpr int M = MAX_COLS<T>;
    const int lv = small_levels(B, sh.k);
    // Only what small_cpl and small_levels can ask for together.
#define JLUST_LAUNCH(N, LV) \
    return launch<T, B, (N <= M ? N : M), LV>(sh, browptr, bcolind, val, Bt, alpha, beta, C, ldc, s)
    if (cpl == 4) {                                        // 13 columns or more
        if constexpr (B <= 4) {
            if (lv == 2) JLUST_LAUNCH(4, 2);
        }
        JLUST_LAUNCH(4, 1);
    }
    if (cpl == 2) {                                        // 7 or more
        if constexpr (B == 2) {
            if (lv == 3) JLUST_LAUNCH(2, 3);
        }
        if (lv == 2) JLUST_LAUNCH(2, 2);
        JLUST_LAUNCH(2, 1);
    }
    if (lv == 3) JLUST_LAUNCH(1, 3);                       // 6 or fewer
    JLUST_LAUNCH(1, 2);
#undef JLUST_LAUNCH
}

}  // namespace

// Columns per pass: as few passes of about equal width as keep B's copy within
// 512 MB, or 1 GB for blocks past 4 x 4, whose values are the larger part of
// what a further pass reads again; 16 columns at least.  us per product, copy
// within 256 MB / 512 MB / 1 GB: 4 x 4 f64 on a band, 2M rows, k = 48: 1311 /
// 1250 / 1433; 2 x 2 f64 mesh of 1M nodes, k = 48: 2139 / 2175 / 2762; 3 x 3
// f32 mesh of 1M nodes, k = 128: 5227 / 4344 / 4380 (one pass: 4932); 4 x 4 f64
// mesh of 422k nodes, k = 24: 1224 / 961 / 954; 8 x 8: 3944 / 3940 / 2969.
static int64_t small_kchunk(int64_t nb, int64_t b, int64_t k, size_t tsz)
{
    const size_t budget = (size_t)(b <= 4 ? 512 : 1024) << 20;
    const int64_t passes = (int64_t)(((size_t)k * (size_t)(nb * b) * tsz + budget - 1) / budget);
    if (passes <= 1) return k;
    return std::min(k, std::max<int64_t>(16, ((k + passes - 1) / passes + 7) / 8 * 8));
}

bool bsr_small_shape(int64_t nb, int64_t b1, int64_t b2, int64_t k, size_t tsz)
{
    if (b1 != b2 || b1 < 2 || b1 > 8 || k < 2) return false;
    // Offsets into B's copy are 32-bit.
    return (uint64_t)(nb * b2 + 1) * (uint64_t)(small_kchunk(nb, b2, k, tsz) + 8) * tsz < 0xff000000ull;
}

size_t bsr_small_copy_bytes(int64_t nb, int64_t b, int64_t k, size_t tsz)
{
    return tsz * (size_t)(nb * b + 1) * (size_t)((small_kchunk(nb, b, k, tsz) + 7) / 8 * 8);
}

// The longest block-row that the kernel takes.  A group of lanes walks its
// block-row alone, 0.5 (2 x 2) to 1.6 us (8 x 8) a block, about 0.2 * b; the
// expansion shares long rows among the card and takes an entry in the time of
// its k values, 64 bytes at least, at 8 TB/s, a plain call 132 bytes more for
// making it.  So a row may have as many blocks as pass while the expansion's
// entries do; 40 in a plan and 512 / b in a plain call, whose expansion takes 90
// us and more, in any case; and 64 or 4 times the mean at most.  us, this kernel /
// the expansion, plan, 4 x 4 f64, k = 24: 512 block-rows of 1024 blocks 644 /
// 196, 2048 of 64 59 / 43, 4096 of 64 59 / 59, 8192 of 128 103 / 193; 8 x 8:
// 1024 of 128 232 / 123, 4096 of 128 281 / 449; f32: 2 x 2, k = 8, 2048 of 1024
// 514 / 75, 16384 of 128 74 / 70; 4 x 4, k = 6, 16384 of 128 105 / 237.  Plain, 4
// x 4 f64, k = 24: 512 of 256 233 / 191, 2048 of 256 224 / 309; 2 x 2 f32, k = 8,
// 4096 of 512 314 / 276, 8192 of 512 302 / 421.  8 block-rows of 65,536 4 x 4
// blocks: 47 ms here, 0.4 by the expansion.
static int64_t small_longest(int64_t mb, int64_t nnzb, int64_t b, int64_t k, size_t tsz, bool plan)
{
    const double entry = std::max(64.0, (double)k * (double)tsz) + (plan ? 0.0 : 132.0);
    const double most = std::max(plan ? 40.0 : 512.0 / (double)b, (double)nnzb * (double)b * entry / 1.6e6);
    return (int64_t)std::min(most, (double)std::max<int64_t>(64, 4 * nnzb / mb));
}

int bsr_small_pattern(int64_t mb, int64_t nnzb, int64_t b, int64_t k, size_t tsz, bool plan, int32_t origin,
                      const int32_t *browptr, hipStream_t s, bool *even)
{
    *even = false;
    if (mb == 0 || nnzb == 0) return JLUST_STATUS_SUCCESS;
    void *ws = nullptr;
    if (int st = scratch((jlust_stream_t)s, 64, &ws)) return st;
    int32_t *d = (int32_t *)ws, h[4] = {0, 0, 0, 0};
    hipLaunchKernelGGL(clear_pair_kernel, dim3(1), dim3(64), 0, s, d);
    hipLaunchKernelGGL(block_row_longest_kernel, dim3((unsigned)min((mb + 255) / 256, (int64_t)512)), dim3(256), 0, s,
                       mb, browptr, d);
    if (int st = check_launch("block_row_longest_kernel")) return st;
    JLUST_HIP_TRY(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s));
    JLUST_HIP_TRY(hipStreamSynchronize(s));
    if (h[2] != origin || (int64_t)h[3] - origin != nnzb || h[1]) return JLUST_STATUS_SUCCESS;
    *even = h[0] <= small_longest(mb, nnzb, b, k, tsz, plan);
    return JLUST_STATUS_SUCCESS;
}

// One pass: its k columns.
template <typename T>
static int small_pass(int64_t mb, int64_t nb, int64_t b, int32_t origin, const int32_t *browptr,
                      const int32_t *bcolind, const T *val, int row_major, int64_t k, T alpha, const T *B, int64_t ldb,
                      T beta, T *C, int64_t ldc, T *Bt, hipStream_t s)
{
    const int cpl = small_cpl<T>(k);
    SmallShape sh{};
    sh.mb = mb;
    sh.k = (int)k;
    sh.ldt = (k + cpl - 1) / cpl * cpl;
    sh.origin = origin;
    sh.row_major = row_major;
    if (int st = spmm_row_major_copy(sizeof(T) == 8 ? 0 : 1, nb * b, k, B, ldb, Bt, sh.ldt, s)) return st;
#define JLUST_B(N) \
    case N: return launch_cpl<T, N>(cpl, sh, browptr, bcolind, val, Bt, alpha, beta, C, ldc, s);
    switch (b) {
        JLUST_B(2)
        JLUST_B(3)
        JLUST_B(4)
        JLUST_B(5)
        JLUST_B(6)
        JLUST_B(7)
        JLUST_B(8)
    }
#undef JLUST_B
    return fail(JLUST_STATUS_INVALID_ARGUMENT, "bsr_small_spmm: block size %lld", (long long)b);
}

template <typename T>
int bsr_small_spmm(int64_t mb, int64_t nb, int64_t b, int32_t origin, const int32_t *browptr, const int32_t *bcolind,
                   const T *val, int row_major, int64_t k, T alpha, const T *B, int64_t ldb, T beta, T *C, int64_t ldc,
                   T *Bt, hipStream_t s)
{
    if (mb == 0) return JLUST_STATUS_SUCCESS;
    const int64_t kc = small_kchunk(nb, b, k, sizeof(T));
    for (int64_t c0 = 0; c0 < k; c0 += kc)
        if (int st = small_pass<T>(mb, nb, b, origin, browptr, bcolind, val, row_major, std::min(kc, k - c0), alpha,
                                   B + c0 * ldb, ldb, beta, C + c0 * ldc, ldc, Bt, s))
            return st;
    return JLUST_STATUS_SUCCESS;
}

template int bsr_small_spmm<double>(int64_t, int64_t, int64_t, int32_t, const int32_t *, const int32_t *,
                                    const double *, int, int64_t, double, const double *, int64_t, double, double *,
                                    int64_t, double *, hipStream_t);
template int bsr_small_spmm<float>(int64_t, int64_t, int64_t, int32_t, const int32_t *, const int32_t *, const float *,
                                   int, int64_t, float, const float *, int64_t, float, float *, int64_t, float *,
                                   hipStream_t);

int preload_bsr_small()
{
    JLUST_PRELOAD_KERNEL(block_row_longest_kernel);
    return JLUST_STATUS_SUCCESS;
}

}  // namespace jlust
