// Sum-of-products SpMM for gfx950: c (R, C) = A (R, K) sparse @ b (K, C) dense row-major, fp32.
// Stands behind mamtorch_kernel_sparsev1::cusparsemm, which the reference implements with cuSPARSE
// (CSR: mamtorch/sparse/kernel/v1/csrc/cuda/cusparsemm_csr.cu:19-77, CUSPARSE_SPMM_CSR_ALG2;
//  COO: mamtorch/sparse/kernel/v1/csrc/cuda/cusparsemm_coo.cu, same call on a COO descriptor),
// int64 indices, alpha = 1, beta = 0, and a cudaMalloc per call that is never freed (:60).
// Here nothing is allocated.
//
// Lanes are output columns: a stored entry (r, k, v) adds v * b[k, :] to c[r, :], and b[k, c0..c0+255]
// is one coalesced 1 KiB load for a wave (4 columns per lane).
//   CSR: a wave owns one row for one panel of 256 columns; column indices and values are wave-uniform
//        scalar loads; the loads of the next 8 entries are in flight while 8 are consumed; the row of c
//        is written once, no atomics, no zero fill.  Workgroups are numbered panel by panel and dealt out so that
//        an XCD works on panels of its own: its L2 then holds the panel of b (1 KiB per row of b) instead of all
//        eight fetching the same one, and c goes past it (non-temporal stores).  4096 x 4096 at 1 % x 4096 columns: 128 ->
//        102 us, 27 TB/s of b rows (0.2 %: 58 -> 29 us; 10 %: 880 -> 870 us, 31.6 TB/s); 90 us where K = 2048 leaves
//        room beside the panel.  Bound by the 64 bytes per clock and CU of the vector memory path (39 TB/s).
//        Entries handed out by v_readlane from lane-held blocks that run on over the wave's rows: 116 us (97 registers, 4
//        waves per SIMD); 2 columns per lane (panels of half the size): 150 us; 4 entries in flight: 108 us.
//        Narrow c: two or four entries per load instead of idle lanes (4096 x 4096 at 5 %, 128 / 64 columns: 26 -> 17, 26 -> 11 us;
//        256 columns 34 and 33 us, 4096 columns at 1 % 102 and 123 us).
//   COO: entries may come in any order and may repeat, so c is cleared first; a wave takes 64
//        consecutive entries, keeps a run of equal row indices in registers and flushes it with
//        atomic adds when the row changes.  On row-sorted input (what Tensor.to_sparse() and
//        coalesce() produce) that is about one flush per row and wave.  A lane's columns are 64 apart: adds of 64
//        neighbouring words (four neighbouring columns a lane, as in the CSR kernel, us: 236641 entries in any order x 2252
//        columns 7180, like this 1970; 24684 x 6871 2840 and 800; 222063 ascending x 704 613 and 178).
// Products are fused multiply-adds in ascending entry order within a wave (narrow c: within each of the two or four
// parts of a row), 64 of them at a time; sums that span waves (COO only) are combined in no fixed order.
#include "mam_common.h"

namespace mam {
namespace spmm {

constexpr int NT = 256;
// loads issued together: fewer where one holds four entries (65536 x 512 with 10 entries a row x 50 columns, 4 and 8: 16.9 and 20.9
// us, 50 entries x 64 columns 42 and 54; one row of 32768 entries alone 1660 and 1560), not where it holds two (10 entries a row x
// 100 columns 17.6 and 20.4, the row alone x 128 columns 2230 and 1730)
constexpr int loads_of(int per) { return per > 2 ? 4 : 8; }
constexpr int COO_CHUNK = 64;  // entries per wave and pass

typedef const __attribute__((address_space(4))) int64_t const_i64;
typedef const __attribute__((address_space(4))) float const_f32;

template <int N> struct Count { static constexpr int value = N; };

template <int TI> struct Vec;
template <> struct Vec<1> { typedef float type; };
template <> struct Vec<4> { typedef float4 type; };

__device__ __forceinline__ void axpy(float (&acc)[1], float v, const float &b) { acc[0] = __builtin_fmaf(v, b, acc[0]); }
__device__ __forceinline__ void axpy(float (&acc)[4], float v, const float4 &b)
{
    acc[0] = __builtin_fmaf(v, b.x, acc[0]);
    acc[1] = __builtin_fmaf(v, b.y, acc[1]);
    acc[2] = __builtin_fmaf(v, b.z, acc[2]);
    acc[3] = __builtin_fmaf(v, b.w, acc[3]);
}

// Which panel of columns a workgroup works on and which block of rows: numbered panel by panel over the XCDs, or a row of the grid
// each, so that all XCDs walk one panel at a time: where the numbers would be more than a launch holds in one dimension, and where the
// panels of eight XCDs are too much for the memory-side cache together (us by XCDs and in turn, 4096 columns: K = 4096 107 / 126, 16384 293 /
// 310, 32768 346 / 346, 65536 354 / 346; 1024 columns, four panels: 65536 91.6 / 93.2).
struct Place { int panel, block; };
// (`panels` by XCD, 0: a row of the grid each.  An argument and no division for one panel: the grid's size would be one more wait, and
// 2^20 rows x 1 column with 0.05 entries each take 171 us with both, 134 without the division, 130 without either; 103 where empty rows are done with at once.)
__device__ __forceinline__ Place place_of(int blocks, int panels)
{
    if (panels == 0) return {(int)blockIdx.y, (int)blockIdx.x};
    const int logical = xcd_remap(blockIdx.x, panels * blocks);
    if (panels == 1) return {0, logical};
    return {logical / blocks, logical % blocks};
}
constexpr int64_t MOST_PANEL_ROWS = 8 * 32768;           // of b, in the panels that are walked at once
static bool by_xcd(int64_t panels, int64_t blocks, int64_t K)
{
    // less than 2^32 threads in a dimension
    return K * (panels < 8 ? panels : 8) <= MOST_PANEL_ROWS && panels * blocks < UINT32_MAX / NT;
}

// four consecutive words, 4-byte aligned; past the L2 whether or not rows of c start lines (past it / to it, us: 4096 x 4096 with 8
// entries a row x 4093 columns 35.4 / 39.9, x 4096 30.5 / 33.2; 65536 x 512 with 10 x 101 22.7 / 24.6, x 50 19 / 19)
typedef float words4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void store4(float *dst, const float (&a)[4])
{
    const words4 v = {a[0], a[1], a[2], a[3]};
    __builtin_nontemporal_store(v, reinterpret_cast<words4 *>(dst));
}
__device__ __forceinline__ void store4(float *, const float (&)[1]) {}

// Whether any workgroup of row_offsets_kernel found that a COO operand may not be summed row by row.  One load per wave, beside
// that of the row offsets.
constexpr int VERDICTS = 256;         // a word of each checking workgroup
__device__ __forceinline__ bool not_by_rows(const uint32_t *verdicts)
{
    const uint4 v = reinterpret_cast<const uint4 *>(verdicts)[threadIdx.x & 63];
    static_assert(VERDICTS == 64 * 4, "four words a lane");
    return __ballot((v.x | v.y | v.z | v.w) != 0) != 0;
}

// verdicts: of a COO operand's rows, nullptr: a CSR operand.  Where they forbid the sum by rows, c is cleared for coo_spmm_kernel.
// PER: entries per load, each by 64 / PER lanes (NEAR only).
// NEAR: b spans less than 4 GiB; a b row is then a buffer load of any alignment (a load of 4 words needs 4 bytes).  PER = 1: C is at
// least 4 and the row's byte offset a scalar register, which the load's range check need not count, so no lane may read past its row:
// lanes that would take the last four columns.  PER > 1: the offset is in the vector register, which the check does count: lanes
// past the last column read on into the next row or, past the end of b, zeros.  Otherwise TI = 4 needs C a multiple of 4 and 16-byte
// aligned rows.
template <int TI, bool NEAR, int PER>
__global__ __launch_bounds__(NT) void csr_spmm_kernel(const int64_t *__restrict__ crow,
                                                      const int64_t *__restrict__ col,
                                                      const float *__restrict__ val,
                                                      const float *__restrict__ b, int64_t ldb, uint32_t b_bytes,
                                                      float *__restrict__ c, int R, int C, int row_blocks, int panels, int width,
                                                      const uint32_t *__restrict__ verdicts)
{
    typedef typename Vec<TI>::type vec;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Place at_block = place_of(row_blocks, panels);
    // (uniform, but the division leaves them in vector registers: 97 of 96 with two entries per load)
    const int panel = __builtin_amdgcn_readfirstlane(at_block.panel), r = __builtin_amdgcn_readfirstlane(at_block.block) * (NT / 64) + wave;
    if (r >= R) return;
    constexpr int EG = loads_of(PER);
    constexpr int LANES = 64 / PER;      // of one entry; the parts are added at the end
    if (PER > 1) width = LANES * TI;     // (one panel)
    const int c0 = panel * width + lane % LANES * TI;
    const bool in = lane % LANES * TI < width && c0 < C;
    // the columns a lane sums: lanes past the panel's last column take its first and store nothing
    const int wanted = in ? c0 : panel * width, cl = TI == 4 && PER == 1 && wanted > C - 4 ? C - 4 : wanted;
    const int part = lane / LANES;

    const_i64 *ccol = (const_i64 *)col;
    const_f32 *cval = (const_f32 *)val;
    const int64_t beg = ((const_i64 *)crow)[r], end = ((const_i64 *)crow)[r + 1];
    const int nnz = verdicts && not_by_rows(verdicts) ? 0 : (int)(end - beg);
    float acc[TI];
#pragma unroll
    for (int t = 0; t < TI; ++t) acc[t] = 0.0f;
    auto put = [&] {
        if (part != 0 || !in) return;
        const int first = PER == 1 ? cl : c0;
        float *dst = c + (int64_t)r * C + first;
        if (TI == 4 && c0 + 3 < C) {
            store4(dst, acc);
        } else {            // (those below c0 are other lanes')
#pragma unroll
            for (int t = 0; t < TI; ++t)
                if (first + t >= c0 && first + t < C) dst[t] = acc[t];
        }
    };
    if (PER > 1 && nnz == 0) return put();

    const float *bl = b + cl;
    const __amdgpu_buffer_rsrc_t near = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(b), 0, (int)b_bytes, 0x00020000);
    const uint32_t row_bytes = (uint32_t)ldb * 4u;
    auto near_row = [&](uint32_t lane_bytes, uint32_t bytes) {
        return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(near, lane_bytes, bytes, 0));
    };
    auto b_row = [&](int64_t e) -> vec {
        if constexpr (PER > 1) {
            uint32_t at = (uint32_t)ccol[e] * row_bytes;
#pragma unroll
            for (int p = 1; p < PER; ++p) {
                const uint32_t other = (uint32_t)ccol[e + p] * row_bytes;
                at = part == p ? other : at;
            }
            return near_row(at + cl * 4, 0);
        } else if constexpr (NEAR) {
            return near_row(cl * 4, (uint32_t)ccol[e] * row_bytes);
        } else {
            return *reinterpret_cast<const vec *>(bl + ccol[e] * ldb);
        }
    };
    auto value = [&](int64_t e) {
        float v = cval[e];
#pragma unroll
        for (int p = 1; p < PER; ++p) {
            const float other = cval[e + p];
            v = part == p ? other : v;
        }
        return v;
    };

    const int ng = nnz / (EG * PER);
    vec xa[EG], xb[EG];
    float wa[EG], wb[EG];
    auto issue = [&](int g, vec (&xv)[EG], float (&wv)[EG]) {
#pragma unroll
        for (int u = 0; u < EG; ++u) {
            xv[u] = b_row(beg + (g * EG + u) * PER);
            wv[u] = value(beg + (g * EG + u) * PER);
        }
    };
    auto consume = [&](const vec (&xv)[EG], const float (&wv)[EG]) {
#pragma unroll
        for (int u = 0; u < EG; ++u) axpy(acc, wv[u], xv[u]);
    };
    // sums of 64 terms are added to a sum of their own, as coo_spmm_kernel adds its to c: a row's rounding errors grow with 64 + n /
    // 64 instead of with n
    float total[TI];
#pragma unroll
    for (int t = 0; t < TI; ++t) total[t] = 0.0f;
    auto fold = [&] {
#pragma unroll
        for (int t = 0; t < TI; ++t) {
            total[t] += acc[t];
            acc[t] = 0.0f;
        }
    };
    if (ng > 0) issue(0, xa, wa);
    for (int g = 0; g < ng; g += 2) {
        if (g % (COO_CHUNK / EG) == 0) fold();
        if (g + 1 < ng) issue(g + 1, xb, wb);
        __builtin_amdgcn_sched_barrier(0);
        consume(xa, wa);
        __builtin_amdgcn_sched_barrier(0);
        if (g + 1 >= ng) break;
        if (g + 2 < ng) issue(g + 2, xa, wa);
        __builtin_amdgcn_sched_barrier(0);
        consume(xb, wb);
        __builtin_amdgcn_sched_barrier(0);
    }
    int i = ng * EG * PER;
    auto few = [&](auto count) {
        constexpr int n = decltype(count)::value;
        if (nnz - i < n * PER) return;
        vec x[n];
        float w[n];
#pragma unroll
        for (int u = 0; u < n; ++u) {
            x[u] = b_row(beg + i + u * PER);
            w[u] = value(beg + i + u * PER);
        }
#pragma unroll
        for (int u = 0; u < n; ++u) axpy(acc, w[u], x[u]);
        i += n * PER;
    };
    few(Count<4>());
    few(Count<2>());
    few(Count<1>());
    if constexpr (PER > 1) {
        if (i + part < nnz) {            // fewer entries than parts
            const int64_t e = beg + i + part;
            axpy(acc, val[e], near_row((uint32_t)col[e] * row_bytes + cl * 4, 0));
        }
    }
#pragma unroll
    for (int t = 0; t < TI; ++t) acc[t] += total[t];
#pragma unroll
    for (int s = LANES; s < 64; s <<= 1)
#pragma unroll
        for (int t = 0; t < TI; ++t) acc[t] += __shfl_xor(acc[t], s);
    put();
}

// A lane's TI columns are 64 apart, so that the adds of a wave, and its loads of b, are of 64 neighbouring words.
template <int TI>
__device__ __forceinline__ void flush_row(float *__restrict__ c, int64_t row, int C, int c0, float (&acc)[TI])
{
    float *dst = c + row * C + c0;
#pragma unroll
    for (int t = 0; t < TI; ++t) {
        if (c0 + 64 * t < C) unsafeAtomicAdd(dst + 64 * t, acc[t]);
        acc[t] = 0.0f;
    }
}

// Panels go to the XCDs as in csr_spmm_kernel.  With verdicts it runs only where they forbid the sum
// by rows, and then in no more workgroups than the chip holds: one per block of entries and panel cost 4 us to find nothing to do.
// NEAR: b spans less than 4 GiB; no lane reads past its row either way (those past the last column read that).
constexpr int FALLBACK_WORKGROUPS = 8 * kNumCU;
template <int TI, bool NEAR>
__global__ __launch_bounds__(NT) void coo_spmm_kernel(const int64_t *__restrict__ row,
                                                      const int64_t *__restrict__ col,
                                                      const float *__restrict__ val, int64_t nnz,
                                                      const float *__restrict__ b, int64_t ldb, uint32_t b_bytes,
                                                      float *__restrict__ c, int C, int chunk_blocks, int64_t total,
                                                      const uint32_t *__restrict__ verdicts)
{
    constexpr int EG = loads_of(1);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (verdicts && !not_by_rows(verdicts)) return;
    // fewer workgroups than blocks (a multiple of the XCDs): an XCD's share in turn, so that it works on panels of its own then too (4096 x
    // 4096 at 1 % with a full row x 4096 columns: 335 -> 240 us)
    const bool turns = total > gridDim.x;
    const int xcd = blockIdx.x % kNumXCD;
    const int64_t end = turns ? total * (xcd + 1) / kNumXCD : total, step = turns ? gridDim.x / kNumXCD : total;
    for (int64_t at = turns ? total * xcd / kNumXCD + blockIdx.x / kNumXCD : xcd_remap(blockIdx.x, gridDim.x); at < end; at += step) {
        const int panel = (int)(at / chunk_blocks);
        const int64_t e0 = ((at - (int64_t)panel * chunk_blocks) * (NT / 64) + wave) * COO_CHUNK;
        if (e0 >= nnz) continue;
        const int n = (int)((nnz - e0) < COO_CHUNK ? (nnz - e0) : COO_CHUNK);
        const int c0 = panel * 64 * TI + lane;
        uint32_t word[TI];
#pragma unroll
        for (int t = 0; t < TI; ++t) word[t] = c0 + 64 * t < C ? c0 + 64 * t : C - 1;
        const __amdgpu_buffer_rsrc_t near = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(b), 0, (int)b_bytes, 0x00020000);
        const uint32_t row_bytes = (uint32_t)ldb * 4u;
        auto b_word = [&](int64_t k, int t) -> float {
            if constexpr (NEAR) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(near, word[t] * 4, (uint32_t)k * row_bytes, 0));
            else return (b + k * ldb)[word[t]];
        };

        const_i64 *crow = (const_i64 *)row;
        const_i64 *ccol = (const_i64 *)col;
        const_f32 *cval = (const_f32 *)val;
        float acc[TI];
#pragma unroll
        for (int t = 0; t < TI; ++t) acc[t] = 0.0f;
        int64_t cur = crow[e0];
        for (int i = 0; i < n; i += EG) {
            // loads of up to EG entries first; entries past the end repeat the last one and are not added
            float xv[EG][TI];
            float wv[EG];
            int64_t rv[EG];
#pragma unroll
            for (int u = 0; u < EG; ++u) {
                const bool ok = i + u < n;
                const int64_t e = e0 + (ok ? i + u : n - 1), k = ccol[e];
#pragma unroll
                for (int t = 0; t < TI; ++t) xv[u][t] = b_word(k, t);
                wv[u] = cval[e];
                rv[u] = crow[e];
            }
#pragma unroll
            for (int u = 0; u < EG; ++u) {
                if (rv[u] != cur) {  // wave-uniform
                    flush_row<TI>(c, cur, C, c0, acc);
                    cur = rv[u];
                }
                if (i + u < n) {
#pragma unroll
                    for (int t = 0; t < TI; ++t) acc[t] = __builtin_fmaf(wv[u], xv[u][t], acc[t]);
                }
            }
        }
        flush_row<TI>(c, cur, C, c0, acc);
    }
}

// crow[r] = entries whose row is below r, for rows in ascending order, a lane per r by halving: the lanes of a wave look at the same lines
// until the last steps, and 2^13 waves are in flight (a wave per r that looks at 64 places a step, us: 4096 rows 4.0, 65536 rows 12 to 33, 2^20 rows
// 210 to 560; this: 4.0, 4 to 5, 12 to 64).  For rows in any other order it ends all the same, inside 0 .. nnz.
// verdicts: the first VERDICTS workgroups look instead whether the rows ascend (a tensor may be flagged as coalesced without
// being so) and none holds more than `longest` entries.
__global__ __launch_bounds__(NT) void row_offsets_kernel(const int64_t *__restrict__ row, int64_t nnz,
                                                         int64_t *__restrict__ crow, int64_t R,
                                                         uint32_t *__restrict__ verdicts, int64_t longest)
{
    const int checking = verdicts ? VERDICTS : 0;
    if ((int)blockIdx.x < checking) {
        bool bad = false;
#pragma unroll 4
        for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < nnz - 1; e += (int64_t)VERDICTS * NT) {
            bad |= row[e + 1] < row[e];
            const int64_t far = longest < nnz - e ? e + longest : nnz - 1;       // (loads without a condition: they are issued together)
            bad |= (row[far] == row[e]) & (far - e == longest);
        }
        const int any = __syncthreads_or(bad);
        if (threadIdx.x == 0) verdicts[blockIdx.x] = any ? 1u : 0u;
        return;
    }
    const int64_t r = (int64_t)((int)blockIdx.x - checking) * NT + threadIdx.x;
    if (r > R) return;
    int64_t lo = 0, count = nnz;          // the place is one of lo .. lo + count
    while (count > 0) {
        const int64_t half = count >> 1;
        const bool below = row[lo + half] < r;
        lo = below ? lo + half + 1 : lo;
        count = below ? count - half - 1 : half;
    }
    crow[r] = lo;
}

static int check_common(const float *b, int64_t ldb, float *c, int64_t R, int64_t K, int64_t C)
{
    if (R < 0 || K < 0 || C < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    if (R > INT32_MAX / 2 || K > INT32_MAX / 2 || C > INT32_MAX / 2)
        return fail(MAM_ERR_UNSUPPORTED, "a dimension exceeds 2^30");
    if (R == 0 || C == 0) return MAM_OK;
    if (!c || (K > 0 && !b)) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    if (ldb < C) return fail(MAM_ERR_INVALID_ARGUMENT, "ldb smaller than the number of columns");
    return MAM_OK;
}

// Scatter of a sparse matrix into a cleared dense one (repeated coordinates add up).  CSR: a wave per row.
// These kernels WRITE at the coordinates they are given, so an entry whose column (or row) lies outside the
// matrix is skipped: nothing is ever written outside `dense`.
__global__ __launch_bounds__(NT) void csr_to_dense_kernel(const int64_t *__restrict__ crow, const int64_t *__restrict__ col,
                                                          const float *__restrict__ val, float *__restrict__ dense,
                                                          int64_t ld, int R, int K)
{
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    if (r >= R) return;
    const int64_t beg = crow[r], end = crow[r + 1];
    float *row = dense + (int64_t)r * ld;
    for (int64_t e = beg + lane; e < end; e += 64) {
        const int64_t cc = col[e];
        if ((uint64_t)cc < (uint64_t)K)
            __hip_atomic_fetch_add(row + cc, val[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

__global__ __launch_bounds__(256) void coo_to_dense_kernel(const int64_t *__restrict__ row, const int64_t *__restrict__ col,
                                                           const float *__restrict__ val, int64_t nnz,
                                                           float *__restrict__ dense, int64_t ld, int R, int K)
{
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nnz; e += stride) {
        const int64_t rr = row[e], cc = col[e];
        if ((uint64_t)rr < (uint64_t)R && (uint64_t)cc < (uint64_t)K)
            __hip_atomic_fetch_add(dense + rr * ld + cc, val[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

static int check_dense(const float *dense, int64_t ld, int64_t R, int64_t K)
{
    if (R < 0 || K < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    if (R > INT32_MAX / 2 || K > INT32_MAX / 2) return fail(MAM_ERR_UNSUPPORTED, "a dimension exceeds 2^30");
    if (R == 0 || K == 0) return MAM_OK;
    if (!dense) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    if (ld < K) return fail(MAM_ERR_INVALID_ARGUMENT, "ld smaller than the number of columns");
    return MAM_OK;
}

// rows of `dense` may be strided: cleared row by row when they are
static int clear_dense(float *dense, int64_t ld, int64_t R, int64_t K, hipStream_t st)
{
    if (ld == K) return fill_zero(dense, R * K, st);
    for (int64_t r = 0; r < R; ++r) {
        const int rc = fill_zero(dense + r * ld, K, st);
        if (rc != MAM_OK) return rc;
    }
    return MAM_OK;
}

static bool wide(const float *b, int64_t ldb, const float *c, int64_t C)
{
    return C % 4 == 0 && ldb % 4 == 0 && (uintptr_t)b % 16 == 0 && (uintptr_t)c % 16 == 0;
}

// Launches of csr_spmm_kernel and coo_spmm_kernel (arguments checked, nothing empty).
static int launch_csr(const int64_t *crow, const int64_t *col, const float *val, const float *b, int64_t ldb, float *c, int64_t R,
                      int64_t K, int64_t C, const uint32_t *verdicts, hipStream_t st)
{
    const int64_t b_bytes = K > 0 ? ((K - 1) * ldb + C) * 4 : 0;
    const bool near = b_bytes < ((int64_t)1 << 32), wide = spmm::wide(b, ldb, c, C);
    const int per = !near ? 1 : C <= 64 ? 4 : C <= 128 ? 2 : 1;          // entries per load
    const int64_t panels = ceil_div(C, near || wide ? 256 / per : 64);
    // panels of one width, whole lines: a narrow last one would leave the XCDs that work on it half idle (4096 x 4096 at 5 % x 260
    // columns as 256 + 4: 64 us, 160 + 100: 54 us; 1 % x 300 columns 18 and 14 us)
    const int width = (int)(ceil_div(ceil_div(C, panels), 32) * 32);
    const int64_t row_blocks = ceil_div(R, NT / 64);
    if (panels > 65535) return fail(MAM_ERR_UNSUPPORTED, "too many columns for the SpMM grid");
    const bool linear = by_xcd(panels, row_blocks, K);
    auto launch = [&](auto kernel) {
        const dim3 grid = linear ? dim3((unsigned)(panels * row_blocks)) : dim3((unsigned)row_blocks, (unsigned)panels);
        hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, st, crow, col, val, b, ldb, (uint32_t)b_bytes, c, (int)R, (int)C, (int)row_blocks,
                           linear ? (int)panels : 0, width, verdicts);
    };
    if (per == 4) launch(csr_spmm_kernel<4, true, 4>);
    else if (per == 2) launch(csr_spmm_kernel<4, true, 2>);
    else if (near) launch(csr_spmm_kernel<4, true, 1>);
    else if (wide) launch(csr_spmm_kernel<4, false, 1>);
    else launch(csr_spmm_kernel<1, false, 1>);
    return check_launch("csr_spmm_kernel");
}

static int launch_coo(const int64_t *row, const int64_t *col, const float *val, int64_t nnz, const float *b, int64_t ldb, float *c,
                      int64_t K, int64_t C, const uint32_t *verdicts, hipStream_t st)
{
    const int64_t gx = ceil_div(nnz, (int64_t)COO_CHUNK * (NT / 64));
    if (gx > INT32_MAX) return fail(MAM_ERR_UNSUPPORTED, "too many entries for the SpMM grid");
    const int64_t b_bytes = K > 0 ? ((K - 1) * ldb + C) * 4 : 0;
    const bool near = b_bytes < ((int64_t)1 << 32);
    // columns per lane: fewer where waves are few, each of which adds up to 64 rows one after the other (4 / 2 / 1, us: 194 entries in any order x 4041
    // columns, 64 waves of four, 26 / 20 / 17; 10207 ascending x 723, 480 waves, 15 / 13 / 14; 103372 ascending x 197, 1616 waves, 15 / 18 / 27)
    const int64_t fours = gx * ceil_div(C, 256);
    const int per_lane = C <= 64 || fours < kNumCU ? 1 : C <= 128 || fours < 4 * kNumCU ? 2 : 4;
    const int64_t panels = ceil_div(C, 64 * per_lane);
    if (panels > 65535) return fail(MAM_ERR_UNSUPPORTED, "too many columns for the SpMM grid");
    const int64_t total = panels * gx, most = verdicts ? FALLBACK_WORKGROUPS : UINT32_MAX / NT / kNumXCD * kNumXCD;      // (2^32 threads in a launch)
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(total < most ? total : most)), dim3(NT), 0, st, row, col, val, nnz, b, ldb,
                           (uint32_t)b_bytes, c, (int)C, (int)gx, total, verdicts);
    };
    if (per_lane == 1) near ? launch(coo_spmm_kernel<1, true>) : launch(coo_spmm_kernel<1, false>);
    else if (per_lane == 2) near ? launch(coo_spmm_kernel<2, true>) : launch(coo_spmm_kernel<2, false>);
    else near ? launch(coo_spmm_kernel<4, true>) : launch(coo_spmm_kernel<4, false>);
    return check_launch("coo_spmm_kernel");
}

// Entries of a COO operand's row that its wave may take one after the other, 0.05 us each (8 in 0.45 us, narrow c: 16 in 0.85), so that
// no row alone takes longer than the COO kernel, 12 us and at least 0.2 us per 2^20 entries times columns, takes for everything.
// (One row full, us by rows / by entries after the look: 4096 x 4096 at 10 % x 1024 columns 393 / 366 and 40, by rows; at 1 % x 4096 301 / 240,
// 64 x 4096 at 1 % x 4096 245 / 23, 4096 x 32768 with 8 entries in the others x 1024 1990 / 59, 300 x 1000 at 1 % x 260 38 / 16.)
static int64_t longest_row(int64_t nnz, int64_t C) { return 256 + (int64_t)((double)nnz * (double)C / (1 << 18)); }

static int launch_row_offsets(const int64_t *row, int64_t nnz, int64_t *crow, int64_t R, uint32_t *verdicts, int64_t longest,
                              hipStream_t st)
{
    hipLaunchKernelGGL(row_offsets_kernel, dim3((unsigned)ceil_div(R + 1, NT) + (verdicts ? VERDICTS : 0)), dim3(NT), 0, st, row, nnz, crow, R, verdicts, longest);
    return check_launch("row_offsets_kernel");
}

}  // namespace spmm
}  // namespace mam

extern "C" int mam_csr_spmm(const int64_t *crow, const int64_t *col, const float *val, const float *b,
                            int64_t ldb, float *c, int64_t R, int64_t K, int64_t C, void *stream)
{
    using namespace mam;
    int rc = spmm::check_common(b, ldb, c, R, K, C);
    if (rc != MAM_OK || R == 0 || C == 0) return rc;
    if (!crow) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    return spmm::launch_csr(crow, col, val, b, ldb, c, R, K, C, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int mam_coo_spmm(const int64_t *row, const int64_t *col, const float *val, int64_t nnz,
                            const float *b, int64_t ldb, float *c, int64_t R, int64_t K, int64_t C,
                            void *stream)
{
    using namespace mam;
    if (nnz < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    int rc = spmm::check_common(b, ldb, c, R, K, C);
    if (rc != MAM_OK || R == 0 || C == 0) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    rc = fill_zero(c, R * C, st);
    if (rc != MAM_OK || nnz == 0) return rc;
    if (!row || !col || !val) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    return spmm::launch_coo(row, col, val, nnz, b, ldb, c, K, C, nullptr, st);
}

extern "C" int mam_coo_row_offsets(const int64_t *row, int64_t nnz, int64_t *crow, int64_t R, void *stream)
{
    using namespace mam;
    if (nnz < 0 || R < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    if (R > INT32_MAX / 2) return fail(MAM_ERR_UNSUPPORTED, "a dimension exceeds 2^30");
    if (!crow || (nnz > 0 && !row)) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    return spmm::launch_row_offsets(row, nnz, crow, R, nullptr, 0, static_cast<hipStream_t>(stream));
}

extern "C" size_t mam_coo_spmm_by_rows_workspace(int64_t R)
{
    return R > 0 ? mam::spmm::VERDICTS * sizeof(uint32_t) + (size_t)(R + 1) * sizeof(int64_t) : 0;
}

extern "C" int mam_coo_spmm_by_rows(const int64_t *row, const int64_t *col, const float *val, int64_t nnz, const float *b, int64_t ldb,
                                    float *c, int64_t R, int64_t K, int64_t C, void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace mam;
    if (nnz < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    int rc = spmm::check_common(b, ldb, c, R, K, C);
    if (rc != MAM_OK || R == 0 || C == 0) return rc;
    if (nnz > 0 && (!row || !col || !val)) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t need = mam_coo_spmm_by_rows_workspace(R);
    if (!workspace || workspace_bytes < need || (uintptr_t)workspace % 16 != 0)
        return fail(MAM_ERR_WORKSPACE, "the sum by rows needs %zu workspace bytes, 16-byte aligned, got %zu", need,
                    workspace ? workspace_bytes : (size_t)0);
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint32_t *verdicts = static_cast<uint32_t *>(workspace);
    int64_t *crow = reinterpret_cast<int64_t *>(verdicts + spmm::VERDICTS);
    rc = spmm::launch_row_offsets(row, nnz, crow, R, verdicts, spmm::longest_row(nnz, C), st);
    if (rc == MAM_OK) rc = spmm::launch_csr(crow, col, val, b, ldb, c, R, K, C, verdicts, st);
    if (rc == MAM_OK && nnz > 0) rc = spmm::launch_coo(row, col, val, nnz, b, ldb, c, K, C, verdicts, st);
    return rc;
}

extern "C" int mam_csr_to_dense(const int64_t *crow, const int64_t *col, const float *val, float *dense, int64_t ld,
                                int64_t R, int64_t K, void *stream)
{
    using namespace mam;
    int rc = spmm::check_dense(dense, ld, R, K);
    if (rc != MAM_OK || R == 0 || K == 0) return rc;
    if (!crow) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    rc = spmm::clear_dense(dense, ld, R, K, st);
    if (rc != MAM_OK) return rc;
    hipLaunchKernelGGL(spmm::csr_to_dense_kernel, dim3((unsigned)ceil_div(R, spmm::NT / 64)), dim3(spmm::NT), 0, st, crow,
                       col, val, dense, ld, (int)R, (int)K);
    return check_launch("csr_to_dense_kernel");
}

extern "C" int mam_coo_to_dense(const int64_t *row, const int64_t *col, const float *val, int64_t nnz, float *dense,
                                int64_t ld, int64_t R, int64_t K, void *stream)
{
    using namespace mam;
    if (nnz < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    int rc = spmm::check_dense(dense, ld, R, K);
    if (rc != MAM_OK || R == 0 || K == 0) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    rc = spmm::clear_dense(dense, ld, R, K, st);
    if (rc != MAM_OK || nnz == 0) return rc;
    if (!row || !col || !val) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    int64_t blocks = ceil_div(nnz, 256);
    if (blocks > 64 * kNumCU) blocks = 64 * kNumCU;
    hipLaunchKernelGGL(spmm::coo_to_dense_kernel, dim3((unsigned)blocks), dim3(256), 0, st, row, col, val, nnz, dense, ld,
                       (int)R, (int)K);
    return check_launch("coo_to_dense_kernel");
}
