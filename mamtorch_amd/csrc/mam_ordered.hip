// MAM forward by magnitude-ordered lists: most products of a MAM neuron are never formed.
//
// max_k(x_k w_k) is attained where |x_k| or |w_k| is large.  Take the entries of a row of x by falling |x_k|;
// once `best` is the largest product seen and U bounds every |x_k| not yet seen, fl(|x_k w_k|) <= fl(U * max|w|)
// for all of those, and U * max|w| < best ends the search: nothing unseen can reach, or tie with, the maximum
// (the same for the minimum with -best).  For x ~ N(0,1) and W ~ U(-a,a) 0.7 % of 4096 products decide an
// output on average and 2.1 % decide 99 % of them; with normal weights 10 %.  The roles may be swapped: lists of
// the rows of w, bounded by max|x|.  Results are those of the scan over every k, bit for bit.
//
// With normal weights as well the largest |w| is far out and one list gets long (10 % on average at K = 4096).  Then
// the leading few percent of the OTHER operand's entries are taken first, for every output; what is left of that
// operand is bounded by its next entry instead of by its largest, and the two short lists together replace the long
// one (an entry in both is met twice, which changes nothing).  K = 768, both normal: 36 % -> 13 % of the products for
// a wave's slowest output, K = 4096: 23 % -> 5.5 %.
//
// Four launches, all decisions on the device:
//   sample_kernel  64 outputs computed in full: how long would their lists have to be, on either side and with any
//                  of LEADS leading shares of the other side?
//   build_kernel   first the decision (two-sided searches and many rows: decide_kernel): the cheapest of these, or none, and then
//                  the dense kernels run instead: where products do not fall off that way (constant magnitudes, products of one
//                  sign), or where the search of so few rows takes longer all the same.
//                  A workgroup per listed row: counting sort of the leading entries by magnitude (512 buckets over 4 octaves),
//                  written chunk by chunk with the bound U of what follows each chunk; and, for a leading share, the
//                  searched operand transposed.
//   forward_kernel the search itself (below).
//   dense kernels  exit at once unless the decision was "none".
//
// Measured against the dense tilings (forward call, hand-over arrays written).  Uniform weights or inputs, one-sided:
// 207 -> 60 to 67 us at 256 x 4096 x 4096, 1.70 -> 0.49 ms and 1.48 -> 0.24 ms for 12608 x 768 -> 3072 -> 768, 10.2 -> 0.72 ms
// (values only) and 3.13 -> 0.36 ms at 16384 x 4096 -> 4096 / 1024.  Normal weights and inputs, two-sided: 1.70 -> 1.36 ms
// at 12608 x 768 -> 3072, 3.12 -> 0.92 ms at 16384 x 4096 -> 1024, 0.84 -> 0.40 ms at 4096 x 2048 x 2048.
#include "mam_ordered.h"

#include <math.h>

namespace mam {
namespace ordered {

constexpr int BUCKETS = 512;          // 128 per octave below the row's largest magnitude
constexpr int BUCKET_SHIFT = 16;
constexpr int BUILD_NT = 256;         // threads of the build, per listed row
constexpr int BUILD_MAX_K = 40 * BUILD_NT;
constexpr int NT = 1024;              // threads of the forward
constexpr int MAX_TILE_BYTES = 152 * 1024;
// N * K * M from which two-sided searches are considered.  They cost two launches and a longer sampling, 7 to 13 us, where they are not
// taken (256 x 4096 -> 4096, uniform weights, 2^32 products: 60 us without, 67 us with them; 64 x 4096 -> 16384, normal weights, by the
// dense tilings: 242 and 255 us): up to 2^33 products 3 to 11 % of the call.  Where they are taken they win earlier (256 x 4096 -> 4096,
// normal weights: 225 us without, 126 us with them; 1024 x 2048 x 2048: 235 and 122).
constexpr int64_t MIN_TWO_SIDED = 1ll << 33;
constexpr int LEAD_CAP = 96;          // leading entries kept per tile row (LDS)
// N * K * M from which a call takes the lists.  Uniform on one side, they win from 2^30 products on (lists / dense, with indices:
// 128 x 2048 -> 4096 46 / 68 us, 128 x 4096 -> 4096 62 / 116), but only the device finds out what the data is, and a call that it
// hands to the dense tilings has paid for sampling and idle launches: 8 to 11 us, 4 to 5 % of the 214 to 240 us that 2^32
// products take there, twice that share at 2^31.
constexpr int64_t MIN_PRODUCTS = 1ll << 32;
constexpr uint32_t INF_BITS = 0x7f800000u;

constexpr int MAX_UNDECIDED = 4096;
constexpr int CHUNK = 8;         // list entries between two tests of the bound
constexpr int BUILD_MAX_CHUNKS = (BUILD_MAX_K / 4 + 64) / CHUNK + 1;
constexpr int SAMPLES = 64;      // sampled outputs of a call, one per lane of a deciding wave
constexpr int LEADS = 9;         // leading shares tried
constexpr int OPTIONS = 2 * LEADS;

// Microseconds of the dense kernels and of the lists of a call, from its sizes alone; launches that come either way are
// left out.  What a search costs per product is not all: its workgroups load their tiles (14.5 us for 128 KiB), a round of 16 blocks
// of rows costs 4 to 6 us beside its products, a round of fewer waves hardly less, and the lists themselves 2 to 10 ns a row.
// Calls of few rows on either side lose there what the search saves (normal x normal, lists / dense: 64 x 4096 -> 16384 357 / 234 us,
// 65536 x 1024 -> 64 822 / 339, 40 x 8000 -> 16384 1499 / 464; 256 x 4096 -> 4096 126 / 214).  Constants fitted to 180 timed
// calls (K 256 .. 8000, N and M 40 .. 65536), most of which they gave within 20 %; the search has become 10 to 25 % faster since, so
// that calls near the border stay with the dense kernels a little longer than they need to.
struct Times {
    struct Side { float fixed, per_entry, rounds, round; };      // of a search of this operand's rows
    float dense, product, led;
    Side one_sided[2], two_sided[2];                             // rows of x are searched, rows of w
    __device__ __forceinline__ float lists_us(int side, int lead, int length, float searched) const
    {
        const Side &s = side == SIDE_X ? (lead > 0 ? two_sided[0] : one_sided[0]) : lead > 0 ? two_sided[1] : one_sided[1];
        return s.fixed + s.per_entry * (float)length + s.rounds * (s.round + product * searched + led * (float)lead);
    }
};

struct Params {
    Call call;
    Times times;
    int *samples;             // [OPTIONS][SAMPLES]: entries of the searched list a sampled output needs
    Decision *decision;
    uint4 *lists_x, *lists_w; // [entry pair][row]: (value, key, value, key)
    float *bound_x, *bound_w; // [chunk][row]: bound on the magnitudes from this chunk on
    float *turned;            // [K][turned_ld]: the searched operand transposed (two-sided searches)
    int turned_ld;            // 0: no room for it, one-sided searches only
    int cap;                  // entries a list can hold (a multiple of CHUNK)
    int pad_x, pad_w;         // rows of the list arrays
    int cus;                  // compute units
    int decided;              // by decide_kernel; otherwise by every workgroup of build_kernel
    int any_size;             // lists wherever they save products, whatever the rest of them costs (option LISTS)
};

// Leading shares in 1/1024 of K.
__device__ const int kLeadShare[LEADS] = {0, 8, 16, 24, 32, 48, 64, 92, 128};
__device__ __forceinline__ int lead_entries(int option, int K)
{
    const int lead = (int)((int64_t)kLeadShare[option % LEADS] * K / 1024 / CHUNK) * CHUNK;
    return lead < LEAD_CAP ? lead : LEAD_CAP;
}

// A list entry's key: (65535 - k) in the upper half, so that the lower k is the larger key, and its place in the
// list + 1 in the lower half (0: not from a list), from which the listed value is found again.
__host__ __device__ __forceinline__ uint32_t key(uint32_t k, uint32_t place) { return ((65535u - k) << 16) | place; }
__device__ __forceinline__ int index_in(uint32_t key) { return (int)(65535u - (key >> 16)); }
__device__ __forceinline__ int place_in(uint32_t key) { return (int)(key & 65535u) - 1; }

// rows of one operand: element (row, k)
struct Rows {
    const float *p;
    int64_t row_stride, k_stride;
    int rows;
    __device__ __forceinline__ const float *at(int64_t row, int64_t k) const { return p + row * row_stride + k * k_stride; }
};
__device__ __forceinline__ Rows x_rows(const Call &c) { return {c.x, c.ldx, 1, (int)c.N}; }
__device__ __forceinline__ Rows w_rows(const Call &c)
{
    return {c.w, c.w_layout == MAM_W_MK ? c.ldw : 1, c.w_layout == MAM_W_MK ? 1 : c.ldw, (int)c.M};
}

__device__ __forceinline__ int wave_sum(int v)
{
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s);
    return v;
}
__device__ __forceinline__ int wave_max(int v)
{
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const int o = __shfl_xor(v, s);
        v = o > v ? o : v;
    }
    return v;
}

// Exclusive prefix over hist[BUCKETS] in LDS, in place, by BUILD_NT threads; the number of buckets that start below
// `len` is returned.  part: one word per wave.
__device__ __forceinline__ uint32_t prefix_buckets(uint32_t *hist, uint32_t *part, uint32_t len)
{
    constexpr int BPT = BUCKETS / BUILD_NT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t own[BPT], sum = 0;
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        own[j] = hist[tid * BPT + j];
        sum += own[j];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const uint32_t o = __shfl_up(incl, s);
        if (lane >= s) incl += o;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
#pragma unroll
    for (int i = 0; i < BUILD_NT / 64; ++i) run += i < wave ? part[i] : 0u;
    int open = 0;
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        hist[tid * BPT + j] = run;
        open += run < len;
        run += own[j];
    }
    open = wave_sum(open);
    __syncthreads();
    if (lane == 0) part[wave] = (uint32_t)open;
    __syncthreads();
    open = 0;
#pragma unroll
    for (int i = 0; i < BUILD_NT / 64; ++i) open += (int)part[i];
    return (uint32_t)open;
}

// ---- sampling ----------------------------------------------------------------------------------------------
// R elements per thread of either row, read once: what counts here is how often a workgroup waits for memory.
template <int R>
__global__ __launch_bounds__(BUILD_NT) void sample_kernel(const Params p)
{
    constexpr int WAVES = BUILD_NT / 64;
    __shared__ uint32_t hist[2][BUCKETS];
    __shared__ uint32_t part[WAVES];
    __shared__ float red[WAVES][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const Call &c = p.call;
    const int K = (int)c.K;
    const uint32_t i = blockIdx.x;
    const int n = (int)((uint64_t)(i * 2 + 1) * (uint64_t)c.N / (2 * SAMPLES));
    const int m = (int)((((uint64_t)(i * 2654435769u)) * (uint64_t)c.M) >> 32);
    const Rows xr = x_rows(c), wr = w_rows(c);
    float hi = -__builtin_inff(), lo = __builtin_inff(), ax = 0.0f, aw = 0.0f;
    float xv[R], wv[R];
#pragma unroll
    for (int t = 0; t < R; ++t) {           // (past the end the last element again: it changes no extreme, and is not counted)
        const int k = t * BUILD_NT + tid < K ? t * BUILD_NT + tid : K - 1;
        xv[t] = *xr.at(n, k);
        wv[t] = *wr.at(m, k);
    }
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const float q = xv[t] * wv[t];
        hi = __builtin_fmaxf(hi, q);
        lo = __builtin_fminf(lo, q);
        ax = __builtin_fmaxf(ax, __builtin_fabsf(xv[t]));
        aw = __builtin_fmaxf(aw, __builtin_fabsf(wv[t]));
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        hi = __builtin_fmaxf(hi, __shfl_xor(hi, s));
        lo = __builtin_fminf(lo, __shfl_xor(lo, s));
        ax = __builtin_fmaxf(ax, __shfl_xor(ax, s));
        aw = __builtin_fmaxf(aw, __shfl_xor(aw, s));
    }
    if (lane == 0) { red[wave][0] = hi; red[wave][1] = lo; red[wave][2] = ax; red[wave][3] = aw; }
    for (int j = tid; j < 2 * BUCKETS; j += BUILD_NT) (&hist[0][0])[j] = 0;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
        hi = __builtin_fmaxf(hi, red[v][0]);
        lo = __builtin_fminf(lo, red[v][1]);
        ax = __builtin_fmaxf(ax, red[v][2]);
        aw = __builtin_fmaxf(aw, red[v][3]);
    }
    const float reach = __builtin_fminf(hi, -lo);      // a bound below this ends both searches
    if (p.turned_ld == 0) {
        // one-sided searches only: options 0 and LEADS
        __shared__ int counts[WAVES][2];
        int nx = 0, nw = 0;
#pragma unroll
        for (int t = 0; t < R; ++t)
            if (t * BUILD_NT + tid < K) {
                nx += !(__builtin_fabsf(xv[t]) * aw < reach);
                nw += !(__builtin_fabsf(wv[t]) * ax < reach);
            }
        nx = wave_sum(nx);
        nw = wave_sum(nw);
        if (lane == 0) { counts[wave][0] = nx; counts[wave][1] = nw; }
        __syncthreads();
        if (tid < 2) {
            int sum = 0;
            for (int v = 0; v < WAVES; ++v) sum += counts[v][tid];
            p.samples[tid * LEADS * SAMPLES + blockIdx.x] = sum;
        }
        return;
    }
    const uint32_t top_x = __float_as_uint(ax), top_w = __float_as_uint(aw);
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const uint32_t bx = (top_x - (__float_as_uint(xv[t]) & 0x7fffffffu)) >> BUCKET_SHIFT;
        const uint32_t bw = (top_w - (__float_as_uint(wv[t]) & 0x7fffffffu)) >> BUCKET_SHIFT;
        const bool there = t * BUILD_NT + tid < K;
        if (there && bx < (uint32_t)BUCKETS) atomicAdd(&hist[0][bx], 1u);
        if (there && bw < (uint32_t)BUCKETS) atomicAdd(&hist[1][bw], 1u);
    }
    __syncthreads();
    prefix_buckets(hist[0], part, 0);
    __syncthreads();
    prefix_buckets(hist[1], part, 0);
    if (tid >= OPTIONS) return;
    // an option: LEADS shares of w ahead of a search of x, then LEADS shares of x ahead of a search of w
    const bool search_x = tid < LEADS;
    const uint32_t *led = hist[search_x ? 1 : 0], *searched = hist[search_x ? 0 : 1];
    const uint32_t top_led = search_x ? top_w : top_x, top_searched = search_x ? top_x : top_w;
    // what is left of the led operand: at most the upper edge of the last bucket that starts inside the share
    const uint32_t lead = (uint32_t)lead_entries(tid, K);
    int b = 0;
    for (int step = BUCKETS / 2; step > 0; step >>= 1)
        if (led[b + step] <= lead) b += step;
    const float left = __uint_as_float(top_led - ((uint32_t)b << BUCKET_SHIFT));
    int need = K;
    if (reach > 0.0f && left > 0.0f) {
        const uint32_t from = __float_as_uint(reach / left);
        if (from > top_searched) {
            need = 0;
        } else {
            const uint32_t d = ((top_searched - from) >> BUCKET_SHIFT) + 1;      // everything down to this bucket
            if (d < (uint32_t)BUCKETS) need = (int)searched[d];
        }
    }
    p.samples[tid * SAMPLES + blockIdx.x] = need;
}

// The COUNT largest of the 64 lanes' values (not negative), in falling order.  Every workgroup of build_kernel waits for this:
// lane shifts instead of trips through the LDS.
template <int COUNT>
__device__ __forceinline__ void largest(int v, int (&top)[COUNT])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
        int m = v;
        auto fold = [&](int other) { m = other > m ? other : m; };
        fold(__builtin_amdgcn_update_dpp(m, m, 0x111, 0xf, 0xf, false));        // row_shr 1, 2, 4, 8
        fold(__builtin_amdgcn_update_dpp(m, m, 0x112, 0xf, 0xf, false));
        fold(__builtin_amdgcn_update_dpp(m, m, 0x114, 0xf, 0xf, false));
        fold(__builtin_amdgcn_update_dpp(m, m, 0x118, 0xf, 0xf, false));
        fold(__builtin_amdgcn_update_dpp(m, m, 0x142, 0xa, 0xf, false));        // last lane of a row of 16 to the next row
        fold(__builtin_amdgcn_update_dpp(m, m, 0x143, 0xc, 0xf, false));        // of the lower half to the upper half
        top[i] = __builtin_amdgcn_readlane(m, 63);
        if (lane == (int)__builtin_ctzll(__ballot(v == top[i]))) v = -1;
    }
}

// rows of the tile operand per workgroup: as many as fit the LDS as whole rows (0: not even 4)
__host__ __device__ __forceinline__ int tile_rows(int64_t K)
{
    for (int tb = 32; tb >= 4; tb /= 2)
        if (K * tb * 4 <= MAX_TILE_BYTES) return tb;
    return 0;
}
constexpr int TWO_SIDED_ROWS = 8;     // of a two-sided search

// Row ranges per tile: three rounds of workgroups over the chip, but at least one block of rows per wave.
__host__ __device__ __forceinline__ int splits_of(int tb, int searched, int tiles, int cus)
{
    const int blocks = (searched + 256 / tb - 1) / (256 / tb);
    const int s = (3 * cus + tiles - 1) / tiles, most = (blocks + NT / 64 - 1) / (NT / 64);
    return s < most ? s : most;
}

// The cheapest option, by all waves of a workgroup.  In units of one product of a dense kernel per output (12608 x 768 x
// 3072: 2.25 us): a searched product costs 3.5, a leading one 6, a wave's slowest output needs ~1.3 times what 95 % of
// the samples need; the launches, outputs and lists cost 0.15 K, a leading share passes over both operands.  Outputs that no list
// finishes (a sampled need beyond the longest list) cost SCAN a product over the whole row, and their waves a whole list first; four
// such samples of 64 need too much by the rule above.  The dense kernels cost K.
constexpr float SCAN = 5.0f;
struct Weighed { float cost, searched, scans; int length; };     // of an option; searched: entries; scans: share of outputs no list finishes
template <int WAVES>
__device__ __forceinline__ Decision decide(const Params &p, Weighed (&weighed)[OPTIONS])
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float K = (float)p.call.K;
    const int step = p.turned_ld > 0 ? 1 : LEADS;         // one-sided searches only: options 0 and LEADS
    for (int o = wave * step; o < OPTIONS; o += WAVES * step) {
        const bool search_x = o < LEADS, two_sided = o % LEADS != 0;
        const int lead = lead_entries(o, (int)p.call.K);
        // the rows of a (K, M) weight are columns in memory: they are not listed, and there is no two-sided search
        const bool possible = (!two_sided || lead > 0) && (p.call.w_layout == MAM_W_MK || search_x);
        const int v = p.samples[o * SAMPLES + lane];
        const float tiled = (float)(search_x ? p.call.M : p.call.N), listed = (float)(search_x ? p.call.N : p.call.M);
        // entries written per list: twice the longest sampled need and 64 more, so that hardly any of the outputs that
        // are finished one by one need more than their list; needs that no list meets do not count
        const int beyond = __popcll(__ballot(v > p.cap));
        int top[5];
        largest<5>(v, top);
        const int second = beyond == 0 ? top[1] : beyond == 1 ? top[2] : beyond == 2 ? top[3] : top[4];
        const int want = (second * 2 + 64 + CHUNK - 1) / CHUNK * CHUNK;
        const int length = want < p.cap ? want : p.cap;
        float searched = 1.3f * (float)top[3];
        if (beyond > 0 && searched < (float)length) searched = (float)length;
        const float scans = (float)beyond / SAMPLES;
        float cost = 0.15f * K + 3.5f * searched + SCAN * K * scans;
        if (two_sided) cost += 6.0f * (float)lead + K * (36.0f / tiled + 18.0f / listed);
        if (lane == 0) weighed[o] = {possible ? cost : 1e30f, searched, scans, length};
    }
    __syncthreads();
    int best = 0;
    for (int o = step; o < OPTIONS; o += step)
        if (weighed[o].cost < weighed[best].cost) best = o;
    Decision d;
    d.side = best < LEADS ? SIDE_X : SIDE_W;
    d.lead = lead_entries(best, (int)p.call.K);
    d.length = weighed[best].length;
    const float us = p.times.lists_us(d.side, d.lead, d.length, weighed[best].searched) + SCAN * weighed[best].scans * p.times.dense;
    if (!(weighed[best].cost < 0.95f * K) || !(p.any_size || us < p.times.dense)) d.side = SIDE_NONE;
    d.pad = 0;
    return d;
}

// Two-sided searches have 18 options: decided once, in a launch of its own (6 us).  The two one-sided ones are decided by
// every workgroup of build_kernel, up to MAX_UNDECIDED of them (build_kernel alone, where none is chosen: 3 us more with 4096, 51 us
// with 16384, 87 us with 65536).
__global__ __launch_bounds__(64 * LEADS) void decide_kernel(const Params p)
{
    __shared__ Weighed weighed[OPTIONS];
    const Decision d = decide<LEADS>(p, weighed);
    if (threadIdx.x == 0) *p.decision = d;
}

// ---- lists -------------------------------------------------------------------------------------------------
// 64 x 64 of `rows` transposed into dst[k][ld] through LDS.
__device__ __forceinline__ void turn_tile(const Rows &rows, int K, float *dst, int ld, int r0, int k0, float (*t)[65])
{
    const int lo = threadIdx.x & 63, hi = threadIdx.x >> 6;
#pragma unroll 8
    for (int i = 0; i < 64; i += BUILD_NT / 64) {
        const int r = r0 + i + hi, k = k0 + lo;
        t[i + hi][lo] = r < rows.rows && k < K ? *rows.at(r, k) : 0.0f;
    }
    __syncthreads();
#pragma unroll 8
    for (int i = 0; i < 64; i += BUILD_NT / 64) {
        const int k = k0 + i + hi, r = r0 + lo;
        if (k < K && r < rows.rows) dst[(int64_t)k * ld + r] = t[lo][i + hi];
    }
}

// The list of one row by a workgroup, R elements per thread in registers.  `place`: entries carry their place.
template <int R>
__device__ __forceinline__ void build_row(const Rows &rows, int row, int K, int len, bool place, uint4 *lists, float *bound, int pad,
                                          uint4 *lds, uint32_t *hist, uint32_t *part, uint32_t *part2, uint32_t *chunk_top)
{
    constexpr int WAVES = BUILD_NT / 64;
    uint2 *items = reinterpret_cast<uint2 *>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunks = len / CHUNK;
    const float *src = rows.at(row, 0);
    float v[R];
#pragma unroll
    for (int t = 0; t < R; ++t) v[t] = t * BUILD_NT + tid < K ? (src + t * BUILD_NT)[(uint32_t)tid] : 0.0f;
#pragma unroll
    for (int j = 0; j < BUCKETS / BUILD_NT; ++j) hist[j * BUILD_NT + tid] = 0;
    for (int j = tid; j < len; j += BUILD_NT) items[j] = make_uint2(0u, key(0, 0));
    uint32_t top = 0;
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const uint32_t bits = __float_as_uint(v[t]) & 0x7fffffffu;
        top = bits > top ? bits : top;
    }
    top = (uint32_t)wave_max((int)top);
    if (lane == 0) part[wave] = top;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WAVES; ++i) top = part[i] > top ? part[i] : top;
    // entries by bucket; what lies below the last bucket is never listed (nor are the clamped k beyond the row:
    // their value is zero, and a zero is listed only in an all-zero row, whose list nobody reads)
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const uint32_t b = (top - (__float_as_uint(v[t]) & 0x7fffffffu)) >> BUCKET_SHIFT;
        if (b < (uint32_t)BUCKETS && t * BUILD_NT + tid < K) atomicAdd(&hist[b], 1u);
    }
    __syncthreads();
    const uint32_t open = prefix_buckets(hist, part2, (uint32_t)len);     // buckets that start inside the list
    uint32_t rest = 0;            // largest magnitude that is not listed
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const uint32_t bits = __float_as_uint(v[t]) & 0x7fffffffu;
        const uint32_t b = (top - bits) >> BUCKET_SHIFT;
        const int k = t * BUILD_NT + tid;
        bool listed = false;
        if (b < open && k < K) {
            const uint32_t at = atomicAdd(&hist[b], 1u);
            if (at < (uint32_t)len) {
                items[at] = make_uint2(__float_as_uint(v[t]), key((uint32_t)k, place ? at + 1 : 0));
                listed = true;
            }
        }
        if (!listed) rest = bits > rest ? bits : rest;
    }
    rest = (uint32_t)wave_max((int)rest);
    if (lane == 0) part[wave] = rest;
    __syncthreads();
    for (int c = tid; c < chunks; c += BUILD_NT) {
        uint32_t t = 0;
#pragma unroll
        for (int e = 0; e < CHUNK; ++e) {
            const uint32_t b = items[c * CHUNK + e].x & 0x7fffffffu;
            t = b > t ? b : t;
        }
        chunk_top[c] = t;
    }
    for (int j = tid; j < len / 2; j += BUILD_NT) lists[(int64_t)j * pad + row] = lds[j];
    __syncthreads();
    if (wave != 0) return;
    // bound[c] = largest magnitude from chunk c on.  A row with a NaN or an infinity gets NaN (never finished by a
    // bound), a row of zeros -1 (finished at once: see the forward).
#pragma unroll
    for (int i = 0; i < WAVES; ++i) rest = part[i] > rest ? part[i] : rest;
    const int per = (chunks + 1 + 63) / 64;
    uint32_t suffix = 0;
    for (int j = per - 1; j >= 0; --j) {
        const int c = lane * per + j;
        if (c < chunks) suffix = chunk_top[c] > suffix ? chunk_top[c] : suffix;
    }
    uint32_t after = suffix;      // maximum over the lanes from this one on
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const uint32_t o = __shfl_down(after, s);
        if (lane + s < 64) after = o > after ? o : after;
    }
    uint32_t tail = __shfl_down(after, 1);
    if (lane == 63) tail = 0;
    tail = rest > tail ? rest : tail;
    const bool special = top >= INF_BITS || top == 0;
    const float instead = top == 0 ? -1.0f : __builtin_nanf("");
    for (int j = per - 1; j >= 0; --j) {
        const int c = lane * per + j;
        if (c < chunks) tail = chunk_top[c] > tail ? chunk_top[c] : tail;
        if (c <= chunks) bound[(int64_t)c * pad + row] = special ? instead : __uint_as_float(tail);
    }
}

// The lists of four consecutive rows by a workgroup, a wave per row with R elements per lane: no barrier but the one before the
// lists are written, 64 bytes of every pair of entries at a time.  Bound by instruction issue where build_row waits at its barriers
// (12608 / 4096 / 2048 / 1024 rows of K = 768 or 1024: 36.6 / 15.2 / 13.2 / 7.4 us by build_row, 23.3 / 10.8 / 10.1 / 8.1 us like this): from 2048 rows on.
// Up to K = 1024: a lane's elements of longer rows take registers that the other path's workgroups lack (K = 2048: 8192 rows 37.9 -> 33.8,
// two-sided call of 4096 x 2048 x 2048 425 -> 436 us; K = 3072 71 -> 112).
constexpr int WAVE_MAX_LENGTH = 256;
constexpr int WAVE_MIN_ROWS = 2048;
constexpr int WAVE_MAX_R = 4;            // of build_kernel: elements per thread of a row's workgroup
struct WaveList {               // of one row, in LDS
    uint32_t hist[BUCKETS];
    uint2 items[WAVE_MAX_LENGTH];
};
template <int R>
__device__ __forceinline__ void build_rows(const Rows &rows, int row0, int K, int len, uint4 *lists, float *bound, int pad, WaveList *all)
{
    static_assert(BUCKETS == 512, "eight buckets a lane");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = row0 + wave;
    WaveList &own = all[wave];
    if (row < rows.rows) {
        const int chunks = len / CHUNK;
        const float *src = rows.at(row, 0);
        float v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) v[t] = t * 64 + lane < K ? (src + t * 64)[(uint32_t)lane] : 0.0f;
        uint4 *const zero = reinterpret_cast<uint4 *>(own.hist);
        zero[lane] = zero[64 + lane] = make_uint4(0, 0, 0, 0);
        for (int j = lane; j < len; j += 64) own.items[j] = make_uint2(0u, key(0, 0));
        uint32_t top = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const uint32_t bits = __float_as_uint(v[t]) & 0x7fffffffu;
            top = bits > top ? bits : top;
        }
        top = (uint32_t)wave_max((int)top);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // (buckets, clamped k and zeros as in build_row)
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const uint32_t b = (top - (__float_as_uint(v[t]) & 0x7fffffffu)) >> BUCKET_SHIFT;
            if (b < (uint32_t)BUCKETS && lane < K - t * 64) atomicAdd(&own.hist[b], 1u);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t count[8], sum = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            count[i] = own.hist[lane * 8 + i];
            sum += count[i];
        }
        uint32_t incl = sum;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {
            const uint32_t o = __shfl_up(incl, s);
            if (lane >= s) incl += o;
        }
        uint32_t run = incl - sum;
        int started = 0;                // buckets that start inside the list
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            own.hist[lane * 8 + i] = run;
            started += run < (uint32_t)len;
            run += count[i];
        }
        const uint32_t open = (uint32_t)wave_sum(started);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t rest = 0;              // largest magnitude that is not listed
        uint32_t top_again = top;       // (the buckets are computed anew: kept, they would take R more registers)
        int lane_again = lane;
        asm volatile("" : "+v"(top_again), "+v"(lane_again));
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const uint32_t bits = __float_as_uint(v[t]) & 0x7fffffffu;
            const uint32_t b = (top_again - bits) >> BUCKET_SHIFT;
            const int k = t * 64 + lane_again;
            bool listed = false;
            if (b < open && k < K) {
                const uint32_t at = atomicAdd(&own.hist[b], 1u);
                if (at < (uint32_t)len) {
                    own.items[at] = make_uint2(__float_as_uint(v[t]), key((uint32_t)k, at + 1));
                    listed = true;
                }
            }
            if (!listed) rest = bits > rest ? bits : rest;
        }
        rest = (uint32_t)wave_max((int)rest);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // bound[c], the special rows: as in build_row, a chunk a lane
        static_assert(WAVE_MAX_LENGTH / CHUNK < 64, "a lane for each chunk and one for what follows");
        uint32_t after = 0;
        if (lane < chunks) {
#pragma unroll
            for (int e = 0; e < CHUNK; ++e) {
                const uint32_t b = own.items[lane * CHUNK + e].x & 0x7fffffffu;
                after = b > after ? b : after;
            }
        } else if (lane == chunks) {
            after = rest;
        }
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {
            const uint32_t o = __shfl_down(after, s);
            if (lane + s < 64) after = o > after ? o : after;
        }
        const bool special = top >= INF_BITS || top == 0;
        const float instead = top == 0 ? -1.0f : __builtin_nanf("");
        if (lane <= chunks) bound[(int64_t)lane * pad + row] = special ? instead : __uint_as_float(after);
    }
    __syncthreads();
    const int which = threadIdx.x & 3;
    if (row0 + which >= rows.rows) return;
    const uint4 *pairs = reinterpret_cast<const uint4 *>(all[which].items);
    for (int j = threadIdx.x >> 2; j < len / 2; j += BUILD_NT / 4) lists[(int64_t)j * pad + row0 + which] = pairs[j];
}

// One work item per workgroup: the rows of the searched operand; with a leading share also the rows of the other one
// and the 64 x 64 tiles of the transpose.
template <int R>
__global__ __launch_bounds__(BUILD_NT) void build_kernel(const Params p)
{
    extern __shared__ uint4 lds[];          // [cap] (value, key) pairs
    __shared__ uint32_t hist[BUCKETS];
    __shared__ uint32_t part[BUILD_NT / 64], part2[BUILD_NT / 64];
    __shared__ uint32_t chunk_top[BUILD_MAX_CHUNKS];
    __shared__ __attribute__((aligned(16))) float turn[64][65];
    // (with turns the decision has been made before; the LDS of one more array would cost a workgroup per CU at K = 3072)
    Weighed (&weighed)[OPTIONS] = reinterpret_cast<Weighed (&)[OPTIONS]>(turn);
    static_assert(sizeof(weighed) <= sizeof(turn), "decision and transpose share LDS");
    Decision d;
    if (p.decided) {
        d = *p.decision;
    } else {
        d = decide<BUILD_NT / 64>(p, weighed);
        d.side = __builtin_amdgcn_readfirstlane(d.side);
        d.length = __builtin_amdgcn_readfirstlane(d.length);
        d.lead = 0;
        if (blockIdx.x == 0 && threadIdx.x == 0) *p.decision = d;       // for the kernels that follow
        __syncthreads();        // every wave has read `weighed`, whose place build_rows takes
    }
    if (d.side == SIDE_NONE) return;
    const bool sx = d.side == SIDE_X;
    const Rows a = sx ? x_rows(p.call) : w_rows(p.call), b = sx ? w_rows(p.call) : x_rows(p.call);
    const int K = (int)p.call.K;
    const int row_tiles = (a.rows + 63) / 64;
    const int turns = d.lead > 0 ? row_tiles * ((K + 63) / 64) : 0;
    const int total = a.rows + (d.lead > 0 ? b.rows : 0) + turns;
    if (R <= WAVE_MAX_R && d.lead == 0 && d.length <= WAVE_MAX_LENGTH && a.rows >= WAVE_MIN_ROWS) {
        constexpr int ROWS = BUILD_NT / 64;
        static_assert(sizeof(WaveList) * ROWS <= sizeof(turn), "rows of a workgroup and the transpose share LDS");
        const int groups = (a.rows + ROWS - 1) / ROWS;
        if ((int)blockIdx.x < groups)
            build_rows<R <= WAVE_MAX_R ? R * ROWS : 1>(a, xcd_remap(blockIdx.x, groups) * ROWS, K, d.length, sx ? p.lists_x : p.lists_w,
                                               sx ? p.bound_x : p.bound_w, sx ? p.pad_x : p.pad_w, reinterpret_cast<WaveList *>(turn));
        return;
    }
    if ((int)blockIdx.x >= total) return;
    const int item = xcd_remap(blockIdx.x, total);
    if (item < total - turns) {
        const bool searched = item < a.rows, is_x = searched == sx;
        build_row<R>(is_x ? x_rows(p.call) : w_rows(p.call), searched ? item : item - a.rows, K, searched ? d.length : d.lead, searched,
                     is_x ? p.lists_x : p.lists_w, is_x ? p.bound_x : p.bound_w, is_x ? p.pad_x : p.pad_w, lds, hist, part, part2,
                     chunk_top);
    } else {
        const int t = item - (total - turns);
        turn_tile(a, K, p.turned, p.turned_ld, t % row_tiles * 64, t / row_tiles * 64, turn);
    }
}

// ---- search ------------------------------------------------------------------------------------------------
typedef uint32_t words4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) words4 global_words4;
typedef const __attribute__((address_space(1))) float global_float;
typedef const __attribute__((address_space(1))) char global_bytes;
// Address in the LDS of a key's place in a column: upper half times the bytes from one k to the next, on top of the
// column's. One instruction (the compiler takes two).
template <int BYTES>
__device__ __forceinline__ uint32_t lds_place(uint32_t key, uint32_t column)
{
    uint32_t at;
    asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(at) : "v"(key), "s"(BYTES), "v"(column));
    return at;
}
typedef const __attribute__((address_space(3))) char lds_bytes;
template <class T>
__device__ __forceinline__ T lds_read(uint32_t at) { return *(const __attribute__((address_space(3))) T *)(uintptr_t)at; }
__device__ __forceinline__ uint32_t lds_address(const float *p) { return (uint32_t)(uintptr_t)(lds_bytes *)p; }
typedef float floats4 __attribute__((ext_vector_type(4)));

// The two running extremes of an output are kept as doubles whose high word is the fp32 product and whose low
// word is the entry's key: for products of one sign, doubles order by (product, lower k first), so v_max_f64 /
// v_min_f64 keep value AND first index in one instruction, in any order of k.  (A product of the wrong sign never decides: an
// output is finished by its bound only with a positive maximum and a negative minimum.  fp32 infinities read as
// finite doubles; NaN products cannot occur in a listed row with finite tile values.)
__device__ __forceinline__ double keyed(float product, uint32_t key)
{
    typedef uint32_t pair_t __attribute__((ext_vector_type(2)));
    pair_t v;
    v.x = key;
    v.y = __float_as_uint(product);
    return __builtin_bit_cast(double, v);
}
__device__ __forceinline__ float product_of(double d) { return __uint_as_float((uint32_t)(__builtin_bit_cast(uint64_t, d) >> 32)); }
__device__ __forceinline__ uint32_t key_of(double d) { return (uint32_t)__builtin_bit_cast(uint64_t, d); }
// (the builtins would canonicalise their operands first: one more instruction each)
__device__ __forceinline__ void max64(double &a, double b) { asm("v_max_f64 %0, %0, %1" : "+v"(a) : "v"(b)); }
__device__ __forceinline__ void min64(double &a, double b) { asm("v_min_f64 %0, %0, %1" : "+v"(a) : "v"(b)); }
__device__ __forceinline__ double lane_value_at(double d, int from)      // from: lane * 4, of each lane its own
{
    const uint64_t b = __builtin_bit_cast(uint64_t, d);
    const uint32_t lo = __builtin_amdgcn_ds_bpermute(from, (uint32_t)b), hi = __builtin_amdgcn_ds_bpermute(from, (uint32_t)(b >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float lane_value_at(float v, int from)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(v)));
}
__device__ __forceinline__ double lane_value(double d, int l)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, d);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, l), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float lane_value(float v, int l)
{
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l));
}

// The running extremes of a lane's 4 outputs: with indices (keyed doubles), or products alone.
template <bool ARGS>
struct Extremes;

template <>
struct Extremes<true> {
    typedef double value;
    double mx[4], mn[4];
    static __device__ __forceinline__ value low() { return keyed(-__builtin_inff(), key(0, 0)); }
    static __device__ __forceinline__ value high() { return keyed(__builtin_inff(), key(0, 0)); }
    static __device__ __forceinline__ value make(float product, int k) { return keyed(product, key((uint32_t)k, 0)); }
    static __device__ __forceinline__ float product(value v) { return product_of(v); }
    static __device__ __forceinline__ void both(value &a, value &b, float product, uint32_t key)
    {
        const double d = keyed(product, key);
        max64(a, d);
        min64(b, d);
    }
    static __device__ __forceinline__ void both(value &a, value &b, const uint4 &it, float w0, float w1)
    {
        both(a, b, __uint_as_float(it.x) * w0, it.y);
        both(a, b, __uint_as_float(it.z) * w1, it.w);
    }
    // a running extreme whose entry is another lane's to know: below every listed entry of the same product
    static __device__ __forceinline__ value start(float product) { return keyed(product, 0); }
    static __device__ __forceinline__ void merge(value &a, value &b, value theirs_a, value theirs_b, int from)
    {
        max64(a, lane_value_at(theirs_a, from));
        min64(b, lane_value_at(theirs_b, from));
    }
    static __device__ __forceinline__ void merge(value &a, value &b, int from) { merge(a, b, a, b, from); }
    // one pair of list entries against 4 tile values each.  Written out because the compiler copies the key into the low
    // word of every key: here two register pairs hold it for the four products of an entry.
    __device__ __forceinline__ void entry(float x, uint32_t key, const floats4 &w)
    {
        asm("v_mov_b32 v120, %9\n\tv_mov_b32 v122, %9\n\t"
            "v_mul_f32 v121, %8, %10\n\tv_mul_f32 v123, %8, %11\n\t"
            "v_max_f64 %0, %0, v[120:121]\n\tv_min_f64 %4, %4, v[120:121]\n\t"
            "v_mul_f32 v121, %8, %12\n\t"
            "v_max_f64 %1, %1, v[122:123]\n\tv_min_f64 %5, %5, v[122:123]\n\t"
            "v_mul_f32 v123, %8, %13\n\t"
            "v_max_f64 %2, %2, v[120:121]\n\tv_min_f64 %6, %6, v[120:121]\n\t"
            "v_max_f64 %3, %3, v[122:123]\n\tv_min_f64 %7, %7, v[122:123]"
            : "+&v"(mx[0]), "+&v"(mx[1]), "+&v"(mx[2]), "+&v"(mx[3]), "+&v"(mn[0]), "+&v"(mn[1]), "+&v"(mn[2]), "+&v"(mn[3])
            : "v"(x), "v"(key), "v"(w.x), "v"(w.y), "v"(w.z), "v"(w.w)
            : "v120", "v121", "v122", "v123");
    }
    __device__ __forceinline__ void entries(const uint4 &it, const floats4 &w0, const floats4 &w1)
    {
        entry(__uint_as_float(it.x), it.y, w0);
        entry(__uint_as_float(it.z), it.w, w1);
    }
};

template <>
struct Extremes<false> {
    typedef float value;
    float mx[4], mn[4];
    static __device__ __forceinline__ value low() { return -__builtin_inff(); }
    static __device__ __forceinline__ value high() { return __builtin_inff(); }
    static __device__ __forceinline__ value make(float product, int) { return product; }
    static __device__ __forceinline__ float product(value v) { return v; }
    static __device__ __forceinline__ void both(value &a, value &b, float product, uint32_t)
    {
        a = __builtin_fmaxf(a, product);
        b = __builtin_fminf(b, product);
    }
    static __device__ __forceinline__ void both(value &a, value &b, const uint4 &it, float w0, float w1)
    {
        const float p0 = __uint_as_float(it.x) * w0, p1 = __uint_as_float(it.z) * w1;
        a = __builtin_fmaxf(__builtin_fmaxf(a, p0), p1);
        b = __builtin_fminf(__builtin_fminf(b, p0), p1);
    }
    static __device__ __forceinline__ value start(float product) { return product; }
    static __device__ __forceinline__ void merge(value &a, value &b, value theirs_a, value theirs_b, int from)
    {
        a = __builtin_fmaxf(a, lane_value_at(theirs_a, from));
        b = __builtin_fminf(b, lane_value_at(theirs_b, from));
    }
    static __device__ __forceinline__ void merge(value &a, value &b, int from) { merge(a, b, a, b, from); }
    __device__ __forceinline__ void entries(const uint4 &it, const floats4 &w0, const floats4 &w1)
    {
        const float x0 = __uint_as_float(it.x), x1 = __uint_as_float(it.z);
        const float f0[4] = {w0.x, w0.y, w0.z, w0.w}, f1[4] = {w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float p0 = x0 * f0[j], p1 = x1 * f1[j];
            mx[j] = __builtin_fmaxf(__builtin_fmaxf(mx[j], p0), p1);       // v_max3_f32
            mn[j] = __builtin_fminf(__builtin_fminf(mn[j], p0), p1);
        }
    }
};

// One output by the whole wave over the rest of its list, 64 entries at a time; whether its bound finished it.
//   column: the output's column of the tile, by 65535 - k; at: chunks already searched; bmax: bound on the tile column
template <int STRIDE, class E>
__device__ __forceinline__ bool finish_by_list(const Params &p, bool sx, int row, const float *column, int at, int chunks, float bmax,
                                               int lane, typename E::value &mx, typename E::value &mn)
{
    const uint4 *lists = sx ? p.lists_x : p.lists_w;
    const float *bound = sx ? p.bound_x : p.bound_w;
    const int pad = sx ? p.pad_x : p.pad_w;
    for (int ch = at; ch < chunks; ch += 64 / CHUNK) {
        const int e = ch * CHUNK + lane;
        const int next = (ch + 64 / CHUNK) < chunks ? ch + 64 / CHUNK : chunks;
        const float u = bound[(int64_t)next * pad + row] * bmax;
        if (e < chunks * CHUNK) {
            const uint2 it = reinterpret_cast<const uint2 *>(lists + (int64_t)(e >> 1) * pad + row)[e & 1];
            E::both(mx, mn, __uint_as_float(it.x) * column[(int)(it.y >> 16) * STRIDE], it.y);
        }
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) E::merge(mx, mn, (lane ^ s) << 2);
        if (E::product(mx) > u && E::product(mn) < -u) return true;
    }
    return false;
}

// What a list does not finish (it is too short, or the row or a tile column holds what no bound covers: NaN, infinity, a zero
// extreme) is scanned over every k, in the exact terms of the ascending scan with ordered strict compares.
struct Scan {
    float hi, lo;
    int ih, il;
    __device__ __forceinline__ void clear()
    {
        hi = -__builtin_inff();
        lo = __builtin_inff();
        ih = il = INT32_MAX;
    }
    __device__ __forceinline__ void take(float q, int k)
    {
        if (q > hi) { hi = q; ih = k; }
        if (q < lo) { lo = q; il = k; }
    }
    __device__ __forceinline__ void merge(int from)         // with another lane's
    {
        const float oh = lane_value_at(hi, from), ol = lane_value_at(lo, from);
        const int jh = __builtin_amdgcn_ds_bpermute(from, ih), jl = __builtin_amdgcn_ds_bpermute(from, il);
        if (oh > hi || (oh == hi && jh < ih)) { hi = oh; ih = jh; }
        if (ol < lo || (ol == lo && jl < il)) { lo = ol; il = jl; }
    }
    // an extreme that was never improved keeps the first k
    template <class E>
    __device__ __forceinline__ void give(typename E::value &mx, typename E::value &mn) const
    {
        mx = E::make(hi, ih == INT32_MAX ? 0 : ih);
        mn = E::make(lo, il == INT32_MAX ? 0 : il);
    }
};

// One output by the whole wave, a lane every 64th k; column as in finish_by_list.
template <int STRIDE, class E>
__device__ __forceinline__ void scan_one(const float *src, int K, const float *column, int lane, typename E::value &mx,
                                         typename E::value &mn)
{
    constexpr int AHEAD = 8;
    Scan r;
    r.clear();
    for (int k0 = 0; k0 < K; k0 += 64 * AHEAD) {
        float v[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int k = k0 + i * 64 + lane;
            v[i] = src[(uint32_t)(k < K ? k : K - 1)];
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int past = k0 + i * 64 + lane, k = past < K ? past : K - 1;     // past the end the last k again
            r.take(v[i] * column[(65535 - k) * STRIDE], k);
        }
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) r.merge((lane ^ s) << 2);
    r.give<E>(mx, mn);
}

// The outputs of one searched row, all columns of the tile, by the whole wave.  A lane takes every RWth k of two columns of its
// own quad (four would cost the search registers); bound by instruction issue, ~35 per k and two columns.  On return each lane
// holds the outputs of its columns.  As many instructions per output as scan_one, but the tile is read contiguously where that one
// reads 4 bytes of every row of it (forward call with 4 % of the rows all +-1, anywhere / next to each other, scan_one and scan_row and dense: 3707 /
// 1595 and 1620 / 1542 and 1680 us at 12608 x 768 -> 3072, 3466 / 11189 and 1716 / 1560 and 3110 us at 16384 x 4096 -> 1024).
//   src: the row, contiguous; by_key: the lane's columns of the tile, by 65535 - k
template <int STRIDE, int RW, int LANE_STEP, class E>
__device__ __forceinline__ void scan_row(const float *src, int K, const float *by_key, int lane, int slice, typename E::value (&mx)[2],
                                         typename E::value (&mn)[2])
{
    constexpr int AHEAD = 4, STEP = AHEAD * RW;
    Scan r[2];
    r[0].clear();
    r[1].clear();
    const char *const end = reinterpret_cast<const char *>(by_key + 65535 * STRIDE);      // k = 0
    auto k_of = [&](int k0, int u) {            // (past the end of the row the last k again)
        const int k = k0 + u * RW + slice;
        return k < K ? k : K - 1;
    };
    auto fetch = [&](float (&v)[AHEAD], int k0) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = src[(uint32_t)k_of(k0, u)];
        asm volatile("" ::: "memory");          // the loads stay ahead of the arithmetic
    };
    auto products = [&](const float (&v)[AHEAD], int k0) {
        float2 w[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) w[u] = *reinterpret_cast<const float2 *>(end - __mul24(k_of(k0, u), STRIDE * 4));
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const float f[2] = {w[u].x, w[u].y};
            const int k = k_of(k0, u);
#pragma unroll
            for (int j = 0; j < 2; ++j) r[j].take(v[u] * f[j], k);
        }
    };
    float first[AHEAD], second[AHEAD];
    fetch(first, 0);
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 2 * STEP) {
        fetch(second, k0 + STEP);
        products(first, k0);
        if (k0 + STEP >= K) break;
        fetch(first, k0 + 2 * STEP);
        products(second, k0 + STEP);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int s = LANE_STEP; s < LANE_STEP * RW; s <<= 1) r[j].merge((lane ^ s) << 2);
        r[j].give<E>(mx[j], mn[j]);
    }
}

// A workgroup holds a tile of TB rows of the other operand in LDS, whole rows, as [K - 1 - k][TB] (a key's upper half
// is then the address but for a constant); a lane owns one
// listed row x 4 consecutive tile rows, and TB / 4 neighbouring lanes share a listed row, so that an entry costs
// each lane one 16-byte LDS read for 4 products and the lanes of a row read TB * 4 contiguous bytes.  Waves take
// blocks of 64 * 4 / TB listed rows in turn and need no barrier after the tile is loaded.  A wave looks at its
// lists chunk by chunk until TOGETHER of its 256 outputs are not yet finished by their bound (41 entries at K = 4096, where all but
// FEW take 90 and the mean output needs 28), then goes on with a lane for each of those -- one product per entry instead of four of
// which most are decided -- and finishes the last FEW one by one with all its lanes.  (Us; TOGETHER, FEW = none, 2 / 32, 2 / 64, 2 / 64, 1 /
// 64, 0: 256 x 4096 x 4096 65.8 / 63.3 / 62.3 / 61.0 / 61.7, 12608 x 768 -> 3072 587 / 581 / 577 / 566 / 560, 16384 x 4096 ->
// 4096 values only 752 / 756 / 758 / 751 / 779, 16384 x 4096 -> 1024 405 / 394 / 386 / 385 / 396; with the lanes in the order of the
// rows, whose list entries are neighbours, 64, 1 and 48, 1: 60.1 and 60.2, 486 and 492, 724 and 729, 360 and 361.  Handing lanes out anew at every
// quarter, 1 to 64 an output, costs more in exchanges than it saves: 64.0 / 625 / 898 / 422.  Lists two chunks ahead: 773 for 745.)
// What bounds it (counters, values only at K = 4096): VALU instructions at 4 cycles take 0.63 of the busy cycles, the random
// 16-byte LDS reads 0.67 (three fifths of it bank conflicts), list entries on their way from the caches to the registers 0.95
// -- but with the lanes of a row loading a quarter or half of its entries each and passing them round the quad the calls take the
// same: 562 / 735 / 384 us for 560 / 745 / 383.  16384 x 4096 -> 4096 with 48: 61 us before the search, 59 us of tile loads, 320 us until
// TOGETHER, 260 us for those (245 in the order of the rows), 42 us for the last one.
constexpr int FEW = 1;
constexpr int TOGETHER = 64;         // at most a wave's lanes
// Outputs of a row that are scanned one by one, 8 to 17 us each beside the other waves' work; the whole row takes 30 to 60 us.
constexpr int FEW_OF_ROW = 4;

// Where a lane sits and how the tile lies in LDS.  One-sided: neighbouring lanes share a searched row, the tile is
// [k][TB], so that the lanes of a row read TB * 4 contiguous bytes and write as many.  Two-sided: neighbouring lanes are
// neighbouring searched rows, which is how the transposed operand is read contiguously; the tile is [TB / 4][k][4],
// so that the lanes of one quad still spread over all banks.  (k descending: a key's upper half is then the address
// but for a constant.)
template <int TB, bool TWO>
struct Lanes {
    static constexpr int Q = TB / 4;               // quads of tile rows
    static constexpr int RW = 64 / Q;              // searched rows per wave
    static constexpr int STRIDE = TWO ? 4 : TB;    // floats from one k to the next
    static __device__ __forceinline__ int quad(int lane) { return TWO ? lane / RW : lane % Q; }
    static __device__ __forceinline__ int row(int lane) { return TWO ? lane % RW : lane / Q; }
    static __device__ __forceinline__ int base(int quad, int K) { return TWO ? quad * K * 4 : quad * 4; }
};

// PAST: stores that are lines by this layout go past the L2 (launch_forward says when they are lines in memory).
template <int TB, bool ARGS, bool TWO, bool PAST>
__global__ __launch_bounds__(NT) void forward_kernel(const Params p)
{
    typedef Extremes<ARGS> E;
    typedef Lanes<TB, TWO> L;
    constexpr int Q = L::Q, RW = L::RW;
    extern __shared__ float tile[];         // the tile; two-sided: then [TB][lead] (value, key)
    __shared__ float tops[TB];
    __shared__ uint8_t places[NT / 64][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Decision d = *p.decision;
    if (d.side == SIDE_NONE || (d.lead > 0) != TWO) return;
    const Call &c = p.call;
    const bool lists_x = d.side == SIDE_X;
    const uint4 *const lists = lists_x ? p.lists_x : p.lists_w, *const lists_b = lists_x ? p.lists_w : p.lists_x;
    const float *const bound = lists_x ? p.bound_x : p.bound_w, *const bound_b = lists_x ? p.bound_w : p.bound_x;
    const int pad = lists_x ? p.pad_x : p.pad_w, pad_b = lists_x ? p.pad_w : p.pad_x;
    const Rows a = lists_x ? x_rows(c) : w_rows(c), b = lists_x ? w_rows(c) : x_rows(c);
    const int K = (int)c.K;
    const int tiles = (b.rows + TB - 1) / TB, splits = splits_of(TB, a.rows, tiles, p.cus);
    if ((int)blockIdx.x >= tiles * splits) return;
    const int logical = xcd_remap(blockIdx.x, tiles * splits);
    const int split = logical / tiles, b0 = (logical - split * tiles) * TB;
    const int chunks = d.length / CHUNK;

    // ---- tile: rows b0 .. b0 + TB - 1 (past the end: the last one again), and the largest magnitude of each ----
    // (bit patterns of magnitudes order as integers; infinities and NaN stay on top)
    uint32_t top[4] = {0, 0, 0, 0};
    auto see = [&](int i, float v) {
        const uint32_t bits = __float_as_uint(v) & 0x7fffffffu;
        top[i] = bits > top[i] ? bits : top[i];
    };
    uint2 *const lead_s = reinterpret_cast<uint2 *>(tile + TB * K);
    for (int i = threadIdx.x; TWO && i < TB * (d.lead / 2); i += NT) {
        const int r = i % TB, pair = i / TB, row = b0 + r < b.rows ? b0 + r : b.rows - 1;
        *reinterpret_cast<uint4 *>(&lead_s[r * d.lead + pair * 2]) = lists_b[(int64_t)pair * pad_b + row];
    }
    if (threadIdx.x < TB) tops[threadIdx.x] = 0.0f;
    int my_quad;
    if (b.k_stride == 1) {
        // consecutive lanes take consecutive k of one quad of rows
        constexpr int STEP = NT / 64 / Q * 64;
        my_quad = wave % Q;
        const float *src[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = b0 + my_quad * 4 + i;
            src[i] = b.at(r < b.rows ? r : b.rows - 1, 0);
        }
#pragma unroll 4
        for (int k = wave / Q * 64 + lane; k < K; k += STEP) {
            float4 v;
            v.x = src[0][(uint32_t)k]; v.y = src[1][(uint32_t)k]; v.z = src[2][(uint32_t)k]; v.w = src[3][(uint32_t)k];
            *reinterpret_cast<float4 *>(&tile[L::base(my_quad, K) + (K - 1 - k) * L::STRIDE]) = v;
            see(0, v.x); see(1, v.y); see(2, v.z); see(3, v.w);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) top[i] = (uint32_t)wave_max((int)top[i]);
    } else {
        // rows of the operand are columns in memory: Q lanes take the TB values of one k
        my_quad = lane % Q;
        const int r0 = b0 + my_quad * 4;
        int r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = (r0 + i) < b.rows ? r0 + i : b.rows - 1;
#pragma unroll 4
        for (int k = threadIdx.x / Q; k < K; k += NT / Q) {
            const float *src = b.p + k * b.k_stride;
            float4 v;
            v.x = src[r[0]]; v.y = src[r[1]]; v.z = src[r[2]]; v.w = src[r[3]];
            *reinterpret_cast<float4 *>(&tile[L::base(my_quad, K) + (K - 1 - k) * L::STRIDE]) = v;
            see(0, v.x); see(1, v.y); see(2, v.z); see(3, v.w);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 32; s >= Q; s >>= 1) {
                const uint32_t o = __shfl_xor(top[i], s);
                top[i] = o > top[i] ? o : top[i];
            }
    }
    __syncthreads();
    if (b.k_stride == 1 ? lane == 0 : lane < Q)
#pragma unroll
        for (int i = 0; i < 4; ++i) atomicMax(reinterpret_cast<uint32_t *>(&tops[my_quad * 4 + i]), top[i]);
    __syncthreads();

    // An output is finished when bound * bmax is below both extremes.  A tile row with an infinity or a NaN gets a
    // NaN for bmax (never finished that way); a zero row on one side gets -1 (finished at once: every product is a
    // zero and the first one decides), zero rows on both sides make +1 and are finished by the full scan.
    const int q = L::quad(lane);
    float bmax[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (TWO) {              // what the leading share leaves of the tile row (the same special values)
            const int r = b0 + q * 4 + j < b.rows ? b0 + q * 4 + j : b.rows - 1;
            bmax[j] = bound_b[(int64_t)(d.lead / CHUNK) * pad_b + r];
            continue;
        }
        const float t = tops[q * 4 + j];
        bmax[j] = t == 0.0f ? -1.0f : t < __builtin_inff() ? t : __builtin_nanf("");
    }
    const float *by_key = tile + L::base(q, K) + (K - 65536) * L::STRIDE;      // element (65535 - k) * STRIDE + row of the quad
    const uint32_t mine = lds_address(by_key);
    const int64_t pair_bytes = (int64_t)pad * 16, bound_bytes = (int64_t)pad * 4;

    // Stores with x searched: a row's outputs lie along the tile rows.  Two-sided, the lanes that hold them change places
    // first (lane r * Q + q takes over from lane q * RW + r).
    const int sq = lane % Q, sr = lane / Q;
    const int swap_from = (sq * RW + sr) * 4;
    const bool whole = b0 + sq * 4 + 3 < b.rows && (c.M & 3) == 0;
    const uint32_t lane_off = lists_x ? (uint32_t)sr * (uint32_t)c.M + sq * 4 : q * 4 * (uint32_t)c.M + L::row(lane);

    const int blocks = (a.rows + RW - 1) / RW;
    const int per_split = (blocks + splits - 1) / splits;
    const int last = (split + 1) * per_split < blocks ? (split + 1) * per_split : blocks;
    for (int blk = split * per_split + wave; blk < last; blk += NT / 64) {
        const int arow = blk * RW + L::row(lane);
        const int row = arow < a.rows ? arow : a.rows - 1;
        const uint32_t list_off = (uint32_t)row * 16u, bound_off = (uint32_t)row * 4u;
        E e;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            e.mx[j] = E::low();
            e.mn[j] = E::high();
        }
        // ---- the leading entries of the tile rows: (value, key) from their lists, the other factor of four
        // consecutive tile rows x neighbouring listed rows from the transposed operand ----
        if constexpr (TWO) {
            const char *turned = reinterpret_cast<const char *>(p.turned);
            const uint32_t ld4 = (uint32_t)p.turned_ld * 4u;
            const uint32_t turned_off = (uint32_t)row * 4u + 65535u * ld4;
            const uint2 *mine_led = lead_s + q * 4 * d.lead;
            auto lead_rows = [&](float (&to)[8], int pair) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint4 l = *reinterpret_cast<const uint4 *>(&mine_led[j * d.lead + pair * 2]);
                    to[2 * j] = *reinterpret_cast<const float *>(turned + (turned_off - __umul24(l.y >> 16, ld4)));
                    to[2 * j + 1] = *reinterpret_cast<const float *>(turned + (turned_off - __umul24(l.w >> 16, ld4)));
                }
                asm volatile("" ::: "memory");
            };
            auto lead_products = [&](const float (&v)[8], int pair) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint4 l = *reinterpret_cast<const uint4 *>(&mine_led[j * d.lead + pair * 2]);
                    E::both(e.mx[j], e.mn[j], v[2 * j] * __uint_as_float(l.x), l.y);
                    E::both(e.mx[j], e.mn[j], v[2 * j + 1] * __uint_as_float(l.z), l.w);
                }
            };
            // rows two pairs ahead of the products; a multiple of 4 pairs (past the end: the last pair again)
            const int pairs = d.lead / 2;
            float v0[8], v1[8], v2[8], v3[8];
            lead_rows(v0, 0);
            lead_rows(v1, 1);
            for (int i = 0; i < pairs; i += 4) {
                lead_rows(v2, i + 2);
                lead_products(v0, i);
                lead_rows(v3, i + 3);
                lead_products(v1, i + 1);
                lead_rows(v0, i + 4 < pairs ? i + 4 : pairs - 1);
                lead_products(v2, i + 2);
                lead_rows(v1, i + 5 < pairs ? i + 5 : pairs - 1);
                lead_products(v3, i + 3);
            }
        }
        int ch = 0;
        uint64_t open[4];
        // a chunk and the bound on what follows it, as global loads: flat ones would count as LDS accesses too, and every read of
        // the tile would wait for them
        auto fetch = [&](uint4 (&to)[CHUNK / 2], float &u, int chunk, uint32_t off) {
            asm volatile("" : "+v"(off));       // scalar base + 32-bit lane offset: the offset is not widened outside the loop
            u = *(global_float *)((global_bytes *)bound + (chunk + 1) * bound_bytes + (off >> 2));
            global_bytes *base = (global_bytes *)lists + (int64_t)chunk * (CHUNK / 2) * pair_bytes;
#pragma unroll
            for (int i = 0; i < CHUNK / 2; ++i, base += pair_bytes) {
                asm volatile("" : "+s"(base));
                const words4 v = *(global_words4 *)(base + off);
                to[i] = make_uint4(v.x, v.y, v.z, v.w);
            }
        };
        constexpr int AHEAD = 1;
        // true when the search is over
        auto step = [&](const uint4 (&cur)[CHUNK / 2], float u, uint4 (&nxt)[CHUNK / 2], float &unxt) {
            fetch(nxt, unxt, ch + 1 < chunks ? ch + 1 : ch, list_off);
            asm volatile("" ::: "memory");      // the loads stay ahead of the arithmetic
#pragma unroll
            for (int i0 = 0; i0 < CHUNK / 2; i0 += AHEAD) {
                floats4 w[2 * AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) {
                    w[2 * i] = lds_read<floats4>(lds_place<L::STRIDE * 4>(cur[i0 + i].y, mine));
                    w[2 * i + 1] = lds_read<floats4>(lds_place<L::STRIDE * 4>(cur[i0 + i].w, mine));
                }
                asm volatile("" ::: "memory");
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) e.entries(cur[i0 + i], w[2 * i], w[2 * i + 1]);
            }
            ++ch;
            int left = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float ub = u * bmax[j];
                open[j] = ~(__ballot(E::product(e.mx[j]) > ub) & __ballot(E::product(e.mn[j]) < -ub));
                left += __popcll(open[j]);
            }
            return left <= TOGETHER || ch == chunks;
        };
        {
            uint4 first[CHUNK / 2], second[CHUNK / 2];
            float u1, u2;
            fetch(first, u1, 0, list_off);
            while (true) {
                if (step(first, u1, second, u2)) break;
                if (step(second, u2, first, u1)) break;
            }
        }
        // the rows past the end are copies of the last one
#pragma unroll
        for (int j = 0; j < 4; ++j) open[j] &= __ballot(arow < a.rows);
        int own = lane;
        asm volatile("" : "+v"(own));           // what is derived from it below is not kept in registers during the search
        // ---- the last TOGETHER outputs: a lane each instead of four on a lane of which most are finished ----
        const int unfinished = __popcll(open[0]) + __popcll(open[1]) + __popcll(open[2]) + __popcll(open[3]);
        if (unfinished > FEW && ch < chunks) {
            // in the order of the lanes, that is of the rows: their list entries are neighbours in memory
            int rank[4], before = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                before = __builtin_amdgcn_mbcnt_hi((uint32_t)(open[j] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)open[j], before));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                rank[j] = before;
                if (open[j] >> own & 1) {
                    places[wave][before] = (uint8_t)(own * 4 + j);
                    ++before;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int task = places[wave][own < unfinished ? own : unfinished - 1], from = task & ~3, tj = task & 3, tl = task >> 2;
            const int trow = blk * RW + L::row(tl) < a.rows ? blk * RW + L::row(tl) : a.rows - 1;
            uint4 first[CHUNK / 2], second[CHUNK / 2];
            float u1, u2;
            fetch(first, u1, ch, (uint32_t)trow * 16u);
            typename E::value tmx = E::start(lane_value_at(E::product(e.mx[0]), from)), tmn = E::start(lane_value_at(E::product(e.mn[0]), from));
            float tb = lane_value_at(bmax[0], from);
#pragma unroll
            for (int j = 1; j < 4; ++j) {
                const float hi = lane_value_at(E::product(e.mx[j]), from), lo = lane_value_at(E::product(e.mn[j]), from);
                const float bj = lane_value_at(bmax[j], from);
                if (tj == j) { tmx = E::start(hi); tmn = E::start(lo); tb = bj; }
            }
            const uint32_t column = lds_address(tile + L::base(L::quad(tl), K) + (K - 65536) * L::STRIDE + tj);
            const uint64_t used = (2ull << (unfinished - 1)) - 1;
            uint64_t still;
            auto tail = [&](const uint4 (&cur)[CHUNK / 2], float u, uint4 (&nxt)[CHUNK / 2], float &unxt) {
                fetch(nxt, unxt, ch + 1 < chunks ? ch + 1 : ch, (uint32_t)trow * 16u);
                asm volatile("" ::: "memory");
#pragma unroll
                for (int i = 0; i < CHUNK / 2; ++i) {
                    const float w0 = lds_read<float>(lds_place<L::STRIDE * 4>(cur[i].y, column));
                    const float w1 = lds_read<float>(lds_place<L::STRIDE * 4>(cur[i].w, column));
                    E::both(tmx, tmn, cur[i], w0, w1);
                }
                ++ch;
                const float ub = u * tb;
                still = ~(__ballot(E::product(tmx) > ub) & __ballot(E::product(tmn) < -ub)) & used;
                return __popcll(still) <= FEW || ch == chunks;
            };
            while (true) {
                if (tail(first, u1, second, u2)) break;
                if (tail(second, u2, first, u1)) break;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool mine = open[j] >> own & 1;
                typename E::value hi = e.mx[j], lo = e.mn[j];
                E::merge(hi, lo, tmx, tmn, rank[j] << 2);
                if (mine) { e.mx[j] = hi; e.mn[j] = lo; }
                open[j] = __ballot(mine && (still >> (rank[j] & 63) & 1));
            }
        }
        // (one copy of the code each: the output's state is picked by selects)
        if (ch < chunks) {
            uint64_t todo[4] = {open[0], open[1], open[2], open[3]};
            while (todo[0] | todo[1] | todo[2] | todo[3]) {
                const int j = todo[0] ? 0 : todo[1] ? 1 : todo[2] ? 2 : 3;
                const int l = __builtin_ctzll(todo[0] ? todo[0] : todo[1] ? todo[1] : todo[2] ? todo[2] : todo[3]);
                typename E::value fx = lane_value(j == 0 ? e.mx[0] : j == 1 ? e.mx[1] : j == 2 ? e.mx[2] : e.mx[3], l);
                typename E::value fn = lane_value(j == 0 ? e.mn[0] : j == 1 ? e.mn[1] : j == 2 ? e.mn[2] : e.mn[3], l);
                const float bm = lane_value(j == 0 ? bmax[0] : j == 1 ? bmax[1] : j == 2 ? bmax[2] : bmax[3], l);
                const bool done = finish_by_list<L::STRIDE, E>(p, lists_x, __builtin_amdgcn_readlane(row, l),
                                                               tile + L::base(L::quad(l), K) + (K - 65536) * L::STRIDE + j, ch, chunks, bm,
                                                               own, fx, fn);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i == j) {
                        todo[i] &= todo[i] - 1;
                        if (done) open[i] &= ~(1ull << l);
                        if (own == l) { e.mx[i] = fx; e.mn[i] = fn; }
                    }
            }
        }
        while (open[0] | open[1] | open[2] | open[3]) {
            const int j = open[0] ? 0 : open[1] ? 1 : open[2] ? 2 : 3;
            const int l = __builtin_ctzll(open[0] ? open[0] : open[1] ? open[1] : open[2] ? open[2] : open[3]);
            const float *src = a.at(__builtin_amdgcn_readlane(row, l), 0);
            const bool mine = L::row(own) == L::row(l);
            const uint64_t lanes = __ballot(mine);
            if (__popcll(open[0] & lanes) + __popcll(open[1] & lanes) + __popcll(open[2] & lanes) + __popcll(open[3] & lanes) > FEW_OF_ROW) {
                // one word of each 128-byte line of the row, so that the scan waits for the memory behind the L2 once
                float touched = 0.0f;
                for (int k = own * 32; k < K; k += 64 * 32) touched += src[(uint32_t)k];
                asm volatile("" ::"v"(touched));
                // (what the row's finished outputs hold already is what the scan gives them)
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    typename E::value fx[2], fn[2];
                    scan_row<L::STRIDE, RW, TWO ? 1 : Q, E>(src, K, by_key + i, own, L::row(own), fx, fn);
                    if (mine) {
                        e.mx[i] = fx[0]; e.mx[i + 1] = fx[1];
                        e.mn[i] = fn[0]; e.mn[i + 1] = fn[1];
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) open[i] &= ~lanes;
            } else {
                typename E::value fx, fn;
                scan_one<L::STRIDE, E>(src, K, tile + L::base(L::quad(l), K) + (K - 65536) * L::STRIDE + j, own, fx, fn);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i == j) {
                        open[i] &= open[i] - 1;
                        if (own == l) { e.mx[i] = fx; e.mn[i] = fn; }
                    }
            }
        }
        // ---- outputs ----
        {
            const float u0 = bound[row];
            const int64_t plane = c.N * c.M;
            float sum[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if ((u0 == -1.0f) != (bmax[j] == -1.0f) && u0 == u0 && bmax[j] == bmax[j]) {
                    const float z = *a.at(row, 0) * tile[L::base(q, K) + (K - 1) * L::STRIDE + j];
                    e.mx[j] = e.mn[j] = E::make(z, 0);
                }
                sum[j] = E::product(e.mx[j]) + E::product(e.mn[j]);
                const int m = lists_x ? b0 + q * 4 + j : arow;
                if (c.bias && m < (int)c.M) sum[j] = sum[j] + c.bias[m];
            }
            // Stores that cover whole 128-byte lines go past the L2 (12608 x 768 -> 3072, seven planes: 560 -> 495 us,
            // 16384 x 4096 -> 1024: 383 -> 363); narrower ones meet their neighbours' there (12608 x 3072 -> 768 past it: 238 ->
            // 473 us).  Uniform base of the block + 32-bit offset of the lane.
            const int64_t base = lists_x ? (int64_t)blk * RW * c.M + b0 : (int64_t)b0 * c.M + blk * RW;
            auto put = [&](float *dst, const float (&v)[4]) {
                float *to = dst + base;
                if (lists_x) {
                    float t[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) t[j] = TWO ? __int_as_float(__builtin_amdgcn_ds_bpermute(swap_from, __float_as_int(v[j]))) : v[j];
                    if (blk * RW + sr >= a.rows) {
                    } else if (whole && ((uintptr_t)dst & 15) == 0) {
                        const floats4 all = {t[0], t[1], t[2], t[3]};
                        if constexpr (PAST && TB == 32) __builtin_nontemporal_store(all, reinterpret_cast<floats4 *>(to + lane_off));
                        else *reinterpret_cast<floats4 *>(to + lane_off) = all;
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (b0 + sq * 4 + j < b.rows) to[lane_off + j] = t[j];
                    }
                } else if (arow < a.rows) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (b0 + q * 4 + j < b.rows) {
                            if constexpr (PAST && RW >= 32) __builtin_nontemporal_store(v[j], to + lane_off + j * (uint32_t)c.M);
                            else to[lane_off + j * (uint32_t)c.M] = v[j];
                        }
                }
            };
            if constexpr (ARGS) {
                if (!c.argmin) {
                    float both[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) both[j] = __int_as_float(pack_picks(index_in(key_of(e.mx[j])), index_in(key_of(e.mn[j]))));
                    put(reinterpret_cast<float *>(c.argmax), both);
                }
#pragma unroll
                for (int side2 = 0; side2 < 2; ++side2) {
                    uint32_t kk[4];
                    float f[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        kk[j] = key_of(side2 ? e.mn[j] : e.mx[j]);
                        f[j] = __int_as_float(index_in(kk[j]));
                    }
                    if (c.argmin) put(reinterpret_cast<float *>(side2 ? c.argmin : c.argmax), f);
                    if (c.wsel || c.xsel) {
                        // the selected operands, of the tile and of the listed row: from the list, which this
                        // XCD's L2 still holds, rather than from anywhere in the row (16384 x 4096 -> 1024: 593 ->
                        // 405 us, 12608 x 3072 -> 768: 345 -> 235 us)
                        float sa[4], sb[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int place = place_in(kk[j]);
                            const char *at = reinterpret_cast<const char *>(lists) + (int64_t)(place >> 1) * pair_bytes;
                            const float *from = reinterpret_cast<const float *>(at + list_off + (place & 1) * 8);
                            if (place < 0) from = a.at(row, index_in(kk[j]));
                            sa[j] = *from;
                            sb[j] = by_key[(int)(kk[j] >> 16) * L::STRIDE + j];
                        }
                        if (c.wsel) put(c.wsel + side2 * plane, lists_x ? sb : sa);
                        if (c.xsel) put(c.xsel + side2 * plane, lists_x ? sa : sb);
                    }
                }
            }
            put(c.c, sum);
        }
    }
}

// ---- host ----------------------------------------------------------------------------------------------------
static int list_cap(int64_t K)
{
    int64_t cap = K / 4 + 64;
    if (cap > K) cap = K;
    return (int)(ceil_div(cap, CHUNK) * CHUNK);
}

// Workgroups of build_kernel: a listed row each, and with a leading share the other rows and the tiles of the transpose.
static int64_t build_items(int64_t N, int64_t K, int64_t M, bool two_sided)
{
    const int64_t longer = N > M ? N : M;
    return two_sided ? N + M + ceil_div(longer, 64) * ceil_div(K, 64) : longer;
}

bool applies(int64_t N, int64_t K, int64_t M)
{
    if (tile_rows(K) == 0 || N * M * K <= 0) return false;
    // A launch holds less than 2^32 threads: calls of more rows stay on the dense tilings.
    if (build_items(N, K, M, true) > UINT32_MAX / BUILD_NT) return false;
    const int choice = option(MAM_OPT_FORWARD_TILING);
    if (choice == MAM_FORWARD_TILING_LISTS) return true;
    return choice == MAM_FORWARD_TILING_AUTO && K >= 128 && N >= 32 && M >= 32 && N * M >= MIN_PRODUCTS / K;
}

// Offsets in the workspace.
struct Layout { size_t lists_x, lists_w, bound_x, bound_w, turned, total; int cap, pad_x, pad_w, turned_ld; };
static Layout layout(int64_t N, int64_t K, int64_t M, int w_layout)
{
    Layout l;
    l.cap = list_cap(K);
    l.pad_x = (int)(ceil_div(N, 64) * 64);
    l.pad_w = w_layout == MAM_W_MK ? (int)(ceil_div(M, 64) * 64) : 0;       // (K, M) weights are not listed
    const size_t chunks = (size_t)l.cap / CHUNK + 1;
    size_t at = 8192;             // decision, samples
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) / 256 * 256;
        return here;
    };
    l.lists_x = take((size_t)l.cap * 8 * l.pad_x);
    l.lists_w = take((size_t)l.cap * 8 * l.pad_w);
    l.bound_x = take(chunks * 4 * l.pad_x);
    l.bound_w = take(chunks * 4 * l.pad_w);
    // the transposed operand is addressed with 32-bit byte offsets, its row length in 24 bits
    l.turned_ld = l.pad_x > l.pad_w ? l.pad_x : l.pad_w;
    if (w_layout != MAM_W_MK || tile_rows(K) < 8 || (N * K * M < MIN_TWO_SIDED && option(MAM_OPT_FORWARD_TILING) != MAM_FORWARD_TILING_LISTS) ||
        (size_t)l.turned_ld * 4 >= (1u << 24) || (size_t)l.turned_ld * 4 * K >= ((size_t)1 << 32)) l.turned_ld = 0;
    if (l.turned_ld == 0) l.turned = at;
    else l.turned = take((size_t)l.turned_ld * 4 * K);
    l.total = at;
    return l;
}

size_t workspace_bytes(int64_t N, int64_t K, int64_t M, int w_layout) { return layout(N, K, M, w_layout).total; }

template <int TB, bool TWO>
static int launch_forward(const Params &p, hipStream_t st)
{
    const size_t lds = (size_t)p.call.K * TB * 4 + (TWO ? LEAD_CAP * TB * 8 : 0);
    const int N = (int)p.call.N, M = (int)p.call.M;
    const int tx = (int)ceil_div(M, TB), tw = (int)ceil_div(N, TB);
    const int64_t bx = (int64_t)tx * splits_of(TB, N, tx, p.cus), bw = (int64_t)tw * splits_of(TB, M, tw, p.cus);
    const unsigned blocks = (unsigned)(bx > bw || p.call.w_layout != MAM_W_MK ? bx : bw);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(NT), lds, st, p); };
    // The 32 words that neighbouring lanes store are whole half lines in memory, 64 bytes, only where rows of c start such halves.  Elsewhere
    // the five or seven planes of a one-sided search had better leave them to the L2 (past it / to it, us: 12608 x 768 -> 3004 862 / 718, -> 3032 727 /
    // 715, -> 3024 561 / 696, -> 3040 559 / 619; 16384 x 4096 -> 1001 444 / 374, -> 1000 390 / 374, -> 1008 368 / 382, -> 1024 353 / 364); the values
    // alone go past it either way (-> 1001 253 / 261, 12608 x 768 -> 3004 401 / 402), and two-sided searches do (12608 x 768 -> 3001 2058 / 2148, 16384 x
    // 2048 -> 1000 645 / 670).
    const Call &c = p.call;
    const bool halves = c.M % 16 == 0 && (((uintptr_t)c.c | (uintptr_t)c.argmax | (uintptr_t)c.argmin | (uintptr_t)c.wsel | (uintptr_t)c.xsel) & 63) == 0;
    constexpr bool always = TWO, never = TB == 16;      // (16 rows: no lines by the layout)
    if (!c.argmax) launch(forward_kernel<TB, false, TWO, true>);
    else if (always || (halves && !never)) launch(forward_kernel<TB, true, TWO, !never>);
    else launch(forward_kernel<TB, true, TWO, always>);
    return check_launch("ordered::forward_kernel");
}

static int setup_device(int)
{
    const void *kernels[] = {
        (const void *)forward_kernel<4, true, false, true>,   (const void *)forward_kernel<4, true, false, false>,
        (const void *)forward_kernel<8, true, false, true>,   (const void *)forward_kernel<8, true, false, false>,
        (const void *)forward_kernel<32, true, false, true>,  (const void *)forward_kernel<32, true, false, false>,
        (const void *)forward_kernel<16, true, false, false>, (const void *)forward_kernel<8, true, true, true>,
        (const void *)forward_kernel<4, false, false, true>,  (const void *)forward_kernel<8, false, false, true>,
        (const void *)forward_kernel<16, false, false, true>, (const void *)forward_kernel<32, false, false, true>,
        (const void *)forward_kernel<8, false, true, true>};
    for (const void *k : kernels)
        if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 158 * 1024) != hipSuccess) {
            (void)hipGetLastError();
            return fail(MAM_ERR_LAUNCH, "could not raise the LDS limit of the list kernels");
        }
    return MAM_OK;
}
static DeviceHookRegistration g_registration(setup_device);

static Times::Side side_times(int64_t listed, int64_t tiled, int64_t K, bool args, bool search_x, bool two_sided, int cus)
{
    const int tb = two_sided ? TWO_SIDED_ROWS : tile_rows(K);
    const int tiles = (int)ceil_div(tiled, tb), splits = splits_of(tb, (int)listed, tiles, cus);
    const int per_split = (int)ceil_div(ceil_div(listed, 256 / tb), splits), waves = NT / 64, last = per_split % waves;
    const float alone = two_sided ? 0.45f : 0.3f;                // of a full round's time, by a single wave
    const float rounds = (float)(per_split / waves) + (last ? alone + (1.0f - alone) * (float)last / (float)waves : 0.0f);
    const float lds = (float)K * (float)tb * 4.0f + (two_sided ? (float)(LEAD_CAP * TWO_SIDED_ROWS * 8) : 0.0f);
    const float load = 4.4e-4f * (float)K * (float)tb * (lds <= 80.0f * 1024.0f ? 0.5f : 1.0f);     // (the fit's: a CU holds one workgroup, by registers, whatever its tile)
    float workgroups = (float)tiles * (float)splits / (float)cus;
    workgroups = workgroups < 4.0f ? ceilf(workgroups) : workgroups + 0.3f;
    const float row = 1e-3f + (K > 16 * BUILD_NT ? 1.4e-6f : 0.95e-6f) * (float)K;
    Times::Side s;
    s.fixed = 4.0f + row * (float)listed + workgroups * load;
    if (two_sided) s.fixed += 0.9f * row * (float)tiled + 4.4e-6f * (float)K * (float)listed;       // lists of the leading entries, transpose
    s.per_entry = 5.3e-6f * (float)listed;
    s.rounds = workgroups * rounds;
    s.round = args ? 6.0f + (search_x ? 0.0f : 0.1f * (float)tb) : 4.0f;                            // (with w searched the stores are columns)
    return s;
}
static Times times_of(const Call &c, int cus)
{
    const bool args = c.argmax != nullptr;
    const int64_t m64 = ceil_div(c.M, 64);
    const bool narrow = m64 % 2 == 1 && m64 <= 5;                // 64 neurons per tile
    const float K = (float)c.K, per = (args ? 0.043f + 11.0f / K : 0.036f + 1.5f / K) * (narrow ? (args ? 1.3f : 1.1f) : 1.0f);
    Times t;
    t.dense = (float)(ceil_div(c.N, 32) * 32) * (float)(narrow ? m64 * 64 : ceil_div(m64, 2) * 128) * K * per * 1e-6f;
    t.product = args ? 0.135f : 0.095f;
    t.led = args ? 0.35f : 0.25f;
    t.one_sided[0] = side_times(c.N, c.M, c.K, args, true, false, cus);
    t.one_sided[1] = side_times(c.M, c.N, c.K, args, false, false, cus);
    t.two_sided[0] = side_times(c.N, c.M, c.K, args, true, true, cus);
    t.two_sided[1] = side_times(c.M, c.N, c.K, args, false, true, cus);
    return t;
}

int launch(const Call &call, void *workspace, Guard &guard, hipStream_t st)
{
    Params p;
    p.call = call;
    const int64_t N = call.N, K = call.K, M = call.M;
    const Layout l = layout(N, K, M, call.w_layout);
    char *base = static_cast<char *>(workspace);
    p.decision = reinterpret_cast<Decision *>(base);
    p.samples = reinterpret_cast<int *>(base + 256);
    p.lists_x = reinterpret_cast<uint4 *>(base + l.lists_x);
    p.lists_w = reinterpret_cast<uint4 *>(base + l.lists_w);
    p.bound_x = reinterpret_cast<float *>(base + l.bound_x);
    p.bound_w = reinterpret_cast<float *>(base + l.bound_w);
    p.turned = reinterpret_cast<float *>(base + l.turned);
    p.turned_ld = l.turned_ld;
    p.cap = l.cap;
    p.pad_x = l.pad_x;
    p.pad_w = l.pad_w;
    guard.decision = p.decision;

    p.cus = num_cus();
    p.times = times_of(call, p.cus);
    const int64_t items = call.w_layout == MAM_W_MK ? build_items(N, K, M, p.turned_ld > 0) : N;
    p.decided = p.turned_ld > 0 || items > MAX_UNDECIDED;
    p.any_size = option(MAM_OPT_FORWARD_TILING) == MAM_FORWARD_TILING_LISTS;
    if (K <= 4 * BUILD_NT) hipLaunchKernelGGL((sample_kernel<4>), dim3(SAMPLES), dim3(BUILD_NT), 0, st, p);
    else if (K <= 16 * BUILD_NT) hipLaunchKernelGGL((sample_kernel<16>), dim3(SAMPLES), dim3(BUILD_NT), 0, st, p);
    else hipLaunchKernelGGL((sample_kernel<40>), dim3(SAMPLES), dim3(BUILD_NT), 0, st, p);
    int rc = check_launch("ordered::sample_kernel");
    if (rc != MAM_OK) return rc;
    if (p.decided) {
        hipLaunchKernelGGL(decide_kernel, dim3(1), dim3(64 * LEADS), 0, st, p);
        rc = check_launch("ordered::decide_kernel");
        if (rc != MAM_OK) return rc;
    }
    const dim3 build_grid((unsigned)items), build_block(BUILD_NT);
    const size_t lds = (size_t)p.cap * 8;
    if (K <= 4 * BUILD_NT) hipLaunchKernelGGL((build_kernel<4>), build_grid, build_block, lds, st, p);
    else if (K <= 8 * BUILD_NT) hipLaunchKernelGGL((build_kernel<8>), build_grid, build_block, lds, st, p);
    else if (K <= 16 * BUILD_NT) hipLaunchKernelGGL((build_kernel<16>), build_grid, build_block, lds, st, p);
    else hipLaunchKernelGGL((build_kernel<40>), build_grid, build_block, lds, st, p);
    rc = check_launch("ordered::build_kernel");
    if (rc != MAM_OK) return rc;
    switch (tile_rows(K)) {
        case 32: rc = launch_forward<32, false>(p, st); break;
        case 16: rc = launch_forward<16, false>(p, st); break;
        case 8: rc = launch_forward<8, false>(p, st); break;
        default: return launch_forward<4, false>(p, st);
    }
    // Narrow tiles for the leading entries: 32 searched rows per wave, 128 contiguous bytes (12608 x 768 -> 3072, normal
    // weights: 1740 / 1515 / 1206 us with 32 / 16 / 8 tile rows, 1730 us dense).
    return rc != MAM_OK || p.turned_ld == 0 ? rc : launch_forward<TWO_SIDED_ROWS, true>(p, st);
}

}  // namespace ordered
}  // namespace mam
