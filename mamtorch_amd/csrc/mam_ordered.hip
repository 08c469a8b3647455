// MAM forward by magnitude-ordered lists: most products of a MAM neuron are never formed.
//
// max_k(x_k w_k) is attained where |x_k| or |w_k| is large.  Take the entries of a row of x by falling |x_k|;
// once `best` is the largest product seen and U bounds every |x_k| not yet seen, fl(|x_k w_k|) <= fl(U * max|w|)
// for all of those, and U * max|w| < best ends the search: nothing unseen can reach, or tie with, the maximum
// (the same for the minimum with -best).  For x ~ N(0,1) and W ~ U(-a,a) 0.7 % of 4096 products decide an
// output on average and 2.1 % decide 99 % of them; with normal weights 10 %.  The roles may be swapped: lists of
// the rows of w, bounded by max|x|.  Results are those of the scan over every k, bit for bit.
//
// Four launches, all decisions on the device:
//   sample_kernel  64 outputs computed in full: how long would their lists have to be, on either side?  Every
//                  later kernel of the call reads these 64 pairs and takes the same decision from them: lists of
//                  x, lists of w, or (when products of a call do not fall off that way: constant magnitudes,
//                  all-positive products) neither, and then the dense kernels run instead.
//   build_kernel   a workgroup per listed row: counting sort of the leading entries by magnitude (512 buckets over 4
//                  octaves), written chunk by chunk with the bound U of what follows each chunk.
//   forward_kernel the search itself (below).
//   dense kernels  exit at once unless the decision was "neither".
//
// Measured against the dense tilings (forward call, hand-over arrays written): 207 -> 66 us at 256 x 4096 x 4096,
// 1.70 -> 0.61 ms and 1.47 -> 0.24 ms for 12608 x 768 -> 3072 -> 768, 10.2 -> 0.82 ms (values only) and 3.13 -> 0.40 ms
// at 16384 x 4096 -> 4096 / 1024.  A wave's search ends with the slowest of its 256 outputs: 92 entries at K = 4096
// where the mean output needs 28.
#include "mam_ordered.h"

namespace mam {
namespace ordered {

constexpr int BUCKETS = 512;          // 128 per octave below the row's largest magnitude
constexpr int BUCKET_SHIFT = 16;
constexpr int BUILD_NT = 256;         // threads of the build, per listed row
constexpr int BUILD_MAX_K = 40 * BUILD_NT;
constexpr int BUILD_MAX_CHUNKS = BUILD_MAX_K * 3 / 8 / CHUNK + 16;
constexpr int NT = 1024;              // threads of the forward
constexpr int MAX_TILE_BYTES = 152 * 1024;
// N * K * M from which a call takes the lists: sampling, lists and the idle dense launches cost ~35 us, which a
// call that then goes to the dense tilings (200 us for 2^32 products) pays as well
constexpr int64_t MIN_PRODUCTS = 1ll << 32;
constexpr uint32_t INF_BITS = 0x7f800000u;

struct Params {
    Call call;
    const Sample *samples;
    uint4 *lists;          // [entry pair][listed row]: (value, key, value, key)
    float *bound;          // [chunk][listed row]: bound on the magnitudes from this chunk on
    int limit;             // longest list a sample may ask for
    int cap;               // entries a list can hold (a multiple of CHUNK)
    int rows_pad;          // listed rows, padded, of the longer operand
    int splits_x, splits_w;   // row ranges per tile when x (w) is listed
};

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

// entries written per list, from the longest sampled need: twice that and 64 more, so that hardly any of the
// outputs that are finished one by one need more than their list (the full scan of an output costs ~20 us, 64
// entries more of its list 1 us)
__device__ __forceinline__ int list_length(const Params &p, int longest)
{
    const int want = (longest * 2 + 64 + CHUNK - 1) / CHUNK * CHUNK;
    return want < p.cap ? want : p.cap;
}

// ---- sampling ----------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sample_kernel(const Params p, Sample *out)
{
    __shared__ float red[4][4];
    __shared__ int cnt[4][2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const Call &c = p.call;
    const int K = (int)c.K;
    const uint32_t i = blockIdx.x;
    const int n = (int)((uint64_t)(i * 2 + 1) * (uint64_t)c.N / (2 * SAMPLES));
    const int m = (int)((((uint64_t)(i * 2654435769u)) * (uint64_t)c.M) >> 32);
    const Rows xr = x_rows(c), wr = w_rows(c);
    float hi = -__builtin_inff(), lo = __builtin_inff(), ax = 0.0f, aw = 0.0f;
#pragma unroll 4
    for (int k = threadIdx.x; k < K; k += 256) {
        const float a = *xr.at(n, k), b = *wr.at(m, k), q = a * b;
        hi = __builtin_fmaxf(hi, q);
        lo = __builtin_fminf(lo, q);
        ax = __builtin_fmaxf(ax, __builtin_fabsf(a));
        aw = __builtin_fmaxf(aw, __builtin_fabsf(b));
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        hi = __builtin_fmaxf(hi, __shfl_xor(hi, s));
        lo = __builtin_fminf(lo, __shfl_xor(lo, s));
        ax = __builtin_fmaxf(ax, __shfl_xor(ax, s));
        aw = __builtin_fmaxf(aw, __shfl_xor(aw, s));
    }
    if (lane == 0) { red[wave][0] = hi; red[wave][1] = lo; red[wave][2] = ax; red[wave][3] = aw; }
    __syncthreads();
    hi = __builtin_fmaxf(__builtin_fmaxf(red[0][0], red[1][0]), __builtin_fmaxf(red[2][0], red[3][0]));
    lo = __builtin_fminf(__builtin_fminf(red[0][1], red[1][1]), __builtin_fminf(red[2][1], red[3][1]));
    ax = __builtin_fmaxf(__builtin_fmaxf(red[0][2], red[1][2]), __builtin_fmaxf(red[2][2], red[3][2]));
    aw = __builtin_fmaxf(__builtin_fmaxf(red[0][3], red[1][3]), __builtin_fmaxf(red[2][3], red[3][3]));
    const float reach = __builtin_fminf(hi, -lo);      // a bound below this ends both searches
    int nx = 0, nw = 0;
#pragma unroll 4
    for (int k = threadIdx.x; k < K; k += 256) {
        nx += !(__builtin_fabsf(*xr.at(n, k)) * aw < reach);
        nw += !(__builtin_fabsf(*wr.at(m, k)) * ax < reach);
    }
    nx = wave_sum(nx);
    nw = wave_sum(nw);
    if (lane == 0) { cnt[wave][0] = nx; cnt[wave][1] = nw; }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[i].need_x = cnt[0][0] + cnt[1][0] + cnt[2][0] + cnt[3][0];
        out[i].need_w = cnt[0][1] + cnt[1][1] + cnt[2][1] + cnt[3][1];
    }
}

// ---- lists -------------------------------------------------------------------------------------------------
// A workgroup per listed row, R elements per thread in registers.  Rows of one 64-byte piece of the list array
// are built on one XCD.
template <int R>
__global__ __launch_bounds__(BUILD_NT) void build_kernel(const Params p)
{
    constexpr int WAVES = BUILD_NT / 64;
    extern __shared__ uint4 lds[];          // [cap] (value, key) pairs
    __shared__ uint32_t hist[BUCKETS];
    __shared__ uint32_t part[WAVES], part2[WAVES];
    __shared__ uint32_t chunk_top[BUILD_MAX_CHUNKS];
    uint2 *items = reinterpret_cast<uint2 *>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int longest;
    const int side = decide(p.samples, p.limit, lane, longest);
    if (side == SIDE_NONE) return;
    const Rows rows = side == SIDE_X ? x_rows(p.call) : w_rows(p.call);
    if ((int)blockIdx.x >= rows.rows) return;
    const int row = xcd_remap(blockIdx.x, rows.rows);
    const int len = list_length(p, longest), chunks = len / CHUNK;
    const int K = (int)p.call.K;
    const float *src = rows.at(row, 0);

    float v[R];
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int k = t * BUILD_NT + tid;
        v[t] = k < K ? src[k * rows.k_stride] : 0.0f;
    }
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
    // exclusive prefix over the buckets, BUCKETS / BUILD_NT consecutive ones per thread
    constexpr int BPT = BUCKETS / BUILD_NT;
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
    if (lane == 63) part2[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
#pragma unroll
    for (int i = 0; i < WAVES - 1; ++i) run += i < wave ? part2[i] : 0u;
    int open = 0;                 // buckets that start inside the list
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        hist[tid * BPT + j] = run;
        open += run < (uint32_t)len;
        run += own[j];
    }
    open = wave_sum(open);
    if (lane == 0) part[wave] = (uint32_t)open;
    __syncthreads();
    open = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) open += (int)part[i];
    uint32_t rest = 0;            // largest magnitude that is not listed
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const uint32_t bits = __float_as_uint(v[t]) & 0x7fffffffu;
        const uint32_t b = (top - bits) >> BUCKET_SHIFT;
        const int k = t * BUILD_NT + tid;
        bool listed = false;
        if (b < (uint32_t)open && k < K) {
            const uint32_t at = atomicAdd(&hist[b], 1u);
            if (at < (uint32_t)len) {
                items[at] = make_uint2(__float_as_uint(v[t]), key((uint32_t)k, at + 1));
                listed = true;
            }
        }
        if (!listed) rest = bits > rest ? bits : rest;
    }
    rest = (uint32_t)wave_max((int)rest);
    if (lane == 0) part2[wave] = rest;
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
    for (int j = tid; j < len / 2; j += BUILD_NT) p.lists[(int64_t)j * p.rows_pad + row] = lds[j];
    __syncthreads();
    if (wave != 0) return;
    // bound[c] = largest magnitude from chunk c on.  A row with a NaN or an infinity gets NaN (never finished by a
    // bound), a row of zeros -1 (finished at once: see the forward).
#pragma unroll
    for (int i = 0; i < WAVES; ++i) rest = part2[i] > rest ? part2[i] : rest;
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
        if (c <= chunks) p.bound[(int64_t)c * p.rows_pad + row] = special ? instead : __uint_as_float(tail);
    }
}

// ---- search ------------------------------------------------------------------------------------------------
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
__device__ __forceinline__ double shfl_xor64(double d, int s)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, d);
    const uint32_t lo = __shfl_xor((uint32_t)b, s), hi = __shfl_xor((uint32_t)(b >> 32), s);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
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
    static __device__ __forceinline__ void merge(value &a, value &b, int s)
    {
        max64(a, shfl_xor64(a, s));
        min64(b, shfl_xor64(b, s));
    }
    // one pair of list entries against 4 tile values each.  Written out because the compiler copies the key into the low
    // word of every key: here two register pairs hold it for the four products of an entry.
    __device__ __forceinline__ void entry(float x, uint32_t key, const float4 &w)
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
    __device__ __forceinline__ void entries(const uint4 &it, const float4 &w0, const float4 &w1)
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
    static __device__ __forceinline__ void merge(value &a, value &b, int s)
    {
        a = __builtin_fmaxf(a, __shfl_xor(a, s));
        b = __builtin_fminf(b, __shfl_xor(b, s));
    }
    __device__ __forceinline__ void entries(const uint4 &it, const float4 &w0, const float4 &w1)
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

// One output by the whole wave: first the rest of its list, 64 entries at a time, then (the list is not enough,
// or the row or the tile column holds what no bound covers: NaN, infinity, a zero extreme) every k, in the exact
// terms of the ascending scan with ordered strict compares.
//   column: the output's column of the tile, by 65535 - k; at: chunks already searched; bmax: bound on the tile column
template <int TB, class E>
__device__ __forceinline__ void finish_one(const Params &p, const Rows &a, int row, const float *column, int at, int chunks,
                                           float bmax, int lane, typename E::value &mx, typename E::value &mn)
{
    for (int ch = at; ch < chunks; ch += 64 / CHUNK) {
        const int e = ch * CHUNK + lane;
        const int next = (ch + 64 / CHUNK) < chunks ? ch + 64 / CHUNK : chunks;
        const float u = p.bound[(int64_t)next * p.rows_pad + row] * bmax;
        if (e < chunks * CHUNK) {
            const uint2 it = reinterpret_cast<const uint2 *>(p.lists + (int64_t)(e >> 1) * p.rows_pad + row)[e & 1];
            E::both(mx, mn, __uint_as_float(it.x) * column[(int)(it.y >> 16) * TB], it.y);
        }
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) E::merge(mx, mn, s);
        if (E::product(mx) > u && E::product(mn) < -u) return;
    }
    float hi = -__builtin_inff(), lo = __builtin_inff();
    int ih = INT32_MAX, il = INT32_MAX;
    const int K = (int)p.call.K;
    const float *src = a.at(row, 0);
    for (int k0 = 0; k0 < K; k0 += 64 * 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + i * 64 + lane;
            v[i] = src[(k < K ? k : K - 1) * a.k_stride];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int past = k0 + i * 64 + lane, k = past < K ? past : K - 1;     // past the end the last k again
            const float q = v[i] * column[(65535 - k) * TB];
            if (q > hi) { hi = q; ih = k; }
            if (q < lo) { lo = q; il = k; }
        }
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const float oh = __shfl_xor(hi, s), ol = __shfl_xor(lo, s);
        const int jh = __shfl_xor(ih, s), jl = __shfl_xor(il, s);
        if (oh > hi || (oh == hi && jh < ih)) { hi = oh; ih = jh; }
        if (ol < lo || (ol == lo && jl < il)) { lo = ol; il = jl; }
    }
    // an extreme that was never improved keeps the first k
    mx = E::make(hi, ih == INT32_MAX ? 0 : ih);
    mn = E::make(lo, il == INT32_MAX ? 0 : il);
}

// A workgroup holds a tile of TB rows of the other operand in LDS, whole rows, as [K - 1 - k][TB] (a key's upper half
// is then the address but for a constant); a lane owns one
// listed row x 4 consecutive tile rows, and TB / 4 neighbouring lanes share a listed row, so that an entry costs
// each lane one 16-byte LDS read for 4 products and the lanes of a row read TB * 4 contiguous bytes.  Waves take
// blocks of 64 * 4 / TB listed rows in turn and need no barrier after the tile is loaded.  A wave looks at its
// lists chunk by chunk until all but FEW of its 256 outputs are finished by their bound, and then finishes those
// one by one with all its lanes (FEW = 0, 1, 2, 4: 75 / 72 / 72 / 73 us at 256 x 4096 x 4096, 608 / 593 / 593 / 602 us at
// 16384 x 4096 -> 1024, while the selected operands still came from the row).  Bound: v_max_f64 / v_min_f64, ~13 of the ~17 cycles per product and SIMD; the random 16-byte
// LDS reads take half of that.  (9.9 T products/s in a loop of its own against 14.3 T with fp32 extremes and no
// indices.)
constexpr int FEW = 2;

template <int TB, bool ARGS>
__global__ __launch_bounds__(NT) void forward_kernel(const Params p)
{
    typedef Extremes<ARGS> E;
    constexpr int Q = TB / 4;               // lanes per listed row
    constexpr int RW = 64 / Q;              // listed rows per wave
    extern __shared__ float tile[];         // [K][TB], k descending
    __shared__ float tops[TB];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int longest;
    const int side = decide(p.samples, p.limit, lane, longest);
    if (side == SIDE_NONE) return;
    const Call &c = p.call;
    const bool lists_x = side == SIDE_X;
    const Rows a = lists_x ? x_rows(c) : w_rows(c), b = lists_x ? w_rows(c) : x_rows(c);
    const int K = (int)c.K;
    const int tiles = (b.rows + TB - 1) / TB, splits = lists_x ? p.splits_x : p.splits_w;
    if ((int)blockIdx.x >= tiles * splits) return;
    const int logical = xcd_remap(blockIdx.x, tiles * splits);
    const int split = logical / tiles, b0 = (logical - split * tiles) * TB;
    const int chunks = list_length(p, longest) / CHUNK;

    // ---- tile: rows b0 .. b0 + TB - 1 (past the end: the last one again), and the largest magnitude of each ----
    // (bit patterns of magnitudes order as integers; infinities and NaN stay on top)
    uint32_t top[4] = {0, 0, 0, 0};
    auto see = [&](int i, float v) {
        const uint32_t bits = __float_as_uint(v) & 0x7fffffffu;
        top[i] = bits > top[i] ? bits : top[i];
    };
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
            *reinterpret_cast<float4 *>(&tile[(K - 1 - k) * TB + my_quad * 4]) = v;
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
            *reinterpret_cast<float4 *>(&tile[(K - 1 - k) * TB + my_quad * 4]) = v;
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
    const int q = lane % Q;
    float bmax[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float t = tops[q * 4 + j];
        bmax[j] = t == 0.0f ? -1.0f : t < __builtin_inff() ? t : __builtin_nanf("");
    }
    const float *by_key = tile + (K - 65536) * TB;      // element (65535 - k) * TB + row
    const char *mine = reinterpret_cast<const char *>(by_key) + q * 16;
    const int64_t pair_bytes = (int64_t)p.rows_pad * 16, bound_bytes = (int64_t)p.rows_pad * 4;

    const bool whole = b0 + q * 4 + 3 < b.rows && (c.M & 3) == 0;
    const uint32_t lane_off = lists_x ? (uint32_t)(lane / Q) * (uint32_t)c.M + q * 4 : q * 4 * (uint32_t)c.M + lane / Q;

    const int blocks = (a.rows + RW - 1) / RW;
    const int per_split = (blocks + splits - 1) / splits;
    const int last = (split + 1) * per_split < blocks ? (split + 1) * per_split : blocks;
    for (int blk = split * per_split + wave; blk < last; blk += NT / 64) {
        const int arow = blk * RW + lane / Q;
        const int row = arow < a.rows ? arow : a.rows - 1;
        const uint32_t list_off = (uint32_t)row * 16u, bound_off = (uint32_t)row * 4u;
        E e;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            e.mx[j] = E::low();
            e.mn[j] = E::high();
        }
        int ch = 0;
        uint64_t open[4];
        auto fetch = [&](uint4 (&to)[CHUNK / 2], int chunk) {
            const char *base = reinterpret_cast<const char *>(p.lists) + (int64_t)chunk * (CHUNK / 2) * pair_bytes;
            asm volatile("" : "+s"(base));      // scalar base + 32-bit lane offset
#pragma unroll
            for (int i = 0; i < CHUNK / 2; ++i) to[i] = *reinterpret_cast<const uint4 *>(base + i * pair_bytes + list_off);
        };
        // true when the search is over
        auto step = [&](const uint4 (&cur)[CHUNK / 2], uint4 (&nxt)[CHUNK / 2]) {
            fetch(nxt, ch + 1 < chunks ? ch + 1 : ch);
            const float u = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(p.bound) + (ch + 1) * bound_bytes + bound_off);
            asm volatile("" ::: "memory");      // the loads stay ahead of the arithmetic
#pragma unroll
            for (int i = 0; i < CHUNK / 2; ++i) {
                const float4 w0 = *reinterpret_cast<const float4 *>(mine + (int)(cur[i].y >> 16) * (TB * 4));
                const float4 w1 = *reinterpret_cast<const float4 *>(mine + (int)(cur[i].w >> 16) * (TB * 4));
                e.entries(cur[i], w0, w1);
            }
            ++ch;
            int left = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float ub = u * bmax[j];
                open[j] = ~(__ballot(E::product(e.mx[j]) > ub) & __ballot(E::product(e.mn[j]) < -ub));
                left += __popcll(open[j]);
            }
            return left <= FEW || ch == chunks;
        };
        {
            uint4 first[CHUNK / 2], second[CHUNK / 2];
            fetch(first, 0);
            while (true) {
                if (step(first, second)) break;
                if (step(second, first)) break;
            }
        }
        while (open[0] | open[1] | open[2] | open[3]) {
            // (one copy of the code: the output's state is picked by selects)
            const int j = open[0] ? 0 : open[1] ? 1 : open[2] ? 2 : 3;
            const int l = __builtin_ctzll(open[0] ? open[0] : open[1] ? open[1] : open[2] ? open[2] : open[3]);
            typename E::value fx = lane_value(j == 0 ? e.mx[0] : j == 1 ? e.mx[1] : j == 2 ? e.mx[2] : e.mx[3], l);
            typename E::value fn = lane_value(j == 0 ? e.mn[0] : j == 1 ? e.mn[1] : j == 2 ? e.mn[2] : e.mn[3], l);
            const float bm = lane_value(j == 0 ? bmax[0] : j == 1 ? bmax[1] : j == 2 ? bmax[2] : bmax[3], l);
            finish_one<TB, E>(p, a, __builtin_amdgcn_readlane(row, l), by_key + (l % Q) * 4 + j, ch, chunks, bm, lane, fx, fn);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i == j) {
                    open[i] &= open[i] - 1;
                    if (lane == l) { e.mx[i] = fx; e.mn[i] = fn; }
                }
        }
        // ---- outputs ----
        if (arow < a.rows) {
            const float u0 = p.bound[row];
            const int64_t plane = c.N * c.M;
            float sum[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if ((u0 == -1.0f) != (bmax[j] == -1.0f) && u0 == u0 && bmax[j] == bmax[j]) {
                    const float z = *a.at(row, 0) * tile[(K - 1) * TB + q * 4 + j];
                    e.mx[j] = e.mn[j] = E::make(z, 0);
                }
                sum[j] = E::product(e.mx[j]) + E::product(e.mn[j]);
                const int m = lists_x ? b0 + q * 4 + j : arow;
                if (c.bias && m < (int)c.M) sum[j] = sum[j] + c.bias[m];
            }
            // uniform base of the block + 32-bit offset of the lane
            const int64_t base = lists_x ? (int64_t)blk * RW * c.M + b0 : (int64_t)b0 * c.M + blk * RW;
            auto put = [&](float *dst, const float (&v)[4]) {
                float *to = dst + base;
                if (lists_x) {
                    if (whole && ((uintptr_t)dst & 15) == 0) {
                        *reinterpret_cast<float4 *>(to + lane_off) = make_float4(v[0], v[1], v[2], v[3]);
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (b0 + q * 4 + j < b.rows) to[lane_off + j] = v[j];
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (b0 + q * 4 + j < b.rows) to[lane_off + j * (uint32_t)c.M] = v[j];
                }
            };
            if constexpr (ARGS) {
#pragma unroll
                for (int side2 = 0; side2 < 2; ++side2) {
                    uint32_t kk[4];
                    float f[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        kk[j] = key_of(side2 ? e.mn[j] : e.mx[j]);
                        f[j] = __int_as_float(index_in(kk[j]));
                    }
                    put(reinterpret_cast<float *>(side2 ? c.argmin : c.argmax), f);
                    if (c.wsel) {
                        // the selected operands, of the tile and of the listed row: from the list, which this
                        // XCD's L2 still holds, rather than from anywhere in the row (16384 x 4096 -> 1024: 593 ->
                        // 405 us, 12608 x 3072 -> 768: 345 -> 235 us)
                        float sa[4], sb[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int place = place_in(kk[j]);
                            const char *at = reinterpret_cast<const char *>(p.lists) + (int64_t)(place >> 1) * pair_bytes;
                            const float *from = reinterpret_cast<const float *>(at + list_off + (place & 1) * 8);
                            if (place < 0) from = a.at(row, index_in(kk[j]));
                            sa[j] = *from;
                            sb[j] = by_key[(int)(kk[j] >> 16) * TB + q * 4 + j];
                        }
                        put(c.wsel + side2 * plane, lists_x ? sb : sa);
                        put(c.xsel + side2 * plane, lists_x ? sa : sb);
                    }
                }
            }
            put(c.c, sum);
        }
    }
}

// ---- host ----------------------------------------------------------------------------------------------------
// rows of the tile operand per workgroup: as many as fit the LDS as whole rows (0: not even 4)
static int tile_rows(int64_t K)
{
    for (int tb = 32; tb >= 4; tb /= 2)
        if (K * tb * 4 <= MAX_TILE_BYTES) return tb;
    return 0;
}

static int list_cap(int64_t K)
{
    int64_t cap = K * 3 / 8;
    if (cap < 128) cap = 128;
    if (cap > K) cap = K;
    return (int)(ceil_div(cap, CHUNK) * CHUNK);
}

bool applies(int64_t N, int64_t K, int64_t M)
{
    if (tile_rows(K) == 0 || N * M * K <= 0 || M > (1 << 24)) return false;
    const int choice = option(MAM_OPT_FORWARD_TILING);
    if (choice == MAM_FORWARD_TILING_LISTS) return true;
    return choice == MAM_FORWARD_TILING_AUTO && K >= 128 && N >= 32 && M >= 32 && N * M >= MIN_PRODUCTS / K;
}

static int64_t rows_padded(int64_t N, int64_t M) { return ceil_div(N > M ? N : M, 64) * 64; }

size_t workspace_bytes(int64_t N, int64_t K, int64_t M)
{
    const size_t cap = (size_t)list_cap(K), rows = (size_t)rows_padded(N, M);
    return 1024 + cap * 8 * rows + ceil_div((cap / CHUNK + 1) * rows * 4, 256) * 256;
}

template <int TB>
static int launch_forward(const Params &p, unsigned blocks, hipStream_t st)
{
    const size_t lds = (size_t)p.call.K * TB * 4;
    if (p.call.argmax)
        hipLaunchKernelGGL((forward_kernel<TB, true>), dim3(blocks), dim3(NT), lds, st, p);
    else
        hipLaunchKernelGGL((forward_kernel<TB, false>), dim3(blocks), dim3(NT), lds, st, p);
    return check_launch("ordered::forward_kernel");
}

static int setup_device(int)
{
    const void *kernels[] = {
        (const void *)forward_kernel<4, true>, (const void *)forward_kernel<8, true>, (const void *)forward_kernel<16, true>,
        (const void *)forward_kernel<32, true>, (const void *)forward_kernel<4, false>, (const void *)forward_kernel<8, false>,
        (const void *)forward_kernel<16, false>, (const void *)forward_kernel<32, false>,
        (const void *)build_kernel<4>, (const void *)build_kernel<8>, (const void *)build_kernel<16>, (const void *)build_kernel<40>};
    for (const void *k : kernels)
        if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_TILE_BYTES) != hipSuccess) {
            (void)hipGetLastError();
            return fail(MAM_ERR_LAUNCH, "could not raise the LDS limit of the list kernels");
        }
    return MAM_OK;
}
static DeviceHookRegistration g_registration(setup_device);

int launch(const Call &call, void *workspace, Guard &guard, hipStream_t st)
{
    Params p;
    p.call = call;
    const int64_t N = call.N, K = call.K, M = call.M;
    char *base = static_cast<char *>(workspace);
    Sample *samples = reinterpret_cast<Sample *>(base);
    p.samples = samples;
    p.cap = list_cap(K);
    p.rows_pad = (int)rows_padded(N, M);
    p.lists = reinterpret_cast<uint4 *>(base + 1024);
    p.bound = reinterpret_cast<float *>(base + 1024 + (size_t)p.cap * 8 * p.rows_pad);
    // a product found through the lists costs two to three dense ones, and the longest search of a wave's 256
    // outputs is what the wave does: the dense kernels are as fast where the sampled searches reach K / 6
    p.limit = (int)(K / 6);
    guard.samples = samples;
    guard.limit = p.limit;

    const int tb = tile_rows(K);
    const int rw = 256 / tb;                      // listed rows per wave
    auto splits = [&](int64_t listed, int64_t tiled) {
        // three rounds of workgroups over the chip, but at least one block of listed rows per wave
        const int64_t tiles = ceil_div(tiled, tb), blocks = ceil_div(listed, rw);
        int64_t s = ceil_div(3 * num_cus(), tiles);
        const int64_t most = ceil_div(blocks, NT / 64);
        return (int)(s < most ? s : most);
    };
    p.splits_x = splits(N, M);
    p.splits_w = splits(M, N);
    const int64_t bx = ceil_div(M, tb) * p.splits_x, bw = ceil_div(N, tb) * p.splits_w;

    hipLaunchKernelGGL(sample_kernel, dim3(SAMPLES), dim3(256), 0, st, p, samples);
    int rc = check_launch("ordered::sample_kernel");
    if (rc != MAM_OK) return rc;
    const dim3 build_grid((unsigned)(N > M ? N : M)), build_block(BUILD_NT);
    const size_t lds = (size_t)p.cap * 8;
    if (K <= 4 * BUILD_NT) hipLaunchKernelGGL((build_kernel<4>), build_grid, build_block, lds, st, p);
    else if (K <= 8 * BUILD_NT) hipLaunchKernelGGL((build_kernel<8>), build_grid, build_block, lds, st, p);
    else if (K <= 16 * BUILD_NT) hipLaunchKernelGGL((build_kernel<16>), build_grid, build_block, lds, st, p);
    else hipLaunchKernelGGL((build_kernel<40>), build_grid, build_block, lds, st, p);
    rc = check_launch("ordered::build_kernel");
    if (rc != MAM_OK) return rc;
    const unsigned blocks = (unsigned)(bx > bw ? bx : bw);
    switch (tb) {
        case 32: return launch_forward<32>(p, blocks, st);
        case 16: return launch_forward<16>(p, blocks, st);
        case 8: return launch_forward<8>(p, blocks, st);
        default: return launch_forward<4>(p, blocks, st);
    }
}

}  // namespace ordered
}  // namespace mam
