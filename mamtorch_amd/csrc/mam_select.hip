// The pruning threshold on the device (gfx950): the element of a given rank among the absolute scores of
// one or several weight matrices, without sorting them.
//
// The reference finds its thresholds with torch.quantile over one layer's |scores|
// (examples/vitb16_imagenet1k/pruning_utils.py:103-104) or by sorting the concatenated |scores| of every
// layer and taking the element of rank int(p * n) (:139-143): a full sort of 16.8 M (one 4096 x 4096 layer)
// to hundreds of millions of floats for ONE number.  Here the number is found by a radix select over the
// bit patterns of the scores: a non-negative fp32 orders like its bit pattern (NaN above infinity, where
// torch.sort puts it too), so three histogram passes over the 31 key bits (11 + 9 + 11 bits, 2048-bin
// histograms in LDS, flushed to a global histogram with integer atomics) narrow the bins down to the one
// key that holds the rank.  Between two passes a prefix sum over the histogram fixes the digit: for one matrix every workgroup
// of the next pass takes it by itself, for several tensors a launch of one workgroup does, after the last of them.
// One or two ranks are followed at once (torch.quantile interpolates between two neighbours), and the
// passes take any number of tensors, so the global rule needs no concatenated copy.  Every pass streams
// the scores once: 3 x 4 bytes per element (plus the second operand of a product or count score).
//
// Scores are those of the pruning kernels (mam_prune.hip): |w|, |w * aux| or aux (+ aux2) selection counts.
#include "mam_common.h"

namespace mam {
namespace selectk {

constexpr int NT = 256;        // begin / advance
constexpr int NT_H = 1024;     // histogram passes
constexpr int BINS = 2048;
constexpr int MAX_RANKS = 2;
constexpr int PASSES = 3;
constexpr int COPIES = 4;                    // histograms per rank and workgroup
constexpr int AHEAD = 4;                     // loads in flight per thread (8: no faster)
constexpr int COPY_STRIDE = BINS + 9;

struct State {
    uint32_t prefix[MAX_RANKS];     // digits fixed so far, right-aligned
    uint32_t nranks, pad;
    int64_t rank[MAX_RANKS];        // rank still to go within the elements that share the prefix
};
// workspace: a State for each pass to start from, then hist[PASSES][MAX_RANKS][BINS] of 64-bit counts (the tensors of one selection may hold
// more than 2^32 elements together; a workgroup's own LDS bins are 32 bits)
typedef unsigned long long count_t;
constexpr size_t kHistWords = (size_t)PASSES * MAX_RANKS * BINS;
constexpr size_t kStateStride = 2;     // 64 bytes from one to the next
static_assert(sizeof(State) == 32 && (PASSES * kStateStride + 1) * sizeof(State) <= 256, "the states precede the histograms");
constexpr size_t kWorkspaceBytes = 256 + kHistWords * sizeof(count_t);

// Keys are 31 bits wide (absolute values: the sign bit is clear): digits of 11, 9 and 11 bits.  The second pass is the
// narrow one: it still sees a twentieth of the scores, spread over all its bins, and every workgroup adds all of them to
// the global histogram (the third sees some thousand scores in all).
__host__ __device__ constexpr int pass_shift(int pass) { return pass == 0 ? 20 : pass == 1 ? 11 : 0; }
__host__ __device__ constexpr int pass_bits(int pass) { return pass == 1 ? 9 : 11; }

template <int MODE>
__device__ __forceinline__ uint32_t key_of(float w, const void *aux, const void *aux2, int64_t idx)
{
    if (MODE == MAM_PRUNE_MAGNITUDE) return __float_as_uint(w) & 0x7fffffffu;
    if (MODE == MAM_PRUNE_WEIGHT_TIMES) return __float_as_uint(w * static_cast<const float *>(aux)[idx]) & 0x7fffffffu;
    int cnt = static_cast<const int32_t *>(aux)[idx];
    if (aux2) cnt += static_cast<const int32_t *>(aux2)[idx];
    return (uint32_t)(cnt < 0 ? -cnt : cnt);
}

__global__ __launch_bounds__(NT) void begin_kernel(State *st, count_t *hist, int64_t r0, int64_t r1, int nranks)
{
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < kHistWords; i += (size_t)gridDim.x * NT) hist[i] = 0ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->prefix[0] = st->prefix[1] = 0u;
        st->nranks = (uint32_t)nranks;
        st->pad = 0u;
        st->rank[0] = r0;
        st->rank[1] = r1;
    }
}

// What `st` becomes once pass `pass` has seen every score: the digit of each rank, found by a prefix sum of the workgroup over
// the histogram (8.3 -> 3.8 us against one thread that walks the bins).  next: LDS; st may be the state that is written afterwards.
template <int THREADS>
__device__ __forceinline__ void advance(const State *__restrict__ st, const count_t *__restrict__ hist, int pass, State *next)
{
    __shared__ int64_t wave_total[MAX_RANKS][THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nr = (int)st->nranks;
    const uint32_t prefix[MAX_RANKS] = {st->prefix[0], st->prefix[1]};
    const int64_t wanted[MAX_RANKS] = {st->rank[0], st->rank[1]};
    const bool one = nr < 2 || prefix[0] == prefix[1];
    const int nbins = 1 << pass_bits(pass);
    constexpr int per = BINS / THREADS;
    int64_t own[MAX_RANKS][per];
#pragma unroll
    for (int s = 0; s < MAX_RANKS; ++s)
#pragma unroll
        for (int b = 0; b < per; ++b) {
            const count_t *h = hist + ((size_t)pass * MAX_RANKS + (one ? 0 : s)) * BINS;
            own[s][b] = s < nr && tid * per + b < nbins ? (int64_t)h[tid * per + b] : 0;
        }
    int64_t sum[MAX_RANKS], upto[MAX_RANKS];       // elements up to and with this thread's bins
#pragma unroll
    for (int s = 0; s < MAX_RANKS; ++s) {
        sum[s] = 0;
#pragma unroll
        for (int b = 0; b < per; ++b) sum[s] += own[s][b];
        upto[s] = sum[s];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int64_t o = __shfl_up(upto[s], off);
            if (lane >= off) upto[s] += o;
        }
        if (lane == 63) wave_total[s][wave] = upto[s];
    }
    __syncthreads();
    if (tid == 0) {
        next->nranks = (uint32_t)nr;
        next->pad = 0u;
        if (nr < MAX_RANKS) {
            next->prefix[1] = prefix[1];
            next->rank[1] = wanted[1];
        }
    }
#pragma unroll
    for (int s = 0; s < MAX_RANKS; ++s) {
        if (s >= nr) break;
        for (int w = 0; w < wave; ++w) upto[s] += wave_total[s][w];
        const int64_t r = wanted[s], before = upto[s] - sum[s];
        if ((before <= r && r < upto[s]) || (tid == THREADS - 1 && r >= upto[s])) {
            int64_t below = before;
            int digit = tid * per;
#pragma unroll
            for (int b = 0; b < per; ++b)
                if (digit == tid * per + b && digit < nbins - 1 && below + own[s][b] <= r) {
                    below += own[s][b];
                    ++digit;
                }
            next->prefix[s] = (prefix[s] << pass_bits(pass)) | (uint32_t)digit;
            next->rank[s] = r - below;
        }
    }
    __syncthreads();
}

// One histogram pass over one matrix.  CHAINED: the only matrix, st is the state before the last pass, whose histogram is complete; the
// state that follows from it is left behind st for the next pass (4096 x 4096: the steps by themselves 13 us and the gaps between four
// launches, 7 us and one launch here).  vec: 16-byte loads (K a multiple of 4, aligned rows).
template <int MODE, bool CHAINED>
__global__ __launch_bounds__(NT_H) void hist_kernel(const float *__restrict__ w, int64_t ldw, const void *aux,
                                                  const void *aux2, int64_t ld_aux, int64_t M, int64_t K, int vec,
                                                  State *st, count_t *hist, int pass)
{
    // Scores crowd into few bins (the first pass looks at the exponent and three mantissa bits), and an LDS atomic
    // costs per lane that shares an address: neighbouring lanes count into copies of the histogram, which start on
    // different banks.  4096 x 4096 normal scores, the three passes: 22 / 21 / 12 us with one histogram per rank, a
    // register for runs of equal digits, an integer division per load and two workgroups per CU; 17.5 / 17.7 / 14 us
    // like this (12 us: the load of 67 MB).  What is left above the load is the histogram's global atomics.
    __shared__ uint32_t bins[MAX_RANKS][COPIES][COPY_STRIDE];
    const int tid = threadIdx.x;
    if (CHAINED) {
        __shared__ State next;
        advance<NT_H>(st, hist, pass - 1, &next);
        if (blockIdx.x == 0 && tid == 0) st[kStateStride] = next;
        st = &next;
    }
    const int nr = (int)st->nranks;
    const int shift = pass_shift(pass), nb = pass_bits(pass);
    const uint32_t mask = (1u << nb) - 1u;
    const uint32_t p0 = st->prefix[0], p1 = st->prefix[1];
    const bool one = nr < 2 || p0 == p1;     // both ranks still in the same bin: one histogram serves both
    const int used = (one ? 1 : MAX_RANKS) * COPIES * COPY_STRIDE;
    for (int i = tid; i < used; i += NT_H) (&bins[0][0][0])[i] = 0u;
    __syncthreads();
    uint32_t *const mine0 = bins[0][tid % COPIES], *const mine1 = bins[1][tid % COPIES];
    auto count = [&](uint32_t key, uint32_t n) {
        const uint32_t hi = pass == 0 ? 0u : key >> (shift + nb);
        const uint32_t digit = (key >> shift) & mask;
        if (hi == p0) atomicAdd(&mine0[digit], n);
        if (!one && hi == p1) atomicAdd(&mine1[digit], n);
    };
    auto take = [&](uint32_t key) { count(key, 1u); };
    // scores that are equal down to this digit (selection counts: the first two digits of all of them) are added at once
    auto take4 = [&](uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
        const uint32_t t = a >> shift;
        const bool same = t == b >> shift && t == c >> shift && t == d >> shift;
        if (__all(same && t == (uint32_t)__builtin_amdgcn_readfirstlane(t))) {
            const uint64_t lanes = __ballot(1);
            if ((tid & 63) == __builtin_ctzll(lanes)) count(a, 4u * (uint32_t)__popcll(lanes));
        } else if (same) {
            count(a, 4u);
        } else {
            take(a); take(b); take(c); take(d);
        }
    };
    const int64_t stride = (int64_t)gridDim.x * NT_H;
    if (vec) {
        const int64_t q = K >> 2, items = M * q;
        for (int64_t it = (int64_t)blockIdx.x * NT_H + tid; it < items; it += stride * AHEAD) {
            uint4 keys[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {      // past the end: the first item again, not counted
                const int64_t i = it + u * stride < items ? it + u * stride : it;
                const int64_t r = M == 1 ? 0 : i / q, c = (i - r * q) * 4;
                const int64_t a = r * ld_aux + c;
                if (MODE == MAM_PRUNE_COUNT) {
                    int4 cnt = *reinterpret_cast<const int4 *>(static_cast<const int32_t *>(aux) + a);
                    if (aux2) {
                        const int4 c2 = *reinterpret_cast<const int4 *>(static_cast<const int32_t *>(aux2) + a);
                        cnt.x += c2.x; cnt.y += c2.y; cnt.z += c2.z; cnt.w += c2.w;
                    }
                    keys[u] = make_uint4(cnt.x < 0 ? -cnt.x : cnt.x, cnt.y < 0 ? -cnt.y : cnt.y, cnt.z < 0 ? -cnt.z : cnt.z,
                                         cnt.w < 0 ? -cnt.w : cnt.w);
                } else {
                    float4 v = *reinterpret_cast<const float4 *>(w + r * ldw + c);
                    if (MODE == MAM_PRUNE_WEIGHT_TIMES) {
                        const float4 f = *reinterpret_cast<const float4 *>(static_cast<const float *>(aux) + a);
                        v.x *= f.x; v.y *= f.y; v.z *= f.z; v.w *= f.w;
                    }
                    keys[u] = make_uint4(__float_as_uint(v.x) & 0x7fffffffu, __float_as_uint(v.y) & 0x7fffffffu,
                                         __float_as_uint(v.z) & 0x7fffffffu, __float_as_uint(v.w) & 0x7fffffffu);
                }
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                if (it + u * stride < items) take4(keys[u].x, keys[u].y, keys[u].z, keys[u].w);
        }
    } else {
        const int64_t items = M * K;
        for (int64_t it = (int64_t)blockIdx.x * NT_H + tid; it < items; it += stride) {
            const int64_t r = M == 1 ? 0 : it / K, c = it - r * K;
            const float wv = MODE == MAM_PRUNE_COUNT ? 0.0f : w[r * ldw + c];
            take(key_of<MODE>(wv, aux, aux2, r * ld_aux + c));
        }
    }
    __syncthreads();
    count_t *out = hist + (size_t)pass * MAX_RANKS * BINS;
    for (int i = tid; i < (one ? 1 : MAX_RANKS) * BINS; i += NT_H) {
        const int rank = i / BINS, bin = i % BINS;
        uint32_t v = 0;
#pragma unroll
        for (int copy = 0; copy < COPIES; ++copy) v += bins[rank][copy][bin];
        if (v) atomicAdd(&out[i], (count_t)v);
    }
}

// After every tensor has been through pass `pass`.
__global__ __launch_bounds__(NT) void advance_kernel(State *st, const count_t *__restrict__ hist, int pass)
{
    __shared__ State next;
    advance<NT>(st, hist, pass, &next);
    if (threadIdx.x == 0) *st = next;
}

// The last digits are in the histogram yet (CHAINED) or in the state.
template <bool CHAINED>
__global__ __launch_bounds__(NT) void result_kernel(const State *st, const count_t *hist, float *out, int as_count)
{
    const int s = threadIdx.x;
    if (CHAINED) {
        __shared__ State next;
        advance<NT>(st, hist, PASSES - 1, &next);
        st = &next;
    }
    if (s < (int)st->nranks) out[s] = as_count ? (float)(int)st->prefix[s] : __uint_as_float(st->prefix[s]);
}

static count_t *hist_of(void *workspace) { return reinterpret_cast<count_t *>(static_cast<char *>(workspace) + 256); }

}  // namespace selectk
}  // namespace mam

extern "C" size_t mam_select_workspace(void) { return mam::selectk::kWorkspaceBytes; }

extern "C" int mam_select_begin(void *workspace, size_t workspace_bytes, const int64_t *ranks, int nranks, void *stream)
{
    using namespace mam;
    if (!workspace || workspace_bytes < selectk::kWorkspaceBytes || (uintptr_t)workspace % 16 != 0)
        return fail(MAM_ERR_WORKSPACE, "the selection needs %zu workspace bytes, 16-byte aligned", selectk::kWorkspaceBytes);
    if (!ranks || nranks < 1 || nranks > selectk::MAX_RANKS)
        return fail(MAM_ERR_INVALID_ARGUMENT, "one or two ranks");
    if (ranks[0] < 0 || (nranks == 2 && ranks[1] < ranks[0]))
        return fail(MAM_ERR_INVALID_ARGUMENT, "ranks must be non-negative and ascending");
    hipLaunchKernelGGL(selectk::begin_kernel, dim3(24), dim3(selectk::NT), 0, static_cast<hipStream_t>(stream),
                       static_cast<selectk::State *>(workspace), selectk::hist_of(workspace), ranks[0],
                       nranks == 2 ? ranks[1] : ranks[0], nranks);
    return check_launch("select begin_kernel");
}

static int accumulate(void *workspace, const float *w, int64_t ldw, int mode, const void *aux, const void *aux2, int64_t ld_aux,
                      int64_t M, int64_t K, int pass, bool chained, void *stream)
{
    using namespace mam;
    if (!workspace) return fail(MAM_ERR_WORKSPACE, "no workspace");
    if (M < 0 || K < 0) return fail(MAM_ERR_INVALID_ARGUMENT, "negative size");
    if (pass < 0 || pass >= selectk::PASSES) return fail(MAM_ERR_INVALID_ARGUMENT, "pass must be 0, 1 or 2");
    if (mode != MAM_PRUNE_MAGNITUDE && mode != MAM_PRUNE_WEIGHT_TIMES && mode != MAM_PRUNE_COUNT)
        return fail(MAM_ERR_INVALID_ARGUMENT, "unknown score mode %d", mode);
    if (M == 0 || K == 0) return MAM_OK;
    if ((mode != MAM_PRUNE_COUNT && !w) || (mode != MAM_PRUNE_MAGNITUDE && !aux))
        return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    if ((mode != MAM_PRUNE_COUNT && ldw < K) || (mode != MAM_PRUNE_MAGNITUDE && ld_aux < K))
        return fail(MAM_ERR_INVALID_ARGUMENT, "leading dimension smaller than the row length");
    // gapless matrices are one row: no division per load, and 16-byte loads wherever M * K is a multiple of 4
    if ((mode == MAM_PRUNE_COUNT || ldw == K) && (mode == MAM_PRUNE_MAGNITUDE || ld_aux == K)) {
        K *= M;
        M = 1;
        ldw = ld_aux = K;
    }
    const bool vec = K % 4 == 0 && (mode == MAM_PRUNE_COUNT || ((uintptr_t)w % 16 == 0 && ldw % 4 == 0)) &&
                     (mode == MAM_PRUNE_MAGNITUDE || ((uintptr_t)aux % 16 == 0 && (uintptr_t)aux2 % 16 == 0 && ld_aux % 4 == 0));
    const int64_t items = vec ? M * (K / 4) : M * K;
    // few, large workgroups: every workgroup ends by adding its non-empty bins to the global histogram, half a million
    // atomics in the second pass with twice as many workgroups and 11 bits there
    int64_t blocks = ceil_div(items, selectk::NT_H * 4);
    const int64_t cap = num_cus();
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // in a chain, pass p > 0 starts from the state that pass p - 1 started from
    selectk::State *state = static_cast<selectk::State *>(workspace) + (chained ? (pass - 1) * selectk::kStateStride : 0);
    selectk::count_t *hist = selectk::hist_of(workspace);
#define MAM_SELECT_LAUNCH(MODE, CHAINED)                                                                             \
    hipLaunchKernelGGL((selectk::hist_kernel<MODE, CHAINED>), dim3((unsigned)blocks), dim3(selectk::NT_H), 0, st, w, ldw, aux, \
                       aux2, ld_aux, M, K, vec ? 1 : 0, state, hist, pass)
    if (mode == MAM_PRUNE_MAGNITUDE && chained) MAM_SELECT_LAUNCH(MAM_PRUNE_MAGNITUDE, true);
    else if (mode == MAM_PRUNE_MAGNITUDE) MAM_SELECT_LAUNCH(MAM_PRUNE_MAGNITUDE, false);
    else if (mode == MAM_PRUNE_WEIGHT_TIMES && chained) MAM_SELECT_LAUNCH(MAM_PRUNE_WEIGHT_TIMES, true);
    else if (mode == MAM_PRUNE_WEIGHT_TIMES) MAM_SELECT_LAUNCH(MAM_PRUNE_WEIGHT_TIMES, false);
    else if (chained) MAM_SELECT_LAUNCH(MAM_PRUNE_COUNT, true);
    else MAM_SELECT_LAUNCH(MAM_PRUNE_COUNT, false);
#undef MAM_SELECT_LAUNCH
    return check_launch("select hist_kernel");
}

extern "C" int mam_select_accumulate(void *workspace, const float *w, int64_t ldw, int mode, const void *aux,
                                     const void *aux2, int64_t ld_aux, int64_t M, int64_t K, int pass, void *stream)
{
    return accumulate(workspace, w, ldw, mode, aux, aux2, ld_aux, M, K, pass, false, stream);
}

extern "C" int mam_select_advance(void *workspace, int pass, void *stream)
{
    using namespace mam;
    if (!workspace) return fail(MAM_ERR_WORKSPACE, "no workspace");
    if (pass < 0 || pass >= selectk::PASSES) return fail(MAM_ERR_INVALID_ARGUMENT, "pass must be 0, 1 or 2");
    hipLaunchKernelGGL(selectk::advance_kernel, dim3(1), dim3(selectk::NT), 0, static_cast<hipStream_t>(stream),
                       static_cast<selectk::State *>(workspace), selectk::hist_of(workspace), pass);
    return check_launch("select advance_kernel");
}

extern "C" int mam_select_result(void *workspace, int mode, float *out, void *stream)
{
    using namespace mam;
    if (!workspace || !out) return fail(MAM_ERR_INVALID_ARGUMENT, "null pointer");
    hipLaunchKernelGGL(selectk::result_kernel<false>, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                       static_cast<const selectk::State *>(workspace), selectk::hist_of(workspace), out, mode == MAM_PRUNE_COUNT ? 1 : 0);
    return check_launch("select result_kernel");
}

extern "C" int mam_select_ranks(const float *w, int64_t ldw, int mode, const void *aux, const void *aux2, int64_t ld_aux, int64_t M,
                                int64_t K, const int64_t *ranks, int nranks, float *out, void *workspace, size_t workspace_bytes,
                                void *stream)
{
    using namespace mam;
    int rc = mam_select_begin(workspace, workspace_bytes, ranks, nranks, stream);
    if (rc == MAM_OK && (!out || M == 0 || K == 0)) {
        // no score to find a digit in: the checks, and what the steps by themselves give
        for (int pass = 0; pass < selectk::PASSES && rc == MAM_OK; ++pass) {
            rc = mam_select_accumulate(workspace, w, ldw, mode, aux, aux2, ld_aux, M, K, pass, stream);
            if (rc == MAM_OK) rc = mam_select_advance(workspace, pass, stream);
        }
        return rc == MAM_OK ? mam_select_result(workspace, mode, out, stream) : rc;
    }
    for (int pass = 0; pass < selectk::PASSES && rc == MAM_OK; ++pass)
        rc = accumulate(workspace, w, ldw, mode, aux, aux2, ld_aux, M, K, pass, pass > 0, stream);
    if (rc != MAM_OK) return rc;
    hipLaunchKernelGGL(selectk::result_kernel<true>, dim3(1), dim3(selectk::NT), 0, static_cast<hipStream_t>(stream),
                       static_cast<const selectk::State *>(workspace) + (selectk::PASSES - 1) * selectk::kStateStride,
                       selectk::hist_of(workspace), out, mode == MAM_PRUNE_COUNT ? 1 : 0);
    return check_launch("select result_kernel");
}
