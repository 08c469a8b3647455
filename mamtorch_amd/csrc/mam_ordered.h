// Forward over magnitude-ordered operand lists: which side of a call is listed, decided on the device.
#pragma once
#include "mam_common.h"

namespace mam {
namespace ordered {

constexpr int SAMPLES = 64;      // sampled outputs of a call, one per lane of the deciding wave
constexpr int CHUNK = 8;         // list entries between two tests of the bound

enum Side { SIDE_NONE = 0, SIDE_X = 1, SIDE_W = 2 };

// What the sampling kernel leaves per sampled output: how many entries of its row of x (of w), taken by
// falling magnitude, have to be looked at before no remaining product can reach either extreme.
struct Sample { int need_x, need_w; };

// `samples` == nullptr: an unconditional launch.  Otherwise every wave of every kernel of the call comes to
// the same decision from the samples: the operand whose lists are shorter, or SIDE_NONE when more than
// MAX_LONG of the samples need more than `limit` entries on either side.
constexpr int MAX_LONG = 3;

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

__device__ __forceinline__ int decide(const Sample *samples, int limit, int lane, int &longest)
{
    const Sample s = samples[lane];
    const int long_x = __popcll(__ballot(s.need_x > limit)), long_w = __popcll(__ballot(s.need_w > limit));
    const int cx = s.need_x < limit ? s.need_x : limit, cw = s.need_w < limit ? s.need_w : limit;
    const int sum_x = wave_sum(cx), sum_w = wave_sum(cw);
    int side = SIDE_NONE;
    if (long_x <= MAX_LONG && (long_w > MAX_LONG || sum_x <= sum_w)) side = SIDE_X;
    else if (long_w <= MAX_LONG) side = SIDE_W;
    const int mine = side == SIDE_W ? s.need_w : s.need_x;
    longest = __builtin_amdgcn_readfirstlane(wave_max(mine > limit ? 0 : mine));
    return __builtin_amdgcn_readfirstlane(side);
}

// The same for kernels that run only when no side was chosen.
struct Guard { const Sample *samples; int limit; };
__device__ __forceinline__ bool guarded_off(const Guard &g)
{
    if (!g.samples) return false;
    const Sample s = g.samples[threadIdx.x & 63];
    return __popcll(__ballot(s.need_x > g.limit)) <= MAX_LONG || __popcll(__ballot(s.need_w > g.limit)) <= MAX_LONG;
}

struct Call {
    const float *x; int64_t ldx;
    const float *w; int64_t ldw; int w_layout;
    const float *bias;
    float *c; int32_t *argmax, *argmin;      // argmax == nullptr: values only
    float *wsel, *xsel;
    int64_t N, K, M;
};

// Whether the path takes a call of this size at all, and the workspace it needs (a multiple of 256).
bool applies(int64_t N, int64_t K, int64_t M);
size_t workspace_bytes(int64_t N, int64_t K, int64_t M);
// Samples, builds the lists and runs the forward where they pay; `guard` is what the caller's dense kernels
// take so that they run only where they do not.
int launch(const Call &call, void *workspace, Guard &guard, hipStream_t stream);

}  // namespace ordered
}  // namespace mam
