// Forward over magnitude-ordered operand lists: which operand is listed, decided on the device.
#pragma once
#include "mam_common.h"

namespace mam {
namespace ordered {

enum Side { SIDE_NONE = 0, SIDE_X = 1, SIDE_W = 2 };

// What build_kernel leaves for the other kernels of a call.
struct Decision {
    int side;    // the operand whose rows are searched entry by entry; SIDE_NONE: the dense kernels run
    int lead;    // entries of the OTHER operand's lists that are taken first (0: none), a multiple of CHUNK
    int length;  // entries per searched list, a multiple of CHUNK
    int pad;
};

// For kernels that run only when no side was chosen (nullptr: unconditional).
struct Guard { const Decision *decision; };
__device__ __forceinline__ bool guarded_off(const Guard &g) { return g.decision && g.decision->side != SIDE_NONE; }

struct Call {
    const float *x; int64_t ldx;
    const float *w; int64_t ldw; int w_layout;
    const float *bias;
    float *c; int32_t *argmax, *argmin;      // argmax == nullptr: values only; argmin == nullptr: both packed in argmax
    float *wsel, *xsel;
    int64_t N, K, M;
};

// Whether the path takes a call of this size at all, and the workspace it needs (a multiple of 256).
bool applies(int64_t N, int64_t K, int64_t M);
size_t workspace_bytes(int64_t N, int64_t K, int64_t M, int w_layout);
// Samples, builds the lists and runs the forward where they pay; `guard` is what the caller's dense kernels
// take so that they run only where they do not.
int launch(const Call &call, void *workspace, Guard &guard, hipStream_t stream);

}  // namespace ordered
}  // namespace mam
