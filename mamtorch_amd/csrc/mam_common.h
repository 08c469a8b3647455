// Shared host/device helpers of libmam_hip.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/mam_hip.h"

namespace mam {

// Records the detail of a failure for mam_last_error() and returns `code`.
int fail(int code, const char *fmt, ...);

// Checks the launch that was just issued on the calling thread.
int check_launch(const char *what);

// Asynchronously sets `count` 32-bit words to zero with a small kernel (graph-capture safe).
int fill_zero(void *ptr, int64_t count, hipStream_t stream);

// ---- per-device set-up ------------------------------------------------------------------------
// Everything that has to happen once per device before kernels are launched there (raising the LDS
// limit of the kernels that use more than 64 KiB, creating the library's second stream and its events,
// taking the address of the file-scope scratch array) is collected in hooks, one per source file, and run
// by ensure_device() under a per-device lock the first time an entry point sees that device -- or by
// mam_init(), which a caller that records HIP graphs calls before capturing.
constexpr int kMaxDevices = 16;
typedef int (*DeviceHook)(int dev);
struct DeviceHookRegistration { explicit DeviceHookRegistration(DeviceHook fn); };
// Returns the current device's index (0..kMaxDevices-1) after its hooks have run, or a negative MAM_ERR_*.
// `st` is the stream the entry point launches on: while it is being captured the hooks still run (they
// create nothing), and the second stream and its events are left for the first call outside a capture.
int ensure_device(hipStream_t st = nullptr);

// Run-time switches (mam_set_option; initial values come from the environment, read once at load).
int option(int which);

// Compute units of the current device (read from the device at its set-up).
int num_cus();

// dst (cols, ld_dst) = transpose of src (rows, cols), row stride ld; columns rows .. ld_dst - 1 repeat the last one.
// `guard` (mam_ordered.h): the kernel exits at once where the guard says that nobody reads the copy.
namespace ordered { struct Guard; }
int transpose(const float *src, int64_t ld, float *dst, int64_t rows, int64_t cols, int64_t ld_dst, hipStream_t stream,
              const ordered::Guard *guard = nullptr);

// dst (rows, ld_dst) = src (rows, cols) with row stride ld, the last element of a row repeated up to ld_dst; two matrices
// in one launch (rows == 0: none).  ld_dst is a multiple of 4, dst 16-byte aligned, at most 65535 rows together.
// range_len > 0: rows are consecutive ranges of range_len (the last one shorter), of which each is lengthened to ld_dst / their number
// (a multiple of 4).
struct LengthenRows { const float *src; int64_t ld; float *dst; int rows; };
// Other ends, of ranges of at least 64: tiles of 64, the last one of which holds the range's last 64; the range, then (64 before
// its copy's end) its last 64 once more.
enum RowsEnd { ROWS_REPEAT_LAST, ROWS_END_WHOLE_TILES, ROWS_AND_LAST_64 };
int lengthen_rows(const LengthenRows &a, const LengthenRows &b, int64_t cols, int64_t ld_dst, int64_t range_len, RowsEnd end,
                  hipStream_t stream, const ordered::Guard *guard = nullptr);

// Two independent kernels of one call side by side: the first runs on a second stream of the library
// (default priority, one per device) between a fork and a join event on the caller's stream.
//   ForkedStream fork(st, units);      // decides; fork.side() is `st` itself when not forked
//   launch A on fork.side(); fork.join_later(); launch B on st; rc = fork.join();
// Between eager launches the two events cost ~15 us, inside a captured graph next to nothing: the fork
// is taken from 2^22 `units` (outputs of the call) on where the caller says that it pays between eager
// launches (`eager_pays`), and from 2^16 on while `st` is being captured, where it pays there (`captured_pays`).
// Option MAM_OPT_BACKWARD_FORK forces it off / on.  The enqueue sequences of concurrent callers on one
// device are serialised (the events are reused), so an object of this class holds that device's lock
// while forked.  The second stream is created by the device's set-up, never inside a capture.
class ForkedStream {
public:
    ForkedStream(hipStream_t st, int64_t units, bool eager_pays = true, bool captured_pays = true);
    ~ForkedStream();
    hipStream_t side() const { return side_; }
    bool forked() const { return forked_; }
    void join_later();   // after the last launch on side(): records the join event
    int join();          // after the launches on the caller's stream: it waits for the side stream
private:
    hipStream_t st_, side_;
    int dev_;
    bool forked_, recorded_;
};

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

constexpr int kNumXCD = 8;   // MI355X: 8 accelerator complex dies, each with its own L2
constexpr int kNumCU = 256;  // 32 active CUs per XCD (fallback when the device cannot be asked)

// Workgroups are handed to the XCDs round-robin by linear id.  This maps the hardware id
// to a logical id such that logical ids [i*per, (i+1)*per) all run on XCD i, so that
// neighbouring logical tiles share one L2.
__device__ __forceinline__ int xcd_remap(int bid, int nblk)
{
    const int xcd = bid % kNumXCD, slot = bid / kNumXCD;
    const int q = nblk / kNumXCD, r = nblk % kNumXCD;
    return slot + xcd * q + (xcd < r ? xcd : r);
}

template <int LAYOUT>
__device__ __forceinline__ float load_w(const float *__restrict__ w, int64_t ldw, int64_t k, int64_t m)
{
    return LAYOUT == MAM_W_MK ? w[m * ldw + k] : w[k * ldw + m];
}

// Both picks of an output in one word (argmin == nullptr, K at most 65535): what a backward reads of the indices, at half the
// planes.  The word of an output that is not there, -1, is a pick that no K has.
constexpr int64_t MOST_PACKED_K = 65535;
__device__ __forceinline__ int32_t pack_picks(int hi, int lo) { return (int32_t)((uint32_t)hi | (uint32_t)lo << 16); }
__device__ __forceinline__ void unpack_picks(int32_t &a1, int32_t &a2)
{
    a2 = (int32_t)((uint32_t)a1 >> 16);
    a1 &= 0xffff;
}

// Q consecutive words of a row of which `left` are left: one load where there are Q, of 4-byte aligned addresses (what a load
// of several words needs), so that neither the number of neurons nor an operand's alignment takes a call off the kernels that read
// several words a lane; past the end of the row `none`.
template <int Q, class T>
__device__ __forceinline__ void row_words(const T *p, int left, T none, T (&v)[Q])
{
    typedef T words __attribute__((ext_vector_type(Q), aligned(4)));
    if (left >= Q) {
        const words t = *reinterpret_cast<const words *>(p);
#pragma unroll
        for (int u = 0; u < Q; ++u) v[u] = t[u];
    } else {
#pragma unroll
        for (int u = 0; u < Q; ++u) v[u] = u < left ? p[u] : none;
    }
}
// (by name and not by index: through arrays mam_bwd_x_rows_kernel takes 73 us for 12608 x 3072 -> 768, like this 65)
typedef float floats4 __attribute__((ext_vector_type(4), aligned(4)));
typedef int ints4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 row_quad(const float *p, int left)
{
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (left >= 4) {
        const floats4 t = *reinterpret_cast<const floats4 *>(p);
        v = make_float4(t.x, t.y, t.z, t.w);
    } else {
        if (left > 0) v.x = p[0];
        if (left > 1) v.y = p[1];
        if (left > 2) v.z = p[2];
    }
    return v;
}
__device__ __forceinline__ int4 row_quad(const int32_t *p, int left)
{
    int4 v = make_int4(-1, -1, -1, -1);
    if (left >= 4) {
        const ints4 t = *reinterpret_cast<const ints4 *>(p);
        v = make_int4(t.x, t.y, t.z, t.w);
    } else {
        if (left > 0) v.x = p[0];
        if (left > 1) v.y = p[1];
        if (left > 2) v.z = p[2];
    }
    return v;
}

// out[m] = sum over s of partial[s][m], in slab order (mam_module.hip).
int sum_slabs(const float *partial, float *out, int64_t M, int64_t slabs, hipStream_t stream);

namespace bwd {
// x_grad (N,K) from the selected weights (2,N,M) written by a forward (mam_backward.hip).
int x_grad_from_selected(const float *grad, const int32_t *argmax, const int32_t *argmin, const float *w_sel,
                         float *x_grad, int64_t N, int64_t K, int64_t M, hipStream_t st);
}  // namespace bwd

}  // namespace mam
