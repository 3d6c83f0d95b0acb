// hostcopy.h -- device-to-host copies of a context's state into the caller's
// ordinary memory (hostcopy.cpp, hostcopy_kernel.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace pic {

// One array to bring to the host: n elements.
enum CopyKind {
    kCopyF64,       // src[0]: double -> dst
    kCopyFix32,     // src[0]: u32 fraction of the box -> double (times 2^-32)
    kCopyUnimod32,  // the same with 0 meaning 1 (positions in (0, 1])
    kCopyPair32,    // src[0], src[1]: float hi, lo -> (hi + lo) * scale
    kCopyPickF64,   // src[*pick ? 1 : 0]: double -> dst (pick: a device word)
};
struct CopyOut {
    CopyKind kind;
    double* dst;
    const void* src[2];
    size_t n;
    double scale;
    const int32_t* pick;
};

// Copies every array of the list (entries without dst are left out) after the
// work that stream, the caller's own, holds so far, which wrote the sources.
// The caller has set the device.  Calls of several threads run side by side.
// Returns a HIP error code (0: done); throws nothing.
hipError_t copy_out(int device, hipStream_t stream, const CopyOut* list, int count);

// The staging buffers exist while some context of the device does: a context
// retains them once when it is made and, if that returned true, releases them
// when it is destroyed.
bool hostcopy_retain(int device);
void hostcopy_release(int device);

// A short list converted by one kernel; off[k]: the first element of array k
// in out.
constexpr int kSmallList = 8;
struct SmallList {
    CopyOut a[kSmallList];
    size_t off[kSmallList + 1];
    int n;
};
hipError_t launch_copy_small(const SmallList& l, double* out, hipStream_t stream);

}  // namespace pic
