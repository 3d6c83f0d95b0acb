// hostcopy.h -- device-to-host copies of a context's state into the caller's
// ordinary memory (hostcopy.cpp).
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

// Copies every array of the list (entries without dst are left out).  The
// caller has synchronised with whatever wrote the sources.  Returns a HIP
// error code (0: done); throws nothing.
hipError_t copy_out(int device, const CopyOut* list, int count);

// The staging buffers exist while some context of the device does: a context
// retains them once when it is made and releases them when it is destroyed.
void hostcopy_retain(int device);
void hostcopy_release(int device);

}  // namespace pic
