// hostcopy_kernel.hip -- a short list of arrays (hostcopy.h) converted into one
// array of doubles, which lies in pinned host memory: the link bounds it.
#include "hostcopy.h"

#include <algorithm>

namespace pic {

__global__ void __launch_bounds__(256) k_copy_small(SmallList l, double* __restrict__ out) {
    const size_t total = l.off[l.n];
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        int k = 0;
        while (i >= l.off[k + 1]) ++k;
        const CopyOut& a = l.a[k];
        const size_t j = i - l.off[k];
        double v;
        if (a.kind == kCopyF64) {
            v = static_cast<const double*>(a.src[0])[j];
        } else if (a.kind == kCopyPickF64) {
            v = static_cast<const double*>(a.src[*a.pick ? 1 : 0])[j];
        } else if (a.kind == kCopyPair32) {
            v = ((double)static_cast<const float*>(a.src[0])[j] + (double)static_cast<const float*>(a.src[1])[j]) * a.scale;
        } else {
            const uint32_t q = static_cast<const uint32_t*>(a.src[0])[j];
            v = a.kind == kCopyUnimod32 && q == 0 ? 1.0 : (double)q * 0x1p-32;
        }
        out[i] = v;
    }
}

hipError_t launch_copy_small(const SmallList& l, double* out, hipStream_t stream) {
    const unsigned blocks = (unsigned)std::min<size_t>((l.off[l.n] + 255) / 256, 512);
    k_copy_small<<<blocks, 256, 0, stream>>>(l, out);
    return hipGetLastError();
}

}  // namespace pic
