// erfc_tail.h -- GENERATED by fit_erfc_tail.py; do not edit.
// erfc(m + 1/2 + u), u in [-1/2, 1/2], in powers of u.
#pragma once
#include <hip/hip_runtime.h>

namespace pic {
// interpolation error 2.3e-22
template <typename T>
__host__ __device__ __forceinline__ T erfc_tail3(T u) {
    T p = T(0x1.78ff49d3f04f5p-33);
    p = __builtin_elementwise_fma(p, u, T(0x1.34a901b26b9c3p-31));
    p = __builtin_elementwise_fma(p, u, T(-0x1.164fdd9fc6a4cp-28));
    p = __builtin_elementwise_fma(p, u, T(0x1.1e83dad877c3cp-27));
    p = __builtin_elementwise_fma(p, u, T(0x1.8a21ba90d495ep-28));
    p = __builtin_elementwise_fma(p, u, T(-0x1.8c962f14619edp-24));
    p = __builtin_elementwise_fma(p, u, T(0x1.43ea28d943826p-22));
    p = __builtin_elementwise_fma(p, u, T(-0x1.dc7e947ad1b07p-22));
    p = __builtin_elementwise_fma(p, u, T(-0x1.dd7f35486d16ap-22));
    p = __builtin_elementwise_fma(p, u, T(0x1.377411d6438e5p-18));
    p = __builtin_elementwise_fma(p, u, T(-0x1.013525f99d85ap-16));
    p = __builtin_elementwise_fma(p, u, T(0x1.1f6304e2293b1p-15));
    p = __builtin_elementwise_fma(p, u, T(-0x1.e827fafa9a49ap-15));
    p = __builtin_elementwise_fma(p, u, T(0x1.46153fb9756a2p-14));
    p = __builtin_elementwise_fma(p, u, T(-0x1.586bafc9b99cap-14));
    p = __builtin_elementwise_fma(p, u, T(0x1.1c07721ac862dp-14));
    p = __builtin_elementwise_fma(p, u, T(-0x1.62ccea63cb0c0p-15));
    p = __builtin_elementwise_fma(p, u, T(0x1.3d0e43d67412ep-16));
    p = __builtin_elementwise_fma(p, u, T(-0x1.6a597219a93dap-18));
    p = __builtin_elementwise_fma(p, u, T(0x1.8ef2a9a18d859p-21));
    return p;
}
// interpolation error 8.6e-22
template <typename T>
__host__ __device__ __forceinline__ T erfc_tail4(T u) {
    T p = T(0x1.0130e006382b6p-34);
    p = __builtin_elementwise_fma(p, u, T(-0x1.ff8471d695744p-36));
    p = __builtin_elementwise_fma(p, u, T(-0x1.feff5b497e711p-32));
    p = __builtin_elementwise_fma(p, u, T(0x1.3380b3f935c1fp-29));
    p = __builtin_elementwise_fma(p, u, T(-0x1.e47b6b3a2c4f4p-28));
    p = __builtin_elementwise_fma(p, u, T(0x1.2cc6700a2f42fp-26));
    p = __builtin_elementwise_fma(p, u, T(-0x1.34eeb3600ab29p-25));
    p = __builtin_elementwise_fma(p, u, T(0x1.0c3ad3c9478e7p-24));
    p = __builtin_elementwise_fma(p, u, T(-0x1.8d2e60635af64p-24));
    p = __builtin_elementwise_fma(p, u, T(0x1.f5f30ee2c8017p-24));
    p = __builtin_elementwise_fma(p, u, T(-0x1.0d678f996672dp-23));
    p = __builtin_elementwise_fma(p, u, T(0x1.e650e3e0951b5p-24));
    p = __builtin_elementwise_fma(p, u, T(-0x1.6b1baf4475855p-24));
    p = __builtin_elementwise_fma(p, u, T(0x1.b598cb3e82ce6p-25));
    p = __builtin_elementwise_fma(p, u, T(-0x1.99b8665622088p-26));
    p = __builtin_elementwise_fma(p, u, T(0x1.180fde419db9bp-27));
    p = __builtin_elementwise_fma(p, u, T(-0x1.f1e3523b419dcp-30));
    p = __builtin_elementwise_fma(p, u, T(0x1.b05cfe2e92156p-33));
    return p;
}
// interpolation error 9.9e-22
template <typename T>
__host__ __device__ __forceinline__ T erfc_tail5(T u) {
    T p = T(-0x1.113a004794de7p-38);
    p = __builtin_elementwise_fma(p, u, T(0x1.136e580b86cc5p-37));
    p = __builtin_elementwise_fma(p, u, T(-0x1.6bd26d7631a81p-37));
    p = __builtin_elementwise_fma(p, u, T(0x1.118eb0fa02d24p-36));
    p = __builtin_elementwise_fma(p, u, T(-0x1.869a2553c8cb9p-36));
    p = __builtin_elementwise_fma(p, u, T(0x1.db082e6a3eca0p-36));
    p = __builtin_elementwise_fma(p, u, T(-0x1.fa5bff3e29463p-36));
    p = __builtin_elementwise_fma(p, u, T(0x1.dbeb2c25fb07cp-36));
    p = __builtin_elementwise_fma(p, u, T(-0x1.84a6d56c05df5p-36));
    p = __builtin_elementwise_fma(p, u, T(0x1.0f737ef08ecbbp-36));
    p = __builtin_elementwise_fma(p, u, T(-0x1.3e4a003309971p-37));
    p = __builtin_elementwise_fma(p, u, T(0x1.31007f87eb3b4p-38));
    p = __builtin_elementwise_fma(p, u, T(-0x1.cb12e5f2b56afp-40));
    p = __builtin_elementwise_fma(p, u, T(0x1.fd39a3c5d9eb8p-42));
    p = __builtin_elementwise_fma(p, u, T(-0x1.725860f353a95p-44));
    p = __builtin_elementwise_fma(p, u, T(0x1.0918294ce3ce5p-47));
    return p;
}
}  // namespace pic
