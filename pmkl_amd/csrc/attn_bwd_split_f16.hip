// Explicit instantiations of the key-split and the eight-wave 16-bit backward for _Float16: compiled as
// a translation unit of its own so that the library's kernels build in parallel
// (attn_capi.hip declares them extern).
#include <hip/hip_runtime.h>

#include "attn_bwd_kernels.hpp"

namespace pmkl_amd {
template __global__ void attn_bwd_dq_kernel<_Float16, 32, true, 2>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 32, false, 2>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 32, true, 2>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 32, false, 2>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 64, true, 2>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 64, false, 2>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 64, true, 2>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 64, false, 2>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 128, true, 2>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 128, false, 2>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 128, true, 2>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 128, false, 2>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 64, true, 1, 8>(BwdParams);
template __global__ void attn_bwd_dq_kernel<_Float16, 64, false, 1, 8>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 64, true, 1, 8>(BwdParams);
template __global__ void attn_bwd_dkdv_kernel<_Float16, 64, false, 1, 8>(BwdParams);
}  // namespace pmkl_amd
