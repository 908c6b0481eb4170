// The 32-lane group kernel (group_kernel32.hip) built for one workgroup per CU: 512 registers a lane
// instead of 256, which keep more of the tracker's values out of private memory.  A launch that
// has at most one workgroup per CU takes this instance, a larger one the instance with two
// waves per SIMD in flight.  512 / 256 registers, n = 22: 601 paths 266 / 320 ms, 1,500 paths 310 / 382,
// 3,000 paths 452 / 462, 7,000 paths 848 / 796.  It is a file of its own because the tracker's
// functions are compiled once per file, for the largest register budget among its kernels.
#define GL 32
#include <hip/hip_runtime.h>

#include "device/hcg_group_run.h"
#include "hcg_group_launch.h"

namespace {

constexpr int kBlock = 256;

__global__ void __launch_bounds__(kBlock, 1) hcg_group_kernel32_wide(hcg_multi_kargs m, const hcg_gsys* sysd, int lds_per_path) {
    extern __shared__ __align__(16) char smem[];
    hcg_group_run<24>(m, sysd, lds_per_path, smem, (int)threadIdx.x);
}

}  // namespace

namespace hcg {

static hipError_t allow_lds(size_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&hcg_group_kernel32_wide),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

hipError_t group_launch32_wide(int grid, size_t shmem, int lds_per_path, hipStream_t stream, const hcg_multi_kargs& m,
                               const hcg_gsys* d_sys) {
    hipError_t e = allow_lds(shmem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(hcg_group_kernel32_wide, dim3(grid), dim3(kBlock), shmem, stream, m, d_sys, lds_per_path);
    return hipGetLastError();
}

hipError_t group_kernel32_wide_blocks_per_cu(size_t shmem, int* blocks) {
    hipError_t e = allow_lds(shmem);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, hcg_group_kernel32_wide, kBlock, shmem);
}

hipError_t group_kernel32_wide_attributes(hipFuncAttributes* attr) {
    return hipFuncGetAttributes(attr, reinterpret_cast<const void*>(&hcg_group_kernel32_wide));
}

}  // namespace hcg
