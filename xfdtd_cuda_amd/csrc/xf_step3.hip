// xf_step3.hip -- k_step3 for one storage type (XF_STEP3_STORE), a
// translation unit of its own so that the types compile in parallel.
#include <type_traits>

#include "xf_kernels.h"

namespace xf {

#include "xf_step3.inl"

template <typename S>
hipError_t step3_launch(const Step3Pass<S>* passes, const int* block_start, int n, int blocks, bool pml, size_t lds,
                        int t_arg, const int* t_dev, hipStream_t stream) {
  const dim3 block(64 * (kStep3Rows + 2));
  if (pml)
    hipLaunchKernelGGL((k_step3<S, true>), dim3(blocks), block, lds, stream, passes, block_start, n, t_arg, t_dev);
  else
    hipLaunchKernelGGL((k_step3<S, false>), dim3(blocks), block, lds, stream, passes, block_start, n, t_arg, t_dev);
  return hipGetLastError();
}

template <typename S>
int step3_blocks_per_cu(bool pml, size_t lds) {
  int n = 0;
  const int threads = 64 * (kStep3Rows + 2);
  const hipError_t e = pml ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_step3<S, true>, threads, lds)
                           : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_step3<S, false>, threads, lds);
  return e == hipSuccess && n > 0 ? n : 1;
}

template int step3_blocks_per_cu<XF_STEP3_STORE>(bool, size_t);
template hipError_t step3_launch<XF_STEP3_STORE>(const Step3Pass<XF_STEP3_STORE>*, const int*, int, int, bool, size_t,
                                                 int, const int*, hipStream_t);

}  // namespace xf
