// The decode matvec kernels of MXFP4 (templates in mmvq.hpp).
#define MMVQ_INSTANTIATE
#include "mmvq.hpp"

namespace hkhip {
template mv_kernel_t pick<HKHIP_MXFP4>(int);
template mv_kernel_t mvr_pick<HKHIP_MXFP4>(int, int, int, bool);
template mv_kernel_t mvs_pick<HKHIP_MXFP4>(int, int);
} // namespace hkhip
