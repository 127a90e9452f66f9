// Matrix-product kernel instances: EPI_RMSNORM.
#include "gemm_launch.h"

template void yr::gm::launch<yr::gm::EPI_RMSNORM>(int, int, bool, bool, const yr::gm::Args&, hipStream_t);
