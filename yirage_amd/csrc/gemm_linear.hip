// Matrix-product kernel instances: EPI_LINEAR.
#include "gemm_launch.h"

template void yr::gm::launch<yr::gm::EPI_LINEAR>(int, int, bool, bool, const yr::gm::Args&, hipStream_t);
