// Matrix-product kernel instances: EPI_GATED.
#include "gemm_launch.h"

template void yr::gm::launch<yr::gm::EPI_GATED>(int, int, bool, bool, const yr::gm::Args&, hipStream_t);
