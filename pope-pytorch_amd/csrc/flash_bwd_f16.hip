// Flash attention backward, fp16 instances (kernels: flash_bwd.hpp).
#include "flash_bwd.hpp"

namespace pope {

hipError_t launch_flash_bwd_f16(const FlashBwdParams& p, hipStream_t s) { return flash_bwd_dispatch<F16>(p, s); }

}  // namespace pope
