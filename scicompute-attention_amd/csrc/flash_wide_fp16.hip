// The wide-row flash kernel's fp16 instantiations (a file per type, so that they compile in parallel).

#include "flash_wide.hpp"

namespace sca_hip {

#define SCA_INSTANTIATE(D)                                                                        \
    template int LaunchFlashWide<F16, D, false>(const sca_flash_params&, const SplitArgs&, hipStream_t); \
    template int LaunchFlashWide<F16, D, true>(const sca_flash_params&, const SplitArgs&, hipStream_t);
#define SCA_INSTANTIATE_VARLEN(D)                                                          \
    template int LaunchFlashVarlen<F16, D, false>(const sca_flash_varlen_params&, hipStream_t); \
    template int LaunchFlashVarlen<F16, D, true>(const sca_flash_varlen_params&, hipStream_t);
SCA_INSTANTIATE(32)
SCA_INSTANTIATE(64)
SCA_INSTANTIATE(96)
SCA_INSTANTIATE(128)
SCA_INSTANTIATE(160)
SCA_INSTANTIATE_VARLEN(64)
SCA_INSTANTIATE_VARLEN(128)

}  // namespace sca_hip
