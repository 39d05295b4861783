// aca_reg_gauss.hip -- the ACA of aca_reg.h for one kernel kind.
#include "aca_reg_kernel.h"

namespace hmg {
template hmg_status aca_reg_launch<HMG_KERNEL_GAUSSIAN>(const AcaArgs&, int, bool, int, hipStream_t);
template hmg_status aca_search_launch<HMG_KERNEL_GAUSSIAN>(const AcaArgs&, int, hipStream_t);
}  // namespace hmg
