// aca_reg_gauss_ref.hip -- the ACA of aca_reg.h for one kernel kind.
#include "aca_reg_kernel.h"

namespace hmg {
template hmg_status aca_reg_launch<HMG_KERNEL_GAUSSIAN_REF>(const AcaArgs&, int, bool, int, hipStream_t);
template hmg_status aca_search_launch<HMG_KERNEL_GAUSSIAN_REF>(const AcaArgs&, int, hipStream_t);
}  // namespace hmg
