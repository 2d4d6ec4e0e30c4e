// rf_tile_inst.hip -- instantiates k_adam8_tile for one (APPLY, MSR, EXACT)
// combination, as rf_adam8_inst.hip does k_adam8.
#include "rf_tile.h"

#if !defined(RFI_APPLY) || !defined(RFI_MSR) || !defined(RFI_EXACT)
#error "build with -DRFI_APPLY=0|1 -DRFI_MSR=0|1 -DRFI_EXACT=0|1"
#endif

#define RF_PICK_NAME2(a, m, e) rf_pick_tile_a##a##_m##m##_e##e
#define RF_PICK_NAME(a, m, e) RF_PICK_NAME2(a, m, e)

namespace rf {

template <int32_t DT>
static adam_kernel_t pick(bool psr, bool nest)
{
    constexpr bool A = RFI_APPLY != 0, M = RFI_MSR != 0, E = RFI_EXACT != 0;
    if constexpr (A) {
        if (psr) return nest ? &k_adam8_tile<DT, A, M, true, true, E> : &k_adam8_tile<DT, A, M, true, false, E>;
    }
    return nest ? &k_adam8_tile<DT, A, M, false, true, E> : &k_adam8_tile<DT, A, M, false, false, E>;
}

// bf16: every leaf of the list has bf16 params and grads
adam_kernel_t RF_PICK_NAME(RFI_APPLY, RFI_MSR, RFI_EXACT)(bool bf16, bool psr, bool nest)
{
    return bf16 ? pick<RF_BF16>(psr, nest) : pick<DT_ANY>(psr, nest);
}

}  // namespace rf
