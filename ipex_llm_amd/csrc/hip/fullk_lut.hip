// Instantiations of the row-finishing low-bit product for decoder kinds: DK_LUT4,DK_FP4
#include "lowbit_fullk.cuh"
namespace illm {
template void launch_fullk_dk<DK_LUT4>(bool, int, const FullkArgs&, hipStream_t);
template void launch_fullk_dk<DK_FP4>(bool, int, const FullkArgs&, hipStream_t);
}  // namespace illm
