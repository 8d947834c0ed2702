// Instantiations of the row-finishing low-bit product for decoder kinds: DK_FP8E4,DK_FP8E5
#include "lowbit_fullk.cuh"
namespace illm {
template void launch_fullk_dk<DK_FP8E4>(bool, int, const FullkArgs&, hipStream_t);
template void launch_fullk_dk<DK_FP8E5>(bool, int, const FullkArgs&, hipStream_t);
}  // namespace illm
