// Instantiations of the row-finishing low-bit product for decoder kinds: DK_INT4S,DK_INT4A
#include "lowbit_fullk.cuh"
namespace illm {
template void launch_fullk_dk<DK_INT4S>(bool, int, const FullkArgs&, hipStream_t);
template void launch_fullk_dk<DK_INT4A>(bool, int, const FullkArgs&, hipStream_t);
}  // namespace illm
