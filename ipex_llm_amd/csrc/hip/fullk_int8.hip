// Instantiations of the row-finishing low-bit product for decoder kinds: DK_INT8S,DK_INT8A
#include "lowbit_fullk.cuh"
namespace illm {
template void launch_fullk_dk<DK_INT8S>(bool, int, const FullkArgs&, hipStream_t);
template void launch_fullk_dk<DK_INT8A>(bool, int, const FullkArgs&, hipStream_t);
}  // namespace illm
