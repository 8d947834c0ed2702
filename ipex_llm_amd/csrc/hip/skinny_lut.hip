// Instantiations of the low-bit skinny GEMM for decoder kinds: DK_LUT4,DK_FP4
#include "lowbit_skinny.cuh"
namespace illm {
template void launch_skinny_dk<DK_LUT4>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
template void launch_skinny_dk<DK_FP4>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
}  // namespace illm
