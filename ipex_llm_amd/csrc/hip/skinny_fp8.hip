// Instantiations of the low-bit skinny GEMM for decoder kinds: DK_FP8E4,DK_FP8E5
#include "lowbit_skinny.cuh"
namespace illm {
template void launch_skinny_dk<DK_FP8E4>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
template void launch_skinny_dk<DK_FP8E5>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
}  // namespace illm
