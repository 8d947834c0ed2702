// Instantiations of the low-bit skinny GEMM for decoder kinds: DK_INT8S,DK_INT8A
#include "lowbit_skinny.cuh"
namespace illm {
template void launch_skinny_dk<DK_INT8S>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
template void launch_skinny_dk<DK_INT8A>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
}  // namespace illm
