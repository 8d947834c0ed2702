// Instantiations of the low-bit skinny GEMM for decoder kinds: DK_INT4S,DK_INT4A
#include "lowbit_skinny.cuh"
namespace illm {
template void launch_skinny_dk<DK_INT4S>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
template void launch_skinny_dk<DK_INT4A>(bool, int, int, int, dim3, const GemvArgs&, hipStream_t);
}  // namespace illm
