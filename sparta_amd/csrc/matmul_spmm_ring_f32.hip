// f32 instantiations of the LDS-ring kernel.
#include "matmul_spmm_ring.hpp"
namespace spx {
template <>
int launch_spmm_ring<float>(const SpmmParams& p, int BN, int batch, int rows, hipStream_t st) {
    return rows == 64 ? launch_spmm_ring_tile<float, 64>(p, BN, batch, st) : launch_spmm_ring_tile<float, 128>(p, BN, batch, st);
}
}  // namespace spx
