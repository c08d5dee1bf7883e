// bf16 instantiations of the LDS-ring kernel.
#include "matmul_spmm_ring.hpp"
namespace spx {
template <>
int launch_spmm_ring<bf16_t>(const SpmmParams& p, int BN, int batch, int rows, hipStream_t st) {
    return rows == 64 ? launch_spmm_ring_tile<bf16_t, 64>(p, BN, batch, st) : launch_spmm_ring_tile<bf16_t, 128>(p, BN, batch, st);
}
}  // namespace spx
