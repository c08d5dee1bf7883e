// bf16 instantiations of the sparse-operand matmul that keeps rows of the dense operand in LDS.
#include "matmul_spmm_rows.hpp"
namespace spx {
template <>
int launch_spmm_rows<bf16_t>(const SpmmParams& p, int BN, int batch, hipStream_t st) {
    return launch_spmm_rows_impl<bf16_t>(p, BN, batch, st);
}
}  // namespace spx
