// f16 instantiations of the sparse-operand matmul that keeps rows of the dense operand in LDS.
#include "matmul_spmm_rows.hpp"
namespace spx {
template <>
int launch_spmm_rows<_Float16>(const SpmmParams& p, int BN, int batch, hipStream_t st) {
    return launch_spmm_rows_impl<_Float16>(p, BN, batch, st);
}
}  // namespace spx
