// bf16 instantiations of the sparse-output matmul whose blocks share A.
#include "matmul_dds_share.hpp"
namespace spx {
template <>
int launch_dds_share<bf16_t>(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st) {
    return launch_dds_share_impl<bf16_t>(p, s, colsum, BM, BN, batch, st);
}
}  // namespace spx
