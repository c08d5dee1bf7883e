// f32 instantiations of the sparse-output matmul whose blocks share A.
#include "matmul_dds_share.hpp"
namespace spx {
template <>
int launch_dds_share<float>(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st) {
    return launch_dds_share_impl<float>(p, s, colsum, BM, BN, batch, st);
}
}  // namespace spx
