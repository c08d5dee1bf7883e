// f16 instantiations of the k-split sparse-output matmul kernel.
#include "matmul_dds_split.hpp"
namespace spx {
template <>
int launch_dds_split<_Float16>(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st) {
    return launch_dds_split_impl<_Float16>(p, s, colsum, BM, BN, batch, st);
}
template <>
int launch_dds_unsliced<_Float16>(const DdsParams& p, int BM, int BN, int nnz_bound, int batch, int share, hipStream_t st) {
    return launch_dds_split<_Float16>(p, DdsSplit{1, 0, nnz_bound, 0, nullptr, nullptr, nullptr, share}, nullptr, BM, BN, batch, st);
}
template int dds_shared_blocks<_Float16>(const DdsParams&, int, int, int, int);
}  // namespace spx
