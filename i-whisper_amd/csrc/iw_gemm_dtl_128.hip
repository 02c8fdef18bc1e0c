// The direct-to-LDS GEMM (iw_gemm_dtl.hpp) on 128 x 128 tiles.
#include "iw_gemm_dtl.hpp"

namespace iw {
namespace dtl {

template int gemm_dtl_tile<Tile128>(const GemmArgs &, hipStream_t);

}  // namespace dtl
}  // namespace iw
