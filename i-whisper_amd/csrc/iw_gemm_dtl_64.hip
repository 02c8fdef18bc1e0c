// The direct-to-LDS GEMM (iw_gemm_dtl.hpp) on 64 x 64 tiles.
#include "iw_gemm_dtl.hpp"

namespace iw {
namespace dtl {

template int gemm_dtl_tile<Tile64>(const GemmArgs &, hipStream_t);

}  // namespace dtl
}  // namespace iw
