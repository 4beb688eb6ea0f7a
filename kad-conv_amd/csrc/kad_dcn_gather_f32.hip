// The gathering deformable convolution for fp32 maps.
#include "kad_dcn_gather.h"

namespace kad {
template int dcn_gather<float>(const kad_dcn_args&, const DcnGeom&, int, hipStream_t);
template int dcn_gather_group<float>(const DcnGroup&, int, hipStream_t);
}  // namespace kad
