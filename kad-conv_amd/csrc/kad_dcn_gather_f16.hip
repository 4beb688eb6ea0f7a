// The gathering deformable convolution for fp16 maps.
#include "kad_dcn_gather.h"

namespace kad {
template int dcn_gather<half_t>(const kad_dcn_args&, const DcnGeom&, int, hipStream_t);
template int dcn_gather_group<half_t>(const DcnGroup&, int, hipStream_t);
}  // namespace kad
