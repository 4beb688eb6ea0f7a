// The gathering deformable convolution for bf16 maps.
#include "kad_dcn_gather.h"

namespace kad {
template int dcn_gather<bf16_t>(const kad_dcn_args&, const DcnGeom&, int, hipStream_t);
template int dcn_gather_group<bf16_t>(const DcnGroup&, int, hipStream_t);
}  // namespace kad
