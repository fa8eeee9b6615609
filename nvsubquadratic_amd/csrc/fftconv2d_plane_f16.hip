// f16 instances of the small-plane 2D convolution.
#include "fftconv2d_plane_impl.h"

namespace nsq {
NSQ_PLANE2_INSTANCES(NSQ_DTYPE_F16)
}  // namespace nsq
