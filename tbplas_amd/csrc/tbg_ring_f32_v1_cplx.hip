// Resident-pass instances: float, 1 state(s) a lane, complex values.
#include "tbg_ring_pass.h"

namespace tbg {
template void launch_ring_rt<float, 1, false>(const RingArgs<float>&, const Ring&, hipStream_t);
template void allow_ring_lds<float, 1, false>(int);
}  // namespace tbg
