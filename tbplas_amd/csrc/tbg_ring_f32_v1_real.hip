// Resident-pass instances: float, 1 state(s) a lane, real values.
#include "tbg_ring_pass.h"

namespace tbg {
template void launch_ring_rt<float, 1, true>(const RingArgs<float>&, const Ring&, hipStream_t);
template void allow_ring_lds<float, 1, true>(int);
}  // namespace tbg
