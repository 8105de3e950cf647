// Resident-pass instances: double, 1 state(s) a lane, complex values.
#include "tbg_ring_pass.h"

namespace tbg {
template void launch_ring_rt<double, 1, false>(const RingArgs<double>&, const Ring&, hipStream_t);
template void allow_ring_lds<double, 1, false>(int);
}  // namespace tbg
