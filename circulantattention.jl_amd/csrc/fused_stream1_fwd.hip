// Instantiations of the streamed kernels, forward, up to 16 real
// components per head (fused_stream_impl.h).
#include "fused_stream_impl.h"

namespace circatt {

CIRCATT_FST_DEF(fwd, fst::FWD, 1)

}  // namespace circatt
