// Instantiations of the streamed kernels, forward, up to 64 real
// components per head (fused_stream_impl.h).
#include "fused_stream_impl.h"

namespace circatt {

CIRCATT_FST_DEF(fwd, fst::FWD, 4)

}  // namespace circatt
