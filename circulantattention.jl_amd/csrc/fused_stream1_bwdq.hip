// Instantiations of the streamed kernels, query-centric, up to 16 real
// components per head (fused_stream_impl.h).
#include "fused_stream_impl.h"

namespace circatt {

CIRCATT_FST_DEF(bwdq, fst::BWDQ, 1)

}  // namespace circatt
