// Instantiations of the streamed kernels, key-centric, up to 64 real
// components per head (fused_stream_impl.h).
#include "fused_stream_impl.h"

namespace circatt {

CIRCATT_FST_DEF(bwdkv, fst::BWDKV, 4)

}  // namespace circatt
