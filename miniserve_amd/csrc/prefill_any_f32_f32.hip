// Any-layout chunked-prefill kernel for f32 queries over f32 caches (see build.py for the flags).
#include "prefill_any.h"

namespace msattn {

MSATTN_DEFINE_PA(float, float)

}  // namespace msattn
