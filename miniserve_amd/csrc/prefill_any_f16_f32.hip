// Any-layout chunked-prefill kernel for f16 queries over f32 caches (see build.py for the flags).
#include "prefill_any.h"

namespace msattn {

MSATTN_DEFINE_PA(_Float16, float)

}  // namespace msattn
