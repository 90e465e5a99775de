// Any-layout chunked-prefill kernel for f16 queries over fp8 caches (see build.py for the flags).
#include "prefill_any.h"

namespace msattn {

MSATTN_DEFINE_PA(_Float16, fp8_t)

}  // namespace msattn
