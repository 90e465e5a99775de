// Any-layout chunked-prefill kernel for bf16 queries over bf16 caches (see build.py for the flags).
#include "prefill_any.h"

namespace msattn {

MSATTN_DEFINE_PA(bf16_t, bf16_t)

}  // namespace msattn
