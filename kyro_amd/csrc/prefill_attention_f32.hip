// prefill_attention.hip for f32 caches, in a translation unit of its own so that it compiles in
// parallel.
#define KYRO_PREFILL_UNIT 2
#include "prefill_attention.hip"
