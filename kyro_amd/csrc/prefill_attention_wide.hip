// prefill_attention.hip at head dims 160, 192, 224 and 256, in a translation unit of its own so that
// it compiles in parallel.
#define KYRO_PREFILL_UNIT 1
#include "prefill_attention.hip"
