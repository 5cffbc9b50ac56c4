// The f32 MFMA attention kernel at head dims 64, 80, 96 and 112, in a translation unit of its own so
// that its instances compile in parallel.
#define KYRO_ATTN_HD_UNIT 3
#include "paged_attention.hip"
