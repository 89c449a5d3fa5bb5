// Decode attention over 128-dim heads with q8_0-style rows on one side or both (tq_attn_rows.h).
#include "tq_attn_rows.h"

using namespace tqattn;

bool tqk_launch_decode_q8(const AttnArgs &a, int kb, int vb, int hg, bool sparse, dim3 grid, unsigned wg, size_t lds, hipStream_t s) {
#define TQ_PAIR(KF, K, V) if (kb == (KF == KFMT_Q8 ? 8 : K) && vb == V) TQ_ATTN_PAIR(KF, K, V, false)
    TQ_PAIR(KFMT_Q8, 3, 2) TQ_PAIR(KFMT_Q8, 3, 3) TQ_PAIR(KFMT_Q8, 3, 4) TQ_PAIR(KFMT_Q8, 3, 8)
    TQ_PAIR(KFMT_TURBO, 2, 8) TQ_PAIR(KFMT_TURBO, 3, 8) TQ_PAIR(KFMT_TURBO, 4, 8)
#undef TQ_PAIR
    return false;
}
