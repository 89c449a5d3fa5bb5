// Decode attention over 256-dim heads (tq_attn_rows.h): turbo K and V of one width, K wider than V, q8_0-style rows on either side.
#include "tq_attn_rows.h"

using namespace tqattn;

bool tqk_launch_decode_256(const AttnArgs &a, int kb, int vb, bool share, bool sparse, dim3 grid, unsigned wg, size_t lds, hipStream_t s) {
#define TQ_SAME(B) if (kb == B && vb == B && share) TQ_ATTN_256(KFMT_TURBO, B, B, true)
#define TQ_PAIR(KF, K, V) if (kb == (KF == KFMT_Q8 ? 8 : K) && vb == V) TQ_ATTN_256(KF, K, V, false)
    TQ_SAME(3) TQ_SAME(4) TQ_SAME(2)
    TQ_PAIR(KFMT_TURBO, 3, 3) TQ_PAIR(KFMT_TURBO, 4, 4) TQ_PAIR(KFMT_TURBO, 2, 2)
    TQ_PAIR(KFMT_TURBO, 4, 2) TQ_PAIR(KFMT_TURBO, 3, 2) TQ_PAIR(KFMT_TURBO, 4, 3)
    TQ_PAIR(KFMT_Q8, 3, 2) TQ_PAIR(KFMT_Q8, 3, 3) TQ_PAIR(KFMT_Q8, 3, 4) TQ_PAIR(KFMT_Q8, 3, 8)
    TQ_PAIR(KFMT_TURBO, 2, 8) TQ_PAIR(KFMT_TURBO, 3, 8) TQ_PAIR(KFMT_TURBO, 4, 8)
#undef TQ_SAME
#undef TQ_PAIR
    return false;
}
