// Block-VQ instances of the matrix-core row kernel (attention_rows.h).
#include "attention_rows.h"

namespace smaq {

template <int KEY>
static void launch_b(const smaq_attn_params& p, const HistAddr& a, const RowsRule& rule, float* slots,
                     const Partials& recent, hipStream_t st) {
  if (p.val_bits == 2) launch_rows_v<KEY, 2, bf16>(p, a, rule, slots, recent, st);
  else launch_rows_v<KEY, 4, bf16>(p, a, rule, slots, recent, st);
}

void launch_rows_vq(const smaq_attn_params& p, const HistAddr& a, const RowsRule& rule, float* slots,
                    const Partials& recent, hipStream_t st) {
  switch (p.vq_block_dim) {
    case 2: launch_b<2>(p, a, rule, slots, recent, st); break;
    case 4: launch_b<4>(p, a, rule, slots, recent, st); break;
    default: launch_b<8>(p, a, rule, slots, recent, st); break;
  }
}

}  // namespace smaq
