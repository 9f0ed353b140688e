// Scalar-key instances of the matrix-core row kernel (attention_rows.h) and
// the rule that says which calls take it.
#include "attention_rows.h"

namespace smaq {

void launch_rows_vq(const smaq_attn_params& p, const HistAddr& a, const RowsRule& rule, float* slots,
                    const Partials& recent, hipStream_t st);

bool rows_supported(const smaq_attn_params& p) {
  const bool known = p.val_dtype == SMAQ_F32 || p.val_dtype == SMAQ_F16 || p.val_dtype == SMAQ_BF16;
  if (p.impl != 0 || !p.has_history || p.max_hist_len <= 0 || !p.arrivals || p.head_dim != 128 || !known) return false;
  if (p.q_len >= 16 || p.val_group != 32) return false;
  if (!(p.val_bits == 2 && p.val_row_bytes == 32) && !(p.val_bits == 4 && p.val_row_bytes == 64)) return false;
  uintptr_t loads = (uintptr_t)p.val_bytes | (uintptr_t)p.q_hist | (uintptr_t)p.key_bytes | (uintptr_t)p.workspace;
  if (p.key_format == SMAQ_KEY_SCALAR) {
    if ((p.key_bits != 3 && p.key_bits != 4) || p.key_row_bytes != 64) return false;
    if (p.norm_dtype != SMAQ_F32 && p.norm_dtype != SMAQ_F16 && p.norm_dtype != SMAQ_BF16) return false;
  } else {
    if (p.vq_block_dim != 2 && p.vq_block_dim != 4 && p.vq_block_dim != 8) return false;
    if (p.vq_centroids < 1 || p.vq_centroids > 256 || p.key_row_bytes != 128 / p.vq_block_dim) return false;
    loads |= (uintptr_t)p.key_lut;  // codewords are read 8 or 16 bytes at a time
  }
  if (loads & 15) return false;
  // (steps are counted in 32 bits)
  const double units = (double)p.batch * p.n_kv_heads * ((p.q_len * (p.n_q_heads / p.n_kv_heads) + kRowsQ - 1) / kRowsQ);
  if (units * ((double)p.max_hist_len / 128.0 + 1.0) > 1e9 || units > 1e6) return false;
  // (16-token halves of a tile lie in one page)
  return !p.block_table || (p.block_size >= 16 && (p.block_size & (p.block_size - 1)) == 0);
}

// Workgroups of the grid: what the device holds at once.
static RowsRule rows_rule(const smaq_attn_params& p, int n_recent) {
  RowsRule r;
  r.rows = p.q_len * (p.n_q_heads / p.n_kv_heads);
  r.tiles = (r.rows + kRowsQ - 1) / kRowsQ;
  const bool scalar = p.key_format == SMAQ_KEY_SCALAR;
  r.groups = device_cu_count() * (scalar ? 2 : 1);
  // A share of at least 512 tokens: a piece costs a partial and a load in the
  // merge (5 query tokens over 4001, whole call: shares from 128 / 256 / 512
  // tokens 177 / 155 / 148 us).
  r.least = scalar ? 4 : 2;
  r.n_recent = n_recent;
  return r;
}

int64_t rows_bytes(const smaq_attn_params& p) {
  const RowsRule r = rows_rule(p, 0);
  return ((int64_t)r.groups + (int64_t)p.batch * p.n_kv_heads * r.tiles) * kRowsSlot * (int64_t)sizeof(float);
}

int launch_rows(const smaq_attn_params& p, const HistAddr& a, void* slots, const Partials& recent, int n_recent,
                hipStream_t st) {
  const RowsRule rule = rows_rule(p, n_recent);
  float* const s = (float*)slots;
  if (p.key_format != SMAQ_KEY_SCALAR) {
    launch_rows_vq(p, a, rule, s, recent, st);
  } else {
    const bool two = p.val_bits == 2;
    switch (p.norm_dtype) {
      case SMAQ_F32: two ? launch_rows_v<0, 2, float>(p, a, rule, s, recent, st) : launch_rows_v<0, 4, float>(p, a, rule, s, recent, st); break;
      case SMAQ_F16: two ? launch_rows_v<0, 2, _Float16>(p, a, rule, s, recent, st) : launch_rows_v<0, 4, _Float16>(p, a, rule, s, recent, st); break;
      default: two ? launch_rows_v<0, 2, bf16>(p, a, rule, s, recent, st) : launch_rows_v<0, 4, bf16>(p, a, rule, s, recent, st); break;
    }
  }
  return launch_status("smaq_attn_hybrid(rows)");
}

}  // namespace smaq
