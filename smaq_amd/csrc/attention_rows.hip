// Scalar-key instances of the matrix-core row kernel (attention_rows.h) and
// the rule that says which calls take it.
#include <algorithm>
#include <cmath>

#include "attention_rows.h"

namespace smaq {

void launch_rows_vq(const smaq_attn_params& p, const HistAddr& a, const RowsRule& rule, float* slots,
                    const Partials& recent, hipStream_t st);

__global__ __launch_bounds__(256) void rows_combine_kernel(smaq_attn_params p, RowsRule rule, int step,
                                                           const float* __restrict__ slots, Partials recent) {
  const int ti = blockIdx.x, h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const RowsShares share = rows_shares(p, rule, step, lane);
  const uint32_t units = (uint32_t)(p.n_kv_heads * rule.tiles), u = (uint32_t)(h * rule.tiles + ti);
  const int64_t len = p.hist_len ? min((int64_t)p.hist_len[b], (int64_t)p.max_hist_len) : (int64_t)p.max_hist_len;
  const uint32_t steps = rows_steps(len, step);
  const uint32_t x = rows_sum_steps(p, step, b, lane) * units + u * steps;
  const uint32_t w0 = share.owner(x), w1 = share.owner(x + steps - 1);
  if (w0 == w1 && rule.n_recent == 0) return;  // written by its workgroup
  rows_merge<1>(p, rule, recent, slots + (int64_t)(w0 + (uint32_t)b * units + u) * kRowsSlot, (int)(w1 - w0) + 1, b, h,
                ti, tid, nullptr);
}

// query tokens: chunks of 64 and more are the prefill kernel's, the automatic
// choice for them being what an explicit impl 3 runs (callers compare the two
// bit for bit), although this kernel is the faster one beyond (30000 tokens,
// 32/8 heads, prefill / this kernel, us: 64 tokens 389 / 213, 128 427 / 386)
constexpr int kRowsMaxT = 63;

bool rows_supported(const smaq_attn_params& p) {
  const bool known = p.val_dtype == SMAQ_F32 || p.val_dtype == SMAQ_F16 || p.val_dtype == SMAQ_BF16;
  if (p.impl != 0 || !p.has_history || p.max_hist_len <= 0 || !p.arrivals || p.head_dim != 128 || !known) return false;
  if (p.q_len > kRowsMaxT || p.val_group != 32 || p.n_kv_heads > 65535 || p.batch > 65535) return false;
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

// Whether this kernel is the faster one, by estimated times in us over units of
// (sequence, KV head), tiles of 8 query rows here and of 16 in the generic
// kernels.  MI355X, whole plan, fitted to 5400 calls (1 to 800 sequences of 16 to
// 30000 tokens, 1 to 63 query tokens, windows of 0 to 16384, 28/4, 32/8 and 8/8
// heads): of the calls in bf16 that differ by more than 4% and 2 us, 84 take the
// slower kernel, by 21% at most.
//
// A unit costs this kernel a chain of round trips whatever its length.
//   Below 16 query tokens the generic kernels are ahead for many sequences of a
// few tokens with block-VQ keys (one workgroup of 8 waves a CU here), where the
// rows fill several tiles badly or a window makes the unit leave a partial: 512
// sequences of 16 tokens, 3 query tokens at 32/8 heads, 8-dim blocks, 293 us here,
// 217 there; of 100 tokens 310 and 430.
//   From 16 query tokens on the prefill kernel serves the call.  It decodes every
// key once into tile images and takes 256 query rows of one head at a time,
// mostly empty ones for a short chunk, where this kernel decodes a key once per
// tile, and the window beside it goes through the recent window's kernel, once
// per tile and without the matrix cores.  Prefill / this kernel: 30000 tokens,
// 32/8 heads, T = 16 344 / 75, 63 363 / 208; with a window of 4096 T = 63
// 448 / 343, of 16384 623 / 728; 500 tokens, T = 63, windows of 128, 1024, 4096
// 76 / 36, 88 / 81, 127 / 164; 512 sequences of 16 and 300 tokens of 8-dim
// block-VQ keys, T = 24, 28/4 heads 888 / 1586 and 1858 / 2008.
bool rows_preferred(const smaq_attn_params& p, bool prefill) {
  const bool scalar = p.key_format == SMAQ_KEY_SCALAR;
  const int g = p.n_q_heads / p.n_kv_heads, rows = p.q_len * g, tiles = (rows + kRowsQ - 1) / kRowsQ;
  const double units = (double)p.batch * p.n_kv_heads, hist = (double)p.max_hist_len;
  const double window = p.has_recent && p.max_recent_len > 0 ? (double)p.max_recent_len : 0.0;
  if (!prefill) {
    if (scalar || (tiles == 1 && window == 0.0)) return true;
    const double blocks = 128.0 / p.vq_block_dim, halves = (rows + 15) / 16;
    const double here = 8.4 + units * (tiles * (0.0323 + 20e-6 * hist) + (tiles > 1 ? 0.0085 : 0.0154));
    const double there = 22.8 + units * (halves * (0.0103 + 0.13e-3 * blocks + (1.08e-3 + 4.6e-6 * blocks) * hist) + 0.0018 * rows);
    return here <= there;
  }
  const bool split = prefill_split_len(p, p.max_hist_len) < p.max_hist_len;  // (a combine launch)
  // Only where its values are as exact in f16 as here: 2-bit codes with bf16 scales
  // and no fp32 window (error beside the generic kernels: 1e-7 to 1e-6 both; fp32
  // or fp16 scales or 4-bit codes 1e-5 to 2e-4 there).
  if (p.val_bits != 2 || p.val_dtype != SMAQ_BF16 || (window > 0.0 && p.recent_dtype == SMAQ_F32)) return true;
  // (the window's kernel takes chunks of 64 tokens)
  const double chunks = std::ceil(window / 64.0) * 9.5e-3;
  const double here = 14.5 + (window > 0.0 ? 9.0 : 0.0) +
                      units * tiles * ((scalar ? 0.0184 : 0.0369) + 26e-6 * hist + chunks);
  const double there = 20.2 + (split ? 8.0 : 0.0) + (window > 0.0 ? 21.9 : 0.0) +
                       units * (g * (0.0216 + 1.24e-3 * p.q_len + 0.217e-3 * hist + 0.358e-3 * window) +
                                0.011 + 0.478e-3 * hist + 0.64e-3 * window);
  return here <= there;
}

// Workgroups of the grid: what the device holds at once.
static RowsRule rows_rule(const smaq_attn_params& p, int n_recent) {
  RowsRule r;
  r.rows = p.q_len * (p.n_q_heads / p.n_kv_heads);
  r.tiles = (r.rows + kRowsQ - 1) / kRowsQ;
  const bool scalar = p.key_format == SMAQ_KEY_SCALAR;
  r.groups = device_cu_count() * (scalar ? 2 : 1);
  // A share of at least 512 tokens: a piece costs a partial and a load in the
  // merge (5 query tokens over 4001 and a window of 100, 4-bit keys and values,
  // whole call: shares from 128 / 256 / 512 / 1024 tokens 37.3 / 35.4 / 33.5 /
  // 37.6 us; 8-dim block-VQ keys from 256 / 512 / 1024 tokens 37.4 / 35.7 / 38.1).
  // But never several units that are whole each: 16 sequences of 16 tokens, 16
  // query tokens at 8/8 heads, 38.6 us with four units a share.
  const int step = kRowsTile * (scalar ? RowsKey<0>::kWaves : RowsKey<8>::kWaves);
  const int64_t steps = (p.max_hist_len + step - 1) / step;
  r.least = (int)std::min<int64_t>(scalar ? 4 : 2, steps);
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
  if (rule.tiles > 1) {
    const int step = (p.key_format == SMAQ_KEY_SCALAR ? RowsKey<0>::kWaves : RowsKey<8>::kWaves) * kRowsTile;
    hipLaunchKernelGGL(rows_combine_kernel, dim3((unsigned)rule.tiles, (unsigned)p.n_kv_heads, (unsigned)p.batch),
                       dim3(256), 0, st, p, rule, step, s, recent);
  }
  return launch_status("smaq_attn_hybrid(rows)");
}

}  // namespace smaq
