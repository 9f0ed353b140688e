// Decode attention on the matrix cores for the shapes that the 4-query-row
// kernel of attention_mfma.hip does not take: block-VQ keys (blocks of 2, 4
// or 8 dims), up to 8 query rows per pass (wide GQA groups, or the rows of a
// few query tokens, causal or not), 2- or 4-bit values.  head_dim 128, value
// groups of 32.
//
// Work split.  Every (sequence, KV head, tile of 8 query rows) is a unit of
// ceil(length / step) steps, and the steps of all units, in order, are dealt
// in equal contiguous shares to as many workgroups as the device runs at
// once: no last round that is nearly empty, whatever the batch, the head
// count and the raggedness, and a workgroup stages its key table once.  A
// unit's tokens are thus cut where a share ends; each piece leaves a partial
// in slot (workgroup + unit), which is unique because either index moves on
// at every cut, and the last piece to arrive merges the unit in piece order
// (rows_combine_kernel does, where a KV head has several tiles).
//
// Per 32-token tile of a wave (two 16-token halves):
//   QK   v_mfma_f32_16x16x32_f16, S^T = K q^T: M = 16 tokens, N = 16 columns
//        (query row r's hi part in column r, its lo part in column 8 + r).
//        A key code becomes its f16 hi/lo pair by one LDS read of a table of
//        all codes (scalar keys: 256 code bytes; block-VQ: every codeword of
//        every block, 128 KB, one workgroup of 8 waves per CU), both halves
//        scaled by a power of two per block that keeps the lo part normal.
//   soft a lane keeps the four tokens of its column's half (columns 0-7 the
//        first, 8-15 the second): the scores need one rotation by 8 lanes,
//        and no LDS.  Base 2, reference raised lazily (attention_mfma.hip),
//        lowered by the exponent of the largest weight * scale so that those
//        products stay inside f16, whatever the scales of tokens of little
//        weight; value groups far apart get a power of two each.
//   PV   v_mfma_f32_16x16x32_f16, O^T = V^T P^T per value group: B is
//        weight * scale split f16 hi (columns 0-7) / lo (8-15), ~22 bits,
//        which the softmax lanes hold in place (the tokens of the K slots are
//        numbered by it); A is the value codes about their middle,
//        (code - mid) * 2^-10: the code bits masked in place are an f16
//        subnormal, and one packed FMA scales and centres it, exactly.
// The zero points, moved by mid * scale, are summed in fp32.  Centred, the two
// sums do not cancel (codes from zero up against the groups' minima left
// 6.3e-6 of relative error at 30000 fp32 tokens, the generic kernel 4.2e-7).
// The QK and PV products are accumulated in fp32 and carry ~22 bits of each
// operand.
//
// What bounds it: VALU issue (349 per tile: 71% of the cycles at 16 x 32768
// tokens of 8-dim block-VQ keys).  Measured, whole call, before (generic
// kernels) and now: that batch at 32/8 heads 4326 -> 114 us (2.3 TB/s of
// 64-byte rows), 64 paged sequences of up to 8000 tokens of 3-bit keys at
// 28/4 heads 2899 -> 68 us (1.8 TB/s of 114-byte rows); its kernel alone over
// one sequence of 65408 tokens of 2-dim block-VQ keys at 28/4 heads 339 (and
// 33 to combine) -> 35 us.
#pragma once

#include "decode_common.h"

namespace smaq {

constexpr int kRowsQ = 8;          // query rows per unit
constexpr int kRowsTile = 32;      // tokens per wave and tile
constexpr int kRowsPitch = 80;     // bytes per code-byte row of the spread value tile
constexpr int kRowsVBytes = 32;    // code bytes of a token per PV pass
// floats of a partial: m[8], l[8], o[8][128]
constexpr int kRowsSlot = kRowsQ * (2 + 128);

// key codes: scalar (3/4 bits, two per byte), or block-VQ by block_dim
template <int KEY>
struct RowsKey {
  static constexpr bool kVq = KEY != 0;
  static constexpr int kLaneBytes = KEY == 8 ? 4 : (KEY == 4 ? 8 : 16);  // code bytes of a lane's 32 dims
  static constexpr int kRowBytes = 4 * kLaneBytes;
  static constexpr int kTable = kVq ? 128 * 256 * 4 : 256 * 8;
  static constexpr int kWaves = kVq ? 8 : 4;                  // per workgroup
};

// The f16 pairs of weight * scale: a row's largest product so far is brought
// to [2^kPairExp, 2^(kPairExp + 1)) and may come to 2^kPairTop (and 0.09 of an
// octave, the error of a log2 taken from a number's bits; f16 ends at 2^16)
// before the exponent follows.  A pair holds 22 bits of a product and multiples
// of 2^-24, so a value group's sum keeps 28 bits or more below its largest
// product (with kPairApart); a higher kPairExp costs the weights' exponents bits.
// (One exponent that followed the largest scale alone lost 2e-3 of the other
// groups beside a channel 1e6 times theirs.  Following products, group by group:
// 64 paged sequences of heavy-tailed keys 62.7 -> 64.0 us, other calls the same.)
constexpr int kPairExp = 6;
constexpr float kPairTop = 15.5f;
constexpr int kPairApart = 2;

// buffer-load policy sc1: agent-coherent, as load_agent
constexpr int kAgentPolicy = 16;

struct RowsRule {
  int rows;     // query rows per (sequence, KV head)
  int tiles;    // units per (sequence, KV head): ceil(rows / 8)
  int groups;   // workgroups of the grid
  int least;    // steps of the smallest share
  int n_recent; // recent partials per row (0: none)
};

typedef _Float16 rf16x2 __attribute__((ext_vector_type(2)));

// The steps of every unit and how they are dealt to workgroups.
struct RowsShares {
  uint32_t total, groups;  // steps; workgroups that have a share
  uint32_t each, more;     // the first `more` shares hold each + 1 steps, the others `each`
  __device__ __forceinline__ uint32_t start(uint32_t w) const { return w * each + min(w, more); }
  // the workgroup whose share holds step y
  __device__ __forceinline__ uint32_t owner(uint32_t y) const {
    const uint32_t low = more * (each + 1);
    return y < low ? y / (each + 1) : more + (y - low) / each;
  }
};

__device__ __forceinline__ uint32_t rows_steps(int64_t len, int step) {
  return len > 0 ? (uint32_t)((len + step - 1) / step) : 1u;
}

// `before`: the steps of one unit of every sequence below b_end, summed (by
// the wave; every lane gets it).
__device__ __forceinline__ uint32_t rows_sum_steps(const smaq_attn_params& p, int step, int b_end, int lane) {
  if (!p.hist_len) return rows_steps(p.max_hist_len, step) * (uint32_t)b_end;
  uint32_t sum = 0;
  for (int b = lane; b < b_end; b += 64)
    sum += rows_steps(min((int64_t)p.hist_len[b], (int64_t)p.max_hist_len), step);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) sum += (uint32_t)__shfl_xor((int)sum, o, 64);
  return (uint32_t)__builtin_amdgcn_readfirstlane(sum);
}

__device__ __forceinline__ RowsShares rows_shares(const smaq_attn_params& p, const RowsRule& rule, int step, int lane) {
  RowsShares s;
  s.total = rows_sum_steps(p, step, p.batch, lane) * (uint32_t)(p.n_kv_heads * rule.tiles);
  s.groups = min((uint32_t)rule.groups, (s.total + rule.least - 1) / rule.least);
  s.each = (uint32_t)__builtin_amdgcn_readfirstlane(s.total / s.groups);
  s.more = s.total - s.each * s.groups;
  return s;
}

// x0, x1 -> packed f16 hi pair and packed f16 pair of what it leaves; `one`
// is an opaque 1.0 (keeps x - hi a mixed-precision FMA)
__device__ __forceinline__ void rows_split2(float x0, float x1, float one, uint32_t& hi, uint32_t& lo) {
  const rf16x2 h = __builtin_convertvector((f32x2){x0, x1}, rf16x2);
  const f32x2 r = {__builtin_fmaf(one, x0, -(float)h[0]), __builtin_fmaf(one, x1, -(float)h[1])};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, rf16x2));
}

// the largest of a query row's 8 lanes (n, n ^ 8 in each 16-lane row)
__device__ __forceinline__ float rows_max8(float x) {
  auto number = [](uint32_t bits) -> float { return __builtin_bit_cast(float, bits); };
  x = fmaxf(x, dpp_row_ror<0x128>(x));
  uint32_t b = __builtin_bit_cast(uint32_t, x);
  const auto p = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  x = fmaxf(number(p[0]), number(p[1]));
  b = __builtin_bit_cast(uint32_t, x);
  const auto q = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  return fmaxf(number(q[0]), number(q[1]));
}

template <int CTRL, int BANKS>
__device__ __forceinline__ uint32_t dpp_bank_move_u(uint32_t old, uint32_t src) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, 0xf, BANKS, false);
}

// N dwords at an address of any alignment
template <int N>
struct __attribute__((packed, aligned(1))) Loose {
  uint32_t w[N];
};
template <int N>
__device__ __forceinline__ void load_loose(const void* src, uint32_t* dst) {
  const Loose<N> v = *(const Loose<N>*)src;
#pragma unroll
  for (int i = 0; i < N; ++i) dst[i] = v.w[i];
}

// element i of storage values kept as loaded
template <typename T>
__device__ __forceinline__ float packed_get(const uint32_t* w, int i) {
  if constexpr (sizeof(T) == 2) return Num<T>::to_f(__builtin_bit_cast(T, (uint16_t)(w[i >> 1] >> (16 * (i & 1)))));
  else return __builtin_bit_cast(float, w[i]);
}
template <typename T>
__device__ __forceinline__ void packed_set(uint32_t* w, int i, T v) {
  if constexpr (sizeof(T) == 2) {
    const uint32_t bits = (uint32_t)__builtin_bit_cast(uint16_t, v);
    w[i >> 1] = (i & 1) ? ((w[i >> 1] & 0xffffu) | (bits << 16)) : bits;
  } else {
    w[i] = __builtin_bit_cast(uint32_t, v);
  }
}

// Two waves per SIMD: with block-VQ keys one workgroup of 8 waves fills a CU
// (its table fills the LDS), with scalar keys two of 4.  (Scalar keys at three
// per SIMD have 168 registers and spill 38: 80.2 against 66.9 us for 64 paged
// sequences of up to 8000 tokens at 28/4 heads.)
constexpr int kRowsPerSimd = 2;


// Merge of one unit (query rows of tile ti of KV head h, sequence b): its np
// partials from `first` on and the recent window's, in that order, by kParts x
// 256 threads (256: 8 rows x 32 dim quads; with 512 the two halves take
// alternate pieces).  A merge is a chain of memory round trips, so each has
// many loads in flight.  `ex`: 11 KB of LDS (kParts 2).
template <int kParts>
__device__ __forceinline__ void rows_merge(const smaq_attn_params& p, const RowsRule& rule, const Partials& recent,
                                           const float* first, int np, int b, int h, int ti, int tid, float* ex) {
  constexpr int kDeep = 8;
  constexpr float kLog2e = 1.4426950408889634f;
  const int g = p.n_q_heads / p.n_kv_heads;
  const int part = tid >> 8, r = (tid & 255) >> 5, d = 4 * (tid & 31);
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(first), (short)0, -1, 0x00020000);
  const int row = ti * kRowsQ + r, n_all = np + rule.n_recent;
  const int64_t rbase =
      rule.n_recent > 0 ? recent.idx(b, h, p.n_kv_heads, rule.rows, min(row, rule.rows - 1), 0) : 0;
  float M = -__builtin_inff(), L = 0.0f;
  f32x4 oh = {0.0f, 0.0f, 0.0f, 0.0f}, orc = oh;
  bool poisoned = false;  // a partial's sum is NaN
  for (int c0 = part; c0 < n_all; c0 += kParts * kDeep) {
    float mv[kDeep], lv[kDeep];
    f32x4 ov[kDeep];
#pragma unroll
    for (int k = 0; k < kDeep; ++k) {
      const int c = c0 + k * kParts;
      mv[k] = -__builtin_inff();
      lv[k] = 0.0f;
      ov[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (c < np) {  // (agent-coherent: written through by the other workgroups)
        const int off = c * kRowsSlot * 4;
        mv[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, r * 4, off, kAgentPolicy));
        lv[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (kRowsQ + r) * 4, off, kAgentPolicy));
        ov[k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    rs, (2 * kRowsQ + r * 128 + d) * 4, off, kAgentPolicy));
      } else if (c < n_all) {  // the recent window's partials (natural-log maxima)
        const int64_t ri = rbase + (c - np);
        mv[k] = recent.m[ri] * kLog2e;
        lv[k] = recent.l[ri];
        ov[k] = *(const f32x4*)&recent.o[ri * 128 + d];
      }
    }
    float Mc = M;
#pragma unroll
    for (int k = 0; k < kDeep; ++k) {
      poisoned |= lv[k] != lv[k];
      Mc = lv[k] > 0.0f ? fmaxf(Mc, mv[k]) : Mc;
    }
    const float c = M == -__builtin_inff() ? 0.0f : fast_exp2(M - Mc);
    L *= c;
    oh *= c;
    orc *= c;
    M = Mc;
#pragma unroll
    for (int k = 0; k < kDeep; ++k) {
      const bool live = lv[k] > 0.0f;
      const float wk = live ? fast_exp2(mv[k] - M) : 0.0f;
      L = live ? fmaf(lv[k], wk, L) : L;
      const bool hist = c0 + k * kParts < np;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = live ? ov[k][i] : 0.0f;
        oh[i] = fmaf(v, hist ? wk : 0.0f, oh[i]);
        orc[i] = fmaf(v, hist ? 0.0f : wk, orc[i]);
      }
    }
  }
  if constexpr (kParts == 2) {
    __syncthreads();
    float* const e = ex + (tid & 255);
    if (part == 1) {
      e[0] = L;
      ((uint32_t*)e)[10 * 256] = poisoned ? 1u : 0u;
      e[256] = M;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        e[(2 + i) * 256] = oh[i];
        e[(6 + i) * 256] = orc[i];
      }
    }
    __syncthreads();
    if (part == 0) {
      const float L2 = e[0], M2 = e[256];
      poisoned |= ((const uint32_t*)e)[10 * 256] != 0u;
      const float Mc = fmaxf(M, M2);
      const float f1 = L > 0.0f ? fast_exp2(M - Mc) : 0.0f, f2 = L2 > 0.0f ? fast_exp2(M2 - Mc) : 0.0f;
      L = L * f1 + (f2 > 0.0f ? L2 * f2 : 0.0f);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        oh[i] = oh[i] * f1 + e[(2 + i) * 256] * f2;
        orc[i] = orc[i] * f1 + e[(6 + i) * 256] * f2;
      }
    }
    __syncthreads();
  }
  if (part != 0 || row >= rule.rows) return;
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  const int t = row / g, j = row - t * g;
  const int64_t oi = (((int64_t)b * p.q_len + t) * p.n_q_heads + (int64_t)h * g + j) * 128 + d;
  float o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[i] = oh[i] * inv;
    // history and recent outputs each in the output dtype, then added
    if (rule.n_recent > 0) o[i] = round_out(p, round_out(p, o[i]) + round_out(p, orc[i] * inv));
    o[i] = poisoned ? kQuietNaN : o[i];
  }
  store_out2(p, oi, o[0], o[1]);
  store_out2(p, oi + 2, o[2], o[3]);
}

// The units of a (sequence, KV head) with several row tiles, merged by one
// workgroup each (the shares as attn_rows_kernel computes them).
__global__ __launch_bounds__(256) void rows_combine_kernel(smaq_attn_params p, RowsRule rule, int step,
                                                           const float* __restrict__ slots, Partials recent);

template <int KEY, int VB, typename TN, typename TV>
__global__ __launch_bounds__(RowsKey<KEY>::kWaves * 64)
    __attribute__((amdgpu_waves_per_eu(kRowsPerSimd, kRowsPerSimd))) void attn_rows_kernel(
        smaq_attn_params p, HistAddr addr, RowsRule rule, float* __restrict__ slots, Partials recent) {
  using K = RowsKey<KEY>;
  constexpr int NW = K::kWaves;
  constexpr int kThreads = NW * 64;
  constexpr int64_t kStep = NW * kRowsTile;
  constexpr int kVRowBytes = VB == 2 ? 32 : 64;      // value code bytes per token
  constexpr int kPasses = kVRowBytes / kRowsVBytes;  // PV passes (32 code bytes each)
  constexpr int kGroups = 4 / kPasses;               // value groups per pass
  constexpr int kNW = sizeof(TN) == 2 ? 2 : 4;       // dwords of four norms
  constexpr int kSW = sizeof(TV) == 2 ? 8 : 16;      // dwords of 4 tokens x 4 groups
  __shared__ __attribute__((aligned(16))) uint8_t table[K::kTable];
  __shared__ __attribute__((aligned(16))) uint8_t vsp[NW][kRowsVBytes * kRowsPitch];
  __shared__ float red_m[NW][kRowsQ], red_l[NW][kRowsQ];
  __shared__ int flag;
  __shared__ int blk_e[K::kVq ? 128 / KEY : 1];  // the blocks' powers of two
  // per-wave outputs of 64 dims, laid over the value tiles between units
  float (*const red_o)[kRowsQ][64] = (float (*)[kRowsQ][64])&vsp[0][0];
  static_assert(sizeof(vsp[0]) >= sizeof(float) * kRowsQ * 64, "red_o");

  const int tid = (int)threadIdx.x;
  const int wg = (int)blockIdx.x;
  const int lane = tid & 63;
  const int wu = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kg = lane >> 4;
  const bool first = n < 8;                      // column half: hi parts, tokens 0-15
  const int q8 = n & 7;
  const int tok0 = 4 * kg + (first ? 0 : 16);    // this lane's softmax tokens tok0 .. tok0 + 3
  const int tq = lane & 7, pq = lane >> 3;       // value loader: tokens 4tq.., bytes 4pq..
  typedef const __attribute__((address_space(4))) int* ConstIntPtr;
  typedef const __attribute__((address_space(4))) int64_t* ConstI64Ptr;
  constexpr float kLog2e = 1.4426950408889634f;
  float one = 1.0f;
  asm volatile("" : "+v"(one));

  // ---- this workgroup's share [x, x_end) of the steps
  const uint32_t per_seq = (uint32_t)(p.n_kv_heads * rule.tiles);  // units per sequence
  auto steps_of = [&](int64_t len) -> uint32_t { return rows_steps(len, (int)kStep); };
  auto length_of = [&](int b) -> int64_t {
    return uniform64(p.hist_len ? min(max(((ConstI64Ptr)p.hist_len)[b], (int64_t)0), (int64_t)p.max_hist_len)
                                : (int64_t)p.max_hist_len);
  };
  const RowsShares share = rows_shares(p, rule, (int)kStep, lane);
  if ((uint32_t)wg >= share.groups) return;
  uint32_t x = share.start((uint32_t)wg);
  const uint32_t x_end = share.start((uint32_t)wg + 1);
  auto owner = [&](uint32_t y) -> uint32_t { return share.owner(y); };
  // the sequence of step x, and the steps before it
  int b = 0;
  uint32_t x_seq = 0;  // first step of sequence b
  if (p.hist_len) {
    const uint32_t want = x / per_seq;
    uint32_t before = 0;
    for (int b0 = 0; b0 < p.batch; b0 += 64) {
      const int bi = b0 + lane;
      const uint32_t st = bi < p.batch ? steps_of(min((int64_t)p.hist_len[bi], (int64_t)p.max_hist_len)) : 0u;
      uint32_t inc = st;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t up = (uint32_t)__shfl_up((int)inc, o, 64);
        if (lane >= o) inc += up;
      }
      const uint64_t past = __ballot(before + inc > want);
      if (past) {
        const int i = __builtin_ctzll(past);
        b = b0 + i;
        x_seq = (before + (uint32_t)__shfl((int)(inc - st), i, 64)) * per_seq;
        break;
      }
      before += (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)inc, 63, 64));
    }
  } else {
    const uint32_t per = steps_of(p.max_hist_len) * per_seq;
    b = (int)(x / per);
    x_seq = (uint32_t)b * per;
  }
  b = __builtin_amdgcn_readfirstlane(b);
  x_seq = (uint32_t)__builtin_amdgcn_readfirstlane(x_seq);

  // ---- key table, each block (scalar keys: all of it) scaled by a power of two
  // that brings its largest entry to [2^13, 2^14): the lo parts of entries down
  // to 2^-17 of it are normal f16.  A block's own power goes into the query's
  // dims, so blocks of any size count alike.
  auto finite = [](float x) -> float { return fabsf(x) < __builtin_inff() ? fabsf(x) : 0.0f; };
  auto exponent = [](float x) -> int { return max(exponent_of(x) - 13, -126); };
  int e_k = 0;
  if constexpr (K::kVq) {
    constexpr int kTpb = kThreads * KEY / 128;  // threads of a block
    constexpr int kPer = 256 / kTpb;            // codewords per thread
    const int nc = p.vq_centroids;
    const int blk = tid / kTpb, sub = tid % kTpb;
    // (rotated by block, so that a wave's writes cover all LDS banks)
    auto code = [&](int i) -> int { return sub + kTpb * ((i + blk) % kPer); };
    float c[kPer][KEY];
    float cmax = 0.0f;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const float* src = p.key_lut + ((int64_t)blk * nc + min(code(i), nc - 1)) * KEY;
      if constexpr (KEY == 2) {
        const float2 v = *(const float2*)src;
        c[i][0] = v.x; c[i][1] = v.y;
      } else {
#pragma unroll
        for (int d = 0; d < KEY; d += 4) {
          const float4 v = *(const float4*)(src + d);
          c[i][d] = v.x; c[i][d + 1] = v.y; c[i][d + 2] = v.z; c[i][d + 3] = v.w;
        }
      }
#pragma unroll
      for (int d = 0; d < KEY; ++d) cmax = fmaxf(cmax, finite(c[i][d]));
    }
#pragma unroll
    for (int o = 1; o < kTpb; o <<= 1) cmax = fmaxf(cmax, __shfl_xor(cmax, o, 64));
    const int e_b = exponent(cmax);
    if (sub == 0) blk_e[blk] = e_b;
    const float ks = ldexpf(1.0f, -e_b);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int e = blk * 256 + code(i);
      uint32_t hi[KEY / 2], lo[KEY / 2];
#pragma unroll
      for (int d = 0; d < KEY; d += 2) rows_split2(c[i][d] * ks, c[i][d + 1] * ks, one, hi[d / 2], lo[d / 2]);
      if constexpr (KEY == 2) *(u32x2*)&table[e * 8] = u32x2{hi[0], lo[0]};
      if constexpr (KEY == 4) *(u32x4*)&table[e * 16] = u32x4{hi[0], hi[1], lo[0], lo[1]};
      if constexpr (KEY == 8) {
        *(u32x4*)&table[e * 16] = u32x4{hi[0], hi[1], hi[2], hi[3]};
        *(u32x4*)&table[65536 + e * 16] = u32x4{lo[0], lo[1], lo[2], lo[3]};
      }
    }
  } else {
    const int nc = 1 << p.key_bits;
    float cmax = 0.0f;
    for (int i = 0; i < nc; ++i) cmax = fmaxf(cmax, finite(p.key_lut[i]));
    e_k = exponent(cmax);
    const float ks = ldexpf(1.0f, -e_k);
    static_assert(K::kVq || kThreads == 256, "one table entry per thread");
    uint32_t hi, lo;
    rows_split2(p.key_lut[tid & (nc - 1)] * ks, p.key_lut[(tid >> p.key_bits) & (nc - 1)] * ks, one, hi, lo);
    *(u32x2*)&table[tid * 8] = u32x2{hi, lo};
  }
  __syncthreads();

  const uint8_t* kbytes = (const uint8_t*)p.key_bytes;
  const uint8_t* vbytes = (const uint8_t*)p.val_bytes;
  const TN* norms = (const TN*)p.key_norms;
  const TV* vsc = (const TV*)p.val_scales;
  const TV* vzr = (const TV*)p.val_zeros;
  const bool paged = __builtin_amdgcn_readfirstlane(addr.table != nullptr ? 1 : 0) != 0;
  const int bshift = paged ? __builtin_ctz((unsigned)addr.block_size) : 0;
  const uint32_t bmask = paged ? (uint32_t)addr.block_size - 1u : 0u;
  typedef const __attribute__((address_space(3))) uint8_t* LdsBytes;
  typedef const __attribute__((address_space(3))) u32x2* LdsPair;
  typedef const __attribute__((address_space(3))) u32x4* LdsQuad;
  const LdsBytes tb = (LdsBytes)&table[0] + (K::kVq ? kg * 32768 / (KEY == 8 ? 2 : 1) : 0);
  uint8_t* const vw = &vsp[wu][kRowsPitch * 4 * pq + (tq < 4 ? 16 * tq : 16 * (tq - 4) + 8)];
  const uint8_t* const vr = &vsp[wu][kRowsPitch * (VB == 2 ? n >> 1 : n) + 16 * kg];
  // the two code fields of a spread byte that this lane's value row (dims
  // 2n, 2n + 1 of a group) takes: 2-bit codes share a byte with the
  // neighbouring row, 4-bit codes fill it
  const uint32_t mask0 = VB == 2 ? 0x00030003u << (4 * (n & 1)) : 0x000f000fu;
  const uint32_t mask1 = mask0 << VB;
  // 2^(14 - field shift), and the middle code, as packed f16 pairs
  constexpr float kMid = VB == 2 ? 1.5f : 7.5f;
  const rf16x2 mul0 = (rf16x2)(_Float16)(VB == 2 && (n & 1) ? 1024.0f : 16384.0f);
  const rf16x2 mul1 = mul0 * (rf16x2)(_Float16)(VB == 2 ? 0.25f : 0.0625f);
  const rf16x2 mid = (rf16x2)(_Float16)(-kMid / 1024.0f);

  // ---- units
  while (x < x_end) {
    const int64_t len = length_of(b);
    const uint32_t steps = steps_of(len);
    const uint32_t rel = x - x_seq;
    if (rel >= steps * per_seq) {  // past sequence b
      x_seq += steps * per_seq;
      ++b;
      continue;
    }
    const uint32_t uis = (uint32_t)__builtin_amdgcn_readfirstlane(rel / steps);  // unit in the sequence
    const uint32_t st0 = rel - uis * steps, st1 = min(steps, st0 + (x_end - x));
    const uint32_t x_unit = x - st0;                     // the unit's first step
    const int h = (int)__builtin_amdgcn_readfirstlane(uis / (uint32_t)rule.tiles);
    const int rt = (int)uis - h * rule.tiles;
    const uint32_t unit = (uint32_t)b * per_seq + uis;
    const int64_t s0 = uniform64((int64_t)st0 * kStep);
    const int64_t s1 = uniform64(min(len, (int64_t)st1 * kStep));
    x += st1 - st0;

    const int g = p.n_q_heads / p.n_kv_heads;
    const int nr = min(kRowsQ, rule.rows - rt * kRowsQ);  // live rows
    // element offset of query row r (of this unit) in [batch][q_len][Hq][128]
    auto row_off = [&](int r) -> int64_t {
      const int row = rt * kRowsQ + r, t = row / g, j = row - t * g;
      return (((int64_t)b * p.q_len + t) * p.n_q_heads + (int64_t)h * g + j) * 128;
    };
    // ---- query operands
    u32x4 bq[8];
    float rfac;
    {
      float qv[32];
      const float* src = p.q_hist + row_off(q8 < nr ? q8 : 0) + 32 * kg;
#pragma unroll
      for (int i = 0; i < 32; i += 4) {
        const float4 v4 = *(const float4*)(src + i);
        qv[i] = v4.x; qv[i + 1] = v4.y; qv[i + 2] = v4.z; qv[i + 3] = v4.w;
      }
      float qmax = 0.0f;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        qv[i] = q8 < nr ? qv[i] : 0.0f;
        if constexpr (K::kVq) qv[i] = __builtin_amdgcn_ldexpf(qv[i], blk_e[(32 * kg + i) / KEY]);
        qmax = fmaxf(qmax, fabsf(qv[i]));
      }
      qmax = fmaxf(qmax, __shfl_xor(qmax, 16, 64));
      qmax = fmaxf(qmax, __shfl_xor(qmax, 32, 64));
      const int e_q = exponent(qmax);
      // The scores are masked (-inf) and their largest found ahead of `rfac`,
      // which has to be positive: the sign of a negative scale goes into the
      // query, and so does a scale of zero or NaN.
      const bool positive = p.scale > 0.0f, negative = p.scale < 0.0f;
      const float qs = ldexpf(positive ? 1.0f : negative ? -1.0f : p.scale, -e_q);
      rfac = fmaxf(ldexpf((positive || negative ? fabsf(p.scale) : 1.0f) * kLog2e, e_q + e_k), 0x1p-126f);
      // the hi (first half) or lo part, met with the keys' hi and lo parts
      uint32_t xw[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        uint32_t hi, lo;
        rows_split2(qv[2 * i] * qs, qv[2 * i + 1] * qs, one, hi, lo);
        xw[i] = first ? hi : lo;
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if constexpr (KEY == 8) {
          const int i = 4 * (t >> 1);
          bq[t] = u32x4{xw[i], xw[i + 1], xw[i + 2], xw[i + 3]};
        } else if constexpr (KEY == 4) {
          bq[t] = u32x4{xw[2 * t], xw[2 * t + 1], xw[2 * t], xw[2 * t + 1]};
        } else {
          bq[t] = u32x4{xw[2 * t], xw[2 * t], xw[2 * t + 1], xw[2 * t + 1]};
        }
      }
    }
    // causal limit of this lane's query row, as a token index (and the
    // smallest of the unit's rows: tiles below it need no mask)
    int64_t qlim = len, qlim_min = len;
    if (p.q_positions) {
      const int row = rt * kRowsQ + (q8 < nr ? q8 : 0);
      qlim = p.q_positions[(int64_t)b * p.q_len + row / g] - p.hist_pos_offset;
      qlim_min = p.q_positions[(int64_t)b * p.q_len + (rt * kRowsQ) / g] - p.hist_pos_offset;
      for (int r = 1; r < nr; ++r)
        qlim_min = min(qlim_min, (int64_t)p.q_positions[(int64_t)b * p.q_len + (rt * kRowsQ + r) / g] - p.hist_pos_offset);
      qlim_min = uniform64(qlim_min);
    }

    // ---- rows
    const int64_t base = uniform64(paged ? 0 : (int64_t)h * addr.head_stride +
        (addr.seq_start ? ((ConstI64Ptr)addr.seq_start)[b] : (int64_t)b * addr.uniform_len));
    const ConstIntPtr tbl =
        (ConstIntPtr)uniform64(paged ? (int64_t)(uintptr_t)(addr.table + (int64_t)b * addr.max_blocks) : 0);
    struct Desc {
      int64_t gA, gB;  // rows of tokens 0 and 16
      int last;        // the last valid token
    };
    auto entries = [&](int64_t t, uint32_t& ea, uint32_t& eb) {
      ea = eb = 0;
      if (paged) {
        const uint32_t ta = (uint32_t)t, tc = (uint32_t)min(t + 16, s1 - 1);
        ea = (uint32_t)__builtin_amdgcn_readfirstlane(tbl[ta >> bshift]);
        eb = (uint32_t)__builtin_amdgcn_readfirstlane(tbl[tc >> bshift]);
      }
    };
    auto rows_at = [&](int64_t t, uint32_t ea, uint32_t eb) -> Desc {
      Desc d;
      d.last = __builtin_amdgcn_readfirstlane((int)min((int64_t)31, s1 - 1 - t));
      if (paged) {
        const uint32_t tt = (uint32_t)t;
        d.gA = (int64_t)((uint64_t)((int64_t)(int)ea * addr.n_kv + h) << bshift) + (int64_t)(tt & bmask);
        d.gB = (int64_t)((uint64_t)((int64_t)(int)eb * addr.n_kv + h) << bshift) + (int64_t)((tt + 16u) & bmask);
        d.gA = uniform64(d.gA);
        d.gB = uniform64(d.gB);
      } else {
        d.gA = uniform64(base + t);
        d.gB = uniform64(base + t + 16);
      }
      return d;
    };
    uint32_t ka[K::kLaneBytes / 4], kb[K::kLaneBytes / 4];
    uint32_t vd[4 * kPasses];
    uint32_t nw[kNW], sw[kSW], zw[kSW];
    auto load_key = [&](int64_t ra, int64_t rb) {
      load_loose<K::kLaneBytes / 4>(kbytes + ra * K::kRowBytes + kg * K::kLaneBytes, ka);
      load_loose<K::kLaneBytes / 4>(kbytes + rb * K::kRowBytes + kg * K::kLaneBytes, kb);
    };
    auto load_keys = [&](const Desc& d) { load_key(d.gA + n, d.gB + n); };
    auto load_value = [&](int i, int64_t r) {
      const uint8_t* src = vbytes + r * kVRowBytes + 4 * pq;
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) vd[4 * ps + i] = *(const uint32_t*)(src + 32 * ps);
    };
    auto load_values = [&](const Desc& d) {
      const int64_t r = tq < 4 ? d.gA + 4 * tq : d.gB + 4 * (tq - 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) load_value(i, r + i);
    };
    auto load_norms = [&](const Desc& d) {
      if constexpr (!K::kVq) load_loose<kNW>(norms + (first ? d.gA : d.gB) + 4 * kg, nw);
    };
    auto load_side = [&](const Desc& d) {
      const int64_t r = (first ? d.gA : d.gB) + 4 * kg;
      load_loose<kSW>(vsc + r * 4, sw);
      load_loose<kSW>(vzr + r * 4, zw);
    };
    // a tile past whose last token lanes read that token's row again
    auto load_tail = [&](const Desc& d) {
      auto rowof = [&](int i) -> int64_t {
        const int c = min(i, d.last);
        return c < 16 ? d.gA + c : d.gB + (c - 16);
      };
      load_key(rowof(n), rowof(16 + n));
#pragma unroll
      for (int i = 0; i < 4; ++i) load_value(i, rowof(4 * tq + i));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t r = rowof(tok0 + i);
        if constexpr (!K::kVq) packed_set<TN>(nw, i, norms[r]);
#pragma unroll
        for (int gg = 0; gg < 4; ++gg) {
          packed_set<TV>(sw, 4 * i + gg, vsc[r * 4 + gg]);
          packed_set<TV>(zw, 4 * i + gg, vzr[r * 4 + gg]);
        }
      }
    };

    // ---- state of this lane's query row (m replicated over its 8 lanes,
    // the sums this lane's share)
    float m_run = -__builtin_inff(), m_thr = -__builtin_inff();
    float mref = -__builtin_inff(), mexp = 0.0f;   // reference, and as the exponent takes it
    // Products weight * scale as f16 pairs: e_fold is the exponent, relative to
    // m_run, of the row's largest (the weights carry 2^(kPairExp - e_fold)),
    // eg that of each value group's.  `apart`: some row's groups are more than
    // 2^kPairApart apart, and a group's products move by its own power of two.
    int e_fold = 0, eg[4] = {-127, -127, -127, -127};
    bool apart = false;
    float p_thr = 0.0f;                            // log2 products (plus 127) that need a look: any, with `apart`
    auto shift_of = [&](int gg) -> int { return min(max(e_fold - eg[gg], -100), 100); };
    float l_run = 0.0f;
    float zacc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[8];                                  // [value group][code field]
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto centred = [&](uint32_t codes, rf16x2 mul) -> uint32_t {
      return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(rf16x2, codes), mul, mid));
    };
    auto spread = [&](int ps) {
      // dword (byte j, tokens 2i, 2i + 1) = [byte of 2i, 0, byte of 2i + 1, 0]
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t sel = 0x0c000c00u | ((uint32_t)(4 + j) << 16) | (uint32_t)j;
        uint2 pr;
        pr.x = __builtin_amdgcn_perm(vd[4 * ps + 1], vd[4 * ps], sel);
        pr.y = __builtin_amdgcn_perm(vd[4 * ps + 3], vd[4 * ps + 2], sel);
        *(uint2*)(vw + kRowsPitch * j) = pr;
      }
    };
    auto tile = [&](int64_t t, int last, auto&& next_values, auto&& next_keys, auto&& next_norms, auto&& next_side) {
      spread(0);
      if constexpr (kPasses == 1) next_values();
      // -- S^T
      f32x4 ca = {0.0f, 0.0f, 0.0f, 0.0f}, cb = ca;
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        u32x4 av, bv;
        if constexpr (KEY == 8) {
          const int i = s >> 1, o = i * 4096 + (s & 1) * 65536;
          av = *(LdsQuad)(tb + ((ka[0] >> (8 * i)) & 0xffu) * 16 + o);
          bv = *(LdsQuad)(tb + ((kb[0] >> (8 * i)) & 0xffu) * 16 + o);
        } else if constexpr (KEY == 4) {
          av = *(LdsQuad)(tb + ((ka[s >> 2] >> (8 * (s & 3))) & 0xffu) * 16 + s * 4096);
          bv = *(LdsQuad)(tb + ((kb[s >> 2] >> (8 * (s & 3))) & 0xffu) * 16 + s * 4096);
        } else {
          constexpr int kBlk = K::kVq ? 2048 : 0;
          const uint32_t wa = ka[s >> 1] >> (16 * (s & 1)), wb = kb[s >> 1] >> (16 * (s & 1));
          const u32x2 a0 = *(LdsPair)(tb + (wa & 0xffu) * 8 + (2 * s) * kBlk);
          const u32x2 a1 = *(LdsPair)(tb + ((wa >> 8) & 0xffu) * 8 + (2 * s + 1) * kBlk);
          const u32x2 b0 = *(LdsPair)(tb + (wb & 0xffu) * 8 + (2 * s) * kBlk);
          const u32x2 b1 = *(LdsPair)(tb + ((wb >> 8) & 0xffu) * 8 + (2 * s + 1) * kBlk);
          av = u32x4{a0[0], a0[1], a1[0], a1[1]};
          bv = u32x4{b0[0], b0[1], b1[0], b1[1]};
        }
        ca = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(av), as_f16x8(bq[s]), ca, 0, 0, 0);
        cb = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(bv), as_f16x8(bq[s]), cb, 0, 0, 0);
      }
      __builtin_amdgcn_s_setprio(0);
      next_keys();
      // -- scores: column r plus column 8 + r; lanes of the first half keep
      // the first 16 tokens, the others the second 16
      float xs[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float mine = first ? ca[v] : cb[v], other = first ? cb[v] : ca[v];
        xs[v] = mine + dpp_row_ror<0x128>(other);
        if constexpr (!K::kVq) xs[v] *= packed_get<TN>(nw, v);
      }
      next_norms();
      if (last < 31 || t + 31 > qlim_min) {  // uniform: an incomplete tile, or a causal cut
        const int lim = (int)max((int64_t)-1, min((int64_t)last, qlim - t));
#pragma unroll
        for (int v = 0; v < 4; ++v) xs[v] = tok0 + v > lim ? -__builtin_inff() : xs[v];
      }
      // scales, and what a unit weight adds to the fp32 sums
      float sv[16], zz[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        sv[i] = packed_get<TV>(sw, i);
        zz[i] = fmaf(kMid, sv[i], packed_get<TV>(zw, i));
        asm volatile("" : "+v"(zz[i]));  // (here, so that `sv` may be scaled in place)
      }
      const float tmax = fmaxf(fmaxf(xs[0], xs[1]), fmaxf(xs[2], xs[3])) * rfac;
      // whether a score or a product is past what the references hold for
      auto grown = [&](float thr) -> bool {
        float smax = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) smax = fmaxf(smax, fabsf(sv[i]));
        // (a number's bits * 2^-23 - 127 is its log2, less at most 0.09)
        return __any((tmax > m_thr) | (fmaf((float)__builtin_bit_cast(uint32_t, smax), 0x1p-23f, tmax) > thr));
      };
      if (__builtin_expect(grown(p_thr), 0)) {
        bool grow = true;
        if (apart) {
#pragma unroll
          for (int i = 0; i < 16; ++i) sv[i] = __builtin_amdgcn_ldexpf(sv[i], shift_of(i & 3));
          grow = grown(mexp + (127.0f + kPairTop));
        }
        if (grow) {
          const bool was = apart;
          int old[4] = {0, 0, 0, 0};  // the groups' powers of two so far
          if (was) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sv[i] = packed_get<TV>(sw, i);
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) old[gg] = shift_of(gg);
          }
          // the row's largest score, and log2 of each group's largest product
          // (as above) beside it
          const float base = tmax == -__builtin_inff() ? 0.0f : tmax;
          float pg[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float w = fast_exp2(fmaf(xs[v], rfac, -base));
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) pg[gg] = fmaxf(pg[gg], fabsf(w * sv[4 * v + gg]));
          }
          const float mt = rows_max8(tmax), m_new = fmaxf(m_run, mt);
          const int drop = m_new > m_run ? (int)fminf(m_new - m_run, 512.0f) : 0;
#pragma unroll
          for (int gg = 0; gg < 4; ++gg) {
            const float lg = rows_max8(fmaf((float)__builtin_bit_cast(uint32_t, pg[gg]), 0x1p-23f, tmax - 127.0f));
            eg[gg] = max(eg[gg] - drop, (int)floorf(fmaxf(lg - m_new, -127.0f)));
          }
          const int e_max = max(max(eg[0], eg[1]), max(eg[2], eg[3]));
          const int e_min = min(min(eg[0], eg[1]), min(eg[2], eg[3]));
          // (clamped where the weights stay far inside fp32's range)
          e_fold = min(max(e_max, -40), 60);
          apart = __any((e_fold - e_min > kPairApart || e_fold < e_max) && m_new > -__builtin_inff());
          m_run = m_new;
          const float r_new = m_run == -__builtin_inff() ? m_run : m_run + (float)(e_fold - kPairExp);
          const float by = mref == -__builtin_inff() ? mref : mref - r_new;
          const float alpha = fast_exp2(by);
          l_run *= alpha;
#pragma unroll
          for (int gg = 0; gg < 4; ++gg) zacc[gg] *= alpha;
          if (was || apart) {
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) {
              const int to = apart ? shift_of(gg) : 0;
              const float beta = fast_exp2(by + (float)(to - old[gg]));
              acc[2 * gg] *= beta;
              acc[2 * gg + 1] *= beta;
#pragma unroll
              for (int v = 0; v < 4; ++v) sv[4 * v + gg] = __builtin_amdgcn_ldexpf(sv[4 * v + gg], to);
            }
          } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] *= alpha;
          }
          mref = r_new;
          mexp = r_new == -__builtin_inff() ? 0.0f : r_new;
          m_thr = m_run + 10.0f;
          p_thr = apart ? -__builtin_inff() : mexp + (127.0f + kPairTop);
        }
      }
      float pw[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        pw[v] = fast_exp2(fmaf(xs[v], rfac, -mexp));
        l_run += pw[v];
#pragma unroll
        for (int gg = 0; gg < 4; ++gg) zacc[gg] = fmaf(pw[v], zz[4 * v + gg], zacc[gg]);
      }
      // -- O^T, kGroups value groups per pass
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        if (ps > 0) {
          wave_sync();
          spread(ps);
          next_values();
        }
        u32x4 bp[kGroups];
#pragma unroll
        for (int gi = 0; gi < kGroups; ++gi) {
          const int gg = ps * kGroups + gi;
          uint32_t h0, h1, l0, l1;
          rows_split2(pw[0] * sv[gg], pw[1] * sv[4 + gg], one, h0, l0);
          rows_split2(pw[2] * sv[8 + gg], pw[3] * sv[12 + gg], one, h1, l1);
          // K slots 0-3 of lane group kg: tokens 4kg.. of the first half,
          // 4-7: of the second; hi parts in columns 0-7, lo in 8-15
          bp[gi] = u32x4{dpp_bank_move_u<0x128, 0xc>(h0, l0), dpp_bank_move_u<0x128, 0xc>(h1, l1),
                         dpp_bank_move_u<0x128, 0x3>(l0, h0), dpp_bank_move_u<0x128, 0x3>(l1, h1)};
        }
        if (ps == kPasses - 1) next_side();
        wave_sync();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int gi = 0; gi < kGroups; ++gi) {
          const int gg = ps * kGroups + gi;
          const u32x4 wv = *(const u32x4*)(vr + kRowsPitch * (32 / kGroups) * gi);
          u32x4 a0, a1;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a0[i] = centred(wv[i] & mask0, mul0);
            a1[i] = centred(wv[i] & mask1, mul1);
          }
          acc[2 * gg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(a0), as_f16x8(bp[gi]), acc[2 * gg], 0, 0, 0);
          acc[2 * gg + 1] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(a1), as_f16x8(bp[gi]), acc[2 * gg + 1], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
      }
      wave_sync();  // this tile's LDS reads come before the next tile's writes
    };

    // ---- this wave's tiles
    {
      int64_t t = s0 + (int64_t)wu * kRowsTile;
      const int full = __builtin_amdgcn_readfirstlane(
          t + kRowsTile <= s1 ? (int)((s1 - t - kRowsTile) / kStep) + 1 : 0);
      if (full > 0) {
        uint32_t ea, eb;
        entries(t, ea, eb);
        const Desc d0 = rows_at(t, ea, eb);
        load_values(d0);
        load_keys(d0);
        load_norms(d0);
        load_side(d0);
        // table entries one tile ahead of the rows, rows one tile ahead of
        // their use; the last tiles load their own rows again
        entries(full > 1 ? t + kStep : t, ea, eb);
        for (int i = 0; i < full; ++i) {
          const int64_t tn = i + 1 < full ? t + kStep : t;
          const Desc dn = rows_at(tn, ea, eb);
          entries(i + 2 < full ? t + 2 * kStep : tn, ea, eb);
          tile(t, 31, [&] { load_values(dn); }, [&] { load_keys(dn); }, [&] { load_norms(dn); }, [&] { load_side(dn); });
          t = uniform64(t + kStep);
        }
      }
      if (t < s1) {
        uint32_t ea, eb;
        entries(t, ea, eb);
        const Desc d = rows_at(t, ea, eb);
        load_tail(d);
        auto none = [] {};
        tile(t, d.last, none, none, none, none);
      }
    }

    // ---- the waves' results
    l_run += dpp_row_ror<0x128>(l_run);
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) {
      zacc[gg] += dpp_row_ror<0x128>(zacc[gg]);
      zacc[gg] += __shfl_xor(zacc[gg], 16, 64);
      zacc[gg] += __shfl_xor(zacc[gg], 32, 64);
    }
    const uint32_t w_first = owner(x_unit), w_last = owner(x_unit + steps - 1);
    const bool direct = w_first == w_last && rule.n_recent == 0;
    float* const slot = slots + (int64_t)((uint32_t)wg + unit) * kRowsSlot;
    if (lane < kRowsQ) {
      red_m[wu][lane] = mref;
      red_l[wu][lane] = l_run;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {  // dims 64 half .. 64 half + 63
      __syncthreads();  // every wave has left its value tile, or read red_o
#pragma unroll
      for (int gi = 0; gi < 2; ++gi) {
        const int gg = 2 * half + gi;
        const float unit = ldexpf(1024.0f, apart ? -shift_of(gg) : 0);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            // value row m = 4kg + v: dim 2m + f of the group
            const float a = acc[2 * gg + f][v];
            const float o = fmaf(a + dpp_row_ror<0x128>(a), unit, zacc[gg]);
            if (first) red_o[wu][q8][32 * gi + 2 * (4 * kg + v) + f] = o;
          }
        }
      }
      __syncthreads();
      for (int i = tid; i < kRowsQ * 32; i += kThreads) {
        const int r = i >> 5, d = 2 * (i & 31);
        float M = -__builtin_inff();
#pragma unroll
        for (int w = 0; w < NW; ++w)
          M = red_l[w][r] > 0.0f ? fmaxf(M, red_m[w][r]) : M;
        float L = 0.0f;
        f32x2 O = {0.0f, 0.0f};
        bool poisoned = false;  // a NaN score reached some wave's sum
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const float lw = red_l[w][r];
          const f32x2 ow = *(const f32x2*)&red_o[w][r][d];
          poisoned |= lw != lw;
          const bool live = lw > 0.0f;
          const float f = live ? fast_exp2(red_m[w][r] - M) : 0.0f;
          L = live ? fmaf(lw, f, L) : L;
          O[0] = live ? fmaf(ow[0], f, O[0]) : O[0];
          O[1] = live ? fmaf(ow[1], f, O[1]) : O[1];
        }
        if (r < nr) {
          if (direct) {
            const float inv = L > 0.0f ? 1.0f / L : 0.0f;
            store_out2(p, row_off(r) + 64 * half + d, poisoned ? kQuietNaN : O[0] * inv,
                       poisoned ? kQuietNaN : O[1] * inv);
          } else {
            store_agent(&slot[2 * kRowsQ + r * 128 + 64 * half + d], O);
            if (half == 0 && d == 0) {
              store_agent(&slot[r], M);
              store_agent(&slot[kRowsQ + r], poisoned ? kQuietNaN : L);
            }
          }
        }
      }
    }
    __syncthreads();  // red_o and red_l before the next unit's tiles
    if (direct) continue;

    // ---- merge: the last piece of a unit to arrive merges it in piece order
    // (the arrival protocol of attention_mfma.hip; the counters are per
    // (sequence, KV head), so several units of one are merged by a launch of
    // their own)
    if (rule.tiles > 1) continue;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(kWaitVmemOnly);
    asm volatile("" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const int pieces = (int)(w_last - w_first) + 1;
      int* const cnt = p.arrivals + ((int64_t)b * p.n_kv_heads + h);
      const int before = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = before == pieces - 1 ? 1 : 0;
      if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      flag = last;
    }
    __syncthreads();
    const bool merging = flag != 0;
    __syncthreads();  // flag is read before the next unit writes it
    if (!merging) continue;
    rows_merge<kThreads / 256>(p, rule, recent, slots + (int64_t)(w_first + unit) * kRowsSlot, (int)(w_last - w_first) + 1,
                               b, h, 0, tid, (float*)&vsp[0][0]);
    __syncthreads();  // (a later unit writes vsp)
  }
}

template <int KEY, int VB, typename TN, typename TV>
inline void launch_rows_k(const smaq_attn_params& p, const HistAddr& a, const RowsRule& rule, float* slots,
                          const Partials& recent, hipStream_t st) {
  hipLaunchKernelGGL((attn_rows_kernel<KEY, VB, TN, TV>), dim3((unsigned)rule.groups),
                     dim3(RowsKey<KEY>::kWaves * 64), 0, st, p, a, rule, slots, recent);
}

template <int KEY, int VB, typename TN>
inline void launch_rows_v(const smaq_attn_params& p, const HistAddr& a, const RowsRule& rule, float* slots,
                          const Partials& recent, hipStream_t st) {
  switch (p.val_dtype) {
    case SMAQ_F32: launch_rows_k<KEY, VB, TN, float>(p, a, rule, slots, recent, st); break;
    case SMAQ_F16: launch_rows_k<KEY, VB, TN, _Float16>(p, a, rule, slots, recent, st); break;
    default: launch_rows_k<KEY, VB, TN, bf16>(p, a, rule, slots, recent, st); break;
  }
}

}  // namespace smaq
