// Block-VQ key encoder for 2-dim blocks (65 to 256 centroids, a multiple of 4
// blocks): the argmin over a few candidates instead of every centroid.
//
// Same indices and tie counts as encode_blockvq_kernel (blockvq_codec.hip),
// whose arithmetic it repeats for every candidate.  Of a 2-dim codebook only a
// handful of centroids can be the nearest to any point of a small rectangle,
// so the plane of a block is cut into 4096 cells and each cell gets the list
// of those that can:
//   build   one workgroup per (block, quarter of its cells), a cell per
//           thread.  A coordinate is mapped by t = (x - mean) / scale,
//           u = t / (1 + |t|), cells are equal in u: fine where the centroids
//           lie, and covering the whole line (scale is 1.5 times the
//           centroids' deviation; the outermost cells, from 22 deviations on
//           with 32 cells an axis, hold no list).  The wider axis gets the more
//           cells (8 to 512), so that cells are about square.  Centroid j is
//           listed when its smallest squared distance to the cell does not
//           exceed the smallest of the centroids' largest ones by more than a
//           margin of 1e-5 (|x|^2 + max |C|^2): every computed distance is
//           within 1e-6 of that sum of its true value, so a centroid left out
//           neither wins nor ties.  The test runs over 2 x 2 cells first.
//   encode  one persistent workgroup of 16 waves per CU with the lists and
//           centroids of 4 blocks in LDS (148 KB), a lane per row: cell, list
//           (4 candidates per LDS read), exact distances.  A lane without a
//           list (outermost cell, a list over 30, a non-finite key or
//           codebook) or with a runner-up within 2e-6 relative has all
//           centroids scanned by its wave.
// The lists live in the caller's workspace and are built by every call.
//
// Bound by VALU issue (220 per 64 rows and block) and the lists' random LDS
// reads.  At 261,632 fp16 rows of 64 blocks (a wave's longest list is 7 to 13
// of 256): build 32 us + encode 110 us against 10,920 us for the full scan
// (whole append with the value pack 10,914 -> 159 us).  Lists over 1,024
// cells left 16 candidates and took 674 us; scanning all centroids lane by lane
// where a list is missing, not by the wave, made one block with too few pool
// words hold its workgroups for 1 ms.
#include "encode_internal.h"

namespace smaq {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kE2Bits = 12;             // log2 of a block's cells
constexpr int kE2N = 1 << kE2Bits;
constexpr int kE2MinBits = 3;           // an axis has at least 8 cells
constexpr int kE2Words = 1536;          // 4-candidate words per quarter
constexpr int kE2Coarse = 64;           // candidates of a 2 x 2 group
constexpr int kE2Full = 31;             // list length that means: scan all
constexpr int kE2Group = 4;             // blocks per encode workgroup
constexpr int kE2Threads = 1024;

// One block's tables, in the workspace and (4 of them) in LDS.
struct E2Block {
  float4 cent[256];                  // c0, c1, |c|^2
  uint16_t cell[kE2N];               // word offset << 5 | candidates (kE2Full: scan all)
  uint32_t pool[4][kE2Words];        // candidate indices, ascending, by quarter (quarter_of)
  float cx, cy, isx, isy;            // the map's centre and 1 / scale
  float E[4];
  int ex, pad[3];                    // log2 of the cells along x
};
static_assert(sizeof(E2Block) % 16 == 0, "copied in 16-byte units");
static_assert(sizeof(E2Block) * kE2Group <= 160 * 1024, "LDS");

// The 2 x 2 group of cell (ix, iy); its low two bits name the quarter.
__device__ __forceinline__ int group_of(int ix, int iy, int ex) { return ((iy >> 1) << (ex - 1)) + (ix >> 1); }

// An axis of the map with 2^bits cells: cells [i, j) (neither outermost) as an
// interval, a little wider than the error with which a key finds its cell.
struct E2Axis {
  float c, scale;
  int bits;
  __device__ __forceinline__ void interval(int i, int j, float* lo, float* hi) const {
    const float w = ldexpf(2.0f, -bits);
    const float u0 = (float)i * w - 1.0f, u1 = (float)j * w - 1.0f;
    const float t0 = u0 / (1.0f - fabsf(u0)), t1 = u1 / (1.0f - fabsf(u1));
    const float t = fmaxf(fabsf(t0), fabsf(t1));
    // (u is found within 5e-7, t within (1 + |t|)^2 of that)
    const float e = 1e-5f * (fmaf(t, t, 1.0f) * scale + fabsf(c));
    *lo = fmaf(t0, scale, c) - e;
    *hi = fmaf(t1, scale, c) + e;
  }
};

struct E2Rect {
  float xl, xh, yl, yh;
  __device__ __forceinline__ float far2(float2 q) const {
    const float mx = fmaxf(q.x - xl, xh - q.x), my = fmaxf(q.y - yl, yh - q.y);
    return fmaf(mx, mx, my * my);
  }
  __device__ __forceinline__ float near2(float2 q) const {
    const float ax = fmaxf(fmaxf(xl - q.x, q.x - xh), 0.0f), ay = fmaxf(fmaxf(yl - q.y, q.y - yh), 0.0f);
    return fmaf(ax, ax, ay * ay);
  }
  // the largest near2 of a listed centroid
  __device__ __forceinline__ float cut(float far, float cm) const {
    const float mx = fmaxf(fabsf(xl), fabsf(xh)), my = fmaxf(fabsf(yl), fabsf(yh));
    return far * (1.0f + 1e-5f) + 1e-5f * (fmaf(mx, mx, my * my) + cm);
  }
};

__global__ __launch_bounds__(kE2Threads) void encode2d_build_kernel(const float* __restrict__ E_blocks,
                                                                    const float* __restrict__ C, int nc,
                                                                    E2Block* __restrict__ out) {
  __shared__ float2 cs[260];  // (every 64 centroids two banks further)
  __shared__ float red[4][4];
  __shared__ int scan[16];
  __shared__ __attribute__((aligned(4))) uint8_t coarse[256][kE2Coarse];
  __shared__ int count[256];
  auto at_id = [](int id) -> int { return id + (id >> 6); };
  const int b = blockIdx.x >> 2, quarter = blockIdx.x & 3, tid = threadIdx.x;
  E2Block& o = out[b];
  // ---- centroids, their mean and deviation (the same in all four quarters)
  float2 c = {0.0f, 0.0f};
  if (tid < 256) {
    if (tid < nc) c = *(const float2*)(C + ((int64_t)b * nc + tid) * 2);
    cs[at_id(tid)] = c;
  }
  const bool mine = tid < nc;
  float sx = mine ? c.x : 0.0f, sy = mine ? c.y : 0.0f;
  if (tid < 256) {
    sx = warp_sum(sx);
    sy = warp_sum(sy);
    if ((tid & 63) == 0) { red[tid >> 6][0] = sx; red[tid >> 6][1] = sy; }
  }
  __syncthreads();
  const float inv = 1.0f / (float)nc;
  const float cx = (red[0][0] + red[1][0] + red[2][0] + red[3][0]) * inv;
  const float cy = (red[0][1] + red[1][1] + red[2][1] + red[3][1]) * inv;
  __syncthreads();
  float vx = mine ? (c.x - cx) * (c.x - cx) : 0.0f, vy = mine ? (c.y - cy) * (c.y - cy) : 0.0f;
  float cm = mine ? fmaf(c.x, c.x, c.y * c.y) : 0.0f;
  if (tid < 256) {
    vx = warp_sum(vx);
    vy = warp_sum(vy);
    cm = warp_max(cm);
    if ((tid & 63) == 0) { red[tid >> 6][0] = vx; red[tid >> 6][1] = vy; red[tid >> 6][2] = cm; }
  }
  __syncthreads();
  vx = (red[0][0] + red[1][0] + red[2][0] + red[3][0]) * inv;
  vy = (red[0][1] + red[1][1] + red[2][1] + red[3][1]) * inv;
  cm = fmaxf(fmaxf(red[0][2], red[1][2]), fmaxf(red[2][2], red[3][2]));
  // (a spread of zero on one axis: cells as fine as the other's, or unit ones)
  const float dx = 1.5f * sqrtf(vx), dy = 1.5f * sqrtf(vy);
  const float least = fmaxf(fmaxf(dx, dy) * 1e-3f, 1e-18f);
  const float sxs = fmaxf(dx, least), sys = fmaxf(dy, least);
  // a non-finite centroid makes the sums so; huge ones leave fp32's range
  const bool sane = vx < 1e30f && vy < 1e30f && cm < 1e30f && fabsf(cx) < 1e18f && fabsf(cy) < 1e18f;

  // cells along x: about square cells, 2^kE2Bits in all
  int ex = 0;
  if (sane) {
    int e = 0;
    frexpf(sxs / sys * 1.41421356f, &e);  // e - 1 = round(log2(sxs / sys))
    ex = min(max((kE2Bits + e - 1) >> 1, kE2MinBits), kE2Bits - kE2MinBits);
  } else {
    ex = kE2Bits / 2;
  }
  const E2Axis ax{cx, sxs, ex}, ay{cy, sys, kE2Bits - ex};
  const int nx = 1 << ex, ny = 1 << (kE2Bits - ex);

  // ---- the 256 groups of this quarter, 4 threads each: centroids that can be
  // nearest to a point of the group's inner cells
  const int gi = (tid >> 2) * 4 + quarter;         // group
  const int gx = 2 * (gi & (nx / 2 - 1)), gy = 2 * (gi >> (ex - 1));
  uint8_t* const group = coarse[tid >> 2];
  int spare;                                       // a centroid outside the group's list
  {
    const int sub = tid & 3;
    E2Rect R;
    ax.interval(max(gx, 1), min(gx + 2, nx - 1), &R.xl, &R.xh);
    ay.interval(max(gy, 1), min(gy + 2, ny - 1), &R.yl, &R.yh);
    const float2* const part = &cs[65 * sub];  // ids 64 sub .. 64 sub + 63
    const int live = min(max(nc - 64 * sub, 0), 64);
    float far = __builtin_inff();
#pragma unroll 8
    for (int i = 0; i < 64; ++i) far = i < live ? fminf(far, R.far2(part[i])) : far;
    far = fminf(far, __shfl_xor(far, 1, 64));
    far = fminf(far, __shfl_xor(far, 2, 64));
    const float cut = R.cut(far, cm);
    uint32_t in[2] = {0u, 0u};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll 8
      for (int i = 0; i < 32; ++i) in[q] |= (32 * q + i < live && R.near2(part[32 * q + i]) <= cut ? 1u : 0u) << i;
    }
    // the group's list in LDS: a thread's ids come after the lower threads'
    const int own = __popc(in[0]) + __popc(in[1]);
    int inc = own;
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) {
      const int up = __shfl_up(inc, o, 64);
      if (sub >= o) inc += up;
    }
    const int all = __shfl(inc, (tid & 60) | 3, 64);
    int at = inc - own;
    if (all <= kE2Coarse) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        for (uint32_t bits = in[q]; bits; bits &= bits - 1)
          group[at++] = (uint8_t)(64 * sub + 32 * q + __builtin_ctz(bits));
    }
    // (at most kE2Coarse of more centroids are listed: one is not)
    const uint32_t out0 = ~in[0], out1 = ~in[1];
    spare = out0 && __builtin_ctz(out0) < live ? 64 * sub + __builtin_ctz(out0)
            : out1 && 32 + __builtin_ctz(out1) < live ? 64 * sub + 32 + __builtin_ctz(out1) : 256;
    spare = min(spare, __shfl_xor(spare, 1, 64));
    spare = min(spare, __shfl_xor(spare, 2, 64));
    // (a group out in the tails: its cells hold no list)
    if (sub == 0) count[tid >> 2] = all <= kE2Coarse ? all : 0;
  }
  __syncthreads();

  // ---- a cell per thread: its group's centroids again
  const int ix = gx + (tid & 1), iy = gy + ((tid >> 1) & 1);
  const int m = count[tid >> 2];
  const bool inner = sane && ix > 0 && ix < nx - 1 && iy > 0 && iy < ny - 1 && m > 0;
  uint32_t in[kE2Coarse / 32] = {};  // bit i: candidate i of the group's list
  int n = 0;
  bool near = false;                 // within 6 deviations of the mean
  if (inner) {
    E2Rect R;
    ax.interval(ix, ix + 1, &R.xl, &R.xh);
    ay.interval(iy, iy + 1, &R.yl, &R.yh);
    near = fmaxf(fabsf(R.xl + R.xh - 2.0f * cx) / sxs, fabsf(R.yl + R.yh - 2.0f * cy) / sys) < 8.0f;
    const uint32_t* const ids = (const uint32_t*)group;
    float far = __builtin_inff();
    for (int i = 0; i < m; i += 4) {
      const uint32_t w = ids[i / 4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float f = R.far2(cs[at_id((w >> (8 * j)) & 0xffu)]);
        far = i + j < m ? fminf(far, f) : far;
      }
    }
    const float cut = R.cut(far, cm);
#pragma unroll
    for (int q = 0; q < kE2Coarse / 32; ++q) {
      for (int i = 0; i < 32 && 32 * q + i < m; i += 4) {
        const uint32_t w = ids[8 * q + i / 4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          in[q] |= (32 * q + i + j < m && R.near2(cs[at_id((w >> (8 * j)) & 0xffu)]) <= cut ? 1u : 0u) << (i + j);
      }
      n += __popc(in[q]);
    }
  }
  const bool list = inner && n > 0 && n < kE2Full;
  const int words = list ? (n + 3) / 4 : 0;
  // offsets, the cells near the mean first (where the pool is too small, far
  // cells go without): an inclusive scan of both counts over the wave, then
  // over the 16 waves
  int inc = near ? words : words << 16;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(inc, o, 64);
    if ((tid & 63) >= o) inc += up;
  }
  if ((tid & 63) == 63) scan[tid >> 6] = inc;
  __syncthreads();
  int total = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < (tid >> 6)) inc += scan[w];
    total += scan[w];
  }
  const int off = near ? (inc & 0xffff) - words : (total & 0xffff) + (inc >> 16) - words;
  const bool fits = list && off + words <= kE2Words;
  o.cell[(iy << ex) + ix] = (uint16_t)(fits ? (off << 5 | n) : kE2Full);
  if (fits) {
    uint8_t* dst = (uint8_t*)&o.pool[quarter][off];
#pragma unroll
    for (int q = 0; q < kE2Coarse / 32; ++q)
      for (uint32_t bits = in[q]; bits; bits &= bits - 1) *dst++ = group[32 * q + __builtin_ctz(bits)];
    // the last word is filled up with a centroid that is not listed (its
    // distance is a true one and can neither win nor tie), so that evaluating
    // a candidate needs no mask
    for (int i = n; i < 4 * words; ++i) *dst++ = (uint8_t)spare;
  }
  if (quarter == 0) {
    if (tid < 256) {
      // |c|^2 in the reference's order (multiply, then add)
      const float s = c.x * c.x;
      o.cent[tid] = float4{c.x, c.y, s + c.y * c.y, 0.0f};
    }
    if (tid == 0) {
      o.cx = cx;
      o.cy = cy;
      o.isx = 1.0f / sxs;
      o.isy = 1.0f / sys;
      o.ex = ex;
    }
    if (tid < 4) o.E[tid] = E_blocks[(int64_t)b * 4 + tid];
  }
}

// The reference's choice for one row over all centroids by the whole wave
// (up to 4 per lane): the first index of the smallest sqrt(d2), a NaN winning
// at its first index; `tie` when another centroid is within 2e-6 relative of
// the smallest d2.
__device__ __forceinline__ int scan_all(const float4* cent, int nc, int lane, float y0, float y1, float xsq, bool* tie) {
  uint64_t key = ~0ull;
  float dmin = __builtin_inff(), d2[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = lane + 64 * j;
    const float4 c = cent[i];
    float a = fmaf(y1, c.y, y0 * c.x);
    a = a + xsq;
    a = a + c.z;
    a = a < 0.0f ? 0.0f : a;  // clamp_min(0); NaN passes
    a = i < nc ? a : __builtin_inff();
    d2[j] = a;
    const bool nan = a != a;
    const uint64_t s = nan ? 0ull : (uint64_t)__float_as_uint(sqrtf(a)) + 1ull;
    const uint64_t kk = i < nc ? (s << 32) | (uint64_t)i : ~0ull;
    key = kk < key ? kk : key;
    dmin = nan ? dmin : fminf(dmin, a);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t other = ((uint64_t)(uint32_t)__shfl_xor((int)(key >> 32), o, 64) << 32) |
                           (uint32_t)__shfl_xor((int)(uint32_t)key, o, 64);
    key = other < key ? other : key;
    dmin = fminf(dmin, __shfl_xor(dmin, o, 64));
  }
  int close = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    close += __popcll(__ballot(lane + 64 * j < nc && d2[j] <= dmin * (1.0f + 2e-6f)));
  // (with every distance infinite the reference's runner-up is its start value)
  *tie = (key >> 32) != 0 && (close >= 2 || !(dmin < __builtin_inff()));
  return (int)(uint32_t)key;
}

// One row's key values of a workgroup's blocks, kept as loaded.
template <typename T>
struct KeyPart {
  static constexpr int kWords = 2 * kE2Group * (int)sizeof(T) / 4;
  uint32_t w[kWords];
  __device__ __forceinline__ void load(const T* p) {
#pragma unroll
    for (int i = 0; i < kWords; i += 4) {
      const u32x4 v = *(const u32x4*)((const uint32_t*)p + i);
      w[i] = v[0]; w[i + 1] = v[1]; w[i + 2] = v[2]; w[i + 3] = v[3];
    }
  }
  __device__ __forceinline__ float get(int i) const {
    if constexpr (sizeof(T) == 2)
      return Num<T>::to_f(__builtin_bit_cast(T, (uint16_t)(w[i >> 1] >> (16 * (i & 1)))));
    else
      return __builtin_bit_cast(float, w[i]);
  }
};

// Workgroup w of an XCD (blockIdx.x % 8) takes block group w % groups: all
// groups of the same rows run on one XCD, whose L2 then holds the rows' lines
// for every group (a group reads 16 or 32 bytes of a row's 128-byte lines).
template <typename T>
__global__ __launch_bounds__(kE2Threads) void encode2d_kernel(const T* __restrict__ k, RowMap map, uint32_t rows,
                                                              int nb, int nc, int chunks,
                                                              const E2Block* __restrict__ tables,
                                                              uint8_t* __restrict__ idx_out,
                                                              unsigned long long* tie_count) {
  __shared__ E2Block L[kE2Group];
  const int tid = threadIdx.x, lane = tid & 63;
  const int groups = nb / kE2Group;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int group = slot % groups, chunk = xcd + 8 * (slot / groups);
  if (chunk >= chunks) return;
  {
    const u32x4* src = (const u32x4*)(tables + (int64_t)group * kE2Group);
    for (int i = tid; i < (int)(sizeof(L) / 16); i += kE2Threads) ((u32x4*)L)[i] = src[i];
  }
  __syncthreads();
  unsigned ties = 0;
  const uint32_t sets = (rows + 63) / 64;
  const uint32_t s1 = (uint32_t)((uint64_t)sets * (chunk + 1) / chunks);
  const uint32_t n_inner = (uint32_t)map.n_inner;
  auto row_at = [&](uint32_t s) -> const T* {
    const uint32_t r = min(s * 64 + lane, rows - 1), o = r / n_inner, i = r - o * n_inner;
    return k + (int64_t)o * map.s_outer + (int64_t)i * map.s_inner + group * (2 * kE2Group);
  };
  uint32_t s = (uint32_t)((uint64_t)sets * chunk / chunks) + (tid >> 6);
  KeyPart<T> next;
  if (s < s1) next.load(row_at(s));
  for (; s < s1; s += kE2Threads / 64) {
    const KeyPart<T> kr = next;
    if (s + kE2Threads / 64 < s1) next.load(row_at(s + kE2Threads / 64));
    const uint32_t r = s * 64 + lane;
    const bool valid = r < rows;
    uint32_t ob = 0u;
#pragma unroll
    for (int b = 0; b < kE2Group; ++b) {
      const E2Block& B = L[b];
      const float k0 = kr.get(2 * b), k1 = kr.get(2 * b + 1);
      const float a0 = fmaf(k1, B.E[1], k0 * B.E[0]), a1 = fmaf(k1, B.E[3], k0 * B.E[2]);
      const float xsq = a0 * a0 + a1 * a1;
      const float y0 = -2.0f * a0, y1 = -2.0f * a1;  // exact
      const float tx = (a0 - B.cx) * B.isx, ty = (a1 - B.cy) * B.isy;
      const float ux = tx * __builtin_amdgcn_rcpf(1.0f + fabsf(tx)), uy = ty * __builtin_amdgcn_rcpf(1.0f + fabsf(ty));
      // (a NaN converts to 0, an outermost cell)
      const int ex = __builtin_amdgcn_readfirstlane(B.ex);
      const int nx = 1 << ex, ny = 1 << (kE2Bits - ex);
      const float hx = (float)(nx / 2), hy = (float)(ny / 2);
      const int ix = min(max((int)fmaf(ux, hx, hx), 0), nx - 1);
      const int iy = min(max((int)fmaf(uy, hy, hy), 0), ny - 1);
      const uint32_t e = B.cell[(iy << ex) + ix];
      const int n = (int)(e & 31u), words = n == kE2Full ? 0 : (n + 3) >> 2;
      const uint32_t* const pool = &B.pool[group_of(ix, iy, ex) & 3][e >> 5];
      float best = __builtin_inff(), second = best;
      uint32_t bi = 0;
      for (int g = 0; g < words; ++g) {
        const uint32_t w = pool[g];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t id = (w >> (8 * j)) & 0xffu;
          const float4 c = B.cent[id];
          float a = fmaf(y1, c.y, y0 * c.x);
          a = a + xsq;
          a = a + c.z;
          bi = a < best ? id : bi;
          second = __builtin_amdgcn_fmed3f(a, best, second);  // (best <= second)
          best = fminf(best, a);
        }
      }
      // (`best` is infinite without a list, the comparison then false; a
      // negative distance counts as zero and ties with its like)
      const bool clear = second > best * (1.0f + 2e-6f) && best < 3.0e38f && best >= 0.0f;
      for (uint64_t todo = __ballot(!clear && valid); todo; todo &= todo - 1) {
        const int t = __builtin_ctzll(todo);
        bool tie;
        const int ci = scan_all(B.cent, nc, lane, __shfl(y0, t, 64), __shfl(y1, t, 64), __shfl(xsq, t, 64), &tie);
        if (lane == t) {
          bi = (uint32_t)ci;
          ties += tie ? 1u : 0u;
        }
      }
      ob |= bi << (8 * b);
    }
    if (valid) {
      const uint32_t o = r / n_inner;
      const int64_t out_row = (int64_t)r + (int64_t)o * (map.out_outer - map.n_inner);
      uint8_t* const dst = idx_out + out_row * nb + group * kE2Group;
      *(uint32_t*)dst = ob;
    }
  }
  add_count(tie_count, ties);
}

}  // namespace

bool encode_2d_supported(int nb, int bd, int nc, int64_t rows, const void* k, int kdtype, long long s_outer,
                         long long s_inner, long long n_inner, const void* C, const void* idx, const void* ws) {
  const int esz = kdtype == SMAQ_F32 ? 4 : 2;
  return bd == 2 && nb % kE2Group == 0 && nb > 0 && nc > kE2Coarse && nc <= 256 && rows < (1ll << 31) - 64 &&
         n_inner < (1ll << 31) &&
         // 16-byte loads of 4 blocks of a row, 8-byte centroid loads, 4-byte
         // index stores, 16-byte table copies
         (((uintptr_t)k | (uintptr_t)(s_outer * esz) | (uintptr_t)(s_inner * esz) | (uintptr_t)ws) & 15) == 0 &&
         ((uintptr_t)C & 7) == 0 && ((uintptr_t)idx & 3) == 0;
}

int64_t encode_2d_bytes(int nb) { return (int64_t)nb * (int64_t)sizeof(E2Block); }

int launch_encode_2d(int kdtype, const void* k, RowMap map, int64_t rows, int nb, int nc, const float* E_blocks,
                     const float* C, uint8_t* idx, unsigned long long* ties, void* ws, hipStream_t st) {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  E2Block* const tables = (E2Block*)ws;
  hipLaunchKernelGGL(encode2d_build_kernel, dim3((unsigned)nb * 4u), dim3(kE2Threads), 0, st, E_blocks, C, nc, tables);
  // one round of workgroups, and at least 64 rows for each of a workgroup's
  // 16 waves
  const int groups = nb / kE2Group;
  int64_t chunks = cus / groups < 1 ? 1 : cus / groups;
  const int64_t most = (rows + kE2Threads - 1) / kE2Threads;
  if (chunks > most) chunks = most;
  const unsigned grid = (unsigned)(8 * groups * ((chunks + 7) / 8));
  switch (kdtype) {
    case SMAQ_F32:
      hipLaunchKernelGGL(encode2d_kernel<float>, dim3(grid), dim3(kE2Threads), 0, st, (const float*)k, map,
                         (uint32_t)rows, nb, nc, (int)chunks, tables, idx, ties);
      break;
    case SMAQ_F16:
      hipLaunchKernelGGL(encode2d_kernel<_Float16>, dim3(grid), dim3(kE2Threads), 0, st, (const _Float16*)k, map,
                         (uint32_t)rows, nb, nc, (int)chunks, tables, idx, ties);
      break;
    default:
      hipLaunchKernelGGL(encode2d_kernel<bf16>, dim3(grid), dim3(kE2Threads), 0, st, (const bf16*)k, map,
                         (uint32_t)rows, nb, nc, (int)chunks, tables, idx, ties);
      break;
  }
  return launch_status("smaq_encode_blockvq(2d)");
}

}  // namespace smaq
