// Scores of the standalone cache in one call (head_dim 128, 3- or 4-bit scalar
// keys): the query rotated, then [compressed, exact] scores written side by
// side, read from the history columns and the exact window in place.
//
// The composition it replaces (rotation table transposed, codes and norms
// copied out of the columns, scores, exact keys transposed, a library product,
// its scaling, a concatenation: 10 launches) left the step host-bound: scores of
// 2 x 8 heads x 8192 fp32 tokens 109 -> 21 us a call, the score kernel 32.3 -> 6.8
// us (it read a code byte at a time).  Any number of query rows gains (512 rows:
// 14237 -> 418 us, 710 with a window of 4096).  Scores are a lane per token: 64 code bytes in four 16-byte loads, each code through
// a 16-entry LDS table, one fmaf chain over the dims per query row in
// scores_scalar_kernel's order (the same bits).  Latency bounds it at the
// sizes of a step.
#include "smaq_common.h"

namespace smaq {
namespace {

constexpr int kCsD = 128;
constexpr int kCsRows = 4;  // query rows per pass over a token

// out[r][j] = sum_d x[r][d] M[j][d]: rotate128_block's sums (eight 16-term
// chains, ((p0 + p1) + (p2 + p3)) + ((p4 + p5) + (p6 + p7))) with M read by
// rows, so the caller needs no transposed copy.  Eight lanes hold an output's
// chains.
__global__ __launch_bounds__(256) void cache_rotate_kernel(const void* __restrict__ x, int xdtype, int64_t rows,
                                                           const float* __restrict__ M, float* __restrict__ out) {
  __shared__ float xs[kCsRows][kCsD];
  const int t = threadIdx.x, c = t & 7;
  const int64_t r0 = (int64_t)blockIdx.x * kCsRows;
  for (int e = t; e < kCsRows * kCsD; e += 256) {
    const int64_t i = r0 * kCsD + e;
    float v = 0.0f;
    if (r0 + e / kCsD < rows) {
      switch (xdtype) {
        case SMAQ_F32: v = ((const float*)x)[i]; break;
        case SMAQ_F16: v = Num<_Float16>::to_f(((const _Float16*)x)[i]); break;
        default: v = Num<bf16>::to_f(((const bf16*)x)[i]); break;
      }
    }
    xs[e / kCsD][e % kCsD] = v;
  }
  float4 m[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int d = 0; d < 4; ++d) m[i][d] = *(const float4*)(M + (32 * i + (t >> 3)) * kCsD + 16 * c + 4 * d);
  __syncthreads();
  for (int r = 0; r < kCsRows && r0 + r < rows; ++r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float a = 0.0f;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float4 xv = *(const float4*)&xs[r][16 * c + 4 * d];
        a = fmaf(xv.x, m[i][d].x, a);
        a = fmaf(xv.y, m[i][d].y, a);
        a = fmaf(xv.z, m[i][d].z, a);
        a = fmaf(xv.w, m[i][d].w, a);
      }
      a += __shfl_xor(a, 1, 64);
      a += __shfl_xor(a, 2, 64);
      a += __shfl_xor(a, 4, 64);
      if (c == 0) out[(r0 + r) * kCsD + 32 * i + (t >> 3)] = a;
    }
  }
}

// Blocks [0, hist_blocks) of x: 256 compressed tokens each; the others: 256
// exact ones.  T: the query's, exact keys' and scores' dtype.
template <typename TN, typename T>
__global__ __launch_bounds__(256) void cache_scores_kernel(
    const float* __restrict__ qrot, const T* __restrict__ q, int64_t nq, int64_t N, const uint8_t* __restrict__ codes,
    int64_t codes_bstride, int bits, const TN* __restrict__ norms, int64_t norm_bstride,
    const float* __restrict__ centroids, int hist_blocks, int64_t R, const T* __restrict__ xk, int64_t xk_bstride,
    float scale, T* __restrict__ out) {
  __shared__ float lut[16];
  __shared__ __attribute__((aligned(16))) float qs[kCsRows][kCsD];
  const int tid = threadIdx.x, b = blockIdx.z;
  const int64_t r0 = (int64_t)blockIdx.y * kCsRows;
  const int nr = (int)min((int64_t)kCsRows, nq - r0);
  const bool hist = (int)blockIdx.x < hist_blocks;
  const int64_t t = (int64_t)((int)blockIdx.x - (hist ? 0 : hist_blocks)) * 256 + tid;
  if (tid < (1 << bits)) lut[tid] = centroids[tid];
  for (int e = tid; e < nr * kCsD; e += 256) {
    const int64_t i = ((int64_t)b * nq + r0) * kCsD + e;
    qs[e / kCsD][e % kCsD] = hist ? qrot[i] : Num<T>::to_f(q[i]);
  }
  __syncthreads();
  T* const o = out + ((int64_t)b * nq + r0) * (N + R) + (hist ? 0 : N) + t;
  if (hist) {
    if (t >= N) return;
    const uint4* const row = (const uint4*)(codes + (int64_t)b * codes_bstride + t * 64);
    uint4 w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = row[i];
    const float norm = Num<TN>::to_f(norms[(int64_t)b * norm_bstride + t]);
    const uint32_t mask = (1u << bits) - 1u;
    float acc[kCsRows] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t word = i % 4 == 0 ? w[i / 4].x : i % 4 == 1 ? w[i / 4].y : i % 4 == 2 ? w[i / 4].z : w[i / 4].w;
      float k[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        k[2 * j] = lut[(word >> (8 * j)) & mask];
        k[2 * j + 1] = lut[(word >> (8 * j + bits)) & mask];
      }
#pragma unroll
      for (int r = 0; r < kCsRows; ++r) {
        if (r < nr) {
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[r] = fmaf(qs[r][8 * i + j], k[j], acc[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < kCsRows; ++r)
      if (r < nr) o[r * (N + R)] = Num<T>::from_f((acc[r] * norm) * scale);
  } else {
    if (t >= R) return;
    const T* const row = xk + (int64_t)b * xk_bstride + t * kCsD;
    float acc[kCsRows][8] = {};
#pragma unroll 2
    for (int i = 0; i < 16; ++i) {
      float k[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) k[j] = Num<T>::to_f(row[8 * i + j]);
#pragma unroll
      for (int r = 0; r < kCsRows; ++r)
        if (r < nr) {
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[r][j] = fmaf(qs[r][8 * i + j], k[j], acc[r][j]);
        }
    }
#pragma unroll
    for (int r = 0; r < kCsRows; ++r) {
      if (r < nr) {
        const float* a = acc[r];
        const float s = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
        // the product in the query's dtype, then the scale (as a library
        // product and a multiplication round them)
        o[r * (N + R)] = Num<T>::from_f(Num<T>::round(s) * scale);
      }
    }
  }
}

template <typename TN, typename T>
void launch_scores(const void* q, int64_t batch, int64_t nq, const float* qrot, int64_t N, const void* codes,
                   int64_t codes_bstride, int bits, const void* norms, int64_t norm_bstride, const float* centroids,
                   int64_t R, const void* xk, int64_t xk_bstride, float scale, void* out, hipStream_t st) {
  const int hist_blocks = (int)((N + 255) / 256);
  const dim3 grid((unsigned)(hist_blocks + (R + 255) / 256), (unsigned)((nq + kCsRows - 1) / kCsRows), (unsigned)batch);
  hipLaunchKernelGGL((cache_scores_kernel<TN, T>), grid, dim3(256), 0, st, qrot, (const T*)q, nq, N,
                     (const uint8_t*)codes, codes_bstride, bits, (const TN*)norms, norm_bstride, centroids, hist_blocks,
                     R, (const T*)xk, xk_bstride, scale, (T*)out);
}

}  // namespace
}  // namespace smaq

using namespace smaq;

extern "C" int smaq_cache_scores(const void* q, int qdtype, long long batch, long long nq, int D, const float* M,
                                 float* qrot, long long N, const void* codes, long long codes_bstride, int bits,
                                 const void* norms, long long norm_bstride, int ndtype, const float* centroids,
                                 long long R, const void* xk, long long xk_bstride, float scale, void* out,
                                 void* stream) {
  SMAQ_REQUIRE(q && M && qrot && codes && norms && centroids && out && (R == 0 || xk), "smaq_cache_scores: null pointer");
  SMAQ_REQUIRE(D == kCsD && (bits == 3 || bits == 4), "smaq_cache_scores: head_dim %d, %d-bit keys unsupported", D, bits);
  SMAQ_REQUIRE(batch > 0 && nq > 0 && N > 0 && R >= 0 && batch < 65536 && (nq + kCsRows - 1) / kCsRows < 65536 &&
                   N + R < (1ll << 38),
               "smaq_cache_scores: bad shape");
  SMAQ_REQUIRE((((uintptr_t)M | (uintptr_t)codes | (uintptr_t)codes_bstride) & 15) == 0,
               "smaq_cache_scores: the metric and the code rows must be 16-byte aligned");
  auto known = [](int t) { return t == SMAQ_F32 || t == SMAQ_F16 || t == SMAQ_BF16; };
  if (!known(qdtype) || !known(ndtype)) {
    set_error("smaq_cache_scores: unsupported %s dtype %d", known(qdtype) ? "norm" : "query",
              known(qdtype) ? ndtype : qdtype);
    return SMAQ_EUNSUPPORTED;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t rows = (int64_t)batch * nq;
  hipLaunchKernelGGL(cache_rotate_kernel, dim3((unsigned)((rows + kCsRows - 1) / kCsRows)), dim3(256), 0, st, q, qdtype,
                     rows, M, qrot);
  int rc = launch_status("smaq_cache_scores(rotation)");
  if (rc != SMAQ_OK) return rc;
#define SMAQ_CS(TN, T)                                                                                       \
  launch_scores<TN, T>(q, batch, nq, qrot, N, codes, codes_bstride, bits, norms, norm_bstride, centroids, R, xk, \
                       xk_bstride, scale, out, st)
#define SMAQ_CS_N(T)                                                                                   \
  switch (ndtype) {                                                                                    \
    case SMAQ_F32: SMAQ_CS(float, T); break;                                                           \
    case SMAQ_F16: SMAQ_CS(_Float16, T); break;                                                        \
    default: SMAQ_CS(bf16, T); break;                                                                  \
  }
  switch (qdtype) {
    case SMAQ_F32: SMAQ_CS_N(float) break;
    case SMAQ_F16: SMAQ_CS_N(_Float16) break;
    default: SMAQ_CS_N(bf16) break;
  }
#undef SMAQ_CS_N
#undef SMAQ_CS
  return launch_status("smaq_cache_scores");
}
