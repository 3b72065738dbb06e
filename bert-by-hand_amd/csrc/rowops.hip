// Memory-bound row kernels: LayerNorm, embedding gather (+ LayerNorm),
// masked mean pool and L2 normalisation.
//
// For 384-wide rows one wavefront owns a row: lane l holds columns
// 2l + 128j (j = 0, 1, 2) as three 4-byte half2 loads, so each load
// instruction of the wavefront covers 256 contiguous bytes.  The row stays in
// registers; mean and variance are two butterfly reductions over those
// registers (two-pass, as src/kernels/layernorm.cu:32-49, but one global read
// instead of three).

#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace bbh {
namespace {

constexpr int kRowsPerBlock = 4;  // one row per wavefront, 256 threads

// y = LN(x [+ residual]) for D == 384 (src/kernels/layernorm.cu:17-59).
__global__ __launch_bounds__(256) void ln384_kernel(const f16* x, const f16* residual,
                                                    const f16* __restrict__ gamma,
                                                    const f16* __restrict__ beta, f16* y,
                                                    int M, float eps) {
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const size_t off = (size_t)row * kHidden;
  const Affine384 aff = load_affine384(gamma, beta, lane);
  float v[6];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int c = 2 * lane + 128 * j;
    const f16x2 a = *reinterpret_cast<const f16x2*>(x + off + c);
    v[2 * j] = (float)a[0];
    v[2 * j + 1] = (float)a[1];
    if (residual) {
      const f16x2 r = *reinterpret_cast<const f16x2*>(residual + off + c);
      v[2 * j] += (float)r[0];
      v[2 * j + 1] += (float)r[1];
    }
  }
  ln_row384(v, eps);
  store_affine384(y + off, v, aff, lane);
}

// Any D: three strided passes per wavefront-owned row, fp32 statistics.
__global__ __launch_bounds__(256) void ln_generic_kernel(const f16* x, const f16* residual,
                                                         const f16* __restrict__ gamma,
                                                         const f16* __restrict__ beta, f16* y,
                                                         int M, int D, float eps) {
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const size_t off = (size_t)row * D;
  auto val = [&](int i) {
    float v = (float)x[off + i];
    if (residual) v += (float)residual[off + i];
    return v;
  };
  float s = 0.f;
  for (int i = lane; i < D; i += 64) s += val(i);
  const float mean = wave_sum(s) / (float)D;
  float q = 0.f;
  for (int i = lane; i < D; i += 64) {
    const float d = val(i) - mean;
    q += d * d;
  }
  const float rstd = rsqrtf(wave_sum(q) / (float)D + eps);
  for (int i = lane; i < D; i += 64)
    y[off + i] = (f16)((val(i) - mean) * rstd * (float)gamma[i] + (float)beta[i]);
}

__device__ __forceinline__ int clamp_id(int v, int n) { return v < 0 ? 0 : (v >= n ? n - 1 : v); }

// One wavefront's row: LN(word[id] + pos[p] + type[tt]), the sum kept in fp32.
__device__ __forceinline__ void embed_row(int id_raw, int tt_raw, int p, const f16* word,
                                          const f16* pos, const f16* type, const f16* gamma,
                                          const f16* beta, f16* dst, float eps, int lane) {
  const int id = clamp_id(id_raw, kVocab), tt = clamp_id(tt_raw, kTypes);
  const f16* wr = word + (size_t)id * kHidden;
  const f16* pr = pos + (size_t)p * kHidden;
  const f16* tr = type + (size_t)tt * kHidden;
  const Affine384 aff = load_affine384(gamma, beta, lane);
  float v[6];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int c = 2 * lane + 128 * j;
    const f16x2 a = *reinterpret_cast<const f16x2*>(wr + c);
    const f16x2 q = *reinterpret_cast<const f16x2*>(pr + c);
    const f16x2 t = *reinterpret_cast<const f16x2*>(tr + c);
    v[2 * j] = (float)a[0] + (float)q[0] + (float)t[0];
    v[2 * j + 1] = (float)a[1] + (float)q[1] + (float)t[1];
  }
  ln_row384(v, eps);
  store_affine384(dst, v, aff, lane);
}

// out[row] = LN(word[id] + pos[row % seq] + type[tt]) (src/model/forward.cu:28-31;
// gather as src/kernels/embedding.cu:20-30, sum kept in fp32 into the LN).
__global__ __launch_bounds__(256) void embedding_ln_kernel(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ types,
    const f16* __restrict__ word, const f16* __restrict__ pos, const f16* __restrict__ type,
    const f16* __restrict__ gamma, const f16* __restrict__ beta, f16* __restrict__ out, int M,
    int seq, float eps) {
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  embed_row(ids[row], types[row], row % seq, word, pos, type, gamma, beta,
            out + (size_t)row * kHidden, eps, lane);
}

// The packed layout: workgroup s embeds sentence s's len tokens, wavefront w
// positions w, w + kPackedEmbWaves, ... (most sentences: one row per wave).
constexpr int kPackedEmbWaves = 8;
__global__ __launch_bounds__(64 * kPackedEmbWaves) void embedding_ln_packed_kernel(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ types,
    const f16* __restrict__ word, const f16* __restrict__ pos, const f16* __restrict__ type,
    const f16* __restrict__ gamma, const f16* __restrict__ beta, f16* __restrict__ out,
    const PackedSentence* __restrict__ sents, float eps) {
  const PackedSentence sn = sents[blockIdx.x];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int p = wave; p < sn.len; p += kPackedEmbWaves)
    embed_row(ids[sn.tok + p], types[sn.tok + p], p, word, pos, type, gamma, beta,
              out + (size_t)(sn.row + p) * kHidden, eps, lane);
}

// Plain gather-sum, any hidden size (src/kernels/embedding.cu:8-31).
__global__ __launch_bounds__(256) void embedding_kernel(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ types,
    const f16* __restrict__ word, const f16* __restrict__ pos, const f16* __restrict__ type,
    f16* __restrict__ out, int seq, int hidden, size_t total) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const size_t row = idx / hidden;
  const int c = idx % hidden;
  const int id = clamp_id(ids[row], kVocab), tt = clamp_id(types[row], kTypes);
  const int p = row % seq;
  out[idx] = (f16)((float)word[(size_t)id * hidden + c] + (float)pos[(size_t)p * hidden + c] +
                   (float)type[(size_t)tt * hidden + c]);
}

// The same for hidden % 8 == 0, eight columns (16 bytes) a thread; 2-byte
// alignment is all that the operands promise.  total8 = rows * hidden / 8 <
// 2^32.  Bound by the bytes: 14336 rows of 384 took 15.8 us with one column
// and one 64-bit division a thread, against 7.9 us here.
typedef f16x8 f16x8_any __attribute__((aligned(2)));
__global__ __launch_bounds__(256) void embedding8_kernel(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ types,
    const f16* __restrict__ word, const f16* __restrict__ pos, const f16* __restrict__ type,
    f16* __restrict__ out, uint32_t seq, uint32_t hidden8, uint32_t total8) {
  const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
  if (idx >= total8) return;
  const uint32_t row = idx / hidden8, c = (idx - row * hidden8) * 8, p = row % seq;
  const size_t hidden = (size_t)hidden8 * 8;
  const int id = clamp_id(ids[row], kVocab), tt = clamp_id(types[row], kTypes);
  const f16x8 a = *reinterpret_cast<const f16x8_any*>(word + id * hidden + c);
  const f16x8 q = *reinterpret_cast<const f16x8_any*>(pos + p * hidden + c);
  const f16x8 t = *reinterpret_cast<const f16x8_any*>(type + tt * hidden + c);
  f16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (f16)((float)a[e] + (float)q[e] + (float)t[e]);
  *reinterpret_cast<f16x8_any*>(out + (size_t)idx * 8) = o;
}

// One workgroup per sentence: the four wavefronts sum disjoint sets of tokens
// (positions w, w+4, ... in increasing order) of the masked mean, combine
// through LDS, then wave 0 divides by max(count, 1) (src/kernels/pooling.cu:
// 21-31) and scales by 1 / max(||x||, 1e-12) (src/kernels/normalize.cu:7,
// 29-30).  `valid(p)` says whether position p is counted and `row(p)` is its
// hidden row.  Each wavefront first lists its counted positions in LDS (one
// ballot per 64 of them), then sums their rows four at a time, so the row
// loads are issued together instead of one mask-dependent load at a time; the
// sum order is the same as one position after another.  `xform(a)` maps a
// loaded row (the lane's three column pairs) to the values that are summed.
struct RowAsIs {
  __device__ __forceinline__ void operator()(f16x2 (&)[3]) const {}
};
template <class Valid, class RowOf, class Xform = RowAsIs>
__device__ __forceinline__ void pool_normalize_body(int seq, Valid valid, RowOf row,
                                                    f16* __restrict__ dst, Xform xform = {}) {
  __shared__ float part[4][kHidden];
  __shared__ int cnt_part[4];
  __shared__ short plist[4][kMaxPos / 4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int n = 0;
  for (int i0 = 0; i0 < (seq + 3) / 4; i0 += kWave) {
    const int p = wave + 4 * (i0 + lane);
    const bool v = p < seq && valid(p);
    const uint64_t bal = __ballot(v);
    if (v) plist[wave][n + __popcll(bal & ((1ull << lane) - 1))] = (short)p;
    n += __popcll(bal);
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's list is in LDS
  __builtin_amdgcn_wave_barrier();
  float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add_rows = [&](auto cnt_c, int k) {
    constexpr int U = decltype(cnt_c)::value;
    f16x2 a[U][3];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const f16* hr = row(plist[wave][k + u]);
#pragma unroll
      for (int j = 0; j < 3; ++j) a[u][j] = *reinterpret_cast<const f16x2*>(hr + 2 * lane + 128 * j);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      xform(a[u]);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        acc[2 * j] += (float)a[u][j][0];
        acc[2 * j + 1] += (float)a[u][j][1];
      }
    }
  };
  int k = 0;
  for (; k + 4 <= n; k += 4) add_rows(std::integral_constant<int, 4>{}, k);
  for (; k < n; ++k) add_rows(std::integral_constant<int, 1>{}, k);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    part[wave][2 * lane + 128 * j] = acc[2 * j];
    part[wave][2 * lane + 128 * j + 1] = acc[2 * j + 1];
  }
  if (lane == 0) cnt_part[wave] = n;
  __syncthreads();
  if (wave != 0) return;
  const int total = cnt_part[0] + cnt_part[1] + cnt_part[2] + cnt_part[3];
  const float inv_cnt = 1.0f / (float)(total > 0 ? total : 1);
  float v[6], ss = 0.f;
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int c = 2 * lane + 128 * j + e;
      v[2 * j + e] = (part[0][c] + part[1][c] + part[2][c] + part[3][c]) * inv_cnt;
      ss += v[2 * j + e] * v[2 * j + e];
    }
  const float inv = 1.0f / fmaxf(sqrtf(wave_sum(ss)), 1e-12f);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    f16x2 o;
    o[0] = (f16)(v[2 * j] * inv);
    o[1] = (f16)(v[2 * j + 1] * inv);
    *reinterpret_cast<f16x2*>(dst + 2 * lane + 128 * j) = o;
  }
}

__global__ __launch_bounds__(256) void pool_normalize_kernel(const f16* __restrict__ hidden,
                                                             const int32_t* __restrict__ mask,
                                                             f16* __restrict__ out, int seq) {
  const int b = blockIdx.x;
  const f16* hb = hidden + (size_t)b * seq * kHidden;
  const int32_t* mb = mask + (size_t)b * seq;
  pool_normalize_body(
      seq, [&](int p) { return mb[p] != 0; }, [&](int p) { return hb + (size_t)p * kHidden; },
      out + (size_t)b * kHidden);
}

// The last encoder layer's residual LayerNorm and the pool in one pass: the
// rows are read before their LayerNorm (y = FFN2 output + residual), each
// counted row is normalised as ln384 does it, rounded to fp16 the same way,
// and summed; so the embedding equals ln384 followed by pool_normalize, bit
// for bit, with one launch and one read of the rows fewer.  Only the pooled
// rows are normalised, and none is written back.
struct RowLayerNorm {
  Affine384 aff;
  float eps;
  __device__ __forceinline__ void operator()(f16x2 (&a)[3]) const {
    float v[6];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      v[2 * j] = (float)a[j][0];
      v[2 * j + 1] = (float)a[j][1];
    }
    ln_row384(v, eps);
#pragma unroll
    for (int j = 0; j < 3; ++j) a[j] = affine384_pair(v, aff, j);
  }
};

__global__ __launch_bounds__(256) void ln_pool_normalize_kernel(
    const f16* __restrict__ y, const int32_t* __restrict__ mask, const f16* __restrict__ gamma,
    const f16* __restrict__ beta, float eps, f16* __restrict__ out, int seq) {
  const int b = blockIdx.x;
  const f16* yb = y + (size_t)b * seq * kHidden;
  const int32_t* mb = mask + (size_t)b * seq;
  const RowLayerNorm ln{load_affine384(gamma, beta, threadIdx.x & 63), eps};
  pool_normalize_body(
      seq, [&](int p) { return mb[p] != 0; }, [&](int p) { return yb + (size_t)p * kHidden; },
      out + (size_t)b * kHidden, ln);
}

// Packed sentences: position p of sentence s is hidden row sents[s].row + p.
__global__ __launch_bounds__(256) void pool_normalize_packed_kernel(
    const f16* __restrict__ hidden, const PackedSentence* __restrict__ sents,
    f16* __restrict__ out) {
  const PackedSentence sn = sents[blockIdx.x];
  const f16* hb = hidden + (size_t)sn.row * kHidden;
  pool_normalize_body(
      sn.len, [&](int) { return true; }, [&](int p) { return hb + (size_t)p * kHidden; },
      out + (size_t)sn.out_row * kHidden);
}

// out[b, d] = masked mean over seq, any dim (src/kernels/pooling.cu:8-32).
__global__ __launch_bounds__(256) void mean_pool_kernel(const f16* __restrict__ hidden,
                                                        const int32_t* __restrict__ mask,
                                                        f16* __restrict__ out, int batch,
                                                        int seq, int dim) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= batch * dim) return;
  const int b = idx / dim, d = idx % dim;
  float acc = 0.f;
  int cnt = 0;
  for (int s = 0; s < seq; ++s) {
    const int m = mask[(size_t)b * seq + s];
    if (m) {
      ++cnt;
      acc += (float)hidden[((size_t)b * seq + s) * dim + d];
    }
  }
  out[idx] = (f16)(acc / (float)(cnt > 0 ? cnt : 1));
}

// The same for dim % 8 == 0 up to kPoolThreads columns of eight: one workgroup
// per sentence, eight columns a thread, the positions dealt to as many row
// groups as the threads allow and the groups' sums added through LDS.  Masked
// rows are not read.  Bound by the row loads' latency, four of which a thread
// keeps in flight: 128 x 112 rows of 384 took 50.6 us with one thread a column
// walking the mask, against 6.1 us here.
constexpr int kPoolThreads = 1024;
__global__ __launch_bounds__(kPoolThreads) void mean_pool8_kernel(
    const f16* __restrict__ hidden, const int32_t* __restrict__ mask, f16* __restrict__ out,
    int seq, int dim) {
  HIP_DYNAMIC_SHARED(float, part);  // [groups][dim], then [groups] counts
  const int cols = dim / 8, groups = min(kPoolThreads / cols, seq);
  const int g = threadIdx.x / cols, c = (threadIdx.x % cols) * 8;
  int* counts = reinterpret_cast<int*>(part + (size_t)groups * dim);
  const size_t b = blockIdx.x;
  const int32_t* mr = mask + b * seq;
  const f16* hr = hidden + b * seq * dim + c;
  if (g < groups) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int n = 0;
    for (int p0 = g; p0 < seq; p0 += 4 * groups) {
      bool on[4];
      f16x8 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int p = p0 + u * groups;
        on[u] = p < seq && mr[p] != 0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (on[u])
          v[u] = *reinterpret_cast<const f16x8_any*>(hr + (size_t)(p0 + u * groups) * dim);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (on[u]) {
          ++n;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] += (float)v[u][e];
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) part[(size_t)g * dim + c + e] = acc[e];
    if (c == 0) counts[g] = n;
  }
  __syncthreads();
  int cnt = 0;
  for (int k = 0; k < groups; ++k) cnt += counts[k];
  const float n = (float)(cnt > 0 ? cnt : 1);
  for (int d = threadIdx.x; d < dim; d += kPoolThreads) {
    float acc = 0.f;
    for (int k = 0; k < groups; ++k) acc += part[(size_t)k * dim + d];
    out[b * dim + d] = (f16)(acc / n);
  }
}

// Rows of x /= max(||row||, 1e-12), one workgroup per row
// (src/kernels/normalize.cu:10-33).
__global__ __launch_bounds__(256) void l2_normalize_kernel(f16* x, int n) {
  __shared__ float part[4];
  f16* r = x + (size_t)blockIdx.x * n;
  float s = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) {
    const float v = (float)r[i];
    s += v * v;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  const float inv = 1.0f / fmaxf(sqrtf(part[0] + part[1] + part[2] + part[3]), 1e-12f);
  for (int i = threadIdx.x; i < n; i += 256) r[i] = (f16)((float)r[i] * inv);
}

// The same for n % 8 == 0 up to 512: one wavefront per row, held in registers
// (128 rows of 384: 4.6 us with two passes of a workgroup over each row,
// 2.4 us here, about what any launch takes).
__global__ __launch_bounds__(256) void l2_normalize8_kernel(f16* x, int n, int batch) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), c = (threadIdx.x & 63) * 8;
  if (row >= batch) return;
  f16* r = x + (size_t)row * n + c;
  f16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (c < n) v = *reinterpret_cast<const f16x8_any*>(r);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s += (float)v[e] * (float)v[e];
  const float inv = 1.0f / fmaxf(sqrtf(wave_sum(s)), 1e-12f);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (f16)((float)v[e] * inv);
  if (c < n) *reinterpret_cast<f16x8_any*>(r) = v;
}

// Exact GELU in place (src/kernels/gelu.h:5-9, gelu.cu): eight values per
// thread with 16-byte accesses; the tail, or a buffer not 16-byte aligned,
// one value per thread.
__global__ __launch_bounds__(256) void gelu8_kernel(f16* x, size_t n8) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  f16x8 v = reinterpret_cast<f16x8*>(x)[i];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (f16)gelu_erf((float)v[j]);
  reinterpret_cast<f16x8*>(x)[i] = v;
}

__global__ __launch_bounds__(256) void gelu1_kernel(f16* x, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] = (f16)gelu_erf((float)x[i]);
}

}  // namespace

hipError_t layernorm(const f16* x, const f16* residual, const f16* gamma, const f16* beta,
                     f16* y, int M, int D, float eps, hipStream_t s) {
  const dim3 grid((M + kRowsPerBlock - 1) / kRowsPerBlock);
  const bool aligned = (((uintptr_t)x | (uintptr_t)residual | (uintptr_t)gamma |
                         (uintptr_t)beta | (uintptr_t)y) & 3) == 0;
  if (D == kHidden && aligned)
    hipLaunchKernelGGL(ln384_kernel, grid, dim3(256), 0, s, x, residual, gamma, beta, y, M, eps);
  else
    hipLaunchKernelGGL(ln_generic_kernel, grid, dim3(256), 0, s, x, residual, gamma, beta, y, M,
                       D, eps);
  return hipGetLastError();
}

hipError_t embedding(const int32_t* ids, const int32_t* types, const f16* word, const f16* pos,
                     const f16* type, f16* out, int batch, int seq, int hidden,
                     hipStream_t s) {
  const size_t total = (size_t)batch * seq * hidden;
  if (hidden % 8 == 0 && total / 8 < (1ull << 31)) {
    const uint32_t total8 = (uint32_t)(total / 8);
    hipLaunchKernelGGL(embedding8_kernel, dim3((total8 + 255) / 256), dim3(256), 0, s, ids, types,
                       word, pos, type, out, (uint32_t)seq, (uint32_t)hidden / 8, total8);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(embedding_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                     ids, types, word, pos, type, out, seq, hidden, total);
  return hipGetLastError();
}

hipError_t embedding_ln(const int32_t* ids, const int32_t* types, const f16* word,
                        const f16* pos, const f16* type, const f16* gamma, const f16* beta,
                        f16* out, int batch, int seq, float eps, hipStream_t s) {
  const int M = batch * seq;
  hipLaunchKernelGGL(embedding_ln_kernel, dim3((M + kRowsPerBlock - 1) / kRowsPerBlock),
                     dim3(256), 0, s, ids, types, word, pos, type, gamma, beta, out, M, seq,
                     eps);
  return hipGetLastError();
}

// Where a workgroup a sentence pays (sentences x seq x dim, us, one thread a
// column -> here):
//  - from kPoolSeq positions, else there is no walk to share (256 x 4 x 384 2.9 ->
//    3.2, 256 x 16 x 384 5.3 -> 3.8);
//  - with most of its threads at work, or all workgroups resident, two a CU
//    (2000 x 16 x 64 5.4 -> 8.0, 20000 x 16 x 64 32 -> 73; 256 x 16 x 64 4.9 -> 3.1, 2000 x
//    16 x 384 17.3 -> 13.1);
//  - up to 1024 columns, or with a sentence for every CU, else fewer CUs work
//    than with a thread a column (16 x 16 x 4096 4.8 -> 5.3, 1 x 512 x 8192 93 -> 180;
//    256 x 16 x 4096 21 -> 6.7);
//  - below 2^22 sentences: a launch holds less than 2^32 threads (a larger one is
//    not refused, its workgroup count wraps).
constexpr int kPoolSeq = 8;
bool pool8_pays(int batch, int seq, int dim) {
  if (dim % 8 != 0 || dim / 8 > kPoolThreads || batch >= (1ll << 32) / kPoolThreads) return false;
  const int cols = dim / 8, busy = cols * std::min(kPoolThreads / cols, seq);
  return seq >= kPoolSeq && (busy >= kPoolThreads * 3 / 4 || batch <= 512) &&
         (dim <= 1024 || batch >= 256);
}

hipError_t mean_pool(const f16* hidden, const int32_t* mask, f16* out, int batch, int seq,
                     int dim, hipStream_t s) {
  if (pool8_pays(batch, seq, dim)) {
    const int groups = std::min(kPoolThreads / (dim / 8), seq);
    const size_t lds = (size_t)groups * (dim + 1) * sizeof(float);  // at most 36 KB
    hipLaunchKernelGGL(mean_pool8_kernel, dim3(batch), dim3(kPoolThreads), lds, s, hidden, mask,
                       out, seq, dim);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(mean_pool_kernel, dim3((batch * dim + 255) / 256), dim3(256), 0, s, hidden,
                     mask, out, batch, seq, dim);
  return hipGetLastError();
}

hipError_t l2_normalize(f16* x, int n, int batch, hipStream_t s) {
  if (n % 8 == 0 && n <= 512)
    hipLaunchKernelGGL(l2_normalize8_kernel, dim3((batch + 3) / 4), dim3(256), 0, s, x, n, batch);
  else
    hipLaunchKernelGGL(l2_normalize_kernel, dim3(batch), dim3(256), 0, s, x, n);
  return hipGetLastError();
}

hipError_t gelu(f16* x, size_t n, hipStream_t s) {
  const size_t n8 = ((uintptr_t)x & 15) ? 0 : n / 8;
  if (n8)
    hipLaunchKernelGGL(gelu8_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, s, x, n8);
  const size_t rest = n - n8 * 8;
  if (rest)
    hipLaunchKernelGGL(gelu1_kernel, dim3((unsigned)((rest + 255) / 256)), dim3(256), 0, s,
                       x + n8 * 8, rest);
  return hipGetLastError();
}

hipError_t embedding_ln_packed(const int32_t* ids, const int32_t* types, const f16* word,
                               const f16* pos, const f16* type, const f16* gamma,
                               const f16* beta, f16* out, const PackedSentence* sents, int n,
                               float eps, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(embedding_ln_packed_kernel, dim3(n), dim3(64 * kPackedEmbWaves), 0, s, ids,
                     types, word, pos, type, gamma, beta, out, sents, eps);
  return hipGetLastError();
}

hipError_t pool_normalize_packed(const f16* hidden, const PackedSentence* sents, int n, f16* out,
                                 hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(pool_normalize_packed_kernel, dim3(n), dim3(256), 0, s, hidden, sents, out);
  return hipGetLastError();
}

hipError_t pool_normalize(const f16* hidden, const int32_t* mask, f16* out, int batch, int seq,
                          hipStream_t s) {
  hipLaunchKernelGGL(pool_normalize_kernel, dim3(batch), dim3(256), 0, s, hidden, mask, out,
                     seq);
  return hipGetLastError();
}

hipError_t ln_pool_normalize(const f16* y, const int32_t* mask, const f16* gamma,
                             const f16* beta, float eps, f16* out, int batch, int seq,
                             hipStream_t s) {
  hipLaunchKernelGGL(ln_pool_normalize_kernel, dim3(batch), dim3(256), 0, s, y, mask, gamma, beta,
                     eps, out, seq);
  return hipGetLastError();
}

}  // namespace bbh
