// Masked multi-head self-attention for head_dim 32, read straight out of the
// fused QKV activations (row stride 3*heads*32, Q | K | V column blocks,
// src/model/weights.h:38-54; strided reads as src/kernels/attention.cu:25-28,
// 74-75) and written straight into the merged (B*S, heads*32) layout
// (attention.cu:87-92).
//
// The reference materialises scores (B*12, S, S) in HBM, runs a separate
// masked softmax over them and a third kernel for P.V
// (src/model/encoder.cu:39-45).  Here one workgroup owns one (sequence, head):
// it stages that head's K (row-major) and V (transposed, [dim][key]) in LDS
// once, then each wavefront walks 32-query tiles with an online softmax, so
// scores never leave the chip (at S = 512 the reference layout is 1.6 GB per
// layer).
//
// Per 32-query x 32-key chunk a wavefront issues four
// v_mfma_f32_32x32x16_f16: two for S^T = K . Q^T (head dims 0-15, 16-31) and
// two for O^T = V^T . P^T (keys 0-15, 16-31).  The 32 K rows of a chunk are
// loaded in the permuted order key_of_row(r) so that the sixteen S^T values a
// lane receives (query lane%32; keys 16*(i/8) + 8*(lane/32) + i%8) are exactly
// the two 8-key groups that lane must supply as operand B of the two P.V
// MFMAs: probabilities go from accumulator to MFMA operand without leaving
// the lane, and V^T is read with one 16-byte LDS load per MFMA.
//
// Softmax in fp32, base 2: the 1/sqrt(32) scale (src/model/encoder.cu:28) and
// log2(e) fold into one FMA before v_exp_f32; the row max needs one
// permlane32 swap (lane ^ 32).  The running max is updated lazily: the
// accumulator is rescaled only when some row's max rises by more than 2^8 in
// probability, so most chunks skip the 16 multiplies and the extra exp.  Row
// sums add the fp16 probabilities (the values the P.V MFMA consumes) with
// v_dot2_f32_f16.  Mask semantics follow src/kernels/softmax.cu:35-62: keys
// with mask 0 are dropped and a query whose keys are all masked gets a zero
// context.  A bitmap of unmasked keys per 32-key chunk, one ballot per 64
// keys, lets fully masked chunks be skipped (their contribution is exactly
// zero) and fully unmasked chunks run without mask arithmetic.
//
// Short sequences are bound by the global round trip: all of a workgroup's
// loads (Q, K, V, mask) are issued before its single barrier, and the output
// goes out through LDS as 16-byte stores of 64 contiguous bytes per row.
// Long sequences are bound by exp + MFMA issue; at 8 and 16 tiles a wavefront takes
// two query tiles at once, sharing each K and V^T operand read between them.

#include <algorithm>

#include "kernels.h"

namespace bbh {
namespace {

// Key (within a 32-key chunk) loaded as row r of the S^T tile.
__device__ __forceinline__ int key_of_row(int r) {
  const int a = r >> 3, c = (r >> 2) & 1, b = r & 3;
  return 16 * (a >> 1) + 8 * c + 4 * (a & 1) + b;
}

// Halves offset of 16-byte chunk c (8 head dims) of key row `key` in the K
// tile; the XOR keeps the 16 rows of one operand fetch on distinct banks.
__device__ __forceinline__ int ks_off(int key, int c) {
  return key * 32 + ((c ^ ((key >> 2) & 3)) << 3);
}

// Stride (halves) of a wavefront's 32 x 32 output staging tile in LDS.
constexpr int kStageLd = 40;

size_t attn_lds_bytes(int seq, int staged_waves) {
  const int seqp = (seq + 31) & ~31;
  return (size_t)seqp * 32 * 2 + (size_t)32 * (seqp + 8) * 2 + (size_t)seqp * 4 +
         (size_t)((seqp / 32 + 3) & ~3) * 4 + (size_t)staged_waves * 32 * kStageLd * 2;
}

// Largest step (log2 units) the running row max may lag the true one: while
// every row's chunk max stays within it of the stored max, probabilities are
// taken against the stored max (each at most 2^kLazy, exact in fp16 and fp32)
// and the accumulator is not rescaled.
constexpr float kLazy = 8.f;

// A wavefront works on T query tiles at once (T = 1 or 2): the tiles share
// every K and V^T operand read from LDS, and their two dependency chains
// (scores -> max -> exp -> P.V) interleave.  The workgroup's NW wavefronts
// take tile groups round robin.
// F: 1 stage the output through LDS, 2 put that staging in the K/V area
// (one tile group per wavefront).
// VL: packed sentences (sents[b] gives the rows and length; every token is
// valid, `mask` and `seq` are unused).
template <int NW, int T, int F, bool VL = false>
__global__ __launch_bounds__(64 * NW, T == 2 || NW > 8 ? 4 : 6) void attention_kernel(
    const f16* __restrict__ qkv, const int32_t* __restrict__ mask, f16* __restrict__ out,
    int batch, int seq, int heads, float c, const PackedSentence* __restrict__ sents,
    int last_first) {
  HIP_DYNAMIC_SHARED(f16, smem);
  // (sequence, head) of this workgroup; the heads of a sequence go to one XCD
  // back to back (but where its span ends), so its QKV rows are fetched into
  // one L2.  last_first: the last sequence first (launch_attention).
  int b, h;
  if (!xcd_item(batch, heads, b, h)) return;
  if (last_first) b = batch - 1 - b;
  size_t row0 = (size_t)b * seq;  // first hidden row of the sentence
  if constexpr (VL) {
    const PackedSentence sn = sents[b];
    seq = sn.len;
    row0 = (size_t)sn.row;
    if (seq == 0) return;  // no tokens: nothing to attend, no rows to write
  }
  const int seqp = (seq + 31) & ~31, nch = seqp >> 5, VLD = seqp + 8;
  f16* Ks = smem;                                              // [seqp][32]
  f16* Vt = Ks + seqp * 32;                                    // [32][VLD]
  float* mb = reinterpret_cast<float*>(Vt + 32 * VLD);         // [seqp]: 0 or -inf
  uint32_t* cm = reinterpret_cast<uint32_t*>(mb + seqp);       // [nch]: unmasked-key bitmaps
  f16* stage = reinterpret_cast<f16*>(cm + ((nch + 3) & ~3));  // [NW*T][32][kStageLd]
  const int hid = heads * kHeadDim, ld = 3 * hid;
  const f16* base = qkv + row0 * ld + h * kHeadDim;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r32 = lane & 31, kh = lane >> 5;
  constexpr int NT = 64 * NW;

  // Q of this wavefront's first tile group, issued before the K/V staging so
  // the two global round trips overlap.  Tile t of group g is
  // wave + NW*(T*g + t); a tile past the sequence (T = 2, odd tile count)
  // reads clamped rows and stores nothing.
  f16x8 q0[T], q1[T];
  auto load_q = [&](int g) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int q = (wave + NW * (T * g + t)) * 32 + r32;
      const f16* qrow = base + (size_t)min(q, seq - 1) * ld;
      q0[t] = *reinterpret_cast<const f16x8*>(qrow + 8 * kh);
      q1[t] = *reinterpret_cast<const f16x8*>(qrow + 16 + 8 * kh);
    }
  };
  load_q(0);

  for (int i = tid; i < seqp * 4; i += NT) {  // K: 16 bytes per (key, 8 dims)
    const int key = i >> 2, ch = i & 3;
    f16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (key < seq) v = *reinterpret_cast<const f16x8*>(base + (size_t)key * ld + hid + ch * 8);
    *reinterpret_cast<f16x8*>(Ks + ks_off(key, ch)) = v;
  }
  for (int i = tid; i < (seqp / 4) * 8; i += NT) {  // V^T: a 4-key x 4-dim block per thread
    const int dq = i & 7, kq = i >> 3;
    f16x4 r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int key = 4 * kq + e;
      r[e] = key < seq ? *reinterpret_cast<const f16x4*>(base + (size_t)key * ld + 2 * hid + 4 * dq)
                       : f16x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f16x4 col = {r[0][e], r[1][e], r[2][e], r[3][e]};
      *reinterpret_cast<f16x4*>(Vt + (4 * dq + e) * VLD + 4 * kq) = col;
    }
  }
  if (wave == NW - 1) {  // key bias and bitmaps of unmasked keys, 64 keys per ballot
    const int32_t* mrow = VL ? nullptr : mask + (size_t)b * seq;
    int mv[kMaxPos / 64];
#pragma unroll
    for (int j = 0; j < kMaxPos / 64; ++j) {
      const int key = 64 * j + lane;
      mv[j] = (64 * j < seq && key < seq) ? (VL ? 1 : mrow[key]) : 0;
    }
#pragma unroll
    for (int j = 0; j < kMaxPos / 64; ++j) {
      if (2 * j >= nch) break;
      if (64 * j + lane < seqp) mb[64 * j + lane] = mv[j] != 0 ? 0.f : -INFINITY;
      const unsigned long long on = __ballot(mv[j] != 0);
      if (lane == 0) cm[2 * j] = (uint32_t)on;
      if (lane == 1 && 2 * j + 1 < nch) cm[2 * j + 1] = (uint32_t)(on >> 32);
    }
  }
  __syncthreads();

  const int krow = key_of_row(r32);
  const uint32_t cml = lane < nch ? cm[lane] : 0u;  // lane j holds chunk j's bitmap
  const float lag = kLazy / c;                      // kLazy in raw-score units
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const f16x2 ones = {(f16)1.f, (f16)1.f};
  for (int g = 0; wave + NW * T * g < nch; ++g) {
    if (g > 0) load_q(g);
    f32x16 o[T];
    float m[T], l[T];  // running max (raw scores) and sum of the fp16 probabilities
#pragma unroll
    for (int t = 0; t < T; ++t) {
      o[t] = zero;
      m[t] = 0.f;
      l[t] = 0.f;
    }
    bool started = false;
    for (int kc = 0; kc < nch; ++kc) {
      const uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)cml, kc);
      if (bits == 0) continue;  // every key of the chunk masked: contributes nothing
      const int key = kc * 32 + krow;
      const f16x8 k0 = *reinterpret_cast<const f16x8*>(Ks + ks_off(key, kh));
      const f16x8 k1 = *reinterpret_cast<const f16x8*>(Ks + ks_off(key, 2 + kh));
      f32x16 s[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        s[t] = mfma32(k0, q0[t], zero);
        s[t] = mfma32(k1, q1[t], s[t]);  // s[i]: key kc*32 + 16*(i/8) + 8*kh + i%8 (raw)
      }
      if (bits != 0xffffffffu) {
        const float* mk = mb + kc * 32 + 8 * kh;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float bias = mk[16 * (i >> 3) + (i & 7)];
#pragma unroll
          for (int t = 0; t < T; ++t) s[t][i] += bias;
        }
      }
      float mx[T];
      bool up = false;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        // IEEE maximum (v_maximum3_f32): scores hold no NaN, and unlike fmaxf
        // it needs no canonicalising v_max_f32 of each MFMA result first.
        float v = __builtin_elementwise_maximum(__builtin_elementwise_maximum(s[t][0], s[t][1]),
                                                s[t][2]);
#pragma unroll
        for (int i = 3; i < 15; i += 2)
          v = __builtin_elementwise_maximum(__builtin_elementwise_maximum(v, s[t][i]), s[t][i + 1]);
        v = __builtin_elementwise_maximum(v, s[t][15]);
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v),
                                                         false, false);
        mx[t] = __builtin_elementwise_maximum(__uint_as_float(sw[0]),
                                              __uint_as_float(sw[1]));  // finite: a key is unmasked
        up = up || mx[t] > m[t] + lag;
      }
      if (!started) {
#pragma unroll
        for (int t = 0; t < T; ++t) m[t] = mx[t];
        started = true;
      } else if (__ballot(up)) {  // the tiles of a group together
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const float mn = fmaxf(m[t], mx[t]);
          const float corr = __builtin_amdgcn_exp2f((m[t] - mn) * c);
          l[t] *= corr;
          o[t] *= corr;
          m[t] = mn;
        }
      }
      const f16* vrow = Vt + r32 * VLD + kc * 32 + 8 * kh;
      const f16x8 va = *reinterpret_cast<const f16x8*>(vrow);
      const f16x8 vb = *reinterpret_cast<const f16x8*>(vrow + 16);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float mc = m[t] * c;
        f16x8 pa, pb;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          pa[i] = (f16)__builtin_amdgcn_exp2f(fmaf(s[t][i], c, -mc));
          pb[i] = (f16)__builtin_amdgcn_exp2f(fmaf(s[t][8 + i], c, -mc));
        }
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          l[t] = __builtin_amdgcn_fdot2(f16x2{pa[i], pa[i + 1]}, ones, l[t], false);
          l[t] = __builtin_amdgcn_fdot2(f16x2{pb[i], pb[i + 1]}, ones, l[t], false);
        }
        o[t] = mfma32(va, pa, o[t]);
        o[t] = mfma32(vb, pb, o[t]);
      }
    }
    float inv[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const float lt = xor32_sum(l[t]);
      inv[t] = lt > 0.f ? 1.0f / lt : 0.f;
    }
    if constexpr (!(F & 1)) {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int q = (wave + NW * (T * g + t)) * 32 + r32;
        if (q < seq) {  // o[i] = O[q][8*(i/4) + 4*kh + i%4]
          f16* dst = out + (row0 + q) * hid + h * kHeadDim + 4 * kh;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            f16x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = (f16)(o[t][4 * j + e] * inv[t]);
            *reinterpret_cast<f16x4*>(dst + 8 * j) = w;
          }
        }
      }
    } else {
      // Through this wavefront's LDS tiles, so that each store instruction
      // writes 16 query rows x 64 contiguous bytes.
      f16* st = stage + wave * T * 32 * kStageLd;
      if ((F & 2) && nch <= NW * T) {  // one group per wavefront: reuse the K/V area once all are done
        if (NW > 1) __syncthreads();
        st = smem + wave * T * 32 * kStageLd;
      }
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f16x4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = (f16)(o[t][4 * j + e] * inv[t]);
          *reinterpret_cast<f16x4*>(st + (t * 32 + r32) * kStageLd + 8 * j + 4 * kh) = w;
        }
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int row = 16 * p + (lane >> 2), cc = lane & 3;
          const int q = (wave + NW * (T * g + t)) * 32 + row;
          const f16x8 w = *reinterpret_cast<const f16x8*>(st + (t * 32 + row) * kStageLd + 8 * cc);
          if (q < seq)
            *reinterpret_cast<f16x8*>(out + (row0 + q) * hid + h * kHeadDim + 8 * cc) = w;
        }
    }
  }
  // A sentence may have fewer query tiles than the workgroup has wavefronts;
  // those wavefronts still take part in the staging barrier.
  if constexpr (F & 2) {
    if (NW > 1 && nch <= NW * T && wave >= nch) __syncthreads();
  }
}

template <int NW, int T, int F, bool VL = false>
hipError_t launch_attention(const f16* qkv, const int32_t* mask, f16* merged, int batch,
                            int heads, int seq, float c, hipStream_t s,
                            const PackedSentence* sents, int rows) {
  const int tiles = (seq + 31) / 32;  // for VL: of the longest sentence
  const int staged = !(F & 1) || ((F & 2) && tiles <= NW * T) ? 0 : NW * T;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(attention_kernel<NW, T, F, VL>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)attn_lds_bytes(kMaxPos, NW * T));
  if (attr != hipSuccess) return attr;
  // Last sequence first where the QKV rows exceed the memory-side cache: the QKV
  // Linear wrote them in ascending order, so the last ones are still there, and
  // an ascending walk would evict each row before it is read (bert_embed 1024 x
  // 128 4.10 -> 4.00 ms, 512 x 256 4.22 -> 4.13, 256 x 512 4.55 -> 4.51, 224 x 512, 264
  // MB, 4.14 -> 4.09; level at 192 x 512, 226 MB, padded and packed).
  const bool last_first = (size_t)rows * 3 * heads * kHeadDim * sizeof(f16) > kMemCache;
  const int grid = xcd_grid(batch, heads);
  hipLaunchKernelGGL((attention_kernel<NW, T, F, VL>), dim3(grid), dim3(64 * NW),
                     attn_lds_bytes(seq, staged), s, qkv, mask, merged, batch, seq, heads, c,
                     sents, (int)last_first);
  return hipGetLastError();
}

// Workgroup shape by query-tile count (tiles = ceil(seq / 32); for packed
// sentences of the longest one).
//  - 2-4 tiles: 4 wavefronts of one tile each, output staged through the K/V
//    area.  More wavefronts than tiles still help to stage K and V, but at two
//    tiles only while all workgroups run at once (six a CU: 1536): 64 x 48 / 128 x
//    64 4.8 / 6.6 us on 2 wavefronts, 4.7 / 6.4 on 4; 130 x 48 / 171 x 64 6.5 / 8.3
//    against 7.2 / 8.9.  At three tiles 4 in every batch (309 x 80 23.0 -> 18.8).
//    Packed sentences of up to 3 tiles: 2 wavefronts, for most sentences are much
//    shorter than the longest.
//  - 8 and 16 tiles: 4 and 8 wavefronts of two tiles, output staged.  The two
//    tiles of a wavefront are rescaled together, which shows in the last bits,
//    so these counts take this shape in every batch (one tile a wavefront: 512 x
//    256 129 us against 122 here, 128 x 512 96 against 94, but 64 x 256 20.7
//    against 21.2).
//  - Else 5-7 tiles: 8 wavefronts, 9-15: 12, one tile at a time and stored
//    straight from the accumulators: more wavefronts than tiles help here, too,
//    and more of them hide the exp and MFMA latencies than 4 or 8 (64 x 144 / 192
//    11.2 / 13.7 -> 9.0 / 12.5 us, 21 x 304 12.5 -> 11.3, 80 x 288 / 480 28.0 / 54.9 ->
//    27.1 / 52.3).  But 9-11 tiles on 8 wavefronts where a CU's share of workgroups
//    fills it anyway (160 x 288 47.2 -> 44.9), and 9-10 where that saves a round,
//    three workgroups a CU against two (43 x 288 / 320 20.8 / 23.7 -> 19.2 / 22.6, 106 x
//    288 37.1 -> 35.4; 65 x 288, two rounds of either, 27.2 on 12, 27.6 on 8).
template <bool VL>
hipError_t attention_any(const f16* qkv, const int32_t* mask, f16* merged, int batch, int heads,
                         int seq, float scale, hipStream_t s, const PackedSentence* sents,
                         int rows) {
  const float c = scale * 1.4426950408889634f;  // scores * c are base-2 exponents
  const int tiles = (seq + 31) / 32;
#define BBH_ATT(NW, T, F) \
  launch_attention<NW, T, F, VL>(qkv, mask, merged, batch, heads, seq, c, s, sents, rows)
  const int wgs = batch * heads;
  if (tiles >= 16) return BBH_ATT(8, 2, 3);
  if (tiles == 8) return BBH_ATT(4, 2, 3);
  auto rounds = [&](int per_cu) { return (wgs + 256 * per_cu - 1) / (256 * per_cu); };
  const bool eight = wgs > 1280 ? tiles <= 11 : tiles <= 10 && rounds(3) < rounds(2);
  if (tiles > 8 && !eight) return BBH_ATT(12, 1, 0);
  if (tiles > 4) return BBH_ATT(8, 1, 0);
  // A launch holds less than 2^32 threads (a larger one is not refused, its
  // workgroup count wraps): 2^24 workgroups and more on 2 wavefronts, too.
  const bool fits4 = (long)xcd_grid(batch, heads) * 256 < 1l << 32;
  if (tiles >= (VL ? 4 : wgs > 1536 ? 3 : 2) && fits4) return BBH_ATT(4, 1, 3);
  if (tiles >= 2) return BBH_ATT(2, 1, 3);
  return BBH_ATT(1, 1, 3);
#undef BBH_ATT
}

}  // namespace

hipError_t attention(const f16* qkv, const int32_t* mask, f16* merged, int batch, int heads,
                     int seq, float scale, hipStream_t s) {
  return attention_any<false>(qkv, mask, merged, batch, heads, seq, scale, s, nullptr,
                              batch * seq);
}

hipError_t attention_packed(const f16* qkv, const PackedSentence* sents, int n, f16* merged,
                            int heads, int max_len, int rows, float scale, hipStream_t s) {
  if (n == 0 || max_len == 0) return hipSuccess;
  return attention_any<true>(qkv, nullptr, merged, n, heads, max_len, scale, s, sents, rows);
}

namespace {

// ---- unfused pieces with the reference's launcher shapes -------------------
// The operands may sit at any element address (only scores' qkv is checked
// for 16 bytes), so these kernels move 16 and 8 bytes at a time through types
// that promise 2-byte alignment: gfx950 takes such global accesses at any
// address, in one instruction.
typedef f16x8 f16x8_any __attribute__((aligned(2)));
typedef f16x4 f16x4_any __attribute__((aligned(2)));
typedef int32_t i32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// scores[z, i, j] = scale * sum_d Q[b, i, d] K[b, j, d], z = b*heads + h
// (src/kernels/attention.cu:17-60), fp32 accumulate, fp16 store.  seq % 16 == 0.
//
// Bound by writing the scores.  A wavefront makes 32 queries x 64 keys (two
// 32x32 MFMA tiles, two k-steps each, operands straight from global memory)
// and stores them through its own LDS tile as 128-byte row runs; a workgroup
// of four covers 128 queries, so its K rows are fetched once into the L1.
// One value per thread (two 64-byte row reads for each 2-byte store) took
// 58.9 us at batch 32 x seq 128, against 9.3 us here (12.6 MB out).
constexpr int kScoreKeys = 64, kScoreLd = kScoreKeys + 8;
__global__ __launch_bounds__(256) void scores_kernel(const f16* __restrict__ qkv,
                                                     f16* __restrict__ scores, int heads,
                                                     int seq, int ld, int q_off, int k_off_,
                                                     float scale) {
  __shared__ __align__(16) f16 stage[4][32 * kScoreLd];
  const int kblocks = (seq + kScoreKeys - 1) / kScoreKeys;
  const int z = blockIdx.y, b = z / heads, h = z % heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r32 = lane & 31, kh = lane >> 5;
  const int q0 = ((int)(blockIdx.x / kblocks) * 4 + wave) * 32;
  const int k0 = (int)(blockIdx.x % kblocks) * kScoreKeys;
  if (q0 >= seq) return;  // no barrier follows: each wavefront keeps to its own LDS tile
  const f16* base = qkv + (size_t)b * seq * ld + h * kHeadDim + 8 * kh;
  // Rows past the sequence read its last row; what they give is not stored.
  const f16* qr = base + (size_t)min(q0 + r32, seq - 1) * ld + q_off;
  const f16x8 qa = *reinterpret_cast<const f16x8_any*>(qr);
  const f16x8 qb = *reinterpret_cast<const f16x8_any*>(qr + 16);
  f16x8 ka[2], kb[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const f16* kr = base + (size_t)min(k0 + 32 * t + r32, seq - 1) * ld + k_off_;
    ka[t] = *reinterpret_cast<const f16x8_any*>(kr);
    kb[t] = *reinterpret_cast<const f16x8_any*>(kr + 16);
  }
  f16* st = stage[wave];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    f32x16 s = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    s = mfma32(ka[t], qa, s);
    s = mfma32(kb[t], qb, s);  // s[i]: query r32, key k0 + 32t + 8*(i/4) + 4*kh + i%4
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f16x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = (f16)(s[4 * j + e] * scale);
      *reinterpret_cast<f16x4*>(st + r32 * kScoreLd + 32 * t + 8 * j + 4 * kh) = w;
    }
  }
  f16* dst = scores + ((size_t)z * seq + q0) * seq + k0;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int row = 8 * p + (lane >> 3), c = (lane & 7) * 8;
    const f16x8 w = *reinterpret_cast<const f16x8*>(st + row * kScoreLd + c);
    if (q0 + row < seq && k0 + c < seq)
      *reinterpret_cast<f16x8_any*>(dst + (size_t)row * seq + c) = w;
  }
}

// Row softmax in place, one wavefront per row (src/kernels/softmax.cu:26-63):
// any N.
__global__ __launch_bounds__(256) void softmax_kernel(f16* x, int M, int N,
                                                      const int32_t* __restrict__ mask,
                                                      int mask_stride) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  f16* r = x + (size_t)row * N;
  const int32_t* mr = mask ? mask + (mask_stride > 0 ? (size_t)(row / mask_stride) * N : 0)
                           : nullptr;
  float m = -INFINITY;
  for (int i = lane; i < N; i += 64)
    if (!mr || mr[i] != 0) m = fmaxf(m, (float)r[i]);
  m = wave_max(m);
  float s = 0.f;
  for (int i = lane; i < N; i += 64)
    if (!mr || mr[i] != 0) s += __expf((float)r[i] - m);
  s = wave_sum(s);
  const float inv = s > 0.f ? 1.0f / s : 0.f;
  for (int i = lane; i < N; i += 64)
    r[i] = (mr && mr[i] == 0) ? (f16)0.f : (f16)(__expf((float)r[i] - m) * inv);
}

// The same for N % 8 == 0 up to 512: LPR lanes hold a row, eight values each
// (the smallest power of two that covers it), so a wavefront takes 64 / LPR
// rows and reads and writes each value once, 16 bytes a lane.  Bound by the
// bytes: 49152 rows of 128 took 23.9 us in three 2-byte passes a row, against
// 8.5 us here.
template <int LPR, class F>
__device__ __forceinline__ float lanes_reduce(float v, F f) {
  if constexpr (LPR > 32) v = xor_op<32>(v, f);
  if constexpr (LPR > 16) v = xor_op<16>(v, f);
  if constexpr (LPR > 8) v = xor_op<8>(v, f);
  if constexpr (LPR > 4) v = xor_op<4>(v, f);
  if constexpr (LPR > 2) v = xor_op<2>(v, f);
  if constexpr (LPR > 1) v = xor_op<1>(v, f);
  return v;
}
template <int LPR>
__global__ __launch_bounds__(256) void softmax8_kernel(f16* x, int M, int N,
                                                       const int32_t* __restrict__ mask,
                                                       int mask_stride) {
  const int lane = threadIdx.x & 63, c = (lane % LPR) * 8;
  const int row = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / LPR) + lane / LPR;
  const bool in = row < M && c < N;  // the other lanes still take part in the reductions
  f16* r = x + (size_t)row * N + c;
  f16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
  uint32_t on = 0;  // bit e: value e counts
  if (in) {
    v = *reinterpret_cast<const f16x8_any*>(r);
    on = 0xff;
    if (mask) {
      const int32_t* mr = mask + (mask_stride > 0 ? (size_t)(row / mask_stride) * N : 0) + c;
      const i32x4_any m0 = *reinterpret_cast<const i32x4_any*>(mr);
      const i32x4_any m1 = *reinterpret_cast<const i32x4_any*>(mr + 4);
      on = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) on |= (m0[e] != 0 ? 1u << e : 0u) | (m1[e] != 0 ? 16u << e : 0u);
    }
  }
  float m = -INFINITY;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (on & (1u << e)) m = fmaxf(m, (float)v[e]);
  m = lanes_reduce<LPR>(m, MaxOp{});
  float p[8], s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    p[e] = 0.f;
    if (on & (1u << e)) {
      p[e] = __expf((float)v[e] - m);
      s += p[e];
    }
  }
  s = lanes_reduce<LPR>(s, AddOp{});
  const float inv = s > 0.f ? 1.0f / s : 0.f;
  if (!in) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (on & (1u << e)) ? (f16)(p[e] * inv) : (f16)0.f;
  *reinterpret_cast<f16x8_any*>(r) = v;
}

// merged[b*seq+i, h*32+d] = sum_j P[z, i, j] V[b, j, d] (attention.cu:65-93):
// any seq, one value per thread.
__global__ __launch_bounds__(256) void context1_kernel(const f16* __restrict__ probs,
                                                       const f16* __restrict__ qkv,
                                                       f16* __restrict__ merged, int heads,
                                                       int seq, int ld, int v_off) {
  const int z = blockIdx.y, b = z / heads, h = z % heads;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= seq * kHeadDim) return;
  const int i = idx / kHeadDim, d = idx % kHeadDim;
  const f16* pr = probs + ((size_t)z * seq + i) * seq;
  const f16* vc = qkv + (size_t)b * seq * ld + v_off + h * kHeadDim + d;
  float acc = 0.f;
  for (int j = 0; j < seq; ++j) acc += (float)pr[j] * (float)vc[(size_t)j * ld];
  merged[((size_t)b * seq + i) * heads * kHeadDim + h * kHeadDim + d] = (f16)acc;
}

// The same for seq % 16 == 0 on the matrix cores: a wavefront makes 32
// queries x 32 dims as O^T = V^T . P^T.  The probabilities are the B operand
// as they lie (a lane's eight keys are contiguous); V is staged transposed
// in LDS, kCtxKeys keys at a time, for the workgroup's NW query tiles.
// Bound by reading the probabilities: batch 32 x seq 128 took 107 us with one
// value per thread (a chain of seq dependent adds), against 6.5 us here.
constexpr int kCtxKeys = 512;
template <int NW>
__global__ __launch_bounds__(64 * NW) void context_kernel(const f16* __restrict__ probs,
                                                          const f16* __restrict__ qkv,
                                                          f16* __restrict__ merged, int heads,
                                                          int seq, int ld, int v_off) {
  HIP_DYNAMIC_SHARED(f16, Vt);  // [32][min(seq, kCtxKeys) + 8]
  const int vld = min(seq, kCtxKeys) + 8;
  const int z = blockIdx.y, b = z / heads, h = z % heads;
  const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, kh = lane >> 5;
  const int q = ((int)blockIdx.x * NW + (tid >> 6)) * 32 + r32;
  const f16* pr = probs + ((size_t)z * seq + min(q, seq - 1)) * seq + 8 * kh;
  const f16* vb = qkv + (size_t)b * seq * ld + v_off + h * kHeadDim;
  f32x16 o = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // The probabilities of up to 128 keys are loaded together (eight k-steps;
  // seq is uniform, so a shorter end only skips steps), the first ones before
  // V is staged.
  f16x8 p[8];
  auto load_p = [&](int k) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + 16 * u < seq) p[u] = *reinterpret_cast<const f16x8_any*>(pr + k + 16 * u);
  };
  load_p(0);
  for (int k0 = 0; k0 < seq; k0 += kCtxKeys) {
    const int nk = min(kCtxKeys, seq - k0);
    if (k0 > 0) __syncthreads();
    for (int i = tid; i < nk * 2; i += 64 * NW) {  // a 4-key x 4-dim block per thread
      const int dq = i & 7, kq = i >> 3;
      f16x4 r[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        r[e] = *reinterpret_cast<const f16x4_any*>(vb + (size_t)(k0 + 4 * kq + e) * ld + 4 * dq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f16x4 col = {r[0][e], r[1][e], r[2][e], r[3][e]};
        *reinterpret_cast<f16x4*>(Vt + (4 * dq + e) * vld + 4 * kq) = col;
      }
    }
    __syncthreads();
    const f16* vt = Vt + r32 * vld + 8 * kh;
    for (int k = 0; k < nk; k += 128) {
      if (k0 + k > 0) load_p(k0 + k);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k + 16 * u < nk)  // o[i] = O[q][8*(i/4) + 4*kh + i%4]
          o = mfma32(*reinterpret_cast<const f16x8*>(vt + k + 16 * u), p[u], o);
    }
  }
  if (q >= seq) return;
  f16* dst = merged + (((size_t)b * seq + q) * heads + h) * kHeadDim + 4 * kh;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f16x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = (f16)o[4 * j + e];
    *reinterpret_cast<f16x4_any*>(dst + 8 * j) = w;
  }
}

template <int NW>
void launch_context(const f16* probs, const f16* qkv, f16* merged, int batch, int heads, int seq,
                    int ld, int v_off, hipStream_t s) {
  const int tiles = (seq + 31) / 32;
  const size_t lds = (size_t)kHeadDim * (std::min(seq, kCtxKeys) + 8) * sizeof(f16);
  hipLaunchKernelGGL(context_kernel<NW>, dim3((tiles + NW - 1) / NW, batch * heads), dim3(64 * NW),
                     lds, s, probs, qkv, merged, heads, seq, ld, v_off);
}

}  // namespace


hipError_t attention_scores(const f16* qkv, f16* scores, int batch, int heads, int seq,
                            int qkv_stride, int q_off, int k_off_, float scale,
                            hipStream_t s) {
  const unsigned qblocks = (seq + 127) / 128, kblocks = (seq + kScoreKeys - 1) / kScoreKeys;
  hipLaunchKernelGGL(scores_kernel, dim3(qblocks * kblocks, batch * heads), dim3(256), 0, s, qkv,
                     scores, heads, seq, qkv_stride, q_off, k_off_, scale);
  return hipGetLastError();
}

// A row of up to 512 values in multiples of eight stays in the registers of
// up to 64 lanes; other rows take three passes over memory.
hipError_t softmax_rows(f16* x, int M, int N, const int32_t* mask, int mask_stride,
                        hipStream_t s) {
#define BBH_SOFTMAX8(LPR)                                                                   \
  hipLaunchKernelGGL(softmax8_kernel<LPR>, dim3((M + 256 / LPR - 1) / (256 / LPR)), dim3(256), 0, \
                     s, x, M, N, mask, mask_stride)
  if (N % 8 != 0 || N > 512)
    hipLaunchKernelGGL(softmax_kernel, dim3((M + 3) / 4), dim3(256), 0, s, x, M, N, mask,
                       mask_stride);
  else if (N <= 16)
    BBH_SOFTMAX8(2);
  else if (N <= 32)
    BBH_SOFTMAX8(4);
  else if (N <= 64)
    BBH_SOFTMAX8(8);
  else if (N <= 128)
    BBH_SOFTMAX8(16);
  else if (N <= 256)
    BBH_SOFTMAX8(32);
  else
    BBH_SOFTMAX8(64);
#undef BBH_SOFTMAX8
  return hipGetLastError();
}

// The matrix cores take 16 keys a step, so other lengths go one value a
// thread.  Up to four query tiles share a workgroup's staged V.
hipError_t attention_context(const f16* probs, const f16* qkv, f16* merged, int batch,
                             int heads, int seq, int qkv_stride, int v_off, hipStream_t s) {
  if (seq % 16 != 0)
    hipLaunchKernelGGL(context1_kernel, dim3((seq * kHeadDim + 255) / 256, batch * heads),
                       dim3(256), 0, s, probs, qkv, merged, heads, seq, qkv_stride, v_off);
  else if (seq <= 32)
    launch_context<1>(probs, qkv, merged, batch, heads, seq, qkv_stride, v_off, s);
  else if (seq <= 64)
    launch_context<2>(probs, qkv, merged, batch, heads, seq, qkv_stride, v_off, s);
  else
    launch_context<4>(probs, qkv, merged, batch, heads, seq, qkv_stride, v_off, s);
  return hipGetLastError();
}

}  // namespace bbh
