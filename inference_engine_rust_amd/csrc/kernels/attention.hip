// Attention over a KV cache laid out per layer as [n_kv][ctx][head_dim] (f32 in the sessions; fp16
// through the op-level entry).
//
// Decode (src/layers/attention.rs:462-655): split-K flash-decode over chunks of keys, GQA groups
// sharing one K/V stream; in a session the chunks are fixed by the cache capacity, so the launch
// shape never changes between captured decode steps, and the live length is read from device memory.
//
// Prefill (attention.rs:175-422): causal attention over the f32 K/V of the prompt (the
// reference attends to the layer's own k_data/v_data, not the cache).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_core.cuh"

namespace iek {

template <int HD, bool EARLY, int SETS, bool COH, typename T>
__global__ __launch_bounds__(256 * SETS) void attn_decode_kernel(const float* __restrict__ q, const T* __restrict__ kc,
                                                                 const T* __restrict__ vc, float* __restrict__ part,
                                                                 float* __restrict__ out, int* __restrict__ counters,
                                                                 int n_heads, int n_kv, int ctx, const int* pos_dev,
                                                                 int total, int window, float scale, int nsplit,
                                                                 int spc, int HG) {
  __shared__ __align__(16) char smem[AttnSmem<HD, SETS, T>::BYTES];
  // all arguments in one batch of scalar loads, ahead of the position they depend on
  asm volatile("" ::"s"(q), "s"(kc), "s"(vc), "s"(part), "s"(out), "s"(counters), "s"(n_heads), "s"(n_kv), "s"(ctx),
               "s"(pos_dev), "s"(total), "s"(window), "s"(scale), "s"(nsplit), "s"(spc), "s"(HG));
  attn_chunk<HD, COH, EARLY, SETS, T>(q, kc, vc, part, out, counters, n_heads, n_kv, ctx, pos_dev, total, window, scale,
                                      nsplit, blockIdx.x / HG, blockIdx.y, spc, smem, blockIdx.x % HG, HG);
}

// head_dim 256 and 512. Latency-bound: one launch reads under 2 MB at the contexts of the models with
// such heads. Against slices of 64 keys staged in LDS (two workgroup barriers a slice, every head's
// wave reading the whole slice back from LDS): 75 keys of one KV head 8.6 -> 6.8 us at 256, 14.8 ->
// 9.5 at 512; 500 keys of 512 17.4 -> 11.8; 8000 keys 54 -> 28.
// The head groups of a KV head are n_kv workgroups apart, so that they share an XCD's L2 when n_kv is a
// multiple of the 8 XCDs (8 KV heads of 64 query heads, 32000 f32 keys of 256: 176 -> 131 us).
template <int HD, int NG, bool EARLY, typename T>
__global__ __launch_bounds__(256) void attn_decode_wide_kernel(const float* __restrict__ q, const T* __restrict__ kc,
                                                               const T* __restrict__ vc, float* __restrict__ part,
                                                               float* __restrict__ out, int* __restrict__ counters,
                                                               int n_heads, int n_kv, int ctx, const int* pos_dev,
                                                               int total, int window, float scale, int nslot, int CK,
                                                               int HG, int first) {
  __shared__ __align__(16) AttnWide<HD> smem;
  asm volatile("" ::"s"(q), "s"(kc), "s"(vc), "s"(part), "s"(out), "s"(counters), "s"(n_heads), "s"(n_kv), "s"(ctx),
               "s"(pos_dev), "s"(total), "s"(window), "s"(scale), "s"(nslot), "s"(CK), "s"(HG), "s"(first));
  attn_chunk_wide<HD, NG, EARLY, T>(q, kc, vc, part, out, counters, n_heads, n_kv, ctx, pos_dev, total, window, scale,
                                    nslot, blockIdx.x % n_kv, first + blockIdx.y, CK, smem, blockIdx.x / n_kv, HG);
}

template <int HD, typename T>
static void attn_decode_hd(hipStream_t st, const float* q, const T* kc, const T* vc, float* out, float* part,
                           int* counters, int n_heads, int n_kv, int ctx, const int* pos_dev, int total, int window,
                           float scale, int max_len) {
  // A group of 8 query heads splits over two workgroups per chunk (four heads each, one per
  // wave) when there are few KV heads to spread over the machine (one KV head: Gemma-4-E2B);
  // each half has its own arrival counter (2 * n_kv counters) and merge.
  const int HG = (n_heads / n_kv == 8 && n_kv < 4) ? 2 : 1;
  // Chunks of spc slices (about 32 chunks per KV head); one partial slot per chunk. Where the host knows
  // the length, one-slice chunks only while all KV heads' fit one to a CU, and at most one chunk per CU
  // (fp16: two). us with chunks of 1 / 2 / 3 / 4 slices at head_dim 128, f32: 8 KV heads, 2000 keys (256
  // slices in all) 13.8 / 13.1 / 15.6 / 16.1; 16, 1100 (288) 14.1 / 12.1 / 14.3 / 15.0; 16, 2600 (656) 29.9 /
  // 21.8 / 17.6 / 18.1; 32, 1500 (768) 32.3 / 20.6 / 17.9 / 18.2; fp16: 16, 2000 (512) 18.1 / 12.5 / 13.4 /
  // 13.8; 32, 2000 (1024) 31.1 / 13.4 / 14.3 / 14.0; 16, 32000 with 512 chunks 50, with 256 59.
  const int nsl = (max_len + SPLIT - 1) / SPLIT;
  int spc = attn_slices_per_chunk(max_len, window, 32);
  if (!pos_dev) {
    const long long live = window > 0 ? std::min(nsl, (window + SPLIT - 1) / SPLIT + 1) : nsl;
    const long long all = live * n_kv * HG, cus = num_cus(), fit = cus * (sizeof(T) == 4 ? 1 : 2);
    spc = std::max({spc, (int)((all + fit - 1) / fit), all > cus ? 2 : 1});
  }
  const int nchunk = (nsl + spc - 1) / spc;
  // Chunks of several slices (long contexts) run two slice streams per workgroup, and publish their
  // partials with coherent stores and a relaxed count (no L2 write-back / invalidate around the
  // arrival, measured faster there; one-slice chunks are faster with plain stores).
  const bool two = spc >= 2;
  auto go = [&](auto kern, int nt) {
    hipLaunchKernelGGL(kern, dim3(n_kv * HG, nchunk), dim3(nt), 0, st, q, kc, vc, part, out, counters, n_heads, n_kv,
                       ctx, pos_dev, total, window, scale, nchunk, spc, HG);
  };
  // without a window the first slice's loads go out before the position is known
  if (window <= 0)
    two ? go(attn_decode_kernel<HD, true, 2, true, T>, 512) : go(attn_decode_kernel<HD, true, 1, false, T>, 256);
  else
    two ? go(attn_decode_kernel<HD, false, 2, true, T>, 512) : go(attn_decode_kernel<HD, false, 1, false, T>, 256);
}

// Partial slots per query head: one per 64 keys; at head_dim 256 and up, whose chunks go down to 8
// keys, one per 8 as far as that keeps n_heads * slots within 4096.
static int attn_slots(int n_heads, int head_dim, int max_len) {
  const int n = (max_len + SPLIT - 1) / SPLIT;
  return head_dim < 256 ? n : std::max(n, std::min((max_len + 7) / 8, 4096 / std::max(n_heads, 1)));
}

template <int HD, typename T>
static void attn_decode_wide(hipStream_t st, const float* q, const T* kc, const T* vc, float* out, float* part,
                             int* counters, int n_heads, int n_kv, int ctx, const int* pos_dev, int total, int window,
                             float scale, int max_len) {
  const int HG = (n_heads / n_kv + 3) / 4;
  // Keys per chunk: a chunk's time grows with its keys and the merge's with the number of chunks,
  // so about sqrt(2 * keys) of them (a window keeps only ~window keys live). Measured with 16 / 32 /
  // 64 chunks per KV head, one KV head of 512: 11.8 / 13.3 / 17.5 us at 500 keys, 20.2 / 17.3 / 19.9
  // at 2000, 49 / 33 / 28 at 8000. In whole steps of the workgroup, within the partial slots and with at
  // most MERGE_SLOTS live chunks (a window touches one more than its own length holds).
  constexpr int UNIT = AttnWide<HD>::UNIT;
  const int span = window > 0 ? std::min(max_len, window) : max_len, slots = attn_slots(n_heads, HD, max_len);
  // Several KV heads fill the chip with fewer chunks each, and more of them only add launches and
  // partials: one chunk of all KV heads per CU, two of an fp16 cache once they hold 512 keys. us with
  // sqrt(2 * keys) / one / two per CU: 16 KV heads of 256, f32, 8000 keys 85 / 48 / 57, fp16 59 / 41 / 43,
  // 32000 196 / 142 / 120; 32 query heads of 8 KV heads of 512, f32, 32000 273 / 206 / 222. A session's
  // chunks are sized for its whole cache, of which any part may be live: 32 per KV head remain there.
  const long long cus = num_cus(), all = (long long)span * n_kv;
  const long long fill = pos_dev         ? std::min<long long>(all * HG / (2 * cus), (span + 31) / 32)
                         : sizeof(T) == 4 ? all / cus
                                          : std::min(all / cus, std::max(512ll, all / (2 * cus)));
  const int keys = std::max({(int)std::sqrt(2.0 * span), (int)fill, (max_len + slots - 1) / slots,
                             (span + MERGE_SLOTS - 2) / (MERGE_SLOTS - 1)});
  const int CK = (keys + UNIT - 1) / UNIT * UNIT, nchunk = (max_len + CK - 1) / CK;
  // the first chunk with a live key, where the host knows the length
  const int first = !pos_dev && window > 0 && total > window ? (total - window) / CK : 0;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(n_kv * HG, nchunk - first), dim3(256), 0, st, q, kc, vc, part, out, counters, n_heads,
                       n_kv, ctx, pos_dev, total, window, scale, nchunk, CK, HG, first);
  };
  // without a window the first step's loads go out before the position is known
  if (n_heads == n_kv)
    window <= 0 ? go(attn_decode_wide_kernel<HD, 1, true, T>) : go(attn_decode_wide_kernel<HD, 1, false, T>);
  else
    window <= 0 ? go(attn_decode_wide_kernel<HD, 4, true, T>) : go(attn_decode_wide_kernel<HD, 4, false, T>);
}

size_t attn_decode_part_floats(int n_heads, int head_dim, int max_len) {
  return (size_t)n_heads * attn_slots(n_heads, head_dim, max_len) * (head_dim + 2);
}

void launch_attn_decode(const float* q, const void* kc, const void* vc, bool kv_f32, float* out, float* part,
                        int* counters, int n_heads, int n_kv, int head_dim, int ctx, const int* pos_dev, int window,
                        float scale, int max_len, hipStream_t st, int total) {
  if (n_kv <= 0 || n_heads % n_kv != 0 || n_heads / n_kv > 8)
    fail(ST_OP, "attention: GQA group must divide the heads and be at most 8");
#define IEK_AD(FN, HD)                                                                                              \
  kv_f32 ? FN<HD>(st, q, (const float*)kc, (const float*)vc, out, part, counters, n_heads, n_kv, ctx, pos_dev,      \
                  total, window, scale, max_len)                                                                    \
         : FN<HD>(st, q, (const __half*)kc, (const __half*)vc, out, part, counters, n_heads, n_kv, ctx, pos_dev,    \
                  total, window, scale, max_len)
  switch (head_dim) {
    case 64:
      IEK_AD(attn_decode_hd, 64);
      break;
    case 128:
      IEK_AD(attn_decode_hd, 128);
      break;
    case 256:
      IEK_AD(attn_decode_wide, 256);
      break;
    case 512:
      IEK_AD(attn_decode_wide, 512);
      break;
    default:
      fail(ST_OP, "attention: head_dim must be 64, 128, 256 or 512");
  }
#undef IEK_AD
}

// Prefill on the matrix cores (v_mfma_f32_16x16x32_f16): one 256-thread workgroup per (head,
// 64-query tile), each wave owning 16 queries; 64-key blocks of K (row-major) and V (transposed)
// are staged in LDS as fp16 (hi, lo) pairs, S = Q K^T and O += P V each take three MFMAs per step
// (hi*hi + hi*lo + lo*hi, products exact in f32), and the softmax is the online form (running max
// per query row, sum rescaled whenever the max grows).
typedef _Float16 ah8_t __attribute__((ext_vector_type(8)));
typedef float af4_t __attribute__((ext_vector_type(4)));
typedef uint32_t au4_t __attribute__((ext_vector_type(4)));

IEK_DEV uint32_t apack2(_Float16 a, _Float16 b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}

IEK_DEV void asplit(float v, _Float16& h, _Float16& l) {
#pragma clang fp contract(off)
  h = (_Float16)v;
  l = (_Float16)(v - (float)h);
}

IEK_DEV af4_t mma3(au4_t ah, au4_t al, au4_t bh, au4_t bl, af4_t c) {
  const ah8_t a_h = __builtin_bit_cast(ah8_t, ah), a_l = __builtin_bit_cast(ah8_t, al);
  const ah8_t b_h = __builtin_bit_cast(ah8_t, bh), b_l = __builtin_bit_cast(ah8_t, bl);
  c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_h, b_h, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_h, b_l, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_l, b_h, c, 0, 0, 0);
  return c;
}

// KB keys per block: 64 up to head_dim 128; 32 at 256 and 512, where the (hi, lo) K block, the
// transposed V block and the P tiles must still fit the 160 KB of LDS.
template <int HD, int KB>
__global__ __launch_bounds__(256) void attn_prefill_mfma_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                                const float* __restrict__ v, float* __restrict__ out,
                                                                int M, int n_heads, int n_kv, int window, float scale) {
  constexpr int JN = KB / 16;    // 16-key column tiles of S
  constexpr int KS = HD / 32;    // MFMA K steps of S = Q K^T
  constexpr int NS = HD / 16;    // 16-wide head-dim subtiles of O
  constexpr int KROW = HD + 8;   // padded LDS rows (halves)
  constexpr int VROW = KB + 8;
  __shared__ __align__(16) _Float16 kh[KB][KROW];
  __shared__ __align__(16) _Float16 kl[KB][KROW];
  __shared__ __align__(16) _Float16 vth[HD][VROW];
  __shared__ __align__(16) _Float16 vtl[HD][VROW];
  __shared__ __align__(16) _Float16 ph[4][16][VROW];
  __shared__ __align__(16) _Float16 pl[4][16][VROW];

  const int h = blockIdx.x, qt = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = n_heads / n_kv, kvh = h / G;
  const int qd = n_heads * HD, kvd = n_kv * HD;
  const int q0 = qt * 64 + 16 * wave;
  const int fr = lane & 15, fk = 8 * (lane >> 4);

  // Q fragments (A operand): row q0 + fr, dims 32 s + fk .. +7, split into fp16 pairs
  au4_t qah[KS], qal[KS];
  {
    const float* qrow = q + (size_t)min(q0 + fr, M - 1) * qd + h * HD;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float4 a = *reinterpret_cast<const float4*>(qrow + 32 * s + fk);
      const float4 b = *reinterpret_cast<const float4*>(qrow + 32 * s + fk + 4);
      const float vv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      _Float16 hh[8], ll[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) asplit(vv[t], hh[t], ll[t]);
      qah[s] = au4_t{apack2(hh[0], hh[1]), apack2(hh[2], hh[3]), apack2(hh[4], hh[5]), apack2(hh[6], hh[7])};
      qal[s] = au4_t{apack2(ll[0], ll[1]), apack2(ll[2], ll[3]), apack2(ll[4], ll[5]), apack2(ll[6], ll[7])};
    }
  }
  af4_t o[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) o[j] = af4_t{0.f, 0.f, 0.f, 0.f};
  float mrow[4], lrow[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    mrow[r] = -INFINITY;
    lrow[r] = 0.f;
  }
  const int last_q = min(M - 1, qt * 64 + 63);
  const int jmin_tile = window > 0 ? max(0, qt * 64 - (window - 1)) : 0;
  for (int kb0 = (jmin_tile / KB) * KB; kb0 <= last_q; kb0 += KB) {
    __syncthreads();  // the previous block's LDS reads are done
    for (int e = tid; e < KB * HD / 4; e += 256) {
      const int j = e / (HD / 4), d4 = 4 * (e % (HD / 4));
      const size_t row = (size_t)min(kb0 + j, M - 1) * kvd + kvh * HD + d4;
      const float4 kk = *reinterpret_cast<const float4*>(k + row);
      const float4 vv = *reinterpret_cast<const float4*>(v + row);
      const float kf[4] = {kk.x, kk.y, kk.z, kk.w}, vf[4] = {vv.x, vv.y, vv.z, vv.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        asplit(kf[t], kh[j][d4 + t], kl[j][d4 + t]);
        asplit(vf[t], vth[d4 + t][j], vtl[d4 + t][j]);
      }
    }
    __syncthreads();
    if (kb0 > q0 + 15) continue;  // every query of this wave precedes the block
    // S = Q K^T for the wave's 16 queries x KB keys
    af4_t sacc[JN];
#pragma unroll
    for (int jn = 0; jn < JN; ++jn) {
      sacc[jn] = af4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const au4_t bh = *reinterpret_cast<const au4_t*>(&kh[16 * jn + fr][32 * s + fk]);
        const au4_t bl = *reinterpret_cast<const au4_t*>(&kl[16 * jn + fr][32 * s + fk]);
        sacc[jn] = mma3(qah[s], qal[s], bh, bl, sacc[jn]);
      }
    }
    // mask, scale, online softmax; lane holds rows 4 * (lane >> 4) + r, key column 16 jn + fr
    float p[JN][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = q0 + 4 * (lane >> 4) + r;
      const int jlo = window > 0 ? max(0, i - (window - 1)) : 0;
      float mx = -INFINITY;
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) {
        const int j = kb0 + 16 * jn + fr;
        const bool ok = j <= i && j >= jlo && j < M && i < M;
        const float sv = sacc[jn][r] * scale;
        p[jn][r] = ok ? sv : -INFINITY;
        mx = fmaxf(mx, p[jn][r]);
      }
      mx = row16_max(mx);
      const float mn = fmaxf(mrow[r], mx);
      const float corr = mn == -INFINITY ? 1.f : expf(mrow[r] - mn);
      float sum = 0.f;
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) {
        const float e = p[jn][r] == -INFINITY ? 0.f : expf(p[jn][r] - mn);
        p[jn][r] = e;
        sum += e;
      }
      sum = row16_sum(sum);
      lrow[r] = lrow[r] * corr + sum;
      mrow[r] = mn;
#pragma unroll
      for (int j = 0; j < NS; ++j) o[j][r] *= corr;
    }
    // P to LDS in A-operand order [query][key] (this wave's slice only)
#pragma unroll
    for (int jn = 0; jn < JN; ++jn)
#pragma unroll
      for (int r = 0; r < 4; ++r) asplit(p[jn][r], ph[wave][4 * (lane >> 4) + r][16 * jn + fr], pl[wave][4 * (lane >> 4) + r][16 * jn + fr]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // O += P V
#pragma unroll
    for (int ks = 0; ks < KB / 32; ++ks) {
      const au4_t pah = *reinterpret_cast<const au4_t*>(&ph[wave][fr][32 * ks + fk]);
      const au4_t pal = *reinterpret_cast<const au4_t*>(&pl[wave][fr][32 * ks + fk]);
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const au4_t bh = *reinterpret_cast<const au4_t*>(&vth[16 * j + fr][32 * ks + fk]);
        const au4_t bl = *reinterpret_cast<const au4_t*>(&vtl[16 * j + fr][32 * ks + fk]);
        o[j] = mma3(pah, pal, bh, bl, o[j]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = q0 + 4 * (lane >> 4) + r;
    if (i < M) {
#pragma unroll
      for (int j = 0; j < NS; ++j) out[(size_t)i * qd + h * HD + 16 * j + fr] = o[j][r] / lrow[r];
    }
  }
}

// ---- prefill attention sharing each K/V block across the query heads of a KV head --------------
// K and V (f32 rows [M][n_kv * HD]) are split once per layer into fp16 (hi, lo) planes laid out for
// the MFMA B operands: K per KV head as [n_kv][M][HD], V transposed as [n_kv][HD][Mp] (Mp = M
// rounded up to 64; the padding is zero). One 64 x 64 tile per workgroup, through LDS for V.
__global__ __launch_bounds__(256) void kv_split_kernel(const float* __restrict__ k, const float* __restrict__ v, int M,
                                                       int n_kv, int hd, int Mp, _Float16* __restrict__ kh,
                                                       _Float16* __restrict__ kl, _Float16* __restrict__ vh,
                                                       _Float16* __restrict__ vl, int* __restrict__ ovf) {
  __shared__ float tile[64][65];
  const int h = blockIdx.z, d0 = blockIdx.y * 64, p0 = blockIdx.x * 64, tid = threadIdx.x;
  const int c4 = 4 * (tid & 15), d = d0 + c4;  // the thread's four head dims (hd is a multiple of 64)
  const size_t kvd = (size_t)n_kv * hd;
  bool big = false;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int pl = (tid >> 4) + 16 * r, p = p0 + pl;
    float vv[4] = {0.f, 0.f, 0.f, 0.f};
    if (p < M) {
      const size_t src = (size_t)p * kvd + (size_t)h * hd + d;
      _Float16 a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float kx = k[src + i];
        vv[i] = v[src + i];
        big |= fmaxf(fabsf(kx), fabsf(vv[i])) > F16_PAIR_MAX;
        asplit(kx, a[i], b[i]);
      }
      const size_t kd = ((size_t)h * M + p) * hd + d;
      *reinterpret_cast<uint2*>(kh + kd) = make_uint2(apack2(a[0], a[1]), apack2(a[2], a[3]));
      *reinterpret_cast<uint2*>(kl + kd) = make_uint2(apack2(b[0], b[1]), apack2(b[2], b[3]));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) tile[pl][c4 + i] = vv[i];
  }
  if (big && ovf) *ovf = 1;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int dl = (tid >> 5) + 8 * r, pl = 2 * (tid & 31);  // Mp is a multiple of 64: every p < Mp
    _Float16 a[2], b[2];
    asplit(tile[pl][dl], a[0], b[0]);
    asplit(tile[pl + 1][dl], a[1], b[1]);
    const size_t vd = ((size_t)h * hd + d0 + dl) * Mp + p0 + pl;
    *reinterpret_cast<uint32_t*>(vh + vd) = apack2(a[0], a[1]);
    *reinterpret_cast<uint32_t*>(vl + vd) = apack2(b[0], b[1]);
  }
}

// The prompt's attention inputs in one pass (replaces RoPE on Q and on K, the KV append and
// kv_split_kernel): workgroup (position tile, 64-dim tile, z); a thread takes four consecutive head
// dims (two RoPE pairs, the arithmetic of rotate() in ops.hip, src/ops/rope.rs:11-59) of rows
// (tid >> 4) + 16 r. z < n_kv: KV head z, whose K rows get RoPE at the prompt positions 0..M-1 in
// registers, then go to the cache at pos0 + p (f32 or fp16, as kv_store_kernel) and to the K
// planes; V goes to the cache and, through LDS, to the transposed V planes. z >= n_kv: query head
// z - n_kv gets RoPE in place.
IEK_DEV void rope4(float4& x, const float* cs, int p, int npairs, int d) {
#pragma clang fp contract(off)
  const float2* e = reinterpret_cast<const float2*>(cs) + (size_t)p * npairs + (d >> 1);
  if (d < 2 * npairs) {
    const float2 c = e[0];
    const float t0 = x.x, t1 = x.y;
    x.x = t0 * c.x - t1 * c.y;
    x.y = t0 * c.y + t1 * c.x;
  }
  if (d + 2 < 2 * npairs) {
    const float2 c = e[1];
    const float t0 = x.z, t1 = x.w;
    x.z = t0 * c.x - t1 * c.y;
    x.w = t0 * c.y + t1 * c.x;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void attn_prep_kernel(float* __restrict__ q, const float* __restrict__ k,
                                                        const float* __restrict__ v, int M, int n_heads, int n_kv,
                                                        int hd, int Mp, const float* __restrict__ cs, int npairs,
                                                        T* __restrict__ kc, T* __restrict__ vc, int ctx, int pos0,
                                                        _Float16* __restrict__ kh, _Float16* __restrict__ kl,
                                                        _Float16* __restrict__ vh, _Float16* __restrict__ vl,
                                                        int* __restrict__ ovf) {
  __shared__ float tile[64][65];
  const int z = blockIdx.z, d0 = blockIdx.y * 64, p0 = blockIdx.x * 64, tid = threadIdx.x;
  const int c4 = 4 * (tid & 15), d = d0 + c4;  // the thread's four head dims
  auto big4 = [](const float4& x) {
    return fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))) > F16_PAIR_MAX;
  };
  if (z >= n_kv) {
    const int h = z - n_kv;
    const size_t qd = (size_t)n_heads * hd;
    bool big = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p = p0 + (tid >> 4) + 16 * r;
      if (p < M && d < hd) {
        float4* e = reinterpret_cast<float4*>(q + (size_t)p * qd + (size_t)h * hd + d);
        float4 x = *e;
        rope4(x, cs, p, npairs, d);
        *e = x;
        big |= big4(x);
      }
    }
    if (big) *ovf = 1;
    return;
  }
  bool big = false;
  const int h = z;
  const size_t kvd = (size_t)n_kv * hd;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int pl = (tid >> 4) + 16 * r, p = p0 + pl;
    float4 vv = make_float4(0.f, 0.f, 0.f, 0.f);
    if (p < M && d < hd) {
      const size_t src = (size_t)p * kvd + (size_t)h * hd + d;
      float4 kx = *reinterpret_cast<const float4*>(k + src);
      vv = *reinterpret_cast<const float4*>(v + src);
      rope4(kx, cs, p, npairs, d);
      big |= big4(kx) || big4(vv);
      const size_t dst = ((size_t)h * ctx + pos0 + p) * hd + d;
      if constexpr (std::is_same<T, float>::value) {
        *reinterpret_cast<float4*>(kc + dst) = kx;
        *reinterpret_cast<float4*>(vc + dst) = vv;
      } else {
        kc[dst] = __float2half_rn(kx.x);
        kc[dst + 1] = __float2half_rn(kx.y);
        kc[dst + 2] = __float2half_rn(kx.z);
        kc[dst + 3] = __float2half_rn(kx.w);
        vc[dst] = __float2half_rn(vv.x);
        vc[dst + 1] = __float2half_rn(vv.y);
        vc[dst + 2] = __float2half_rn(vv.z);
        vc[dst + 3] = __float2half_rn(vv.w);
      }
      _Float16 a[4], b[4];
      asplit(kx.x, a[0], b[0]);
      asplit(kx.y, a[1], b[1]);
      asplit(kx.z, a[2], b[2]);
      asplit(kx.w, a[3], b[3]);
      const size_t kd = ((size_t)h * M + p) * hd + d;
      *reinterpret_cast<uint2*>(kh + kd) = make_uint2(apack2(a[0], a[1]), apack2(a[2], a[3]));
      *reinterpret_cast<uint2*>(kl + kd) = make_uint2(apack2(b[0], b[1]), apack2(b[2], b[3]));
    }
    tile[pl][c4] = vv.x;
    tile[pl][c4 + 1] = vv.y;
    tile[pl][c4 + 2] = vv.z;
    tile[pl][c4 + 3] = vv.w;
  }
  if (big) *ovf = 1;
  __syncthreads();
#pragma unroll 4
  for (int r = 0; r < 16; ++r) {
    const int dt = (tid >> 6) + 4 * r, pl = tid & 63, dd = d0 + dt, p = p0 + pl;
    if (dd < hd && p < Mp) {
      _Float16 a, b;
      asplit(tile[pl][dt], a, b);
      const size_t vd = ((size_t)h * hd + dd) * Mp + p;
      vh[vd] = a;
      vl[vd] = b;
    }
  }
}

// One workgroup of NW waves per (KV head, group of up to 4 query heads, query tile): wave w takes
// query head w % G4 and query sub-tile w / G4 (G4 = min(G, 4)), TMQ 16-query MFMA tiles of it. Each
// KB-key block (64; 32 at head_dim 256) of K and V^T is staged once in LDS (16-byte copies of the split planes, the next
// block's loads in flight during the current block's MFMAs) and serves every query head of the
// KV head. The scores are computed transposed, S^T = K Q^T with the keys as MFMA rows: a lane's
// 16 scores of a block then all belong to one query (lane & 15), and with the K rows staged in the
// order krow() gives, the lane's keys of block steps 2t and 2t + 1 are exactly the 8 consecutive
// keys 32t + 8(lane >> 4) .. + 7 that it supplies as the B operand of O^T += V^T P^T. P stays in
// registers (no LDS round trip, no wave barrier), and 72 KB of LDS lets two workgroups share a
// CU (NW = 4) or gives eight waves one staged block (NW = 8). Every product takes three MFMAs (hi*hi +
// hi*lo + lo*hi of the fp16 pairs, exact in f32); the softmax is the online form per query. The longest
// (latest) query tiles are dispatched first.
// KG = 2: two sets of NW waves take the tile's key blocks in turn, each with its own staged block,
// and the second set's (max, sum, O) are folded in through LDS at the end (head_dim 256 where the
// grid leaves CUs idle: 800 rows of 8 query heads are 100 workgroups). `ovf` (when q was not
// checked before): set when a q value is beyond the fp16 pair's range.
template <int HD, int TMQ, int NW, int KB, int KG = 1>
__global__ __launch_bounds__(64 * NW * KG, 8 / (NW * KG) > 0 ? 8 / (NW * KG) : 1) void attn_prefill_gqa_kernel(const float* __restrict__ q,
                                                                  const _Float16* __restrict__ kh,
                                                                  const _Float16* __restrict__ kl,
                                                                  const _Float16* __restrict__ vh,
                                                                  const _Float16* __restrict__ vl,
                                                                  float* __restrict__ out, int M, int Mp, int n_heads,
                                                                  int n_kv, int window, float scale,
                                                                  int* __restrict__ ovf) {
  static_assert(KB == 32 || KB == 64, "keys per block");
  constexpr int JN = KB / 16;    // 16-key row tiles of S^T
  constexpr int KS = HD / 32;    // MFMA K steps of S^T
  constexpr int NS = HD / 16;    // 16-wide head-dim row tiles of O^T
  constexpr int KROW = HD + 8;   // padded LDS rows (halves)
  constexpr int VROW = KB + 8;
  constexpr int QW = 16 * TMQ;   // queries per wave
  constexpr int NT = 64 * NW;
  constexpr int CPT = KB * HD / 8 / NT;  // 16-byte chunks per thread per plane of a K (or V^T) block
  static_assert(CPT >= 1 && (KB * HD / 8) % NT == 0, "block must divide over the threads");
  struct Block {
    _Float16 kh[KB][KROW], kl[KB][KROW], vh[HD][VROW], vl[HD][VROW];
  };
  __shared__ __align__(16) Block blk[KG];

  const int G = n_heads / n_kv, G4 = min(G, 4), HG = (G + 3) / 4;
  const int kvh = blockIdx.x / HG, hg = blockIdx.x % HG;
  const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
  const int tid = KG == 1 ? threadIdx.x : threadIdx.x % NT, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto& ksh = blk[kg].kh;
  auto& ksl = blk[kg].kl;
  auto& vsh = blk[kg].vh;
  auto& vsl = blk[kg].vl;
  const int hl = wave % G4, qs = wave / G4, h = 4 * hg + hl;
  const bool active = h < G && qs < NW / G4;
  const int QT = QW * (NW / G4);
  const int qt = gridDim.y - 1 - blockIdx.y;  // latest tiles first
  const int wq0 = qt * QT, wq1 = min(M - 1, wq0 + QT - 1);
  const int q0 = wq0 + qs * QW;
  const int hq = kvh * G + min(h, G - 1);
  const int qd = n_heads * HD;
  const int fr = lane & 15, lg = lane >> 4, fk = 8 * lg;

  // Q fragments (B operand of S^T: lane = query fr, dims fk .. fk + 7 of each 32-dim step) of the
  // wave's TMQ query tiles, scaled by scale * log2(e) so that the scores come out in base-2 units
  // (the softmax below is exp2(s - max), the same function), split into fp16 pairs
  const float qscale = scale * 1.44269504088896341f;
  au4_t qah[TMQ][KS], qal[TMQ][KS];
  bool qbig = false;
#pragma unroll
  for (int i = 0; i < TMQ; ++i) {
    const float* qrow = q + (size_t)min(q0 + 16 * i + fr, M - 1) * qd + (size_t)hq * HD;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float4 a = *reinterpret_cast<const float4*>(qrow + 32 * s + fk);
      const float4 b = *reinterpret_cast<const float4*>(qrow + 32 * s + fk + 4);
      const float vv[8] = {a.x * qscale, a.y * qscale, a.z * qscale, a.w * qscale,
                           b.x * qscale, b.y * qscale, b.z * qscale, b.w * qscale};
      if (ovf)
        qbig |= fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                      fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w)))) > F16_PAIR_MAX;
      _Float16 hh[8], ll[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) asplit(vv[t], hh[t], ll[t]);
      qah[i][s] = au4_t{apack2(hh[0], hh[1]), apack2(hh[2], hh[3]), apack2(hh[4], hh[5]), apack2(hh[6], hh[7])};
      qal[i][s] = au4_t{apack2(ll[0], ll[1]), apack2(ll[2], ll[3]), apack2(ll[4], ll[5]), apack2(ll[6], ll[7])};
    }
  }
  if (ovf && qbig) *ovf = 1;
  // O^T accumulators (lane: query fr, dims 16j + 4lg .. + 3) and the lane's query's softmax state
  // (running max in base-2 units, running sum)
  af4_t o[TMQ][NS];
  float mrow[TMQ], lrow[TMQ];
#pragma unroll
  for (int i = 0; i < TMQ; ++i) {
#pragma unroll
    for (int j = 0; j < NS; ++j) o[i][j] = af4_t{0.f, 0.f, 0.f, 0.f};
    mrow[i] = -INFINITY;
    lrow[i] = 0.f;
  }

  // staged block: K rows [row][dim] in krow order and V^T rows [dim][key], both planes
  const _Float16* khp = kh + (size_t)kvh * M * HD;
  const _Float16* klp = kl + (size_t)kvh * M * HD;
  const _Float16* vhp = vh + (size_t)kvh * HD * Mp;
  const _Float16* vlp = vl + (size_t)kvh * HD * Mp;
  // LDS row of key j of a block: key 32t + 8g + 4u + e goes to row 16(2t + u) + 4g + e, so that S^T
  // row tile jn = 2t + u holds, in lane group g's four output rows, keys 32t + 8g + 4u .. + 3
  auto krow = [](int j) { return (j & 32) + 16 * ((j >> 2) & 1) + 4 * ((j >> 3) & 3) + (j & 3); };
  au4_t rk[2][CPT], rv[2][CPT];
  auto fetch = [&](int kb0) {
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int e = tid + NT * c;
      const int j = e / (HD / 8), kc = e % (HD / 8);
      const size_t ks = (size_t)min(kb0 + j, M - 1) * HD + 8 * kc;
      rk[0][c] = *reinterpret_cast<const au4_t*>(khp + ks);
      rk[1][c] = *reinterpret_cast<const au4_t*>(klp + ks);
      const int d = e / (KB / 8), vc = e % (KB / 8);
      const size_t vs = (size_t)d * Mp + kb0 + 8 * vc;
      rv[0][c] = *reinterpret_cast<const au4_t*>(vhp + vs);
      rv[1][c] = *reinterpret_cast<const au4_t*>(vlp + vs);
    }
  };
  const int kb_start = window > 0 ? (max(0, wq0 - (window - 1)) / KB) * KB : 0;
  fetch(min(kb_start + KB * kg, Mp - KB));
  for (int kb1 = kb_start; kb1 <= wq1; kb1 += KB * KG) {
    const int kb0 = kb1 + KB * kg;  // (the last round may leave the second set without a block)
    __syncthreads();  // the previous block's LDS reads are done
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int e = tid + NT * c;
      const int j = e / (HD / 8), kc = e % (HD / 8);
      *reinterpret_cast<au4_t*>(&ksh[krow(j)][8 * kc]) = rk[0][c];
      *reinterpret_cast<au4_t*>(&ksl[krow(j)][8 * kc]) = rk[1][c];
      const int d = e / (KB / 8), vc = e % (KB / 8);
      *reinterpret_cast<au4_t*>(&vsh[d][8 * vc]) = rv[0][c];
      *reinterpret_cast<au4_t*>(&vsl[d][8 * vc]) = rv[1][c];
    }
    __syncthreads();
    if (kb0 + KB * KG <= wq1) fetch(kb0 + KB * KG);
    // the wave's queries all precede the block, or the block is older than all their windows
    if (!active || (KG > 1 && kb0 > wq1) || kb0 > q0 + QW - 1 || (window > 0 && kb0 + KB - 1 < q0 - (window - 1))) continue;
    // query tiles that reach into the block (uniform); each K and V^T fragment is read from LDS
    // once and serves all of them
    bool live[TMQ];
#pragma unroll
    for (int i = 0; i < TMQ; ++i) live[i] = kb0 <= q0 + 16 * i + 15;
    af4_t sacc[TMQ][JN];
#pragma unroll
    for (int i = 0; i < TMQ; ++i)
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) sacc[i][jn] = af4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int jn = 0; jn < JN; ++jn)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const au4_t ah = *reinterpret_cast<const au4_t*>(&ksh[16 * jn + fr][32 * s + fk]);
        const au4_t al = *reinterpret_cast<const au4_t*>(&ksl[16 * jn + fr][32 * s + fk]);
#pragma unroll
        for (int i = 0; i < TMQ; ++i)
          if (live[i]) sacc[i][jn] = mma3(ah, al, qah[i][s], qal[i][s], sacc[i][jn]);
        // keeps the fragment loads next to their MFMAs (hoisted, they would not fit the registers)
        if (TMQ > 1) __builtin_amdgcn_sched_barrier(0);
      }
    // per query tile: the online softmax of the lane's query, then P^T as the B operands of the two
    // 32-key steps (fp16 pairs); sacc[i][jn][r] is key kb0 + 32(jn >> 1) + 8lg + 4(jn & 1) + r
    au4_t pbh[TMQ][KB / 32], pbl[TMQ][KB / 32];
#pragma unroll
    for (int i = 0; i < TMQ; ++i) {
      if (!live[i]) continue;
      const int qi0 = q0 + 16 * i, qi = qi0 + fr;
      // every key of the block is visible to every query of the tile: no per-score mask
      const bool interior = kb0 + KB - 1 <= qi0 && kb0 + KB <= M && (window <= 0 || kb0 >= qi0 + 16 - window);
      float p[JN][4];
      float mx = -INFINITY;
      if (interior) {
#pragma unroll
        for (int jn = 0; jn < JN; ++jn)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[jn][r] = sacc[i][jn][r];
            mx = fmaxf(mx, p[jn][r]);
          }
      } else {
        const int jlo = window > 0 ? max(0, qi - (window - 1)) : 0;
#pragma unroll
        for (int jn = 0; jn < JN; ++jn)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = kb0 + 32 * (jn >> 1) + fk + 4 * (jn & 1) + r;
            const bool ok = j <= qi && j >= jlo && j < M && qi < M;
            p[jn][r] = ok ? sacc[i][jn][r] : -INFINITY;
            mx = fmaxf(mx, p[jn][r]);
          }
      }
      // lanes fr, fr + 16, fr + 32, fr + 48 hold the same query
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mn = fmaxf(mrow[i], mx);
      float sum = 0.f;
      if (mn == -INFINITY) {  // no visible key yet
#pragma unroll
        for (int jn = 0; jn < JN; ++jn)
#pragma unroll
          for (int r = 0; r < 4; ++r) p[jn][r] = 0.f;
      } else {
#pragma unroll
        for (int jn = 0; jn < JN; ++jn)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[jn][r] = __builtin_amdgcn_exp2f(p[jn][r] - mn);  // exp2(-inf) = 0 for a hidden key
            sum += p[jn][r];
          }
      }
      sum += __shfl_xor(sum, 16);
      sum += __shfl_xor(sum, 32);
      // the running max grows in a few blocks only: rescale when some lane's did
      if (__any(mn != mrow[i])) {
        const float corr = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(mrow[i] - mn);
        lrow[i] *= corr;
#pragma unroll
        for (int j = 0; j < NS; ++j) o[i][j] *= corr;
      }
      lrow[i] += sum;
      mrow[i] = mn;
#pragma unroll
      for (int t = 0; t < KB / 32; ++t) {
        _Float16 ph[8], pl[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) asplit(p[2 * t + (e >> 2)][e & 3], ph[e], pl[e]);
        pbh[i][t] = au4_t{apack2(ph[0], ph[1]), apack2(ph[2], ph[3]), apack2(ph[4], ph[5]), apack2(ph[6], ph[7])};
        pbl[i][t] = au4_t{apack2(pl[0], pl[1]), apack2(pl[2], pl[3]), apack2(pl[4], pl[5]), apack2(pl[6], pl[7])};
      }
    }
    // O^T += V^T P^T over the block's two 32-key steps; the B operand is the lane's own P
#pragma unroll
    for (int t = 0; t < KB / 32; ++t)
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const au4_t ah = *reinterpret_cast<const au4_t*>(&vsh[16 * j + fr][32 * t + fk]);
        const au4_t al = *reinterpret_cast<const au4_t*>(&vsl[16 * j + fr][32 * t + fk]);
#pragma unroll
        for (int i = 0; i < TMQ; ++i)
          if (live[i]) o[i][j] = mma3(ah, al, pbh[i][t], pbl[i][t], o[i][j]);
        if (TMQ > 1) __builtin_amdgcn_sched_barrier(0);
      }
  }
  if constexpr (KG == 2) {
    static_assert(KG == 1 || (TMQ == 1 && sizeof(Block) >= (size_t)NW * 64 * 4 * (4 * NS + 2)), "hand-over fits a block");
    // [wave][value][lane], in the first set's block
    float* hand = reinterpret_cast<float*>(&blk[0]) + (size_t)wave * 64 * (4 * NS + 2) + lane;
    __syncthreads();
    if (kg == 1) {
      hand[0] = mrow[0];
      hand[64] = lrow[0];
#pragma unroll
      for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) hand[64 * (2 + 4 * j + r)] = o[0][j][r];
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = hand[0], l1 = hand[64];
    const float mn = fmaxf(mrow[0], m1);
    const float w0 = mrow[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mrow[0] - mn);
    const float w1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - mn);
    lrow[0] = lrow[0] * w0 + l1 * w1;
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[0][j][r] = o[0][j][r] * w0 + hand[64 * (2 + 4 * j + r)] * w1;
  }
  if (!active) return;
#pragma unroll
  for (int i = 0; i < TMQ; ++i) {
    const int qi = q0 + 16 * i + fr;
    if (qi < M) {
      // o / l with one reciprocal per query: its rounding error is taken out of each quotient by the
      // remainder (l is a sum of exponentials, 1 or more; a full division per value was ten
      // instructions)
      const float l = lrow[i];
      float rc = __builtin_amdgcn_rcpf(l);
      rc = fmaf(fmaf(-l, rc, 1.f), rc, rc);
      auto quot = [&](float x) {
        const float y = x * rc;
        return fmaf(fmaf(-y, l, x), rc, y);
      };
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const af4_t v = o[i][j];
        *reinterpret_cast<float4*>(out + (size_t)qi * qd + (size_t)hq * HD + 16 * j + 4 * lg) =
            make_float4(quot(v[0]), quot(v[1]), quot(v[2]), quot(v[3]));
      }
    }
  }
}

// Prefill attention on f32 inputs (taken when a q, k or v value is beyond the fp16 pair's range):
// the reference's per-(position, head) loop (src/layers/attention.rs:364-415) with an online
// softmax. One wave per (query row i, head h): keys j in [j_min, i] (j_min = i - (window - 1)
// with a window) in chunks of 64, lane = key for the scores (dot * scale in f32), lane = head
// dims for P V. q and k carry RoPE; k and v rows are [M][n_kv * hd], KV head h / (n_heads / n_kv).
__global__ __launch_bounds__(64) void attn_prefill_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                              const float* __restrict__ v, float* __restrict__ out,
                                                              int M, int n_heads, int n_kv, int hd, int window,
                                                              float scale) {
#pragma clang fp contract(off)
  constexpr int DPL = 8;  // head dims per lane (hd <= 512)
  __shared__ float qs[512];
  __shared__ float ps[64];
  const int i = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int kvh = h / (n_heads / n_kv);
  const size_t qd = (size_t)n_heads * hd, kvd = (size_t)n_kv * hd;
  for (int d = lane; d < hd; d += 64) qs[d] = q[(size_t)i * qd + (size_t)h * hd + d];
  __syncthreads();
  const int j0 = window > 0 ? max(0, i - (window - 1)) : 0;
  float m = -INFINITY, l = 0.f, o[DPL];
#pragma unroll
  for (int t = 0; t < DPL; ++t) o[t] = 0.f;
  for (int jb = j0; jb <= i; jb += 64) {
    const int j = jb + lane;
    float sc = -INFINITY;
    if (j <= i) {
      const float* kr = k + (size_t)j * kvd + (size_t)kvh * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; ++d) dot += qs[d] * kr[d];
      sc = dot * scale;
    }
    const float cm = wave_max(sc);
    const float mn = fmaxf(m, cm);
    const float p = j <= i ? expf(sc - mn) : 0.f;
    const float corr = expf(m - mn);  // 0 on the first chunk (m = -inf)
    l = l * corr + wave_sum(p);
#pragma unroll
    for (int t = 0; t < DPL; ++t) o[t] *= corr;
    m = mn;
    ps[lane] = p;
    __syncthreads();
    const int nj = min(64, i + 1 - jb);
    for (int jj = 0; jj < nj; ++jj) {
      const float pj = ps[jj];
      const float* vr = v + (size_t)(jb + jj) * kvd + (size_t)kvh * hd;
#pragma unroll
      for (int t = 0; t < DPL; ++t) {
        const int d = lane + 64 * t;
        if (d < hd) o[t] += pj * vr[d];
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < DPL; ++t) {
    const int d = lane + 64 * t;
    if (d < hd) out[(size_t)i * qd + (size_t)h * hd + d] = o[t] / l;
  }
}

void launch_attn_prefill_f32(const float* q, const float* k, const float* v, float* out, int M, int n_heads, int n_kv,
                             int head_dim, int window, float scale, hipStream_t st) {
  if (M <= 0) return;
  if (head_dim <= 0 || head_dim > 512 || n_kv <= 0 || n_heads % n_kv != 0)
    fail(ST_OP, "prefill attention (f32): head_dim <= 512 and whole GQA groups");
  hipLaunchKernelGGL(attn_prefill_f32_kernel, dim3(M, n_heads), dim3(64), 0, st, q, k, v, out, M, n_heads, n_kv,
                     head_dim, window, scale);
}

// Scratch halves the shared-K/V path needs: four planes of n_kv * HD * Mp.
size_t attn_prefill_scratch_halves(int M, int n_kv, int head_dim) {
  const size_t Mp = (size_t)((M + 63) / 64) * 64;
  return 4 * (size_t)n_kv * head_dim * Mp;
}

// The split K / V^T planes and attn_prefill_gqa_kernel: head_dim 64, 128 and (through
// kv_split_kernel only) 256.
static bool attn_planes_ok(int M, int n_heads, int n_kv, int head_dim, const void* scratch, size_t scratch_halves) {
  return scratch && M >= 1 && n_kv >= 1 && (head_dim == 64 || head_dim == 128 || head_dim == 256) &&
         n_heads % n_kv == 0 && scratch_halves >= attn_prefill_scratch_halves(M, n_kv, head_dim);
}

bool launch_attn_prefill_prep(float* q, const float* k, const float* v, int M, int n_heads, int n_kv, int head_dim,
                              const float* cs, int npairs, void* kc, void* vc, bool kv_f32, int ctx, int pos0,
                              void* scratch, size_t scratch_halves, int* ovf, hipStream_t st) {
  if (!attn_planes_ok(M, n_heads, n_kv, head_dim, scratch, scratch_halves) || head_dim > 128 || npairs < 0 ||
      2 * npairs > head_dim || !ovf)
    return false;
  if (pos0 < 0 || (size_t)pos0 + (size_t)M > (size_t)ctx) fail(ST_KVCACHE, "attention prep: the prompt does not fit the cache");
  const int Mp = ((M + 63) / 64) * 64;
  const size_t plane = (size_t)n_kv * head_dim * Mp;
  _Float16* s16 = static_cast<_Float16*>(scratch);
  _Float16 *kh = s16, *kl = s16 + plane, *vh = s16 + 2 * plane, *vl = s16 + 3 * plane;
  const dim3 grid(Mp / 64, (head_dim + 63) / 64, n_kv + n_heads);
  if (kv_f32)
    hipLaunchKernelGGL(attn_prep_kernel<float>, grid, dim3(256), 0, st, q, k, v, M, n_heads, n_kv, head_dim, Mp, cs,
                       npairs, (float*)kc, (float*)vc, ctx, pos0, kh, kl, vh, vl, ovf);
  else
    hipLaunchKernelGGL(attn_prep_kernel<__half>, grid, dim3(256), 0, st, q, k, v, M, n_heads, n_kv, head_dim, Mp, cs,
                       npairs, (__half*)kc, (__half*)vc, ctx, pos0, kh, kl, vh, vl, ovf);
  return true;
}

void launch_attn_prefill(const float* q, const float* k, const float* v, float* out, int M, int n_heads, int n_kv,
                         int head_dim, int window, float scale, hipStream_t st, void* scratch, size_t scratch_halves,
                         bool planes_ready, int* ovf) {
  const int G = n_heads / n_kv;
  if (attn_planes_ok(M, n_heads, n_kv, head_dim, scratch, scratch_halves) && G >= 1) {
    const int Mp = ((M + 63) / 64) * 64;
    const size_t plane = (size_t)n_kv * head_dim * Mp;
    _Float16* s16 = static_cast<_Float16*>(scratch);
    _Float16 *kh = s16, *kl = s16 + plane, *vh = s16 + 2 * plane, *vl = s16 + 3 * plane;
    if (!planes_ready)
      hipLaunchKernelGGL(kv_split_kernel, dim3(Mp / 64, (head_dim + 63) / 64, n_kv), dim3(256), 0, st, k, v, M, n_kv,
                         head_dim, Mp, kh, kl, vh, vl, ovf);
    int* qovf = planes_ready ? nullptr : ovf;
    const int G4 = std::min(G, 4), HG = (G + 3) / 4;
    // query tile of NW waves of TMQ 16-query tiles each
    auto tile = [&](int tmq, int nw) { return 16 * tmq * (nw / G4); };
    auto wgs = [&](int qt) { return (size_t)n_kv * HG * ((M + qt - 1) / qt); };
#define IEK_GQA(HD, TMQ, NW, KB, KG)                                                                                \
  hipLaunchKernelGGL((attn_prefill_gqa_kernel<HD, TMQ, NW, KB, KG>),                                                \
                     dim3(n_kv * HG, (M + tile(TMQ, NW) - 1) / tile(TMQ, NW)), dim3(64 * NW * KG), 0, st, q, kh, kl, \
                     vh, vl, out, M, Mp, n_heads, n_kv, window, scale, qovf)
    // eight waves of two query tiles each per staged block once the grid fills the machine twice
    // over (4096 rows of 32 heads: 393 us against 510), four waves of one tile below that (2045
    // rows: 146 against 176; four waves of two tiles 171)
    const bool wide = wgs(tile(2, 8)) >= 2 * (size_t)num_cus();
    if (head_dim == 256) {
      // 32-key blocks (the K and V^T planes of a block take 75 KB). Two sets of four waves while the
      // grid holds at most two workgroups per CU, which is what fits of one set: whole calls at 8
      // heads of one KV head, one set / two, us: 2045 rows (256 workgroups) 215 / 172, 4096 (512) 411 /
      // 331, window 512 121 / 118, 5000 (626) 500 / 514, 6500 (814) 665 / 807, 8192 (1024) 980 / 1139; 32
      // heads of 8, 2045 rows (1024) 288 / 341.
      if (wgs(tile(1, 4)) <= 2 * (size_t)num_cus()) IEK_GQA(256, 1, 4, 32, 2);
      else IEK_GQA(256, 1, 4, 32, 1);
    } else if (head_dim == 128) {
      if (wide) IEK_GQA(128, 2, 8, 64, 1);
      else IEK_GQA(128, 1, 4, 64, 1);
    } else {
      if (wide) IEK_GQA(64, 2, 8, 64, 1);
      else IEK_GQA(64, 1, 4, 64, 1);
    }
#undef IEK_GQA
    return;
  }
  // the kernel below splits q, k and v into fp16 pairs itself
  if (!planes_ready && ovf)
    launch_range_flag3(q, (size_t)M * n_heads * head_dim, k, v, (size_t)M * n_kv * head_dim, ovf, st);
  dim3 grid(n_heads, (M + 63) / 64);
  switch (head_dim) {
#define IEK_AP(HD, KB)                                                                                          \
  hipLaunchKernelGGL((attn_prefill_mfma_kernel<HD, KB>), grid, dim3(256), 0, st, q, k, v, out, M, n_heads, n_kv, \
                     window, scale)
    case 64:
      IEK_AP(64, 64);
      break;
    case 128:
      IEK_AP(128, 64);
      break;
    case 256:
      IEK_AP(256, 32);
      break;
    case 512:
      IEK_AP(512, 32);
      break;
#undef IEK_AP
    default:
      fail(ST_OP, "prefill attention: head_dim must be 64, 128, 256 or 512");
  }
}

}  // namespace iek
