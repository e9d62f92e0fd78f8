// Prefill matmul for few activation rows (short prompts): out[m, n] = sum_k a[m, k] * W(k, n) with
// the operands and exact products of gemm_q.hip (fp16 (hi, lo) activations, integer weights w').
//
// At a few rows the call is bound by streaming the weights, and the 64 x 256 tiles of gemm_q.hip
// leave most of the chip idle (N = 4096 gives them 16 column tiles) behind one barrier per 64 of K.
// Here a workgroup of eight waves owns 64 columns (four waves of 16) and up to 64 rows, two waves
// split its K range, and workgroups split K further until the chip is full (S of them per column
// group; the last to arrive adds the S partial sums in their order). Weights go straight into MFMA
// operand registers, two units of 256 in flight per wave; the activation is staged through LDS, so
// its waits (LDS counter) never wait for a younger weight load, and each workgroup reads it once
// per 64 columns (per 16 columns, straight from L2, the activation's L2 traffic was the bound).
// Up to 8 rows the hi and lo planes share one MFMA (PK: operand rows 0-7 hi, 8-15 lo).
#include <algorithm>
#include <type_traits>

#include "kq_core.cuh"

namespace iek {

namespace {

// 16 bytes at a 2-byte aligned address (the native Q6_K and Q8_0 blocks) of a tensor that ends at
// `end`; bytes past the end read as zero.
struct __attribute__((packed, aligned(2))) U128A2 {
  uint32_t x, y, z, w;
};
IEK_DEV qu4_t ld16_a2(const uint8_t* p, const uint8_t* end) {
  if (p + 16 <= end) {
    const U128A2 v = *reinterpret_cast<const U128A2*>(p);
    return qu4_t{v.x, v.y, v.z, v.w};
  }
  uint32_t h[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) h[i] = p + 2 * i + 2 <= end ? *reinterpret_cast<const uint16_t*>(p + 2 * i) : 0u;
  return qu4_t{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
}
IEK_DEV qu4_t ld16(const uint8_t* p) { return *reinterpret_cast<const qu4_t*>(p); }
IEK_DEV uint2 lds8(const uint8_t* p) { return *reinterpret_cast<const uint2*>(p); }

// Weight formats. A unit is 256 consecutive k of one weight row (eight K steps of 32); the lane of
// k group g (lane >> 4) holds k = 8g .. 8g + 7 of every step, in plane_pos order. A wave copies its
// 16 rows' raw bytes as CH chunks of 16 per row, consecutive lanes taking consecutive bytes, into a
// strip of LDS of its own (rows STRIDE bytes apart, which spreads the banks) and reads them back
// per lane: loaded straight in operand order, 16 neighbouring lanes touch 16 rows and every load
// costs 64 cache lookups (14336 x 4096 at 4 rows: 17 us). `prep` readies a unit's factors, b<S>
// builds step S's operand (lo: the part of w' beyond fp16, Q6_K only). FOLD: the steps between
// folds of the partial sums into the accumulator (by d(S)).
//
// Q4_K: masking leaves each nibble as the fp16 subnormal q * 2^-24; times sc * 2^10 that is the
// exact normal number sc * q * 2^-14 (the matrix cores take subnormal operands too, but then drop
// low bits of the products: 7e-6 of error).
struct SkQ4K {
  static constexpr bool LO = false, MINS = true;
  static constexpr int FOLD = 8, CH = 9, STRIDE = 144;
  struct Raw {
    uint4 h;
    uint2 q[4];
  };
  struct Pre {
    uint32_t sc[2], m[2];
    float d, dm;
  };
  IEK_DEV static qu4_t chunk(const uint8_t* row, int u, int c, int, const uint8_t*) {
    return ld16(row + (size_t)u * Q4K_BYTES + 16 * c);
  }
  IEK_DEV static void read(const uint8_t* l, int lg, int, Raw& o) {
    o.h = *reinterpret_cast<const uint4*>(l);
#pragma unroll
    for (int c = 0; c < 4; ++c) o.q[c] = lds8(l + 16 + 32 * c + 8 * lg);
  }
  IEK_DEV static Pre prep(const Raw& r) {
    return Pre{{r.h.y & 0x3F3F3F3Fu, (r.h.w & 0x0F0F0F0Fu) | ((r.h.y >> 2) & 0x30303030u)},
               {r.h.z & 0x3F3F3F3Fu, ((r.h.w >> 4) & 0x0F0F0F0Fu) | ((r.h.z >> 2) & 0x30303030u)},
               half_bits_to_float(r.h.x) * 16384.f,
               half_bits_to_float(r.h.x >> 16)};
  }
  template <int S>
  IEK_DEV static void b(const Raw& r, const Pre& p, qu4_t& bh, qu4_t&) {
    constexpr int n = 4 * (S & 1), i = S & 3;
    // {sc, sc} * 2^10: (1024 + sc) by a byte permute, less 1024, times 1024
    const qh2_t sc = (__builtin_bit_cast(qh2_t, mag16(p.sc[S >> 2], 0x04000400u | i | (i << 16))) -
                      qh2_t{1024.0f16, 1024.0f16}) *
                     qh2_t{1024.0f16, 1024.0f16};
    const uint2 q = r.q[S >> 1];
    const uint32_t v[4] = {(q.x >> n) & 0x000F000Fu, (q.x >> (8 + n)) & 0x000F000Fu, (q.y >> n) & 0x000F000Fu,
                           (q.y >> (8 + n)) & 0x000F000Fu};
#pragma unroll
    for (int t = 0; t < 4; ++t) bh[t] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(qh2_t, v[t]) * sc);
  }
  template <int S>
  IEK_DEV static float d(const Raw&, const Pre& p) { return p.d; }
  // the eight mins in plane_pos order, like the per-32 sums
  IEK_DEV static qu4_t mins(const Pre& p, bool live) {
    qu4_t r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r[i] = live ? pk_fma16(mag16(p.m[i >> 1], (i & 1) ? SEL13 : SEL02), H2_ONE, H2_M1024) : 0u;
    return r;
  }
  IEK_DEV static float dmin(const Pre& p) { return p.dm; }
};

// Q6_K: per 128-wide half the raw bytes l0 / l1 (low nibbles of quarters 0, 2 / 1, 3) and h (high
// bits), and sc, the lane's four scale bytes (one per quarter). Step S is quarter S & 3 of half
// S >> 2. The scale changes every 16 k, within a step, so it stays in the operand.
struct SkQ6K {
  static constexpr bool LO = true, MINS = false;
  static constexpr int FOLD = 8;
  struct Raw {
    uint2 l0[2], l1[2], h[2];
    uint32_t sc[2], d;
  };
  struct Pre {
    uint32_t scb[2];
    float d;
  };
  IEK_DEV static Pre prep(const Raw& r) {
    return Pre{{r.sc[0] ^ 0x80808080u, r.sc[1] ^ 0x80808080u}, half_bits_to_float(r.d)};
  }
  template <int S>
  IEK_DEV static void b(const Raw& r, const Pre& p, qu4_t& bh, qu4_t& bl) {
    constexpr int hf = S >> 2, qd = S & 3;
    const qh2_t s2 =
        __builtin_bit_cast(qh2_t, mag16(p.scb[hf], 0x04000400u | qd | (qd << 16))) - qh2_t{1152.0f16, 1152.0f16};
    const uint2 l = (qd & 1) ? r.l1[hf] : r.l0[hf], h = r.h[hf];
    const uint32_t qx = ((l.x >> (4 * (qd >> 1))) & 0x0F0F0F0Fu) | (((h.x >> (2 * qd)) << 4) & 0x30303030u);
    const uint32_t qy = ((l.y >> (4 * (qd >> 1))) & 0x0F0F0F0Fu) | (((h.y >> (2 * qd)) << 4) & 0x30303030u);
    const uint32_t v[4] = {mag16(qx, SEL02), mag16(qx, SEL13), mag16(qy, SEL02), mag16(qy, SEL13)};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const qh2_t qm = __builtin_bit_cast(qh2_t, v[t]) - qh2_t{1056.0f16, 1056.0f16};  // q - 32, exact
      const qh2_t hi = qm * s2;
      bh[t] = __builtin_bit_cast(uint32_t, hi);
      bl[t] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(qm, s2, -hi));  // exact remainder
    }
  }
  template <int S>
  IEK_DEV static float d(const Raw&, const Pre& p) { return p.d; }
  IEK_DEV static qu4_t mins(const Pre&, bool) { return qu4_t{0u, 0u, 0u, 0u}; }
  IEK_DEV static float dmin(const Pre&) { return 0.f; }
};
// from the native 210-byte blocks
struct SkQ6KN : SkQ6K {
  static constexpr int CH = 14, STRIDE = 240;
  IEK_DEV static qu4_t chunk(const uint8_t* row, int u, int c, int, const uint8_t* end) {
    return ld16_a2(row + (size_t)u * Q6K_BYTES + 16 * c, end);
  }
  IEK_DEV static void read(const uint8_t* l, int lg, int, Raw& o) {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      o.l0[hf] = lds8(l + 64 * hf + 8 * lg);
      o.l1[hf] = lds8(l + 64 * hf + 32 + 8 * lg);
      o.h[hf] = lds8(l + 128 + 32 * hf + 8 * lg);
      const uint2 s = lds8(l + 192 + 8 * hf);
      o.sc[hf] = __builtin_amdgcn_perm(s.y, s.x, 0x06040200u + 0x01010101u * (uint32_t)(lg >> 1));
    }
    o.d = *reinterpret_cast<const uint16_t*>(l + 208);
  }
};
// from the regrouped rows (DT_Q6K_R: per superblock four 48-byte lane chunks, then the scale
// dwords of every chunk, then d; d's chunk is the 16 bytes of eight superblocks)
struct SkQ6KR : SkQ6K {
  static constexpr int CH = 14, STRIDE = 240;
  IEK_DEV static qu4_t chunk(const uint8_t* row, int u, int c, int nsb, const uint8_t*) {
    const uint8_t* p = row + (size_t)u * 192 + 16 * c;
    if (c == 12) p = row + (size_t)nsb * 192 + 16 * u;
    if (c == 13) p = row + (size_t)nsb * 208 + 16 * (u >> 3);
    return ld16(p);
  }
  IEK_DEV static void read(const uint8_t* l, int lg, int u, Raw& o) {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int ch = 2 * hf + (lg >> 1);
      const uint8_t* b = l + 48 * ch + 8 * (lg & 1);
      o.l0[hf] = lds8(b);
      o.l1[hf] = lds8(b + 16);
      o.h[hf] = lds8(b + 32);
      o.sc[hf] = *reinterpret_cast<const uint32_t*>(l + 192 + 4 * ch);
    }
    o.d = *reinterpret_cast<const uint16_t*>(l + 208 + 2 * (u & 7));
  }
};

// Q8_0, native 34-byte blocks: one block per step; steps past the row's last block (K % 256 != 0)
// hold another row's bytes and count with d = 0.
struct SkQ80 {
  static constexpr bool LO = false, MINS = false;
  static constexpr int FOLD = 1, CH = 17, STRIDE = 272;
  struct Raw {
    uint2 q[8];
    uint32_t d[8];
  };
  struct Pre {};
  IEK_DEV static qu4_t chunk(const uint8_t* row, int u, int c, int, const uint8_t* end) {
    return ld16_a2(row + (size_t)u * (8 * Q8_0_BYTES) + 16 * c, end);
  }
  IEK_DEV static void read(const uint8_t* l, int lg, int, Raw& o) {
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      // bytes 34 s + 2 + 8 lg: dword-aligned for odd s, two past a dword for even s
      const uint32_t* p = reinterpret_cast<const uint32_t*>(l + (34 * s + 2 + 8 * lg - (s & 1 ? 0 : 2)));
      if (s & 1) {
        o.q[s] = make_uint2(p[0], p[1]);
      } else {
        const uint32_t a = p[0], b = p[1], c = p[2];
        o.q[s] = make_uint2(__builtin_amdgcn_alignbyte(b, a, 2), __builtin_amdgcn_alignbyte(c, b, 2));
      }
      o.d[s] = *reinterpret_cast<const uint16_t*>(l + 34 * s);
    }
  }
  IEK_DEV static Pre prep(const Raw&) { return Pre{}; }
  template <int S>
  IEK_DEV static void b(const Raw& r, const Pre&, qu4_t& bh, qu4_t&) {
    const uint32_t x = r.q[S].x ^ 0x80808080u, y = r.q[S].y ^ 0x80808080u;
    const uint32_t v[4] = {mag16(x, SEL02), mag16(x, SEL13), mag16(y, SEL02), mag16(y, SEL13)};
#pragma unroll
    for (int t = 0; t < 4; ++t)
      bh[t] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(qh2_t, v[t]) - qh2_t{1152.0f16, 1152.0f16});
  }
  template <int S>
  IEK_DEV static float d(const Raw& r, const Pre&) { return half_bits_to_float(r.d[S]); }
  IEK_DEV static qu4_t mins(const Pre&, bool) { return qu4_t{0u, 0u, 0u, 0u}; }
  IEK_DEV static float dmin(const Pre&) { return 0.f; }
};

constexpr int CW = 4, KW = 2;     // waves along the columns (16 each) and along K
constexpr int SK_COLS = 16 * CW;  // columns per workgroup (GLU: 32 gate and the same 32 up)

// MT: 16-row tiles (PK: one tile holding at most 8 rows, hi and lo planes). A round is one unit per
// K wave, its activation in one of NB LDS buffers.
template <class F, int MT, bool PK, bool GLU>
__global__ __launch_bounds__(512, 2) void gemm_skinny_kernel(GemmQArgs g) {
  static_assert(!PK || MT == 1, "packed planes are one row tile");
  constexpr int NB = MT == 1 || (MT == 2 && F::STRIDE <= 240) ? 2 : 1;  // LDS buffers (160 KB in all)
  constexpr int NP = PK ? 1 : 2;             // activation operands per row tile and step
  constexpr int AT = 8 * MT * NP;            // 1 KB operand tiles per K wave and round
  constexpr int AU = KW * AT / 8;            // of them staged per wave
  static_assert(KW * AT % 8 == 0, "the eight waves share the staging evenly");
  __shared__ __align__(16) qu4_t As[NB][KW * AT * 64];
  constexpr int WCH = (16 * F::CH + 63) / 64;  // chunks per lane and unit
  __shared__ __align__(16) uint8_t Ws[CW * KW][16 * F::STRIDE];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4, wc = wave & (CW - 1), wk = wave / CW;
  const int M = g.M, K = g.K, kb = K / 32;
  const int nu = (kb + 7) / 8, nfmt = std::is_same<F, SkQ80>::value ? kb : K / QK_K;
  const int S = g.ksplit, ntile = blockIdx.x / S, ks = blockIdx.x % S, m0 = blockIdx.y * 16 * MT;
  const int s = GLU ? 0 : (ntile < g.tile_start[1] ? 0 : (ntile < g.tile_start[2] ? 1 : 2));
  const int N = s == 0 ? g.n[0] : (s == 1 ? g.n[1] : g.n[2]);
  const int ts = s == 0 ? 0 : (s == 1 ? g.tile_start[1] : g.tile_start[2]);
  const int col0 = GLU ? 32 * ntile : (ntile - ts) * SK_COLS;
  const uint8_t* w = GLU ? (wc < 2 ? g.w[0] : g.w[1]) : (s == 0 ? g.w[0] : (s == 1 ? g.w[1] : g.w[2]));
  const uint8_t* wend = w + g.row_bytes * (size_t)N;
  // chunk i of this lane: row (64 i + lane) / CH of the wave's 16, chunk (64 i + lane) % CH
  const uint8_t* wrow[WCH];
  uint8_t* wl = Ws[wave];
  uint32_t wdst[WCH];
  int wch[WCH];
  const int wcol = col0 + 16 * (GLU ? (wc & 1) : wc);
#pragma unroll
  for (int i = 0; i < WCH; ++i) {
    const int c = min(64 * i + lane, 16 * F::CH - 1);  // (spare lanes of the last pass repeat its last chunk)
    wch[i] = c % F::CH;
    wrow[i] = w + (size_t)min(wcol + c / F::CH, N - 1) * g.row_bytes;
    wdst[i] = (uint32_t)((c / F::CH) * F::STRIDE + 16 * wch[i]);
  }

  // this workgroup's units, split over the K waves (the first takes the odd one)
  const int glo = (int)((long long)nu * ks / S), ghi = (int)((long long)nu * (ks + 1) / S);
  const int half = (ghi - glo + 1) / 2;
  const int u0 = wk == 0 ? glo : glo + half, u1 = wk == 0 ? glo + half : ghi;
  const int rounds = half;

  // activation staging: operand tile t of a round is (K wave, unit, step, row tile, plane); its 64
  // chunks are in plane_chunk order in memory (row, k group) and (k group, row) in LDS, the row
  // xor-ed with the k group's, which keeps both sides free of bank conflicts
  const qu4_t* xh = reinterpret_cast<const qu4_t*>(g.xh);
  const qu4_t* xl = reinterpret_cast<const qu4_t*>(g.xl);
  const int sr = lane >> 2, sg = lane & 3, st_pos = sg * 16 + (sr ^ (4 * sg));
  auto load_a = [&](int round, qu4_t (&o)[AU]) {
#pragma unroll
    for (int i = 0; i < AU; ++i) {
      const int t = wave + 8 * i;
      const int pl = t % NP, rt = (t / NP) % MT, step = (t / (NP * MT)) & 7, kw = t / AT;
      const int un = min((kw == 0 ? glo : glo + half) + round, nu - 1);
      const int kst = min(8 * un + step, kb - 1), rtile = min((m0 >> 4) + rt, (M - 1) >> 4);
      const size_t base = ((size_t)rtile * kb + kst) * 64;
      if constexpr (PK) o[i] = lane < 32 ? xh[base + lane] : xl[base + (lane - 32)];
      else o[i] = (pl == 0 ? xh : xl)[base + lane];
    }
  };
  auto store_a = [&](int buf, const qu4_t (&o)[AU]) {
#pragma unroll
    for (int i = 0; i < AU; ++i) As[buf][(wave + 8 * i) * 64 + st_pos] = o[i];
  };

  // per-32 sums (Q4_K's min term): k group 0 reads the hi plane, 1 the lo plane (PK: group 0 only,
  // by the row's plane)
  const _Float16* sp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = min(m0 + 16 * i + (PK ? (lr & 7) : lr), M - 1);
    sp[i] = reinterpret_cast<const _Float16*>(g.xs) + (size_t)(m + ((PK ? lr >= 8 : (lg & 1)) ? M : 0)) * kb;
  }
  struct Unit {
    qu4_t w[WCH];
    qu4_t xs[MT];
  };
  auto fetch = [&](int u, Unit& o) {
#pragma unroll
    for (int i = 0; i < WCH; ++i) o.w[i] = F::chunk(wrow[i], u, wch[i], nfmt, wend);
    if constexpr (F::MINS) {
#pragma unroll
      for (int i = 0; i < MT; ++i) o.xs[i] = *reinterpret_cast<const qu4_t*>(sp[i] + 8 * u);
    }
  };

  const qf4_t zero{0.f, 0.f, 0.f, 0.f};
  qf4_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = zero;
  const int rd_pos = lg * 16 + (lr ^ (4 * lg));
  auto compute = [&](int u, const Unit& o, const qu4_t* a) {  // a: the unit's operand tiles
    qf4_t part[MT];
    // through the wave's own strip (LDS operations of one wave stay in order)
#pragma unroll
    for (int i = 0; i < WCH; ++i) *reinterpret_cast<qu4_t*>(wl + wdst[i]) = o.w[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    typename F::Raw raw;
    F::read(wl + lr * F::STRIDE, lg, u, raw);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if constexpr (std::is_same<F, SkQ80>::value) {
#pragma unroll
      for (int t = 0; t < 8; ++t)
        if (8 * u + t >= kb) raw.d[t] = 0u;
    }
    const typename F::Pre pre = F::prep(raw);
    auto step = [&](auto T) {
      constexpr int t = decltype(T)::value;
      qu4_t bh, bl;
      F::template b<t>(raw, pre, bh, bl);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const qu4_t a0 = a[((t * MT + i) * NP) * 64 + rd_pos];
        part[i] = mfma16(a0, bh, t % F::FOLD == 0 ? zero : part[i]);
        if constexpr (NP == 2) part[i] = mfma16(a[((t * MT + i) * NP + 1) * 64 + rd_pos], bh, part[i]);
        if constexpr (F::LO) part[i] = mfma16(a0, bl, part[i]);
      }
      if constexpr ((t + 1) % F::FOLD == 0) {
        const float d = F::template d<t>(raw, pre);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][r] += d * part[i][r];
      }
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
    step(std::integral_constant<int, 4>{});
    step(std::integral_constant<int, 5>{});
    step(std::integral_constant<int, 6>{});
    step(std::integral_constant<int, 7>{});
    if constexpr (F::MINS) {
      const float dm = F::dmin(pre);
      const qu4_t mb = F::mins(pre, PK ? lg == 0 : lg < 2);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const qf4_t mp = mfma16(o.xs[i], mb, zero);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] -= dm * mp[r];
      }
    }
  };

  // Weight ring of two units; a slot is refilled two rounds on right after its use. Fetches past the
  // range re-read its last unit (a K wave without units the workgroup's last).
  const int ul = max(min(u1, nu) - 1, 0);
  Unit ring[2];
  qu4_t ar[AU];
  load_a(0, ar);
  fetch(min(u0, ul), ring[0]);
  fetch(min(u0 + 1, ul), ring[1]);
  store_a(0, ar);
  __syncthreads();
  for (int q0 = 0; q0 < rounds; q0 += 2) {
#pragma unroll
    for (int qi = 0; qi < 2; ++qi) {
      const int q = q0 + qi;
      if (q >= rounds) break;
      load_a(q + 1, ar);
      __builtin_amdgcn_sched_barrier(0);
      if (u0 + q < u1) compute(u0 + q, ring[qi], &As[qi % NB][wk * AT * 64]);
      __builtin_amdgcn_sched_barrier(0);
      fetch(min(u0 + q + 2, ul), ring[qi]);
      __builtin_amdgcn_sched_barrier(0);
      if (NB == 1) __syncthreads();
      store_a((qi ^ 1) % NB, ar);
      __syncthreads();
    }
  }

  // sums: the second K wave's through LDS, then the other workgroups' through g.kpart
  float4* red = reinterpret_cast<float4*>(&As[0][0]);
  if (wk == 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
      red[(wc * MT + i) * 64 + lane] = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
  }
  __syncthreads();
  if (wk == 0) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const float4 v = red[(wc * MT + i) * 64 + lane];
      acc[i][0] += v.x;
      acc[i][1] += v.y;
      acc[i][2] += v.z;
      acc[i][3] += v.w;
    }
  }
  if (S > 1) {
    const int grp = blockIdx.y * (gridDim.x / S) + ntile;
    float* part = g.kpart + ((size_t)grp * S * CW * MT + (size_t)wc * MT) * 256;
    if (wk == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        float* p = part + ((size_t)ks * CW * MT + i) * 256 + 4 * lane;
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          const float2 f2 = make_float2(acc[i][r], acc[i][r + 1]);
          __hip_atomic_store(reinterpret_cast<unsigned long long*>(p + r), __builtin_bit_cast(unsigned long long, f2),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // the coherent stores are done before the arrival
    __syncthreads();
    if (tid == 0) {
      const int old = __hip_atomic_fetch_add(&g.sk_cnt[grp], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = old == S - 1;
      if (s_last) __hip_atomic_store(&g.sk_cnt[grp], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    // row tile i by K wave i % KW; the loads go out in batches (one after the other they cost a
    // memory round trip each)
    constexpr int BT = MT == 1 ? 8 : 4;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (i % KW != wk) continue;
      acc[i] = zero;
      for (int q0 = 0; q0 < S; q0 += BT) {
        float4 v[BT];
#pragma unroll
        for (int q = 0; q < BT; ++q)
          v[q] = ld_coh4(reinterpret_cast<const float4*>(part + ((size_t)min(q0 + q, S - 1) * CW * MT + i) * 256) + lane);
#pragma unroll
        for (int q = 0; q < BT; ++q) {
          if (q0 + q >= S) break;
          acc[i][0] += v[q].x;
          acc[i][1] += v[q].y;
          acc[i][2] += v[q].z;
          acc[i][3] += v[q].w;
        }
      }
    }
  }
  // the K wave that holds row tile i's total
  const bool spread = S > 1;
  auto mine = [&](int i) { return wk == (spread ? i % KW : 0); };
  if constexpr (PK) {  // rows 0-7: the hi plane's sums plus the lo plane's, 32 lanes on
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[0][r] += __shfl_xor(acc[0][r], 32, 64);
  }
  if constexpr (GLU) {
    if (!spread) __syncthreads();  // (with a K split the arrival's barriers are past red's readers)
#pragma unroll
    for (int i = 0; i < MT; ++i)
      if (mine(i)) red[(wc * MT + i) * 64 + lane] = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
    __syncthreads();
    if (wave >= MT) return;
    qf4_t v[1][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float4 t = red[(c * MT + wave) * 64 + lane];
      v[0][c] = qf4_t{t.x, t.y, t.z, t.w};
    }
    const float one[4] = {1.f, 1.f, 1.f, 1.f};
    glu_epilogue<1>(g, v, one, false, m0 + 16 * wave, col0, lane);
  } else {
    float* out = s == 0 ? g.out[0] : (s == 1 ? g.out[1] : g.out[2]);
    const float* resid = s == 0 ? g.resid : nullptr;
    const int n = col0 + 16 * wc + lr;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * i + 4 * lg + r;
        if (mine(i) && m < M && n < N) {
          float x = acc[i][r];
          if (g.row_scale) x *= g.row_scale[m];
          if (resid) x = resid[(size_t)m * N + n] + x;
          out[(size_t)m * N + n] = x;
        }
      }
  }
}

// Workgroups that share a column group's K, for t column groups: split until one workgroup per CU
// and row block, while each still has two units (two per CU measured slower: 14336 x 4096 Q4_K at 4
// rows 16.1 against 13.9 us). So a split has at most 256 column groups and K parts, and with at most
// four row blocks (SK_MAX_ROWS) at most SK_MAX_GROUPS counters. It does not depend on the rows: a row's
// sums keep their order from 9 rows on (up to 8, the packed planes add the lo products at the end).
int k_split(int t, int K) { return std::max(1, std::min(std::min(num_cus(), 256) / t, (K / 32 + 7) / 8 / 2)); }

template <class F, int MT, bool PK, bool GLU>
void skinny_launch(GemmQArgs& g, hipStream_t st) {
  int t = 0;
  for (int i = 0; i < g.nseg; ++i) {
    g.tile_start[i] = t;
    t += (g.n[i] + SK_COLS - 1) / SK_COLS;
  }
  if (GLU) t = g.n[0] / 32;
  for (int i = GLU ? 1 : g.nseg; i <= 3; ++i) g.tile_start[i] = t;
  const int mt = (g.M + 16 * MT - 1) / (16 * MT);
  g.ksplit = g.sk_cnt && g.kpart ? k_split(t, g.K) : 1;
  hipLaunchKernelGGL((gemm_skinny_kernel<F, MT, PK, GLU>), dim3(t * g.ksplit, mt), dim3(512), 0, st, g);
}

template <class F, bool GLU>
void skinny_rows(GemmQArgs& g, hipStream_t st) {
  if (g.M <= 8) skinny_launch<F, 1, true, GLU>(g, st);
  else if (g.M <= 16) skinny_launch<F, 1, false, GLU>(g, st);
  else if (g.M <= 32) skinny_launch<F, 2, false, GLU>(g, st);
  else if constexpr (F::STRIDE <= 240) skinny_launch<F, 4, false, GLU>(g, st);
  else skinny_launch<F, 2, false, GLU>(g, st);
}

template <class F>
void skinny(GemmQArgs& g, bool glu, hipStream_t st) {
  if constexpr (!std::is_same<F, SkQ80>::value) {
    if (glu) {
      skinny_rows<F, true>(g, st);
      return;
    }
  }
  skinny_rows<F, false>(g, st);
}

}  // namespace

// Few rows: every output column of up to 64 rows costs this kernel one pass over the weights, where
// the 64 x 256 tiles of gemm_q.hip cost the same for 64 rows as for one until they fill the chip.
// Whole op-level calls, us, this kernel / the tiles with their split-K and row-scale passes, N x K:
//   Q4_K 4096 x 4096    23 rows 26 / 50   64 30 / 52   65 46 / 52   128 50 / 55   129  66 / 54   256  89 / 59
//        6144 x 4096                      64 38 / 52   65 62 / 52
//        14336 x 4096   23 rows 33 / 53   33 51 / 53   64 55 / 55   128 99 / 63
//        6144 x 1536                      64 27 / 31   65 41 / 32
//        1024 x 4096                                                128 28 / 51   129  36 / 51   256  43 / 54
//        4096 x 14336                                               128 102 / 149 192 144 / 149  256 187 / 155
//   Q6_K 4096 x 14336   23 rows 42 / 265  64 60 / 271  128 105 / 273  256 198 / 275
//        14336 x 4096                     64 57 / 106  65 98 / 107  128 102 / 112  200 191 / 180
//        6144 x 1536                      64 28 / 49   128 46 / 52  129  62 / 51   256  66 / 56
// So this kernel takes any width up to 32 rows (Q6_K, whose tiles take three MFMAs per product, up to
// 64), and further rows while columns times row blocks stay where it costs less. The lines are on the
// safe side of where the two cross, not on it: narrow Q4_K at 129 to 256 rows, Q4_K of large K and wide
// Q6_K above 64 rows stay with the tiles although this kernel is faster there.
// Q8_0 above 32 rows takes two or more passes of 32 here, and gemm_q80.hip's tiles are as fast once they
// are enough of them (this kernel / those): 64 rows 4096 x 14336 65 / 92, 1536 x 6144 34 / 45, 6144 x
// 1536 31 / 24, 14336 x 4096 62 / 43; 128 rows 512 x 4096 25 / 38, 1536 x 6144 51 / 49, 1536 x 2048
// 28 / 26, 6144 x 1536 41 / 34, 4096 x 14336 113 / 93.
bool gemm_skinny_ok(int dt, int M, int N) {
  const long long c = (long long)N * ((M + 63) / 64);
  switch (dt) {
    case DT_Q4K: return M <= 32 || (M <= 128 && c <= 8192);
    case DT_Q6K:
    case DT_Q6K_R: return M <= 64 || (M <= SK_MAX_ROWS && c <= 16384);
    case DT_Q8_0: return M <= 32 || (M <= 128 && (long long)N * ((M + 31) / 32) <= (M <= 64 ? 8192 : 5120));
    default: return false;
  }
}

bool gemm_skinny_splits(int K, int N) { return k_split((N + SK_COLS - 1) / SK_COLS, K) > 1; }

void launch_gemm_skinny(int dt, GemmQArgs& g, bool glu, hipStream_t st) {
  switch (dt) {
    case DT_Q4K: skinny<SkQ4K>(g, glu, st); break;
    case DT_Q6K: skinny<SkQ6KN>(g, glu, st); break;
    case DT_Q6K_R: skinny<SkQ6KR>(g, glu, st); break;
    default: skinny<SkQ80>(g, glu, st); break;
  }
}

}  // namespace iek
