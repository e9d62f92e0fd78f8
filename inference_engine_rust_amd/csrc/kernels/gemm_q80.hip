// Prefill matmul for Q8_0 weights and more rows than the few-row kernel takes: out[m, n] =
// sum_k a[m, k] * W(k, n) with the operands and exact products of gemm_q.hip.
//
// A workgroup owns 64 x 64 outputs and its four waves a quarter of K each, so every wave has a
// 64 x 64 tile: an activation operand serves four MFMAs and a decoded weight operand eight, the
// waves share nothing until the end and no barrier stands in the K loop. The activation planes are
// stored in MFMA operand order, so its operands come straight from L2 (one coalesced 1 KB load
// each). Weights are copied as raw bytes in memory order through a strip of LDS of the wave's own.
//
// Against the tiles it took over from (64 x 64 with both operands staged through LDS as fp16, a wave
// of 16 x 64 reading six LDS operands for eight MFMAs, one barrier per 32 of K), whole op-level calls,
// us: 256 x 6144 x 1536 42.0 -> 29.0; 130 x 4096 x 14336 229 -> 93; 256 x 1536 x 6144 110 -> 50;
// 512 x 14336 x 4096 279 -> 194. With tiles left over the bound is a wave's chain of steps (~0.8 us
// per 32 of K with one wave per SIMD); prefetching the activation two blocks ahead instead of one
// changed nothing (98 / 99 at 130 x 4096 x 14336), so it is not the loads' latency.
#include <algorithm>

#include "kq_core.cuh"
#include "../iek_internal.h"

namespace iek {

namespace {

constexpr int Q80_T = 64;                       // rows and columns per workgroup
constexpr int Q80_U = 4, Q80_UB = 34 * Q80_U;   // a unit: four blocks (128 k) of a weight row
constexpr int Q80_CH = Q80_UB / 8;              // its 8-byte chunks (and those per lane of 64 rows)
static_assert(Q80_CH == 17, "chunk_off divides by 17");

struct __attribute__((packed, aligned(2))) U64A2 {
  uint32_t x, y;
};

__global__ __launch_bounds__(256, 2) void gemm_q80_kernel(GemmQArgs g) {
  constexpr int RED = 4 * 4 * 4 * 64 * 16, STRIP = Q80_T * Q80_UB;
  static_assert(RED >= 4 * STRIP, "the strips fit the hand-over's LDS");
  __shared__ __align__(16) uint8_t smem[RED];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int M = g.M, kb = g.K / 32, mtiles = (M + Q80_T - 1) / Q80_T;
  // workgroup b runs on XCD b % 8: with xcd_remap an XCD takes a contiguous run of tiles, so the row
  // tiles of a weight tile share its L2
  int tile = blockIdx.x;
  if (g.xcd_remap) tile = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  const int mt = tile % mtiles, ntile = tile / mtiles;
  const int s = ntile < g.tile_start[1] ? 0 : (ntile < g.tile_start[2] ? 1 : 2);
  const uint8_t* w = s == 0 ? g.w[0] : (s == 1 ? g.w[1] : g.w[2]);
  const int N = s == 0 ? g.n[0] : (s == 1 ? g.n[1] : g.n[2]);
  const int ts = s == 0 ? 0 : (s == 1 ? g.tile_start[1] : g.tile_start[2]);
  const int m0 = mt * Q80_T, n0 = (ntile - ts) * Q80_T;
  const uint8_t* wend = w + g.row_bytes * (size_t)N;
  const uint8_t* wt = w + g.row_bytes * (size_t)n0;
  uint8_t* strip = smem + wave * STRIP;

  // this wave's units
  const int nu = (kb + Q80_U - 1) / Q80_U, u0 = nu * wave / 4, u1 = nu * (wave + 1) / 4;
  // Chunk i of this lane: row c / CH of the tile's 64 (the last live one past N) for c = 64 i + lane,
  // so a wave load takes consecutive bytes; the strip holds the chunks in the same order. (Worked out
  // anew for each unit: kept, the offsets cost 17 registers.) A row's last, partial unit runs into
  // the next row, but not past the tensor: its last eight bytes are read instead and shifted.
  const int last_row = N - 1 - n0;
  auto chunk_off = [&](int i, int ln) {
    const uint32_t c = 64 * i + ln, row = c * 241 >> 12;  // c / 17 for c < 1088
    return min(row, (uint32_t)last_row) * (uint32_t)g.row_bytes + 8 * (c - Q80_CH * row);
  };
  auto fetch_w = [&](int u, uint2 (&o)[Q80_CH]) {
    const uint8_t* p = wt + (size_t)u * Q80_UB;
    const uint32_t lim = (uint32_t)min((size_t)(wend - 8 - p), (size_t)0x7FFFFFF8);
    int ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int i = 0; i < Q80_CH; ++i) {
      const U64A2 v = *reinterpret_cast<const U64A2*>(p + min(chunk_off(i, ln), lim));
      o[i] = make_uint2(v.x, v.y);
    }
  };
  auto shift_w = [&](int u, uint2 (&o)[Q80_CH]) {  // a partial unit's chunks over the tensor's end
    const uint32_t lim = (uint32_t)min((size_t)(wend - 8 - (wt + (size_t)u * Q80_UB)), (size_t)0x7FFFFFF8);
    int ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int i = 0; i < Q80_CH; ++i) {
      const uint32_t off = chunk_off(i, ln), by = off > lim ? min(off - lim, 7u) : 0u;  // (8 and more: unused bytes)
      const uint64_t v = (((uint64_t)o[i].y << 32) | o[i].x) >> (8 * by);
      o[i] = make_uint2((uint32_t)v, (uint32_t)(v >> 32));
    }
  };
  const qu4_t* xh = reinterpret_cast<const qu4_t*>(g.xh);
  const qu4_t* xl = reinterpret_cast<const qu4_t*>(g.xl);
  const int la = 4 * lr + lg;  // this lane's chunk of a 16 x 32 plane tile
  size_t at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) at[i] = (size_t)min((m0 >> 4) + i, (M - 1) >> 4) * kb * 64;
  auto fetch_a = [&](int i, int k, qu4_t (&o)[2]) {  // row tile i, block k of K
    const size_t off = at[i] + (size_t)min(k, kb - 1) * 64;
    o[0] = (xh + off)[la];
    o[1] = (xl + off)[la];
  };

  const qf4_t zero{0.f, 0.f, 0.f, 0.f};
  qf4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero;
  // Block t (a constant) of the unit in the strip, block k of K. A row tile's operands of the next
  // block go out once its MFMAs have read these; a tile's sums are folded in under the next one's
  // MFMAs.
  auto step = [&](int t, int k, qu4_t (&a)[4][2]) {
    qu4_t b[4];
    float d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint8_t* row = strip + (16 * j + lr) * Q80_UB;
      // bytes 34 t + 2 + 8 lg: dword-aligned for odd t, two past a dword for even t
      const uint32_t* p = reinterpret_cast<const uint32_t*>(row + (34 * t + 2 + 8 * lg - (t & 1 ? 0 : 2)));
      uint32_t x, y;
      if (t & 1) {
        x = p[0], y = p[1];
      } else {
        const uint32_t q0 = p[0], q1 = p[1], q2 = p[2];
        x = __builtin_amdgcn_alignbyte(q1, q0, 2), y = __builtin_amdgcn_alignbyte(q2, q1, 2);
      }
      d[j] = half_bits_to_float(*reinterpret_cast<const uint16_t*>(row + 34 * t));
      x ^= 0x80808080u, y ^= 0x80808080u;
      const uint32_t v[4] = {mag16(x, SEL02), mag16(x, SEL13), mag16(y, SEL02), mag16(y, SEL13)};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        b[j][e] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(qh2_t, v[e]) - qh2_t{1152.0f16, 1152.0f16});
    }
    __builtin_amdgcn_sched_barrier(0);
    qf4_t part[2][4];
    auto fold = [&](int i) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] += d[j] * part[i & 1][j][r];
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) part[i & 1][j] = mfma16(a[i][0], b[j], zero);
#pragma unroll
      for (int j = 0; j < 4; ++j) part[i & 1][j] = mfma16(a[i][1], b[j], part[i & 1][j]);
      fetch_a(i, k + 1, a[i]);
      if (i > 0) fold(i - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    fold(3);
  };

  if (u0 < u1) {
    uint2 wr[Q80_CH];
    qu4_t a[4][2];
    fetch_w(u0, wr);
#pragma unroll
    for (int i = 0; i < 4; ++i) fetch_a(i, Q80_U * u0, a[i]);
    for (int u = u0; u < u1; ++u) {
      if (Q80_U * (u + 1) > kb) shift_w(u, wr);
      // (LDS operations of one wave stay in order)
#pragma unroll
      for (int i = 0; i < Q80_CH; ++i) *reinterpret_cast<uint2*>(strip + 8 * (64 * i + lane)) = wr[i];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int t = 0; t < Q80_U; ++t) {
        if (Q80_U * u + t >= kb) break;  // uniform, in K's last unit only
        if (t == 0) fetch_w(min(u + 1, u1 - 1), wr);
        __builtin_amdgcn_sched_barrier(0);
        step(t, Q80_U * u + t, a);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }

  // wave i finishes row tile i: the others' sums of it through LDS, added in the waves' order
  __syncthreads();
  float4* red = reinterpret_cast<float4*>(smem);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      red[((wave * 4 + i) * 4 + j) * 64 + lane] = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  __syncthreads();
  float* out = s == 0 ? g.out[0] : (s == 1 ? g.out[1] : g.out[2]);
  const float* resid = s == 0 ? g.resid : nullptr;
  const int mb = m0 + 16 * wave + 4 * lg;
  float f[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) f[r] = g.row_scale ? g.row_scale[min(mb + r, M - 1)] : 1.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 p = red[((q * 4 + wave) * 4 + j) * 64 + lane];
      v[0] += p.x, v[1] += p.y, v[2] += p.z, v[3] += p.w;
    }
    const int n = n0 + 16 * j + lr;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mb + r;
      if (m < M && n < N) {
        float x = v[r] * f[r];
        if (resid) x = resid[(size_t)m * N + n] + x;
        out[(size_t)m * N + n] = x;
      }
    }
  }
}

}  // namespace

void launch_gemm_q80(GemmQArgs& g, hipStream_t st) {
  int t = 0;
  for (int i = 0; i < g.nseg; ++i) {
    g.tile_start[i] = t;
    t += (g.n[i] + Q80_T - 1) / Q80_T;
  }
  for (int i = g.nseg; i <= 3; ++i) g.tile_start[i] = t;
  const int tiles = (g.M + Q80_T - 1) / Q80_T * t;
  g.xcd_remap = tiles % 8 == 0;
  hipLaunchKernelGGL(gemm_q80_kernel, dim3(tiles), dim3(256), 0, st, g);
}

}  // namespace iek
