// Device pieces shared by the matrix-core K-quant GEMMs (gemm_q.hip: 64-row tiles for prompts;
// gemm_skinny.hip: few rows): the launch arguments, the exact fp16 weight operands and the SwiGLU
// epilogue.
#pragma once
#include "common.cuh"

namespace iek {

struct GemmQArgs {
  const uint8_t* w[3];
  float* out[3];
  int n[3];
  int tile_start[4];  // first N tile of each segment; tile_start[nseg] = total N tiles
  int nseg;
  int M, K;
  size_t row_bytes;
  const __half* xh;
  const __half* xl;
  const float* xs;
  const float* resid;  // segment 0 only
  int xcd_remap;
  // split-K (wave-tiled kernel, one segment): the second half of the superblocks writes its
  // partial sums to kpart [M, N], which a follow-up pass adds to out
  int ksplit;
  float* kpart;
  // gate/up + SwiGLU (wave-tiled kernel instantiated with GLU, segments 0 = gate and 1 = up of
  // equal N): each wave computes 32 gate and the same 32 up columns; the epilogue writes
  // act = silu(gate) * up as the down projection's input: fp16 (hi, lo) planes, their
  // per-32 sums (glu_sums, optional) and the f32 act (glu_out, optional)
  _Float16 *glu_h, *glu_l, *glu_sums;
  float* glu_out;
  // op level: out[m] *= row_scale[m] (the power-of-two factors of launch_split_scaled), or null
  const float* row_scale;
  // few-row kernel: with ksplit > 1 kpart holds the workgroups' partial sums and sk_cnt their arrival
  // counters, which the kernel leaves zero again
  int* sk_cnt;
  int* ovf;  // GLU: set when an act value or per-32 sum is beyond the fp16 pair's range
};

namespace {

typedef _Float16 qh8_t __attribute__((ext_vector_type(8)));
typedef float qf4_t __attribute__((ext_vector_type(4)));
typedef uint32_t qu4_t __attribute__((ext_vector_type(4)));

typedef _Float16 qh2_t __attribute__((ext_vector_type(2)));

IEK_DEV uint32_t pk_fma16(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(qh2_t, a), __builtin_bit_cast(qh2_t, b),
                                                                __builtin_bit_cast(qh2_t, c)));
}
// (1024 + byte) as fp16 in each half: bytes of x picked by the selector's bytes 0 and 2.
IEK_DEV uint32_t mag16(uint32_t x, uint32_t sel) { return __builtin_amdgcn_perm(0x64646464u, x, sel); }
// weights in plane_pos order: bytes (0, 2) and (1, 3) of a dword
constexpr uint32_t SEL02 = 0x04020400u, SEL13 = 0x04030401u;
constexpr uint32_t H2_M1024 = 0xE400E400u;  // (-1024, -1024)
constexpr uint32_t H2_ONE = 0x3C003C00u;    // (1, 1)

// {sc, sc} and {-1024 sc, -1024 sc} for the 6-bit scale in byte `i` of `scs`.
IEK_DEV void q4k_scale2(uint32_t scs, uint32_t i, uint32_t& s2, uint32_t& c2) {
  s2 = pk_fma16(mag16(scs, 0x04000400u | i | (i << 16)), H2_ONE, H2_M1024);
  c2 = pk_fma16(s2, H2_M1024, 0u);
}

// B operand of sub-block 2P + H (H = 0: low nibbles, 1: high nibbles) for one 16-column tile.
template <int P, int H>
IEK_DEV qu4_t q4k_b(const uint4& hdr, uint2 q) {
  const uint32_t scs = P < 2 ? (hdr.y & 0x3F3F3F3Fu) : ((hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u));
  uint32_t sc, c;
  q4k_scale2(scs, 2 * (P & 1) + H, sc, c);
  const uint32_t x = (q.x >> (4 * H)) & 0x0F0F0F0Fu, y = (q.y >> (4 * H)) & 0x0F0F0F0Fu;
  return qu4_t{pk_fma16(mag16(x, SEL02), sc, c), pk_fma16(mag16(x, SEL13), sc, c), pk_fma16(mag16(y, SEL02), sc, c),
               pk_fma16(mag16(y, SEL13), sc, c)};
}

// The eight 6-bit mins of a superblock as fp16 (k groups 0 and 1; zero for groups 2 and 3).
IEK_DEV qu4_t q4k_mins(const uint4& hdr, bool live) {
  const uint32_t m03 = hdr.z & 0x3F3F3F3Fu;
  const uint32_t m47 = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
  qu4_t r{pk_fma16(mag16(m03, SEL02), H2_ONE, H2_M1024), pk_fma16(mag16(m03, SEL13), H2_ONE, H2_M1024),
          pk_fma16(mag16(m47, SEL02), H2_ONE, H2_M1024), pk_fma16(mag16(m47, SEL13), H2_ONE, H2_M1024)};
  return live ? r : qu4_t{0u, 0u, 0u, 0u};
}

IEK_DEV qf4_t mfma16(qu4_t a, qu4_t b, qf4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(qh8_t, a), __builtin_bit_cast(qh8_t, b), c, 0, 0, 0);
}

// SwiGLU epilogue of a gate/up tile (GLU): column groups 0-1 of a wave are gate columns and 2-3
// the same up columns, so each lane holds matching gate / up sums. act = silu(g) * u with the
// arithmetic of swiglu_split_kernel (src/ops/swiglu.rs:24-36: two-branch stable sigmoid,
// (g * s) * u), then its fp16 (hi, lo) pair and, per 32 columns, the sum in emit_split8's order
// (pairs, pairs of pairs, then the eight quarter sums one after the other from zero), so the down
// projection's input has the bits the separate pass would write.
// (Staging the fp16 pair through LDS for 16-byte stores measured no faster.)
template <int TM, typename AccT>
IEK_DEV void glu_epilogue(const GemmQArgs& g, const AccT& acc, const float (&Dc)[4], bool rescaled, int m0, int wcol,
                          int lane) {
#pragma clang fp contract(off)
  const int lr = lane & 15, lg = lane >> 4;
  const int M = g.M, N = g.n[0];
  const size_t nb = (size_t)N / 32;
  bool big = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 16 * i + 4 * lg + r;
      float vv[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = wcol + 16 * j + lr;
        const float x = rescaled ? acc[i][j][r] * Dc[j] : acc[i][j][r];
        const float u = rescaled ? acc[i][j + 2][r] * Dc[j + 2] : acc[i][j + 2][r];
        float sg;
        if (x >= 0.0f) {
          const float z = expf(-x);
          sg = 1.0f / (1.0f + z);
        } else {
          const float z = expf(x);
          sg = z / (1.0f + z);
        }
        const float v = x * sg * u;
        if (m < M && n < N) {
          const size_t o = 8 * plane_chunk(m, n >> 3, N / 32) + plane_pos(n & 7);
          const _Float16 h = (_Float16)v;
          g.glu_h[o] = h;
          g.glu_l[o] = (_Float16)(v - (float)h);
          if (g.glu_out) g.glu_out[(size_t)m * N + n] = v;
          big |= fabsf(v) > F16_PAIR_MAX;
        }
        vv[j] = v;
      }
      if (g.glu_sums) {
        // (v0 + v1) + (v2 + v3) over each aligned group of four columns, at the group's first lane
        float qs[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float s1 = vv[j] + __shfl_xor(vv[j], 1, 64);
          qs[j] = s1 + __shfl_xor(s1, 2, 64);
        }
        // the wave's 32 columns are one block; its eight quarter sums sit at lanes 0, 4, 8, 12 of
        // the lane's row of 16 (same m) for j = 0, then j = 1
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t) sum += __shfl(qs[j], (lane & ~15) + 4 * t, 64);
        if (lr == 0 && m < M && wcol < N) {
          const int b = wcol / 32;
          const size_t o = (size_t)m * nb + sums_pos(b, (int)nb);
          const _Float16 h = (_Float16)sum;
          g.glu_sums[o] = h;
          g.glu_sums[(size_t)M * nb + o] = (_Float16)(sum - (float)h);
          big |= fabsf(sum) > F16_PAIR_MAX;
        }
      }
    }
  if (big && g.ovf) *g.ovf = 1;
}

}  // namespace

void launch_gemm_skinny(int dt, GemmQArgs& g, bool glu, hipStream_t st);
void launch_gemm_q80(GemmQArgs& g, hipStream_t st);

}  // namespace iek
