// Token-parallel GEMMs for chunks of positions (teacher-forced encode).
//
// Mapping: one lane = one position (token) of the chunk, one wave = up to 64
// positions x R weight rows.  Every (row, position) output is a dependent
// f32 chain that its lane walks in the reference's order; the wave
// dequantises each weight once into LDS and all 64 lanes read it back as a
// broadcast, so the decode cost is shared by the whole chunk and the inner
// loop is one multiply + one add per weight (Q4_K) or one int8 dot4 per four
// weights (Q6_K, Q8_0).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <array>

#include "dtl_blocks.h"
#include "dtl_device.h"
#include "dtl_numerics.h"

namespace dtl {

namespace {

constexpr int kWaves = 4;  // waves per workgroup
constexpr int kGgmlQ4_0 = 2, kGgmlQ4K = 12, kGgmlQ6K = 14, kGgmlQ8_0 = 8;

__device__ __forceinline__ void flag(int* err, int bit) { atomicOr(err, bit); }

__device__ __forceinline__ uint32_t byte_of(const uint32_t w[3], int i) {
  return (w[i >> 2] >> (8 * (i & 3))) & 0xffu;
}

// Q4_K 6-bit scale and min of sub-block j from the 12 packed bytes held as
// three little-endian words (det-quant lib.rs:519-529).
__device__ __forceinline__ void q4k_scale_min_w(const uint32_t s[3], int j, int* sc, int* mn) {
  if (j < 4) {
    *sc = (int)(byte_of(s, j) & 0x3f);
    *mn = (int)(byte_of(s, j + 4) & 0x3f);
  } else {
    *sc = (int)((byte_of(s, j + 4) & 0x0f) | ((byte_of(s, j - 4) >> 6) << 4));
    *mn = (int)((byte_of(s, j + 4) >> 4) | ((byte_of(s, j) >> 6) << 4));
  }
}

__device__ __forceinline__ bool store_epilogue(float v, float* out, size_t o, const float* bias, int r,
                                               int epi) {
  bool ok = finite(v);
  if (epi == EPI_BIAS) v = v + bias[r];
  else if (epi == EPI_RESIDUAL) v = out[o] + v;
  out[o] = v;
  return ok && finite(v);
}

// The value the epilogue adds (bias[r], or the residual out[o]), read
// without a branch so that a kernel can load it ahead, long before its
// store: a load under a branch is waited for at once, and one such wait per
// output put a round trip per output on the kernel's tail.  With EPI_STORE
// the read (of out[o]) goes unused.
__device__ __forceinline__ float epilogue_operand(const float* out, size_t o, const float* bias, int r,
                                                  int epi) {
  return *(epi == EPI_BIAS ? bias + r : out + o);
}

__device__ __forceinline__ bool store_epilogue_pre(float v, float pre, float* out, size_t o, int epi) {
  bool ok = finite(v);
  if (epi == EPI_BIAS) v = v + pre;
  else if (epi == EPI_RESIDUAL) v = pre + v;
  out[o] = v;
  return ok && finite(v);
}

}  // namespace

// ---------------------------------------------------------------------------
// Q4_K: dot_q4_k_q8a (det-quant lib.rs:281-315).  Each lane's chain adds
// weight*activation for every element of the row in ascending order.
// PAIR computes rows of two matrices with the same shape (gate and up) and
// writes silu(gate)*up (det-model lib.rs:2420-2434) in the epilogue.
template <int R, bool PAIR>
__global__ void __launch_bounds__(256) k_q4k_tok(DevMat W0, DevMat W1, const float* __restrict__ af,
                                                 int T, float* out0, float* out1, float* ffo,
                                                 const float* bias, int epi, int* err) {
  constexpr int NM = PAIR ? 2 : 1;
  __shared__ __align__(16) float wl[kWaves][NM * R][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = (blockIdx.x * kWaves + wave) * R;
  const int t = blockIdx.y * 64 + lane;
  const bool tok = t < T;
  const int rows = W0.rows, cols = W0.cols, nsb = W0.nb;
  const float* arow = af + (size_t)(tok ? t : 0) * cols;
  float acc[NM * R];
#pragma unroll
  for (int k = 0; k < NM * R; k++) acc[k] = 0.0f;
  // lane -> four consecutive elements of one sub-block
  const int wi = lane & 31, hh = lane >> 5;
  const int sub = 2 * (wi >> 3) + hh;
  const int e0 = sub * 32 + (wi & 7) * 4;

  for (int sb = 0; sb < nsb; sb++) {
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const DevMat& W = m ? W1 : W0;
#pragma unroll
      for (int r = 0; r < R; r++) {
        int row = row0 + r;
        float4 w4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < rows) {
          size_t blk = (size_t)row * nsb + sb;
          const uint32_t* h = (const uint32_t*)(W.hdr + blk * 16);
          uint32_t h0 = h[0];
          uint32_t s[3] = {h[1], h[2], h[3]};
          float d = f16_to_f32((uint16_t)(h0 & 0xffff));
          float dmin = f16_to_f32((uint16_t)(h0 >> 16));
          int sc, mn;
          q4k_scale_min_w(s, sub, &sc, &mn);
          float dsc = d * (float)sc, dm = dmin * (float)mn;
          uint32_t qw = ((const uint32_t*)((const uint8_t*)W.w + blk * 128))[wi];
          uint32_t q = (qw >> (4 * hh)) & 0x0f0f0f0fu;
          w4.x = dsc * (float)(q & 0xff) - dm;
          w4.y = dsc * (float)((q >> 8) & 0xff) - dm;
          w4.z = dsc * (float)((q >> 16) & 0xff) - dm;
          w4.w = dsc * (float)(q >> 24) - dm;
        }
        *(float4*)&wl[wave][m * R + r][e0] = w4;
      }
    }
    __builtin_amdgcn_wave_barrier();
    // 16 activations per slice held in registers; each row's 16 weights
    // come from LDS as four broadcast 128-bit reads.
#pragma unroll 1
    for (int s = 0; s < 16; s++) {
      float a[16];
      const float4* ap = (const float4*)(arow + sb * 256 + s * 16);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float4 v = ap[i];  // rows past T read row 0 and are never stored
        a[4 * i] = v.x;
        a[4 * i + 1] = v.y;
        a[4 * i + 2] = v.z;
        a[4 * i + 3] = v.w;
      }
#pragma unroll
      for (int k = 0; k < NM * R; k++) {
        const float4* wp = (const float4*)&wl[wave][k][s * 16];
        float c = acc[k];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float4 w = wp[i];
          c += w.x * a[4 * i];
          c += w.y * a[4 * i + 1];
          c += w.z * a[4 * i + 2];
          c += w.w * a[4 * i + 3];
        }
        acc[k] = c;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (!tok) return;
  bool ok = true;
#pragma unroll
  for (int r = 0; r < R; r++) {
    int row = row0 + r;
    if (row >= rows) continue;
    size_t o = (size_t)t * rows + row;
    if (PAIR) {
      float g = acc[r], u = acc[R + r];
      float v = silu_det(g) * u;
      ok &= finite(g) && finite(u) && finite(v);
      if (out0) out0[o] = g;
      if (out1) out1[o] = u;
      ffo[o] = v;
    } else {
      ok &= store_epilogue(acc[r], out0, o, bias, row, epi);
    }
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

// ---------------------------------------------------------------------------
// Q6_K: dot_q6_k_q8k (det-quant lib.rs:353-397).  The eight lane sums
// aux32[l] (l = element index mod 8) are exact integers: with the Q8_K
// activations stored class-major (class l at bytes 32l..32l+31 of each
// 256-block) and W' = scale*q6 split into int8 planes hi = W' >> 6 and
// lo = W' & 63 in the same order, aux32[l] = 64*dot(hi_l, q_l) + dot(lo_l, q_l),
// eight dot4 per plane.  Then sums[l] += (dw*da)*aux32[l] per superblock and
// the final sequential combine 0 + s0 + ... + s7.
template <int R>
__global__ void __launch_bounds__(256) k_q6k_tok(DevMat W, const int8_t* __restrict__ qk,
                                                 const float* __restrict__ dk, int T, float* out,
                                                 const float* bias, int epi, int* err) {
  __shared__ __align__(16) int8_t hl[kWaves][R][2][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = (blockIdx.x * kWaves + wave) * R;
  const int t = blockIdx.y * 64 + lane;
  const bool tok = t < T;
  const int rows = W.rows, cols = W.cols, nsb = W.nb;
  const int8_t* arow = qk + (size_t)(tok ? t : 0) * cols;
  const float* drow = dk + (size_t)(tok ? t : 0) * nsb;
  float sums[R][8];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int l = 0; l < 8; l++) sums[r][l] = 0.0f;
  // lane -> elements e0..e0+3 (same half, part and 16-element scale group)
  const int e0 = lane * 4;
  const int half = e0 >> 7, within = e0 & 127, l0 = within & 31, part = within >> 5;

  for (int sb = 0; sb < nsb; sb++) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      int row = row0 + r;
      uint32_t hiw = 0, low = 0;
      if (row < rows) {
        const uint8_t* body = (const uint8_t*)W.w + ((size_t)row * nsb + sb) * 208;
        uint32_t qlw = *(const uint32_t*)(body + half * 64 + l0 + (part & 1) * 32);
        uint32_t qhw = *(const uint32_t*)(body + 128 + half * 32 + l0);
        int scale = (int)(int8_t)body[192 + (e0 >> 4)];
        uint32_t nib = (part < 2 ? qlw : (qlw >> 4)) & 0x0f0f0f0fu;
        uint32_t two = (qhw >> (2 * part)) & 0x03030303u;
        uint32_t q6 = nib | (two << 4);  // four 6-bit codes
#pragma unroll
        for (int k = 0; k < 4; k++) {
          int v = (int)((q6 >> (8 * k)) & 0xff) - 32;
          int wp = scale * v;           // in [-4064, 4096]
          int hi = wp >> 6, lo = wp & 63;
          hiw |= (uint32_t)(uint8_t)hi << (8 * k);
          low |= (uint32_t)(uint8_t)lo << (8 * k);
        }
      }
      // scatter the four bytes to their class-major positions
#pragma unroll
      for (int k = 0; k < 4; k++) {
        int e = e0 + k;
        int p = (e & 7) * 32 + (e >> 3);
        hl[wave][r][0][p] = (int8_t)(hiw >> (8 * k));
        hl[wave][r][1][p] = (int8_t)(low >> (8 * k));
      }
    }
    __builtin_amdgcn_wave_barrier();
    float da = drow[sb];
    float d[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      int row = row0 + r < rows ? row0 + r : rows - 1;
      d[r] = f16_to_f32(W.d16[(size_t)row * nsb + sb]) * da;
    }
#pragma unroll
    for (int l = 0; l < 8; l++) {
      // the 32 class-l activation quants of this superblock
      const int4* ap = (const int4*)(arow + sb * 256 + l * 32);
      int4 a0 = ap[0];
      int4 a1 = ap[1];
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int4* hp = (const int4*)&hl[wave][r][0][l * 32];
        const int4* lp = (const int4*)&hl[wave][r][1][l * 32];
        int4 h0 = hp[0], h1 = hp[1], q0 = lp[0], q1 = lp[1];
        int dh = 0, dl = 0;
        dh = __builtin_amdgcn_sdot4(h0.x, a0.x, dh, false);
        dh = __builtin_amdgcn_sdot4(h0.y, a0.y, dh, false);
        dh = __builtin_amdgcn_sdot4(h0.z, a0.z, dh, false);
        dh = __builtin_amdgcn_sdot4(h0.w, a0.w, dh, false);
        dh = __builtin_amdgcn_sdot4(h1.x, a1.x, dh, false);
        dh = __builtin_amdgcn_sdot4(h1.y, a1.y, dh, false);
        dh = __builtin_amdgcn_sdot4(h1.z, a1.z, dh, false);
        dh = __builtin_amdgcn_sdot4(h1.w, a1.w, dh, false);
        dl = __builtin_amdgcn_sdot4(q0.x, a0.x, dl, false);
        dl = __builtin_amdgcn_sdot4(q0.y, a0.y, dl, false);
        dl = __builtin_amdgcn_sdot4(q0.z, a0.z, dl, false);
        dl = __builtin_amdgcn_sdot4(q0.w, a0.w, dl, false);
        dl = __builtin_amdgcn_sdot4(q1.x, a1.x, dl, false);
        dl = __builtin_amdgcn_sdot4(q1.y, a1.y, dl, false);
        dl = __builtin_amdgcn_sdot4(q1.z, a1.z, dl, false);
        dl = __builtin_amdgcn_sdot4(q1.w, a1.w, dl, false);
        int aux = dh * 64 + dl;
        sums[r][l] += d[r] * (float)aux;
      }
      // keep the loads of one class from being hoisted over the previous one
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (!tok) return;
  bool ok = true;
#pragma unroll
  for (int r = 0; r < R; r++) {
    int row = row0 + r;
    if (row >= rows) continue;
    float v = 0.0f;
#pragma unroll
    for (int l = 0; l < 8; l++) v += sums[r][l];
    ok &= store_epilogue(v, out, (size_t)t * rows + row, bias, row, epi);
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

// ---------------------------------------------------------------------------
// Q4_K from an exact f32 copy of the weights (Q4kF32Args, the modes in
// dtl_device.h; one matrix, or two concatenated), every output one chain of
// products in element order.  The lanes of a wave are split over positions and rows, and each lane
// holds a PP x RP block of chains: lane = (p = lane % PW, r = lane / PW),
// RW = 64 / PW; the lane's positions are p + PW i (i < PP) and its rows
// r + RW j (j < RP), one chain per (position, row), every chain in
// element order.  A wave covers PW PP positions of RW RP
// rows; a workgroup is WP x WR waves covering PB positions of RB rows and
// stages each 64-element slice of those positions' activations and rows'
// weights in LDS once (double-buffered, the next slice's global loads in
// flight).  Per four elements a lane reads PP activation and RP weight
// float4 for PP RP chains: the blocking divides the LDS bytes per
// multiply-add, which bound the one-chain mapping, by the block's size
// over its perimeter.
template <int PW, int PP, int RP, int WP, int WR, int MODE>
__global__ void __launch_bounds__(64 * WP * WR) k_q4k_f32m(Q4kF32Args p) {
  static_assert(MODE != MODE_PAIR, "gate + up runs on k_q4k_mfp");
  constexpr int NT = 64 * WP * WR;
  constexpr int NM = 1;
  constexpr int RW = 64 / PW;
  constexpr int PWV = PW * PP, RWV = RW * RP;  // positions, rows per wave
  constexpr int PB = WP * PWV;                 // positions per workgroup
  constexpr int RB = WR * RWV;                 // rows per workgroup
  constexpr int NR = PB + NM * RB;             // staged LDS rows per slice
  constexpr int SL = 64, LD = SL + 4;          // elements per slice, padded LDS row
  constexpr int F = NR * SL / 4;               // float4 per slice
  constexpr int PERT = (F + NT - 1) / NT;
  static_assert(PERT >= 1 && PERT <= 8, "staging slots per thread");
  static_assert(2 * NR * LD * 4 <= 64 * 1024, "LDS tile");
  __shared__ __align__(16) float st[2][NR][LD];
  const int cols = p.cols, T = p.T;
  const int rows_total = MODE == MODE_CAT ? p.rows0 + p.rows1 : p.rows0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wr = wave / WP;
  const int pl = lane % PW, rl = lane / PW;
  const int prow = wp * PWV + pl;   // LDS row of position i: prow + PW i
  const int rrow = wr * RWV + rl;   // workgroup row of row j: rrow + RW j
  float acc[NM][PP][RP];
#pragma unroll
  for (int m = 0; m < NM; m++)
#pragma unroll
    for (int i = 0; i < PP; i++)
#pragma unroll
      for (int j = 0; j < RP; j++) acc[m][i][j] = 0.0f;

  // Staging slot k of thread x moves float4 f = x + k NT of the slice: LDS
  // row f / 16 (activations of position f / 16 first, then the weight rows,
  // matrix by matrix), columns 4 (f % 16).  Out-of-range positions and rows
  // read the last valid one; slots past the slice load a valid address and
  // store nothing, so every load is unconditional.
  auto slot_src = [&](int f) -> const float* {
    const int sr = f < F ? f >> 4 : 0, c4 = f & 15;
    if (sr < PB) {
      const int tt = blockIdx.y * PB + sr;
      return p.af + (size_t)(tt < T ? tt : T - 1) * cols + c4 * 4;
    }
    const int wrow = sr - PB;
    int gg = blockIdx.x * RB + wrow;
    gg = gg < rows_total ? gg : rows_total - 1;
    const bool m = MODE == MODE_CAT && gg >= p.rows0;
    return (m ? p.w1 : p.w0) + (size_t)(m ? gg - p.rows0 : gg) * cols + c4 * 4;
  };
  // Up to eight slots as named registers (an indexed array of them is not
  // kept in registers by the compiler across the conditional load/store).
  const int x = threadIdx.x;
#define DTL_SLOT_DECL(n)                                                      \
  const float* s##n = slot_src(x + (n) * NT);                                 \
  const int d##n = ((x + (n) * NT) >> 4) * LD + ((x + (n) * NT) & 15) * 4;    \
  const bool k##n = x + (n) * NT < F;                                         \
  float4 q##n;
  DTL_SLOT_DECL(0) DTL_SLOT_DECL(1) DTL_SLOT_DECL(2) DTL_SLOT_DECL(3)
  DTL_SLOT_DECL(4) DTL_SLOT_DECL(5) DTL_SLOT_DECL(6) DTL_SLOT_DECL(7)
#undef DTL_SLOT_DECL
#define DTL_ISSUE_M(e0)                                                       \
  do {                                                                        \
    q0 = *(const float4*)(s0 + (e0));                                         \
    if (PERT > 1) q1 = *(const float4*)(s1 + (e0));                           \
    if (PERT > 2) q2 = *(const float4*)(s2 + (e0));                           \
    if (PERT > 3) q3 = *(const float4*)(s3 + (e0));                           \
    if (PERT > 4) q4 = *(const float4*)(s4 + (e0));                           \
    if (PERT > 5) q5 = *(const float4*)(s5 + (e0));                           \
    if (PERT > 6) q6 = *(const float4*)(s6 + (e0));                           \
    if (PERT > 7) q7 = *(const float4*)(s7 + (e0));                           \
  } while (0)
#define DTL_COMMIT_M(b)                                                       \
  do {                                                                        \
    float* sb_ = &st[b][0][0];                                                \
    if (k0) *(float4*)(sb_ + d0) = q0;                                        \
    if (PERT > 1 && k1) *(float4*)(sb_ + d1) = q1;                            \
    if (PERT > 2 && k2) *(float4*)(sb_ + d2) = q2;                            \
    if (PERT > 3 && k3) *(float4*)(sb_ + d3) = q3;                            \
    if (PERT > 4 && k4) *(float4*)(sb_ + d4) = q4;                            \
    if (PERT > 5 && k5) *(float4*)(sb_ + d5) = q5;                            \
    if (PERT > 6 && k6) *(float4*)(sb_ + d6) = q6;                            \
    if (PERT > 7 && k7) *(float4*)(sb_ + d7) = q7;                            \
  } while (0)
  DTL_ISSUE_M(0);
  DTL_COMMIT_M(0);
  __syncthreads();
  int buf = 0;
  for (int e0 = 0; e0 < cols; e0 += SL) {
    const bool more = e0 + SL < cols;
    if (more) DTL_ISSUE_M(e0 + SL);
    const float* sb = &st[buf][0][0];
#pragma unroll 4
    for (int e = 0; e < SL; e += 4) {
      float4 a[PP], w[NM][RP];
#pragma unroll
      for (int i = 0; i < PP; i++) a[i] = *(const float4*)(sb + (prow + PW * i) * LD + e);
#pragma unroll
      for (int m = 0; m < NM; m++)
#pragma unroll
        for (int j = 0; j < RP; j++)
          w[m][j] = *(const float4*)(sb + (PB + m * RB + rrow + RW * j) * LD + e);
#pragma unroll
      for (int m = 0; m < NM; m++)
#pragma unroll
        for (int i = 0; i < PP; i++)
#pragma unroll
          for (int j = 0; j < RP; j++) {
            float c = acc[m][i][j];
            c += w[m][j].x * a[i].x;
            c += w[m][j].y * a[i].y;
            c += w[m][j].z * a[i].z;
            c += w[m][j].w * a[i].w;
            acc[m][i][j] = c;
          }
    }
    if (more) DTL_COMMIT_M(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
#undef DTL_ISSUE_M
#undef DTL_COMMIT_M
  bool ok = true;
#pragma unroll
  for (int i = 0; i < PP; i++) {
    const int t = blockIdx.y * PB + prow + PW * i;
    if (t >= T) continue;
#pragma unroll
    for (int j = 0; j < RP; j++) {
      const int g = blockIdx.x * RB + rrow + RW * j;  // row of the concatenation
      if (g >= rows_total) continue;
      const bool m = MODE == MODE_CAT && g >= p.rows0;
      const int local = m ? g - p.rows0 : g;
      const int R = m ? p.rows1 : p.rows0;
      ok &= store_epilogue(acc[0][i][j], m ? p.out1 : p.out0, (size_t)t * R + local,
                           m ? p.bias1 : p.bias0, local, p.epi);
    }
  }
  if (!ok) flag(p.err, ERRBIT_NON_FINITE);
}

// Exact f32 copy of a Q4_K matrix: q4_k_value for every element.
__global__ void k_dequant_q4k(DevMat W, float* out) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t total = (size_t)W.rows * W.cols;
  if (i >= total) return;
  int row = (int)(i / W.cols), c = (int)(i % W.cols);
  int sb = c / 256, idx = c % 256, sub = idx / 32, within = idx % 32;
  size_t blk = (size_t)row * W.nb + sb;
  const uint32_t* h = (const uint32_t*)(W.hdr + blk * 16);
  uint32_t h0 = h[0];
  uint32_t s[3] = {h[1], h[2], h[3]};
  float d = f16_to_f32((uint16_t)(h0 & 0xffff)), dmin = f16_to_f32((uint16_t)(h0 >> 16));
  int sc, mn;
  q4k_scale_min_w(s, sub, &sc, &mn);
  uint8_t byte = ((const uint8_t*)W.w)[blk * 128 + (sub / 2) * 32 + within];
  int q = (sub & 1) ? (byte >> 4) : (byte & 0x0f);
  out[i] = (d * (float)sc) * (float)q - (dmin * (float)mn);
}

void launch_dequant_q4k(const DevMat& W, float* out, hipStream_t s) {
  size_t total = (size_t)W.rows * W.cols;
  launch_kernel(k_dequant_q4k, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, W, out);
}

// ---------------------------------------------------------------------------
// Q6_K on the int8 matrix cores (dot_q6_k_q8k, det-quant lib.rs:353-397).
// Per superblock sb and class c (element index mod 8) the reference's exact
// integer sums aux_c = sum_j W'[8j+c] * qa[8j+c] over the 32 elements of
// the class form a [rows x positions] product with K = 32.  With
// W' = scale*q6 = 64*hi + lo held as two int8 planes, aux_c is
// 64*(hi . qa) + (lo . qa): two v_mfma_i32_16x16x64_i8 (K quarters 2 and 3
// zero), exact in i32.  The f32 part, sums[c] += (dw*da)*aux_c per
// superblock in order and the final 0 + sums[0] + ... + sums[7], runs on the
// VALU as in the reference.  The Q8_K activations are class-major within
// each 256-block, so class c's 32 bytes are contiguous.
//
// One workgroup per 16-row tile x NT tiles of 16 positions.  MFMA
// operand layout (16x16x64 i8): lane l supplies row / position l % 16 and
// K quarter l / 16 (16 bytes); result register i of lane l is row
// 4 (l / 16) + i, position l % 16.
typedef int dtl_v4i __attribute__((ext_vector_type(4)));
typedef float dtl_v4f __attribute__((ext_vector_type(4)));

__global__ void k_q6k_planes(DevMat W, int rows_pad, int8_t* planes) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = W.nb;
  const size_t total = (size_t)rows_pad * nb * 256;
  if (idx >= total) return;
  const int row = (int)(idx / ((size_t)nb * 256));
  const int rem = (int)(idx % ((size_t)nb * 256));
  const int sb = rem >> 8, k = rem & 255;
  const int c = k >> 5, j = k & 31;
  int wp = 0;
  if (row < W.rows) {
    const uint8_t* body = (const uint8_t*)W.w + ((size_t)row * nb + sb) * 208;
    const int e = 8 * j + c;
    wp = q6k_scale(body, e) * q6k_quant(body, e);
  }
  const size_t base = ((((size_t)(row >> 4) * nb + sb) * 8 + c) * 2) * 512 + (row & 15) * 32 + j;
  planes[base] = (int8_t)(wp >> 6);
  planes[base + 512] = (int8_t)(wp & 63);
}

size_t q6k_planes_bytes(const DevMat& W) {
  return (size_t)((W.rows + 15) / 16) * 16 * W.nb * 256 * 2;
}

void launch_q6k_planes(const DevMat& W, int8_t* planes, hipStream_t s) {
  const int rows_pad = (W.rows + 15) / 16 * 16;
  const size_t total = (size_t)rows_pad * W.nb * 256;
  launch_kernel(k_q6k_planes, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, W, rows_pad,
                planes);
}

// K steps in flight per wave in the int8 MFMA GEMMs (slots r0, r1, ...):
// the Q6_K superblock's operands are four times a Q8_0 block pair's.
constexpr int kQ6kRing = 2;

template <int NT>
__global__ void __launch_bounds__(256) k_q6k_mfma(const int8_t* __restrict__ planes,
                                                  const uint16_t* __restrict__ d16, int rows,
                                                  int nb, const int8_t* __restrict__ qk,
                                                  const float* __restrict__ dk, int T, float* out,
                                                  const float* bias, int epi, int* err) {
  // The eight class chains are independent until the final combine: wave w
  // runs classes 2w and 2w+1 of the workgroup's tile.
  __shared__ float part[8][NT][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rt = blockIdx.x;
  const int p0 = blockIdx.y * 16 * NT;
  const int q = lane >> 4, li = lane & 15;
  const int cols = nb * 256;
  const dtl_v4i zero = {0, 0, 0, 0};
  // A operand: row li of the tile, bytes 16 (q & 1) .. of the class run
  // (quarters 2 and 3 read the same bytes and are zeroed).
  const int8_t* abase = planes + (size_t)rt * nb * 8192 + (size_t)(2 * wave) * 1024 + li * 32 +
                        (q & 1) * 16;
  // B operand: position p0 + 16 j + li (clamped to T - 1; not stored).
  const int8_t* bsrc[NT];
  const float* dsrc[NT];
#pragma unroll
  for (int j = 0; j < NT; j++) {
    int pos = p0 + 16 * j + li;
    pos = pos < T ? pos : T - 1;
    bsrc[j] = qk + (size_t)pos * cols + (2 * wave) * 32 + (q & 1) * 16;
    dsrc[j] = dk + (size_t)pos * nb;
  }
  // Rows of this lane's results: 16 rt + 4 q + i.
  const uint16_t* dwsrc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int row = rt * 16 + 4 * q + i;
    row = row < rows ? row : rows - 1;
    dwsrc[i] = d16 + (size_t)row * nb;
  }
  float sums[NT][2][4];
#pragma unroll
  for (int j = 0; j < NT; j++)
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) sums[j][c][i] = 0.0f;
  // Operands of one superblock for this wave's two classes; the next
  // superblock's are in flight while the current one is multiplied.
  struct Ops {
    dtl_v4i a[2][2];
    dtl_v4i b[NT][2];
    uint16_t dw[4];
    float da[NT];
  };
  auto load = [&](Ops& o, int sb) {
    const int8_t* ab = abase + (size_t)sb * 8192;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      o.a[c][0] = *(const dtl_v4i*)(ab + (2 * c) * 512);
      o.a[c][1] = *(const dtl_v4i*)(ab + (2 * c + 1) * 512);
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int c = 0; c < 2; c++) o.b[j][c] = *(const dtl_v4i*)(bsrc[j] + sb * 256 + c * 32);
#pragma unroll
    for (int i = 0; i < 4; i++) o.dw[i] = dwsrc[i][sb];
#pragma unroll
    for (int j = 0; j < NT; j++) o.da[j] = dsrc[j][sb];
  };
  // valid false (a ring slot past the last superblock): every term added is
  // +0.0f, which leaves the sums' bits unchanged (a sum that starts at +0.0f
  // is never -0.0f), so the loop needs no branch around it.
  auto compute = [&](const Ops& o, bool valid) {
    float dd[NT][4];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) dd[j][i] = f16_to_f32(o.dw[i]) * o.da[j];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const dtl_v4i ahi = q < 2 ? o.a[c][0] : zero;
      const dtl_v4i alo = q < 2 ? o.a[c][1] : zero;
#pragma unroll
      for (int j = 0; j < NT; j++) {
        dtl_v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ahi, o.b[j][c], zero, 0, 0, 0);
        acc = acc * 64;
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(alo, o.b[j][c], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float term = dd[j][i] * (float)acc[i];
          sums[j][c][i] += valid ? term : 0.0f;
        }
      }
    }
  };
  // kQ6kRing superblocks in flight.  Every pass refills its slot (the
  // index clamped to the last superblock): with the refill under a branch
  // the compiler waits for every load in flight before the next compute.
  // (Named slots, not an array, and each refill after the last use of the
  // slot: otherwise the loop-carried registers get copies at the back edge,
  // and the copies wait for the loads.)
  auto last = [&](int i) { return i < nb ? i : nb - 1; };
  Ops r0, r1;
  load(r0, last(0));
  load(r1, last(1));
  // the epilogue's operands of this wave's outputs (see the final combine),
  // in flight with the first superblocks
  float pre[NT];
#pragma unroll
  for (int k = 0; k < NT; k++) {
    const int o = wave + 4 * k, j = o >> 2, i = o & 3;
    int pos = p0 + 16 * j + li;
    pos = pos < T ? pos : T - 1;
    int row = rt * 16 + 4 * q + i;
    row = row < rows ? row : rows - 1;
    pre[k] = epilogue_operand(out, (size_t)pos * rows + row, bias, row, epi);
  }
#define DTL_MFMA_STEP(r, i)                                                                \
  compute(r, (i) < nb);                                                                    \
  __builtin_amdgcn_sched_barrier(0);                                                       \
  load(r, last((i) + kQ6kRing));                                                           \
  __builtin_amdgcn_sched_barrier(0)
  for (int s0 = 0; s0 < nb; s0 += kQ6kRing) {
    DTL_MFMA_STEP(r0, s0);
    DTL_MFMA_STEP(r1, s0 + 1);
  }
#undef DTL_MFMA_STEP
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) part[2 * wave + c][j][i][lane] = sums[j][c][i];
  __syncthreads();
  // Final combine 0 + sums[0] + ... + sums[7] in class order; the four
  // waves split the (position tile, register) outputs.
  bool ok = true;
#pragma unroll
  for (int k = 0; k < NT; k++) {
    const int o = wave + 4 * k, j = o >> 2, i = o & 3;
    const int pos = p0 + 16 * j + li;
    const int row = rt * 16 + 4 * q + i;
    if (row < rows && pos < T) {
      float v = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; c++) v += part[c][j][i][lane];
      ok &= store_epilogue_pre(v, pre[k], out, (size_t)pos * rows + row, epi);
    }
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

// ---------------------------------------------------------------------------
// Q8_0 / Q4_0 on the int8 matrix cores: dot_q8_0_q8a / dot_q4_0_q8a
// (det-quant lib.rs:237-279).  Per 32-element block b the reference forms
// the exact integer isum = sum_e qw[e] * qa[e], then c = (dw * da) * isum
// and one f32 chain per (row, position) over the blocks in order.  With K =
// 64 covering blocks 2p and 2p+1, v_mfma_i32_16x16x64_i8 gives block 2p's
// isum when the A operand's K quarters 2 and 3 are zero and block 2p+1's
// when quarters 0 and 1 are: both exact in i32.  The f32 part runs on the
// VALU in the reference's order: four instructions per block and output
// (convert, dw * da, times isum, add), which bound the large launches, the
// matrix cores taking a quarter of their time.  Q4_0 uses the int8 copy of
// its weights (nibble - 8, element order) built at load.
//
// MFMA operand layout (16x16x64 i8): lane l supplies row / position l % 16
// and K quarter l / 16 (16 bytes); result register i of lane l is row
// 4 (l / 16) + i, position l % 16.
//
// A wave owns RW x PW tiles of 16 rows x 16 positions (4 RW PW chains a
// lane), a workgroup WR x WP waves.  Stages of 128 bytes of K (four blocks)
// of the workgroup's rows and positions, with their scales as f32, pass
// through LDS, double-buffered, with two further stages in flight in
// registers; rows are padded to 144 bytes, so sixteen lanes' operand reads
// fall in distinct banks.  Blocks past the row have zero scales (their terms
// are +-0, which change no sum).  V4: a row's block count is a multiple of
// four, so its four scales are one load.  Up to three matrices share a
// launch over concatenated rows; PAIR alternates the rows of gate and up
// (tile row i is matrix i % 2, row i / 2) and writes silu(gate) * up.
//
// Workgroups are numbered row tile first.  Numbered so that the position
// tiles of a row tile run on one XCD, for its L2, the launches took 1 to 2%
// longer (output projection at 512 positions 452 against 442 us).
namespace {
// A weight scale (a finite f16) by the hardware's conversion, exact.
__device__ __forceinline__ float half_to_f32(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
// The matrix and row of row tr of row tile rt (clamped to the last row; false
// past it).
template <bool PAIR, int TR>
__device__ __forceinline__ bool q8_locate(const Q8Mats& M, int rt, int tr, int* mat, int* row) {
  if (PAIR) {
    const int r = rt * (TR / 2) + (tr >> 1);
    *mat = tr & 1;
    *row = r < M.rows[0] ? r : M.rows[0] - 1;
    return r < M.rows[0];
  }
  const int g = rt * TR + tr;
  const int gc = g < M.total_rows ? g : M.total_rows - 1;
  *mat = (gc >= M.row_end[0] ? 1 : 0) + (gc >= M.row_end[1] ? 1 : 0);
  *row = gc - (*mat == 0 ? 0 : (*mat == 1 ? M.row_end[0] : M.row_end[1]));
  return g < M.total_rows;
}
}  // namespace

template <int RW, int PW, int WR, int WP, bool V4, bool PAIR>
__global__ void __launch_bounds__(64 * WR * WP) k_q8_tile(Q8Mats M, const int8_t* __restrict__ qa,
                                                          const float* __restrict__ da, int T, int* err) {
  constexpr int NT = 64 * WR * WP, TR = 16 * RW * WR, TP = 16 * PW * WP;
  constexpr int KB = 128, LD = KB + 16;
  constexpr int NA = (TR * 8 + NT - 1) / NT, NB = (TP * 8 + NT - 1) / NT;  // 16-byte chunks per thread
  static_assert(TR * 8 % NT == 0 && TR + TP <= NT, "staging slots");
  constexpr int D = 2;  // stages of loads in flight per thread (four measured no faster)
  __shared__ __align__(16) int8_t sa[2][TR * LD];
  __shared__ __align__(16) int8_t sb[2][TP * LD];
  __shared__ __align__(16) float ss[2][4][TR + TP];  // the rows' scales, then the positions'
  const int rt = blockIdx.x, pt = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WP, wp = wave % WP;
  const int q = lane >> 4, li = lane & 15;
  const int nb = M.nb, cols = nb * 32;
  auto locate = [&](int tr, int* mat, int* row) -> bool { return q8_locate<PAIR, TR>(M, rt, tr, mat, row); };
  // Staging: chunk f = tid + k NT is byte column 16 (f % 8) of row f / 8.
  const int cc = 16 * (tid & 7);
  const int8_t* asrc[NA];
  const int8_t* bsrc[NB];
#pragma unroll
  for (int k = 0; k < NA; k++) {
    int mat, row;
    (void)locate((tid + k * NT) >> 3, &mat, &row);
    asrc[k] = pick3(M.w, mat) + (size_t)row * cols;
  }
#pragma unroll
  for (int k = 0; k < NB; k++) {
    int p = pt * TP + ((tid + k * NT) >> 3);
    p = p < T ? p : T - 1;
    bsrc[k] = qa + (size_t)p * cols;
  }
  // Scales: thread t < TR moves tile row t's, TR <= t < TR + TP a position's
  // (both loads on every thread, clamped: no load under a branch).
  const bool is_w = tid < TR;
  const uint16_t* wsc;
  {
    int mat, row;
    (void)locate(is_w ? tid : 0, &mat, &row);
    wsc = pick3(M.d16, mat) + (size_t)row * nb;
  }
  int dp = pt * TP + (is_w ? 0 : tid - TR);
  dp = dp < T ? dp : T - 1;
  const float* dsc = da + (size_t)dp * nb;
  struct Regs {
    dtl_v4i a[NA], b[NB];
    uint16_t w[4];
    float d[4];
  };
  auto issue = [&](Regs& r, int s) {
    const int col = s * KB + cc < cols ? s * KB + cc : 0;
#pragma unroll
    for (int k = 0; k < NA; k++) r.a[k] = *(const dtl_v4i*)(asrc[k] + col);
#pragma unroll
    for (int k = 0; k < NB; k++) r.b[k] = *(const dtl_v4i*)(bsrc[k] + col);
    if constexpr (V4) {
      const int b0 = 4 * s < nb ? 4 * s : 0;
      const uint2 u = *(const uint2*)(wsc + b0);
      r.w[0] = (uint16_t)(u.x & 0xffffu);
      r.w[1] = (uint16_t)(u.x >> 16);
      r.w[2] = (uint16_t)(u.y & 0xffffu);
      r.w[3] = (uint16_t)(u.y >> 16);
      const float4 f = *(const float4*)(dsc + b0);
      r.d[0] = f.x;
      r.d[1] = f.y;
      r.d[2] = f.z;
      r.d[3] = f.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int b = 4 * s + k < nb ? 4 * s + k : 0;
        r.w[k] = wsc[b];
        r.d[k] = dsc[b];
      }
    }
  };
  auto commit = [&](const Regs& r, int buf, int s) {
#pragma unroll
    for (int k = 0; k < NA; k++) *(dtl_v4i*)(sa[buf] + ((tid + k * NT) >> 3) * LD + cc) = r.a[k];
#pragma unroll
    for (int k = 0; k < NB; k++)
      if (NB * NT == TP * 8 || tid + k * NT < TP * 8) *(dtl_v4i*)(sb[buf] + ((tid + k * NT) >> 3) * LD + cc) = r.b[k];
    if (TR + TP == NT || tid < TR + TP) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const float v = is_w ? half_to_f32(r.w[k]) : r.d[k];
        ss[buf][k][tid] = 4 * s + k < nb ? v : 0.0f;
      }
    }
  };
  float sums[RW][PW][4];
#pragma unroll
  for (int i = 0; i < RW; i++)
#pragma unroll
    for (int j = 0; j < PW; j++)
#pragma unroll
      for (int c = 0; c < 4; c++) sums[i][j][c] = 0.0f;
  const dtl_v4i zero = {0, 0, 0, 0};
  auto compute = [&](int buf) {
#pragma unroll
    for (int pp = 0; pp < 2; pp++) {
      dtl_v4i a[RW], b[PW];
#pragma unroll
      for (int i = 0; i < RW; i++) a[i] = *(const dtl_v4i*)(sa[buf] + ((wr * RW + i) * 16 + li) * LD + 64 * pp + 16 * q);
#pragma unroll
      for (int j = 0; j < PW; j++) b[j] = *(const dtl_v4i*)(sb[buf] + ((wp * PW + j) * 16 + li) * LD + 64 * pp + 16 * q);
      // the blocks' K quarters of the positions, zeros in the others
      dtl_v4i bm[2][PW];
      float dv[2][PW];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int j = 0; j < PW; j++) {
          bm[h][j] = (q >> 1) == h ? b[j] : zero;
          dv[h][j] = ss[buf][2 * pp + h][TR + (wp * PW + j) * 16 + li];
        }
      // Row tile n % RW of block n / RW: its MFMAs are issued ahead of the
      // arithmetic on the one before, whose latency they cover.  The empty
      // asms keep that order (hoisted, a stage's results needed 430
      // registers).
      dtl_v4i acc[2][PW];
#pragma unroll
      for (int j = 0; j < PW; j++) acc[0][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], bm[0][j], zero, 0, 0, 0);
#pragma unroll
      for (int n = 0; n < 2 * RW; n++) {
        const int h = n / RW, i = n % RW;
        if (n + 1 < 2 * RW) {
          const int h1 = (n + 1) / RW, i1 = (n + 1) % RW;
          asm volatile("" : "+v"(a[i1]));
#pragma unroll
          for (int j = 0; j < PW; j++)
            acc[(n + 1) & 1][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i1], bm[h1][j], zero, 0, 0, 0);
        }
        const float4 dw = *(const float4*)&ss[buf][2 * pp + h][(wr * RW + i) * 16 + 4 * q];
#pragma unroll
        for (int j = 0; j < PW; j++) {
          const dtl_v4i r = acc[n & 1][j];
          sums[i][j][0] += (dw.x * dv[h][j]) * (float)r[0];
          sums[i][j][1] += (dw.y * dv[h][j]) * (float)r[1];
          sums[i][j][2] += (dw.z * dv[h][j]) * (float)r[2];
          sums[i][j][3] += (dw.w * dv[h][j]) * (float)r[3];
        }
#pragma unroll
        for (int j = 0; j < PW; j++)
          asm volatile("" : "+v"(sums[i][j][0]), "+v"(sums[i][j][1]), "+v"(sums[i][j][2]), "+v"(sums[i][j][3]));
      }
    }
  };
  const int ns = (nb + 3) / 4;
  Regs r[D];
#pragma unroll
  for (int u = 0; u < D; u++) {
    issue(r[u], u);
    __builtin_amdgcn_sched_barrier(0);
  }
  // The epilogue's operands (the residual, the bias), in flight with the
  // first stages where the tile leaves registers for them.
  constexpr bool kPre = !PAIR && RW * PW <= 2;
  float pre[kPre ? RW : 1][kPre ? PW : 1][4];
  auto load_pre = [&](int i, int j, float (&p)[4]) {
    int pos = pt * TP + (wp * PW + j) * 16 + li;
    pos = pos < T ? pos : T - 1;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      int mat, row;
      (void)locate((wr * RW + i) * 16 + 4 * q + c, &mat, &row);
      p[c] = epilogue_operand(pick3(M.out, mat), (size_t)pos * pick3(M.rows, mat) + row, pick3(M.bias, mat), row,
                              pick3(M.epi, mat));
    }
  };
  if constexpr (kPre) {
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
      for (int j = 0; j < PW; j++) load_pre(i, j, pre[i][j]);
  }
  commit(r[0], 0, 0);
  issue(r[0], D);
  __syncthreads();
  for (int s0 = 0; s0 < ns; s0 += D) {
#pragma unroll
    for (int u = 0; u < D; u++) {
      if (s0 + u < ns) compute(u & 1);
      commit(r[(u + 1) % D], (u + 1) & 1, s0 + u + 1);
      issue(r[(u + 1) % D], s0 + u + 1 + D);
      __syncthreads();
    }
  }
  bool ok = true;
  const bool any_operand = M.epi[0] != EPI_STORE || M.epi[1] != EPI_STORE || M.epi[2] != EPI_STORE;
#pragma unroll
  for (int i = 0; i < RW; i++)
#pragma unroll
    for (int j = 0; j < PW; j++) {
      const int pos = pt * TP + (wp * PW + j) * 16 + li;
      const int tr = (wr * RW + i) * 16 + 4 * q;
      int mat, row;
      if constexpr (PAIR) {
#pragma unroll
        for (int c = 0; c < 4; c += 2) {
          if (!locate(tr + c, &mat, &row) || pos >= T) continue;
          const float gv = sums[i][j][c], uv = sums[i][j][c + 1];
          const float v = silu_det(gv) * uv;
          ok &= finite(gv) && finite(uv) && finite(v);
          M.out[0][(size_t)pos * M.rows[0] + row] = v;
        }
      } else {
        float p[4];
        if constexpr (kPre) {
#pragma unroll
          for (int c = 0; c < 4; c++) p[c] = pre[i][j][c];
        } else {
          p[0] = p[1] = p[2] = p[3] = 0.0f;
          if (any_operand) load_pre(i, j, p);
        }
        const bool live = locate(tr, &mat, &row) && pos < T;
        const int R = pick3(M.rows, mat), epi = pick3(M.epi, mat);
        if (live && row + 3 < R && ((row | R) & 3) == 0) {
          // four rows of one matrix at a 16-byte aligned place
          float v[4];
#pragma unroll
          for (int c = 0; c < 4; c++) {
            v[c] = sums[i][j][c];
            ok &= finite(v[c]);
            if (epi == EPI_BIAS) v[c] = v[c] + p[c];
            else if (epi == EPI_RESIDUAL) v[c] = p[c] + v[c];
            ok &= finite(v[c]);
          }
          *(float4*)(pick3(M.out, mat) + (size_t)pos * R + row) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++)
            if (locate(tr + c, &mat, &row) && pos < T)
              ok &= store_epilogue_pre(sums[i][j][c], p[c], pick3(M.out, mat),
                                       (size_t)pos * pick3(M.rows, mat) + row, pick3(M.epi, mat));
        }
      }
    }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

// The same blocks for launches of few tiles, where k_q8_tile's waves walk K
// alone on their SIMDs: a workgroup of W waves owns one tile of 16 rows x 16
// positions and splits K.  Per round each wave forms the terms (dw * da) *
// isum of its four blocks, its operands straight from memory, and leaves them
// in LDS; then each of 256 threads adds the round's 4 W terms of its output in
// block order.  Two rounds of loads are in flight; the terms are double
// buffered, so a round has one barrier.
template <int W, bool V4, bool PAIR>
__global__ void __launch_bounds__(64 * W) k_q8_split(Q8Mats M, const int8_t* __restrict__ qa,
                                                     const float* __restrict__ da, int T, int* err) {
  constexpr int BR = 4 * W;  // blocks of a round
  __shared__ __align__(16) float terms[2][BR][256];  // [block][position * 16 + row]
  const int rt = blockIdx.x, pt = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, li = lane & 15;
  const int nb = M.nb, cols = nb * 32;
  auto locate = [&](int tr, int* mat, int* row) -> bool { return q8_locate<PAIR, 16>(M, rt, tr, mat, row); };
  int mat, row;
  (void)locate(li, &mat, &row);
  const int8_t* asrc = pick3(M.w, mat) + (size_t)row * cols;
  const uint16_t* wsc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    (void)locate(4 * q + i, &mat, &row);
    wsc[i] = pick3(M.d16, mat) + (size_t)row * nb;
  }
  int p = pt * 16 + li;
  p = p < T ? p : T - 1;
  const int8_t* bsrc = qa + (size_t)p * cols;
  const float* dsc = da + (size_t)p * nb;
  struct Regs {
    dtl_v4i a[2], b[2];
    uint2 w[4];  // four f16 scales of each row
    dtl_v4f d;
  };
  auto issue = [&](Regs& r, int s) {
    const int b0 = (s * W + wave) * 4;
#pragma unroll
    for (int pp = 0; pp < 2; pp++) {
      int col = b0 * 32 + 64 * pp + 16 * q;
      col = col < cols ? col : 0;
      r.a[pp] = *(const dtl_v4i*)(asrc + col);
      r.b[pp] = *(const dtl_v4i*)(bsrc + col);
    }
    if constexpr (V4) {
      const int b = b0 < nb ? b0 : 0;
#pragma unroll
      for (int i = 0; i < 4; i++) r.w[i] = *(const uint2*)(wsc[i] + b);
      r.d = *(const dtl_v4f*)(dsc + b);
    } else {
      int b[4];
#pragma unroll
      for (int k = 0; k < 4; k++) b[k] = b0 + k < nb ? b0 + k : 0;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        r.w[i].x = (uint32_t)wsc[i][b[0]] | ((uint32_t)wsc[i][b[1]] << 16);
        r.w[i].y = (uint32_t)wsc[i][b[2]] | ((uint32_t)wsc[i][b[3]] << 16);
      }
#pragma unroll
      for (int k = 0; k < 4; k++) r.d[k] = dsc[b[k]];
    }
  };
  const dtl_v4i zero = {0, 0, 0, 0};
  auto form = [&](const Regs& r, int buf, int s) {
    const int b0 = (s * W + wave) * 4;
    dtl_v4i acc[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const dtl_v4i bm = (q >> 1) == (k & 1) ? r.b[k >> 1] : zero;
      acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r.a[k >> 1], bm, zero, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float dv = b0 + k < nb ? r.d[k] : 0.0f;  // past the row: terms of +-0
      dtl_v4f t;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t u = k < 2 ? r.w[i].x : r.w[i].y;
        const float dw = half_to_f32((uint16_t)((k & 1) ? u >> 16 : u & 0xffffu));
        t[i] = (dw * dv) * (float)acc[k][i];
      }
      *(dtl_v4f*)&terms[buf][4 * wave + k][li * 16 + 4 * q] = t;
    }
  };
  const int ns = (nb + BR - 1) / BR;
  Regs r[2];
  issue(r[0], 0);
  __builtin_amdgcn_sched_barrier(0);
  issue(r[1], 1);
  __builtin_amdgcn_sched_barrier(0);
  // the thread's output: row tid % 16, position tid / 16
  const int o = tid & 255;
  const int pos = pt * 16 + (o >> 4);
  const bool live = locate(o & 15, &mat, &row) && pos < T;
  const int R = pick3(M.rows, mat), epi = pick3(M.epi, mat);
  const size_t at = (size_t)(pos < T ? pos : T - 1) * R + row;
  const float pre = PAIR ? 0.0f : epilogue_operand(pick3(M.out, mat), at, pick3(M.bias, mat), row, epi);
  float sum = 0.0f;
  for (int s0 = 0; s0 < ns; s0 += 2) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      if (s0 + u < ns) {
        form(r[u], u, s0 + u);
        issue(r[u], s0 + u + 2);
        __syncthreads();
        float t[BR];
#pragma unroll
        for (int k = 0; k < BR; k++) t[k] = terms[u][k][o];
#pragma unroll
        for (int k = 0; k < BR; k++) sum += t[k];
      }
    }
  }
  if (tid >= 256) return;
  bool ok = true;
  if constexpr (PAIR) {
    const float other = __shfl_xor(sum, 1);
    if (live && !(o & 1)) {
      const float v = silu_det(sum) * other;
      ok = finite(sum) && finite(other) && finite(v);
      M.out[0][at] = v;
    }
  } else if (live) {
    ok = store_epilogue_pre(sum, pre, pick3(M.out, mat), at, epi);
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

// int8 copy of a Q4_0 matrix in element order (nibble - 8; det-quant
// lib.rs:259-279: element i < 16 is the low nibble of byte i, element
// i + 16 its high nibble), the A operand of k_q8_tile.
__global__ void k_q4_0_i8(DevMat W, int8_t* out) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)W.rows * W.cols;
  if (idx >= total) return;
  const size_t blk = idx / 32;
  const int e = (int)(idx % 32);
  const uint8_t b = ((const uint8_t*)W.w)[blk * 16 + (e & 15)];
  out[idx] = (int8_t)((e < 16 ? (b & 15) : (b >> 4)) - 8);
}

void launch_q4_0_i8(const DevMat& W, int8_t* out, hipStream_t s) {
  const size_t total = (size_t)W.rows * W.cols;
  launch_kernel(k_q4_0_i8, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, W, out);
}

// ---------------------------------------------------------------------------
// launchers

namespace {
// Rows per wave: enough waves to cover every SIMD, more rows when the
// matrix is tall so the per-row decode is amortised over fewer LDS refills.
int rows_per_wave(int rows) {
  if (rows >= 8192) return 4;
  if (rows >= 4096) return 2;
  return 1;
}

// Which Q4_K chunk GEMM serves a launch.  The products on the matrix cores
// (k_q4k_mfp) own 16 x 16 (row, position) chains per wave, so a launch of
// wo / ffn_down or wq + wk at 64 positions has 512-576 waves: with other
// chunks' launches in flight (the pipelined encode) they and the gate + up
// pair (2816 waves) run there.  Alone on the chip a launch needs about three
// waves per CU there; below, one chain per lane of k_q4k_f32m, 8 x 8 lanes,
// 2 x 2 waves over 16 positions x 16 rows, fills the chip better.  us per
// launch, k_q4k_f32m against k_q4k_mfp, wo and ffn_down on average / wq + wk
// of the TinyLlama-1.1B shape: 64 positions (512 / 576 waves) 38 against 51 /
// 33 against 33; 96 (768 / 864) 51.7 against 51.6 / 42.2 against 41.9; 128
// 66 against 52 / 50 against 42; 512 229 against 131 / 163 against 98.
constexpr long kMfpWaves = 768;

template <int PW, int PP, int RP, int WP, int WR, int MODE>
void launch_q4k_f32m(const Q4kF32Args& a, int rows_total, hipStream_t s) {
  constexpr int RB = WR * RP * 64 / PW, PB = WP * PW * PP;
  dim3 grid((rows_total + RB - 1) / RB, (a.T + PB - 1) / PB);
  launch_kernel(k_q4k_f32m<PW, PP, RP, WP, WR, MODE>, grid, dim3(64 * WP * WR), 0, s, a);
}

template <int MODE>
void launch_q4k_f32w(const Q4kF32Args& a, bool overlapped, hipStream_t s) {
  const int rows_total = MODE == MODE_CAT ? a.rows0 + a.rows1 : a.rows0;
  const long waves = (long)((rows_total + 15) / 16) * ((a.T + 15) / 16);
  if (MODE == MODE_PAIR || overlapped || waves >= kMfpWaves) return launch_q4k_mfp(a, MODE, s);
  launch_q4k_f32m<8, 1, 1, 2, 2, MODE == MODE_CAT ? MODE_CAT : MODE_SINGLE>(a, rows_total, s);
}

Q4kF32Args q4k_args(const DevMat& W0, const DevMat* W1, const DevAct& A, int T, float* out0,
                    float* out1, float* ffo, const float* bias0, const float* bias1, int epi,
                    int* err) {
  Q4kF32Args a{};
  a.w0 = W0.w32;
  a.w1 = W1 ? W1->w32 : nullptr;
  a.rows0 = W0.rows;
  a.rows1 = W1 ? W1->rows : 0;
  a.cols = W0.cols;
  a.af = A.af;
  a.T = T;
  a.out0 = out0;
  a.out1 = out1;
  a.ffo = ffo;
  a.bias0 = bias0;
  a.bias1 = bias1;
  a.epi = epi;
  a.err = err;
  return a;
}
}  // namespace

namespace {
template <int RW, int PW, int WR, int WP, bool V4, bool PAIR>
void launch_q8_tile(const Q8Mats& M, const DevAct& A, int T, int* err, hipStream_t s) {
  constexpr int TR = 16 * RW * WR, TP = 16 * PW * WP;
  const int rows = PAIR ? 2 * M.rows[0] : M.total_rows;
  const int rt = (rows + TR - 1) / TR, pt = (T + TP - 1) / TP;
  launch_kernel((k_q8_tile<RW, PW, WR, WP, V4, PAIR>), dim3(rt, pt), dim3(64 * WR * WP), 0, s, M, A.qa, A.da, T, err);
}

// Up to 300 tiles of 16 x 16 (512 where a row has 64 blocks or more) the
// kernel that splits K.  us per launch, k_q8_split against k_q8_tile, 896 x
// 896 and 896 x 4864 on average: 8.3 / 8.8 / 8.4 / 11.8 / 21.3 at 16 / 32 /
// 64 / 128 / 256 positions (56 tiles each 16) against 13.7 / 15.1 / 15.0 /
// 15.0 / 14.9; 1152 x 896 5.0 / 6.8 / 9.2 at 16 / 64 / 128 (72) against 6.7 /
// 7.2 / 7.1; 960 x 576 5.8 / 7.7 at 64 / 128 (240, 480) against 7.5 / 7.8;
// gate + up with SwiGLU 3072 x 576 5.5 at 16 (192) against 6.2, 9728 x 896
// 9.8 (608) against 8.5.  Eight waves instead of four were never faster.
//
// Else the largest tile that still gives every CU two workgroups (one for 32 x
// 64): a larger tile reads LDS less often per product, a smaller one spreads
// a short launch.  Up to 16 positions one position tile, 64 rows where that
// fills the chip, else 16.  us per launch, Qwen2.5-0.5B shape, against the
// kernel without LDS staging that these replace (one to four position tiles
// a wave, every operand straight from memory): output projection (151936 x
// 896) 30 / 70 / 126 / 233 / 444 at 9 / 64 / 128 / 256 / 512 positions
// against 595 (one lane per row) / 157 / 291 / 566 / 1111; gate + up with
// SwiGLU 49 at 512 against 2 x 49 + 8; wo and down on average 14 at 9, 19 at
// 512.  Large launches run at about 0.36 of the 424 T multiply-adds/s that
// four VALU instructions per block and output allow.
template <bool V4, bool PAIR>
void launch_q8_tiles(const Q8Mats& M, const DevAct& A, int T, int* err, hipStream_t s) {
  const int rows = PAIR ? 2 * M.rows[0] : M.total_rows;
  auto wgs = [&](int tr, int tp) { return (long)((rows + tr - 1) / tr) * ((T + tp - 1) / tp); };
  if (wgs(16, 16) <= (M.nb >= 64 ? 512 : 300))
    launch_kernel((k_q8_split<4, V4, PAIR>), dim3((rows + 15) / 16, (T + 15) / 16), dim3(256), 0, s, M, A.qa, A.da, T,
                  err);
  else if (T <= 16 && wgs(64, 16) >= 256) launch_q8_tile<1, 1, 4, 1, V4, PAIR>(M, A, T, err, s);
  else if (T <= 16) launch_q8_tile<1, 1, 1, 1, V4, PAIR>(M, A, T, err, s);
  else if (wgs(128, 64) >= 512) launch_q8_tile<4, 2, 2, 2, V4, PAIR>(M, A, T, err, s);
  else if (wgs(64, 64) >= 512) launch_q8_tile<2, 2, 2, 2, V4, PAIR>(M, A, T, err, s);
  else if (T > 32 && wgs(32, 64) >= 256) launch_q8_tile<1, 2, 2, 2, V4, PAIR>(M, A, T, err, s);
  else launch_q8_tile<1, 1, 2, 2, V4, PAIR>(M, A, T, err, s);
}

const int8_t* q8_weights(const DevMat& W) {
  return W.type == kGgmlQ8_0 ? static_cast<const int8_t*>(W.w) : (W.type == kGgmlQ4_0 ? W.i8 : nullptr);
}
}  // namespace

bool q8_mats_fit(const DevMat* const* mats, int nm, bool pair) {
  if (nm < 1 || nm > 3 || (pair && nm != 2)) return false;
  for (int i = 0; i < nm; i++) {
    const DevMat& m = *mats[i];
    if (!q8_weights(m) || m.cols != mats[0]->cols || m.rows <= 0) return false;
    if (pair && m.rows != mats[0]->rows) return false;
  }
  return true;
}

bool launch_q8_mats(const DevMat* const* mats, int nm, bool pair, const DevAct& A, int T, float* const* outs,
                    const float* const* biases, const int* epis, int* err, hipStream_t s) {
  if (T < 1 || !q8_mats_fit(mats, nm, pair)) return false;
  Q8Mats M{};
  int acc = 0;
  for (int i = 0; i < 3; i++) {
    if (i < nm) {
      M.w[i] = q8_weights(*mats[i]);
      M.d16[i] = mats[i]->d16;
      M.rows[i] = mats[i]->rows;
      acc += mats[i]->rows;
      if (!pair) {
        M.out[i] = outs[i];
        M.bias[i] = biases[i];
        M.epi[i] = epis[i];
      }
    }
    M.row_end[i] = acc;
  }
  if (pair) M.out[0] = outs[0];
  M.total_rows = acc;
  M.nb = mats[0]->nb;
  if (M.nb % 4 == 0) {
    if (pair) launch_q8_tiles<true, true>(M, A, T, err, s);
    else launch_q8_tiles<true, false>(M, A, T, err, s);
  } else {
    if (pair) launch_q8_tiles<false, true>(M, A, T, err, s);
    else launch_q8_tiles<false, false>(M, A, T, err, s);
  }
  return true;
}

bool gemm_tok_supported(const DevMat& W) {
  return W.type == kGgmlQ4K || W.type == kGgmlQ6K || W.type == kGgmlQ8_0 ||
         (W.type == kGgmlQ4_0 && W.i8);
}

void launch_gemm_tok(const DevMat& W, const DevAct& A, int T, float* out, const float* bias,
                     int epi, int* err, hipStream_t s) {
  DevMat none{};
  if (W.type == kGgmlQ4K && W.w32) {
    launch_q4k_f32w<MODE_SINGLE>(
        q4k_args(W, nullptr, A, T, out, nullptr, nullptr, bias, nullptr, epi, err), A.overlapped, s);
    return;
  }
  if (W.type == kGgmlQ6K && W.planes) {
    // Matrices of 2048 rows and more: 32 positions per wave share each
    // weight-plane load; shorter ones split positions over waves to fill the
    // chip.  (The TinyLlama encode's 2048-row ffn_down: 98.5 against 99.1 ms
    // per pipelined step with 16 positions per wave, in a same-box A/B.)
    const int rt = (W.rows + 15) / 16;
    if (W.rows >= 2048) {
      launch_kernel(k_q6k_mfma<2>, dim3(rt, (T + 31) / 32), dim3(256), 0, s, W.planes, W.d16,
                    W.rows, W.nb, A.qk, A.dk, T, out, bias, epi, err);
    } else {
      launch_kernel(k_q6k_mfma<1>, dim3(rt, (T + 15) / 16), dim3(256), 0, s, W.planes, W.d16,
                    W.rows, W.nb, A.qk, A.dk, T, out, bias, epi, err);
    }
    return;
  }
  {
    const DevMat* mats[1] = {&W};
    if (launch_q8_mats(mats, 1, false, A, T, &out, &bias, &epi, err, s)) return;
  }
  int R = rows_per_wave(W.rows);
  dim3 grid((W.rows + kWaves * R - 1) / (kWaves * R), (T + 63) / 64);
  dim3 block(kWaves * 64);
  switch (W.type) {
    case kGgmlQ4K:
      if (R == 4)
        launch_kernel((k_q4k_tok<4, false>), grid, block, 0, s, W, none, A.af, T, out, nullptr, nullptr, bias, epi, err);
      else if (R == 2)
        launch_kernel((k_q4k_tok<2, false>), grid, block, 0, s, W, none, A.af, T, out, nullptr, nullptr, bias, epi, err);
      else
        launch_kernel((k_q4k_tok<1, false>), grid, block, 0, s, W, none, A.af, T, out, nullptr, nullptr, bias, epi, err);
      break;
    default:
      if (R == 4)
        launch_kernel((k_q6k_tok<4>), grid, block, 0, s, W, A.qk, A.dk, T, out, bias, epi, err);
      else if (R == 2)
        launch_kernel((k_q6k_tok<2>), grid, block, 0, s, W, A.qk, A.dk, T, out, bias, epi, err);
      else
        launch_kernel((k_q6k_tok<1>), grid, block, 0, s, W, A.qk, A.dk, T, out, bias, epi, err);
      break;
  }
}

void launch_gemm_pair_swiglu_q4k(const DevMat& G, const DevMat& U, const DevAct& A, int T, float* g,
                                 float* u, float* ffo, int* err, hipStream_t s) {
  if (G.w32 && U.w32 && !g && !u) {
    launch_q4k_f32w<MODE_PAIR>(
        q4k_args(G, &U, A, T, nullptr, nullptr, ffo, nullptr, nullptr, EPI_STORE, err), A.overlapped, s);
    return;
  }
  int R = rows_per_wave(2 * G.rows) >= 2 ? 2 : 1;
  dim3 grid((G.rows + kWaves * R - 1) / (kWaves * R), (T + 63) / 64);
  dim3 block(kWaves * 64);
  if (R == 2)
    launch_kernel((k_q4k_tok<2, true>), grid, block, 0, s, G, U, A.af, T, g, u, ffo, nullptr, 0, err);
  else
    launch_kernel((k_q4k_tok<1, true>), grid, block, 0, s, G, U, A.af, T, g, u, ffo, nullptr, 0, err);
}

bool launch_gemm_cat_q4k(const DevMat& W0, const DevMat& W1, const DevAct& A, int T, float* out0,
                         float* out1, const float* bias0, const float* bias1, int epi, int* err,
                         hipStream_t s) {
  if (T <= kQ4kGemvMaxT || W0.type != kGgmlQ4K || W1.type != kGgmlQ4K || !W0.w32 || !W1.w32 ||
      W0.cols != W1.cols)
    return false;
  launch_q4k_f32w<MODE_CAT>(q4k_args(W0, &W1, A, T, out0, out1, nullptr, bias0, bias1, epi, err),
                            A.overlapped, s);
  return true;
}

}  // namespace dtl
