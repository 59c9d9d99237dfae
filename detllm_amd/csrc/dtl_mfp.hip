// Q4_K chunk GEMMs (teacher-forced encode) with the products formed on the
// matrix cores and the chains' adds on the VALU: the rows x positions of
// k_q4k_f32m (dtl_gemm.hip), value for value, at one VALU instruction per
// multiply-add instead of two.  Built with the VGPR form of the MFMA
// results (-mllvm -amdgpu-mfma-vgpr-form): the VALU adds read them
// directly, where results in accumulation registers would need a copy
// (v_accvgpr_read) per product.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dtl_device.h"
#include "dtl_numerics.h"

namespace dtl {

namespace {

__device__ __forceinline__ void flag(int* err, int bit) { atomicOr(err, bit); }

__device__ __forceinline__ bool store_epilogue(float v, float* out, size_t o, const float* bias, int r,
                                               int epi) {
  bool ok = finite(v);
  if (epi == EPI_BIAS) v = v + bias[r];
  else if (epi == EPI_RESIDUAL) v = out[o] + v;
  out[o] = v;
  return ok && finite(v);
}

}  // namespace

// The same chains with the products formed on the matrix cores.  An f32
// MFMA with one element of K and a zero accumulator is an outer product:
// v_mfma_f32_16x16x1f32 forms, in four blocks, D_b[i][j] = A_b[i] B_b[j]
// + 0, each rounded once, which is the rounded product w a (bit for bit,
// denormals included; a product of -0 comes out +0, which no chain that
// starts at +0.0 can tell apart, as x + -0 = x + +0 for every x but -0,
// and a sum of products from +0.0 is never -0).  The VALU then does only
// the chains' adds, one instruction per multiply-add instead of two.
//   wave tile  16 rows x 16 positions, 4 chains per lane: lane l holds rows
//              4 (l / 16) + c (c < 4) at position l % 16 (the D layout:
//              lane j + 16 (i / 4), register 4 b + i % 4)
//   16 elements per four MFMAs: MFMA m's block b takes element k0 + 4 b + m,
//              so a lane's A operands over the four are one float4 of its
//              row at k0 + 4 (l / 16) (A_b[i] comes from lane i + 16 b), and
//              its B operands one float4 of its position there; register
//              4 b + c of MFMA m is chain c's product at k0 + 4 b + m, and
//              the adds run b-major, then m: element order
//   pair       the wave's 16 tile rows alternate gate and up rows (tile row
//              i is matrix i % 2, row i / 2), so each lane holds a gate and
//              an up chain of two rows for the SwiGLU epilogue
// A workgroup of WP x WR waves stages 16 WP positions and 16 WR tile rows
// per 64-element slice in LDS, double-buffered as in k_q4k_f32m.
typedef float dtl_v4f __attribute__((ext_vector_type(4)));
typedef float dtl_v16f __attribute__((ext_vector_type(16)));

template <int WP, int WR, int MODE>
__global__ void __launch_bounds__(64 * WP * WR) k_q4k_mfp(Q4kF32Args p) {
  constexpr int NT = 64 * WP * WR;
  constexpr int PB = WP * 16;        // positions per workgroup
  constexpr int TR = WR * 16;        // tile rows per workgroup
  constexpr int NR = PB + TR;        // staged LDS rows per slice
  constexpr int SL = 64, LD = SL + 4;
  constexpr int F = NR * SL / 4;
  constexpr int PERT = (F + NT - 1) / NT;
  static_assert(PERT >= 1 && PERT <= 8, "staging slots per thread");
  static_assert(2 * NR * LD * 4 <= 64 * 1024, "LDS tile");
  __shared__ __align__(16) float st[2][NR][LD];
  const int cols = p.cols, T = p.T;
  const int rows_total = MODE == MODE_CAT ? p.rows0 + p.rows1 : p.rows0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wr = wave / WP;
  const int l16 = lane & 15, q = lane >> 4;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};

  // Staging slot k of thread x moves float4 f = x + k NT of the slice: LDS
  // row f / 16 (the positions, then the tile rows), columns 4 (f % 16);
  // clamped sources and unconditional loads as in k_q4k_f32m.
  auto slot_src = [&](int f) -> const float* {
    const int sr = f < F ? f >> 4 : 0, c4 = f & 15;
    if (sr < PB) {
      const int tt = blockIdx.y * PB + sr;
      return p.af + (size_t)(tt < T ? tt : T - 1) * cols + c4 * 4;
    }
    const int tr = sr - PB;
    if (MODE == MODE_PAIR) {
      const int rr = blockIdx.x * (TR / 2) + (tr >> 1);
      return ((tr & 1) ? p.w1 : p.w0) + (size_t)(rr < p.rows0 ? rr : p.rows0 - 1) * cols + c4 * 4;
    }
    int gg = blockIdx.x * TR + tr;
    gg = gg < rows_total ? gg : rows_total - 1;
    const bool m = MODE == MODE_CAT && gg >= p.rows0;
    return (m ? p.w1 : p.w0) + (size_t)(m ? gg - p.rows0 : gg) * cols + c4 * 4;
  };
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
  dtl_v16f zero;
#pragma unroll
  for (int i = 0; i < 16; i++) zero[i] = 0.0f;
  const int boff = (wp * 16 + l16) * LD + 4 * q;       // this lane's position
  const int aoff = (PB + wr * 16 + l16) * LD + 4 * q;  // this lane's tile row
  int buf = 0;
  for (int e0 = 0; e0 < cols; e0 += SL) {
    const bool more = e0 + SL < cols;
    if (more) DTL_ISSUE_M(e0 + SL);
    const float* sb = &st[buf][0][0];
    dtl_v4f a4 = *(const dtl_v4f*)(sb + boff);
    dtl_v4f w4 = *(const dtl_v4f*)(sb + aoff);
#pragma unroll
    for (int g = 0; g < SL; g += 16) {
      dtl_v16f d[4];
#pragma unroll
      for (int m = 0; m < 4; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(w4[m], a4[m], zero, 0, 0, 0);
      // the next group's operands read while these products are added
      if (g + 16 < SL) {
        a4 = *(const dtl_v4f*)(sb + boff + g + 16);
        w4 = *(const dtl_v4f*)(sb + aoff + g + 16);
      }
      // the four MFMAs issue back to back, ahead of the adds: an add placed
      // right after the MFMA it reads waits out that MFMA's latency
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
          for (int c = 0; c < 4; c++) acc[c] += d[m][4 * b + c];
      // The next group's MFMAs take operands that pass through this empty
      // asm with the sums, so they follow these adds: one group's 64
      // results are live at a time (hoisted, the sixteen MFMAs of a slice
      // needed 256 registers).
      asm volatile("" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(a4), "+v"(w4));
    }
    if (more) DTL_COMMIT_M(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
#undef DTL_ISSUE_M
#undef DTL_COMMIT_M
  const int t = blockIdx.y * PB + wp * 16 + l16;
  if (t >= T) return;
  bool ok = true;
  if (MODE == MODE_PAIR) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int row = blockIdx.x * (TR / 2) + wr * 8 + 2 * q + h;
      if (row >= p.rows0) continue;
      const float gv = acc[2 * h], uv = acc[2 * h + 1];
      const float v = silu_det(gv) * uv;
      ok &= finite(gv) && finite(uv) && finite(v);
      p.ffo[(size_t)t * p.rows0 + row] = v;
    }
  } else {
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int g = blockIdx.x * TR + wr * 16 + 4 * q + c;
      if (g >= rows_total) continue;
      const bool m = MODE == MODE_CAT && g >= p.rows0;
      const int local = m ? g - p.rows0 : g;
      const int R = m ? p.rows1 : p.rows0;
      ok &= store_epilogue(acc[c], m ? p.out1 : p.out0, (size_t)t * R + local, m ? p.bias1 : p.bias0,
                           local, p.epi);
    }
  }
  if (!ok) flag(p.err, ERRBIT_NON_FINITE);
}

namespace {
template <int WP, int WR, int MODE>
void launch_mfp(const Q4kF32Args& a, hipStream_t s) {
  constexpr int PB = WP * 16, TR = WR * 16;
  const int rows_grid = MODE == MODE_PAIR ? 2 * a.rows0 : (MODE == MODE_CAT ? a.rows0 + a.rows1 : a.rows0);
  dim3 grid((rows_grid + TR - 1) / TR, (a.T + PB - 1) / PB);
  launch_kernel(k_q4k_mfp<WP, WR, MODE>, grid, dim3(64 * WP * WR), 0, s, a);
}
}  // namespace

// F32 weights (dot_f32_ref: chain c of eight adds the products of elements
// c, c + 8, ... in order, then the combine tree), products on the matrix
// cores as in k_q4k_mfp.  The eight chains are independent, so two waves
// share each 16 x 16 tile of outputs, wave half h holding chains 4 h .. 4 h +
// 3 (sixteen sums a lane): twice the waves for the same work, which short
// matrices need to fill the chip.  Per 32 elements a wave issues four MFMAs,
// MFMA m's block b taking element 8 b + 4 h + m (a lane's operands are the
// float4 at 8 (lane / 16) + 4 h of its row and of its position), and 64 adds:
// register 4 b + c of MFMA m is the next term of chain 4 h + m of row c, so
// b ascending is the chain's order and sixteen adds in a row are independent.
// A workgroup of eight waves covers 32 rows x 32 positions and stages
// 64-element slices as k_q4k_mfp does; columns past the row are staged as
// zeros (both operands: the products are +0.0, which changes no sum).
//
// Measured: 32000 x 1024 at 256 positions 307 us (27.4 T multiply-adds/s of
// the 33.7 the pattern reaches), gate + up of that width (2 x 2816 rows) 61
// us; short matrices are bound by the one workgroup per CU that they fill
// (576-row q/k/v 10 us from 5 to 256 positions).  One lane per (row,
// position), the kernel before: 607 us per launch on average over a
// 100-position chunk of the SmolLM2-135M shape, 29 ms for six layers and the
// output projection against 0.64.
template <bool PAIR>
__global__ void __launch_bounds__(512) k_f32_mfp(F32Mats M, const float* __restrict__ x, int T, int* err) {
  constexpr int PB = 32, TR = 32, SL = 64, LD = SL + 4;
  __shared__ __align__(16) float st[2][PB + TR][LD];
  __shared__ __align__(16) float halves[4][64][4];
  const int cols = M.cols;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = wave & 1, wp = (wave >> 1) & 1, wr = wave >> 2;
  const int l16 = lane & 15, q = lane >> 4;
  // The matrix and row of tile row tr (clamped to the last row).
  auto locate = [&](int tr, int* mat, int* row) -> bool {
    if (PAIR) {
      const int rr = blockIdx.x * (TR / 2) + (tr >> 1);
      *mat = tr & 1;
      *row = rr < M.rows[0] ? rr : M.rows[0] - 1;
      return rr < M.rows[0];
    }
    const int g = blockIdx.x * TR + tr;
    const int gc = g < M.total_rows ? g : M.total_rows - 1;
    *mat = (gc >= M.row_end[0] ? 1 : 0) + (gc >= M.row_end[1] ? 1 : 0);
    *row = gc - (*mat == 0 ? 0 : (*mat == 1 ? M.row_end[0] : M.row_end[1]));
    return g < M.total_rows;
  };
  // Staging: thread x moves column float4 x % 16 of position x / 16 and of
  // tile row x / 16.
  const int sr = tid >> 4, c4 = (tid & 15) * 4;
  int sm, srow;
  (void)locate(sr, &sm, &srow);
  const int tt = blockIdx.y * PB + sr;
  const float* xs = x + (size_t)(tt < T ? tt : T - 1) * cols;
  const float* ws = pick3(M.w, sm) + (size_t)srow * cols;
  // Two slices of loads in flight (even slices in the first pair of slots),
  // for launches with one workgroup per CU.
  // (named registers: as struct members or array elements they went to scratch)
  float4 x0, w0, x1, w1;
#define DTL_ISSUE_F(n, e0)                                 \
  do {                                                     \
    const int e_ = (e0) + c4 < cols ? (e0) + c4 : 0;       \
    x##n = *reinterpret_cast<const float4*>(xs + e_);      \
    w##n = *reinterpret_cast<const float4*>(ws + e_);      \
  } while (0)
#define DTL_COMMIT_F(n, b, e0)                                                                         \
  do {                                                                                                 \
    const bool in_ = (e0) + c4 < cols;                                                                 \
    *reinterpret_cast<float4*>(&st[b][sr][c4]) =                                                       \
        make_float4(in_ ? x##n.x : 0.0f, in_ ? x##n.y : 0.0f, in_ ? x##n.z : 0.0f, in_ ? x##n.w : 0.0f); \
    *reinterpret_cast<float4*>(&st[b][PB + sr][c4]) =                                                  \
        make_float4(in_ ? w##n.x : 0.0f, in_ ? w##n.y : 0.0f, in_ ? w##n.z : 0.0f, in_ ? w##n.w : 0.0f); \
  } while (0)
  DTL_ISSUE_F(0, 0);
  DTL_ISSUE_F(1, SL);
  DTL_COMMIT_F(0, 0, 0);
  DTL_ISSUE_F(0, 2 * SL);
  __syncthreads();
  dtl_v16f zero;
#pragma unroll
  for (int i = 0; i < 16; i++) zero[i] = 0.0f;
  float acc[4][4];
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[m][c] = 0.0f;
  const int boff = (wp * 16 + l16) * LD + 8 * q + 4 * h;
  const int aoff = (PB + wr * 16 + l16) * LD + 8 * q + 4 * h;
  auto slice = [&](int buf) {
    const float* sb = &st[buf][0][0];
    dtl_v4f a4 = *(const dtl_v4f*)(sb + boff);
    dtl_v4f w4 = *(const dtl_v4f*)(sb + aoff);
#pragma unroll
    for (int g = 0; g < SL; g += 32) {
      dtl_v16f d[4];
#pragma unroll
      for (int m = 0; m < 4; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(w4[m], a4[m], zero, 0, 0, 0);
      if (g + 32 < SL) {
        a4 = *(const dtl_v4f*)(sb + boff + g + 32);
        w4 = *(const dtl_v4f*)(sb + aoff + g + 32);
      }
      __builtin_amdgcn_sched_barrier(0);  // as in k_q4k_mfp
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
          for (int c = 0; c < 4; c++) acc[m][c] += d[m][4 * b + c];
      // the next group's MFMAs after all of these adds
      asm volatile("" : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[0][2]), "+v"(acc[0][3]), "+v"(acc[1][0]),
                   "+v"(acc[1][1]), "+v"(acc[1][2]), "+v"(acc[1][3]), "+v"(a4));
      asm volatile("" : "+v"(acc[2][0]), "+v"(acc[2][1]), "+v"(acc[2][2]), "+v"(acc[2][3]), "+v"(acc[3][0]),
                   "+v"(acc[3][1]), "+v"(acc[3][2]), "+v"(acc[3][3]), "+v"(w4));
    }
  };
  // Slices past the end are staged as zeros and add nothing (their adds run
  // at most once, when the slice count is odd); refills are unconditional.
  for (int e0 = 0; e0 < cols; e0 += 2 * SL) {
    slice(0);
    DTL_COMMIT_F(1, 1, e0 + SL);
    DTL_ISSUE_F(1, e0 + 3 * SL);
    __syncthreads();
    slice(1);
    DTL_COMMIT_F(0, 0, e0 + 2 * SL);
    DTL_ISSUE_F(0, e0 + 4 * SL);
    __syncthreads();
  }
#undef DTL_ISSUE_F
#undef DTL_COMMIT_F
  // ((a0 + a1) + (a2 + a3)) + ((a4 + a5) + (a6 + a7)): the second half's sum
  // through LDS
  float half[4];
#pragma unroll
  for (int c = 0; c < 4; c++) half[c] = (acc[0][c] + acc[1][c]) + (acc[2][c] + acc[3][c]);
  if (h == 1) *reinterpret_cast<float4*>(halves[wave >> 1][lane]) = make_float4(half[0], half[1], half[2], half[3]);
  __syncthreads();
  if (h == 1) return;
  const float4 o4 = *reinterpret_cast<const float4*>(halves[wave >> 1][lane]);
  const float v4[4] = {half[0] + o4.x, half[1] + o4.y, half[2] + o4.z, half[3] + o4.w};
  const int t = blockIdx.y * PB + wp * 16 + l16;
  if (t >= T) return;
  bool ok = true;
  int mat, row;
  if (PAIR) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if (!locate(wr * 16 + 4 * q + 2 * i, &mat, &row)) continue;
      const float gv = v4[2 * i], uv = v4[2 * i + 1];
      const float v = silu_det(gv) * uv;
      ok &= finite(gv) && finite(uv) && finite(v);
      M.out[0][(size_t)t * M.rows[0] + row] = v;
    }
  } else {
#pragma unroll
    for (int c = 0; c < 4; c++) {
      if (!locate(wr * 16 + 4 * q + c, &mat, &row)) continue;
      ok &= store_epilogue(v4[c], pick3(M.out, mat), (size_t)t * pick3(M.rows, mat) + row, pick3(M.bias, mat), row, pick3(M.epi, mat));
    }
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

void launch_f32_mfp(const F32Mats& M, bool pair, const float* x, int T, int* err, hipStream_t s) {
  const int rows = pair ? 2 * M.rows[0] : M.total_rows;
  const dim3 grid((rows + 31) / 32, (T + 31) / 32);
  if (pair) launch_kernel(k_f32_mfp<true>, grid, dim3(512), 0, s, M, x, T, err);
  else launch_kernel(k_f32_mfp<false>, grid, dim3(512), 0, s, M, x, T, err);
}

// ---------------------------------------------------------------------------
// Chunk attention in three launches: the scores and the P.V sums as products
// on the matrix cores, the softmax between them through the score rows in
// memory.  A KV group's query rows (position t, head h) are numbered r = t G +
// h % G, so a tile of rows shares the group's keys and has rows of nearly the
// same length.  Every value is formed as in k_attention (dtl_kernels.hip):
// scores in dot_f32_ref's order, then * scale; max, clamped exps, the eight Z
// chains, divisions; out[d] += p_j * v_j[d] with j ascending (lib.rs:2319-2420).
//
// Bound by P.V's serial sums when the rows are few (a wave adds 16 keys in
// about 400 cycles), by the adds of both products when they are many.  128-wide
// heads, 8 query / 2 key heads, us per layer at 1000 keys and 5 / 16 / 64 /
// 128 / 512 positions: 37 / 37 / 44 / 51 / 106, against 344 to 350 up to 64
// positions of the kernel these widths ran before (one workgroup per KV group
// and position, K and V through one LDS tile).

// Scores of 32 query rows x 32 keys, HD contracted: the wave pair and chain
// split of k_f32_mfp, all of HD staged at once.
template <int HD>
__global__ void __launch_bounds__(512) k_attn_qk_mfp(const float* __restrict__ q, const float* __restrict__ kc,
                                                     int layer, int T, int pos0, int H, int KV, int n_ctx,
                                                     float scale, float* __restrict__ scores, int* err) {
  constexpr int KP = (HD + 31) / 32 * 32, LD = KP + 4, F4 = KP / 4;
  __shared__ __align__(16) float sq[32][LD];
  __shared__ __align__(16) float sk[32][LD];
  __shared__ __align__(16) float halves[4][64][4];
  const int G = H / KV, rows = T * G;
  const int g = blockIdx.z, r0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  const int rlast = (r0 + 31 < rows ? r0 + 31 : rows - 1);
  if (j0 > pos0 + rlast / G) return;  // no row of the tile sees these keys
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = wave & 1, wp = (wave >> 1) & 1, wr = wave >> 2;
  const int l16 = lane & 15, qd = lane >> 4;
  const float* keys = kc + ((size_t)layer * KV + g) * n_ctx * HD;
  const int jmax = pos0 + T - 1;
  for (int f = tid; f < 32 * F4; f += 512) {
    const int i = f / F4, c = 4 * (f % F4);
    const int r = r0 + i < rows ? r0 + i : rows - 1, j = j0 + i < jmax ? j0 + i : jmax;
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
    if (HD == KP || c < HD) {
      a = *reinterpret_cast<const float4*>(q + ((size_t)(r / G) * H + g * G + r % G) * HD + c);
      b = *reinterpret_cast<const float4*>(keys + (size_t)j * HD + c);
    }
    *reinterpret_cast<float4*>(&sq[i][c]) = a;
    *reinterpret_cast<float4*>(&sk[i][c]) = b;
  }
  __syncthreads();
  dtl_v16f zero;
#pragma unroll
  for (int i = 0; i < 16; i++) zero[i] = 0.0f;
  float acc[4][4];
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[m][c] = 0.0f;
  // MFMA rows are keys (a lane's four results are consecutive keys of one
  // query row), columns query rows
  const float* ap = &sk[wr * 16 + l16][8 * qd + 4 * h];
  const float* bp = &sq[wp * 16 + l16][8 * qd + 4 * h];
#pragma unroll
  for (int k0 = 0; k0 < KP; k0 += 32) {
    dtl_v4f a4 = *(const dtl_v4f*)(ap + k0);
    dtl_v4f b4 = *(const dtl_v4f*)(bp + k0);
    asm volatile("" : "+v"(a4), "+v"(b4));
    dtl_v16f d[4];
#pragma unroll
    for (int m = 0; m < 4; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(a4[m], b4[m], zero, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int m = 0; m < 4; m++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[m][c] += d[m][4 * b + c];
    asm volatile("" : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[0][2]), "+v"(acc[0][3]), "+v"(acc[1][0]),
                 "+v"(acc[1][1]), "+v"(acc[1][2]), "+v"(acc[1][3]));
    asm volatile("" : "+v"(acc[2][0]), "+v"(acc[2][1]), "+v"(acc[2][2]), "+v"(acc[2][3]), "+v"(acc[3][0]),
                 "+v"(acc[3][1]), "+v"(acc[3][2]), "+v"(acc[3][3]));
  }
  float half[4];
#pragma unroll
  for (int c = 0; c < 4; c++) half[c] = (acc[0][c] + acc[1][c]) + (acc[2][c] + acc[3][c]);
  if (h == 1) *reinterpret_cast<float4*>(halves[wave >> 1][lane]) = make_float4(half[0], half[1], half[2], half[3]);
  __syncthreads();
  if (h == 1) return;
  const float4 o4 = *reinterpret_cast<const float4*>(halves[wave >> 1][lane]);
  const int r = r0 + wp * 16 + l16, j = j0 + wr * 16 + 4 * qd;
  if (r >= rows) return;
  const int pos = pos0 + r / G;
  float* srow = scores + ((size_t)(r / G) * H + g * G + r % G) * n_ctx;
  const float s4[4] = {(half[0] + o4.x) * scale, (half[1] + o4.y) * scale, (half[2] + o4.z) * scale,
                       (half[3] + o4.w) * scale};
  bool ok = true;
#pragma unroll
  for (int c = 0; c < 4; c++)
    if (j + c <= pos) {
      ok &= finite(s4[c]);
      srow[j + c] = s4[c];
    }
  if (!ok && pos > 0) flag(err, ERRBIT_NON_FINITE);  // a single score is never formed
}

// softmax_in_place (lib.rs:2361-2388) of one score row, in place; the row's
// places up to the chunk's last position are set to zero, so that a tile of
// rows can be summed over one range.  LDS: the row, and its exps chain-major
// (element j at chain j % 8, slot j / 8).
__host__ __device__ inline int softmax_zs(int maxlen) { return (((maxlen + 7) / 8 + 3) & ~3) + 4; }

__global__ void __launch_bounds__(256) k_attn_softmax(float* scores, int T, int pos0, int H, int n_ctx, int* err) {
  extern __shared__ __align__(16) float lds[];
  __shared__ float red[4];
  __shared__ float zc[8];
  const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x;
  const int len = pos0 + t + 1, end = pos0 + T;
  const int zs = softmax_zs(end);
  float* zcm = lds;             // [8][zs]
  float* row = lds + 8 * zs;    // [len]
  float* srow = scores + ((size_t)t * H + h) * n_ctx;
  for (int j = len + tid; j < end; j += 256) srow[j] = 0.0f;
  if (len == 1) {
    if (tid == 0) srow[0] = 1.0f;
    return;
  }
  float mx = -__builtin_huge_valf();
  for (int j0 = tid; j0 < len; j0 += 1024) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = srow[j0 + 256 * k < len ? j0 + 256 * k : len - 1];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (j0 + 256 * k < len) row[j0 + 256 * k] = v[k];
      mx = fmaxf(mx, v[k]);
    }
  }
  mx = wave_fmax(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const int n8 = (len + 7) & ~7;
#pragma unroll 4
  for (int j = tid; j < n8; j += 256) {
    // padded to the longest chain with +0.0, which no sum of exps changes
    const float e = j < len ? exp_clamped(row[j < len ? j : 0] - mx) : 0.0f;
    if (j < len) row[j] = e;
    zcm[(j & 7) * zs + (j >> 3)] = e;
  }
  __syncthreads();
  if (tid < 128) {
    const float z = chain_group_lds<16>(0.0f, zcm + (tid >> 4) * zs, n8 / 8);
    if ((tid & 15) == 0) zc[tid >> 4] = z;
  }
  __syncthreads();
  const float z = finish_8lane(zc);
  bool ok = finite(z) && z != 0.0f;
#pragma unroll 4
  for (int j = tid; j < len; j += 256) {
    const float p = row[j] / z;
    ok &= finite(p);
    srow[j] = p;
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

// out[r][d] = sum over j of p_r[j] v_j[d], one chain per output, j ascending
// (the pattern of k_q4k_mfp): MFMA rows are sixteen dimensions, columns
// sixteen query rows, the wave's 16 keys per group the four MFMAs' K.  A
// workgroup has a wave per (sixteen dimensions, row tile) of RT row tiles and
// stages 64 keys of its rows' probabilities and of V, double-buffered.
// Keys past a row's own position have probability +0.0 (products +-0, which
// change no sum).
template <int HD>
constexpr int pv_row_tiles() { return HD <= 64 ? 2 : 1; }

template <int HD>
__global__ void __launch_bounds__(HD / 16 * pv_row_tiles<HD>() * 64) k_attn_pv_mfp(
    const float* __restrict__ scores, const float* __restrict__ vc, int layer, int T, int pos0, int H, int KV,
    int n_ctx, float* __restrict__ out, int* err) {
  constexpr int DT = HD / 16, RT = pv_row_tiles<HD>(), NT = 64 * DT * RT, SL = 64;
  constexpr int LDV = HD + 4, LDP = SL + 4;
  constexpr int NV = SL * HD / 4 / NT, NP = (16 * RT * SL + NT - 1) / NT;  // staging slots per thread
  static_assert(SL * HD / 4 % NT == 0, "whole staging rounds");
  __shared__ __align__(16) float sv[2][SL][LDV];
  __shared__ __align__(16) float sp[2][16 * RT][LDP];
  const int G = H / KV, rows = T * G;
  const int g = blockIdx.y, r0 = blockIdx.x * 16 * RT;
  const int rlast = r0 + 16 * RT - 1 < rows ? r0 + 16 * RT - 1 : rows - 1;
  const int end = pos0 + rlast / G + 1;  // keys the tile's longest row sees
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dt = wave % DT, rt = wave / DT;
  const int l16 = lane & 15, qd = lane >> 4;
  const float* vals = vc + ((size_t)layer * KV + g) * n_ctx * HD;
  const float* prow[NP];
#pragma unroll
  for (int k = 0; k < NP; k++) {
    const int r = r0 + (tid + k * NT) / SL, rc = r < rows ? r : rows - 1;
    prow[k] = scores + ((size_t)(rc / G) * H + g * G + rc % G) * n_ctx;
  }
  dtl_v4f v[NV];
  float p[NP];
  auto issue = [&](int k0) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int f = tid + k * NT, j = k0 + f / (HD / 4);
      v[k] = *reinterpret_cast<const dtl_v4f*>(vals + (size_t)(j < end ? j : 0) * HD + 4 * (f % (HD / 4)));
    }
#pragma unroll
    for (int k = 0; k < NP; k++) {
      const int j = k0 + (tid + k * NT) % SL;
      p[k] = prow[k][j < end ? j : 0];
    }
  };
  auto commit = [&](int b, int k0) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int f = tid + k * NT;
      *reinterpret_cast<dtl_v4f*>(&sv[b][f / (HD / 4)][4 * (f % (HD / 4))]) = v[k];
    }
#pragma unroll
    for (int k = 0; k < NP; k++) {
      const int f = tid + k * NT;
      if (16 * RT * SL % NT == 0 || f < 16 * RT * SL) sp[b][f / SL][f % SL] = k0 + f % SL < end ? p[k] : 0.0f;
    }
  };
  dtl_v16f zero;
#pragma unroll
  for (int i = 0; i < 16; i++) zero[i] = 0.0f;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  issue(0);
  commit(0, 0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < end; k0 += SL) {
    issue(k0 + SL);  // unconditional: past the end row 0, not summed
    const float* ap = &sv[buf][4 * qd][dt * 16 + l16];
    const float* bp = &sp[buf][rt * 16 + l16][4 * qd];
#pragma unroll
    for (int e = 0; e < SL; e += 16) {
      dtl_v4f a4 = {ap[e * LDV], ap[(e + 1) * LDV], ap[(e + 2) * LDV], ap[(e + 3) * LDV]};
      dtl_v4f b4 = *(const dtl_v4f*)(bp + e);
      asm volatile("" : "+v"(a4), "+v"(b4));
      dtl_v16f d[4];
#pragma unroll
      for (int m = 0; m < 4; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(a4[m], b4[m], zero, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
          for (int c = 0; c < 4; c++) acc[c] += d[m][4 * b + c];
      asm volatile("" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
    }
    commit(buf ^ 1, k0 + SL);
    __syncthreads();
    buf ^= 1;
  }
  const int r = r0 + rt * 16 + l16, d0 = dt * 16 + 4 * qd;
  if (r >= rows) return;
  float4 o = make_float4(acc[0], acc[1], acc[2], acc[3]);
  if (pos0 + r / G == 0) o = *reinterpret_cast<const float4*>(vals + d0);  // a single score copies V exactly
  else if (!(finite(o.x) && finite(o.y) && finite(o.z) && finite(o.w))) flag(err, ERRBIT_NON_FINITE);
  *reinterpret_cast<float4*>(out + ((size_t)(r / G) * H + g * G + r % G) * HD + d0) = o;
}

namespace {
constexpr size_t kSoftmaxLds = 150 * 1024;
size_t softmax_smem(int maxlen) { return ((size_t)8 * softmax_zs(maxlen) + ((maxlen + 3) & ~3)) * sizeof(float); }

template <int HD>
void launch_attention_hd(const float* q, const float* kc, const float* vc, int layer, int T, int pos0, int H, int KV,
                         int n_ctx, float scale, float* scores, float* out, int* err, hipStream_t s) {
  const int rows = T * (H / KV), end = pos0 + T;
  constexpr int RT = 16 * pv_row_tiles<HD>();
  launch_kernel(k_attn_qk_mfp<HD>, dim3((rows + 31) / 32, (end + 31) / 32, KV), dim3(512), 0, s, q, kc, layer, T,
                pos0, H, KV, n_ctx, scale, scores, err);
  static const bool attr = hipFuncSetAttribute((const void*)k_attn_softmax,
                                               hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)kSoftmaxLds) == hipSuccess;
  (void)attr;
  launch_kernel(k_attn_softmax, dim3(H, T), dim3(256), softmax_smem(end), s, scores, T, pos0, H, n_ctx, err);
  launch_kernel(k_attn_pv_mfp<HD>, dim3((rows + RT - 1) / RT, KV), dim3(HD / 16 * pv_row_tiles<HD>() * 64), 0, s,
                scores, vc, layer, T, pos0, H, KV, n_ctx, out, err);
}
}  // namespace

bool launch_attention_mfp(const float* q, const float* kc, const float* vc, int layer, int T, int pos0, int H, int KV,
                          int hd, int n_ctx, float scale, float* scores, float* out, int* err, hipStream_t s) {
  if (softmax_smem(pos0 + T) > kSoftmaxLds) return false;
#define DTL_ATTN_HD(w) \
  case w: launch_attention_hd<w>(q, kc, vc, layer, T, pos0, H, KV, n_ctx, scale, scores, out, err, s); return true
  switch (hd) {
    DTL_ATTN_HD(16);
    DTL_ATTN_HD(32);
    DTL_ATTN_HD(64);
    DTL_ATTN_HD(80);
    DTL_ATTN_HD(96);
    DTL_ATTN_HD(128);
  }
#undef DTL_ATTN_HD
  return false;
}

// Measurement support: the rate of k_q4k_mfp's inner pattern on a chip
// with nothing else to do, four 16x16x1 outer products (4096 products per
// wave) and the 64 ordered adds per lane that take them into four chains,
// with operands the compiler must treat as new each iteration.  A SIMD runs
// the f32 MFMAs and the VALU adds one after the other, not side by side, so
// this, not either unit's own peak, bounds the Q4_K chunk GEMMs.  Four
// waves per SIMD (k_q4k_mfp's occupancy); the result is written only for a
// value no input produces, which keeps the work live.
__global__ void __launch_bounds__(256) k_mfp_probe(float* out, float a0, float b0, int iters) {
  const int lane = threadIdx.x & 63;
  dtl_v4f a4, w4;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    a4[m] = a0 + (float)(lane + m);
    w4[m] = b0 - (float)(lane * m);
  }
  dtl_v16f zero;
#pragma unroll
  for (int i = 0; i < 16; i++) zero[i] = 0.0f;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int it = 0; it < iters; it++) {
    dtl_v16f d[4];
#pragma unroll
    for (int m = 0; m < 4; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(w4[m], a4[m], zero, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int m = 0; m < 4; m++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[c] += d[m][4 * b + c];
    asm volatile("" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(a4), "+v"(w4));
  }
  const float s = acc[0] + acc[1] + acc[2] + acc[3];
  if (s == -1.0f) out[threadIdx.x] = s;
}

void launch_mfp_probe(float* out, int workgroups, int iters, hipStream_t s) {
  launch_kernel(k_mfp_probe, dim3(workgroups), dim3(256), 0, s, out, 1.0001f, 0.5f, iters);
}

// Tiles (waves over positions x rows): 2 x 2.  For the short matrices 4 x 1
// (one row tile, four position tiles) was the faster with 64-position launches
// side by side; from 96 positions on 2 x 2 is: us per launch alone, wo and
// ffn_down on average / wq + wk of the TinyLlama-1.1B shape, 4 x 1 against 2 x
// 2: 96 positions 51.4 against 48.5 / 42.1 against 31.7, 256 66.3 against 64.2
// / 61.7 against 59.1, 512 130.6 against 115.4 / 97.9 against 93.0; the
// pipelined 2048-token window 88.5 against 88.3 ms (86.8 against 88.3 in
// chunks of 512).
void launch_q4k_mfp(const Q4kF32Args& a, int mode, hipStream_t s) {
  if (mode == MODE_PAIR) return launch_mfp<2, 2, MODE_PAIR>(a, s);
  if (mode == MODE_CAT) return launch_mfp<2, 2, MODE_CAT>(a, s);
  launch_mfp<2, 2, MODE_SINGLE>(a, s);
}

}  // namespace dtl
