// GEMVs of a few positions with F32 weights (F32 and widened F16 models):
// dot_f32_ref's order (det-num reduce.rs: eight interleaved chains and the
// combine tree), one launch for the matrices that share an input.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dtl_device.h"
#include "dtl_numerics.h"

namespace dtl {

namespace {

constexpr int kGgmlF32 = 0;

__device__ __forceinline__ void flag(int* err, int bit) { atomicOr(err, bit); }

// Lane I of each quad, to the quad's four lanes.
template <int I>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), I * 0x55, 0xf, 0xf, true));
}

// Lane i ^ 8 within each row of sixteen.
__device__ __forceinline__ float row_swap8(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));  // row_ror:8
}

}  // namespace

// A wave covers eight weight rows, eight lanes each, and TT positions.  Of a
// row's next 32 elements, lane (half h, q) of its eight loads the float4 at
// 8 q + 4 h: the eight lanes read one 128-byte line, the four lanes of a quad
// hold consecutive terms of the same four chains (4 h .. 4 h + 3), and each
// forms its own rounded products.  Every lane of the quad then adds the four
// products of each chain in order, taking them from the quad's lanes by DPP:
// per 32 elements and row one load, four multiplies and sixteen adds a lane,
// no LDS and no barrier.  The chains' sums join by finish_8lane's tree.
//
// Bound by the weights' stream on tall matrices (49152 x 576, 113 MB: 17.4 us
// per launch at one position, 6.5 TB/s), by the launch, one memory round
// trip and the adds (cols / 8 per chain) on short ones (q/k/v, gate + up and
// wo / down of the SmolLM2-135M shape: 4.8, 5.1 and 6.4 us).  One lane per
// row, the kernel these shapes ran before: 225 us per token of the two-layer
// 64-wide model against 125.
//
// PAIR: the wave's eight rows alternate gate and up (four rows of each);
// silu(gate) * up is written to out[0].
template <int TT, bool PAIR>
__global__ void __launch_bounds__(256) k_gemv_f32(F32Mats M, const float* __restrict__ x, int T, int* err) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int grp = lane >> 3, h = (lane >> 2) & 1, q = lane & 3;
  const int t0 = blockIdx.y * TT;
  const int cols = M.cols;
  // this lane's row: its matrix and its index there
  int m, r;
  bool live;
  if (PAIR) {
    m = grp & 1;
    r = wave * 4 + (grp >> 1);
    live = r < M.rows[0];
    r = live ? r : M.rows[0] - 1;
  } else {
    const int g = wave * 8 + grp;
    live = g < M.total_rows;
    const int gc = live ? g : M.total_rows - 1;
    m = (gc >= M.row_end[0] ? 1 : 0) + (gc >= M.row_end[1] ? 1 : 0);
    r = gc - (m == 0 ? 0 : (m == 1 ? M.row_end[0] : M.row_end[1]));
  }
  const float* w = pick3(M.w, m) + (size_t)r * cols;
  const float* xr[TT];
#pragma unroll
  for (int t = 0; t < TT; t++) xr[t] = x + (size_t)(t0 + t < T ? t0 + t : T - 1) * cols;
  float acc[TT][4];
#pragma unroll
  for (int t = 0; t < TT; t++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[t][c] = 0.0f;
  const int off = 8 * q + 4 * h;
  auto add_in_order = [&](float (&a)[4], const float4& p) {
    a[0] += quad_lane<0>(p.x);
    a[1] += quad_lane<0>(p.y);
    a[2] += quad_lane<0>(p.z);
    a[3] += quad_lane<0>(p.w);
    a[0] += quad_lane<1>(p.x);
    a[1] += quad_lane<1>(p.y);
    a[2] += quad_lane<1>(p.z);
    a[3] += quad_lane<1>(p.w);
    a[0] += quad_lane<2>(p.x);
    a[1] += quad_lane<2>(p.y);
    a[2] += quad_lane<2>(p.z);
    a[3] += quad_lane<2>(p.w);
    a[0] += quad_lane<3>(p.x);
    a[1] += quad_lane<3>(p.y);
    a[2] += quad_lane<3>(p.z);
    a[3] += quad_lane<3>(p.w);
  };
  // U lines of the row in flight per lane
  constexpr int U = TT == 1 ? 8 : (TT == 2 ? 4 : 2);
  const int whole = cols / (32 * U) * (32 * U);
  for (int e0 = 0; e0 < whole; e0 += 32 * U) {
    float4 wv[U], xv[U][TT];
#pragma unroll
    for (int u = 0; u < U; u++) {
      wv[u] = *reinterpret_cast<const float4*>(w + e0 + 32 * u + off);
#pragma unroll
      for (int t = 0; t < TT; t++) xv[u][t] = *reinterpret_cast<const float4*>(xr[t] + e0 + 32 * u + off);
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < TT; t++)
        add_in_order(acc[t], make_float4(wv[u].x * xv[u][t].x, wv[u].y * xv[u][t].y, wv[u].z * xv[u][t].z,
                                         wv[u].w * xv[u][t].w));
  }
  // The rest: addresses clamped to the row, terms past it added as +0.0 (a
  // sum that starts at +0.0 is never -0.0, so its bits do not change).
  for (int e0 = whole; e0 < cols; e0 += 32) {
    const int e = e0 + off;
    const bool in = e < cols;
    const int ec = in ? e : 0;
    const float4 wv = *reinterpret_cast<const float4*>(w + ec);
#pragma unroll
    for (int t = 0; t < TT; t++) {
      const float4 xv = *reinterpret_cast<const float4*>(xr[t] + ec);
      add_in_order(acc[t], make_float4(in ? wv.x * xv.x : 0.0f, in ? wv.y * xv.y : 0.0f,
                                       in ? wv.z * xv.z : 0.0f, in ? wv.w * xv.w : 0.0f));
    }
  }
  // lane s of a row's eight stores position s
  const int s = lane & 7;
  float v = 0.0f;
#pragma unroll
  for (int t = 0; t < TT; t++) {
    const float half = (acc[t][0] + acc[t][1]) + (acc[t][2] + acc[t][3]);
    const float sum = half + dpp_f32<kDppMirror8>(half);
    v = s == t ? sum : v;
  }
  bool ok = true;
  if (PAIR) {
    const float other = row_swap8(v);
    if (live && s < TT && t0 + s < T && m == 0) {
      const float p = silu_det(v) * other;
      ok = finite(v) && finite(other) && finite(p);
      M.out[0][(size_t)(t0 + s) * M.rows[0] + r] = p;
    }
  } else if (live && s < TT && t0 + s < T) {
    float* o = pick3(M.out, m) + (size_t)(t0 + s) * pick3(M.rows, m) + r;
    ok = finite(v);
    if (pick3(M.epi, m) == EPI_BIAS) v = v + pick3(M.bias, m)[r];
    else if (pick3(M.epi, m) == EPI_RESIDUAL) v = *o + v;
    *o = v;
    ok = ok && finite(v);
  }
  if (!ok) flag(err, ERRBIT_NON_FINITE);
}

namespace {
template <bool PAIR>
void launch_gemv_f32(const F32Mats& M, const float* x, int T, int* err, hipStream_t s) {
  const int rows = PAIR ? 2 * M.rows[0] : M.total_rows;
  const int waves = (rows + 7) / 8;
  // Short matrices: one wave per workgroup, so that every wave has a CU's
  // load path to itself.
  const int per = waves >= 2048 ? 4 : 1;
  const int TT = T == 1 ? 1 : (T == 2 ? 2 : 4);
  const dim3 grid((waves + per - 1) / per, (T + TT - 1) / TT), block(64 * per);
  if (TT == 1) launch_kernel((k_gemv_f32<1, PAIR>), grid, block, 0, s, M, x, T, err);
  else if (TT == 2) launch_kernel((k_gemv_f32<2, PAIR>), grid, block, 0, s, M, x, T, err);
  else launch_kernel((k_gemv_f32<4, PAIR>), grid, block, 0, s, M, x, T, err);
}
}  // namespace

bool f32_mats_fit(const DevMat* const* mats, int nm, bool pair) {
  if (nm < 1 || nm > 3 || (pair && nm != 2)) return false;
  for (int i = 0; i < nm; i++) {
    const DevMat& m = *mats[i];
    // whole float4 per row, every row 16-byte aligned
    if (m.type != kGgmlF32 || m.cols != mats[0]->cols || m.cols % 4 != 0 || m.rows <= 0) return false;
    if (pair && m.rows != mats[0]->rows) return false;
  }
  return true;
}

bool launch_f32_mats(const DevMat* const* mats, int nm, bool pair, const float* x, int T, float* const* outs,
                     const float* const* biases, const int* epis, int* err, hipStream_t s) {
  if (T < 1 || !f32_mats_fit(mats, nm, pair)) return false;
  F32Mats M{};
  int acc = 0;
  for (int i = 0; i < 3; i++) {
    if (i < nm) {
      M.w[i] = static_cast<const float*>(mats[i]->w);
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
  M.cols = mats[0]->cols;
  if (T > kF32GemvMaxT) {
    launch_f32_mfp(M, pair, x, T, err, s);
  } else if (pair) {
    launch_gemv_f32<true>(M, x, T, err, s);
  } else {
    launch_gemv_f32<false>(M, x, T, err, s);
  }
  return true;
}

}  // namespace dtl
