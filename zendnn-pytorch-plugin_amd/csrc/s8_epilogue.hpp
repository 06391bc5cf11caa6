// Epilogue of the tiled int8 GEMMs (dynq_kernels.hip, s8_prefill.hip), four
// columns of a row at a time; the arithmetic of dyn_epilogue.
#pragma once

#include "zt_gemm_tile.hpp"
#include "zt_launch.hpp"

namespace zt {

// What the epilogue of one column quad n..n+3 needs for every row.
struct QuadScales {
  float sw[4], bias[4], inv, zp;
  int32_t cs[4];
  bool has_bias;

  __device__ __forceinline__ void load(const DynArgs &a, int n, int N) {
    has_bias = a.bias != nullptr;
    inv = a.out_scale ? __fdiv_rn(1.0f, *a.out_scale) : 0.f;
    zp = a.out_zp ? (float)*a.out_zp : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const bool in = n + r < N;
      sw[r] = in && a.sw ? load_elem(a.sw, a.sw_dt, a.sw_bcast ? 0 : n + r) : 0.f;
      bias[r] = in && has_bias ? load_elem(a.bias, a.b_dt, n + r) : 0.f;
      cs[r] = in && a.azp ? a.colsum[n + r] : 0;
    }
  }

  // the arithmetic of dyn_epilogue: ((acc - azp colsum) sx) sw + bias
  __device__ __forceinline__ i32x4_t correct(i32x4_t v, int32_t azp) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] -= azp * cs[r];
    return v;
  }
  __device__ __forceinline__ void scale(i32x4_t v, float sx, float (&f)[4]) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float t = (float)v[r] * sx * sw[r];
      f[r] = has_bias ? t + bias[r] : t;
    }
  }
};

// Whether the post-ops are at most one relu, which costs one instruction on
// the way to the store and no pass of its own.
__host__ __device__ __forceinline__ bool at_most_relu(const PostOps &p) {
  return p.count == 0 || (p.count == 1 && p.ids[0] == ZT_PO_RELU);
}

// Columns n..n+3 of row m of the raw sums / of y.
__device__ __forceinline__ void store_sums4(const DynArgs &a, int m, int n, int N, i32x4_t v) {
  int32_t *dst = reinterpret_cast<int32_t *>(a.y) + (int64_t)m * N + n;
  if (n + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
    *reinterpret_cast<i32x4_t *>(dst) = v;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) dst[r] = v[r];
  }
}

__device__ __forceinline__ void store_y4(const DynArgs &a, const QuadScales &q, int m, int n, int N,
                                         float (&f)[4], bool relu) {
  if (relu)
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = unary_op(ZT_PO_RELU, f[r]);
  if (a.y_dt != ZT_DT_U8 && a.y_dt != ZT_DT_S8) {
    store4(a.y, a.y_dt, N, m, n, N, f);
    return;
  }
  const float lo = a.y_dt == ZT_DT_U8 ? 0.f : -128.f, hi = a.y_dt == ZT_DT_U8 ? 255.f : 127.f;
  uint32_t b[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    b[r] = (uint32_t)(int)fminf(fmaxf(rintf(f[r] * q.inv) + q.zp, lo), hi) & 0xffu;
  uint8_t *dst = reinterpret_cast<uint8_t *>(a.y) + (int64_t)m * N + n;
  if (n + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 3u) == 0) {
    *reinterpret_cast<uint32_t *>(dst) = b[0] | b[1] << 8 | b[2] << 16 | b[3] << 24;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) dst[r] = (uint8_t)b[r];
  }
}

}  // namespace zt
