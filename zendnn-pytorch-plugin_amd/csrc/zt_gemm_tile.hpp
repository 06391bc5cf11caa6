// Device helpers shared by the large-tile prefill GEMMs (woq_prefill.hip,
// s8_prefill.hip): LDS DMA, step waits, tile order and the four-column
// epilogue.
#pragma once

#include <type_traits>

#include "zt_common.hpp"

namespace zt {

typedef __attribute__((address_space(3))) void *tile_lds_ptr_t;

__device__ __forceinline__ uint32_t lds_address(void *p) {
  return (uint32_t)(uintptr_t)(tile_lds_ptr_t)p;
}

// Raw buffer descriptor as four scalars, for dma16.
__device__ __forceinline__ i32x4_t dma_rsrc(const void *p, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return i32x4_t{__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff),
                 __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}

// One 16-byte-per-lane load of buffer bytes voff + soff straight into LDS at
// lds + 16 * lane; a lane whose voff is kOobOffset gets zeros.  Written as
// assembly because the compiler, seeing the builtin, waits for every such load in flight before each later
// LDS read it cannot prove disjoint (vmcnt(0) in the middle of the step that
// the loads were issued ahead of); it has no register result, and the
// callers wait for it themselves (wait_step) before the barrier that
// publishes the stage.  Writing M0 needs one wait state before the load; the
// kernels that call this hold nothing else in M0 (it cannot be named as a
// clobber: the compiler reserves it), so they use no builtin that does.
__device__ __forceinline__ void dma16(i32x4_t rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\t"
               "s_nop 0\n\t"
               "buffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
               : "memory");
}

// At most N of this wave's loads outstanding (they retire in order) and its
// LDS accesses done, then the workgroup barrier.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);
  asm volatile("s_barrier" ::: "memory");
}

// All of this wave's loads and LDS accesses done, then the workgroup barrier.
__device__ __forceinline__ void wait_step() { wait_loads<0>(); }

// Tile (tm, tn) of workgroup b: groups of group_m row tiles walked column by
// column, each XCD on one contiguous range of that order.
__device__ __forceinline__ void grouped_tile(int b, int tiles_m, int tiles_n, int group_m,
                                             int &tm, int &tn) {
  const int t = xcd_contiguous_tile(b, tiles_m * tiles_n);
  const int per_group = group_m * tiles_n;
  const int g = t / per_group, tg = t - g * per_group;
  const int gm = min(group_m, tiles_m - g * group_m);
  tm = g * group_m + tg % gm;
  tn = tg / gm;
}

// Post-ops on columns n..n+3 of row m (valid[r]: column n + r exists), the
// binary operands as one 8- or 16-byte load where their address allows it.
// Same arithmetic, in the same order, as apply_post_ops per element.
__device__ __forceinline__ void post_ops4(float (&f)[4], const PostOps &p, int64_t m, int n,
                                          int N) {
  int b = 0;
  for (int i = 0; i < p.count; ++i) {
    const int id = p.ids[i];
    if (id == ZT_PO_ADD || id == ZT_PO_MUL) {
      float o[4] = {0.f, 0.f, 0.f, 0.f};
      const int64_t at = m * p.ld[b] + n;
      const bool f32 = p.dts[b] == ZT_DT_F32;
      const char *src = static_cast<const char *>(p.bufs[b]) + at * (f32 ? 4 : 2);
      if (n + 3 < N && (reinterpret_cast<uintptr_t>(src) & (f32 ? 15u : 7u)) == 0) {
        if (f32) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t *>(src);
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = v[r];
        } else {
          const u32x2_t v = *reinterpret_cast<const u32x2_t *>(src);
          o[0] = bf16_bits_to_f32(v[0] & 0xffffu);
          o[1] = __uint_as_float(v[0] & 0xffff0000u);
          o[2] = bf16_bits_to_f32(v[1] & 0xffffu);
          o[3] = __uint_as_float(v[1] & 0xffff0000u);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) o[r] = load_elem(p.bufs[b], p.dts[b], at + r);
      }
      ++b;
#pragma unroll
      for (int r = 0; r < 4; ++r) f[r] = id == ZT_PO_ADD ? f[r] + o[r] : f[r] * o[r];
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) f[r] = unary_op(id, f[r]);
    }
  }
}

// Post-ops over a wave's 32-row slab of fp32 results in LDS, in place: lane
// holds column quads c4 of rows r0 + t * RP (t < T), global row mb + that and
// column n.  Op by op over the whole slab and not quad by quad: the binary
// operands of all T rows are then in flight together (a quad at a time each
// waited for its own load, 32 round trips per tile), and the unary functions'
// code exists once for all rows.
template <int T, int RP>
__device__ __forceinline__ void post_ops_slab(float *slab, int pitch, int c4, int r0,
                                              const PostOps &p, int mb, int n, int M, int N) {
  int b = 0;
  for (int i = 0; i < p.count; ++i) {
    const int id = p.ids[i];
    if (id == ZT_PO_ADD || id == ZT_PO_MUL) {
      const bool f32 = p.dts[b] == ZT_DT_F32;
      const int es = f32 ? 4 : 2;
      const char *base = static_cast<const char *>(p.bufs[b]) + (int64_t)n * es;
      const int64_t ld = p.ld[b] * es;
      const bool vec =
          n + 3 < N && ((reinterpret_cast<uintptr_t>(base) | ld) & (f32 ? 15 : 7)) == 0;
      auto row = [&](int t) { return base + min(mb + t * RP + r0, M - 1) * ld; };
      auto apply = [&](int t, f32x4_t w) {
        f32x4_t *q = reinterpret_cast<f32x4_t *>(slab + (t * RP + r0) * pitch + c4);
        *q = id == ZT_PO_ADD ? *q + w : *q * w;
      };
      if (vec && f32) {
        constexpr int U = T < 8 ? T : 8;  // rows in flight
        static_assert(T % U == 0, "whole batches");
#pragma unroll 1
        for (int t0 = 0; t0 < T; t0 += U) {
          f32x4_t o[U];
#pragma unroll
          for (int t = 0; t < U; ++t) o[t] = *reinterpret_cast<const f32x4_t *>(row(t0 + t));
#pragma unroll
          for (int t = 0; t < U; ++t) apply(t0 + t, o[t]);
        }
      } else if (vec) {
        u32x2_t o[T];
#pragma unroll
        for (int t = 0; t < T; ++t) o[t] = *reinterpret_cast<const u32x2_t *>(row(t));
#pragma unroll
        for (int t = 0; t < T; ++t)
          apply(t, f32x4_t{bf16_bits_to_f32(o[t][0] & 0xffffu), __uint_as_float(o[t][0] & 0xffff0000u),
                           bf16_bits_to_f32(o[t][1] & 0xffffu), __uint_as_float(o[t][1] & 0xffff0000u)});
      } else {
        // rows that are not whole aligned quads: element by element, four rows'
        // loads in flight (columns past N read column N - 1, and are not stored)
        auto elements = [&](auto *src) {
          constexpr int U = T % 4 == 0 ? 4 : 1;
#pragma unroll 1
          for (int t0 = 0; t0 < T; t0 += U) {
            f32x4_t o[U];
#pragma unroll
            for (int t = 0; t < U; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const auto v =
                    src[min(mb + (t0 + t) * RP + r0, M - 1) * p.ld[b] + min(n + r, N - 1)];
                if constexpr (sizeof(v) == 4) o[t][r] = v;
                else o[t][r] = bf16_bits_to_f32(v);
              }
#pragma unroll
            for (int t = 0; t < U; ++t) apply(t0 + t, o[t]);
          }
        };
        if (f32) elements(static_cast<const float *>(p.bufs[b]));
        else elements(static_cast<const uint16_t *>(p.bufs[b]));
      }
      ++b;
    } else {
      // four rows at a time, so that their latencies overlap, each function in
      // code of its own.  Row by row a gelu, sigmoid or tanh took 12 us of a 4096 x
      // 4096 call at M = 699 (44 us without), a silu 9 of 14336 x 4096 at M = 200.
      auto rows = [&](auto op) {
        constexpr int U = T % 4 == 0 ? 4 : 1;
#pragma unroll 1
        for (int t0 = 0; t0 < T; t0 += U) {
          f32x4_t v[U];
#pragma unroll
          for (int t = 0; t < U; ++t)
            v[t] = *reinterpret_cast<f32x4_t *>(slab + ((t0 + t) * RP + r0) * pitch + c4);
#pragma unroll
          for (int t = 0; t < U; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[t][r] = unary_op(op.value, v[t][r]);
            *reinterpret_cast<f32x4_t *>(slab + ((t0 + t) * RP + r0) * pitch + c4) = v[t];
          }
        }
      };
      switch (id) {
      case ZT_PO_RELU: rows(std::integral_constant<int, ZT_PO_RELU>{}); break;
      case ZT_PO_GELU_TANH: rows(std::integral_constant<int, ZT_PO_GELU_TANH>{}); break;
      case ZT_PO_GELU_ERF: rows(std::integral_constant<int, ZT_PO_GELU_ERF>{}); break;
      case ZT_PO_SILU: rows(std::integral_constant<int, ZT_PO_SILU>{}); break;
      case ZT_PO_SIGMOID: rows(std::integral_constant<int, ZT_PO_SIGMOID>{}); break;
      case ZT_PO_TANH: rows(std::integral_constant<int, ZT_PO_TANH>{}); break;
      default: break;
      }
    }
  }
}

// Columns n..n+3 of row m of y, in one store where the row allows it.
__device__ __forceinline__ void store4(void *y, int y_dt, int64_t ldy, int64_t m, int n, int N,
                                       const float (&f)[4]) {
  char *dst = static_cast<char *>(y) + (m * ldy + n) * (y_dt == ZT_DT_F32 ? 4 : 2);
  const uintptr_t at = reinterpret_cast<uintptr_t>(dst);
  if (n + 3 < N && y_dt == ZT_DT_BF16 && (at & 7u) == 0) {
    *reinterpret_cast<u32x2_t *>(dst) =
        u32x2_t{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])};
  } else if (n + 3 < N && y_dt == ZT_DT_F32 && (at & 15u) == 0) {
    *reinterpret_cast<f32x4_t *>(dst) = f32x4_t{f[0], f[1], f[2], f[3]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) store_elem(y, y_dt, m * ldy + n + r, f[r]);
  }
}

}  // namespace zt
