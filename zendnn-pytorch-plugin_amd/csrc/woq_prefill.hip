// Large-tile int4 weight-only GEMM for gfx950 (prefill, any zero-point and
// scale type, groups of 32 and up).
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "woq_dequant.hpp"
#include "zt_gemm_tile.hpp"
#include "zt_launch.hpp"
#include "zt_tuning.hpp"

namespace zt {

namespace {

// How the workgroup dequantises: signed int4 with bf16 scales (one FMA per
// weight), unsigned int4 with bf16 scales and 8-bit integer zero points (and
// half a packed fp16 one), or any scale / zero-point type.
enum DequantMode { kDqS4 = 0, kDqU4 = 1, kDqAny = 2 };

// Cost model of woq_prefill_plan, microseconds: a tile's prologue and
// epilogue; one of its 64-k steps with few CUs busy and with all of them
// (clocks and L2 make the difference; the 128 x 128 tile runs two workgroups per
// CU past one round); and the K-split reduction.
constexpr double kPfFixed[3] = {4.0, 5.1, 7.9};
constexpr double kPfStepFew[3] = {0.70, 0.83, 1.15}, kPfStepAll[3] = {1.15, 1.04, 1.45};
constexpr double kPfReduce = 3.8, kPfReduceRate = 2.9e6;  // bytes per us

constexpr int kPfBK = 64;     // k per step
constexpr int kPfRow = 128;   // bytes of one LDS row: a step of bf16

// row pitch of the K splits' fp32 partials [split][M][pitch]
__host__ __device__ constexpr int64_t pf_pitch(int64_t N) { return (N + 3) / 4 * 4; }

// two stages of x and dequantised W rows (the epilogue's slabs, 32 rows x 68
// floats per wave, fit in them)
template <int BM, int BN>
constexpr size_t pf_lds() {
  return 2 * (size_t)(BM + BN) * kPfRow;
}

// Scale and zero point of one weight row's group, as loaded: converting them
// only where they are used keeps the wait for the loads there.
struct GroupRaw {
  uint32_t s, z;
};

// Scale and zero point number sn + g of the two arrays (sn per lane).
template <int DQ, typename R>
__device__ __forceinline__ GroupRaw load_group(const WoqArgs &a, R s_rs, R z_rs, uint32_t sn,
                                               uint32_t g) {
  auto u32 = [&](R rs) { return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, sn * 4, g * 4, 0); };
  auto u16 = [&](R rs) {
    return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, sn * 2, g * 2, 0);
  };
  auto u8 = [&](R rs) {
    return (uint32_t)(uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rs, sn, g, 0);
  };
  GroupRaw q{0, 0};
  q.s = DQ == kDqAny && a.s_dt == ZT_DT_F32 ? u32(s_rs) : u16(s_rs);
  if (DQ == kDqU4) {
    q.z = u8(z_rs);
  } else if (DQ == kDqAny) {
    if (a.zp_dt == ZT_DT_F32 || a.zp_dt == ZT_DT_S32) q.z = u32(z_rs);
    else if (a.zp_dt == ZT_DT_BF16) q.z = u16(z_rs);
    else if (a.zp_dt != ZT_DT_NONE) q.z = u8(z_rs);
  }
  return q;
}

struct GroupQ {
  float s, z;
};

// Their values, without branches: floats by a shift (0 or 16), 8-bit
// integers by their sign bit zsx (0x80 signed, 0 unsigned or 32-bit).
struct GroupFormat {
  int sshift, zshift, zsx;
  bool zint;
};

__device__ __forceinline__ GroupFormat group_format(const WoqArgs &a) {
  GroupFormat f;
  f.sshift = a.s_dt == ZT_DT_F32 ? 0 : 16;
  f.zshift = a.zp_dt == ZT_DT_BF16 ? 16 : 0;
  f.zsx = a.zp_dt == ZT_DT_S8 ? 0x80 : 0;
  f.zint = a.zp_dt == ZT_DT_S8 || a.zp_dt == ZT_DT_U8 || a.zp_dt == ZT_DT_S32;
  return f;
}

template <int DQ>
__device__ __forceinline__ GroupQ group_of(const GroupFormat &f, GroupRaw r) {
  GroupQ q;
  q.s = __uint_as_float(r.s << (DQ == kDqAny ? f.sshift : 16));
  const float zi = (float)(((int)r.z ^ f.zsx) - f.zsx);
  q.z = DQ == kDqS4 ? 0.f : (DQ == kDqU4 || f.zint) ? zi : __uint_as_float(r.z << f.zshift);
  return q;
}

template <int DQ>
__device__ __forceinline__ u32x4_t dequant8(uint32_t w, const GroupQ &q, int zmode) {
  if (DQ == kDqS4) return dq8_s4_bf16scale(w, q.s, q.s * 0.0625f, -1032.f * q.s, -72.f * q.s);
  if (DQ == kDqU4) return dq8_u4_scale(w, q.s, q.z);
  return dq8_general(w, dq_general_params(zmode, q.s, q.z));
}

// A register copy made here and not at the loop's back edge, where the
// compiler would put it after (and waiting for) the load that refills v.
__device__ __forceinline__ uint32_t copy_now(uint32_t v) {
  uint32_t r;
  asm volatile("v_mov_b32 %0, %1" : "=&v"(r) : "v"(v));
  return r;
}

// y tile of BM x BN on v_mfma_f32_32x32x16_bf16, WM x WN waves, K in steps of 64
// over two LDS stages [x rows | dequantised W rows] of 128-byte rows (16-byte
// chunk c of row r at c ^ ((r >> 1) & 7), so the 16 rows of a fragment read meet
// 16 bank groups).  x moves into LDS by DMA; the packed weights go through
// registers and are dequantised once per workgroup, not once per wave that
// multiplies with them.  A = W, B = x, so D is [n][m].  GU is the merged
// gate_up: every wave's 64 columns are 32 gate rows of W and their 32 up rows.
//
// Bound: the 256 x 256 tile reads 192 KB of fragments from LDS and writes 64
// per step, 2048 clocks at 128 B/clk, beside 2048 clocks of MFMAs, and on
// random data the chip's power holds the MFMAs fed from LDS to 1.53 PFLOP/s.
// 28672 x 4096 at M = 4096 runs at 1.19 PFLOP/s, at M = 2048 (3.5
// rounds of tiles) in 435-450 us; the kernels before it, which dequantised in
// every wave and waited for each step's DMA before the step's first LDS read,
// took 472-480.  Taking the dequantisation out saved 19 % of the time, the
// fragment reads 19 %, the DMA 8 %, all three 35 %.
template <int BM, int BN, int WM, int WN, int DQ, bool GU>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2, 2)))
void woq_prefill_kernel(WoqArgs a, int tiles_m, int tiles_n, int group_m, int gshift, int gmask,
                        float *partial, int sps) {
  constexpr int NT = 64 * WM * WN, NW = WM * WN;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // 32 x 32 tiles per wave
  constexpr int STAGE = (BM + BN) * kPfRow;
  constexpr int XL = BM / 8 / NW;  // 1 KB x loads (8 rows) per wave and step
  constexpr int TPR = NT / BN;   // threads per row of W, each WPT packed words a step
  constexpr int WPT = 8 / TPR;
  static_assert((TPR == 2 || TPR == 4) && TN == 2 && XL * NW * 8 == BM, "tile shape");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / WN, wn = wv % WN;
  const int hl = lane >> 5, l32 = lane & 31;
  int tm, tn;
  grouped_tile(blockIdx.x, tiles_m, tiles_n, group_m, tm, tn);
  const int M = (int)a.M, N = (int)a.N, K = (int)a.K;
  // columns of y; a merged gate_up tile is BN / 2 gate rows of W and their
  // BN / 2 up rows
  const int NY = GU ? N / 2 : N;
  const int m0 = tm * BM, n0 = tn * (GU ? BN / 2 : BN);
  const int ldx2 = (int)a.ldx * 2, KB = K / 2;
  const int nk = K / kPfBK;
  const int kb = partial ? (int)blockIdx.y * sps : 0;  // this workgroup's steps [kb, ke)
  const int ke = partial ? min(kb + sps, nk) : nk;

  // x: 8 rows x 128 B per load, chunk c of row r at c ^ ((r >> 1) & 7)
  const i32x4_t x_rs = dma_rsrc(a.x, (uint32_t)((int64_t)M * ldx2));
  const uint32_t lds0 = lds_address(smem);
  uint32_t xsrc[XL];
#pragma unroll
  for (int q = 0; q < XL; ++q) {
    const int row = (wv * XL + q) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    xsrc[q] = m0 + row < M ? (uint32_t)((m0 + row) * ldx2 + chunk * 16) : kOobOffset;
  }
  auto dma = [&](int step, int st) {
    const uint32_t at = lds0 + st * STAGE, k = (uint32_t)min(step, nk - 1) * (kPfBK * 2);
#pragma unroll
    for (int q = 0; q < XL; ++q) dma16(x_rs, at + (wv * XL + q) * 1024, xsrc[q], k);
  };

  // W: thread wq of the TPR of a row has its words wq * WPT ..
  const int wrow = tid / TPR, wq = tid % TPR;
  // merged gate_up: each wave's 64 columns are 32 gate rows and their up rows
  const int wcol = n0 + (GU ? (wrow >> 6) * 32 + (wrow & 31) : wrow);
  const bool w_in = wcol < NY;
  const int wn_row = wcol + (GU && (wrow & 32) ? NY : 0);
  const auto w_rs = make_rsrc(a.w, (uint32_t)((int64_t)N * KB));
  const uint32_t wsrc = w_in ? (uint32_t)(wn_row * KB + wq * (WPT * 4)) : kOobOffset;
  // its scale and zero point: byte offset of the row in a group's row of N,
  // and of the step's group.  Groups of 32 (gshift 0) put the two halves of a
  // step into different groups.
  const int64_t gb = (int64_t)a.G * N;
  const int se = a.s_dt == ZT_DT_F32 ? 4 : 2;
  const int ze = a.zp_dt == ZT_DT_F32 || a.zp_dt == ZT_DT_S32 ? 4 : a.zp_dt == ZT_DT_BF16 ? 2 : 1;
  const auto s_rs = make_rsrc(a.scales, (uint32_t)(gb * se));
  const auto z_rs = make_rsrc(a.zp, a.zp ? (uint32_t)(gb * ze) : 0u);
  const uint32_t sn = w_in ? (uint32_t)(wn_row + (gshift == 0 ? wq * WPT / 4 * N : 0)) : kOobOffset / 4;
  const int zmode = !a.zp ? 0 : (a.zp_dt == ZT_DT_F32 || a.zp_dt == ZT_DT_BF16) ? 1 : 2;
  // (steps past the last load the last one again, into places nothing reads)
  typedef unsigned words_t __attribute__((ext_vector_type(WPT)));
  auto load_w = [&](int step) {
    const int k = min(step, nk - 1) * (kPfBK / 2);
    if constexpr (WPT == 4)
      return __builtin_bit_cast(words_t, __builtin_amdgcn_raw_buffer_load_b128(w_rs, wsrc, k, 0));
    else
      return __builtin_bit_cast(words_t, __builtin_amdgcn_raw_buffer_load_b64(w_rs, wsrc, k, 0));
  };
  auto load_q = [&](int step) {
    const uint32_t g = (uint32_t)(((2 * min(step, nk - 1)) >> gshift) & gmask) * (uint32_t)N;
    return load_group<DQ>(a, s_rs, z_rs, sn, g);
  };
  const GroupFormat gf = group_format(a);
  const int wdst = BM * kPfRow + wrow * kPfRow;
  const int wswz = (wrow >> 1) & 7;
  auto put_w = [&](int st, int j, uint32_t word, GroupQ q) {
    *reinterpret_cast<u32x4_t *>(smem + st * STAGE + wdst +
                                 (((wq * WPT + j) ^ wswz) * 16)) = dequant8<DQ>(word, q, zmode);
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int fsw = (l32 >> 1) & 7;
  const int xrow = (wm * (BM / WM) + l32) * kPfRow;
  const int brow = (BM + wn * (BN / WN) + l32) * kPfRow;
  bf16x8_t xf[2][TM], wf[2][TN];
  auto read = [&](const unsigned char *stage, int sub, int buf) {
    const int pos = ((2 * sub + hl) ^ fsw) * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      wf[buf][j] = *reinterpret_cast<const bf16x8_t *>(stage + brow + j * 32 * kPfRow + pos);
#pragma unroll
    for (int i = 0; i < TM; ++i)
      xf[buf][i] = *reinterpret_cast<const bf16x8_t *>(stage + xrow + i * 32 * kPfRow + pos);
  };

  // Step ks computes on stage (ks - kb) & 1 while the dequantised weights of
  // step ks + 1 go into the other one.  The step's barrier stands before its
  // last sub-step: by then every wave holds the stage's last fragments in
  // registers, so behind it the stage takes the DMA of step ks + 2 and the
  // first fragments of step ks + 1 are read under the last MFMAs.  x and the
  // packed weights have one whole step to arrive.
  // Word j of a step's weights is dequantised in sub-step j - 1 of the step
  // before (word 0 in the last sub-step of the one before that), one word's
  // VALU work beside each sub-step's MFMAs.
  dma(kb, 0);
  words_t w = load_w(kb), wnext = load_w(kb + 1), wfar = load_w(kb + 2);
  GroupRaw qr = load_q(kb), qnext = load_q(kb + 1), qfar = load_q(kb + 2);
  {
    const GroupQ first = group_of<DQ>(gf, qr);
#pragma unroll
    for (int j = 0; j < WPT; ++j) put_w(0, j, w[j], first);
  }
  w = wnext, qr = qnext;
  wnext = wfar, qnext = qfar;
  GroupQ q = group_of<DQ>(gf, qr);
  put_w(1, 0, w[0], q);
  wait_step();
  // (opaque, so that the loop carries the loaded words as they are: as
  // 8- or 16-bit values it would extend them, and wait, at its top)
  asm volatile("" : "+v"(qnext.s), "+v"(qnext.z));
  dma(kb + 1, 1);
  // the epilogue's columns and their bias, loaded ahead of the main loop
  constexpr int SP = 64 + 4;            // slab pitch, floats
  constexpr int Q = GU ? 8 : 16;        // column quads of y per wave and row
  constexpr int RP = 64 / Q;            // rows per pass
  const int c4 = (lane % Q) * 4, r0 = lane / Q;
  const int n = n0 + wn * 4 * Q + c4;
  float bias[4] = {0.f, 0.f, 0.f, 0.f}, ubias[4] = {0.f, 0.f, 0.f, 0.f};
  if (a.bias && !partial)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < NY) {
        bias[r] = load_elem(a.bias, a.b_dt, n + r);
        if (GU) ubias[r] = load_elem(a.bias, a.b_dt, NY + n + r);
      }
  read(smem, 0, 0);
  int cur = 0;
  for (int ks = kb; ks < ke; ++ks, cur ^= 1) {
    const unsigned char *stage = smem + cur * STAGE;
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      if (sub < 3) {
        read(stage, sub + 1, (sub + 1) & 1);
        if (sub + 1 < WPT) put_w(cur ^ 1, sub + 1, w[sub + 1], q);
      } else {
        wait_step();
#pragma unroll
        for (int j = 0; j < WPT; ++j) w[j] = copy_now(wnext[j]);
        qr.s = copy_now(qnext.s);
        if (DQ != kDqS4) qr.z = copy_now(qnext.z);
        q = group_of<DQ>(gf, qr);
        __builtin_amdgcn_sched_barrier(0);
        read(smem + (cur ^ 1) * STAGE, 0, 0);
        dma(ks + 2, cur);
        wnext = load_w(ks + 3);
        qnext = load_q(ks + 3);
        put_w(cur, 0, w[0], q);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[sub & 1][j], xf[sub & 1][i],
                                                              acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  wait_step();

  // Epilogue, each wave by itself through a 32-row LDS slab of its own (D is
  // [n][m]: register r of lane l holds n = 8 (r / 4) + 4 (l / 32) + r % 4 and
  // m = l % 32; the slab turns it into rows of four columns per lane).  The
  // loops stay rolled: the code runs once per tile, and unrolled its
  // instruction fetches alone took 30 us.
  float *slab = reinterpret_cast<float *>(smem) + wv * (32 * SP);
  const bool has_bias = a.bias != nullptr;
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    const int mb = m0 + wm * (BM / WM) + i * 32;
    if (mb >= M) break;  // rows past M: nothing to store (few rows of a short K, last tiles)
#pragma unroll
    for (int ii = 0; ii < TM; ++ii)
      if (ii == i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4_t *>(slab + l32 * SP + j * 32 + 8 * r + 4 * hl) =
                f32x4_t{acc[ii][j][4 * r], acc[ii][j][4 * r + 1], acc[ii][j][4 * r + 2],
                        acc[ii][j][4 * r + 3]};
    __builtin_amdgcn_wave_barrier();
    if (GU || (a.post.count && !partial)) {
#pragma unroll GU ? 1 : 4
      for (int t = 0; t < 32 / RP; ++t) {
        float *at = slab + (t * RP + r0) * SP + c4;
        f32x4_t v = *reinterpret_cast<const f32x4_t *>(at);
        if (GU) {
          const f32x4_t u = *reinterpret_cast<const f32x4_t *>(at + 32);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float g = has_bias ? v[r] + bias[r] : v[r];
            float up = has_bias ? u[r] + ubias[r] : u[r];
            if (a.y_dt == ZT_DT_BF16) up = bf16_bits_to_f32(f32_to_bf16_bits(up));
            v[r] = unary_op(ZT_PO_SILU, g) * up;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = has_bias ? v[r] + bias[r] : v[r];
        }
        *reinterpret_cast<f32x4_t *>(at) = v;
      }
      if (!GU) post_ops_slab<32 / RP, RP>(slab, SP, c4, r0, a.post, mb, n, M, N);
    }
    if (partial) {  // rows of whole quads
#pragma unroll 4
      for (int t = 0; t < 32 / RP; ++t) {
        const int row = t * RP + r0, m = mb + row;
        if (m < M && n < N)
          *reinterpret_cast<f32x4_t *>(partial + ((size_t)blockIdx.y * M + m) * pf_pitch(N) + n) =
              *reinterpret_cast<const f32x4_t *>(slab + row * SP + c4);
      }
    } else {
      const bool add = has_bias && !GU && !a.post.count;
#pragma unroll 4
      for (int t = 0; t < 32 / RP; ++t) {
        const int row = t * RP + r0, m = mb + row;
        const f32x4_t v = *reinterpret_cast<const f32x4_t *>(slab + row * SP + c4);
        float f[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) f[r] = add ? v[r] + bias[r] : v[r];
        if (m < M && n < NY) store4(a.y, a.y_dt, a.ldy, m, n, NY, f);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int BM, int BN, int WM, int WN, bool GU>
hipError_t launch_pf(const WoqArgs &a, hipStream_t s, float *partial, int splits) {
  const int64_t ny = GU ? a.N / 2 : a.N;
  constexpr int CN = GU ? BN / 2 : BN;
  const int tiles_m = (int)((a.M + BM - 1) / BM), tiles_n = (int)((ny + CN - 1) / CN);
  const int group_m = tiles_m < 4 ? tiles_m : 4;
  int gshift = 31, gmask = 0;  // per channel
  if (a.G > 1) {
    gmask = 0x7fffffff;
    for (gshift = 0; ((int64_t)32 << gshift) < a.K / a.G;) ++gshift;
  }
  const int nk = (int)(a.K / kPfBK);
  const int sps = partial ? (nk + splits - 1) / splits : nk;
  const dim3 grid((unsigned)(tiles_m * tiles_n), partial ? (unsigned)splits : 1u);
  const dim3 block(64 * WM * WN);
  const bool bf16s = a.s_dt == ZT_DT_BF16;
  if (bf16s && !a.zp)
    woq_prefill_kernel<BM, BN, WM, WN, kDqS4, GU><<<grid, block, pf_lds<BM, BN>(), s>>>(
        a, tiles_m, tiles_n, group_m, gshift, gmask, partial, sps);
  else if (bf16s && (a.zp_dt == ZT_DT_S8 || a.zp_dt == ZT_DT_U8))
    woq_prefill_kernel<BM, BN, WM, WN, kDqU4, GU><<<grid, block, pf_lds<BM, BN>(), s>>>(
        a, tiles_m, tiles_n, group_m, gshift, gmask, partial, sps);
  else
    woq_prefill_kernel<BM, BN, WM, WN, kDqAny, GU><<<grid, block, pf_lds<BM, BN>(), s>>>(
        a, tiles_m, tiles_n, group_m, gshift, gmask, partial, sps);
  return hipGetLastError();
}

// y = epilogue of the sum of the K splits' partials, in split order, four
// columns per thread; every split's load is issued before the first add
// (the partials come from other XCDs, a round trip each).
template <int S>
__global__ __launch_bounds__(256) void woq_prefill_reduce_kernel(WoqArgs a, const float *partial,
                                                                 int splits) {
  const int64_t pitch = pf_pitch(a.N), quads = pitch / 4;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * quads) return;
  const int64_t m = idx / quads;
  const int n = (int)(idx - m * quads) * 4, N = (int)a.N;
  const float *p = partial + idx * 4;
  f32x4_t q[S];
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < splits) q[i] = *reinterpret_cast<const f32x4_t *>(p + i * a.M * pitch);
  f32x4_t v = q[0];
#pragma unroll
  for (int i = 1; i < S; ++i)
    if (i < splits) v += q[i];
  float f[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    f[r] = a.bias && n + r < N ? v[r] + load_elem(a.bias, a.b_dt, n + r) : v[r];
  post_ops4(f, a.post, m, n, N);
  store4(a.y, a.y_dt, a.ldy, m, n, N, f);
}

hipError_t launch_reduce(const WoqArgs &a, const float *partial, int splits, hipStream_t s) {
  const dim3 grid((unsigned)((a.M * (pf_pitch(a.N) / 4) + 255) / 256)), block(256);
  if (splits <= 2) woq_prefill_reduce_kernel<2><<<grid, block, 0, s>>>(a, partial, splits);
  else if (splits <= 4) woq_prefill_reduce_kernel<4><<<grid, block, 0, s>>>(a, partial, splits);
  else woq_prefill_reduce_kernel<8><<<grid, block, 0, s>>>(a, partial, splits);
  return hipGetLastError();
}

}  // namespace

bool woq_prefill_ok(const WoqArgs &a) {
  const int64_t gs = a.K / a.G, g32 = gs / 32;
  auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return a.x_dt == ZT_DT_BF16 && a.K % kPfBK == 0 && a.ldx % 8 == 0 && aligned16(a.x) &&
         aligned16(a.w) && (a.G == 1 || (gs % 32 == 0 && (g32 & (g32 - 1)) == 0)) &&
         a.M * a.ldx * 2 < (int64_t)kOobOffset && a.N * (a.K / 2) < (int64_t)kOobOffset &&
         a.G * a.N * 4 < (int64_t)kOobOffset;
}

// Tile and K split of least estimated time.  Against a sweep of both over
// 4096 x 4096, 6144 x 4096, 4096 x 14336, 28672 x 4096, 5120 x 5120 and
// 16384 x 3072 at 65 to 2048 rows the choice is the fastest one at 56 of 60
// points and within 5 % at the others; the time is 9 % below the previous
// kernels' on average there (4096 x 14336 at M = 777 149.5 -> 113 us,
// 28672 x 4096 at M = 65 65.8 -> 45.7, 4096 x 4096 at M = 2048 equal).
PrefillPlan woq_prefill_plan(int64_t M, int64_t N, int64_t K, bool gate_up) {
  PrefillPlan best{};
  if (M < 1 || N < 1 || K < kPfBK) return best;
  const char *e = knob(kKnobWoqGemm);
  const bool forced = e && e[0] == 'p' && e[1] >= '0' && e[1] <= '2';
  const int nk = (int)(K / kPfBK);
  // Splits: up to 8, but no more than woq_gemm_splits gives a shape it splits,
  // so that such a shape's workspace stays the size callers know it by.  (The
  // cap costs nothing: against up to 8 splits everywhere 9 shapes at 65 to 512 rows
  // run 1 % faster on average, 6144 x 4096 at M = 256 28.5 against 33.4 us, 2048 x
  // 2048 at M = 65 15.5 against 13.5.)
  const int known = woq_gemm_splits(M, N, K);
  const int most = gate_up ? 1 : forced || known < 2 ? 8 : known;
  static const int bm[3] = {128, 128, 256}, bn[3] = {128, 256, 256};
  for (int t = 0; t < 3; ++t) {
    if (forced && e[1] != '0' + t) continue;
    const int64_t tiles = ((M + bm[t] - 1) / bm[t]) * ((N + bn[t] - 1) / bn[t]);
    for (int sp = 1; sp <= most; ++sp) {
      if (sp > 1 && nk / sp < 4) break;
      if (forced && e[2] && !gate_up && std::atoi(e + 2) != sp) continue;
      const int sps = (nk + sp - 1) / sp;
      if ((nk + sps - 1) / sps != sp) continue;  // a split would be empty
      const int64_t wg = tiles * sp, slots = t == 0 ? 512 : 256;
      auto round = [&](int64_t w) {
        const double step = t == 0 ? (w <= 256 ? kPfStepFew[0] : kPfStepAll[0])
                                   : kPfStepFew[t] + (kPfStepAll[t] - kPfStepFew[t]) * w / 256;
        return kPfFixed[t] + sps * step;
      };
      double us = wg / slots * round(slots) + (wg % slots ? round(wg % slots) : 0.0);
      if (sp > 1) us += kPfReduce + (double)(2 * sp + 1) * M * N * 2 / kPfReduceRate;
      if (best.tile < 0 || us < best.us) best.tile = t, best.splits = sp, best.us = us;
    }
  }
  return best;
}

// Both sides from graph replays at 17 to 64 rows of 28 shapes, 256 x 256 to
// 28672 x 4096 (bf16 zero points; fp32 scales; 8-bit zero points where N % 4
// keeps the wide kernel away), those of fp32 scales fitted again over 18 shapes at 17
// to 40 rows.  The choice is the faster one, or within 2 %, at 422 of 427 points of the
// first and within 5 % at those of the second past K = 704; 17 x 4096 x 4096 took 22.3 / 23.6 us (zero points /
// fp32 scales) here against 14.4 / 13.0 in blocks, 64 x 4096 x 4096 24 / 25 against 31 /
// 28, 24 x 18944 x 3584 35 / 40 against 70 / 54, 20 x 4096 x 14336 with fp32 scales 44
// against 39.
bool woq_prefill_beats_row_blocks(const WoqArgs &a) {
  const PrefillPlan p = woq_prefill_plan(a.M, a.N, a.K, false);
  const double plan = p.us;
  const bool f32 = a.s_dt == ZT_DT_F32;
  // (the plan's constants are those of the two one-FMA dequantisations)
  const double here = f32                                               ? 1.35 * plan + 0.0002 * a.K
                      : a.zp_dt == ZT_DT_S8 || a.zp_dt == ZT_DT_U8 ? 0.9 * plan
                                                                        : 1.13 * plan + 1.6;
  // (unsplit, in few waves: post-ops past one relu or operand, 5 us of 512 x 1000 at M =
  // 48, and columns that are not whole quads and are stored one by one)
  const double epilogue =
      p.splits > 1 ? 0.0
                   : (double)a.M * ((a.N % 4 ? 0.045 : 0.0) + (long_post_ops(a.post) ? 0.1 : 0.0));
  // a round of 256 row tiles of 16, x whole in LDS (stream kernel) or not
  const double k = (double)a.K;
  const double round =
      16 * (a.K + 8) * 2 <= 160 * 1024
          ? std::min(0.7 + 0.0035 * k, f32 ? 2.7 + 0.00045 * k : 2.5 + 0.0007 * k)
          : (f32 ? 0.0014 : 0.0016) * k;
  const int64_t rounds = ((a.N + 15) / 16 + 255) / 256, blocks = (a.M + 15) / 16;
  const double last = 0.6 + 0.4 / 16 * (double)(a.M - 16 * (blocks - 1));
  return here + epilogue < (3.0 + rounds * round) * (blocks - 1 + last);
}

size_t woq_prefill_workspace(int64_t M, int64_t N, int64_t K) {
  const PrefillPlan p = woq_prefill_plan(M, N, K, false);
  return p.splits > 1 ? (size_t)p.splits * (size_t)M * (size_t)pf_pitch(N) * sizeof(float) : 0;
}

hipError_t launch_woq_prefill(const WoqArgs &a, bool gate_up, void *workspace,
                              size_t workspace_bytes, hipStream_t s) {
  const PrefillPlan p = woq_prefill_plan(a.M, a.N, a.K, gate_up);
  float *partial = nullptr;
  if (p.splits > 1 && workspace && workspace_bytes >= woq_prefill_workspace(a.M, a.N, a.K) &&
      (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0)
    partial = static_cast<float *>(workspace);
  const int sp = partial ? p.splits : 1;
  if (knob(kKnobWoqDebug))
    std::fprintf(stderr, "[zt] woq prefill M=%lld N=%lld K=%lld: tile %d, %d K splits%s\n",
                 (long long)a.M, (long long)a.N, (long long)a.K, p.tile, sp,
                 gate_up ? ", gate_up" : "");
  if (gate_up) {
    if (p.tile == 2) return launch_pf<256, 256, 2, 4, true>(a, s, nullptr, 1);
    if (p.tile == 1) return launch_pf<128, 256, 2, 4, true>(a, s, nullptr, 1);
    return launch_pf<128, 128, 2, 2, true>(a, s, nullptr, 1);
  }
  const hipError_t err = p.tile == 2   ? launch_pf<256, 256, 2, 4, false>(a, s, partial, sp)
                         : p.tile == 1 ? launch_pf<128, 256, 2, 4, false>(a, s, partial, sp)
                                       : launch_pf<128, 128, 2, 2, false>(a, s, partial, sp);
  if (err != hipSuccess || !partial) return err;
  return launch_reduce(a, partial, sp, s);
}

}  // namespace zt
