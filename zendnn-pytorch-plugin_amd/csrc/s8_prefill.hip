// Large-tile int8 GEMM for gfx950: the dynamic and static int8 linears past
// 128 tokens.
#include <cstdio>

#include "s8_epilogue.hpp"
#include "zt_gemm_tile.hpp"
#include "zt_launch.hpp"
#include "zt_tuning.hpp"

namespace zt {

namespace {

constexpr int kPqBK = 128;   // k, and bytes of an LDS row, per step

// two stages of x and W rows
template <int BM, int BN>
constexpr size_t pq_lds() {
  return 2 * (size_t)(BM + BN) * kPqBK;
}

// y tile of BM x BN on v_mfma_i32_32x32x32_i8, WM x WN waves of 128 x 64, K in
// steps of 128 over two LDS stages of 128-byte x and W rows, both moved by DMA.
// A = W, B = x: D is [n][m].  Exact int32 sums.
//
// Bound: per step 2048 clocks of MFMAs beside 2048 of LDS traffic (192 KB of
// fragments read, 64 KB written), and the chip's power: MFMAs fed from LDS
// sustain 3.0 POP/s on random bytes (4.4 on zeros).  Quantisation included,
// 28672 x 4096 at M = 4096 takes 478 us (2.0 POP/s, 555 on 256 x 128 tiles),
// 14336 x 4096 at M = 2048 140 (160), 4096 x 14336 at M = 4096 230 (258), 4096 x 4096 at
// M = 4096 79 (91).  256 x 192 tiles on six waves were no faster than these, 128 x
// 256 in three stages than the load-wave kernel's 256 x 128.
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2, 2)))
void s8_prefill_kernel(DynArgs a, int tiles_m, int tiles_n, int group_m) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // 32 x 32 tiles per wave
  constexpr int STAGE = (BM + BN) * kPqBK;
  constexpr int LPW = (BM + BN) / 8 / NW;  // 1 KB loads (8 rows) per wave and step
  static_assert(TN == 2 && BM % 64 == 0 && LPW * NW * 8 == BM + BN, "tile shape");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / WN, wn = wv % WN;
  const int hl = lane >> 5, l32 = lane & 31;
  int tm, tn;
  grouped_tile(blockIdx.x, tiles_m, tiles_n, group_m, tm, tn);
  const int M = (int)a.M, N = (int)a.N, K = (int)a.K;
  const int m0 = tm * BM, n0 = tn * BN;
  const int nk = (K + kPqBK - 1) / kPqBK;

  // rows of the [x | W] slab, 8 per load, 16-byte chunk c of row r at
  // c ^ ((r >> 1) & 7); a load lies wholly in x or in W
  const i32x4_t x_rs = dma_rsrc(a.qx, (uint32_t)((int64_t)M * K));
  const i32x4_t w_rs = dma_rsrc(a.w, (uint32_t)((int64_t)N * K));
  const uint32_t lds0 = lds_address(smem);
  uint32_t src[LPW];
  const int chunk = (lane & 7) ^ ((wv * 4 + (lane >> 4)) & 7);  // of all its rows
  static_assert(NW % 2 == 0, "the chunk of load q does not depend on q");
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int row = (q * NW + wv) * 8 + (lane >> 3);
    const int at = row < BM ? m0 + row : n0 + row - BM;
    src[q] = at < (row < BM ? M : N) ? (uint32_t)(at * K + chunk * 16) : kOobOffset;
  }
  // K % 16 == 0: a 16-byte chunk lies wholly inside or past its row; past it
  // in the last step's load the lane reads zeros
  const uint32_t past = K % kPqBK && (nk - 1) * kPqBK + chunk * 16 >= K ? kOobOffset : 0u;
  auto dma = [&](int step, int st, int q) {
    const uint32_t at = lds0 + st * STAGE, k = (uint32_t)min(step, nk - 1) * kPqBK;
    const uint32_t cut = step == nk - 1 ? past : 0u;
    const int li = q * NW + wv;
    dma16(li * 8 < BM ? x_rs : w_rs, at + li * 1024, src[q] | cut, k);
  };

  i32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  const int fsw = (l32 >> 1) & 7;
  const int xrow = (wm * (BM / WM) + l32) * kPqBK;
  const int brow = (BM + wn * (BN / WN) + l32) * kPqBK;
  i32x4_t xf[2][TM], wf[2][TN];
  auto read = [&](int st, int sub, int buf) {
    const unsigned char *stage = smem + st * STAGE;
    const int pos = ((2 * sub + hl) ^ fsw) * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      wf[buf][j] = *reinterpret_cast<const i32x4_t *>(stage + brow + j * 32 * kPqBK + pos);
#pragma unroll
    for (int i = 0; i < TM; ++i)
      xf[buf][i] = *reinterpret_cast<const i32x4_t *>(stage + xrow + i * 32 * kPqBK + pos);
  };

  // As woq_prefill_kernel: the step's barrier stands before its last
  // sub-step, whose fragments every wave then holds, so the stage takes the
  // DMA of step ks + 2 behind it and the next step's first fragments are read
  // under the last MFMAs.
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < LPW; ++q) dma(p, p, q);
  wait_loads<LPW>();
  // the epilogue's row scales and offsets: rows lane and lane + 64 of the
  // wave's, and its columns',
  // loaded ahead of the main loop
  float row_sx[BM / WM / 64];
  int32_t row_azp[BM / WM / 64];
#pragma unroll
  for (int p = 0; p < BM / WM / 64; ++p) {
    const int m = min(m0 + wm * (BM / WM) + p * 64 + lane, M - 1);
    row_sx[p] = a.sx ? a.sx[m] : 0.f;
    row_azp[p] = a.azp ? a.azp[m] : 0;
  }
  const int c4 = (lane % 16) * 4, r0 = lane / 16;
  const int n = n0 + wn * 64 + c4;
  QuadScales qs;
  qs.load(a, n, N);

  read(0, 0, 0);
  int cur = 0;
  for (int ks = 0; ks < nk; ++ks) {
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      if (sub < 3) {
        read(cur, sub + 1, (sub + 1) & 1);
      } else {
        wait_step();
        read(cur ^ 1, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        // the stage's refill, one load after each MFMA pair's first: a load
        // the buffer unit cannot take yet holds up what is behind it
        if (sub == 3)
#pragma unroll
          for (int q = i * LPW / TM; q < (i + 1) * LPW / TM; ++q) dma(ks + 2, cur, q);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[sub & 1][j], xf[sub & 1][i],
                                                            acc[i][j], 0, 0, 0);
        if (sub == 3) __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    cur ^= 1;
  }
  wait_step();

  // epilogue: as woq_prefill_kernel's, each wave through a slab of its own,
  // the row scales and offsets of its rows beside it (a load per row and pass
  // would be a round trip each)
  constexpr int SP = 64 + 4, WR = BM / WM;
  int32_t *slab = reinterpret_cast<int32_t *>(smem) + wv * (32 * SP + 2 * WR);
  float *fslab = reinterpret_cast<float *>(slab);
  float *sx_l = fslab + 32 * SP;
  int32_t *azp_l = slab + 32 * SP + WR;
#pragma unroll
  for (int p = 0; p < WR / 64; ++p) {
    sx_l[p * 64 + lane] = row_sx[p];
    azp_l[p * 64 + lane] = row_azp[p];
  }
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    const int mb = m0 + wm * WR + i * 32;
    if (mb >= M) break;  // rows past M: nothing to store
#pragma unroll
    for (int ii = 0; ii < TM; ++ii)
      if (ii == i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            *reinterpret_cast<i32x4_t *>(slab + l32 * SP + j * 32 + 8 * r + 4 * hl) =
                i32x4_t{acc[ii][j][4 * r], acc[ii][j][4 * r + 1], acc[ii][j][4 * r + 2],
                        acc[ii][j][4 * r + 3]};
    __builtin_amdgcn_wave_barrier();
    auto sums = [&](int t) {
      return *reinterpret_cast<const i32x4_t *>(slab + (t * 4 + r0) * SP + c4);
    };
    if (a.y_dt == ZT_DT_S32) {
#pragma unroll 4
      for (int t = 0; t < 8; ++t) {
        const int row = t * 4 + r0, m = mb + row;
        const i32x4_t v = sums(t);
        if (m < M && n < N) store_sums4(a, m, n, N, qs.correct(v, azp_l[i * 32 + row]));
      }
    } else if (at_most_relu(a.post)) {
#pragma unroll 4
      for (int t = 0; t < 8; ++t) {
        const int row = t * 4 + r0, m = mb + row;
        float f[4];
        qs.scale(qs.correct(sums(t), azp_l[i * 32 + row]), sx_l[i * 32 + row], f);
        if (m < M && n < N) store_y4(a, qs, m, n, N, f, a.post.count != 0);
      }
    } else {
#pragma unroll 4
      for (int t = 0; t < 8; ++t) {
        const int row = t * 4 + r0;
        float f[4];
        qs.scale(qs.correct(sums(t), azp_l[i * 32 + row]), sx_l[i * 32 + row], f);
        *reinterpret_cast<f32x4_t *>(fslab + row * SP + c4) = f32x4_t{f[0], f[1], f[2], f[3]};
      }
      post_ops_slab<8, 4>(fslab, SP, c4, r0, a.post, mb, n, M, N);
#pragma unroll 4
      for (int t = 0; t < 8; ++t) {
        const int row = t * 4 + r0, m = mb + row;
        const f32x4_t v = *reinterpret_cast<const f32x4_t *>(fslab + row * SP + c4);
        float f[4] = {v[0], v[1], v[2], v[3]};
        if (m < M && n < N) store_y4(a, qs, m, n, N, f, false);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Estimated microseconds of the 256 x 256 tile here and of the 256 x 128 tile
// of s8_gemm_ws_kernel: per round of tiles, a prologue and epilogue and the
// 128-k steps, whose time grows with the CUs that are busy.
double rounds_us(int64_t wg, int64_t nk, double fixed, double few, double all) {
  const int64_t rest = wg % 256;
  return wg / 256 * (fixed + nk * all) + (rest ? fixed + nk * (few + (all - few) * rest / 256) : 0.0);
}

}  // namespace

// (constants from graph replays of both kernels at 2743 shapes of 129 to 4096 rows,
// K 192 to 18944: the choice is the faster kernel or within 3 % at all but 1 % of
// those outside the 192 zone below, at most 10 % behind in it.  A tile's fixed cost
// fitted to K >= 1024 only, 11 and 8 us, took 256 x 256 tiles for few k steps and a
// nearly empty last round: 16460 x 784 at M = 1023 53 us against 45.  Post-ops and
// requantised outputs lengthen the other kernel's epilogue by more.)
bool s8_prefill_better(const DynArgs &a) {
  const char *e = knob(kKnobS8Kind);
  if (e) return e[0] == 'p';
  const int64_t nk = (a.K + kPqBK - 1) / kPqBK, tm = (a.M + 255) / 256;
  const bool floats = a.y_dt == ZT_DT_BF16 || a.y_dt == ZT_DT_F32;
  // The load-wave kernel's 256 x 192 tiles where they make one round and its
  // 256 x 128 do not: ahead up to K = 4096 (quantisation included, M = 2048: 6144 x 2048
  // 42.4 against 43.3 us, 5120 x 4096 59.7 against 61.1), behind at most shapes past it
  // (5120 x 5120 81.0 against 75.3, 6144 x 8192 120.7 against 118).  That tile's epilogue
  // takes post-ops and requantised outputs quad by quad (s8_tile_epilogue): with any of
  // them it was behind at all 267 shapes (4096 x 1024 at M = 2520 with an add 83
  // us against 37, 14420 x 736 at M = 601 to u8 78 against 29).
  if (tm * ((a.N + 127) / 128) > 256 && tm * ((a.N + 191) / 192) <= 256)
    return a.K > 4096 || a.post.count || !floats;
  const double fixed = at_most_relu(a.post) && floats ? 14.2 : 12.0;
  return rounds_us(tm * ((a.N + 255) / 256), nk, fixed, 1.10, 1.80) <
         rounds_us(tm * ((a.N + 127) / 128), nk, 7.1, 0.56, 1.07);
}

hipError_t launch_s8_prefill(const DynArgs &a, hipStream_t s) {
  constexpr int BM = 256, BN = 256;
  const int tiles_m = (int)((a.M + BM - 1) / BM), tiles_n = (int)((a.N + BN - 1) / BN);
  if (knob(kKnobWoqDebug))
    std::fprintf(stderr, "[zt] s8 prefill M=%lld N=%lld K=%lld\n", (long long)a.M, (long long)a.N,
                 (long long)a.K);
  s8_prefill_kernel<BM, BN, 2, 4><<<dim3((unsigned)(tiles_m * tiles_n)), dim3(512),
                                    pq_lds<BM, BN>(), s>>>(a, tiles_m, tiles_n,
                                                           tiles_m < 4 ? tiles_m : 4);
  return hipGetLastError();
}

}  // namespace zt
