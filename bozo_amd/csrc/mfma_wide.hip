// bf16 MFMA kernels of local windows wider than one 64-row tile (head dim 64,
// no bias, tau or dTau): the global block's layout (mfma_global.hip) over a
// band.  A workgroup owns a 64-row tile and streams the 64-row blocks of its
// band through an LDS ring (global_load_lds); wave (w & 1, w >> 1) takes
// 32 of the tile's rows against 32 rows of every block, so a fragment read from
// LDS feeds two MFMAs (the split kernels' 16-row waves read twice the LDS per
// MFMA and stage through registers); the two halves of a row meet once, through
// LDS, at the end.  Only the blocks that cross a band edge are masked, and a
// wave skips the 32 x 32 quarters that lie outside.
//
// A masked pair enters the second products as weight 0 times its row, so an
// infinity or NaN in that row would reach the result.  Products are left out 16
// result rows x 32 summed rows at a time where no pair of the group lies on the
// band, the same groups as in the split kernels: a non-finite row reaches the
// result rows it has a pair with and those that share such a group with it.
//
// Bound by each workgroup's own latencies (first loads, five dependent blocks at
// W = 256, the merge) at two or three workgroups per CU, over an HBM floor of 13
// to 20 us.  B8 H16 T1024 W256, valid count, sustained (split kernels -> these):
// forward 28.1 -> 25.1 us, dQ 33.8 -> 35.5, dK / dV 49.5 -> 45.7.  Which calls
// take them, phase by phase: wide_from in capi.hip; forward + backward of that
// call, with dQ on the split kernels, 106.5 -> 104.8 us.
#include <type_traits>

#include "mfma_common.h"

namespace tension {
namespace {

// No pair of NQ queries from qa and NK keys from ka on the band (query t sees
// keys t - W .. t - 1).  In a 32 x 32 quarter that has pairs, 16 rows without any
// can only lie past the band's far edge: the later queries, or the earlier keys.
template <int NQ, int NK>
__device__ __forceinline__ bool pairs_out(int qa, int ka, int W) {
  return ka > qa + NQ - 2 || ka + NK - 1 < qa - W;
}

__device__ __forceinline__ bool pair_on(int q, int k, int W) { return k < q && k >= q - W; }

struct Range {
  int first, n;
};

// Key blocks of query tile `tile`, and query blocks of key tile `tile`.
__device__ __forceinline__ Range key_blocks(const BandParams& p, int tile) {
  const int lo = tile * kTile - p.win;
  const int first = lo > 0 ? lo >> 6 : 0;
  return {first, tile - first + 1};
}

__device__ __forceinline__ Range query_blocks(const BandParams& p, int tile) {
  // keys of the tile reach queries up to its last key + W (win < 2^30)
  const int64_t hi = ((int64_t)tile * kTile + kTile - 1 + p.win) >> 6;
  const int last = hi < p.ntiles - 1 ? (int)hi : p.ntiles - 1;
  return {tile, last - tile + 1};
}

__device__ __forceinline__ float count_norm(int t, int W) {
  const int n = t < W ? t : W;
  return 1.f / (float)(n > 1 ? n : 1);
}

constexpr int kRing = 3;  // ring slots

// A ring over blocks [first, first + n) of two tensors (slot s: lds[s] and
// lds[kRing + s]): body(block, slot) once per block.  One barrier per block:
// past it every wave has left block i - 1, whose slot takes block i + kRing - 1.
// Every copy past the last block is clamped to it, so each wait leaves exactly
// kRing - 2 blocks' copies in flight: 4 instructions each, and the NX that
// extra(block, slot) adds.  The caller owns the LDS at entry and exit.  (Two
// slots with two barriers per block: 2 to 4% slower in each kernel; four slots
// cost the forward a workgroup per CU, 36 against 29 us, and gain nothing in
// the others.)
template <int NX, typename Extra, typename Body>
__device__ __forceinline__ void ring(const TileSrc& a, const TileSrc& b, const Range& r, bf16 (*lds)[kDTile], int wave,
                                     Extra extra, Body body) {
  const int last = r.first + r.n - 1;
  auto copy = [&](int blk, int slot) __attribute__((always_inline)) {
    blk = blk < last ? blk : last;
    tile_async_src(a, blk * kTile, lds[slot], wave);
    tile_async_src(b, blk * kTile, lds[kRing + slot], wave);
    extra(blk, slot);
  };
#pragma unroll
  for (int i = 0; i + 1 < kRing; ++i) copy(r.first + i, i);
  int slot = 0, free = kRing - 1;
  for (int i = 0; i < r.n; ++i) {
    wait_vm<(4 + NX) * (kRing - 2)>();
    lds_barrier();
    copy(r.first + i + kRing - 1, free);
    body(r.first + i, slot);
    free = slot;
    slot = slot + 1 < kRing ? slot + 1 : 0;
  }
  wait_vm<0>();
  __syncthreads();
}

// S^T and, with V rows, dP^T of a wave's 32 keys (rows krow..) x 32 queries.
__device__ __forceinline__ void product32(const bf16* tile, int row0, const bf16x8 (*f)[2], int g, int c,
                                          f32x4 (*s)[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const bf16x8 a0 = dt_row8(tile, row0 + 16 * j + c, g), a1 = dt_row8(tile, row0 + 16 * j + c, 4 + g);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      f32x4 z = {};
      z = mfma(a0, f[i][0], z);
      s[i][j] = mfma(a1, f[i][1], z);
    }
  }
}

// The half of a wave pair's sums that the partner keeps goes through LDS: wave
// (own, other) keeps row tile i = other and hands tile 1 - other over.
template <int N>
__device__ __forceinline__ void meet(float* red, int own, int other, int lane, const float (*x)[N], float* mine) {
  float* dst = red + (2 * own + other) * N * 64 + lane;
#pragma unroll
  for (int e = 0; e < N; ++e) dst[e * 64] = other == 0 ? x[1][e] : x[0][e];
  __syncthreads();
  const float* src = red + (2 * own + (1 - other)) * N * 64 + lane;
#pragma unroll
  for (int e = 0; e < N; ++e) mine[e] = (other == 0 ? x[0][e] : x[1][e]) + src[e * 64];
  __syncthreads();
}

}  // namespace

template <int NORM>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3, 8))) void wl_fwd(BandArgs args) {
  touch_args(args);
  const BandParams p = band_params(args);
  __shared__ __attribute__((aligned(16))) bf16 lds[2 * kRing][kDTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15, qh = wave & 1, kh = wave >> 1;
  const TileId id = tile_id(p, false);
  const int b = id.b, h = id.h, T = p.T, W = p.win, t0 = id.tile * kTile, qa = t0 + 32 * qh;

  const bf16* qb = (const bf16*)p.q.p + b * p.q.s0 + h * p.q.s2;
  bf16x8 qf[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) load_qfrag(qb, p.q.s1, qa + 16 * i + c, T, g, qf[i]);
  const TileSrc ks = tile_src((const bf16*)p.k.p + b * p.k.s0 + h * p.k.s2, p.k.s1, T, wave, lane);
  const TileSrc vs = tile_src((const bf16*)p.v.p + b * p.v.s0 + h * p.v.s2, p.v.s1, T, wave, lane);
  const float k2 = -kLog2e * (float)(1.0 / p.scale);
  f32x4 acc[2][4] = {};
  float msum[2] = {0.f, 0.f};

  auto block = [&](const bf16* Ks, const bf16* Vs, int ka, auto mask_tag) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_tag)::value;
    f32x4 s[2][2];
    product32(Ks, 32 * kh, qf, g, c, s);
    TrRead vr[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) vr[m] = dt_tr8_issue(Vs, m, 32 * kh, g, c);
    bf16x8 vt[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (MASK && i == 1 && pairs_out<16, 32>(qa + 16, ka, W)) break;
      float pr[2][4];
      const int q = qa + 16 * i + c;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[i][j][r] * k2));
          pr[j][r] = !MASK || pair_on(q, ka + 16 * j + 4 * g + r, W) ? x : 0.f;
          if (NORM == NORM_MASS_) msum[i] += pr[j][r];
        }
      const bf16x8 pb = pack_b(pr[0], pr[1]);
      if (i == 0) {
        tr_wait4(vr);
#pragma unroll
        for (int m = 0; m < 4; ++m) vt[m] = tr_join(vr[m]);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[i][m] = mfma(vt[m], pb, acc[i][m]);
    }
  };
  ring<0>(ks, vs, key_blocks(p, id.tile), lds, wave, [](int, int) {}, [&](int blk, int slot) __attribute__((always_inline)) {
    const int ka = blk * kTile + 32 * kh;
    if (pairs_out<32, 32>(qa, ka, W)) return;
    if (ka + 31 < qa && ka >= qa + 31 - W) block(lds[slot], lds[kRing + slot], ka, std::false_type{});
    else block(lds[slot], lds[kRing + slot], ka, std::true_type{});
  });

  // 16 features and the mass per lane
  float x[2][17], o[17];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) x[i][e] = acc[i][e >> 2][e & 3];
    x[i][16] = NORM == NORM_MASS_ ? wave_sum_g(msum[i]) : 0.f;
  }
  meet<17>((float*)&lds[0][0], qh, kh, lane, x, o);
  const int r0 = qa + 16 * kh, tq = r0 + c;  // the wave's rows
  f32x4 of[4];
#pragma unroll
  for (int e = 0; e < 16; ++e) of[e >> 2][e & 3] = o[e];
  const float f = NORM == NORM_MASS_ ? 1.f / (o[16] > kMassEps ? o[16] : kMassEps)
                  : NORM == NORM_COUNT_ ? count_norm(tq, W)
                                        : 1.f;
  store_rows_staged((bf16*)p.out.p + b * p.out.s0 + (int64_t)r0 * p.out.s1 + h * p.out.s2, p.out.s1, T - r0, of, f, g,
                    c, lane, &lds[0][0] + wave * (16 * kTile));
  if (NORM == NORM_MASS_ && p.mass.p && tq < T && g == 0)
    st<float>(p.mass, b * p.mass.s0 + (int64_t)tq * p.mass.s1 + h * p.mass.s2, o[16]);
}

// dQ; with tau mass a first pass over the band forms a_t = 1 / m_t and
// c_t = sum P dP / m_t^2 in float32 (they also go to the workspace for wl_dkv).
template <int NORM>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 8))) void wl_dq(BandArgs args) {
  touch_args(args);
  const BandParams p = band_params(args);
  __shared__ __attribute__((aligned(16))) bf16 lds[2 * kRing][kDTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15, qh = wave & 1, kh = wave >> 1;
  const TileId id = tile_id(p, false);
  const int b = id.b, h = id.h, T = p.T, W = p.win, t0 = id.tile * kTile, qa = t0 + 32 * qh;

  const bf16* qb = (const bf16*)p.q.p + b * p.q.s0 + h * p.q.s2;
  const bf16* gb = (const bf16*)p.dout.p + b * p.dout.s0 + h * p.dout.s2;
  bf16x8 qf[2][2], gf[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    load_qfrag(qb, p.q.s1, qa + 16 * i + c, T, g, qf[i]);
    load_qfrag(gb, p.dout.s1, qa + 16 * i + c, T, g, gf[i]);
  }
  const TileSrc ks = tile_src((const bf16*)p.k.p + b * p.k.s0 + h * p.k.s2, p.k.s1, T, wave, lane);
  const TileSrc vs = tile_src((const bf16*)p.v.p + b * p.v.s0 + h * p.v.s2, p.v.s1, T, wave, lane);
  const float k2 = -kLog2e * (float)(1.0 / p.scale);
  const Range kr = key_blocks(p, id.tile);
  float ca[2] = {1.f, 1.f}, cc[2] = {0.f, 0.f};
  if (NORM == NORM_COUNT_) {
    ca[0] = count_norm(qa + c, W);
    ca[1] = count_norm(qa + 16 + c, W);
  }
  auto each = [&](auto body) __attribute__((always_inline)) {
    ring<0>(ks, vs, kr, lds, wave, [](int, int) {}, [&](int blk, int slot) __attribute__((always_inline)) {
      const int ka = blk * kTile + 32 * kh;
      if (pairs_out<32, 32>(qa, ka, W)) return;
      if (ka + 31 < qa && ka >= qa + 31 - W) body(lds[slot], lds[kRing + slot], ka, std::false_type{});
      else body(lds[slot], lds[kRing + slot], ka, std::true_type{});
    });
  };
  if constexpr (NORM == NORM_MASS_) {
    float sums[2][2] = {};  // [query tile][mass, sum P dP]
    each([&](const bf16* Ks, const bf16* Vs, int ka, auto mask_tag) __attribute__((always_inline)) {
      constexpr bool MASK = decltype(mask_tag)::value;
      f32x4 s[2][2], dp[2][2];
      product32(Ks, 32 * kh, qf, g, c, s);
      product32(Vs, 32 * kh, gf, g, c, dp);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool on = !MASK || pair_on(qa + 16 * i + c, ka + 16 * j + 4 * g + r, W);
            const float x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[i][j][r] * k2));
            const float pv = on ? x : 0.f;
            sums[i][0] += pv;
            sums[i][1] = fmaf(pv, on ? dp[i][j][r] : 0.f, sums[i][1]);
          }
    });
    // the key halves' sums meet: every wave needs both of its query tiles
    float* red = (float*)&lds[0][0];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        sums[i][e] = wave_sum_g(sums[i][e]);
        red[(wave * 4 + 2 * i + e) * 64 + lane] = sums[i][e];
      }
    __syncthreads();
    const int64_t nws = (int64_t)p.B * T * p.H;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float* o = red + ((wave ^ 2) * 4 + 2 * i) * 64 + lane;
      const float m = sums[i][0] + o[0], d = sums[i][1] + o[64];
      ca[i] = 1.f / (m > kMassEps ? m : kMassEps);
      cc[i] = m >= kMassEps ? d * ca[i] * ca[i] : 0.f;
      const int tq = qa + 16 * i + c;
      if (kh == 0 && g == 0 && tq < T) {
        const int64_t wi = ((int64_t)b * T + tq) * p.H + h;
        ((float*)p.ws)[wi] = ca[i];
        ((float*)p.ws)[nws + wi] = cc[i];
      }
    }
    __syncthreads();  // the ring takes the LDS back
  }

  f32x4 acc[2][4] = {};
  each([&](const bf16* Ks, const bf16* Vs, int ka, auto mask_tag) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_tag)::value;
    f32x4 s[2][2], dp[2][2];
    product32(Ks, 32 * kh, qf, g, c, s);
    product32(Vs, 32 * kh, gf, g, c, dp);
    TrRead kt_[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) kt_[m] = dt_tr8_issue(Ks, m, 32 * kh, g, c);
    bf16x8 kt[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (MASK && i == 1 && pairs_out<16, 32>(qa + 16, ka, W)) break;
      float gd[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[i][j][r] * k2));
          const float gv = (NORM == NORM_RAW ? dp[i][j][r] : fmaf(dp[i][j][r], ca[i], -cc[i])) * (x - x * x);
          gd[j][r] = !MASK || pair_on(qa + 16 * i + c, ka + 16 * j + 4 * g + r, W) ? gv : 0.f;
        }
      const bf16x8 pb = pack_b(gd[0], gd[1]);
      if (i == 0) {
        tr_wait4(kt_);
#pragma unroll
        for (int m = 0; m < 4; ++m) kt[m] = tr_join(kt_[m]);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[i][m] = mfma(kt[m], pb, acc[i][m]);
    }
  });

  float x[2][16], o[16];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) x[i][e] = acc[i][e >> 2][e & 3];
  meet<16>((float*)&lds[0][0], qh, kh, lane, x, o);
  f32x4 of[4];
#pragma unroll
  for (int e = 0; e < 16; ++e) of[e >> 2][e & 3] = o[e];
  const int r0 = qa + 16 * kh;
  store_rows_staged((bf16*)p.dq.p + b * p.dq.s0 + (int64_t)r0 * p.dq.s1 + h * p.dq.s2, p.dq.s1, T - r0, of,
                    (float)(1.0 / p.scale), g, c, lane, &lds[0][0] + wave * (16 * kTile));
}

// dK / dV: key-centric, wave (kh = w & 1, qh = w >> 1); the queries' a_t / c_t
// pass through the LDS ring with the Q / dO rows.
template <int NORM>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 8))) void wl_dkv(BandArgs args) {
  touch_args(args);
  const BandParams p = band_params(args);
  // one LDS object (see gl_dkv): the ring, then coef[slot][a, c][query]
  __shared__ __attribute__((aligned(16))) bf16 lds[2 * kRing * kDTile + (NORM == NORM_RAW ? 0 : 4 * kRing * kTile)];
  float(*coef)[2][kTile] = (float(*)[2][kTile])(lds + 2 * kRing * kDTile);
  bf16(*tiles)[kDTile] = (bf16(*)[kDTile])lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15, kh = wave & 1, qh = wave >> 1;
  const TileId id = tile_id(p, false);
  const int b = id.b, h = id.h, T = p.T, W = p.win, k0 = id.tile * kTile, ka = k0 + 32 * kh;

  const bf16* kb = (const bf16*)p.k.p + b * p.k.s0 + h * p.k.s2;
  const bf16* vb = (const bf16*)p.v.p + b * p.v.s0 + h * p.v.s2;
  bf16x8 kf[2][2], vf[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    load_qfrag(kb, p.k.s1, ka + 16 * i + c, T, g, kf[i]);
    load_qfrag(vb, p.v.s1, ka + 16 * i + c, T, g, vf[i]);
  }
  const TileSrc qs = tile_src((const bf16*)p.q.p + b * p.q.s0 + h * p.q.s2, p.q.s1, T, wave, lane);
  const TileSrc gs = tile_src((const bf16*)p.dout.p + b * p.dout.s0 + h * p.dout.s2, p.dout.s1, T, wave, lane);
  const Range qr = query_blocks(p, id.tile);
  const float k2 = -kLog2e * (float)(1.0 / p.scale);
  f32x4 dk[2][4] = {}, dv[2][4] = {};

  // a (waves 0, 2) or c (1, 3) of query block qb, one query per lane, by DMA with
  // the block's rows (a load of its own would be waited for in order, behind
  // the copies ahead of it); rows past T read T - 1's (their pairs are masked).
  // Valid count: computed.
  auto coef_copy = [&](int qb, int slot) __attribute__((always_inline)) {
    int t = qb * kTile + lane;
    t = t < T ? t : T - 1;
    if constexpr (NORM == NORM_MASS_) {
      const int64_t nws = (int64_t)p.B * T * p.H;
      const float* src = (const float*)p.ws + (wave & 1) * nws + ((int64_t)b * T + t) * p.H + h;
      __builtin_amdgcn_global_load_lds((const void*)src, (lds_void*)&coef[slot][wave & 1][0], 4, 0, 0);
    } else if constexpr (NORM == NORM_COUNT_) {
      if (wave == 0) coef[slot][0][lane] = count_norm(t, W);
    }
  };
  auto block = [&](const bf16* Qs, const bf16* Gs, const float(*cf)[kTile], int qa, auto mask_tag)
                   __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_tag)::value;
    f32x4 s[2][2], dp[2][2];  // [key tile i][query tile j]
    product32(Qs, 32 * qh, kf, g, c, s);
    product32(Gs, 32 * qh, vf, g, c, dp);
    f32x4 a4[2], c4[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a4[j] = f32x4{1.f, 1.f, 1.f, 1.f};
      c4[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (NORM != NORM_RAW) a4[j] = *(const f32x4*)&cf[0][32 * qh + 16 * j + 4 * g];
      if (NORM == NORM_MASS_) c4[j] = *(const f32x4*)&cf[1][32 * qh + 16 * j + 4 * g];
    }
    TrRead qt_[4], gt_[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      qt_[m] = dt_tr8_issue(Qs, m, 32 * qh, g, c);
      gt_[m] = dt_tr8_issue(Gs, m, 32 * qh, g, c);
    }
    bf16x8 qt[4], gt[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float pa[2][4], gd[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int q = qa + 16 * j + 4 * g + r;
          const float x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[i][j][r] * k2));
          const bool on = !MASK || (q < T && pair_on(q, ka + 16 * i + c, W));
          const float dt = NORM == NORM_RAW ? dp[i][j][r] : fmaf(dp[i][j][r], a4[j][r], -c4[j][r]);
          pa[j][r] = on ? (NORM == NORM_RAW ? x : x * a4[j][r]) : 0.f;
          gd[j][r] = on ? dt * (x - x * x) : 0.f;
        }
      const bf16x8 pb = pack_b(pa[0], pa[1]), gbv = pack_b(gd[0], gd[1]);
      if (i == 0) {
        tr_wait4(qt_);
        tr_wait4(gt_);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          qt[m] = tr_join(qt_[m]);
          gt[m] = tr_join(gt_[m]);
        }
      }
      // (left out from the pairs' arithmetic on, in either order of i, the kernel
      // spills 12 to 27 registers; so only the products are)
      if (MASK && i == 0 && pairs_out<32, 16>(qa, ka, W)) continue;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        dv[i][m] = mfma(gt[m], pb, dv[i][m]);
        dk[i][m] = mfma(qt[m], gbv, dk[i][m]);
      }
    }
  };
  ring<NORM == NORM_MASS_ ? 1 : 0>(qs, gs, qr, tiles, wave, coef_copy, [&](int blk, int slot) __attribute__((always_inline)) {
    const int qa = blk * kTile + 32 * qh;
    if (pairs_out<32, 32>(qa, ka, W)) return;
    if (ka + 31 < qa && ka >= qa + 31 - W && qa + 31 < T) block(tiles[slot], tiles[kRing + slot], coef[slot], qa, std::false_type{});
    else block(tiles[slot], tiles[kRing + slot], coef[slot], qa, std::true_type{});
  });

  float x[2][32], o[32];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      x[i][e] = dk[i][e >> 2][e & 3];
      x[i][16 + e] = dv[i][e >> 2][e & 3];
    }
  meet<32>((float*)lds, kh, qh, lane, x, o);
  f32x4 ok[4], ov[4];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    ok[e >> 2][e & 3] = o[e];
    ov[e >> 2][e & 3] = o[16 + e];
  }
  const int r0 = ka + 16 * qh;
  bf16* sb = lds + wave * (16 * kTile);
  store_rows_staged((bf16*)p.dk.p + b * p.dk.s0 + (int64_t)r0 * p.dk.s1 + h * p.dk.s2, p.dk.s1, T - r0, ok,
                    (float)(1.0 / p.scale), g, c, lane, sb);
  store_rows_staged((bf16*)p.dv.p + b * p.dv.s0 + (int64_t)r0 * p.dv.s1 + h * p.dv.s2, p.dv.s1, T - r0, ov, 1.f, g, c,
                    lane, sb);
}

// Phase 0 forward, 1 dQ, 2 dK / dV; one workgroup per 64-row tile (n of them).
void launch_wide(int phase, const BandParams& p, hipStream_t st, unsigned n, int norm) {
  const BandArgs a = to_args(p);
#define WL(K)                                                                                        \
  do {                                                                                               \
    if (norm == NORM_MASS_) hipLaunchKernelGGL((K<NORM_MASS_>), dim3(n), dim3(kThreads), 0, st, a);  \
    else if (norm == NORM_COUNT_) hipLaunchKernelGGL((K<NORM_COUNT_>), dim3(n), dim3(kThreads), 0, st, a); \
    else hipLaunchKernelGGL((K<NORM_RAW>), dim3(n), dim3(kThreads), 0, st, a);                        \
  } while (0)
  if (phase == 0) WL(wl_fwd);
  else if (phase == 1) WL(wl_dq);
  else WL(wl_dkv);
#undef WL
}

}  // namespace tension
