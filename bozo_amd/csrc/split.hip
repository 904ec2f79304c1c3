// Dispatch of the split-operand band kernels (split_band.h): grid size and
// the per-phase, per-precision instantiation units.
#include "kernels.h"

namespace tension {

void launch_split_fwd_bf16(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dq_bf16(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dkv_bf16(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_fwd_f32(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dq_f32(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dkv_f32(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_fwd_f32v(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dq_f32v(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dkv_f32v(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_fwd_f16(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dq_f16(const BandParams& p, hipStream_t st, unsigned n);
void launch_split_dkv_f16(const BandParams& p, hipStream_t st, unsigned n);

static thread_local int g_key_groups = 0;

int last_key_groups() { return g_key_groups; }

int launch_split(int phase, int flow, const BandParams& p_in, hipStream_t st, hipError_t* err) {
  if (flow < SPLIT_FLOW_BF16 || flow > SPLIT_FLOW_F16) return -1;
  if (phase < 0 || phase > 2) return -1;
  BandArgs probe;
  if (!band_args(p_in, &probe)) return -1;  // the kernels take 32-bit strides
  BandParams p = p_in;
  if (p.D != 32 && p.D != 64) return -1;
  p.ntiles = (p.T + 63) / 64;
  int64_t nwg = (int64_t)p.B * p.H * p.ntiles;
  if (nwg <= 0) return -1;
  if (nwg > 0x7fffffff) return kGridTooLarge;
  // p.chunk > 0: runs of consecutive tiles per workgroup (p.chunk runs per
  // (b, h)) for a local window W <= 64: the forward, sized for about three
  // resident workgroups per CU, and the backward kernels for about two: dK /
  // dV (float32 throughout at head dim 64: see below), and dQ for float32 Q / K with a bf16 V at head dim 32 without dTau
  // (where its run kernel measured faster); 0: one tile per workgroup; -1: see
  // below
  p.chunk = 0;
  const bool dq_runs = flow == SPLIT_FLOW_F32 && p.D == 32 && p.dtau.p == nullptr;
  if ((phase != 1 || dq_runs) && !p.glob && p.win >= 1 && p.win <= 64) {
    const int64_t bh = (int64_t)p.B * p.H;
    const int64_t per_cu = phase == 0 ? 3 : 2;
    const int64_t slots = per_cu * (int64_t)device_cus();
    int64_t runs = (slots + bh / 2) / bh;
    bool take = true;
    if (phase == 2 && flow == SPLIT_FLOW_F32V && p.D == 64) {
      // the float32 kernel holds exactly two workgroups per CU, so a few runs over
      // would be a round of their own, and the runs are worth it only where they
      // fill their rounds: to 60%, with a bias or a dTau (where they gain less over
      // one tile per workgroup) to 90%, to 75% when a run has four tiles at most (an
      // empty place costs little).  One tile -> runs, valid count, W 64, us:
      // 96 (b, h) of T1000 51 -> 45, with dTau 59 -> 58; 128 64 -> 54, 75 -> 69; 192
      // (three runs each, 2.25 per CU) 88 -> 99, 104 -> 135; 514 220 -> 269, 251 ->
      // 374; of T256, 704 83 -> 77, 99 -> 102; 448 59 -> 49, 70 -> 63; 1024 117 -> 100,
      // 140 -> 124.
      runs = slots / bh;
      const int64_t wg = bh * (runs < 1 ? 1 : runs), rounds = (wg + slots - 1) / slots;
      const bool side = p.dtau.p || p.bias.p;
      take = 20 * wg >= (!side ? 12 : p.ntiles <= 4 ? 15 : 18) * rounds * slots;
    }
    if (runs < 1) runs = 1;
    if (take && runs < p.ntiles) {
      p.chunk = (int)runs;
      nwg = bh * runs;
    }
  }
  // a forward whose windows are wider than a key block, on a grid of at most one
  // workgroup per CU: two key groups per workgroup (p.chunk < 0, xb_fwd).  B1
  // H16 T1024, autocast / float32: W256 14.5 -> 12.6 / 18.0 -> 15.9 us, with tau
  // 20.2 -> 17.7 / 23.7 -> 20.1, global 36.6 -> 27.6 / 47.9 -> 36.8; past one per
  // CU the larger workgroups no longer all fit at once (B2 H12 T1024 with tau
  // 25.8 -> 31.8 / 30.4 -> 35.8)
  if (phase == 0 && (p.glob || p.win > 64) && nwg <= device_cus()) p.chunk = -1;
  if (phase == 0) g_key_groups = p.chunk < 0 ? 2 : 1;
  const unsigned n = (unsigned)nwg;
  typedef void (*Launch)(const BandParams&, hipStream_t, unsigned);
  static const Launch table[4][3] = {
      {launch_split_fwd_bf16, launch_split_dq_bf16, launch_split_dkv_bf16},
      {launch_split_fwd_f32, launch_split_dq_f32, launch_split_dkv_f32},
      {launch_split_fwd_f32v, launch_split_dq_f32v, launch_split_dkv_f32v},
      {launch_split_fwd_f16, launch_split_dq_f16, launch_split_dkv_f16}};
  table[flow][phase](p, st, n);
  *err = hipGetLastError();
  return 0;
}

}  // namespace tension
