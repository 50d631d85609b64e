// lstm_resident.h — QuantLSTM forward recurrence with all of a member's W_hh in registers.
// Included by lstm_fwd.hip after its argument structs and activation tables.
//
// A workgroup holds the int8 W_hh operands of its hidden units (all four gates) in VGPRs for the
// whole launch: up to H = 256 that is the whole layer, so a step exchanges nothing with other
// workgroups; up to H = 512 a cluster of up to four workgroups of 128 units shares eight
// sequences and exchanges only the new h codes (cluster.h).  A wave computes one or two tiles of
// 16 units over the full K range, so no sums meet across waves, and every lane finishes whole
// (sequence, unit) elements: gates, cell and hidden update in registers, one LDS exchange and one
// barrier per step.
//
// MFMA rows (16 of v_mfma_i32_16x16x64_i8): lane group g (lanes 16 g .. 16 g + 15) receives rows
// 4 g .. 4 g + 3, so sequence s' of group g with plane q of h is row 4 g + s' NPL + q: the plane
// sums of an element arrive in one lane's accumulator.
//
// Activations are table lookups (one entry per input code): gate tables in LDS, or in global
// memory where four grids do not fit; the cell's tanh as 16-bit entries in LDS for a 16-bit cell
// grid (128 KB, which the weights no longer need) where they fit, else in global memory.
//
// Measured (recurrence alone; before: clusters of 64-unit members on 16 sequences with W_hh in LDS):
// H = 256, B = 64, T = 50, 8 bits, inference: 294 -> 55 us; H = 512, B = 512, T = 100, 16-bit cell,
// saved codes: 868 -> 479 us.  What bounds it: up to H = 256 the chain of one step (LDS reads, 32
// MFMA per wave, about 130 VALU, the barrier); above, the exchange (1.5 us of 4.8) and two
// elements per lane.  Packing the saved codes into 8-byte stores by quad transposes: no gain.
#pragma once

#include "resident.h"

namespace rxmet {
namespace lstm {

enum { kLresInfer = 0, kLresCodes = 1, kLresFloat = 2 };
// gates and tanh in LDS; gates and a 16-bit tanh table in LDS; gates in LDS, tanh in global memory;
// both in global memory
enum { kTabLds = 0, kTabLds16 = 1, kTabGlobalTanh = 2, kTabGlobal = 3 };
constexpr int kLresMember = 128;             // units of a cluster member (8 waves x 16)
constexpr int kLresTile = 8;                 // sequences of a cluster

// The step's scalar parameters, reduced to what the float-domain forms use.
struct LresGate {
  float h2g_mult, in_zp, in_lo, in_hi;
  int h2g_shift, base;   // table index of an input code: code + base
  int out_c, out_lo;     // centred output: entry / 2 + out_c; code: entry / 2 + out_lo
};
struct LresParams {
  LresGate g[4];
  float lin_zp, lin_lo, lin_hi;
  float c_zp, c_lo, c_hi, ratio_f, ratio_i, c_scale;
  int t_base, t_c, t_lo, c_min;
  float h_zp, h_lo, h_hi, h_scale, hid_mult;
  int hid_shift;
  const uint32_t *gate_tab;  // global gate tables (lds_gates = 0)
  const uint32_t *tanh_tab;  // global tanh table
  int lds_gates;             // entries of the LDS table copied from lds_src (gates, perhaps tanh)
  const uint32_t *lds_src;
  int tanh_n;
  // cluster (G > 1): members, clusters, h exchange, barrier
  int G, ncl, ntiles;
  int8_t *hx;
  unsigned *counters;
  int *timeout;
  unsigned spin_limit;
};

// s clamped to [lo, hi]; bit is set where it was outside.
__device__ __forceinline__ float lres_clamp(float s, float lo, float hi, unsigned bit, unsigned &m) {
  if (s < lo || s > hi) m |= bit;
  return fminf(fmaxf(s, lo), hi);
}

// LDS beside the dynamic part: the meeting's flags of cluster.h (two words), rounded up.
constexpr size_t kLresStaticLds = 64;

constexpr size_t lres_lds_bytes(int npl, int ks, int ns, int lds_gates, int tanh16) {
  return static_cast<size_t>(2) * ns * npl * (64 * ks + 16) + 4 * static_cast<size_t>(lds_gates) +
         2 * static_cast<size_t>(tanh16);
}

// NS sequences per workgroup (2, 4; 8 in a cluster), UPW unit tiles per wave.
// TAB: where the tables are.  A run-time choice between an LDS and a global pointer would become
// one flat load, which waits for every store in flight.
template <int NPL, int KS, int UPW, int NS, int MODE, int TAB>
__global__ __launch_bounds__(512) void lstm_recurrence_res(RecArgs a, LresParams p) {
  constexpr bool kCluster = NS == kLresTile;
  constexpr int SPG = kCluster ? 2 : 1;            // sequences per lane group
  constexpr bool kMerge = UPW == 2 && NS == 2;     // two tiles' sums share one pass of the lanes
  constexpr int NP = kCluster ? 2 : (UPW == 2 && !kMerge ? 2 : 1);
  // the input branch is loaded two steps ahead; one where the registers are short (a cluster's
  // loads have the barrier to return in)
  constexpr bool kDeep = NP == 1;
  constexpr int ROW = 64 * KS + 16, HB = NS * NPL * ROW;
  extern __shared__ __align__(16) unsigned char smem[];
  int8_t *hs = reinterpret_cast<int8_t *>(smem);  // [2][NS * NPL][ROW] (a cluster uses the first)
  uint32_t *lut = reinterpret_cast<uint32_t *>(smem + 2 * HB);
  uint16_t *lut16 = reinterpret_cast<uint16_t *>(lut + p.lds_gates);
  const int H = a.H, C = 4 * H, B = a.B, T = a.T;
  const int tid = threadIdx.x, w = tid / 64, l = tid % 64, grp = l / 16, e = l % 16;
  cluster::Place place = {static_cast<int>(blockIdx.x), 0};
  if (kCluster) place = cluster::place(p.G, p.ncl);
  const int ut0 = kCluster ? place.member * (kLresMember / 16) : 0, UT = H / 16;

  for (int i = tid; i < 2 * HB / 4; i += blockDim.x) reinterpret_cast<int *>(hs)[i] = 0;
  for (int i = tid; i < p.lds_gates; i += blockDim.x) lut[i] = p.lds_src[i];
  if (TAB == kTabLds16)
    for (int i = tid; i < p.tanh_n; i += blockDim.x) lut16[i] = static_cast<uint16_t>(p.tanh_tab[i]);

  v4i wf[UPW][4][KS];
#pragma unroll
  for (int u = 0; u < UPW; ++u)
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int ut = ut0 + UPW * w + u;
        wf[u][g][s] = ut < UT && s < a.KS
                          ? a.frag[(static_cast<size_t>(g * UT + ut) * a.KS + s) * 64 + l]
                          : v4i{0, 0, 0, 0};
      }
  // channel constants of the lane's units (one set per unit tile it finishes)
  constexpr int NC = NP == 2 && !kCluster ? 2 : 1;
  float mult[NC][4], bacc[NC][4];
  int hk[NC][4], shift[NC][4];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int ut = ut0 + UPW * w + (kMerge ? grp / 2 : k), j = ut < UT ? 16 * ut + e : 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const ChanRun r = a.run[g * H + j];
      const ChanHost h = a.ch[g * H + j];
      mult[k][g] = h.hh_mult;
      shift[k][g] = -h.hh_shift;
      bacc[k][g] = r.hh_bacc;
      hk[k][g] = r.hh_k;
    }
  }
  const int ar = SPG == 2 ? (e % 4 < SPG * NPL ? (e / 4) * SPG * NPL + e % 4 : 0)
                          : (e / 4 < NS && e % 4 < NPL ? (e / 4) * NPL + e % 4 : 0);
  const int8_t *hr = hs + ar * ROW + 16 * grp;
  const unsigned step_h = 4u * static_cast<unsigned>(B) * H, step_c = 4u * step_h;
  const unsigned nblk = static_cast<unsigned>((B + 15) / 16) * (H / 16);  // code blocks of a step
  unsigned *counter = kCluster ? p.counters + cluster::kCounterStride * place.cluster : nullptr;
  unsigned epoch = 0;
  bool alive = true;

  for (int tile = place.cluster; tile < (kCluster ? p.ntiles : place.cluster + 1) && alive;
       tile += kCluster ? p.ncl : 1) {
    // the elements this lane finishes: pass k, (sequence b, unit j), and their offsets in a step
    float cst[NP], hv[NP];
    unsigned oi[NP], oh[NP], ob[NP], oq[NP];
    int8_t *hw[NP];
    int sq[NP], uj[NP];
    bool own[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int seq = kCluster ? SPG * grp + k : (kMerge ? grp % 2 : grp);
      const int ut = ut0 + UPW * w + (kMerge ? grp / 2 : (kCluster ? 0 : k));
      const int b = NS * tile + seq, j = 16 * ut + e;
      own[k] = seq < NS && ut < UT;
      sq[k] = seq;
      uj[k] = j;
      const bool ok = own[k] && b < B;
      const unsigned row = static_cast<unsigned>(b) * H + j;
      oi[k] = ok ? 4u * (static_cast<unsigned>(b) * C + j) : kResSkip;
      oh[k] = ok ? 4u * row : kResSkip;
      // codes: the block's offset and the element's place in it; float format: mask offsets
      const unsigned blk = static_cast<unsigned>(b / 16) * (H / 16) + ut;
      ob[k] = MODE == kLresCodes ? (ok ? blk * kLckBlock : kResSkip)
                                 : (ok ? static_cast<unsigned>(b) * C + j : kResSkip);
      oq[k] = MODE == kLresCodes ? (ok ? 2u * (blk * kLcellBlock + (b % 16) * 16 + e) : kResSkip)
                                 : (ok ? row : kResSkip);
      cst[k] = ok ? a.c0q[row] : p.c_zp;
      hv[k] = ok ? a.h0q[row] : p.h_zp;
      hw[k] = hs + (own[k] ? seq * NPL * ROW + j : 0);
    }
    // the row inside its block of 16 sequences (codes format)
    const int R0 = (NS * tile) % 16;
    const unsigned plane_stride = static_cast<unsigned>(kLresTile) * H;
    const unsigned xpar = NPL * plane_stride * static_cast<unsigned>(p.ntiles);
    const unsigned xtile = NPL * plane_stride * static_cast<unsigned>(tile);
    // new h codes: to the other buffer of this workgroup, or to the cluster's exchange
    auto put_h = [&](int buf) {
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        const int hc = static_cast<int>(hv[k] - a.h_offset);
        if constexpr (kCluster) {
          unsigned char *dst = reinterpret_cast<unsigned char *>(p.hx) + buf * xpar + xtile +
                               (own[k] ? static_cast<unsigned>(sq[k]) * H + uj[k] : 0);
#pragma unroll
          for (int q = 0; q < NPL; ++q) {
            // four lanes of a quad hold four consecutive bytes: lane 0 of it stores the word
            unsigned v = static_cast<unsigned>(NPL == 1 ? hc : (q == 0 ? (hc & 255) - 128 : hc >> 8)) & 255u;
            v |= quad_xor1(v) << 8;
            v |= quad_xor2(v) << 16;
            if (own[k] && e % 4 == 0)
              cluster::store_coherent(reinterpret_cast<unsigned *>(dst + q * plane_stride), v);
          }
        } else if (own[k]) {
          int8_t *dst = hw[k] + buf * HB;
          dst[0] = static_cast<int8_t>(NPL == 1 ? hc : (hc & 255) - 128);
          if (NPL == 2) dst[ROW] = static_cast<int8_t>(hc >> 8);
        }
      }
    };
    // the cluster's h codes of a step, from the exchange into LDS (16 bytes per thread)
    const auto xr = cluster::buffer_rsrc(p.hx, 2u * xpar);
    auto get_h = [&](int buf) {
      const int n = NPL * kLresTile * H / 16, cpr = H / 16;
      for (int i = tid; i < n; i += 512) {
        const int q = i / (kLresTile * cpr), s = (i / cpr) % kLresTile, c = i % cpr;
        const int4 v = cluster::load_coherent16(
            xr, buf * xpar + xtile + q * plane_stride + static_cast<unsigned>(s) * H + 16u * c);
        *reinterpret_cast<int4 *>(hs + (s * NPL + q) * ROW + 16 * c) = v;
      }
    };
    auto load_in = [&](int t, float (&lh)[NP][4]) {
      const auto r = cluster::buffer_rsrc(a.lhs + static_cast<size_t>(t < T ? t : T - 1) * B * C, step_c);
#pragma unroll
      for (int k = 0; k < NP; ++k)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          lh[k][g] = buf_load_f32(r, oi[k] + 4u * g * H);
    };

    auto step = [&](int t, int par, float (&lh)[NP][4]) {
      v4i acc[UPW][4];
#pragma unroll
      for (int u = 0; u < UPW; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[u][g] = v4i{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const v4i hf = *reinterpret_cast<const v4i *>(hr + (kCluster ? 0 : par * HB) + 64 * s);
#pragma unroll
        for (int u = 0; u < UPW; ++u)
#pragma unroll
          for (int g = 0; g < 4; ++g) acc[u][g] = mfma_i8(hf, wf[u][g][s], acc[u][g]);
      }
      unsigned ge[NP][4], gm[NP][4], te[NP], cm[NP];
      float cnew[NP], hnew[NP];
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        constexpr int kOne = 0;
        const int kc = NC == 2 ? k : kOne;
        float go[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          int sum[NPL];
#pragma unroll
          for (int q = 0; q < NPL; ++q) {
            if constexpr (kMerge)
              sum[q] = __builtin_amdgcn_permlane32_swap(acc[0][g][q], acc[UPW - 1][g][q], false, false)[0];
            else
              sum[q] = kCluster ? acc[0][g][k * NPL + q] : acc[k < UPW ? k : 0][g][q];
          }
          int v = sum[0] + hk[kc][g];
          if (NPL == 2) v += 256 * sum[NPL - 1];
          unsigned m = 0;
          const float accf = static_cast<float>(v) + bacc[kc][g];
          const float lin = lres_clamp(rintf(ldexpf(accf * mult[kc][g], shift[kc][g])) + p.lin_zp,
                                       p.lin_lo, p.lin_hi, 1u, m);
          const float rhs = rintf(ldexpf((lin - p.lin_zp) * p.g[g].h2g_mult, -p.g[g].h2g_shift));
          const float gi = lres_clamp((lh[k][g] + rhs) + p.g[g].in_zp, p.g[g].in_lo, p.g[g].in_hi,
                                      2u, m);
          const int idx = static_cast<int>(gi) + p.g[g].base;
          if constexpr (TAB == kTabGlobal)
            ge[k][g] = p.gate_tab[idx];
          else
            ge[k][g] = lut[idx];
          gm[k][g] = m;
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          gm[k][g] |= (ge[k][g] & 1u) << 2;
          go[g] = static_cast<float>(static_cast<int>(ge[k][g] >> 1) + p.g[g].out_c);
        }
        const float pf = go[1] * (cst[k] - p.c_zp), pi = go[0] * go[2];
        const float sum = pf * p.ratio_f + pi * p.ratio_i;
        unsigned m = 0;
        cnew[k] = lres_clamp(rintf(sum) + p.c_zp, p.c_lo, p.c_hi, 1u, m);
        const int ti = static_cast<int>(cnew[k]) + p.t_base;
        if constexpr (TAB == kTabLds)
          te[k] = lut[ti];
        else if constexpr (TAB == kTabLds16)
          te[k] = lut16[ti];
        else
          te[k] = p.tanh_tab[ti];
        m |= (te[k] & 1u) << 1;
        const float raw = go[3] * static_cast<float>(static_cast<int>(te[k] >> 1) + p.t_c);
        hnew[k] = lres_clamp(rintf(ldexpf(raw * p.hid_mult, -p.hid_shift)) + p.h_zp, p.h_lo, p.h_hi,
                             4u, m);
        cm[k] = m;
        cst[k] = cnew[k];
        hv[k] = hnew[k];
      }
      put_h(par ^ 1);
      if constexpr (kCluster) {
        cluster::arrive(counter);
        ++epoch;
      } else {
        lds_barrier();
      }
      // everything below is independent of the next step's reads
      load_in(t + (kDeep ? 2 : 1), lh);
      const size_t t64 = static_cast<size_t>(t);
      const auto ro = cluster::buffer_rsrc(a.output + t64 * B * H, step_h);
#pragma unroll
      for (int k = 0; k < NP; ++k) buf_f32(ro, (hv[k] - p.h_zp) * p.h_scale, oh[k]);
      if constexpr (MODE != kLresInfer) {
        const auto rhd = cluster::buffer_rsrc(a.hidden + t64 * B * H, step_h);
#pragma unroll
        for (int k = 0; k < NP; ++k) buf_f32(rhd, hv[k], oh[k]);
      }
      if constexpr (MODE == kLresCodes) {
        const auto rb = cluster::buffer_rsrc(a.ckb + t64 * nblk * kLckBlock, nblk * kLckBlock);
        const auto rc = cluster::buffer_rsrc(a.cellc + (t64 + 1) * nblk * kLcellBlock,
                                             2u * nblk * kLcellBlock);
#pragma unroll
        for (int k = 0; k < NP; ++k) {
          const unsigned R = static_cast<unsigned>(R0 + sq[k]) % 16;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            buf_u16(rb, ge[k][g] >> 1, ob[k] + 2u * ((R * 4 + g) * 16 + e));
            buf_u8(rb, gm[k][g], ob[k] + kLckGm + (g * 16 + R) * 16 + e);
          }
          buf_u16(rb, te[k] >> 1, ob[k] + kLckTanh + 2u * (R * 16 + e));
          buf_u8(rb, cm[k], ob[k] + kLckCm + R * 16 + e);
          buf_u16(rc, static_cast<unsigned>(static_cast<int>(cnew[k]) - p.c_min), oq[k]);
        }
      } else if constexpr (MODE == kLresFloat) {
        const auto rg = cluster::buffer_rsrc(a.gate_out + t64 * B * C, step_c);
        const auto r0 = cluster::buffer_rsrc(a.hh_lin_m + t64 * B * C, step_h);
        const auto r1 = cluster::buffer_rsrc(a.gate_in_m + t64 * B * C, step_h);
        const auto r2 = cluster::buffer_rsrc(a.gate_out_m + t64 * B * C, step_h);
        const auto rc = cluster::buffer_rsrc(a.cell + t64 * B * H, step_h);
        const auto rt = cluster::buffer_rsrc(a.cell_tanh + t64 * B * H, step_h);
        const auto m0 = cluster::buffer_rsrc(a.cell_m + t64 * B * H, step_h / 4);
        const auto m1 = cluster::buffer_rsrc(a.cell_tanh_m + t64 * B * H, step_h / 4);
        const auto m2 = cluster::buffer_rsrc(a.hidden_m + t64 * B * H, step_h / 4);
#pragma unroll
        for (int k = 0; k < NP; ++k) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            buf_f32(rg, static_cast<float>(static_cast<int>(ge[k][g] >> 1) + p.g[g].out_lo),
                     oi[k] + 4u * g * H);
            buf_u8(r0, gm[k][g] & 1u, ob[k] + g * H);
            buf_u8(r1, (gm[k][g] >> 1) & 1u, ob[k] + g * H);
            buf_u8(r2, gm[k][g] >> 2, ob[k] + g * H);
          }
          buf_f32(rc, cnew[k], oh[k]);
          buf_f32(rt, static_cast<float>(static_cast<int>(te[k] >> 1) + p.t_lo), oh[k]);
          buf_u8(m0, cm[k] & 1u, oq[k]);
          buf_u8(m1, (cm[k] >> 1) & 1u, oq[k]);
          buf_u8(m2, cm[k] >> 2, oq[k]);
        }
      }
      if constexpr (kCluster) {
        alive = cluster::wait(counter, epoch * p.G, p.timeout, p.spin_limit);
        if (alive && t + 1 < T) {
          get_h(par ^ 1);
          lds_barrier();
        }
      }
    };

    float la[NP][4], lb[NP][4];
    load_in(0, la);
    if constexpr (kDeep) load_in(1, lb);
    put_h(0);
    if constexpr (kCluster) {
      alive = cluster::sync(counter, ++epoch * p.G, p.timeout, p.spin_limit);
      if (!alive) break;
      get_h(0);
    }
    lds_barrier();  // h, the zeroed rows and the tables are in LDS
    if constexpr (kDeep) {
      for (int t = 0;;) {
        step(t, 0, la);
        if (++t >= T) break;
        step(t, 1, lb);
        if (++t >= T) break;
      }
    } else {
      for (int t = 0; t < T && alive; ++t) step(t, t & 1, la);
    }
    if (!alive) break;
    const auto rhn = cluster::buffer_rsrc(a.h_n, step_h), rcn = cluster::buffer_rsrc(a.c_n, step_h);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      buf_f32(rhn, (hv[k] - p.h_zp) * p.h_scale, oh[k]);
      buf_f32(rcn, (cst[k] - p.c_zp) * p.c_scale, oh[k]);
    }
  }
}

template <int NPL, int MODE, int TAB>
static const void *lres_kernel(int H, int ns) {
  if (H > 256)
    return reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 8, 1, kLresTile, MODE, TAB>);
  if (H > 128)
    return ns == 2 ? reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 4, 2, 2, MODE, TAB>)
                   : reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 4, 2, 4, MODE, TAB>);
  if (H > 64)
    return ns == 2 ? reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 2, 1, 2, MODE, TAB>)
                   : reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 2, 1, 4, MODE, TAB>);
  return ns == 2 ? reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 1, 1, 2, MODE, TAB>)
                 : reinterpret_cast<const void *>(&lstm_recurrence_res<NPL, 1, 1, 4, MODE, TAB>);
}

template <int NPL, int MODE>
static const void *lres_kernel(int H, int ns, int tab) {
  return tab == kTabLds     ? lres_kernel<NPL, MODE, kTabLds>(H, ns)
         : tab == kTabLds16 ? lres_kernel<NPL, MODE, kTabLds16>(H, ns)
         : tab == kTabGlobalTanh ? lres_kernel<NPL, MODE, kTabGlobalTanh>(H, ns)
                                 : lres_kernel<NPL, MODE, kTabGlobal>(H, ns);
}

}  // namespace lstm
}  // namespace rxmet
