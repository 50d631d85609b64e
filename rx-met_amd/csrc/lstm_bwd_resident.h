// lstm_bwd_resident.h — QuantLSTM backward recurrence with a member's W_hh in registers.
// Included by lstm_bwd.hip after its argument structs.
//
// Up to H = 256 a workgroup owns two or four sequences and holds all of W_hh^T as int8 MFMA
// operands: a step exchanges nothing with other workgroups.  Up to H = 512 a cluster of up to four
// workgroups shares eight sequences; member m owns 128 units, that is 512 of the 4H channels, and
// holds W_hh of those channels for every unit.  It multiplies its own gate gradients only, and the
// members exchange partial dh (32 KB per member and step) instead of gate gradients (64 KB).
//
// The gate gradients scaled by W's channel scales become 31-bit fixed point on one exponent per
// (sequence, group of 64 units), in four signed byte digits; row 4 s + q of
// v_mfma_i32_16x16x64_i8 is digit q of sequence s, so the four digit sums of a (sequence, unit) over
// a group's 256 channels arrive in one lane.  Each term is off by at most 2^-30 of its group's
// largest; the rest is exact up to the order of a few sums in double: the digit sums and their
// combination per group, the groups' and the members' (which meet as doubles), rounded once to fp32.
// The clustered form's groups are the same, with 22 bits.  (One exponent per workgroup, sums met and
// combined in fp32: 731 us in place of the 803 below, and a group whose gradients are far below
// another's loses its bits.)
// Gradients of a whole training step against 64 bits: 5.0e-7 (clustered form: 5.1e-7).
//
// Measured (recurrence of B = 512, T = 100, H = 512, saved codes): 949 -> 803 us against clusters of
// 64-unit members on 16 sequences.  What bounds it there: two elements per lane (some 500 VALU per
// step), 64 MFMA per wave and the exchange.
#pragma once

#include "resident.h"

namespace rxmet {
namespace lstm {

constexpr int kBresMember = 128;  // units of a cluster member
constexpr int kBresTile = 8;      // sequences of a cluster

struct BresParams {
  float gs[4], gz[4];  // gate outputs: (code - gz) gs; with saved codes the code's offset
  float c_s, c_z, t_s, t_z;
  const v4i *frag;     // lstm_pack_bres
  int G, ncl, ntiles;  // cluster
  double *xp;          // [2][ntiles][G dst][G src][8][128] partial dh
  unsigned *counters;
  int *timeout;
  unsigned spin_limit;
};

// W_hh codes [4H][H] -> frag[((m UT + jt) KS + s) 64 + lane]: channels 64 s + 16 (lane / 16) .. + 15 of
// member m's, in groups of 64 units and by gate inside a group (K step s: gate s % 4 of units m U +
// 64 (s / 4) .. + 63), against unit 16 jt + lane % 16 (zero beyond H).
__global__ __launch_bounds__(64) void lstm_pack_bres(int H, int U, int KS, const float *__restrict__ wq,
                                                     v4i *__restrict__ frag) {
  const int lane = threadIdx.x, idx = blockIdx.x, UT = H / 16;
  const int s = idx % KS, jt = (idx / KS) % UT, m = idx / (KS * UT);
  const int j = 16 * jt + lane % 16;
  int wd[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    int by[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int g = s % 4, u = m * U + 64 * (s / 4) + 16 * (lane / 16) + 4 * q + e;
      by[e] = u < H ? static_cast<int>(wq[static_cast<size_t>(g * H + u) * H + j]) : 0;
    }
    wd[q] = pack4_i8(by[0], by[1], by[2], by[3]);
  }
  frag[static_cast<size_t>(idx) * 64 + lane] = v4i{wd[0], wd[1], wd[2], wd[3]};
}

// One element's step inputs as they are in memory.  Narrow values of a quad's four units come in
// one wide load per lane (lane i: gate i of the four units) and are transposed when used.
template <bool CODES>
struct BresRaw {
  float gd;
  float v[CODES ? 1 : 6];      // float format: gate outputs, tanh, previous cell
  unsigned gc[CODES ? 2 : 1];  // gate codes (quad words)
  unsigned tc, pc, cm;         // tanh and previous-cell codes, cell-phase mask bits
  unsigned gm, ih;             // gate mask bytes, ih mask bytes (quad words)
  unsigned m3[CODES ? 1 : 2];  // float format: gate-in and gate-out masks (gm: hh)
};

constexpr size_t bres_lds_bytes(int ks, int ns) {
  return 512 + static_cast<size_t>(4) * ns * (64 * ks + 16);
}

template <int KS, int UPW, int NS, bool CODES>
__global__ __launch_bounds__(512) void lstm_bwd_recurrence_res(BwdArgs a, BresParams p) {
  constexpr bool kCluster = NS == kBresTile;
  constexpr bool kMerge = UPW == 2 && NS == 2;
  constexpr int NP = kCluster ? 2 : (UPW == 2 && !kMerge ? 2 : 1);
  constexpr int RB = kCluster ? 2 : 1;   // blocks of 16 digit rows
  constexpr bool kDeep = NP == 1;        // inputs loaded two steps ahead
  constexpr int ROW = 64 * KS + 16;
  constexpr int NG = KS / 4;                               // groups of 64 units
  constexpr int WPG = UPW == 2 && !kCluster ? 2 : 4;       // waves whose elements make a group
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned *smax = reinterpret_cast<unsigned *>(smem);  // [NS][8]: a wave's largest per sequence
  unsigned *stop = smax + 64;                           // [8][2]: a cluster's largest per group
  int8_t *pl = reinterpret_cast<int8_t *>(smem + 512);  // [4 NS][ROW] digit rows
  const int H = a.H, C = 4 * H, B = a.B, T = a.T, UT = H / 16;
  const int U = kCluster ? kBresMember : H;             // units of the workgroup
  const int tid = threadIdx.x, w = tid / 64, l = tid % 64, grp = l / 16, e = l % 16;
  cluster::Place place = {static_cast<int>(blockIdx.x), 0};
  if (kCluster) place = cluster::place(p.G, p.ncl);
  const int m0 = place.member, ut0 = kCluster ? m0 * (kBresMember / 16) : 0;

  for (int i = tid; i < NS * ROW; i += blockDim.x) reinterpret_cast<int *>(pl)[i] = 0;
  for (int i = tid; i < 128; i += blockDim.x) smax[i] = 0u;
  // operands: the units whose dh this wave sums (all of the layer's in a cluster)
  v4i wf[UPW][KS];
  const int ksn = 4 * ((U + 63) / 64);
#pragma unroll
  for (int u = 0; u < UPW; ++u)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int jt = UPW * w + u;
      wf[u][s] = jt < UT && s < ksn
                     ? p.frag[((static_cast<size_t>(m0) * UT + jt) * ksn + s) * 64 + l]
                     : v4i{0, 0, 0, 0};
    }
  const int8_t *ar[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) ar[rb] = pl + (16 * rb + e % (4 * NS < 16 ? 4 * NS : 16)) * ROW + 16 * grp;
  const unsigned step_h = 4u * static_cast<unsigned>(B) * H, step_c = 4u * step_h;
  const unsigned nblk = static_cast<unsigned>((B + 15) / 16) * (H / 16);
  unsigned *counter = kCluster ? p.counters + cluster::kCounterStride * place.cluster : nullptr;
  unsigned epoch = 0;
  bool alive = true;

  for (int tile = place.cluster; tile < (kCluster ? p.ntiles : place.cluster + 1) && alive;
       tile += kCluster ? p.ncl : 1) {
    // the elements this lane finishes: pass k, (sequence b, unit j)
    float dh[NP], dc[NP], sw[NP][4];
    unsigned os[NP], ol[NP], og[NP], ob[NP], oq[NP];
    int8_t *pw[NP];
    int sq[NP];
    unsigned rw[NP];
    bool own[NP], ok[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int seq = kCluster ? 2 * grp + k : (kMerge ? grp % 2 : grp);
      // a cluster's element tile is the wave's; else the tiles it also sums
      const int utl = kCluster ? w : UPW * w + (kMerge ? grp / 2 : k), ut = ut0 + utl;
      const int b = NS * tile + seq, bc = b < B ? b : B - 1, j = 16 * ut + e;
      sq[k] = seq;
      rw[k] = static_cast<unsigned>(bc) % 16;
      own[k] = seq < NS && ut < UT;
      ok[k] = own[k] && b < B;
      const int jc = ut < UT ? j : e, utc = ut < UT ? ut : 0;
      const unsigned row = static_cast<unsigned>(bc) * H + jc;
      os[k] = ok[k] ? 4u * (static_cast<unsigned>(b) * C + j) : kResSkip;
      ol[k] = 4u * row;
      og[k] = static_cast<unsigned>(bc) * C + (e % 4) * H + (jc & ~3);  // quad mask words
      if (CODES) {
        const unsigned blk = static_cast<unsigned>(bc / 16) * (H / 16) + utc;
        ob[k] = blk * kLckBlock;
        oq[k] = 2u * (blk * kLcellBlock + (bc % 16) * 16 + e);
      } else {
        ob[k] = 4u * (static_cast<unsigned>(bc) * C + jc);
        oq[k] = row;
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) sw[k][g] = a.s_whh[g * H + jc];
      dh[k] = a.grad_hn && ok[k] ? a.grad_hn[row] : 0.0f;
      dc[k] = a.grad_cn && ok[k] ? a.grad_cn[row] : 0.0f;
      pw[k] = pl + (own[k] ? (4 * seq + e % 4) * ROW + 256 * (utl / 4) + 16 * (utl % 4) + (e & ~3) : 0);
    }
    auto load = [&](int t, BresRaw<CODES> (&r)[NP]) {
      const size_t tt = static_cast<size_t>(t > 0 ? t : 0);
      const auto rg = cluster::buffer_rsrc(a.grad_out + tt * B * H, step_h);
      const auto ri = cluster::buffer_rsrc(a.ih_m + tt * B * C, step_h);
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        r[k].gd = buf_load_f32(rg, ol[k]);
        r[k].ih = buf_load_u32(ri, og[k]);
      }
      if constexpr (CODES) {
        const auto rb = cluster::buffer_rsrc(a.ckb + tt * nblk * kLckBlock, nblk * kLckBlock);
        const auto rc = cluster::buffer_rsrc(a.cellc + tt * nblk * kLcellBlock, 2u * nblk * kLcellBlock);
#pragma unroll
        for (int k = 0; k < NP; ++k) {
          const unsigned R = rw[k];
          const auto v = __builtin_amdgcn_raw_buffer_load_b64(
              rb, ob[k] + 2u * ((R * 4 + e % 4) * 16 + (e & ~3)), 0, 0);
          r[k].gc[0] = v[0];
          r[k].gc[1] = v[1];
          r[k].gm = buf_load_u32(rb, ob[k] + kLckGm + ((e % 4) * 16 + R) * 16 + (e & ~3));
          r[k].tc = buf_load_u16(rb, ob[k] + kLckTanh + 2u * (R * 16 + e));
          r[k].cm = buf_load_u8(rb, ob[k] + kLckCm + R * 16 + e);
          r[k].pc = buf_load_u16(rc, oq[k]);
        }
      } else {
        const auto ro = cluster::buffer_rsrc(a.gate_out + tt * B * C, step_c);
        const auto rt = cluster::buffer_rsrc(a.cell_tanh + tt * B * H, step_h);
        const auto rc = cluster::buffer_rsrc(tt == 0 ? a.c0_q : a.cell + (tt - 1) * B * H, step_h);
        const auto m0_ = cluster::buffer_rsrc(a.hh_m + tt * B * C, step_h);
        const auto m1_ = cluster::buffer_rsrc(a.gin_m + tt * B * C, step_h);
        const auto m2_ = cluster::buffer_rsrc(a.gout_m + tt * B * C, step_h);
        const auto n0 = cluster::buffer_rsrc(a.cell_m + tt * B * H, step_h / 4);
        const auto n1 = cluster::buffer_rsrc(a.tanh_m + tt * B * H, step_h / 4);
        const auto n2 = cluster::buffer_rsrc(a.hid_m + tt * B * H, step_h / 4);
#pragma unroll
        for (int k = 0; k < NP; ++k) {
#pragma unroll
          for (int g = 0; g < 4; ++g) r[k].v[g] = buf_load_f32(ro, ob[k] + 4u * g * H);
          r[k].v[4] = buf_load_f32(rt, ol[k]);
          r[k].v[5] = buf_load_f32(rc, ol[k]);
          r[k].gm = buf_load_u32(m0_, og[k]);
          r[k].m3[0] = buf_load_u32(m1_, og[k]);
          r[k].m3[1] = buf_load_u32(m2_, og[k]);
          r[k].cm = buf_load_u8(n0, oq[k]);
          r[k].tc = buf_load_u8(n1, oq[k]);
          r[k].pc = buf_load_u8(n2, oq[k]);
        }
      }
    };

    auto step = [&](int t, BresRaw<CODES> (&r)[NP]) {
      float li[NP][4], lh[NP][4], sv[NP][4];
      unsigned mx[NP];
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        // the STE pointwise in the reference's order; masks (1 = clamped) that meet on one value
        // combined before the product
        float go[4], ct, pc;
        unsigned m_gi, m_go, m_hh;  // byte g: gate g
        unsigned m_c, m_t, m_h;
        const unsigned ihw = quad_transpose8(r[k].ih, e);
        if constexpr (CODES) {
          const v2u c = quad_transpose16(r[k].gc[0], r[k].gc[1], e);
          const unsigned v[4] = {c[0] & 0xffffu, c[0] >> 16, c[1] & 0xffffu, c[1] >> 16};
#pragma unroll
          for (int g = 0; g < 4; ++g) go[g] = static_cast<float>(v[g]);
          ct = static_cast<float>(r[k].tc);
          pc = static_cast<float>(r[k].pc);
          const unsigned gm = quad_transpose8(r[k].gm, e);
          m_hh = gm;
          m_gi = gm >> 1;
          m_go = gm >> 2;
          m_c = r[k].cm;
          m_t = r[k].cm >> 1;
          m_h = r[k].cm >> 2;
        } else {
#pragma unroll
          for (int g = 0; g < 4; ++g) go[g] = r[k].v[g];
          ct = r[k].v[4];
          pc = r[k].v[5];
          m_hh = quad_transpose8(r[k].gm, e);
          m_gi = quad_transpose8(r[k].m3[0], e);
          m_go = quad_transpose8(r[k].m3[1], e);
          m_c = r[k].cm;
          m_t = r[k].tc;
          m_h = r[k].pc;
        }
        const auto keep = [](unsigned m, int sh) { return static_cast<float>(((m >> sh) & 1u) ^ 1u); };
        const unsigned mg = m_gi | m_go, mi = mg | ihw, mh = mg | m_hh;
#pragma unroll
        for (int g = 0; g < 4; ++g) go[g] = (go[g] - p.gz[g]) * p.gs[g];
        ct = (ct - p.t_z) * p.t_s;
        pc = (pc - p.c_z) * p.c_s;
        const float dht = (dh[k] + r[k].gd) * keep(m_h, 0);
        const float d_o = dht * ct;
        const float dct = dht * go[3] * keep(m_t, 0);
        const float dcv = dc[k] + dct * (1.0f - ct * ct);
        const float mdc = dcv * keep(m_c, 0);
        const float pre[4] = {mdc * go[2] * go[0] * (1.0f - go[0]), mdc * pc * go[1] * (1.0f - go[1]),
                              mdc * go[0] * (1.0f - go[2] * go[2]), d_o * go[3] * (1.0f - go[3])};
        unsigned m = 0u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          li[k][g] = pre[g] * keep(mi, 8 * g);
          lh[k][g] = pre[g] * keep(mh, 8 * g);
          sv[k][g] = lh[k][g] * sw[k][g];
          m = max(m, __builtin_bit_cast(unsigned, sv[k][g]) & 0x7fffffffu);  // a NaN is the largest
        }
        dc[k] = mdc * go[1];
        mx[k] = own[k] ? m : 0u;
      }
      // the largest magnitude of each sequence's groups: a wave's lanes, then the waves through LDS
      if constexpr (kCluster) {
#pragma unroll
        for (int k = 0; k < NP; ++k) {
          const unsigned v = row16_max(mx[k]);
          if (e == 0) smax[sq[k] * 8 + w] = v;
        }
      } else {
        unsigned v = mx[0];
        if (NP == 2) v = max(v, mx[NP - 1]);
        v = row16_max(v);
        if constexpr (kMerge) {
          const auto x = __builtin_amdgcn_permlane32_swap(v, v, false, false);
          v = max(x[0], x[1]);
        }
        if (e == 0 && (kMerge ? grp < 2 : grp < NS)) smax[sq[0] * 8 + w] = v;
      }
      lds_barrier();
      auto store = [&]() {
        const auto r0 = cluster::buffer_rsrc(a.dli + static_cast<size_t>(t) * B * C, step_c);
        const auto r1 = cluster::buffer_rsrc(a.dlh + static_cast<size_t>(t) * B * C, step_c);
#pragma unroll
        for (int k = 0; k < NP; ++k)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            buf_f32(r0, li[k][g], os[k] + 4u * g * H);
            buf_f32(r1, lh[k][g], os[k] + 4u * g * H);
          }
      };
      if constexpr (!kCluster) {
        load(t - (kDeep ? 2 : 1), r);
        store();
      }
      auto top_of = [&](int s, int g) {  // of sequence s, group g
        const unsigned *m = smax + s * 8 + WPG * g;
        const uint2 x = *reinterpret_cast<const uint2 *>(m);
        unsigned v = max(x.x, x.y);
        if constexpr (WPG == 4) {
          const uint2 y = *reinterpret_cast<const uint2 *>(m + 2);
          v = max(v, max(y.x, y.y));
        }
        return v;
      };
      unsigned top[kCluster ? NP : NG];  // of the lane's elements' group; else of all groups
#pragma unroll
      for (int k = 0; k < (kCluster ? NP : NG); ++k)
        top[k] = kCluster ? top_of(sq[k % NP], w / WPG) : top_of(sq[0] < NS ? sq[0] : 0, k);
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        const unsigned own_top = kCluster ? top[k] : top_of(sq[0] < NS ? sq[0] : 0, w / WPG);
        const int ex = fixed_exp(own_top);
        const bool bad = fixed_bad(own_top);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const unsigned d = quad_transpose8(bad ? 0u : fixed_digits(sv[k][g], ex), e);
          if (own[k]) *reinterpret_cast<unsigned *>(pw[k] + 64 * g) = d;
        }
        if (kCluster && w % WPG == 0 && e == 0) stop[2 * sq[k] + w / WPG] = own_top;
      }
      lds_barrier();
      // a group's part of dh of the block's sequences for the wave's units, in digit sums
      auto product = [&](int rb, int q, v4i (&acc)[UPW]) {
#pragma unroll
        for (int u = 0; u < UPW; ++u) acc[u] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int s = 4 * q; s < 4 * q + 4; ++s) {
          const v4i af = *reinterpret_cast<const v4i *>(ar[rb] + 64 * s);
#pragma unroll
          for (int u = 0; u < UPW; ++u) acc[u] = mfma_i8(af, wf[u][s], acc[u]);
        }
      };
      v4i acc[UPW];
      if constexpr (kCluster) {
        // partial dh of sequence 4 rb + grp for the wave's 64 units, to the member that owns them
        const unsigned par = t & 1, G = static_cast<unsigned>(p.G);
        const unsigned base = (par * p.ntiles + tile) * G * G;
        const unsigned dst = w / 2;
        if (dst < G) {
          double *x = p.xp + static_cast<size_t>((base + dst * G + m0) * kBresTile) * kBresMember +
                     64 * (w % 2) + e;
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            double v[UPW];
#pragma unroll
            for (int q = 0; q < NG; ++q) {
              product(rb, q, acc);
              const unsigned tp = stop[2 * (4 * rb + grp) + q];
              const int ex = fixed_exp(tp);
              const bool bad = fixed_bad(tp);
#pragma unroll
              for (int u = 0; u < UPW; ++u) {
                const double f = bad ? static_cast<double>(NAN)
                                     : fixed_sum(fixed_pair(acc[u][0], acc[u][1]),
                                                 fixed_pair(acc[u][2], acc[u][3]), ex);
                v[u] = q == 0 ? f : v[u] + f;
              }
            }
#pragma unroll
            for (int u = 0; u < UPW; ++u)
              cluster::store_coherent(
                  reinterpret_cast<unsigned long long *>(x + (4 * rb + grp) * kBresMember + 16 * u),
                  __builtin_bit_cast(unsigned long long, v[u]));
          }
        }
        cluster::arrive(counter);
        ++epoch;
        load(t - 1, r);
        store();
        alive = cluster::wait(counter, epoch * G, p.timeout, p.spin_limit);
        if (!alive) return;
        const auto xr = cluster::buffer_rsrc(p.xp, 16u * p.ntiles * G * G * kBresTile * kBresMember);
        double part[NP][4];
#pragma unroll
        for (int k = 0; k < NP; ++k)
#pragma unroll
          for (unsigned s = 0; s < 4; ++s) {
            const unsigned src = s < G ? s : 0;
            part[k][s] = __builtin_bit_cast(
                double, __builtin_amdgcn_raw_buffer_load_b64(
                           xr, 8u * (((base + m0 * G + src) * kBresTile + sq[k]) * kBresMember + 16 * w + e),
                           0, 16 /* sc1: from the coherence point */));
          }
#pragma unroll
        for (int k = 0; k < NP; ++k) {
          double v = part[k][0];
#pragma unroll
          for (unsigned s = 1; s < 4; ++s)
            if (s < G) v += part[k][s];
          dh[k] = static_cast<float>(v);
        }
      } else {
        double sum[NP];
        bool bad = false;
#pragma unroll
        for (int q = 0; q < NG; ++q) {
          product(0, q, acc);
          bad |= fixed_bad(top[q]);
#pragma unroll
          for (int k = 0; k < NP; ++k) {
            const v4i &d = acc[k < UPW ? k : 0];
            int lo = fixed_pair(d[0], d[1]), hi = fixed_pair(d[2], d[3]);
            if constexpr (kMerge) {
              const v4i &d1 = acc[UPW - 1];
              lo = __builtin_amdgcn_permlane32_swap(lo, fixed_pair(d1[0], d1[1]), false, false)[0];
              hi = __builtin_amdgcn_permlane32_swap(hi, fixed_pair(d1[2], d1[3]), false, false)[0];
            }
            const double f = fixed_sum(lo, hi, fixed_exp(top[q]));
            sum[k] = q == 0 ? f : sum[k] + f;
          }
        }
#pragma unroll
        for (int k = 0; k < NP; ++k) dh[k] = bad ? NAN : static_cast<float>(sum[k]);
      }
    };

    BresRaw<CODES> ra[NP], rb[NP];
    load(T - 1, ra);
    if constexpr (kDeep) load(T - 2, rb);
    __syncthreads();  // the zeroed rows are in LDS
    if constexpr (kDeep) {
      for (int t = T - 1;;) {
        step(t, ra);
        if (--t < 0) break;
        step(t, rb);
        if (--t < 0) break;
      }
    } else {
      for (int t = T - 1; t >= 0 && alive; --t) step(t, ra);
    }
    if (!alive) break;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      if (!ok[k]) continue;
      const unsigned o = ol[k] / 4;
      a.dh0[o] = dh[k] * (a.h0_m[o] ? 0.0f : 1.0f);
      a.dc0[o] = dc[k] * (a.c0_m[o] ? 0.0f : 1.0f);
    }
  }
}

template <int NS, bool CODES>
static const void *bres_kernel(int H) {
  if (H <= 64) return reinterpret_cast<const void *>(&lstm_bwd_recurrence_res<4, 1, NS, CODES>);
  if (H <= 128) return reinterpret_cast<const void *>(&lstm_bwd_recurrence_res<8, 1, NS, CODES>);
  // four sequences in the float format would need more than the 256 VGPRs of a wave
  return reinterpret_cast<const void *>(&lstm_bwd_recurrence_res<16, 2, (CODES ? NS : 2), CODES>);
}

template <bool CODES>
static const void *bres_kernel(int H, int ns) {
  if (H > 256) return reinterpret_cast<const void *>(&lstm_bwd_recurrence_res<8, 4, kBresTile, CODES>);
  return ns == 2 ? bres_kernel<2, CODES>(H) : bres_kernel<4, CODES>(H);
}

// Fragments and exchange of the form that takes H (v4i elements, doubles).
static size_t bres_frags(int H) {
  const size_t U = H > 256 ? kBresMember : H, G = (H + U - 1) / U;
  return G * (H / 16) * (4 * ((U + 63) / 64)) * 64;
}
static size_t bres_exchange(int B, int H) {
  const size_t G = (H + kBresMember - 1) / kBresMember, nt = (B + kBresTile - 1) / kBresTile;
  return H > 256 ? 2 * nt * G * G * kBresTile * kBresMember : 0;
}

// Resident recurrence; 1 when launched (with the timeout flag of a cluster in *timeout_flag), 0 when
// another form takes the call: W_hh of 8 bits, H <= 512, grids within 2^24 codes (the float-domain
// forms), rows aligned for the quad loads.  Up to H = 256 two sequences per workgroup while every
// workgroup then has a CU of its own, else four; above, clusters of ceil(H / 128) on eight.  A
// forced poll limit (the timeout tests) asks for the clustered form up to H = 256.
static int lstm_bwd_res_launch(const BwdArgs &a, const StepParams &sp, const float *whh_q, v4i *frag,
                               double *xp, unsigned *sync, hipStream_t stream, int **timeout_flag) {
  const int H = a.H, B = a.B;
  const bool clustered = H > 256, codes = a.ckb != nullptr;
  if (H > kMaxHB || std::getenv("RXMET_NO_CLUSTER") != nullptr ||
      (!clustered && cluster::spin_limit() != cluster::kSpinLimit))
    return 0;
  auto fits = [](const Grid &g) { return g.lo > -(1 << 24) && g.hi < (1 << 24); };
  if (!fits(sp.c) || !fits(sp.tanh_c)) return 0;
  for (int g = 0; g < 4; ++g)
    if (!fits(sp.gout[g])) return 0;
  // one step's rows are addressed with 31-bit byte offsets (gates: 16 bytes per unit)
  if (16.0 * ((B + 15) / 16 * 16) * H >= 2147483648.0) return 0;
  if (8.0 * bres_exchange(B, H) >= 2147483648.0) return 0;
  BresParams p{};
  for (int g = 0; g < 4; ++g) {
    p.gs[g] = static_cast<float>(sp.gout[g].dscale);
    p.gz[g] = static_cast<float>(sp.gout[g].zp - (codes ? sp.gout[g].lo : 0));
  }
  p.c_s = static_cast<float>(sp.c.dscale);
  p.c_z = static_cast<float>(sp.c.zp - (codes ? sp.c.lo : 0));
  p.t_s = static_cast<float>(sp.tanh_c.dscale);
  p.t_z = static_cast<float>(sp.tanh_c.zp - (codes ? sp.tanh_c.lo : 0));
  p.frag = frag;
  const int U = clustered ? kBresMember : H, ksn = 4 * ((U + 63) / 64);
  p.G = (H + U - 1) / U;
  int device = 0, ncu = 0;
  RXMET_CHECK_HIP(hipGetDevice(&device));
  RXMET_CHECK_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device));
  const int ns = clustered ? kBresTile : ((B + 1) / 2 <= ncu || (!codes && H > 128) ? 2 : 4);
  const int ks = clustered ? 8 : (H <= 64 ? 4 : (H <= 128 ? 8 : 16)), upw = clustered ? 4 : (ks == 16 ? 2 : 1);
  const void *fn = codes ? bres_kernel<true>(H, ns) : bres_kernel<false>(H, ns);
  const size_t lds = bres_lds_bytes(ks, ns);
  RXMET_CHECK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds)));
  int per_cu = 0;
  if (clustered) {
    p.ntiles = (B + kBresTile - 1) / kBresTile;
    RXMET_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 512, lds));
    p.ncl = std::min(per_cu * ncu / p.G, p.ntiles);
    if (p.ncl < 1) return 0;
    if (p.ncl >= 8) p.ncl -= p.ncl % 8;
  }
  hipLaunchKernelGGL(lstm_pack_bres, dim3(p.G * (H / 16) * ksn), dim3(64), 0, stream, H, U, ksn, whh_q,
                     frag);
  RXMET_CHECK_LAUNCH();
  void *args[] = {const_cast<BwdArgs *>(&a), &p};
  if (!clustered) {
    const int waves = (H / 16 + upw - 1) / upw;
    rxmet::prof::Scope ps__("lstm_bwd_recurrence", stream);
    RXMET_CHECK_HIP(hipLaunchKernel(fn, dim3((B + ns - 1) / ns), dim3(64 * waves), args, lds, stream));
    return 1;
  }
  p.xp = xp;
  p.counters = sync;
  p.timeout = reinterpret_cast<int *>(p.counters + cluster::kCounterStride * p.ncl);
  p.spin_limit = cluster::spin_limit();
  hipLaunchKernelGGL(cluster::zero_words, dim3(1), dim3(256), 0, stream, p.counters,
                     cluster::kCounterStride * p.ncl + 1);
  RXMET_CHECK_LAUNCH();
  rxmet::prof::Scope ps__("lstm_bwd_recurrence", stream);
  RXMET_CHECK_HIP(cluster::launch(fn, dim3(p.ncl * p.G), dim3(512), args, static_cast<unsigned>(lds),
                                  stream));
  *timeout_flag = p.timeout;
  return 1;
}

}  // namespace lstm
}  // namespace rxmet
