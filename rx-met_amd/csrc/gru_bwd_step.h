// gru_bwd_step.h — the stepped GRU backward (any H up to 1024, any recurrent weight width), one
// launch per step for every direction; included by gru_bwd.hip.
//
// Launch t takes the gate gradients of step t + 1, computes dh_t = dhl + (dq_{t+1} scale_R) R_q^T
// for its tile of sequences x units and goes straight on to the STE pointwise of step t for that
// tile, whose dq it leaves for the next launch; launch -1 ends with dh0.  The boundary between two
// launches is what orders the exchange: dq of one step is read by workgroups on every XCD, which
// inside one launch would have to bypass the L2 (3 x 6 bytes per unit and reader: 300 MB per step
// at B = H = 1024, 38 us at the 8 TB/s of the coherence point against 10 us from the L2s).
//
// The product runs on bf16 MFMA: dq scale_R as its exact three bf16 terms (split3x8), made once by
// the pointwise that produces it, against R_q's codes, with fp32 sums of at most 384 channels per
// wave, the eight waves' sums added in order.  Both operands lie in MFMA fragment order, 1 KB per
// 16 rows x 32 channels, so each lane loads its fragments from global memory as contiguous pieces
// and no operand goes through LDS.  (Through LDS, every wave pair read its operands from it again:
// 64 KB per 64 channels, 35 us for the product alone at B = H = 1024 where it now takes 20.  dq as
// fp32, split by every wave that reads it: 31 us, bound by the vector unit.)
//
// Two tile shapes (step_big): 64 x 64, whose 4 x 4 fragments per wave read the fewest bytes per
// product, when that gives half of the CUs a workgroup; else 32 x 32, for four times as many.
//
// Measured, per step, w4a16 codes: B = H = 1024 62 us in two launches -> 40 us (20 the product, at
// 20 TB/s from the L2s; the rest launch, the pointwise and its 48 MB of stores, which nothing
// hides); a whole training step of 50 time steps, I = 256: B 64, H 512 1855 -> 1168 us; B 200,
// H 512, both directions 4032 -> 2049; B 300, H 320 2127 -> 1409; B 1024, H 1024 7742 -> 6931.
#pragma once

namespace rxmet {
namespace gru {

constexpr int kStepFrag = 512;  // bf16 of one fragment: 16 rows (or columns) x 32 channels

// One direction of the stepped backward.  Channels are padded per gate: k = gate Hk + unit.
struct StepArgs {
  BwdArgs a;
  const __bf16 *rb;  // [planes of R][H / 16][KR][kStepFrag], zero from chunk KC on
  __bf16 *dqp;       // [2 parities][3 terms][MT][KC][kStepFrag]
  float *dhl;        // [B, H]: the part of dh that does not pass through R
};
struct StepShape {
  int t, ndir, tm, tn;  // tiles of one direction
  int Hk, KC, KR, MT;   // channels per gate (a multiple of 32), 32-channel chunks, those of rb,
                        // row fragments
  size_t rbplane;       // elements of one plane of rb
};

// R_q [H][3H] as B fragments, in planes (bf16 of the code and, for codes of more than 8 bits, the
// exact rest).  One workgroup of 64 per (column fragment, chunk).
template <int NPB>
__global__ __launch_bounds__(64) void pack_rt_step(int H, int Hk, int KR, const float *__restrict__ Rq,
                                                   __bf16 *__restrict__ dst, size_t plane) {
  const int l = threadIdx.x, kc = blockIdx.x % KR, nt = blockIdx.x / KR;
  const int n = 16 * nt + l % 16;
  __bf16 p[2][8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = 32 * kc + 8 * (l / 16) + e, g = k / Hk, j = k % Hk;
    const float v = g < 3 && j < H ? Rq[static_cast<size_t>(n) * 3 * H + g * H + j] : 0.0f;
    p[0][e] = static_cast<__bf16>(v);
    p[1][e] = static_cast<__bf16>(v - static_cast<float>(p[0][e]));
  }
  __bf16 *d = dst + (static_cast<size_t>(nt) * KR + kc) * kStepFrag + 8 * l;
#pragma unroll
  for (int pl = 0; pl < NPB; ++pl)
#pragma unroll
    for (int e = 0; e < 8; ++e) d[pl * plane + e] = p[pl][e];
}

// The step inputs of (sequence b, unit j) as they are in memory.  No load depends on a branch (a
// branch per element would wait for each element's loads before the next one's): absent operands
// read another buffer that is at least as large, and their value is replaced afterwards.
template <bool CODES>
__device__ __forceinline__ void step_load_raw(const BwdArgs &a, int t, int b, int j,
                                              BwdRaw<CODES> &r) {
  const int H = a.H;
  const uint32_t BH = static_cast<uint32_t>(a.B) * H, tH = static_cast<uint32_t>(t) * BH;
  const uint32_t oH = static_cast<uint32_t>(b) * H + j;
  const bool view = a.gv_on && a.gv;
  const float *gp = view ? a.gv : (a.gv_on ? a.h : a.dh_new + BH);
  const int64_t go = view ? (a.gv_rev ? a.T - 1 - t : t) * a.gv_t + b * a.gv_b + (a.gv_col0 + j) * a.gv_k
                          : static_cast<int64_t>(tH + oH);
  const float g = gp[go];
  r.g = a.gv_on && !a.gv ? 0.0f : g;
  r.h = a.h[tH + oH];
  if constexpr (CODES) {
    const uint32_t nt = static_cast<uint32_t>(a.B + 15) / 16;
    const uint32_t row = ((static_cast<uint32_t>(t) * nt + static_cast<uint32_t>(b) / 16) *
                              (static_cast<uint32_t>(H) / 16) + static_cast<uint32_t>(j) / 16) * 16 +
                         static_cast<uint32_t>(b) % 16;
    const uint32_t e = static_cast<uint32_t>(j) % 16;
#pragma unroll
    for (int q = 0; q < 4; ++q) r.c[q] = a.vc[64 * row + 16 * q + e];
    r.c[4] = a.mb[16 * row + e];
  } else {
    const uint32_t m = 3u * tH + 3u * static_cast<uint32_t>(b) * H + j;
    const uint32_t v0 = 4u * tH + 4u * static_cast<uint32_t>(b) * H + j;
#pragma unroll
    for (int q = 0; q < 4; ++q) r.v[q] = a.v[v0 + q * H];
    const uint8_t *none = reinterpret_cast<const uint8_t *>(a.v);
    const uint8_t *fam[4] = {a.ih_m, a.hh_m, a.gin_m, a.gout_m};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int g3 = 0; g3 < 3; ++g3) {
        const unsigned v = (fam[q] ? fam[q] : none)[m + g3 * H];
        r.c[3 * q + g3] = fam[q] ? v : 1u;
      }
    const unsigned v = (a.h_m ? a.h_m : none)[tH + oH];
    r.c[12] = a.h_m ? v : 1u;
  }
}

// One workgroup (512 threads): tile (tile % tn) of BT units and (tile / tn) of BT sequences.
template <int BT, int NPB, bool CODES>
__global__ __launch_bounds__(512) void bwd_step(StepArgs s0, StepArgs s1, StepShape sh) {
  constexpr int NT = BT / 16;          // fragments along either side of the tile
  constexpr int ROW = BT + 4;          // floats per row of a tile in LDS
  constexpr int PT = BT * BT / 512;    // elements per thread of the pointwise
  constexpr int TY = 512 / BT;         // its row groups
  // the waves' partial dh tiles, then the scaled dq, then the bias sums
  __shared__ __align__(16) float smem[8 * BT * ROW];

  const int total = sh.ndir * sh.tm * sh.tn;
  // consecutive tiles (one row of tiles after the other) on one XCD: they share dq rows
  const int per = (static_cast<int>(gridDim.x) + 7) / 8;
  const int idx = static_cast<int>(blockIdx.x) % 8 * per + static_cast<int>(blockIdx.x) / 8;
  if (idx >= total) return;  // whole workgroup
  const StepArgs &s = idx >= sh.tm * sh.tn ? s1 : s0;
  const BwdArgs &a = s.a;
  const int tile = idx % (sh.tm * sh.tn), m0 = tile / sh.tn * BT, n0 = tile % sh.tn * BT;
  const int t = sh.t, H = a.H, B = a.B, C = 3 * H, KC = sh.KC;
  const int tid = threadIdx.x, l = tid % 64;
  const int w = __builtin_amdgcn_readfirstlane(tid / 64);  // uniform: addresses in scalars
  const bool gemm = t != a.T - 1;
  const int mt0 = m0 / 16, nt0 = n0 / 16, ntmax = H / 16 - 1;
  const size_t aplane = static_cast<size_t>(sh.MT) * KC * kStepFrag;
  const __bf16 *pin = s.dqp + static_cast<size_t>((t + 1) & 1) * 3 * aplane;
  __bf16 *pout = s.dqp + static_cast<size_t>(t & 1) * 3 * aplane;

  // the tile's elements of this thread: unit n0 + tx, sequences m0 + ty + TY i
  const int tx = tid % BT, ty = tid / BT;
  const int j = n0 + tx;
  const bool on = j < H;
  // in flight under the products, except the float format's 20 values per element, which do not
  // fit beside the 64 x 64 tile's sums: those are loaded afterwards, four elements at a time
  constexpr bool kEarly = CODES || BT < 64;
  constexpr int LB = kEarly ? PT : 4;
  BwdRaw<CODES> raw[LB];
  float carry[PT];
  auto load_point = [&](int i0) {
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int b = m0 + ty + TY * (i0 + i);
      // absent elements repeat one that is there
      step_load_raw<CODES>(a, t, b < B ? b : B - 1, on ? j : 0, raw[i]);
    }
    if (t == a.T - 1 && a.gv_on && a.gv_hn) {  // the gradient of h_n
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const int b = m0 + ty + TY * (i0 + i);
        raw[i].g += a.gv_hn[static_cast<uint32_t>(b < B ? b : B - 1) * H + (on ? j : 0)];
      }
    }
  };
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int b = m0 + ty + TY * i;
    const float c = s.dhl[static_cast<uint32_t>(b < B ? b : B - 1) * H + (on ? j : 0)];
    carry[i] = gemm ? c : 0.0f;  // step T - 1 comes first: nothing is carried into it
  }
  if (kEarly && t >= 0) load_point(0);

  float dhc[PT];
#pragma unroll
  for (int i = 0; i < PT; ++i) dhc[i] = 0.0f;
  if (gemm) {
    // wave w takes chunks w, w + 8, ..: at most 384 channels each, summed in order at the end
    v4f acc[NT][NT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int q = 0; q < NT; ++q) acc[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
    // Every wave runs the same number of chunks, those past the last against zeros of rb (their A
    // is the last chunk again), so that the loop is one block: with a branch in it the compiler
    // sinks the loads across it to their uses.  64 x 64: a row's fragments are loaded again for
    // the wave's next chunk as their products are issued, B two sets; 32 x 32: two sets of both.
    constexpr int S = 2, SA = BT == 64 ? 1 : 2;
    v8bf fa[SA][NT][3], fb[S][NT][NPB];
    auto load_a = [&](v8bf (&f)[3], int c, int i) {
      const __bf16 *q = pin + (static_cast<size_t>(mt0 + i) * KC + min(c, KC - 1)) * kStepFrag;
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) f[pl] = *reinterpret_cast<const v8bf *>(q + pl * aplane + 8 * l);
    };
    auto load_b = [&](v8bf (&f)[NT][NPB], int c) {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const __bf16 *q = s.rb + (static_cast<size_t>(min(nt0 + n, ntmax)) * sh.KR +
                                  min(c, sh.KR - 1)) * kStepFrag;
#pragma unroll
        for (int pl = 0; pl < NPB; ++pl)
          f[n][pl] = *reinterpret_cast<const v8bf *>(q + pl * sh.rbplane + 8 * l);
      }
    };
    auto products = [&](int i, const v8bf (&x)[3], const v8bf (&y)[NT][NPB]) {
#pragma unroll
      for (int pl = 0; pl < NPB; ++pl)
#pragma unroll
        for (int e = 2; e >= 0; --e)  // smallest terms first; a sum's products apart
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[i][n] = mfma_bf16(x[e], y[n][pl], acc[i][n]);
    };
    auto chunk = [&](int c, v8bf (&xa)[NT][3], v8bf (&xb)[NT][NPB]) {
      constexpr int ahead = 8 * SA;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        products(i, xa[i], xb);
        load_a(xa[i], c + ahead, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      load_b(xb, c + 8 * S);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int k = 0; k < S; ++k) {
      load_b(fb[k], w + 8 * k);
      if (k < SA)
#pragma unroll
        for (int i = 0; i < NT; ++i) load_a(fa[k][i], w + 8 * k, i);
    }
    for (int c = w; c < sh.KR; c += 8 * S) {
#pragma unroll
      for (int k = 0; k < S; ++k) chunk(c + 8 * k, fa[k % SA], fb[k]);
    }
    float *d = smem + w * BT * ROW;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int q = 0; q < NT; ++q)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          d[(16 * i + 4 * (l / 16) + rr) * ROW + 16 * q + l % 16] = acc[i][q][rr];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int o = (ty + TY * i) * ROW + tx;
      float v = smem[o];
#pragma unroll
      for (int k = 1; k < 8; ++k) v += smem[k * BT * ROW + o];
      dhc[i] = carry[i] + v;
    }
    __syncthreads();
  }

  if (t < 0) {  // dh0
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int b = m0 + ty + TY * i;
      if (!on || b >= B) continue;
      const uint32_t o = static_cast<uint32_t>(b) * H + j;
      a.dh0[o] = a.h0_m ? dhc[i] * static_cast<float>(a.h0_m[o]) : dhc[i];
    }
    return;
  }

  // ---- pointwise of step t; scaled dq to LDS, [gate][sequence][unit] ----
  auto gate_tile = [&](int g) { return smem + g * BT * ROW; };
  float er[3];
#pragma unroll
  for (int g = 0; g < 3; ++g) er[g] = on ? a.eff_r[g * H + j] : 0.0f;
  double sb[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  const uint32_t BH = static_cast<uint32_t>(B) * H;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    if (!kEarly && i % LB == 0) load_point(i);
    const int r = ty + TY * i, b = m0 + r;
    float dpv[3] = {0.f, 0.f, 0.f}, dqv[3] = {0.f, 0.f, 0.f};
    if (on && b < B) {
      s.dhl[static_cast<uint32_t>(b) * H + j] = bwd_point_raw<CODES>(raw[i % LB], a, dhc[i], dpv, dqv);
      const uint32_t m = 3u * static_cast<uint32_t>(t) * BH + 3u * static_cast<uint32_t>(b) * H + j;
#pragma unroll
      for (int g = 0; g < 3; ++g) {
        a.dp[m + g * H] = dpv[g];
        a.dq[m + g * H] = dqv[g];
        sb[g] += static_cast<double>(dpv[g]);
        sb[3 + g] += static_cast<double>(dqv[g]);
      }
    }
#pragma unroll
    for (int g = 0; g < 3; ++g) gate_tile(g)[r * ROW + tx] = dqv[g] * er[g];  // units past H: zero
  }
  __syncthreads();
  // its three bf16 terms, one fragment per wave and pass
  constexpr int NF = 3 * NT * (BT / 32);
#pragma unroll
  for (int f0 = 0; f0 < NF; f0 += 8) {
    const int f = f0 + w, g = f / (NT * (BT / 32)), m = f / (BT / 32) % NT, k = f % (BT / 32);
    if (f >= NF || n0 + 32 * k >= sh.Hk) continue;
    const float *p = gate_tile(g) + (16 * m + l % 16) * ROW + 32 * k + 8 * (l / 16);
    const float4 x0 = *reinterpret_cast<const float4 *>(p),
                 x1 = *reinterpret_cast<const float4 *>(p + 4);
    const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    uint4 q[3];
    split3x8(v, q[0], q[1], q[2]);
    __bf16 *d = pout + (static_cast<size_t>(mt0 + m) * KC + (g * sh.Hk + n0) / 32 + k) * kStepFrag +
                8 * l;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<uint4 *>(d + pl * aplane) = q[pl];
  }
  __syncthreads();
  // bias partials of the tile's sequences, added to those of the later steps
  double *red = reinterpret_cast<double *>(smem);  // [TY - 1][6][BT]
  static_assert((TY - 1) * 6 * BT * 8 <= sizeof(smem), "bias reduction fits");
  if (ty > 0)
#pragma unroll
    for (int e = 0; e < 6; ++e) red[((ty - 1) * 6 + e) * BT + tx] = sb[e];
  __syncthreads();
  if (ty == 0 && on) {
#pragma unroll
    for (int k = 0; k < TY - 1; ++k)
#pragma unroll
      for (int e = 0; e < 6; ++e) sb[e] += red[(k * 6 + e) * BT + tx];
    double *p = a.bias_partial + static_cast<size_t>(m0 / BT) * 2 * C;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const double mw = a.bw_m ? static_cast<double>(a.bw_m[g * H + j]) : 1.0;
      const double mr = a.br_m ? static_cast<double>(a.br_m[g * H + j]) : 1.0;
      p[g * H + j] = (gemm ? p[g * H + j] : 0.0) + sb[g] * mw;
      p[C + g * H + j] = (gemm ? p[C + g * H + j] : 0.0) + sb[3 + g] * mr;
    }
  }
}

// Chunks of rb: every wave runs the same number, two sets of eight at a time.
inline int step_kr(int KC) { return (KC + 15) / 16 * 16; }
// Elements of one parity's dq terms and of one plane of R's fragments.
inline size_t step_terms(int B, int H) {
  return static_cast<size_t>(3) * ((B + 63) / 64 * 4) * (3 * ((H + 31) / 32)) * kStepFrag;
}
inline size_t step_rplane(int H) {
  return static_cast<size_t>((H + 15) / 16) * step_kr(3 * ((H + 31) / 32)) * kStepFrag;
}

}  // namespace gru
}  // namespace rxmet
