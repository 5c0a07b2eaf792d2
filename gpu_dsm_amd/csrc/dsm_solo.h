// dsm_solo.h -- the solo form of the KMC jump kernels: one chain per wave, for the long
// and the few.  Included by dsm_solo_inst.hip.
//
// Why.  Where chains are few, or one of them is much longer than the others, a pass ends
// with the serial run of a chain: its time is the latency of one jump.  The wave form
// (dsm_kmc.h) holds a chain in registers, four positions a lane and group, and works on
// all of them at every jump.  Here the chain lies in LDS and a jump touches what it needs:
// the 256 positions around the event for the canonical sums, four strands for the rates.
// The rates before the event, after a Kuhn step to the right and after one to the left
// are evaluated side by side in three rows of lanes, so a jump passes once through the
// tables and the exponential; what follows from them is picked by the wave's scalar unit.
// Every sum and rate is formed from the same operands in the same order as in the other
// forms, so a chain makes the same jumps bit for bit.
//
// What bounds it: alone on a SIMD, instruction latency -- about 3,000 cycles a jump whatever
// the chain's length (window and rates 800, clock 400, sums 400, sub-event 250), 6,000 for
// one that splits or merges strands (a third of the jumps of a chain of 12 strands, a tenth
// of one of 125); with four waves a SIMD, their instructions.  Strand vectors are touched
// by splits, merges and samples alone and stay in the chain arrays, so a position takes 16
// bytes of LDS and a CU holds eight chains of 1,024 positions.  Measured against the wave
// forms: 1,500 chains of Nk 1000, 4 tau_K: 1.68 against 4.48 ms; 32,768 of Nk 600: 8.4 / 15.1;
// 65,536 of Nk 300: 15.5 / 16.8 (two chains a wave); 1000 of Nk 25, 64 tau_K: 1.10 / 1.15; 64
// of Nk 16: 0.86 / 0.84.
#pragma once
#include "dsm_lane.h"

namespace dsm {

__device__ __forceinline__ float lane_read(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ int lane_read(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// the last lane of each row into the next row, for the rows of `MASK`
template <int MASK>
__device__ __forceinline__ float row_carry(float v, float old) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), 0x142, MASK, 0xf, false));
}

// A wave's chain in LDS: per position the rate R (of the pair to its right; the chain-end
// rates' sum at Z-1), |Q|^2, the CD rate w and the strand's length with its slot among the
// chain's strand vectors (LaneRec).  Behind the chain R, q2 and w are zero, the length is 1
// and the slots are the free ones.  The canonical sums of 256 positions (a group: four
// 64-position blocks, one a row of lanes) are formed at a time; MULTI: chains of more than
// one group, whose block totals are kept, one a lane.
template <bool MULTI>
struct Solo {
  LaneCtx C;
  lds_f *R, *q2, *w;
  lds_i* ns;
  int cap;
  int g;            // the group in the registers below
  float s[4], X;    // sums within a quad, and before it within its block
  float cb, P;      // sum before the lane's block, and through the lane's quad
  float tot;        // MULTI: lane b: total of block b
  int nb;           // blocks of the chain
  __device__ __forceinline__ int len(int p) const { return ns[p] & 0xffff; }
  // sums of group `group`
  __device__ __forceinline__ void scan(int group) {
    g = group;
    const int j = 64 * g + C.lane;
    vf4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (4 * j < cap) v = ((lds_f4*)R)[j];
    s[0] = v.x;
    s[1] = s[0] + v.y;
    s[2] = s[1] + v.z;
    s[3] = s[2] + v.w;
    float H = s[3];
    H = H + dppf<kRowShr1>(H, 0.0f);
    H = H + dppf<kRowShr2>(H, 0.0f);
    H = H + dppf<kRowShr4>(H, 0.0f);
    H = H + dppf<kRowShr8>(H, 0.0f);
    X = dppf<kRowShr1>(H, 0.0f);
  }
  // the same with the sum c0 before the group: the blocks' totals added in order
  __device__ __forceinline__ void carry(float c0) {
    const float I = X + s[3];
    cb = c0;
    P = cb + I;
    cb = row_carry<2>(P, cb);
    P = cb + I;
    cb = row_carry<4>(P, cb);
    P = cb + I;
    cb = row_carry<8>(P, cb);
    P = cb + I;
  }
  // after rates of the group changed
  __device__ __forceinline__ void refresh(int group) {
    scan(group);
    if constexpr (MULTI) {
      const float t = from_lane(X + s[3], 16 * (C.lane & 3) + 15);
      tot = C.lane >> 2 == g ? t : tot;
    } else {
      carry(0.0f);
    }
  }
  __device__ __forceinline__ void refresh_to(int g0, int g1) {
    if constexpr (MULTI) {
      for (int k = g1; k > g0; --k) refresh(k);
    }
    refresh(g0);
  }
};

// The chain's total rate; c: the sums over the blocks (MULTI: lane b: blocks 0 .. b, added
// in order; further rounds leave them as they are).
template <bool MULTI>
__device__ __forceinline__ float solo_total(const Solo<MULTI>& S, float& c) {
  if constexpr (!MULTI) return lane_read(S.P, 63);
  c = S.tot;
  for (int b = 1; b < S.nb; b += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = S.tot + dppf<kWaveShr1>(c, 0.0f);
  }
  return lane_read(c, S.nb - 1);
}

// The first position whose inclusive sum exceeds pr (-1: none, or behind the chain, whose
// sums may round above its last one), and the sum before it.  Of a chain of many groups a
// block can hold it only if the sum before the block plus the block's total, with more
// than the rounding of its inner sums to spare, exceeds pr.
template <bool MULTI>
__device__ __forceinline__ int solo_pick(Solo<MULTI>& S, float c, float pr, int Z, float& before) {
  const int lane = S.C.lane;
  float cin = 0.0f;
  uint64_t cand = 1;
  if constexpr (MULTI) {
    cin = dppf<kWaveShr1>(c, 0.0f);  // lane b: the sum before block b
    cand = __ballot(cin + S.tot * (1.0f + 0x1p-19f) > pr) & (~0ull >> (64 - S.nb));
  }
  while (cand) {
    const int g = MULTI ? (int)__builtin_ctzll(cand) >> 2 : 0;
    float c0 = 0.0f;
    if constexpr (MULTI) {
      if (g != __builtin_amdgcn_readfirstlane(S.g)) S.scan(g);
      c0 = lane_read(cin, 4 * g);
      S.carry(c0);
    }
    const uint64_t m = __ballot(S.P > pr);
    if (m) {
      // in every lane: the position within its quad, and the sum before it
      const float g0 = S.cb + (S.X + S.s[0]), g1 = S.cb + (S.X + S.s[1]), g2 = S.cb + (S.X + S.s[2]);
      const float gl = dppf<kWaveShr1>(S.P, c0);
      const bool h0 = g0 > pr, h1 = g1 > pr, h2 = g2 > pr;
      const int i = h0 ? 0 : (h1 ? 1 : (h2 ? 2 : 3));
      const float b = h0 ? gl : (h1 ? g0 : (h2 ? g1 : g2));
      const int l = (int)__builtin_ctzll(m);
      before = lane_read(b, l);
      const int p = 4 * (64 * g + l) + lane_read(i, l);
      return p < Z ? p : -1;
    }
    if constexpr (!MULTI) break;
    cand &= g < 15 ? ~0ull << (4 * (g + 1)) : 0ull;
  }
  return -1;
}

// The pairs of four strands in lanes 0..3 of a row: positions x, lengths N, |Q|^2 and CD
// rates of consecutive strands of a chain of Z; lane i gets the rates of the pair (i, i+1).
struct SoloPairs {
  float wp, wm, R;
};
template <bool MULTI>
__device__ __forceinline__ SoloPairs solo_pairs(const Solo<MULTI>& S, const LaneChain& H, int x, int N, float q,
                                                float w, int Z) {
  SoloPairs W;
  const LaneStrand t = lane_strand(S.C, N, q, x == 0 || x == Z - 1);
  LaneStrand u;  // the next strand's
  u.a = dppf<kRowShl1>(t.a, 0.0f);
  u.b = dppf<kRowShl1>(t.b, 0.0f);
  u.pp = dppf<kRowShl1>(t.pp, 0.0f);
  u.pm = dppf<kRowShl1>(t.pm, 0.0f);
  u.xp = dppi<kRowShl1>(t.xp, 0);
  u.xm = dppi<kRowShl1>(t.xm, 0);
  const bool far = lane_pair(S.C, t, u, W.wp, W.wm);
  W.R = lane_total(H.cd, H.cc, N, W.wp, W.wm, w);
  const int Nn = dppi<kRowShl1>(N, 1);
  const bool any = S.C.rl < 3 && (uint32_t)x < (uint32_t)(Z - 1) && (far || N + Nn >= kLaneN);
  if (__ballot(any)) {
    const float qn = dppf<kRowShl1>(q, 0.0f);
    if (any) lane_pair_any(H.ens, H.cd, N, Nn, q, qn, w, x == 0, x + 2 == Z, W.wp, W.wm, W.R);
  }
  return W;
}

// Moves the positions first .. end-1 of the arrays by one: from the left (open) or the
// right neighbour.
template <bool MULTI>
__device__ __forceinline__ void solo_move(const Solo<MULTI>& S, int first, int end, bool open) {
  if (first >= end) return;
  const int g0 = MULTI ? first >> 8 : 0, g1 = MULTI ? (end - 1) >> 8 : 0;
  for (int i = 0; i <= g1 - g0; ++i) {
    const int g = open ? g1 - i : g0 + i;
    const int j = 64 * g + S.C.lane, p0 = 4 * j;
    const bool on = p0 + 3 >= first && p0 < end;
    // (lanes beyond the arrays read their last quad)
    const int jc = min(j, (S.cap >> 2) - 1), pn = min(max(open ? p0 - 1 : p0 + 4, 0), S.cap - 1);
    vi4 v[4];
    int e[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      lds_i* A = a == 0 ? S.ns : (lds_i*)(a == 1 ? S.R : (a == 2 ? S.q2 : S.w));
      v[a] = ((lds_i4*)A)[jc];
      e[a] = A[pn];
    }
    wave_lds_sync();
    if (on) {
      const bool m0 = p0 >= first, m1 = p0 + 1 >= first && p0 + 1 < end, m2 = p0 + 2 >= first && p0 + 2 < end,
                 m3 = p0 + 3 < end;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        lds_i* A = a == 0 ? S.ns : (lds_i*)(a == 1 ? S.R : (a == 2 ? S.q2 : S.w));
        const vi4 o = v[a];
        ((lds_i4*)A)[j] = vi4{m0 ? (open ? e[a] : o.y) : o.x, m1 ? (open ? o.x : o.z) : o.y,
                              m2 ? (open ? o.y : o.w) : o.z, m3 ? (open ? o.z : e[a]) : o.w};
      }
    }
    wave_lds_sync();
  }
}

// A split or merge of strands (LaneEvent).
template <bool MULTI>
__device__ __forceinline__ void solo_event(Solo<MULTI>& S, const KmcArgs& a, LaneChain& H, int Z) {
  const int rl = S.C.rl;
  LaneEvent E;
  E.place(H);
  const int e = __builtin_amdgcn_readfirstlane(E.e);
  const bool open = __builtin_amdgcn_readfirstlane(E.dir) > 0;
  // the old strands e-1 .. e+2 in lanes 0..3
  const int x = e - 1 + rl, xc = min(max(x, 0), S.cap - 1);
  const bool in = rl < 4 && (uint32_t)x < (uint32_t)Z;
  const int n = S.ns[xc], fs = S.ns[min(Z, S.cap - 1)];  // (the first free slot)
  float q = S.q2[xc], w = S.w[xc];
  int N = in ? n & 0xffff : 1;
  const int sl0 = (int)((uint32_t)lane_read(n, 1) >> 16), sl2 = (int)((uint32_t)lane_read(n, 2) >> 16);
  const int sl1 = open ? (int)((uint32_t)__builtin_amdgcn_readfirstlane(fs) >> 16) : sl2;
  const int64_t v0 = H.base + sl0, v1 = H.base + (open ? sl0 : sl2);
  const float ax = a.ch.Qx[v0], ay = a.ch.Qy[v0], az = a.ch.Qz[v0];
  const float bx = a.ch.Qx[v1], by = a.ch.Qy[v1], bz = a.ch.Qz[v1];
  solo_move(S, open ? e + 2 : e + 1, open ? Z + 1 : Z - 1, open);
  E.apply(a, H, lane_read(N, 0), lane_read(N, 1), lane_read(N, 2), lane_read(N, 3), lane_read(w, 1), lane_read(w, 2),
          ax, ay, az, bx, by, bz);
  const int Zn = open ? Z + 1 : Z - 1;
  S.nb = (Zn + 63) >> 6;
  // the new ones in the same lanes
  const bool l1 = rl == 1, l2 = rl == 2;
  const float ex = l1 ? E.x0 : E.x1, ey = l1 ? E.y0 : E.y1, ez = l1 ? E.z0 : E.z1;
  const float eq = q2_of(ex, ey, ez), ew = l1 ? E.w0 : E.w1;
  const int en = l1 ? E.n0 : E.n1;
  {
    const int Nm = open ? dppi<kRowShr1>(N, 1) : dppi<kRowShl1>(N, 1);
    const float qm = open ? dppf<kRowShr1>(q, 0.0f) : dppf<kRowShl1>(q, 0.0f);
    const bool mine = l1 || (l2 && open);
    N = mine ? en : (rl < 2 ? N : (rl == 3 && !open ? 1 : Nm));
    q = mine ? eq : (rl < 2 ? q : qm);
    w = mine ? ew : w;
  }
  // a merge's free slot goes behind the chain
  if (S.C.row == 0 && (l1 || l2)) {
    const bool freed = l2 && !open;
    const int at = l1 ? e : (open ? e + 1 : Z - 1);
    const int sl = l1 ? sl0 : sl1;
    S.ns[at] = (freed ? 1 : en) | sl << 16;
    S.q2[at] = freed ? 0.0f : eq;
    S.w[at] = freed ? 0.0f : ew;
    if (!freed) {
      const int64_t o = H.base + sl;
      a.ch.Qx[o] = ex; a.ch.Qy[o] = ey; a.ch.Qz[o] = ez;
    }
  }
  const SoloPairs W = solo_pairs(S, H, x, N, q, w, Zn);
  const float eend = lane_ends(H).total();
  {
    // the pairs around (a merge leaves the one behind it as it was, moved), the chain end
    // and the position a merge left
    const int at = rl < 3 ? x : (rl == 3 ? Zn - 1 : Z - 1);
    const float v = rl < 3 ? W.R : (rl == 3 ? eend : 0.0f);
    const bool on = rl < 3 ? (rl < 2 || open) && (uint32_t)x < (uint32_t)(Zn - 1) : (rl == 3 || (rl == 4 && !open));
    if (S.C.row == 0 && on) S.R[at] = v;
  }
  wave_lds_sync();
  S.refresh_to(max(e - 1, 0) >> 8, (max(Z, Zn) - 1) >> 8);
}

// One jump.  Strands p-1 .. p+2 lie in lanes 0..3 of a row, the pairs they form in lanes
// 0..2: row 0 as they are, row 1 after a Kuhn step from p+1 to p, row 2 after one from p to
// p+1.
template <bool MULTI>
__device__ __forceinline__ void solo_jump(Solo<MULTI>& S, LaneChain& H, const uint4& rnd, int Z) {
  float c = 0.0f, before = 0.0f;
  const float W = solo_total(S, c);
  const float pr = W * u01(rnd.x);
  if (!lane_clock(H, W, rnd)) return;
  const int p = solo_pick(S, c, pr, Z, before);
  if (p < 0) return;  // no position: the clock moves, the chain does not
  const int rl = S.C.rl, row = S.C.row;
  const int x = p - 1 + rl, xc = min(max(x, 0), S.cap - 1);
  const float q = S.q2[xc], w = S.w[xc];
  const int n = S.ns[xc];
  const int step = row == 1 ? 1 : (row == 2 ? -1 : 0);
  const int N = ((rl < 4 && (uint32_t)x < (uint32_t)Z) ? n & 0xffff : 1) + (rl == 1 ? step : (rl == 2 ? -step : 0));
  const SoloPairs V = solo_pairs(S, H, x, N, q, w, Z);
  float r = p == 0 ? pr : pr - before;
  int kind = lane_kind(H, p < Z - 1, w, V.wp, V.wm, N, r);  // (lane 1 has the picked pair's)
  kind = lane_read(kind, 1);
  if (kind != kEvShiftP && kind != kEvShiftM) {
    H.kind = kind;
    H.p = p;
    H.r = lane_read(r, 1);
    H.rz = rnd.z;
    H.rw = rnd.w;
    return;
  }
  const int rs = kind == kEvShiftP ? 1 : 2;
  if (row == rs && rl < 3) {
    if ((uint32_t)x < (uint32_t)(Z - 1)) S.R[x] = V.R;
    if (rl > 0) S.ns[x] = N | (n & ~0xffff);
  }
  const int g = p >> 8;
  if (p <= 1 || p >= Z - 3) {
    lane_shift_ends(H, p, lane_read(N, 16 * rs + 1), lane_read(N, 16 * rs + 2));
    lane_end_rates(H);
    const float eend = lane_ends(H).total();
    if (S.C.lane == 0) S.R[Z - 1] = eend;
    wave_lds_sync();
    if constexpr (MULTI) {
      if ((Z - 1) >> 8 != g) S.refresh((Z - 1) >> 8);
    }
  }
  wave_lds_sync();
  if constexpr (MULTI) {
    if ((p & 255) == 255) S.refresh(g + 1);
    if ((p & 255) == 0 && p > 0) S.refresh(g - 1);
  }
  S.refresh(g);
}

// Sum of the canonical block sums over the groups, block by block; I: the inclusive sum of
// lane 15 of each row is the block's.
__device__ __forceinline__ void solo_add(float& sum, float I, int g, int nb) {
  const float b0 = lane_read(I, 15), b1 = lane_read(I, 31), b2 = lane_read(I, 47), b3 = lane_read(I, 63);
  sum = g == 0 ? b0 : sum + b0;
  if (4 * g + 1 < nb) sum = sum + b1;
  if (4 * g + 2 < nb) sum = sum + b2;
  if (4 * g + 3 < nb) sum = sum + b3;
}

// One G(t) or MSD sample (eq_sample and com_sample in dsm_kmc.h) into the staging rows.
template <bool MULTI>
__device__ __forceinline__ void solo_sample(const Solo<MULTI>& S, const KmcArgs& a, const LaneChain& H) {
  const int Z = __builtin_amdgcn_readfirstlane(H.Z), ng = (Z + 255) >> 8;
  const EnsParams* P = a.ens + H.ens;
  float tot[3] = {0.0f, 0.0f, 0.0f}, carry[3] = {0.0f, 0.0f, 0.0f};
  const float nkf = (float)a.ch.nk[H.c];
  for (int g = 0; g < ng; ++g) {
    const int p0 = 4 * (64 * g + S.C.lane);
    float x[3][4];
    int n[4] = {1, 1, 1, 1};
#pragma unroll
    for (int k = 0; k < 4; ++k) x[0][k] = x[1][k] = x[2][k] = 0.0f;
    if (p0 < Z) {
      const vi4 v = ((lds_i4*)S.ns)[p0 >> 2];
      const int e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        n[k] = e[k] & 0xffff;
        const bool on = p0 + k < Z;
        const int64_t o = H.base + (on ? (int)((uint32_t)e[k] >> 16) : 0);
        const float qx = a.ch.Qx[o], qy = a.ch.Qy[o], qz = a.ch.Qz[o];
        x[0][k] = on ? qx : 0.0f;
        x[1][k] = on ? qy : 0.0f;
        x[2][k] = on ? qz : 0.0f;
      }
    }
#pragma unroll
    for (int comp = 0; comp < 3; ++comp) {
      float v[4], I[4];
      if (H.msd) {
        block_scan4(x[comp][0], x[comp][1], x[comp][2], x[comp][3], I);
        const float b0 = lane_read(I[3], 15), b1 = lane_read(I[3], 31), b2 = lane_read(I[3], 47),
                    b3 = lane_read(I[3], 63);
        const float c0 = carry[comp], c1 = g == 0 ? b0 : c0 + b0, c2 = c1 + b1, c3 = c2 + b2;
        carry[comp] = c3 + b3;
        const int row = S.C.row;
        const float cb = row == 0 ? c0 : (row == 1 ? c1 : (row == 2 ? c2 : c3));
        float out[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) out[k] = g == 0 && row == 0 ? I[k] : cb + I[k];
        const float before = dppf<kRowShr1>(out[3], 0.0f);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float Pk = k > 0 ? out[k > 0 ? k - 1 : 0] : (S.C.rl == 0 ? cb : before);
          v[k] = p0 + k < Z ? ((Pk + x[comp][k] * 0.5f) * (float)n[k]) / nkf : 0.0f;
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool on = p0 + k < Z;
          const float t3 = on ? 3.0f / (float)n[k] : 0.0f;
          const float u = comp == 1 ? x[1][k] : x[0][k], z = comp == 0 ? x[1][k] : x[2][k];
          v[k] = on ? (u * z) * t3 : 0.0f;
        }
      }
      block_scan4(v[0], v[1], v[2], v[3], I);
      solo_add(tot[comp], I[3], g, S.nb);
    }
  }
  if (S.C.lane == 0 && H.next_sample >= P->k0) {
    float* o = a.stage + P->stage_off + ((H.next_sample - P->k0) * P->nchains + a.ch.local[H.c]) * 3;
    if (H.msd) {
      const float* r = a.ch.R1 + 3 * (int64_t)H.c;
      o[0] = tot[0] + r[0]; o[1] = tot[1] + r[1]; o[2] = tot[2] + r[2];
    } else {
      o[0] = -tot[0]; o[1] = -tot[1]; o[2] = -tot[2];
    }
  }
}

// Chain H.c from the chain arrays into LDS, its rates and sums.
template <bool MULTI>
__device__ __forceinline__ void solo_load(Solo<MULTI>& S, const KmcArgs& a, const LaneChain& H) {
  const int Z = __builtin_amdgcn_readfirstlane(H.Z), ng = (S.cap + 255) >> 8;
  S.nb = (Z + 63) >> 6;
  for (int g = 0; g < ng; ++g) {
    const int j = 64 * g + S.C.lane, p0 = 4 * j;
    if (p0 >= S.cap) continue;
    vf4 q = {0.f, 0.f, 0.f, 0.f}, w = q;
    vi4 n = {p0 << 16 | 1, (p0 + 1) << 16 | 1, (p0 + 2) << 16 | 1, (p0 + 3) << 16 | 1};
    if (p0 < Z) {
      const int64_t o = H.base + p0;
      const float4 x = *(const float4*)(a.ch.Qx + o), y = *(const float4*)(a.ch.Qy + o),
                   z = *(const float4*)(a.ch.Qz + o), ww = *(const float4*)(a.ch.w + o);
      const int4 m = *(const int4*)(a.ch.N + o);
      const bool i1 = p0 + 1 < Z, i2 = p0 + 2 < Z, i3 = p0 + 3 < Z;
      q = vf4{q2_of(x.x, y.x, z.x), i1 ? q2_of(x.y, y.y, z.y) : 0.f, i2 ? q2_of(x.z, y.z, z.z) : 0.f,
              i3 ? q2_of(x.w, y.w, z.w) : 0.f};
      w = vf4{ww.x, i1 ? ww.y : 0.f, i2 ? ww.z : 0.f, i3 ? ww.w : 0.f};
      n = vi4{p0 << 16 | m.x, (p0 + 1) << 16 | (i1 ? m.y : 1), (p0 + 2) << 16 | (i2 ? m.z : 1),
              (p0 + 3) << 16 | (i3 ? m.w : 1)};
    }
    ((lds_f4*)S.q2)[j] = q;
    ((lds_f4*)S.w)[j] = w;
    ((lds_i4*)S.ns)[j] = n;
  }
  wave_lds_sync();
  const float ee = lane_ends(H).total();
  for (int g = 0; g < ng; ++g) {
    const int j = 64 * g + S.C.lane, p0 = 4 * j;
    if (p0 < S.cap) {
      float R[4] = {0.f, 0.f, 0.f, 0.f};
      if (p0 < Z) {
        const vf4 qv = ((lds_f4*)S.q2)[j], wv = ((lds_f4*)S.w)[j];
        const vi4 nv = ((lds_i4*)S.ns)[j];
        const int pn = min(p0 + 4, S.cap - 1);
        const int N[5] = {nv.x & 0xffff, nv.y & 0xffff, nv.z & 0xffff, nv.w & 0xffff, p0 + 4 < Z ? S.len(pn) : 1};
        const float q[5] = {qv.x, qv.y, qv.z, qv.w, S.q2[pn]}, ww[4] = {wv.x, wv.y, wv.z, wv.w};
        lane_quad_rates(S.C, H.ens, H.cd, H.cc, Z, p0, N, q, ww, ee, R);
      }
      ((lds_f4*)S.R)[j] = vf4{R[0], R[1], R[2], R[3]};
    }
  }
  wave_lds_sync();
  S.tot = 0.0f;
  S.refresh_to(0, (Z - 1) >> 8);
}

// The chain back into the chain arrays, strand vectors in position order (through the
// chain's LDS, which is not needed any more).
template <bool MULTI>
__device__ __forceinline__ void solo_store(const Solo<MULTI>& S, const KmcArgs& a, const LaneChain& H) {
  const int Z = __builtin_amdgcn_readfirstlane(H.Z), ng = (Z + 255) >> 8;
  for (int g = 0; g < ng; ++g) {
    const int j = 64 * g + S.C.lane, p0 = 4 * j;
    if (p0 < Z) {
      const int64_t o = H.base + p0;
      const vi4 n = ((lds_i4*)S.ns)[j];
      const vf4 w = ((lds_f4*)S.w)[j];
      *(int4*)(a.ch.N + o) = make_int4(n.x & 0xffff, n.y & 0xffff, n.z & 0xffff, n.w & 0xffff);
      *(float4*)(a.ch.w + o) = make_float4(w.x, w.y, w.z, w.w);
      const int e[4] = {n.x, n.y, n.z, n.w};
      float x[4], y[4], z[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int64_t v = H.base + (p0 + k < Z ? (int)((uint32_t)e[k] >> 16) : 0);
        x[k] = a.ch.Qx[v]; y[k] = a.ch.Qy[v]; z[k] = a.ch.Qz[v];
      }
      ((lds_f4*)S.R)[j] = vf4{x[0], x[1], x[2], x[3]};
      ((lds_f4*)S.q2)[j] = vf4{y[0], y[1], y[2], y[3]};
      ((lds_f4*)S.w)[j] = vf4{z[0], z[1], z[2], z[3]};
    }
  }
  wave_lds_sync();
  for (int g = 0; g < ng; ++g) {
    const int j = 64 * g + S.C.lane, p0 = 4 * j;
    if (p0 < Z) {
      const int64_t o = H.base + p0;
      const vf4 x = ((lds_f4*)S.R)[j], y = ((lds_f4*)S.q2)[j], z = ((lds_f4*)S.w)[j];
      *(float4*)(a.ch.Qx + o) = make_float4(x.x, x.y, x.z, x.w);
      *(float4*)(a.ch.Qy + o) = make_float4(y.x, y.y, y.z, y.w);
      *(float4*)(a.ch.Qz + o) = make_float4(z.x, z.y, z.z, z.w);
    }
  }
  wave_lds_sync();
}

// Persistent waves, one a workgroup: each runs chains from the work list until it is
// exhausted; a chain that could outgrow `cap` positions is handed on.
template <bool MULTI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MULTI ? 3 : 4))) kmc_solo_kernel(KmcArgs a) {
  extern __shared__ float lds_dyn[];
  Solo<MULTI> S;
  S.cap = a.cap;
  S.C.tab = (lds_f*)lds_dyn;
  S.C.lane = lane_id();
  S.C.row = S.C.lane >> 4;
  S.C.rl = S.C.lane & 15;
  S.R = S.C.tab + kLaneTabFloats;
  S.q2 = S.R + S.cap;
  S.w = S.q2 + S.cap;
  S.ns = (lds_i*)(S.w + S.cap);
  S.g = 0; S.X = 0.0f; S.cb = 0.0f; S.P = 0.0f; S.tot = 0.0f; S.nb = 1;
  for (auto& v : S.s) v = 0.0f;
  const int n_work = *a.n_work;
  if ((int)blockIdx.x >= n_work) return;  // more waves than chains: nothing is left for it
  for (int i = S.C.lane; i < kLaneTabFloats; i += 64) S.C.tab[i] = a.lane_tab[i];
  wave_lds_sync();
  const double kNever = __longlong_as_double(0x7ff0000000000000ll);
  LaneChain H;
  for (;;) {
    int ent = 0;
    if (S.C.lane == 0) ent = atomicAdd(a.queue, 1);
    ent = __builtin_amdgcn_readfirstlane(ent);
    if (ent >= n_work) break;
    const int c = __builtin_amdgcn_readfirstlane(a.work[ent]);
    if (c < 0 || a.ch.stall[c] != 0) continue;
    const int z = __builtin_amdgcn_readfirstlane(a.ch.Z[c]);
    if (z >= S.cap) {
      if (S.C.lane == 0) a.overflow[atomicAdd(a.n_overflow, 1)] = c;
      continue;
    }
    H.c = c;
    H.Z = z;
    lane_begin(a, H);
    solo_load(S, a, H);
    uint64_t ev0 = H.ev;                             // lane k: random words of jump ev0 + k
    uint4 rnd = lane_step_words(H, ev0 + S.C.lane);
    bool outgrown = false;
    for (;;) {
      while (__builtin_amdgcn_readfirstlane(H.t > H.t_next)) {
        solo_sample(S, a, H);
        ++H.next_sample;
        const EnsParams* P = a.ens + H.ens;
        H.t_next = H.next_sample < P->k_end ? (double)H.next_sample * P->delta : kNever;
      }
      if (!__builtin_amdgcn_readfirstlane(H.stall == 0 && H.t < H.t_end && H.left > 0)) break;
      const int Zc = __builtin_amdgcn_readfirstlane(H.Z);
      if (Zc >= S.cap) { outgrown = true; break; }
      int k = __builtin_amdgcn_readfirstlane((int)(H.ev - ev0));
      if (k >= 64) {
        ev0 = H.ev;
        rnd = lane_step_words(H, ev0 + S.C.lane);
        k = 0;
      }
      uint4 r;
      r.x = (uint32_t)lane_read((int)rnd.x, k);
      r.y = (uint32_t)lane_read((int)rnd.y, k);
      r.z = (uint32_t)lane_read((int)rnd.z, k);
      r.w = (uint32_t)lane_read((int)rnd.w, k);
      solo_jump(S, H, r, Zc);
      if (__builtin_amdgcn_readfirstlane(H.kind) != kEvNone) solo_event(S, a, H, Zc);
    }
    solo_store(S, a, H);
    if (S.C.lane == 0) {
      a.ch.Z[c] = H.Z; a.ch.stall[c] = H.stall; a.ch.next_sample[c] = H.next_sample; a.ch.t[c] = H.t;
      a.ch.ev[c] = H.ev; a.ch.zsum[c] += H.zsum; a.ch.dt_prev[c] = H.dt_prev;
      if (outgrown) a.overflow[atomicAdd(a.n_overflow, 1)] = c;
    }
  }
}

}  // namespace dsm
