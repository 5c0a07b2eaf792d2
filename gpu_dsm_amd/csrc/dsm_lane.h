// dsm_lane.h -- the lane form of the KMC jump kernels: one chain per lane, 64 per wave.
// Included by dsm_lane_inst.hip.
//
// Why.  The row, pair and wave forms (dsm_kmc.h) give a chain 16 to 64 lanes and scan all
// its positions at every jump: about 430-580 VALU instructions per wave step for one to
// four chains.  A jump changes three pair rates, though, and needs only (a) the exact
// canonical total W, (b) the position whose inclusive sum first exceeds W*u and (c) the
// rates next to it.  Here every lane does that for its own chain: the canonical tree of a
// 64-position block (serial over four slots, Hillis-Steele over 16 quads, dsm_kmc.h) is a
// function of the quad sums alone, so a lane keeps those in registers, evaluates the tree
// from them (49 additions a block), reads the picked quad's four rates and the strands
// around the position, and rewrites at most three quad sums.  Every sum is formed from the
// same operands in the same order, so a chain makes the same jumps bit for bit.
//
// State while a chain runs: the cached rates R (of the pair to a position's right; the
// chain-end rates' sum at Z-1) in LDS, four positions side by side in a column per lane;
// a 12-byte record {|Q|^2, w, N} per position in `rec` (L2 / Infinity Cache); Q in the
// chain arrays; header and quad sums in registers.
//
// What bounds it (131,072 chains of Nk 100, one 16 tau_K window, 76 positions: 5.1 ms against
// 9.0 ms in the row form plus 0.76 ms for its overflow in the wave form): per jump 35 VALU
// instructions instead of 103, issued on about half of the cycles.  LDS holds two waves a
// SIMD (512 lanes a CU at 76 positions), so the loads from L2 and Infinity Cache
// are only partly hidden, and 38 of a wave's 64 lanes are
// ready in an average step, the others waiting for row work.  Rates and records both in
// memory (three waves a SIMD): 9.1 ms, at 640 bytes of traffic a jump; rates, lengths and
// quad sums all in LDS (one wave a SIMD): 7.8 ms.
//
// What is not one lane's work is done by 16-lane rows, four chains at a time: loading a
// chain from the chain arrays, writing it back, taking a sample, and the one-position
// shift of the arrays in memory after a split or merge of strands.  Lanes that need one
// of these wait until enough of the wave's lanes do, since the step costs the wave the
// same for one lane as for many.
#pragma once
#include "dsm_kmc.h"
#include "dsm_launch.h"

namespace dsm {

// LDS of a workgroup: {SP, SM, PP, PM}[N < kLaneN], FR[x < kLaneFR] (all ensembles and
// waves share them: these tables depend on N alone), then per wave R[NQ][S][4] for S lane
// columns (S odd, so a row that walks one lane's column meets every bank group once).
struct LaneTab {
  float sp, sm, pp, pm;
};

// dexpf for |x| <= 87 (the same operations; the power of two is applied by ldexp, exact
// here as the product is); anything for other arguments, which the callers look for
__device__ __forceinline__ float lane_exp(float x) {
  const float n = __builtin_rintf(x * 0x1.715476p+0f);
  float r = __builtin_fmaf(-n, 0x1.62e4p-1f, x);
  r = __builtin_fmaf(-n, 0x1.7f7d1cp-20f, r);
  float q = 0x1.a01a02p-13f;
  q = __builtin_fmaf(q, r, 0x1.6c16c2p-10f);
  q = __builtin_fmaf(q, r, 0x1.111112p-7f);
  q = __builtin_fmaf(q, r, 0x1.555556p-5f);
  q = __builtin_fmaf(q, r, 0x1.555556p-3f);
  q = __builtin_fmaf(q, r, 0x1p-1f);
  q = __builtin_fmaf(q, r, 1.0f);
  q = __builtin_fmaf(q, r, 1.0f);
  return __builtin_amdgcn_ldexpf(q, (int)n);
}

// Philox with the 32 x 32 -> 64 products taken in one instruction each
__device__ __forceinline__ uint4 lane_philox(uint4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
    const uint64_t m0 = (uint64_t)0xD2511F53u * c.x, m1 = (uint64_t)0xCD9E8D57u * c.z;
    c = make_uint4((uint32_t)(m1 >> 32) ^ c.y ^ k0, (uint32_t)m1, (uint32_t)(m0 >> 32) ^ c.w ^ k1, (uint32_t)m0);
  }
  return c;
}

// One position in `rec`: |Q|^2, the CD rate, and the strand's length with the place of
// its vector among the chain's strand slots in the upper 16 bits.  While a chain runs,
// strand vectors stay where they are when positions shift; lane_store puts them in order.
struct LaneRec {
  float q2, w;
  int ns;
  __device__ __forceinline__ int N() const { return ns & 0xffff; }
  __device__ __forceinline__ int slot() const { return (int)((uint32_t)ns >> 16); }
};
static_assert(sizeof(LaneRec) == kLaneRecFloats * sizeof(float), "record layout");

// One lane's chain.
struct LaneChain {
  int c;                 // chain index; -1 none, -2 past the end of the list
  int ens, Z, left, stall;
  uint32_t cid, key0, key1;
  int64_t base;
  double t, t_next, t_end;
  int64_t next_sample;
  uint64_t ev;
  uint64_t zsum;         // sum of Z over the jumps made here
  float dt_prev;
  float beta, cc;        // cc: CD creation per N - 1 (0: CD off)
  float eh, et;          // creation or destruction rates at the head and the tail
  int cd, exp_wait, msd, pd;  // pd: float offset of the partner tables (-1: none)
  int N0, N1, Nz, Nz2;   // lengths at both ends: positions 0, 1, Z-1, Z-2
  uint4 rnd;             // Philox words of the next jump
  int kind, p;           // a split or merge waiting to be applied (kEvNone: none), its position,
  float r;               // the remainder of the pick and its jump's third and fourth word
  uint32_t rz, rw;
  uint32_t used[4];      // strand slots in use
};

// Chain-end rates (end_rates in dsm_kmc.h) from the lengths in registers; the tables EC,
// ED, ED2 are quotients, formed here by the same IEEE division.  eh and et change with
// the lengths at their end and between Z = 2 and the rest.
__device__ __forceinline__ void lane_end_rates(LaneChain& H) {
  const bool z2 = H.Z == 2, h1 = H.N0 == 1, t1 = H.Nz == 1;
  const float f0 = (float)H.N0, f1 = (float)H.N1, fz = (float)H.Nz, fz2 = (float)H.Nz2;
  const float hd = h1 ? (z2 ? 0.75f + (f1 + 0.25f) : 0.75f + 0.5f * f1) : H.beta * (f0 + 0.5f);
  const float td = t1 ? (z2 ? 0.75f + (fz2 + 0.25f) : 0.75f + 0.5f * fz2) : H.beta * (fz + 0.5f);
  H.eh = (h1 ? 1.0f : 2.0f) / hd;
  H.et = (t1 ? 1.0f : 2.0f) / td;
}
__device__ __forceinline__ EndRates lane_ends(const LaneChain& H) {
  const bool h1 = H.N0 == 1, t1 = H.Nz == 1;
  EndRates e;
  e.cdcz = H.cc * (float)(H.Nz - 1);
  e.sdc1 = h1 ? 0.0f : H.eh;
  e.sdcz = t1 ? 0.0f : H.et;
  e.sdd1 = h1 ? H.eh : 0.0f;
  e.sddz = t1 ? H.et : 0.0f;
  if (H.Z == 1) {  // one strand: its length is Nk
    e.sdc1 = 1.0f / (H.beta * (float)H.N0);
    e.sdcz = e.sdc1;
    e.sdd1 = 0.0f;
    e.sddz = 0.0f;
  }
  return e;
}

struct LaneCtx {
  lds_f* tab;    // {SP, SM, PP, PM}[kLaneN], FR[kLaneFR]
  lds_f4* rq;    // [quad][S]: rates R of four positions
  LaneRec* rec;
  int S;
  int lane, row, rl;
  __device__ __forceinline__ LaneTab pt(int N) const {
    const vf4 v = *(lds_f4*)(tab + 4 * N);
    return LaneTab{v.x, v.y, v.z, v.w};
  }
  __device__ __forceinline__ float fr(int x) const { return tab[4 * kLaneN + x]; }
  // rate of position p of lane column c
  __device__ __forceinline__ lds_f* rp(int p, int c) const { return (lds_f*)(rq + ((p >> 2) * S + c)) + (p & 3); }
};

// What a strand of length N and |Q|^2 = q2 contributes to the rates of the two pairs it
// belongs to (pair_rate in dsm_kmc.h): at a chain end the friction index counts 4N +- 1
// instead of 2N and the length factors are 1.  pm is zero for N = 1, at the ends too: a
// strand of one Kuhn step gives none away, and its rate is 0 * exp = 0.
struct LaneStrand {
  float a, b;    // q2 SP(N), q2 SM(N)
  float pp, pm;
  int xp, xm;
};
__device__ __forceinline__ LaneStrand lane_strand(const LaneCtx& X, int N, float q2, bool end) {
  const int n = min(N, kLaneN - 1);  // (longer ones take the general form)
  const LaneTab t = X.pt(n);
  const int x = end ? 4 * n : 2 * n, d = end ? 1 : 0;
  const float one = N > 1 ? 1.0f : 0.0f;
  return LaneStrand{q2 * t.sp, q2 * t.sm, end ? 1.0f : t.pp, end ? one : t.pm, x + d, x - d};
}
// Shift rates of the pair (i, j) and whether an exponent left the range of lane_exp.
__device__ __forceinline__ bool lane_pair(const LaneCtx& X, const LaneStrand& i, const LaneStrand& j, float& wp,
                                          float& wm) {
  const float ep = i.a - j.b, em = j.a - i.b;
  wp = ((X.fr(i.xp + j.xm) * i.pp) * j.pm) * lane_exp(ep);
  wm = ((X.fr(i.xm + j.xp) * i.pm) * j.pp) * lane_exp(em);
  // (a NaN |Q|^2 makes both NaN, an infinite one at least one infinite or both NaN)
  return !(fmaxf(__builtin_fabsf(ep), __builtin_fabsf(em)) <= 87.0f);
}
__device__ __forceinline__ float lane_total(int cd, float cc, int Ni, float wp, float wm, float we) {
  return cd ? (wp + wm) + (we + cc * (float)(Ni - 1)) : (wp + wm);
}

// The kernel's arguments read again where they are needed: held over the loop, their
// pointers would take more scalar registers than there are.
__device__ __forceinline__ KmcArgs fresh_args() {
  typedef const __attribute__((address_space(4))) KmcArgs* args4;
  args4 p = (args4)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  KmcArgs b;
  __builtin_memcpy(&b, (const void*)p, sizeof(b));
  return b;
}

// The general form, through the ensemble's tables in global memory: lengths or exponents
// beyond the fast form's tables and range.
__device__ __forceinline__ void lane_pair_any(int ens, int cd, int Ni, int Nj, float q2i, float q2j, float we,
                                              bool endi, bool endj, float& wp, float& wm, float& R) {
  const KmcArgs a = fresh_args();
  const EnsParams* P = a.ens + ens;
  Tabs<false> T;
  T.n = P->nmax + 2;
  T.b = (TabPtr<false>::type)(a.tabs + P->tab_off);
  pair_rate<false>(T, cd, Ni, Nj, q2i, q2j, we, endi, endj, wp, wm, R);
}

// Rates of the pairs (A+i, A+i+1), i = 0..2, from the records of positions A..A+3 of a
// chain of Z strands; pairs outside 0..Z-2 get a value nobody reads.  Lengths of
// positions outside the chain must be given as 1.
__device__ __forceinline__ void lane_pairs3(const LaneCtx& X, const LaneChain& H, int A, int Z, const int (&N)[4],
                                            const float (&q)[4], const float (&w)[3], float (&R)[3]) {
  LaneStrand t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = lane_strand(X, N[i], q[i], A + i == 0 || A + i == Z - 1);
  bool slow = N[0] + N[1] + N[2] + N[3] >= kLaneN;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    float wp, wm;
    slow |= lane_pair(X, t[i], t[i + 1], wp, wm);
    R[i] = lane_total(H.cd, H.cc, N[i], wp, wm, w[i]);
  }
  if (slow) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float wp, wm;
      if (A + i >= 0 && A + i <= Z - 2)
        lane_pair_any(H.ens, H.cd, N[i], N[i + 1], q[i], q[i + 1], w[i], A + i == 0, A + i + 2 == Z, wp, wm, R[i]);
    }
  }
}

// The canonical tree over the quads [16 B, min(NQ, 16 B + 16)) of a block: X[l] = sum
// before quad l (the exclusive lane prefix), I3[l] = X[l] + s[l] the inclusive sum of quad
// l; returns the block's total (I3 of lane 15).  Quads beyond NQ hold no position: their
// sums are zero, so additions with them are left out (x + 0 = x; rates are never -0).
template <int NQ, int B>
__device__ __forceinline__ float lane_tree(const float (&lf)[NQ], float (&X)[16], float (&I3)[16]) {
  constexpr int n = NQ - 16 * B < 16 ? NQ - 16 * B : 16;
  float h[16];
  bool z[16];
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    z[l] = l >= n;
    h[l] = l < n ? lf[16 * B + (l < n ? l : 0)] : 0.0f;
  }
#pragma unroll
  for (int d = 1; d < 16; d *= 2) {
#pragma unroll
    for (int l = 15; l >= 1; --l) {
      if (l < d) continue;
      if (z[l]) { h[l] = h[l - d]; z[l] = z[l - d]; }
      else if (!z[l - d]) h[l] = h[l] + h[l - d];
    }
  }
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    X[l] = l > 0 ? h[l > 0 ? l - 1 : 0] : 0.0f;
    I3[l] = l < n ? (l > 0 ? X[l] + lf[16 * B + (l < n ? l : 0)] : lf[16 * B]) : X[l];
  }
  return I3[15];
}

// Quad sums of the lane's own column (the rates at positions >= Z are zero there).
template <int NQ>
__device__ __forceinline__ void lane_leaves(const LaneCtx& C, float (&lf)[NQ]) {
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const vf4 v = C.rq[j * C.S + C.lane];
    lf[j] = ((v.x + v.y) + v.z) + v.w;
  }
}

// ------------------------------------------------------------------ row work
// Four chains at a time: row r works for the lane `src` of its turn in `m` (-1: none);
// m loses the lanes taken.
__device__ __forceinline__ int row_take(uint64_t& m, int row) {
  int src = -1;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (m) {
      const int s = (int)__builtin_ctzll(m);
      m &= m - 1;
      src = row == r ? s : src;
    }
  }
  return src;
}
__device__ __forceinline__ int from_lane(int v, int src) { return __builtin_amdgcn_ds_bpermute(src << 2, v); }
__device__ __forceinline__ float from_lane(float v, int src) {
  return __int_as_float(from_lane(__float_as_int(v), src));
}
__device__ __forceinline__ int64_t from_lane(int64_t v, int src) {
  const int lo = from_lane((int)(uint32_t)(uint64_t)v, src), hi = from_lane((int)(v >> 32), src);
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// four records at a position that is a multiple of four (48 bytes, 16-byte aligned)
template <int A, int B>
__device__ __forceinline__ void rec_put4(LaneRec* r, const float (&q)[A], const float (&w)[B], const int (&N)[4]) {
  float4* o = (float4*)r;
  o[0] = make_float4(q[0], w[0], __int_as_float(N[0]), q[1]);
  o[1] = make_float4(w[1], __int_as_float(N[1]), q[2], w[2]);
  o[2] = make_float4(__int_as_float(N[2]), q[3], w[3], __int_as_float(N[3]));
}
__device__ __forceinline__ void rec_get4(const LaneRec* r, float (&q)[4], float (&w)[4], int (&N)[4]) {
  const float4* o = (const float4*)r;
  const float4 a = o[0], b = o[1], c = o[2];
  q[0] = a.x; w[0] = a.y; N[0] = __float_as_int(a.z); q[1] = a.w;
  w[1] = b.x; N[1] = __float_as_int(b.y); q[2] = b.z; w[2] = b.w;
  N[2] = __float_as_int(c.x); q[3] = c.y; w[3] = c.z; N[3] = __float_as_int(c.w);
}

// Rates of the quad of positions p0 .. p0+3 of a chain of Z strands: of the pair to a
// position's right, the chain-end rates' sum `ee` at Z-1, zero behind it.  N, q: lengths and
// |Q|^2 of positions p0 .. p0+4, lengths outside the chain given as 1.
__device__ __forceinline__ void lane_quad_rates(const LaneCtx& C, int ens, int cd, float cc, int Z, int p0,
                                                const int (&N)[5], const float (&q)[5], const float (&ww)[4], float ee,
                                                float (&R)[4]) {
  LaneStrand t[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) t[k] = lane_strand(C, N[k], q[k], p0 + k == 0 || p0 + k == Z - 1);
  bool slow = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int p = p0 + k;
    float wp, wm;
    const bool far = lane_pair(C, t[k], t[k + 1], wp, wm) || N[k] + N[k + 1] >= kLaneN;
    slow = slow || (far && p <= Z - 2);
    R[k] = p <= Z - 2 ? lane_total(cd, cc, N[k], wp, wm, ww[k]) : (p == Z - 1 ? ee : 0.0f);
  }
  if (slow) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float wp, wm;
      if (p0 + k <= Z - 2)
        lane_pair_any(ens, cd, N[k], N[k + 1], q[k], q[k + 1], ww[k], p0 + k == 0, p0 + k + 2 == Z, wp, wm, R[k]);
    }
  }
}

// Load the chains of lanes `m` from the chain arrays: rates into LDS, records into `rec`.
template <int NQ>
__device__ __forceinline__ void lane_load(const LaneCtx& C, const KmcArgs& a, const LaneChain& H, uint64_t m) {
  const float eend = lane_ends(H).total();
  while (m) {
    const int src0 = row_take(m, C.row);
    const bool act = src0 >= 0;
    const int src = act ? src0 : C.lane;
    const int Z = from_lane(H.Z, src), cd = from_lane(H.cd, src), ens = from_lane(H.ens, src);
    const int64_t base = from_lane(H.base, src);
    const float cc = from_lane(H.cc, src), ee = from_lane(eend, src);
    for (int b = 0; 16 * b < NQ; ++b) {
      const bool row_on = act && 64 * b < Z;
      if (!__ballot(row_on)) break;
      const int p0 = 64 * b + 4 * C.rl;
      float R[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (row_on && p0 < Z) {
        const int64_t o = base + p0;
        const float4 x = *(const float4*)(a.ch.Qx + o), y = *(const float4*)(a.ch.Qy + o),
                     z = *(const float4*)(a.ch.Qz + o), w = *(const float4*)(a.ch.w + o);
        const int4 n = *(const int4*)(a.ch.N + o);
        const bool more = p0 + 4 < Z;
        const int64_t o4 = o + (more ? 4 : 0);
        const float x4 = a.ch.Qx[o4], y4 = a.ch.Qy[o4], z4 = a.ch.Qz[o4];
        const int n4 = a.ch.N[o4];
        const int N[5] = {n.x, p0 + 1 < Z ? n.y : 1, p0 + 2 < Z ? n.z : 1, p0 + 3 < Z ? n.w : 1, more ? n4 : 1};
        const float q[5] = {q2_of(x.x, y.x, z.x), q2_of(x.y, y.y, z.y), q2_of(x.z, y.z, z.z), q2_of(x.w, y.w, z.w),
                            q2_of(x4, y4, z4)};
        const float ww[4] = {w.x, w.y, w.z, w.w};
        lane_quad_rates(C, ens, cd, cc, Z, p0, N, q, ww, ee, R);
        const int ns[4] = {N[0] | p0 << 16, N[1] | (p0 + 1) << 16, N[2] | (p0 + 2) << 16, N[3] | (p0 + 3) << 16};
        rec_put4(C.rec + o, q, ww, ns);
        C.rq[(p0 >> 2) * C.S + src] = vf4{R[0], R[1], R[2], R[3]};
      }
    }
  }
}

// Write the chains of lanes `m` back: lengths, CD rates, and the strand vectors from their
// slots into position order (every vector of a chain is read before one is written).
template <int NQ>
__device__ __forceinline__ void lane_store(const LaneCtx& C, const KmcArgs& a, const LaneChain& H, uint64_t m) {
  constexpr int NB = (NQ + 15) / 16;
  while (m) {
    const int src0 = row_take(m, C.row);
    const bool act = src0 >= 0;
    const int src = act ? src0 : C.lane;
    const int Z = from_lane(H.Z, src);
    const int64_t base = from_lane(H.base, src);
    float x[NB][4], y[NB][4], z[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int p0 = 64 * b + 4 * C.rl;
      if (act && p0 < Z) {
        const int64_t o = base + p0;
        float q[4], w[4];
        int ns[4];
        rec_get4(C.rec + o, q, w, ns);
        *(int4*)(a.ch.N + o) = make_int4(ns[0] & 0xffff, ns[1] & 0xffff, ns[2] & 0xffff, ns[3] & 0xffff);
        *(float4*)(a.ch.w + o) = make_float4(w[0], w[1], w[2], w[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int64_t v = base + (p0 + k < Z ? (int)((uint32_t)ns[k] >> 16) : 0);
          x[b][k] = a.ch.Qx[v]; y[b][k] = a.ch.Qy[v]; z[b][k] = a.ch.Qz[v];
        }
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int p0 = 64 * b + 4 * C.rl;
      if (act && p0 < Z) {
        const int64_t o = base + p0;
        *(float4*)(a.ch.Qx + o) = make_float4(x[b][0], x[b][1], x[b][2], x[b][3]);
        *(float4*)(a.ch.Qy + o) = make_float4(y[b][0], y[b][1], y[b][2], y[b][3]);
        *(float4*)(a.ch.Qz + o) = make_float4(z[b][0], z[b][1], z[b][2], z[b][3]);
      }
    }
  }
}

// One G(t) sample of the chains of lanes `m` (eq_sample in dsm_kmc.h) into the staging
// rows.
template <int NQ>
__device__ __forceinline__ void lane_sample(const LaneCtx& C, const KmcArgs& a, const LaneChain& H, uint64_t m) {
  while (m) {
    const int src0 = row_take(m, C.row);
    const bool act = src0 >= 0;
    const int src = act ? src0 : C.lane;
    const int Z = from_lane(H.Z, src), ens = from_lane(H.ens, src), c = from_lane(H.c, src);
    const int64_t base = from_lane(H.base, src), ns = from_lane(H.next_sample, src);
    float tot[3] = {0.0f, 0.0f, 0.0f};
    for (int b = 0; 16 * b < NQ; ++b) {
      const bool row_on = act && 64 * b < Z;
      if (!__ballot(row_on)) break;
      const int p0 = 64 * b + 4 * C.rl;
      float u[4] = {0.f, 0.f, 0.f, 0.f}, v[4] = {0.f, 0.f, 0.f, 0.f}, d[4] = {0.f, 0.f, 0.f, 0.f};
      if (row_on && p0 < Z) {
        const LaneRec* rr = C.rec + base + p0;
        int ns4[4];
        float xs[4], ys[4], zs[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) ns4[k] = rr[k].ns;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int64_t v = base + (p0 + k < Z ? (int)((uint32_t)ns4[k] >> 16) : 0);
          xs[k] = a.ch.Qx[v]; ys[k] = a.ch.Qy[v]; zs[k] = a.ch.Qz[v];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool on = p0 + k < Z;
          const float t3 = on ? 3.0f / (float)(ns4[k] & 0xffff) : 0.0f;
          u[k] = on ? (xs[k] * ys[k]) * t3 : 0.0f;
          v[k] = on ? (ys[k] * zs[k]) * t3 : 0.0f;
          d[k] = on ? (xs[k] * zs[k]) * t3 : 0.0f;
        }
      }
      float I[4];
      block_scan4(u[0], u[1], u[2], u[3], I);
      const float B0 = row_last(I[3]);
      block_scan4(v[0], v[1], v[2], v[3], I);
      const float B1 = row_last(I[3]);
      block_scan4(d[0], d[1], d[2], d[3], I);
      const float B2 = row_last(I[3]);
      if (row_on) {
        tot[0] = b == 0 ? B0 : tot[0] + B0;
        tot[1] = b == 0 ? B1 : tot[1] + B1;
        tot[2] = b == 0 ? B2 : tot[2] + B2;
      }
    }
    if (act && C.rl == 0) {
      const EnsParams* P = a.ens + ens;
      if (ns >= P->k0) {
        float* o = a.stage + P->stage_off + ((ns - P->k0) * P->nchains + a.ch.local[c]) * 3;
        o[0] = -tot[0]; o[1] = -tot[1]; o[2] = -tot[2];
      }
    }
  }
}

// One MSD sample of the chains of lanes `m`: the centre of mass (com_sample in dsm_kmc.h)
// plus R1.
template <int NQ>
__device__ __forceinline__ void lane_sample_com(const LaneCtx& C, const KmcArgs& a, const LaneChain& H, uint64_t m) {
  while (m) {
    const int src0 = row_take(m, C.row);
    const bool act = src0 >= 0;
    const int src = act ? src0 : C.lane;
    const int Z = from_lane(H.Z, src), ens = from_lane(H.ens, src), c = from_lane(H.c, src);
    const int64_t base = from_lane(H.base, src), ns = from_lane(H.next_sample, src);
    const float nkf = act ? (float)a.ch.nk[c] : 1.0f;
    float tot[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int comp = 0; comp < 3; ++comp) {
      const float* Q = comp == 0 ? a.ch.Qx : (comp == 1 ? a.ch.Qy : a.ch.Qz);
      float carry = 0.0f;
      for (int b = 0; 16 * b < NQ; ++b) {
        const bool row_on = act && 64 * b < Z;
        if (!__ballot(row_on)) break;
        const int p0 = 64 * b + 4 * C.rl;
        float q[4] = {0.f, 0.f, 0.f, 0.f}, n[4] = {0.f, 0.f, 0.f, 0.f}, I[4], v[4];
        if (row_on && p0 < Z) {
          const LaneRec* rr = C.rec + base + p0;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int s4 = rr[k].ns;
            const bool on = p0 + k < Z;
            const float x = Q[base + (on ? (int)((uint32_t)s4 >> 16) : 0)];
            q[k] = on ? x : 0.0f;
            n[k] = (float)(s4 & 0xffff);
          }
        }
        block_scan4(q[0], q[1], q[2], q[3], I);
        const float Bt = row_last(I[3]);
        float out[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) out[k] = b == 0 ? I[k] : carry + I[k];
        const float before = dppf<kRowShr1>(out[3], 0.0f);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float P = k > 0 ? out[k > 0 ? k - 1 : 0] : (C.rl == 0 ? carry : before);
          v[k] = p0 + k < Z ? ((P + q[k] * 0.5f) * n[k]) / nkf : 0.0f;
        }
        block_scan4(v[0], v[1], v[2], v[3], I);
        const float Bv = row_last(I[3]);
        if (row_on) {
          tot[comp] = b == 0 ? Bv : tot[comp] + Bv;
          carry = b == 0 ? Bt : carry + Bt;
        }
      }
    }
    if (act && C.rl == 0) {
      const EnsParams* P = a.ens + ens;
      if (ns >= P->k0) {
        float* o = a.stage + P->stage_off + ((ns - P->k0) * P->nchains + a.ch.local[c]) * 3;
        const float* r = a.ch.R1 + 3 * (int64_t)c;
        o[0] = tot[0] + r[0]; o[1] = tot[1] + r[1]; o[2] = tot[2] + r[2];
      }
    }
  }
}

// ------------------------------------------------------------------ one jump of every ready lane
__device__ __forceinline__ uint4 lane_step_words(const LaneChain& H, uint64_t ev) {
  return lane_philox(make_uint4((uint32_t)ev, (uint32_t)(ev >> 32), H.cid, kPurposeStep), H.key0, H.key1);
}

// The header of chain H.c of H.Z strands.
__device__ __forceinline__ void lane_begin(const KmcArgs& a, LaneChain& H) {
  const double kNever = __longlong_as_double(0x7ff0000000000000ll);
  const int c = H.c;
  const ChainArrays& ch = a.ch;
  H.ens = ch.ens[c]; H.stall = 0; H.cid = ch.cid[c];
  H.base = ch.base[c]; H.t = ch.t[c]; H.next_sample = ch.next_sample[c]; H.ev = ch.ev[c]; H.zsum = 0;
  H.dt_prev = ch.dt_prev[c];
  const uint64_t stop = a.use_ev_stop ? ch.ev_stop[c] : ~0ull;
  H.left = stop <= H.ev ? 0 : (stop - H.ev > 0x7fffffffull ? 0x7fffffff : (int)(stop - H.ev));
  const EnsParams* P = a.ens + H.ens;
  H.key0 = P->key0; H.key1 = P->key1; H.beta = P->beta; H.cd = P->cd; H.exp_wait = P->exp_wait;
  H.cc = P->cd ? P->c_create : 0.0f;
  H.t_end = P->t_end;
  H.t_next = H.next_sample < P->k_end && P->sample_mode != kSampleNone ? (double)H.next_sample * P->delta : kNever;
  H.N0 = ch.N[H.base]; H.N1 = ch.N[H.base + (H.Z > 1 ? 1 : 0)];
  H.Nz = ch.N[H.base + H.Z - 1]; H.Nz2 = ch.N[H.base + (H.Z > 1 ? H.Z - 2 : 0)];
  lane_end_rates(H);
  H.rnd = lane_step_words(H, H.ev);
  H.msd = P->sample_mode == kSampleMsd;
  H.pd = P->partner ? P->pd_off : -1;
  H.kind = kEvNone;
}

// A chain's total rate and, once W*u is known, the quad of the first position whose
// inclusive sum exceeds it, from its quad sums.
template <int NQ>
struct LanePick {
  float X0[16], I0[16], X1[16], I1[16], B0;
  float Xl, Gl, cin;  // sums before the quad: within its block, over the chain; before the block
  __device__ __forceinline__ float total(const float (&lf)[NQ], int Z) {
    B0 = lane_tree<NQ, 0>(lf, X0, I0);
    float B1 = 0.0f;
    if constexpr (NQ > 16) B1 = lane_tree<NQ, 1>(lf, X1, I1);
    return NQ > 16 && Z > 64 ? B0 + B1 : B0;
  }
  // (block 1 adds block 0's total; 4 * NQ: none)
  __device__ __forceinline__ int quad(float pr) {
    int qp = 4 * NQ;
    Xl = 0.0f;
    Gl = 0.0f;
#pragma unroll
    for (int k = NQ - 1; k >= 16; --k) {
      const int l = k - 16;
      const bool g = B0 + I1[l] > pr;
      qp = g ? k : qp;
      Xl = g ? X1[l] : Xl;
      Gl = g ? (l > 0 ? B0 + I1[l > 0 ? l - 1 : 0] : B0) : Gl;
    }
#pragma unroll
    for (int k = (NQ < 16 ? NQ : 16) - 1; k >= 0; --k) {
      const bool g = I0[k] > pr;
      qp = g ? k : qp;
      Xl = g ? X0[k] : Xl;
      Gl = g ? (k > 0 ? I0[k > 0 ? k - 1 : 0] : 0.0f) : Gl;
    }
    cin = NQ > 16 && qp >= 16 ? B0 : 0.0f;
    return qp;
  }
  // the position in the quad with rates R (0..3) and the sum before it
  __device__ __forceinline__ int slot(const float (&R)[4], float pr, float& before) const {
    const float s0 = R[0], s1 = s0 + R[1], s2 = s1 + R[2];
    const float g0 = cin + (Xl + s0), g1 = cin + (Xl + s1), g2 = cin + (Xl + s2);
    const int k = g0 > pr ? 0 : (g1 > pr ? 1 : (g2 > pr ? 2 : 3));
    before = k == 0 ? Gl : (k == 1 ? g0 : (k == 2 ? g1 : g2));
    return k;
  }
};

// Waiting time and clock of a jump with total rate W; false: the chain stalls.
__device__ __forceinline__ bool lane_clock(LaneChain& H, float W, const uint4& rnd) {
  float dt;
  if (H.exp_wait) dt = (-dlogf(u01(rnd.y))) / W;
  else dt = 1.0f / W;
  if (__builtin_amdgcn_classf(dt, 0x263)) {  // zero, NaN or +infinity
    H.stall = dt == 0.0f ? 1 : (dt != dt ? 2 : 3);
    return false;
  }
  H.t += (double)dt;
  H.dt_prev = dt;
  H.ev += 1;
  H.zsum += (uint64_t)H.Z;
  --H.left;
  return true;
}

// The sub-event of position p in the reference order: of a pair, from its CD and shift
// rates; at the end position, from the chain-end rates.  r becomes what is left of it.
__device__ __forceinline__ int lane_kind(const LaneChain& H, bool pair, float w, float wp, float wm, int N, float& r) {
  float v0 = H.cd ? w : 0.0f, v1 = wp, v2 = wm, v3 = H.cc * (float)(N - 1), v4 = 0.0f;
  if (!pair) {
    const EndRates er = lane_ends(H);
    v0 = er.cdcz; v1 = er.sdc1; v2 = er.sdcz; v3 = er.sdd1; v4 = er.sddz;
  }
  const float x = r;
  const bool t0 = v0 > 0.0f && x < v0;
  const float x1 = x - v0;
  const bool t1 = v1 > 0.0f && x1 < v1;
  const float x2 = x1 - v1;
  const bool t2 = v2 > 0.0f && x2 < v2;
  const float x3 = x2 - v2;
  const bool t3 = v3 > 0.0f && x3 < v3;
  const float x4 = x3 - v3;
  const bool t4 = v4 > 0.0f && x4 < v4;
  const int m = t0 ? 0 : (t1 ? 1 : (t2 ? 2 : (t3 ? 3 : (t4 ? 4 : 5))));
  r = t0 ? x : (t1 ? x1 : (t2 ? x2 : (t3 ? x3 : x4)));
  // four bits a kind
  constexpr uint32_t kPair = kEvCDd | kEvShiftP << 4 | kEvShiftM << 8 | kEvCDc << 12;
  constexpr uint32_t kEnd = kEvCDcTail | kEvSDcHead << 4 | kEvSDcTail << 8 | kEvSDdHead << 12 | kEvSDdTail << 16;
  static_assert(kEvNone == 0, "what is not listed");
  return (int)(((pair ? kPair : kEnd) >> (4 * m)) & 15);
}

// Lengths at the chain's ends after a shift that left N at p and M at p + 1; true when one
// of them changed.
__device__ __forceinline__ bool lane_shift_ends(LaneChain& H, int p, int N, int M) {
  const int Z = H.Z;
  if (p == 0) { H.N0 = N; H.N1 = M; }
  if (p == 1) H.N1 = N;
  if (p == Z - 2) { H.Nz2 = N; H.Nz = M; }
  if (p == Z - 3) H.Nz2 = M;
  return p <= 1 || p >= Z - 3;
}

// Picks the event, applies it when it is a shift of one Kuhn step across a link, and
// leaves a split or merge in (kind, p, r) for lane_rare.
template <int NQ>
__device__ __forceinline__ void lane_jump(const LaneCtx& C, LaneChain& H, float (&lf)[NQ]) {
  const uint4 rnd = H.rnd;
  const int Z = H.Z;
  LanePick<NQ> K;
  const float W = K.total(lf, Z);
  if (!lane_clock(H, W, rnd)) return;
  const float pr = W * u01(rnd.x);
  const int qp = K.quad(pr);
  if (qp > (Z - 1) >> 2) {  // no position: the clock moves, the chain does not
    H.rnd = lane_step_words(H, H.ev);
    return;
  }
  const int p4 = 4 * qp;
  const vf4 Rv = C.rq[qp * C.S + C.lane];
  float R[4] = {Rv.x, Rv.y, Rv.z, Rv.w};
  float before;
  const int k = K.slot(R, pr, before);
  const int p = p4 + k;
  float r = p == 0 ? pr : pr - before;
  // the window p-1 .. p+2 (clamped into the chain)
  LaneRec* rb = C.rec + H.base;
  const int pm1 = max(p - 1, 0), pp1 = min(p + 1, Z - 1), pp2 = min(p + 2, Z - 1);
  const LaneRec c0 = rb[pm1], c1 = rb[p], c2 = rb[pp1], c3 = rb[pp2];
  // the next jump's random words, while the window is on its way
  H.rnd = lane_step_words(H, H.ev);
  int N[4] = {c0.N(), c1.N(), c2.N(), c3.N()};
  const float q[4] = {c0.q2, c1.q2, c2.q2, c3.q2}, w[3] = {c0.w, c1.w, c2.w};
  N[2] = p + 1 < Z ? N[2] : 1;
  N[3] = p + 2 < Z ? N[3] : 1;
  const bool pair = p < Z - 1;
  float wp, wm, rr;
  const bool far = lane_pair(C, lane_strand(C, N[1], q[1], p == 0), lane_strand(C, N[2], q[2], p + 2 == Z), wp, wm);
  if ((far || N[1] + N[2] >= kLaneN) && pair)
    lane_pair_any(H.ens, H.cd, N[1], N[2], q[1], q[2], w[1], p == 0, p + 2 == Z, wp, wm, rr);
  const int kind = lane_kind(H, pair, w[1], wp, wm, N[1], r);
  if (kind != kEvShiftP && kind != kEvShiftM) {
    H.kind = kind;
    H.p = p;
    H.r = r;
    H.rz = rnd.z;
    H.rw = rnd.w;
    return;
  }
  // a shift: one Kuhn step from one strand of the pair to the other
  const int dn = kind == kEvShiftP ? 1 : -1;
  N[1] += dn;
  N[2] -= dn;
  rb[p].ns = c1.ns + dn;
  rb[p + 1].ns = c2.ns - dn;
  const bool ends = lane_shift_ends(H, p, N[1], N[2]);
  float Rn[3];
  lane_pairs3(C, H, p - 1, Z, N, q, w, Rn);
  float eend = 0.0f;
  if (ends) {
    lane_end_rates(H);
    eend = lane_ends(H).total();
  }
  const bool last = p + 1 == Z - 1;  // p + 1 is the end position
  const float Rr = last ? eend : Rn[2];
  // the new rates into the quad
  if (k == 0) { R[0] = Rn[1]; R[1] = Rr; }
  if (k == 1) { R[0] = Rn[0]; R[1] = Rn[1]; R[2] = Rr; }
  if (k == 2) { R[1] = Rn[0]; R[2] = Rn[1]; R[3] = Rr; }
  if (k == 3) { R[2] = Rn[0]; R[3] = Rn[1]; }
  const int ze = Z - 1 - p4;  // the end position within the quad (0..3) or beyond
  if (ends) {
    if (ze == 1) R[1] = eend;
    if (ze == 2) R[2] = eend;
    if (ze == 3) R[3] = eend;
  }
  C.rq[qp * C.S + C.lane] = vf4{R[0], R[1], R[2], R[3]};
  const float v0 = ((R[0] + R[1]) + R[2]) + R[3];
  // the neighbouring quad, when a changed pair lies there, and the end position's
  const int qend = (Z - 1) >> 2;
  const bool left_q = k == 0 && p > 0, right_q = k == 3;
  int side = -1, endq = -1;
  float vs = 0.0f, ve = 0.0f;
  if (left_q || right_q) {
    side = left_q ? qp - 1 : qp + 1;
    const vf4 o = C.rq[side * C.S + C.lane];
    const int zr = Z - 1 - 4 * side;
    const bool re = ends && right_q;
    const float e0 = left_q ? o.x : Rr;
    const float e1 = re && zr == 1 ? eend : o.y;
    const float e2 = re && zr == 2 ? eend : o.z;
    const float e3 = left_q ? Rn[0] : (re && zr == 3 ? eend : o.w);
    C.rq[side * C.S + C.lane] = vf4{e0, e1, e2, e3};
    vs = ((e0 + e1) + e2) + e3;
  }
  if (ends && qend != qp && !(right_q && side == qend)) {
    endq = qend;
    const vf4 o = C.rq[qend * C.S + C.lane];
    const int ke = (Z - 1) & 3;
    const float e0 = ke == 0 ? eend : o.x, e1 = ke == 1 ? eend : o.y, e2 = ke == 2 ? eend : o.z,
                e3 = ke == 3 ? eend : o.w;
    C.rq[qend * C.S + C.lane] = vf4{e0, e1, e2, e3};
    ve = ((e0 + e1) + e2) + e3;
  }
#pragma unroll
  for (int j = 0; j < NQ; ++j) lf[j] = j == qp ? v0 : (j == side ? vs : (j == endq ? ve : lf[j]));
}

// ------------------------------------------------------------------ splits and merges
// One position's shift of the records of eight chains, eight lanes a chain: each lane has
// eight positions of a 64-position block.  take chooses the chains, load fetches a block,
// store writes it back moved (splits go from the last block down, merges up).
struct RowShift {
  int gl, first, end, Z;
  bool any, open, mv, two;
  int64_t base;
  LaneRec* r;
  int p0;
  float qa[4], wa[4], qb[4], wb[4];
  int na[4], nb[4];
  LaneRec ce;
  __device__ __forceinline__ void take(const LaneCtx& C, uint64_t& mm, int e, int dir, int zold, int64_t b0) {
    const int grp = C.lane >> 3;
    gl = C.lane & 7;
    int src0 = -1;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (mm) {
        const int s = (int)__builtin_ctzll(mm);
        mm &= mm - 1;
        src0 = grp == k ? s : src0;
      }
    }
    any = src0 >= 0;
    const int src = any ? src0 : C.lane;
    // (read on every lane: a group without a chain may hold another group's source lane)
    const int re = from_lane(e, src), rd = from_lane(dir, src);
    Z = from_lane(zold, src);
    base = from_lane(b0, src);
    open = rd > 0;
    first = open ? re + 2 : re + 1;  // positions first .. end-1 move
    end = open ? Z + 1 : Z - 1;
  }
  __device__ __forceinline__ void load(const LaneCtx& C, int i, int NB) {
    const int b = open ? NB - 1 - i : i;
    p0 = 64 * b + 8 * gl;
    mv = any && p0 + 7 >= first && p0 < end;
    two = p0 + 4 < end;  // the second quad lies in the chain
    if (mv) {
      r = C.rec + base + p0;
      ce = r[open ? (p0 > 0 ? -1 : 0) : (p0 + 8 < Z ? 8 : 0)];
      rec_get4(r, qa, wa, na);
      rec_get4(r + (p0 + 4 < Z || two ? 4 : 0), qb, wb, nb);
    }
  }
  template <typename T>
  __device__ __forceinline__ T pick(T lo, T mid, T hi, int k) const {
    return p0 + k >= first && p0 + k < end ? (open ? lo : hi) : mid;
  }
  template <typename T>
  __device__ __forceinline__ void move(const T (&x)[4], const T (&y)[4], T c, T (&d)[8]) const {
    d[0] = pick(c, x[0], x[1], 0); d[1] = pick(x[0], x[1], x[2], 1); d[2] = pick(x[1], x[2], x[3], 2);
    d[3] = pick(x[2], x[3], y[0], 3); d[4] = pick(x[3], y[0], y[1], 4); d[5] = pick(y[0], y[1], y[2], 5);
    d[6] = pick(y[1], y[2], y[3], 6); d[7] = pick(y[2], y[3], c, 7);
  }
  __device__ __forceinline__ void store() {
    if (mv) {
      float q[8], w[8];
      int n[8];
      move(qa, qb, ce.q2, q);
      move(wa, wb, ce.w, w);
      move(na, nb, ce.ns, n);
      float4* o = (float4*)r;
      o[0] = make_float4(q[0], w[0], __int_as_float(n[0]), q[1]);
      o[1] = make_float4(w[1], __int_as_float(n[1]), q[2], w[2]);
      o[2] = make_float4(__int_as_float(n[2]), q[3], w[3], __int_as_float(n[3]));
      if (two) {
        o[3] = make_float4(q[4], w[4], __int_as_float(n[4]), q[5]);
        o[4] = make_float4(w[5], __int_as_float(n[5]), q[6], w[6]);
        o[5] = make_float4(__int_as_float(n[6]), q[7], w[7], __int_as_float(n[7]));
      }
    }
  }
};

// Applies the waiting events of lanes `m`.  Merge(e) joins strands e and e+1 (CD
// destruction of link e; SD destruction at the head, e = 0, or tail, e = Z-2); split(e)
// cuts strand e in two (CD creation, SD creation at the head, e = 0, or either at the
// tail, e = Z-1).  The lane computes the new values, the rows shift the arrays by one
// position behind the event, the lane writes its values, and the rows rebuild the quad
// sums.
struct LaneEvent {
  int e, dir;              // strand; +1 split, -1 merge
  int n0, n1;              // lengths at e and (split) e + 1
  float x0, y0, z0, x1, y1, z1, w0, w1;
  // The strand the waiting event acts on.
  __device__ __forceinline__ void place(const LaneChain& H) {
    const uint32_t k = 1u << H.kind;
    e = k & (1u << kEvSDcHead | 1u << kEvSDdHead) ? 0 : H.p;
    e = k & (1u << kEvSDdTail) ? H.Z - 2 : e;
    dir = k & (1u << kEvCDd | 1u << kEvSDdHead | 1u << kEvSDdTail) ? -1 : 1;
  }
  // New strands from the old lengths at e-1 .. e+2 (m), CD rates (we, we1) and vectors
  // (a, b) at e and e+1; the header follows.
  __device__ __forceinline__ void apply(const KmcArgs& A, LaneChain& H, int m0, int m1, int m2, int m3, float we,
                                        float we1, float ax, float ay, float az, float bx, float by, float bz) {
    const int Z = H.Z, kind = H.kind;
    const bool tail = kind == kEvCDcTail || kind == kEvSDcTail;
    const bool sd = kind == kEvSDcHead || kind == kEvSDcTail;
    x0 = y0 = z0 = x1 = y1 = z1 = 0.0f;
    w1 = 0.0f;
    n1 = 0;
    if (dir < 0) {
      n0 = m1 + m2;
      if (kind == kEvCDd && !(e == 0 || e == Z - 2)) { x0 = ax + bx; y0 = ay + by; z0 = az + bz; }
      if (H.msd && e == 0 && kind != kEvSDdTail) {  // the first entanglement goes: R1 moves forward by the old Q_1
        float* r1 = A.ch.R1 + 3 * (int64_t)H.c;
        r1[0] = r1[0] + bx; r1[1] = r1[1] + by; r1[2] = r1[2] + bz;
      }
      w0 = kind == kEvSDdTail ? 0.0f : we1;
      H.Z = Z - 1;
      if (e == 0) { H.N0 = n0; H.N1 = e + 2 < Z ? m3 : 1; }
      if (e == 1) H.N1 = n0;
      if (e == Z - 2) { H.Nz = n0; H.Nz2 = e > 0 ? m0 : 1; }
      if (e == Z - 3) H.Nz2 = n0;
    } else {
      // the lifetime law's constants (on their way during the random numbers): rate_ft
      // (s_At s_Ct s_Dt s_taud_inv s_one_minus_g) or rate_fdt (s_Adt s_Bdt s_Cdt s_Ddt
      // s_taud_inv)
      const EnsParams* P = A.ens + H.ens;
      const float* law = H.pd >= 0 ? A.tabs + H.pd + 5 * ((sd ? 0 : kPartnerK) + (int)(H.rw >> (32 - kPartnerBits)))
                                   : (sd ? P->law_ft : P->law_fdt);
      const float l0 = law[0], l1 = law[1], l2 = law[2], l3 = law[3], l4 = law[4];
      const uint64_t evj = H.ev - 1;
      const uint4 gr = lane_philox(make_uint4((uint32_t)evj, (uint32_t)(evj >> 32), H.cid, kPurposeGauss), H.key0, H.key1);
      float g0, g1, g2, g3;
      boxmuller(gr.x, gr.y, g0, g1);
      boxmuller(gr.z, gr.w, g2, g3);
      const float u = u01(H.rz);
      const float thr = sd ? l4 : l1, D = sd ? l2 : l3, ex = sd ? l1 : l2, slow = sd ? l3 : l4;
      const float wn = u < thr ? dpowf(__builtin_fmaf(u, l0, D), ex) : slow;
      const int Ne = m1;
      const float wc = H.cc * (float)(Ne - 1);
      n0 = kind == kEvSDcHead ? 1 : (kind == kEvSDcTail ? Ne - 1 : split_newn(H.r, Ne, wc));
      n1 = Ne - n0;
      w0 = sd && !H.cd ? 0.0f : wn;
      w1 = tail ? 0.0f : we;
      // the vectors: all zero but the new strand's at the ends
      const float num = tail ? (float)n0 : (e == 0 ? (float)n1 : (float)n0 * (float)n1);
      const float den = tail || e == 0 ? 3.0f : 3.0f * (float)Ne;
      const float sig = sqrtf(num / den);
      const float gx = g0 * sig, gy = g1 * sig, gz = g2 * sig;
      if (tail || e == 0) {
        if (Z != 1) {
          if (tail) { x0 = gx; y0 = gy; z0 = gz; }
          else { x1 = gx; y1 = gy; z1 = gz; }
        }
      } else {
        const float ratio = (float)n0 / (float)Ne;
        x0 = gx + (ax * ratio);
        y0 = gy + (ay * ratio);
        z0 = gz + (az * ratio);
        x1 = ax - x0; y1 = ay - y0; z1 = az - z0;
      }
      if (H.msd && ((kind == kEvCDc && e == 0) || kind == kEvSDcHead)) {  // a new first one: back by the new Q_1
        float* r1 = A.ch.R1 + 3 * (int64_t)H.c;
        r1[0] = r1[0] - x1; r1[1] = r1[1] - y1; r1[2] = r1[2] - z1;
      }
      H.Z = Z + 1;
      if (e == 0) { H.N0 = n0; H.N1 = n1; }
      if (e == 1) H.N1 = n0;
      if (e == Z - 1) { H.Nz2 = n0; H.Nz = n1; }
      if (e == Z - 2) H.Nz2 = n1;
    }
    H.kind = kEvNone;
    lane_end_rates(H);
  }
};

template <int NQ>
__device__ __forceinline__ void lane_rare(const LaneCtx& C, const KmcArgs& a, LaneChain& H, float (&lf)[NQ],
                                          uint64_t m) {
  const bool on = (m >> C.lane) & 1;
  LaneEvent E;
  E.e = 0;
  E.dir = 0;
  int zold = 1, sl0 = 0, sl1 = 0;
  float q0 = 0.f, q1 = 0.f;
  if (on) {
    const int Z = H.Z;
    zold = Z;
    E.place(H);
    const int e = E.e;
    // the old values at e-1 .. e+2, clamped into the chain
    const LaneRec* rb = C.rec + H.base;
    const LaneRec o0 = rb[max(e - 1, 0)], o1 = rb[e], o2 = rb[min(e + 1, Z - 1)], o3 = rb[min(e + 2, Z - 1)];
    const int64_t v1 = H.base + o1.slot(), v2 = H.base + o2.slot();
    const float ax = a.ch.Qx[v1], ay = a.ch.Qy[v1], az = a.ch.Qz[v1];
    const float bx = a.ch.Qx[v2], by = a.ch.Qy[v2], bz = a.ch.Qz[v2];
    E.apply(a, H, o0.N(), o1.N(), o2.N(), o3.N(), o1.w, o2.w, ax, ay, az, bx, by, bz);
    q0 = q2_of(E.x0, E.y0, E.z0);
    q1 = q2_of(E.x1, E.y1, E.z1);
    sl0 = o1.slot();
    const bool split = E.dir > 0;
    // a merge frees the slot of e+1, a split takes the first free one
    if (split) {
#pragma unroll
      for (int k = (NQ + 7) / 8 - 1; k >= 0; --k) sl1 = ~H.used[k] ? 32 * k + __builtin_ctz(~H.used[k]) : sl1;
    }
    const int sx = split ? sl1 : o2.slot();
#pragma unroll
    for (int k = 0; k < (NQ + 7) / 8; ++k) {
      const uint32_t bit = (sx >> 5) == k ? 1u << (sx & 31) : 0u;
      H.used[k] = split ? H.used[k] | bit : H.used[k] & ~bit;
    }
    const int N[4] = {e > 0 ? o0.N() : 1, E.n0, split ? E.n1 : (e + 2 < Z ? o3.N() : 1),
                      split && e + 1 < Z ? o2.N() : 1};
    const float q[4] = {o0.q2, q0, split ? q1 : o3.q2, split ? o2.q2 : 0.0f};
    const float w[3] = {o0.w, E.w0, E.w1};
    const int dir = E.dir;
    float Rn[3];
    lane_pairs3(C, H, e - 1, H.Z, N, q, w, Rn);
    // the rates behind the event move by one position in the lane's own column: position
    // p > e+1 takes the old p-1 (split), position p > e the old p+1 (merge; a zero follows
    // the last rate)
    const bool open = dir > 0;
    const int first = open ? e + 2 : e + 1;
    {
      int j = first >> 2;
      const int jl = (max(zold, H.Z) - 1) >> 2;
      if (j <= jl) {
        vf4 v = C.rq[j * C.S + C.lane];
        float pv;
        {
          const int d = first & 3;
          const float nx = j + 1 < NQ ? *C.rp(4 * j + 4, C.lane) : 0.0f;
          const float px = *C.rp(max(4 * j - 1, 0), C.lane);
          const vf4 n = {d == 0 ? (open ? px : v.y) : v.x, d <= 1 ? (open ? v.x : v.z) : v.y,
                         d <= 2 ? (open ? v.y : v.w) : v.z, open ? v.z : nx};
          C.rq[j * C.S + C.lane] = n;
          pv = v.w;
        }
        for (++j; j <= jl; ++j) {
          v = C.rq[j * C.S + C.lane];
          const float nx = !open && j + 1 < NQ ? *C.rp(4 * j + 4, C.lane) : 0.0f;
          const vf4 n = {open ? pv : v.y, open ? v.x : v.z, open ? v.y : v.w, open ? v.z : nx};
          C.rq[j * C.S + C.lane] = n;
          pv = v.w;
        }
      }
    }
    if (e > 0) *C.rp(e - 1, C.lane) = Rn[0];
    *C.rp(e, C.lane) = Rn[1];
    if (open) *C.rp(e + 1, C.lane) = Rn[2];
    *C.rp(H.Z - 1, C.lane) = lane_ends(H).total();
    lane_leaves<NQ>(C, lf);
  }
  // the records likewise, eight chains at a time: eight lanes a chain, eight positions a
  // lane
  constexpr int NB = (NQ + 15) / 16;
  for (uint64_t mm = m; mm;) {
    RowShift row;
    row.take(C, mm, E.e, E.dir, zold, H.base);
#pragma unroll 1
    for (int i = 0; i < NB; ++i) {
      row.load(C, i, NB);
      row.store();
    }
  }
  wave_lds_sync();
  if (on) {  // the lane's new strands
    const int64_t o = H.base + E.e, v = H.base + sl0;
    C.rec[o] = LaneRec{q0, E.w0, E.n0 | sl0 << 16};
    a.ch.Qx[v] = E.x0; a.ch.Qy[v] = E.y0; a.ch.Qz[v] = E.z0;
    if (E.dir > 0) {
      const int64_t v1 = H.base + sl1;
      C.rec[o + 1] = LaneRec{q1, E.w1, E.n1 | sl1 << 16};
      a.ch.Qx[v1] = E.x1; a.ch.Qy[v1] = E.y1; a.ch.Qz[v1] = E.z1;
    }
  }
}

// LDS floats of a workgroup, S columns of NQ quads a wave
__host__ __device__ constexpr int lane_lds_floats(int NQ, int S) { return kLaneTabFloats + kLaneWaves * 4 * NQ * S; }

// ------------------------------------------------------------------ the kernel
// Each wave keeps up to a.lanes of its lanes busy with chains from the work list until
// it is exhausted; a chain leaves its lane at its targets, at a stall, or when it could
// outgrow NQ quads (then it is handed on).
template <int NQ>
__global__ void __launch_bounds__(64 * kLaneWaves) __attribute__((amdgpu_waves_per_eu(2))) kmc_lane_kernel(KmcArgs a0) {
  extern __shared__ float lds_dyn[];
  constexpr int CAP = 4 * NQ;
  LaneCtx C;
  const int lanes = a0.lanes;
  C.S = lanes | 1;
  C.tab = (lds_f*)lds_dyn;
  C.rq = (lds_f4*)(C.tab + kLaneTabFloats) + (threadIdx.x >> 6) * NQ * C.S;
  C.rec = (LaneRec*)a0.rec;
  C.lane = lane_id();
  C.row = C.lane >> 4;
  C.rl = C.lane & 15;
  for (int i = threadIdx.x; i < kLaneTabFloats; i += 64 * kLaneWaves) C.tab[i] = a0.lane_tab[i];
  __syncthreads();  // the only meeting of the workgroup's waves
  const int n_work = *a0.n_work;
  // The first chains go by place, the others by the queue: the list is in decreasing
  // order of work, so the workgroup's waves take far-apart parts of it, and waves w and
  // w + 4, which share a SIMD, opposite ones (parts w and 7 - w).
  const int n_first = kLaneWaves * gridDim.x * lanes;
  const int wv = threadIdx.x >> 6, part = wv < kLaneWaves / 2 ? wv : kLaneWaves + kLaneWaves / 2 - 1 - wv;
  int first_ent = C.lane < lanes ? (part * (int)gridDim.x + (int)blockIdx.x) * lanes + C.lane : -1;
  const double kNever = __longlong_as_double(0x7ff0000000000000ll);
  float lf[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) lf[j] = 0.0f;
  LaneChain H;
  H.c = C.lane < lanes ? -1 : -2;
  H.ens = 0; H.Z = 1; H.left = 0; H.stall = 0; H.cid = 0; H.key0 = 0; H.key1 = 0;
  H.base = 0; H.t = 0.0; H.t_next = 0.0; H.t_end = 0.0; H.next_sample = 0; H.ev = 0; H.zsum = 0;
  H.dt_prev = 0.f; H.beta = 1.f; H.cc = 0.f; H.cd = 0; H.exp_wait = 0; H.msd = 0; H.pd = -1; H.eh = 0.f; H.et = 0.f;
  for (auto& u : H.used) u = 0;
  H.N0 = 1; H.N1 = 1; H.Nz = 1; H.Nz2 = 1;
  H.rnd = make_uint4(0, 0, 0, 0);
  H.kind = kEvNone; H.p = 0; H.r = 0.f; H.rz = 0; H.rw = 0;
  for (;;) {
    const bool run = H.c >= 0;
    const bool rare = run && H.kind != kEvNone;
    const bool samp = run && !rare && H.t > H.t_next;
    const bool more = run && !rare && !samp && H.stall == 0 && H.t < H.t_end && H.left > 0;
    const bool outgrown = more && H.Z >= CAP;
    const bool ready = more && !outgrown;
    const bool fin = run && !rare && !samp && !ready;
    const uint64_t mj = __ballot(ready), mr = __ballot(rare), ms = __ballot(samp), mf = __ballot(fin);
    const uint64_t me = __ballot(H.c == -1);
    const int nrun = __popcll(mj | mr | ms);
    if (mr && (__popcll(mr) * 3 >= nrun || !mj)) {
      const KmcArgs a = fresh_args();
      lane_rare<NQ>(C, a, H, lf, mr);
      wave_lds_sync();
      continue;
    }
    if (ms && (__popcll(ms) >= min(nrun / 4, 8) || !mj)) {
      const KmcArgs a = fresh_args();
      const uint64_t mc = __ballot(samp && H.msd);
      if (ms & ~mc) lane_sample<NQ>(C, a, H, ms & ~mc);
      if (mc) lane_sample_com<NQ>(C, a, H, mc);
      if (samp) {
        ++H.next_sample;
        const EnsParams* P = a.ens + H.ens;
        H.t_next = H.next_sample < P->k_end ? (double)H.next_sample * P->delta : kNever;
      }
      continue;
    }
    const int nfree = __popcll(mf | me);
    if (nfree && (nfree >= max(1, lanes / 8) || !mj)) {
      const KmcArgs a = fresh_args();
      if (mf) {
        lane_store<NQ>(C, a, H, mf);
        if (fin) {
          const int c = H.c;
          a.ch.Z[c] = H.Z; a.ch.stall[c] = H.stall; a.ch.next_sample[c] = H.next_sample; a.ch.t[c] = H.t;
          a.ch.ev[c] = H.ev; a.ch.zsum[c] += H.zsum; a.ch.dt_prev[c] = H.dt_prev;
          if (outgrown) a.overflow[atomicAdd(a.n_overflow, 1)] = c;
          H.c = -1;
        }
      }
      // free lanes take chains until they hold a live one or the list is exhausted
      const bool need = H.c == -1;
      if (need) {
        for (;;) {
          const int ent = first_ent >= 0 ? first_ent : n_first + atomicAdd(a.queue, 1);
          first_ent = -1;
          if (ent >= n_work) { H.c = -2; break; }
          const int c = a.work[ent];
          if (c < 0) continue;
          const int z = a.ch.Z[c];
          if (a.ch.stall[c] != 0) continue;
          if (z >= CAP) { a.overflow[atomicAdd(a.n_overflow, 1)] = c; continue; }
          H.c = c;
          H.Z = z;
          break;
        }
        if (H.c >= 0) {
          lane_begin(a, H);
#pragma unroll
          for (int k = 0; k < (NQ + 7) / 8; ++k) {
            const int z = H.Z - 32 * k;
            H.used[k] = z >= 32 ? ~0u : (z > 0 ? (1u << z) - 1u : 0u);
          }
        }
      }
      const uint64_t ml = __ballot(need && H.c >= 0);
      if (ml) {
        if (need && H.c >= 0) {
#pragma unroll
          for (int j = 0; j < NQ; ++j) C.rq[j * C.S + C.lane] = vf4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        wave_lds_sync();
        lane_load<NQ>(C, a, H, ml);
        wave_lds_sync();
        if (need && H.c >= 0) lane_leaves<NQ>(C, lf);
      }
      continue;
    }
    if (!mj) break;  // nothing runs and the list is exhausted
    if (ready) lane_jump<NQ>(C, H, lf);
    wave_lds_sync();
  }
}

}  // namespace dsm
