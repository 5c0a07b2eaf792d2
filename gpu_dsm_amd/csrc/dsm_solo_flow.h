// dsm_solo_flow.h -- the solo form for passes with flow: one chain per wave, all of its
// rates at every jump.  Included by dsm_solo_inst.hip.
//
// Why.  The affine step after a jump changes every rate, so the wave form (dsm_kmc.h) under
// flow stages all strands and rates in LDS at every jump, for the sake of the cross-lane
// reads that follow.  Here a chain's strands stay in registers, four positions a lane and
// group of 256: a jump deforms them, evaluates the pairs (the next lane's first strand comes
// by a lane shift), sums the rates where they are, and reads what the picked lane holds;
// what depends on the pick runs in the wave's scalar unit.  Splits and merges shift the
// registers by one position.  Same operands in the same order as the other forms.
//
// What bounds it: alone on a SIMD, instruction latency; with more waves, about 550 VALU
// instructions a jump and group, most of them the pairs' (64 chains of Nk 30,
// 4 tau_K: 0.15 against 0.24 ms in the wave form; 100 of Nk 500, 2 tau_K: 1.14 / 1.92).
#pragma once
#include "dsm_solo.h"

namespace dsm {

// (by value: a choice between two elements would be one of their addresses)
template <typename T>
__device__ __forceinline__ T pick(bool c, T a, T b) {
  return c ? a : b;
}

// A wave's chain: position 256 g + 4 lane + k in element 4 g + k.  Behind the chain the
// vectors and CD rates are of no use, the lengths are read as 1.
template <int G>
struct SoloFlow {
  LaneCtx C;
  float x[4 * G], y[4 * G], z[4 * G], w[4 * G];
  int N[4 * G];
  __device__ __forceinline__ int pos(int i) const { return 256 * (i >> 2) + 4 * C.lane + (i & 3); }
  // the value at position p (uniform)
  template <typename T>
  __device__ __forceinline__ T get(const T (&v)[4 * G], int p) const {
    T r = v[0];
#pragma unroll
    for (int i = 1; i < 4 * G; ++i) r = pick<T>(((p >> 8) << 2 | (p & 3)) == i, v[i], r);
    return lane_read(r, (p >> 2) & 63);
  }
  // positions first .. move by one: each takes its left (open) or right neighbour's value;
  // those at e and, opened, e + 1 get a and b
  template <typename T>
  __device__ __forceinline__ void move(T (&v)[4 * G], int e, bool open, T a, T b) const {
    T o[4 * G];
#pragma unroll
    for (int i = 0; i < 4 * G; ++i) o[i] = v[i];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (open) {
        T in = lane_prev(o[4 * g + 3]);  // (position -1 is never read)
        if (g > 0) in = pick<T>(C.lane == 0, lane_read(o[4 * (g > 0 ? g - 1 : 0) + 3], 63), in);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int i = 4 * g + k, p = pos(i);
          const T left = pick<T>(k > 0, o[4 * g + (k > 0 ? k - 1 : 0)], in);
          v[i] = pick<T>(p > e + 1, left, pick<T>(p == e + 1, b, pick<T>(p == e, a, o[i])));
        }
      } else {
        T in = lane_next(o[4 * g]);
        if (g + 1 < G) in = pick<T>(C.lane == 63, lane_read(o[4 * (g + 1 < G ? g + 1 : 0)], 0), in);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int i = 4 * g + k, p = pos(i);
          const T right = pick<T>(k < 3, o[4 * g + (k < 3 ? k + 1 : 0)], in);
          v[i] = pick<T>(p > e, right, pick<T>(p == e, a, o[i]));
        }
      }
    }
  }
  static __device__ __forceinline__ float lane_prev(float v) { return dppf<kWaveShr1>(v, 0.0f); }
  static __device__ __forceinline__ int lane_prev(int v) { return dppi<kWaveShr1>(v, 0); }
  static __device__ __forceinline__ float lane_next(float v) { return dppf<kWaveShl1>(v, 0.0f); }
  static __device__ __forceinline__ int lane_next(int v) { return dppi<kWaveShl1>(v, 0); }
};

// The affine step Q <- Q + dt kappa Q (deform in dsm_kmc.h).
template <int G>
__device__ __forceinline__ void solo_deform(SoloFlow<G>& S, const float* kappa, float dt, int Z) {
  float dk[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) dk[i] = dt * kappa[i];
#pragma unroll
  for (int i = 0; i < 4 * G; ++i) {
    const float x = S.x[i], y = S.y[i], z = S.z[i];
    S.x[i] = __builtin_fmaf(dk[2], z, __builtin_fmaf(dk[1], y, __builtin_fmaf(dk[0], x, x)));
    S.y[i] = __builtin_fmaf(dk[5], z, __builtin_fmaf(dk[4], y, __builtin_fmaf(dk[3], x, y)));
    S.z[i] = __builtin_fmaf(dk[8], z, __builtin_fmaf(dk[7], y, __builtin_fmaf(dk[6], x, z)));
  }
}

// Canonical sums of one group of four positions a lane: within the quad (s), before it in
// its block (X), before the block (cb, from c0 before the group) and through the quad (P).
struct SoloSums {
  float s[4], X, cb, P;
  __device__ __forceinline__ void form(float v0, float v1, float v2, float v3, float c0) {
    s[0] = v0;
    s[1] = s[0] + v1;
    s[2] = s[1] + v2;
    s[3] = s[2] + v3;
    float H = s[3];
    H = H + dppf<kRowShr1>(H, 0.0f);
    H = H + dppf<kRowShr2>(H, 0.0f);
    H = H + dppf<kRowShr4>(H, 0.0f);
    H = H + dppf<kRowShr8>(H, 0.0f);
    X = dppf<kRowShr1>(H, 0.0f);
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
};

struct SoloChoice {
  int p, kind, N;  // position (-1: none), sub-event, length
  float r;
};
// The position of lane l's quad whose sum first exceeds pr, in the group from p0 on, and its
// sub-event; w, N, wp, wm: the group's.  In every lane: the position within its quad, the sum
// before it, and what its sub-event would be; lane l's are read.
__device__ __forceinline__ SoloChoice solo_choose(const SoloSums& T, float c0, float pr, int l, int p0, int Z,
                                                  const LaneChain& H, const float* w, const int* N, const float* wp,
                                                  const float* wm) {
  const float g0 = T.cb + (T.X + T.s[0]), g1 = T.cb + (T.X + T.s[1]), g2 = T.cb + (T.X + T.s[2]);
  const float gl = dppf<kWaveShr1>(T.P, c0);
  const bool h0 = g0 > pr, h1 = g1 > pr, h2 = g2 > pr;
  auto at = [&](auto v0, auto v1, auto v2, auto v3) { return h0 ? v0 : (h1 ? v1 : (h2 ? v2 : v3)); };
  const int i = at(0, 1, 2, 3);
  SoloChoice k;
  k.p = p0 + 4 * l + lane_read(i, l);
  const float before = at(gl, g0, g1, g2);
  float r = k.p == 0 ? pr : pr - before;
  const int n = at(N[0], N[1], N[2], N[3]);
  const int kind = lane_kind(H, k.p < Z - 1, at(w[0], w[1], w[2], w[3]), at(wp[0], wp[1], wp[2], wp[3]),
                             at(wm[0], wm[1], wm[2], wm[3]), n, r);
  k.kind = lane_read(kind, l);
  k.r = lane_read(r, l);
  k.N = lane_read(n, l);
  if (k.p >= Z) k.p = -1;  // (sums behind the chain may round above its last one)
  return k;
}

// One jump; a split or merge is left in (kind, p, r).
template <int G>
__device__ __forceinline__ void solo_flow_jump(SoloFlow<G>& S, LaneChain& H, const uint4& rnd, int Z) {
  const int lane = S.C.lane;
  const float ee = lane_ends(H).total();
  float wp[4 * G], wm[4 * G], R[4 * G];
  {
    LaneStrand t[4 * G];
    float q2[4 * G];
    int N[4 * G];
#pragma unroll
    for (int i = 0; i < 4 * G; ++i) {
      const int p = S.pos(i);
      const bool in = p < Z;
      N[i] = in ? S.N[i] : 1;
      q2[i] = in ? q2_of(S.x[i], S.y[i], S.z[i]) : 0.0f;
      t[i] = lane_strand(S.C, N[i], q2[i], p == 0 || p == Z - 1);
    }
    // the strand behind each: the lane's next, behind its last the next lane's first
    LaneStrand u[4 * G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      u[4 * g] = t[4 * g + 1];
      u[4 * g + 1] = t[4 * g + 2];
      u[4 * g + 2] = t[4 * g + 3];
      LaneStrand f;
      f.a = S.lane_next(t[4 * g].a); f.b = S.lane_next(t[4 * g].b);
      f.pp = S.lane_next(t[4 * g].pp); f.pm = S.lane_next(t[4 * g].pm);
      f.xp = S.lane_next(t[4 * g].xp); f.xm = S.lane_next(t[4 * g].xm);
      if constexpr (G > 1) {
        const int j = g + 1 < G ? 4 * g + 4 : 0;  // (behind the last group lies no strand)
        const bool l = lane == 63 && g + 1 < G;
        const float a = lane_read(t[j].a, 0), b = lane_read(t[j].b, 0), pp = lane_read(t[j].pp, 0),
                    pm = lane_read(t[j].pm, 0);
        const int xp = lane_read(t[j].xp, 0), xm = lane_read(t[j].xm, 0);
        f.a = l ? a : f.a; f.b = l ? b : f.b; f.pp = l ? pp : f.pp; f.pm = l ? pm : f.pm;
        f.xp = l ? xp : f.xp; f.xm = l ? xm : f.xm;
      }
      u[4 * g + 3] = f;
    }
    bool slow = false;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = 4 * g + k, p = S.pos(i);
        const bool far = lane_pair(S.C, t[i], u[i], wp[i], wm[i]);
        // (a long strand is beside its pair's other one, or in its own pair too)
        slow = slow || (p <= Z - 2 && far) || N[i] >= kLaneN / 2;
        R[i] = p <= Z - 2 ? lane_total(H.cd, H.cc, N[i], wp[i], wm[i], S.w[i]) : (p == Z - 1 ? ee : 0.0f);
      }
    }
    if (__ballot(slow)) {
      // some pair needs the general form: every lane looks at its own
#pragma unroll
      for (int i = 0; i < 4 * G; ++i) {
        const int p = S.pos(i), g = i >> 2;
        int Nj;
        float qj;
        if ((i & 3) < 3) {
          Nj = N[(i & 3) < 3 ? i + 1 : i];
          qj = q2[(i & 3) < 3 ? i + 1 : i];
        } else {
          Nj = S.lane_next(N[4 * g]);
          qj = S.lane_next(q2[4 * g]);
          if (g + 1 < G) {
            Nj = lane == 63 ? lane_read(N[4 * (g + 1 < G ? g + 1 : 0)], 0) : Nj;
            qj = lane == 63 ? lane_read(q2[4 * (g + 1 < G ? g + 1 : 0)], 0) : qj;
          }
        }
        if (p <= Z - 2)
          lane_pair_any(H.ens, H.cd, N[i], Nj, q2[i], qj, S.w[i], p == 0, p + 2 == Z, wp[i], wm[i], R[i]);
      }
    }
  }
  SoloSums T[G];
  float c0[G + 1];
  c0[0] = 0.0f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    T[g].form(R[4 * g], R[4 * g + 1], R[4 * g + 2], R[4 * g + 3], c0[g]);
    c0[g + 1] = lane_read(T[g].P, 63);
  }
  const float W = c0[G];
  const float pr = W * u01(rnd.x);
  if (!lane_clock(H, W, rnd)) return;
  SoloChoice k{-1, kEvNone, 0, 0.0f};
  const uint64_t m0 = __ballot(T[0].P > pr);
  if (m0) {
    k = solo_choose(T[0], c0[0], pr, (int)__builtin_ctzll(m0), 0, Z, H, S.w, S.N, wp, wm);
  } else if constexpr (G > 1) {
    const uint64_t m1 = __ballot(T[1].P > pr);
    if (m1)
      k = solo_choose(T[1], c0[1], pr, (int)__builtin_ctzll(m1), 256, Z, H, S.w + 4, S.N + 4, wp + 4, wm + 4);
  }
  const int p = k.p, kind = k.kind, Nk = k.N;
  const float r = k.r;
  if (p < 0) return;  // no position: the clock moves, the chain does not
  if (kind != kEvShiftP && kind != kEvShiftM) {
    H.kind = kind;
    H.p = p;
    H.r = r;
    H.rz = rnd.z;
    H.rw = rnd.w;
    return;
  }
  const int dn = kind == kEvShiftP ? 1 : -1;
  if (p <= 1 || p >= Z - 3) {
    lane_shift_ends(H, p, Nk + dn, S.get(S.N, p + 1) - dn);
    lane_end_rates(H);
  }
#pragma unroll
  for (int i = 0; i < 4 * G; ++i) S.N[i] += S.pos(i) == p ? dn : (S.pos(i) == p + 1 ? -dn : 0);
}

// A split or merge of strands (LaneEvent).
template <int G>
__device__ __forceinline__ void solo_flow_event(SoloFlow<G>& S, const KmcArgs& a, LaneChain& H, int Z) {
  LaneEvent E;
  E.place(H);
  const int e = __builtin_amdgcn_readfirstlane(E.e), f = min(e + 1, Z - 1);
  const bool open = __builtin_amdgcn_readfirstlane(E.dir) > 0;
  E.apply(a, H, S.get(S.N, max(e - 1, 0)), S.get(S.N, e), S.get(S.N, f), S.get(S.N, min(e + 2, Z - 1)),
          S.get(S.w, e), S.get(S.w, f), S.get(S.x, e), S.get(S.y, e), S.get(S.z, e), S.get(S.x, f), S.get(S.y, f),
          S.get(S.z, f));
  S.move(S.x, e, open, E.x0, E.x1);
  S.move(S.y, e, open, E.y0, E.y1);
  S.move(S.z, e, open, E.z0, E.z1);
  S.move(S.w, e, open, E.w0, E.w1);
  S.move(S.N, e, open, E.n0, E.n1);
}

// Canonical total over the chain of v, zero behind it, by blocks (-0 stays what a chain's
// own blocks make it).
template <int G>
__device__ __forceinline__ float solo_chain_sum(const float (&v)[4 * G], int Z) {
  float tot = 0.0f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (g > 0 && Z <= 256 * g) break;
    float I[4];
    block_scan4(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3], I);
    solo_add(tot, I[3], g, (Z + 63) >> 6);
  }
  return tot;
}

// One G(t) or flow sample (eq_sample, flow_sample in dsm_kmc.h) into the staging rows.
template <int G>
__device__ __forceinline__ void solo_flow_sample(const SoloFlow<G>& S, const KmcArgs& a, const LaneChain& H, int Z) {
  const EnsParams* E = a.ens + H.ens;
  const bool flow = E->sample_mode == kSampleFlow;
  float t3[4 * G], v[4 * G], out[7];
#pragma unroll
  for (int i = 0; i < 4 * G; ++i) t3[i] = S.pos(i) < Z ? 3.0f / (float)S.N[i] : 0.0f;
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    // the G(t) sample has components 3, 4 and 5 of the flow sample
    if (!flow && (q < 3 || q == 6)) continue;
#pragma unroll
    for (int i = 0; i < 4 * G; ++i) {
      const bool on = S.pos(i) < Z;
      const float x = S.x[i], y = S.y[i], z = S.z[i];
      const float s = q == 0 ? x * x : q == 1 ? y * y : q == 2 ? z * z : q == 3 ? x * y : q == 4 ? y * z : x * z;
      v[i] = on ? (q < 6 ? s * t3[i] : sqrtf(q2_of(x, y, z))) : 0.0f;
    }
    out[q] = solo_chain_sum<G>(v, Z);
  }
  if (S.C.lane == 0 && H.next_sample >= E->k0) {
    float* o = a.stage + E->stage_off + ((H.next_sample - E->k0) * E->nchains + a.ch.local[H.c]) * (flow ? 8 : 3);
    if (flow) {
#pragma unroll
      for (int q = 0; q < 6; ++q) o[q] = -out[q];
      o[6] = out[6];
      o[7] = (float)Z;
    } else {
      o[0] = -out[3]; o[1] = -out[4]; o[2] = -out[5];
    }
  }
}

// Persistent waves as in kmc_solo_kernel; chains of ensembles with and without flow (no MSD
// sampling), to 256 G - 1 positions.
template <int G>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(G > 1 ? 2 : 3))) kmc_solo_flow_kernel(KmcArgs a) {
  extern __shared__ float lds_dyn[];
  const int n_work = *a.n_work;
  if ((int)blockIdx.x >= n_work) return;
  SoloFlow<G> S;
  S.C.tab = (lds_f*)lds_dyn;
  S.C.lane = lane_id();
  S.C.row = S.C.lane >> 4;
  S.C.rl = S.C.lane & 15;
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
    if (z >= 256 * G) {
      if (S.C.lane == 0) a.overflow[atomicAdd(a.n_overflow, 1)] = c;
      continue;
    }
    H.c = c;
    H.Z = z;
    lane_begin(a, H);
    const EnsParams* E = a.ens + H.ens;
    const bool flow = E->flow != 0, flow_rows = E->sample_mode == kSampleFlow;
    float kappa[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) kappa[i] = E->kappa[i];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int p0 = 256 * g + 4 * S.C.lane;
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f), y = x, zz = x, w = x;
      int4 n = make_int4(1, 1, 1, 1);
      if (p0 < z) {
        const int64_t o = H.base + p0;
        x = *(const float4*)(a.ch.Qx + o); y = *(const float4*)(a.ch.Qy + o); zz = *(const float4*)(a.ch.Qz + o);
        w = *(const float4*)(a.ch.w + o); n = *(const int4*)(a.ch.N + o);
      }
      S.x[4 * g] = x.x; S.x[4 * g + 1] = x.y; S.x[4 * g + 2] = x.z; S.x[4 * g + 3] = x.w;
      S.y[4 * g] = y.x; S.y[4 * g + 1] = y.y; S.y[4 * g + 2] = y.z; S.y[4 * g + 3] = y.w;
      S.z[4 * g] = zz.x; S.z[4 * g + 1] = zz.y; S.z[4 * g + 2] = zz.z; S.z[4 * g + 3] = zz.w;
      S.w[4 * g] = w.x; S.w[4 * g + 1] = w.y; S.w[4 * g + 2] = w.z; S.w[4 * g + 3] = w.w;
      S.N[4 * g] = n.x; S.N[4 * g + 1] = n.y; S.N[4 * g + 2] = n.z; S.N[4 * g + 3] = n.w;
    }
    uint64_t ev0 = H.ev;  // lane k: random words of jump ev0 + k
    uint4 rnd = lane_step_words(H, ev0 + S.C.lane);
    bool outgrown = false;
    for (;;) {
      int Zc = __builtin_amdgcn_readfirstlane(H.Z);
      if (flow) {
        if (__builtin_amdgcn_readfirstlane(H.dt_prev != 0.0f)) solo_deform(S, kappa, H.dt_prev, Zc);
        H.dt_prev = 0.0f;
      }
      while (__builtin_amdgcn_readfirstlane(flow_rows ? H.t >= H.t_next : H.t > H.t_next)) {
        solo_flow_sample(S, a, H, Zc);
        ++H.next_sample;
        const EnsParams* P = a.ens + H.ens;
        H.t_next = H.next_sample < P->k_end ? (double)H.next_sample * P->delta : kNever;
      }
      if (!__builtin_amdgcn_readfirstlane(H.stall == 0 && H.t < H.t_end && H.left > 0)) break;
      if (Zc >= 256 * G) { outgrown = true; break; }
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
      solo_flow_jump(S, H, r, Zc);
      if (__builtin_amdgcn_readfirstlane(H.kind) != kEvNone) solo_flow_event(S, a, H, Zc);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int p0 = 256 * g + 4 * S.C.lane;
      if (p0 < H.Z) {
        const int64_t o = H.base + p0;
        *(float4*)(a.ch.Qx + o) = make_float4(S.x[4 * g], S.x[4 * g + 1], S.x[4 * g + 2], S.x[4 * g + 3]);
        *(float4*)(a.ch.Qy + o) = make_float4(S.y[4 * g], S.y[4 * g + 1], S.y[4 * g + 2], S.y[4 * g + 3]);
        *(float4*)(a.ch.Qz + o) = make_float4(S.z[4 * g], S.z[4 * g + 1], S.z[4 * g + 2], S.z[4 * g + 3]);
        *(float4*)(a.ch.w + o) = make_float4(S.w[4 * g], S.w[4 * g + 1], S.w[4 * g + 2], S.w[4 * g + 3]);
        *(int4*)(a.ch.N + o) = make_int4(S.N[4 * g], S.N[4 * g + 1], S.N[4 * g + 2], S.N[4 * g + 3]);
      }
    }
    if (S.C.lane == 0) {
      a.ch.Z[c] = H.Z; a.ch.stall[c] = H.stall; a.ch.next_sample[c] = H.next_sample; a.ch.t[c] = H.t;
      a.ch.ev[c] = H.ev; a.ch.zsum[c] += H.zsum; a.ch.dt_prev[c] = H.dt_prev;
      if (outgrown) a.overflow[atomicAdd(a.n_overflow, 1)] = c;
    }
  }
}

}  // namespace dsm
