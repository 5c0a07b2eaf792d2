// dsm_lane_flow.h -- the lane form (dsm_lane.h) under flow: one chain per lane.  Included by
// dsm_lane_flow_inst.hip.
//
// Why.  The affine step after every jump changes all of a chain's rates, so a jump deforms
// every strand and evaluates every pair.  The row form does that with 16 lanes a chain, four
// positions a lane: a chain of 25 strands uses seven of them, and picking and applying the
// event costs the four chains of a wave what it would cost 64.  Here a lane walks its own
// chain, strand by strand: deformed, its part of the two pairs it belongs to, the pair to
// its left, a quad's sum; no position is idle but those beyond the shorter chains of the
// wave.  A chain's strands {Q, w} and lengths lie in LDS, a column a lane (18 bytes a
// position); the picked quad's rates are evaluated a second time rather than kept.  Splits
// and merges move the column behind them; nothing but loading, writing back and samples'
// rows touches memory.  Same operands in the same order as the other forms.
//
// What bounds it: VALU issue, about 60 instructions a position and jump, on the 27 to 64
// lanes of a wave that LDS has room for (flow_max_lanes: 64 up to 16 positions, 33 at 32, 31
// at 36, 27 at 40), or fewer where the chains come in rounds of that many (262,144 at 36
// positions: five rounds of 26).  262,144 chains of 16 sheared ensembles, 8 tau_K: Nk 50 9.6
// against 11.8 ms in the row form, Nk 25 3.4 / 7.9, Nk 12 1.5 / 5.5.  A version with the strand
// vectors in registers (64 lanes at 44 positions) spilled hundreds of them; whether it would
// have with its elements selected by value only (dsm_solo_flow.h) was not tried.
#pragma once
#include "dsm_lane.h"

namespace dsm {

typedef __attribute__((address_space(3))) uint16_t lds_h;

struct FlowChain : LaneChain {
  float kappa[9];
};

// A wave's columns: strand p of lane l at q[p * S + l], its length at n[p * S + l].
template <int P>
struct FlowCols {
  LaneCtx C;
  lds_f4* q;
  lds_h* n;
  __device__ __forceinline__ int at(int p) const { return min(p, P - 1) * C.S + C.lane; }
};

// One strand: what its pairs need.  Outside the chain: length 1, zero.
struct FlowStrand {
  LaneStrand t;
  int N;
  float q2, w;
};
// Strand p of the lane's chain, after the affine step Q <- Q + dt kappa Q (deform in
// dsm_kmc.h) when `step` (dk = dt kappa).
template <int P, bool DEFORM>
__device__ __forceinline__ FlowStrand flow_strand(const FlowCols<P>& F, int p, int Z, bool step, const float (&dk)[9]) {
  const int i = F.at(p);
  vf4 v = F.q[i];
  const int n = F.n[i];
  const bool in = p < Z;
  FlowStrand s;
  s.N = in ? n : 1;
  if constexpr (DEFORM) {
    const float x = v.x, y = v.y, z = v.z;
    const float dx = __builtin_fmaf(dk[2], z, __builtin_fmaf(dk[1], y, __builtin_fmaf(dk[0], x, x)));
    const float dy = __builtin_fmaf(dk[5], z, __builtin_fmaf(dk[4], y, __builtin_fmaf(dk[3], x, y)));
    const float dz = __builtin_fmaf(dk[8], z, __builtin_fmaf(dk[7], y, __builtin_fmaf(dk[6], x, z)));
    v.x = step ? dx : x;
    v.y = step ? dy : y;
    v.z = step ? dz : z;
    F.q[i] = v;  // (the last row, which stands for all behind it, holds no strand: Z < P)
  }
  s.q2 = in ? q2_of(v.x, v.y, v.z) : 0.0f;
  s.w = v.w;
  s.t = lane_strand(F.C, s.N, s.q2, p == 0 || p == Z - 1);
  return s;
}

// Rates of quad j: of the pairs to the right of positions 4j .. 4j+3, the chain-end rates'
// sum ee at Z-1, zero behind it; s: strand 4j, then strand 4j+4.
template <int P, bool DEFORM>
__device__ __forceinline__ void flow_quad(const FlowCols<P>& F, const FlowChain& H, int j, int Z, float ee, bool step,
                                          const float (&dk)[9], FlowStrand& s, float (&R)[4], float (&wp)[4],
                                          float (&wm)[4], float (&w)[4], int (&N)[4]) {
  const int p0 = 4 * j;
  FlowStrand u[5];
  u[0] = s;
#pragma unroll
  for (int k = 1; k < 5; ++k) u[k] = flow_strand<P, DEFORM>(F, p0 + k, Z, step, dk);
  bool slow = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int p = p0 + k;
    const bool far = lane_pair(F.C, u[k].t, u[k + 1].t, wp[k], wm[k]) || u[k].N + u[k + 1].N >= kLaneN;
    slow = slow || (far && p <= Z - 2);
    R[k] = p <= Z - 2 ? lane_total(H.cd, H.cc, u[k].N, wp[k], wm[k], u[k].w) : (p == Z - 1 ? ee : 0.0f);
    w[k] = u[k].w;
    N[k] = u[k].N;
  }
  if (slow) {
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
      // (one copy of the general form: the values by selection)
      FlowStrand a = u[0], b = u[1];
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        a.N = i == k ? u[i].N : a.N; a.q2 = i == k ? u[i].q2 : a.q2; a.w = i == k ? u[i].w : a.w;
        b.N = i == k ? u[i + 1].N : b.N; b.q2 = i == k ? u[i + 1].q2 : b.q2;
      }
      if (p0 + k <= Z - 2) {
        float vp, vm, r;
        lane_pair_any(H.ens, H.cd, a.N, b.N, a.q2, b.q2, a.w, p0 + k == 0, p0 + k + 2 == Z, vp, vm, r);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          wp[i] = i == k ? vp : wp[i];
          wm[i] = i == k ? vm : wm[i];
          R[i] = i == k ? r : R[i];
        }
      }
    }
  }
  s = u[4];
}

// The affine step alone, of a chain that will not jump now (a sample, or its end).
template <int P>
__device__ __forceinline__ void flow_deform(const FlowCols<P>& F, FlowChain& H) {
  float dk[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) dk[i] = H.dt_prev * H.kappa[i];
  for (int p = 0; p < H.Z; ++p) (void)flow_strand<P, true>(F, p, H.Z, true, dk);
  H.dt_prev = 0.0f;
}

// One jump of every ready lane: the affine step of the last one, all rates, the event; a
// split or merge is left in (kind, p, r) for flow_rare.
template <int P>
__device__ __forceinline__ void flow_jump(const FlowCols<P>& F, FlowChain& H) {
  constexpr int NQ = P / 4;
  const uint4 rnd = lane_step_words(H, H.ev);
  const int Z = H.Z;
  const bool step = H.dt_prev != 0.0f;
  float dk[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) dk[i] = H.dt_prev * H.kappa[i];
  H.dt_prev = 0.0f;
  const float ee = lane_ends(H).total();
  float R[4], wp[4], wm[4], w[4], lf[NQ];
  int N[4];
  {
    FlowStrand s = flow_strand<P, true>(F, 0, Z, step, dk);
#pragma unroll
    for (int j = 0; j < NQ; ++j) lf[j] = 0.0f;
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      if (!__ballot(4 * j < Z)) break;
      flow_quad<P, true>(F, H, j, Z, ee, step, dk, s, R, wp, wm, w, N);
      lf[j] = ((R[0] + R[1]) + R[2]) + R[3];
    }
  }
  LanePick<NQ> K;
  const float W = K.total(lf, Z);
  if (!lane_clock(H, W, rnd)) return;
  const float pr = W * u01(rnd.x);
  const int qp = K.quad(pr);
  if (qp > (Z - 1) >> 2) return;  // no position: the clock moves, the chain does not
  FlowStrand s = flow_strand<P, false>(F, 4 * qp, Z, false, dk);
  flow_quad<P, false>(F, H, qp, Z, ee, false, dk, s, R, wp, wm, w, N);
  float before;
  const int k = K.slot(R, pr, before);
  const int p = 4 * qp + k;
  float r = p == 0 ? pr : pr - before;
  const float wk = k == 0 ? w[0] : (k == 1 ? w[1] : (k == 2 ? w[2] : w[3]));
  const float wpk = k == 0 ? wp[0] : (k == 1 ? wp[1] : (k == 2 ? wp[2] : wp[3]));
  const float wmk = k == 0 ? wm[0] : (k == 1 ? wm[1] : (k == 2 ? wm[2] : wm[3]));
  const int Nk = k == 0 ? N[0] : (k == 1 ? N[1] : (k == 2 ? N[2] : N[3]));
  const int kind = lane_kind(H, p < Z - 1, wk, wpk, wmk, Nk, r);
  if (kind != kEvShiftP && kind != kEvShiftM) {
    H.kind = kind;
    H.p = p;
    H.r = r;
    H.rz = rnd.z;
    H.rw = rnd.w;
    return;
  }
  const int dn = kind == kEvShiftP ? 1 : -1;
  const int a = F.at(p), b = F.at(p + 1);
  const int M = F.n[b];
  F.n[a] = (uint16_t)(Nk + dn);
  F.n[b] = (uint16_t)(M - dn);
  if (lane_shift_ends(H, p, Nk + dn, M - dn)) lane_end_rates(H);
}

// Applies the waiting split or merge of a lane (LaneEvent) and moves the strands behind it
// by one.
template <int P>
__device__ __forceinline__ void flow_rare(const FlowCols<P>& F, const KmcArgs& a, FlowChain& H) {
  const int Z = H.Z;
  LaneEvent E;
  E.place(H);
  const int e = E.e;
  const int i0 = F.at(max(e - 1, 0)), i1 = F.at(e), i2 = F.at(min(e + 1, Z - 1)), i3 = F.at(min(e + 2, Z - 1));
  const vf4 v = F.q[i1], u = F.q[i2];
  E.apply(a, H, F.n[i0], F.n[i1], F.n[i2], F.n[i3], v.w, u.w, v.x, v.y, v.z, u.x, u.y, u.z);
  // four strands at a time, from the end that moves away
  const bool open = E.dir > 0;
  const int last = open ? e + 2 : Z - 2, dir = open ? -1 : 1;  // (Z < P)
  for (int p = open ? Z : e + 1; dir * p <= dir * last; p += 4 * dir) {
    vf4 x[4];
    uint16_t n[4];
    int i[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      i[k] = max(p + k * dir, 0);
      const int j = F.at(max(p + (k + 1) * dir, 0));
      x[k] = F.q[j];
      n[k] = F.n[j];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (dir * (p + k * dir) <= dir * last) {
        F.q[F.at(i[k])] = x[k];
        F.n[F.at(i[k])] = n[k];
      }
    }
  }
  if (open) {
    const int o = F.at(e + 1);
    F.q[o] = vf4{E.x1, E.y1, E.z1, E.w1};
    F.n[o] = (uint16_t)E.n1;
  }
  F.q[i1] = vf4{E.x0, E.y0, E.z0, E.w0};
  F.n[i1] = (uint16_t)E.n0;
}

// One flow sample (flow_sample in dsm_kmc.h) of the chains of lanes `m` into the staging
// rows, four chains at a time, a row of lanes each.
template <int P>
__device__ __forceinline__ void flow_lane_sample(const FlowCols<P>& F, const KmcArgs& a, const FlowChain& H, uint64_t m) {
  const LaneCtx& C = F.C;
  while (m) {
    const int src0 = row_take(m, C.row);
    const bool act = src0 >= 0;
    const int src = act ? src0 : C.lane;
    const int Z = from_lane(H.Z, src), ens = from_lane(H.ens, src), c = from_lane(H.c, src);
    const int64_t ns = from_lane(H.next_sample, src);
    float tot[7];
#pragma unroll
    for (int q = 0; q < 7; ++q) tot[q] = 0.0f;
    for (int b = 0; 64 * b < P; ++b) {
      const bool row_on = act && 64 * b < Z;
      if (!__ballot(row_on)) break;
      const int p0 = 64 * b + 4 * C.rl;
      float v[7][4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool on = row_on && p0 + k < Z;
        const int i = (on ? p0 + k : 0) * C.S + src;
        const vf4 x = F.q[i];
        const float t3 = on ? 3.0f / (float)F.n[i] : 0.0f;
        v[0][k] = on ? (x.x * x.x) * t3 : 0.0f;
        v[1][k] = on ? (x.y * x.y) * t3 : 0.0f;
        v[2][k] = on ? (x.z * x.z) * t3 : 0.0f;
        v[3][k] = on ? (x.x * x.y) * t3 : 0.0f;
        v[4][k] = on ? (x.y * x.z) * t3 : 0.0f;
        v[5][k] = on ? (x.x * x.z) * t3 : 0.0f;
        v[6][k] = on ? sqrtf(q2_of(x.x, x.y, x.z)) : 0.0f;
      }
#pragma unroll
      for (int q = 0; q < 7; ++q) {
        float I[4];
        block_scan4(v[q][0], v[q][1], v[q][2], v[q][3], I);
        const float B = row_last(I[3]);
        if (row_on) tot[q] = b == 0 ? B : tot[q] + B;
      }
    }
    if (act && C.rl == 0) {
      const EnsParams* P0 = a.ens + ens;
      if (ns >= P0->k0) {
        float* o = a.stage + P0->stage_off + ((ns - P0->k0) * P0->nchains + a.ch.local[c]) * 8;
#pragma unroll
        for (int q = 0; q < 6; ++q) o[q] = -tot[q];
        o[6] = tot[6];
        o[7] = (float)Z;
      }
    }
  }
}

// The chains of lanes `m` between the chain arrays and their columns.
template <int P, bool LOAD>
__device__ __forceinline__ void flow_move(const FlowCols<P>& F, const KmcArgs& a, const FlowChain& H, uint64_t m) {
  const LaneCtx& C = F.C;
  while (m) {
    const int src0 = row_take(m, C.row);
    const bool act = src0 >= 0;
    const int src = act ? src0 : C.lane;
    const int Z0 = from_lane(H.Z, src), Z = act ? Z0 : 0;
    const int64_t base = from_lane(H.base, src);
    for (int p0 = 4 * C.rl; p0 < Z; p0 += 64) {  // (p0 + 3 < P: both are multiples of four)
      const int64_t o = base + p0;
      const int i = p0 * C.S + src, S = C.S;
      if constexpr (LOAD) {
        const float4 x = *(const float4*)(a.ch.Qx + o), y = *(const float4*)(a.ch.Qy + o),
                     z = *(const float4*)(a.ch.Qz + o), w = *(const float4*)(a.ch.w + o);
        const int4 n = *(const int4*)(a.ch.N + o);
        F.q[i] = vf4{x.x, y.x, z.x, w.x};
        F.q[i + S] = vf4{x.y, y.y, z.y, w.y};
        F.q[i + 2 * S] = vf4{x.z, y.z, z.z, w.z};
        F.q[i + 3 * S] = vf4{x.w, y.w, z.w, w.w};
        F.n[i] = (uint16_t)n.x;
        F.n[i + S] = (uint16_t)n.y;
        F.n[i + 2 * S] = (uint16_t)n.z;
        F.n[i + 3 * S] = (uint16_t)n.w;
      } else {
        const vf4 v0 = F.q[i], v1 = F.q[i + S], v2 = F.q[i + 2 * S], v3 = F.q[i + 3 * S];
        *(float4*)(a.ch.Qx + o) = make_float4(v0.x, v1.x, v2.x, v3.x);
        *(float4*)(a.ch.Qy + o) = make_float4(v0.y, v1.y, v2.y, v3.y);
        *(float4*)(a.ch.Qz + o) = make_float4(v0.z, v1.z, v2.z, v3.z);
        *(float4*)(a.ch.w + o) = make_float4(v0.w, v1.w, v2.w, v3.w);
        *(int4*)(a.ch.N + o) = make_int4(F.n[i], F.n[i + S], F.n[i + 2 * S], F.n[i + 3 * S]);
      }
    }
  }
}

// One workgroup of eight waves a CU: LDS bounds the chains in flight; two waves a SIMD issue
// while the other waits (four waves of twice the lanes: 14.0 against 12.9 ms at 44 positions).
template <int P>
__global__ void __launch_bounds__(64 * kFlowWaves) __attribute__((amdgpu_waves_per_eu(2))) kmc_lane_flow_kernel(KmcArgs a0) {
  extern __shared__ float lds_dyn[];
  FlowCols<P> F;
  LaneCtx& C = F.C;
  const int lanes = a0.lanes, wv = threadIdx.x >> 6;
  C.S = lanes | 1;
  C.tab = (lds_f*)lds_dyn;
  C.rq = nullptr;
  C.rec = nullptr;
  F.q = (lds_f4*)(C.tab + kLaneTabFloats + wv * flow_wave_floats(P, C.S));
  F.n = (lds_h*)(F.q + P * C.S);
  C.lane = lane_id();
  C.row = C.lane >> 4;
  C.rl = C.lane & 15;
  for (int i = threadIdx.x; i < kLaneTabFloats; i += 64 * kFlowWaves) C.tab[i] = a0.lane_tab[i];
  __syncthreads();  // the only meeting of the workgroup's waves
  const int n_work = *a0.n_work;
  // the first chains by place, the others by the queue (kmc_lane_kernel)
  const int n_first = kFlowWaves * gridDim.x * lanes;
  int first_ent = C.lane < lanes ? (wv * (int)gridDim.x + (int)blockIdx.x) * lanes + C.lane : -1;
  const double kNever = __longlong_as_double(0x7ff0000000000000ll);
  FlowChain H;
  H.c = C.lane < lanes ? -1 : -2;
  H.ens = 0; H.Z = 1; H.left = 0; H.stall = 0; H.cid = 0; H.key0 = 0; H.key1 = 0;
  H.base = 0; H.t = 0.0; H.t_next = 0.0; H.t_end = 0.0; H.next_sample = 0; H.ev = 0; H.zsum = 0;
  H.dt_prev = 0.f; H.beta = 1.f; H.cc = 0.f; H.cd = 0; H.exp_wait = 0; H.msd = 0; H.pd = -1; H.eh = 0.f; H.et = 0.f;
  H.N0 = 1; H.N1 = 1; H.Nz = 1; H.Nz2 = 1;
  H.kind = kEvNone; H.p = 0; H.r = 0.f; H.rz = 0; H.rw = 0;
#pragma unroll
  for (int i = 0; i < 9; ++i) H.kappa[i] = 0.f;
  for (;;) {
    // a chain's turn after a jump: its split or merge, the affine step, samples, then the
    // next jump or the end
    const bool run = H.c >= 0;
    const bool rare = run && H.kind != kEvNone;
    const bool samp = run && !rare && H.t >= H.t_next;
    const bool more = run && !rare && !samp && H.stall == 0 && H.t < H.t_end && H.left > 0;
    const bool outgrown = more && H.Z >= P;
    const bool ready = more && !outgrown;
    const bool fin = run && !rare && !samp && !ready;
    const uint64_t mj = __ballot(ready), mr = __ballot(rare), ms = __ballot(samp), mf = __ballot(fin);
    const uint64_t me = __ballot(H.c == -1);
    const int nrun = __popcll(mj | mr | ms);
    if (mr && (__popcll(mr) * 4 >= nrun || !mj)) {
      const KmcArgs a = fresh_args();
      if (rare) flow_rare(F, a, H);
      wave_lds_sync();
      continue;
    }
    if (ms && (__popcll(ms) >= min(nrun / 4, 8) || !mj)) {
      const KmcArgs a = fresh_args();
      if (samp && H.dt_prev != 0.0f) flow_deform(F, H);
      wave_lds_sync();
      flow_lane_sample(F, a, H, ms);
      if (samp) {
        ++H.next_sample;
        const EnsParams* E = a.ens + H.ens;
        H.t_next = H.next_sample < E->k_end ? (double)H.next_sample * E->delta : kNever;
      }
      continue;
    }
    const int nfree = __popcll(mf | me);
    if (nfree && (nfree >= max(1, lanes / 8) || !mj)) {
      const KmcArgs a = fresh_args();
      if (mf) {
        if (fin && H.dt_prev != 0.0f) flow_deform(F, H);
        wave_lds_sync();
        flow_move<P, false>(F, a, H, mf);
        if (fin) {
          const int c = H.c;
          a.ch.Z[c] = H.Z; a.ch.stall[c] = H.stall; a.ch.next_sample[c] = H.next_sample; a.ch.t[c] = H.t;
          a.ch.ev[c] = H.ev; a.ch.zsum[c] += H.zsum; a.ch.dt_prev[c] = H.dt_prev;
          if (outgrown) a.overflow[atomicAdd(a.n_overflow, 1)] = c;
          H.c = -1;
        }
      }
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
          if (z >= P) { a.overflow[atomicAdd(a.n_overflow, 1)] = c; continue; }
          H.c = c;
          H.Z = z;
          break;
        }
        if (H.c >= 0) {
          lane_begin(a, H);
          const EnsParams* E = a.ens + H.ens;
#pragma unroll
          for (int i = 0; i < 9; ++i) H.kappa[i] = E->kappa[i];
        }
      }
      const uint64_t ml = __ballot(need && H.c >= 0);
      wave_lds_sync();
      if (ml) flow_move<P, true>(F, a, H, ml);
      wave_lds_sync();
      continue;
    }
    if (!mj) break;  // nothing runs and the list is exhausted
    if (ready) flow_jump(F, H);
    wave_lds_sync();
  }
}

}  // namespace dsm
