// dsm_kernels.hip -- MI355X (gfx950) kernels for the Discrete Slip-Link Model ensemble KMC path.
//
// One wave64 owns one chain.  Strand i sits in lane i%64 of register slot i/64
// (S slots per lane, S a template parameter, so a chain of up to 64*S strands
// lives in VGPRs).  A KMC jump (ktaletsk/gpu_dsm common/eq_ensemble_kernel.cu:242-663,
// common/ensemble_kernel.cu:188-502) is:
//   1. per-pair rates (sliding + constraint dynamics) cached per lane; the five
//      chain-end rates summed into the last position,
//   2. a wave64 inclusive scan (DPP tree) -> total W, dt = 1/W, FP64 clock += dt,
//   3. pr = W*u from Philox(seed, chain, event); the pair is the first lane
//      whose inclusive sum exceeds pr (ballot + ffs); the sub-event follows the
//      reference order CDd, SD+, SD-, CDc (pairs) / CDc tail, SDc head/tail,
//      SDd head/tail (ends),
//   4. the effect: N updates for shifts; split/merge as in-wave shifts of all
//      strand records; only the pair rates next to the change are recomputed.
// Two forms share this code:
//   * plain:   one jump per chain per launch, state read from and written to HBM
//              (the reference's one-step-per-launch structure);
//   * batched: persistent waves pull chains from a work queue, keep the chain in
//              registers for many jumps (until its clock passes the window end),
//              then write it back once.
#include "dsm_kmc.h"
#include "dsm_launch.h"

namespace dsm {

// ------------------------------------------------------------------ equilibrium init
// G lanes (a 16-lane row, or four) per chain of first .. first+n-1.  Inner Kuhn-step boundary i (1 <= i < nk)
// carries an entanglement iff Philox word (i-1) < 2^32/(1+beta): Z-1 ~ Binomial(nk-1,
// 1/(1+beta)) and N|Z uniform over compositions (the laws of common/chain.cu:38-88).
// Internal strands get Q ~ N(0, N/3) per component (common/chain.cu:90-102), links get CD
// rates from f_t (common/chain.cu:155-158), with the partner length of each link drawn from
// the background distribution when there is one (:141-149).  A lane has the four words of
// one Philox call in each part; a cut's strand index is the count of cuts before it, and
// the cut positions are kept in the strand-length array until the lengths are their
// differences.  One thread a chain, all of it in turn, a row and a quad of lanes, 262,144 chains,
// us: Nk 100 1039, 225, 324; Nk 30 362, 108, 100; Nk 12 106, 90, 49; Nk 6 55, 85, 42; Nk 4 31, 76, 34;
// 20,000 of Nk 20 43, 22, 24.
// inclusive sums over the G lanes of a chain, and their last lane's value
template <int G>
__device__ __forceinline__ int lanes_scan(int v, int gl) {
  if constexpr (G == 16) {
    v += dppi<kRowShr1>(v, 0);
    v += dppi<kRowShr2>(v, 0);
    v += dppi<kRowShr4>(v, 0);
    v += dppi<kRowShr8>(v, 0);
  } else {
    const int a = dppi<kRowShr1>(v, 0);
    v += gl >= 1 ? a : 0;
    const int b = dppi<kRowShr2>(v, 0);
    v += gl >= 2 ? b : 0;
  }
  return v;
}
template <int G>
__device__ __forceinline__ int lanes_last(int v) {
  if constexpr (G == 16) return row_last(v);
  else return dppi<0xFF>(v, 0);  // quad_perm 3 3 3 3
}
template <int G>
__global__ void __launch_bounds__(256) init_eq_kernel(ChainArrays ch, const EnsParams* ens, const float* tabs,
                                                        int first, int n) {
  static_assert(G == 16 || G == 4, "a row of lanes, or a quad");
  const int rl = threadIdx.x & (G - 1);
  const int idx = blockIdx.x * (256 / G) + threadIdx.x / G;
  const bool on = idx < n;  // rows past the end run along, without a store
  const int c = first + (on ? idx : 0);
  const EnsParams& P = ens[ch.ens[c]];
  const uint32_t k0 = P.key0, k1 = P.key1;
  const int nk = ch.nk[c];
  const uint32_t cid = ch.cid[c];
  const int64_t b = ch.base[c];
  int Z = 0;
  for (int w0 = 0; __ballot(w0 < nk); w0 += 4 * G) {
    const int wi = w0 + 4 * rl;  // words wi..wi+3: boundaries wi+1..wi+4; boundary nk always ends a strand
    uint4 x = make_uint4(0, 0, 0, 0);
    if (wi < nk - 1) x = philox4x32_10(make_uint4((uint32_t)(wi >> 2), 0u, cid, kPurposeInitCut), k0, k1);
    const uint32_t word[4] = {x.x, x.y, x.z, x.w};
    int cut[4], cnt = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = wi + k + 1;
      cut[k] = i == nk || (i < nk && word[k] < P.cut_threshold) ? 1 : 0;
      cnt += cut[k];
    }
    const int before = lanes_scan<G>(cnt, rl);  // inclusive
    const int total = lanes_last<G>(before);
    int at = Z + before - cnt;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (cut[k]) {
        if (on) ch.N[b + at] = wi + k + 1;
        ++at;
      }
    Z += total;
  }
  // The lanes' cut positions are complete (same wave, in issue order); lengths from the
  // last block of G strands down, each read before the strand below is rewritten
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const int zmax = Z;
  for (int s0 = (zmax - 1) & ~(G - 1); __ballot(s0 >= 0); s0 -= G) {
    const int k = s0 + rl;
    const bool in = s0 >= 0 && k < Z;
    int N = 0;
    if (in) N = ch.N[b + k] - (k > 0 ? ch.N[b + k - 1] : 0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (in && on) {
      float qx = 0.0f, qy = 0.0f, qz = 0.0f;
      if (k > 0 && k < Z - 1) {
        const uint4 g = philox4x32_10(make_uint4((uint32_t)k, 0u, cid, kPurposeInitQ), k0, k1);
        float g0, g1, g2, g3;
        boxmuller(g.x, g.y, g0, g1);
        boxmuller(g.z, g.w, g2, g3);
        const float sig = sqrtf((float)N / 3.0f);
        qx = g0 * sig; qy = g1 * sig; qz = g2 * sig;
      }
      ch.Qx[b + k] = qx; ch.Qy[b + k] = qy; ch.Qz[b + k] = qz;
      ch.N[b + k] = N;
    }
  }
  const float* pd = tabs + P.pd_off;
  for (int s0 = 0; __ballot(s0 < Z); s0 += 4 * G) {
    const int k = s0 + 4 * rl;
    if (k >= Z || !on) continue;
    uint4 x = make_uint4(0, 0, 0, 0), y = x;
    if (P.cd && k < Z - 1) {
      x = philox4x32_10(make_uint4((uint32_t)(k >> 2), 0u, cid, kPurposeInitTau), k0, k1);
      if (P.partner) y = philox4x32_10(make_uint4((uint32_t)(k >> 2), 0u, cid, kPurposeInitPartner), k0, k1);
    }
    const uint32_t word[4] = {x.x, x.y, x.z, x.w}, pw[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (k + q >= Z) continue;
      float w = 0.0f;
      if (P.cd && k + q < Z - 1)
        w = P.partner ? rate_ft_partner(pd, (int)(pw[q] >> (32 - kPartnerBits)), u01(word[q])) : rate_ft(&P, u01(word[q]));
      ch.w[b + k + q] = w;
    }
  }
  if (on && rl == 0) {
    ch.Z[c] = Z; ch.stall[c] = 0; ch.t[c] = 0.0; ch.ev[c] = 0; ch.dt_prev[c] = 0.0f; ch.zsum[c] = 0;
    ch.next_sample[c] = (P.sample_mode == kSampleFlow) ? 1 : 0;
    float* r1 = ch.R1 + 3 * (int64_t)c;  // common/chain.cu:207
    r1[0] = 0.0f; r1[1] = 0.0f; r1[2] = 0.0f;
  }
}

// ------------------------------------------------------------------ utility kernels
__global__ void fill_u32_kernel(uint32_t* p, uint32_t v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// one block: out[0] += sum of ev, out[1] += sum of zsum over a chain range
// SET: one block, out[0..1] the sums, out[2..n_zero) zero; otherwise added to out[0..1].
template <bool SET>
__global__ void __launch_bounds__(1024) sum_counters_kernel(const uint64_t* ev, const uint64_t* zsum, int chain0,
                                                             int n, unsigned long long* out, int n_zero) {
  __shared__ unsigned long long r0[1024], r1[1024];
  unsigned long long a0 = 0, a1 = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    a0 += ev[chain0 + i];
    a1 += zsum[chain0 + i];
  }
  r0[threadIdx.x] = a0;
  r1[threadIdx.x] = a1;
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) { r0[threadIdx.x] += r0[threadIdx.x + h]; r1[threadIdx.x] += r1[threadIdx.x + h]; }
    __syncthreads();
  }
  if constexpr (SET) {
    if (threadIdx.x < (unsigned)n_zero) out[threadIdx.x] = threadIdx.x == 0 ? r0[0] : (threadIdx.x == 1 ? r1[0] : 0ull);
  } else {
    if (threadIdx.x == 0) { atomicAdd(out, r0[0]); atomicAdd(out + 1, r1[0]); }
  }
}

__global__ void set_ev_stop_kernel(const uint64_t* ev, uint64_t* ev_stop, int chain0, int n, uint64_t add) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) ev_stop[chain0 + i] = ev[chain0 + i] + add;
}

// Chains of a pass into per-geometry lists by their current Z.  Geometry b takes a chain
// whose Z is below its capacity -- for the wave-form geometries (b >= 2) below 7/8 of it,
// so that a long chain, whose Z drifts by a few tens over a window, rarely outgrows its
// geometry mid-pass (it would then finish alone in the late round, after everything
// else; measured on the polydisperse melt, the same margin at the row and pair
// boundaries costs more in the first round than it saves in the late one).  Stalled
// chains go to geometry 0, which skips them.  Lists are cap entries apart, counts[b]
// their lengths.
// One global atomic per block and geometry (one per wave took 197 us for 262,144 chains, all
// on a line of L2): the waves of a geometry get consecutive slots of the block's.
// margin_div > 0: a chain within capacity/margin_div of a wave-form geometry's capacity
// starts in the next one (it would likely outgrow it during the pass)
// lane_cap > 0: list 0 takes the chains that will stay below that many positions (three
// standard deviations above the equilibrium Z, eight above now) whatever their geometry, the
// row form's others join list 1.
__global__ void __launch_bounds__(1024) split_geoms_kernel(const int* src, int n, const ChainArrays ch, const EnsParams* ens, int* lists,
                                   int cap, int* counts, int margin_div, int lane_cap) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = i < n ? src[i] : -1;
  int b = -1;
  if (c >= 0) {
    const int z = ch.Z[c];
    b = 0;
    bool fits = false;
    if (lane_cap > 0) {
      const float nk = (float)ch.nk[c], beta = ens[ch.ens[c]].beta;
      fits = z + 8 < lane_cap && lane_room(nk, beta) < (float)lane_cap;
      b = fits ? 0 : 1;
    }
    if (ch.stall[c] == 0 && !fits)
      while (b + 1 < kNumGeoms &&
             z >= kmc_geom_capacity(b) - (b >= 2 && margin_div > 0 ? kmc_geom_capacity(b) / margin_div : 0))
        ++b;
  }
  __shared__ int num[kNumGeoms], base[kNumGeoms];
  if (threadIdx.x < kNumGeoms) num[threadIdx.x] = 0;
  __syncthreads();
  const int lane = (int)__lane_id();
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int at = 0;  // within the block's share of the list
#pragma unroll
  for (int g = 0; g < kNumGeoms; ++g) {
    const uint64_t m = __ballot(b == g);
    if (m == 0) continue;
    const int leader = (int)__builtin_ctzll(m);
    int o = 0;
    if (lane == leader) o = atomicAdd(num + g, __popcll(m));
    o = __shfl(o, leader) + __popcll(m & below);
    at = b == g ? o : at;
  }
  __syncthreads();
  if (threadIdx.x < kNumGeoms && num[threadIdx.x] > 0)
    base[threadIdx.x] = atomicAdd(counts + threadIdx.x, num[threadIdx.x]);
  __syncthreads();
  if (b >= 0) lists[(int64_t)b * cap + base[b] + at] = c;
}

// Work list in decreasing Z (16 buckets of `width` positions; Z >= 16 * width first,
// stalled chains last): the chains started last, at the end of a pass, are the shortest.
__device__ __forceinline__ int zbucket(const int* Z, const int* stall, int width, int c) {
  if (stall[c] != 0) return 16;
  const int z = Z[c];
  return z >= 16 * width ? 0 : 15 - z / width;
}
constexpr int kZBuckets = kZOrderScratch;

// Block-local histograms in LDS, one global atomic per block and bucket (a per-element
// global atomic on 17 counters serialises in L2).  Grid-stride over the elements.
// src == null: the chains first .. first+n-1 (one ensemble's range)
__global__ void __launch_bounds__(1024) zhist_kernel(const int* src, int first, int n, const int* Z, const int* stall,
                                                     int width, int* hist) {
  __shared__ int lh[kZBuckets];
  if (threadIdx.x < kZBuckets) lh[threadIdx.x] = 0;
  __syncthreads();
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = src ? src[i] : first + i;
    if (c >= 0) atomicAdd(lh + zbucket(Z, stall, width, c), 1);
  }
  __syncthreads();
  if (threadIdx.x < kZBuckets && lh[threadIdx.x]) atomicAdd(hist + threadIdx.x, lh[threadIdx.x]);
}

// hist -> exclusive offsets (in place), total into *n_out
__global__ void zscan_kernel(int* hist, int* n_out) {
  if (threadIdx.x != 0) return;
  int acc = 0;
  for (int g = 0; g < kZBuckets; ++g) { const int h = hist[g]; hist[g] = acc; acc += h; }
  *n_out = acc;
}

// Each block reserves its range of every bucket with one atomic, then places its
// elements with LDS atomics (order within a bucket is arbitrary).
__global__ void __launch_bounds__(1024) zscatter_kernel(const int* src, int first, int n, const int* Z,
                                                        const int* stall, int width, int* cursor, int* dst) {
  __shared__ int lh[kZBuckets], base[kZBuckets];
  if (threadIdx.x < kZBuckets) lh[threadIdx.x] = 0;
  __syncthreads();
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = src ? src[i] : first + i;
    if (c >= 0) atomicAdd(lh + zbucket(Z, stall, width, c), 1);
  }
  __syncthreads();
  if (threadIdx.x < kZBuckets) {
    base[threadIdx.x] = lh[threadIdx.x] ? atomicAdd(cursor + threadIdx.x, lh[threadIdx.x]) : 0;
    lh[threadIdx.x] = 0;
  }
  __syncthreads();
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = src ? src[i] : first + i;
    if (c >= 0) {
      const int b = zbucket(Z, stall, width, c);
      dst[base[b] + atomicAdd(lh + b, 1)] = c;
    }
  }
}

// The whole of it, and the counts of a sequential pass (init_counts_kernel), in one block:
// short lists, where a pass's time is its launches.
__global__ void __launch_bounds__(1024) zorder_block_kernel(const int* src, int first, int n, const int* Z,
                                                            const int* stall, int width, int* cnt, int n_cnt, int n0,
                                                            int* dst, int* n_out) {
  __shared__ int lh[kZBuckets], at[kZBuckets];
  for (int i = threadIdx.x; i < n_cnt; i += 1024) cnt[i] = i == 0 ? n0 : 0;
  if (threadIdx.x < kZBuckets) lh[threadIdx.x] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 1024) {
    const int c = src ? src[i] : first + i;
    if (c >= 0) atomicAdd(lh + zbucket(Z, stall, width, c), 1);
  }
  __syncthreads();
  if (threadIdx.x < kZBuckets) {
    int before = 0;
    for (int b = 0; b < (int)threadIdx.x; ++b) before += lh[b];
    at[threadIdx.x] = before;
    if (threadIdx.x == kZBuckets - 1) *n_out = before + lh[kZBuckets - 1];  // (behind the counts' zeros)
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 1024) {
    const int c = src ? src[i] : first + i;
    if (c >= 0) dst[atomicAdd(at + zbucket(Z, stall, width, c), 1)] = c;
  }
}

// counts of a sequential pass: cnt[0] = n0, the rest (lists, queues, order scratch) zero
__global__ void init_counts_kernel(int* cnt, int n, int n0) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cnt[i] = i == 0 ? n0 : 0;
}

__global__ void iota_kernel(int* p, int start, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = start + i;
}

// flow stress: per (sample, ensemble) FP64 sums of the 8 components over healthy
// chains (stall == 0, finite, recorded); out[...*9 + 8] = chain count.
// (common/ensemble_call_block.cu:452-505 averages in FP32 on the host.)
// A row of a chain counts when the chain recorded it (Z column >= 1: staging rows start
// at zero and a chain that has stalled records nothing after the stall) and it holds no
// NaN, so a chain that stalls mid-window keeps the rows it recorded before, as the
// reference excludes a stalled chain only from the outputs after its stall
// (common/ensemble_call_block.cu:471-491, per output step).
// Block (row, part) sums one of gridDim.y parts of the chains into part[row][part][9]; with
// one part that is the row's result, otherwise flow_parts_kernel adds the parts in order.
// (One block a row: 87 us for 8 rows of 16,384 chains, four parts in flight a row.)
__global__ void __launch_bounds__(256) flow_reduce_kernel(const float* stage, int nchains, double* part) {
  const int row = blockIdx.x;
  const int per = (nchains + gridDim.y - 1) / gridDim.y;
  const int lo = blockIdx.y * per, hi = min(nchains, lo + per);
  __shared__ double red[9][4];
  double acc[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) acc[q] = 0.0;
  for (int c = lo + threadIdx.x; c < hi; c += blockDim.x) {
    const float4* o4 = (const float4*)(stage + ((int64_t)row * nchains + c) * 8);
    const float4 a = o4[0], b = o4[1];
    const float o[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    bool ok = o[7] > 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) ok = ok && (o[q] == o[q]);
    if (ok) {
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] += (double)o[q];
      acc[8] += 1.0;
    }
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    for (int d = 32; d > 0; d >>= 1) acc[q] += __shfl_down(acc[q], d, 64);
    if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = acc[q];
  }
  __syncthreads();
  if (threadIdx.x < 9)
    part[((int64_t)row * gridDim.y + blockIdx.y) * 9 + threadIdx.x] =
        ((red[threadIdx.x][0] + red[threadIdx.x][1]) + red[threadIdx.x][2]) + red[threadIdx.x][3];
}
__global__ void __launch_bounds__(256) flow_parts_kernel(const double* part, int parts, int nrows, double* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrows * 9) return;
  const int row = i / 9, q = i - 9 * row;
  double acc = 0.0;
  for (int k = 0; k < parts; ++k) acc += part[((int64_t)row * parts + k) * 9 + q];
  out[i] = acc;
}

// ------------------------------------------------------------------ multi-tau correlator
// Thread per chain (lanes = consecutive chains -> every access below is coalesced).
// Per-chain FP64 state: D[level][slot][3], A[level][3], C[level][lag]
// (C accumulates the sum of the three component products).  The level
// counters are identical for all chains (sampling is synchronous) and are
// passed in; the host advances its copy by the same rule after each launch.
// Insert rule, block averages and lag products: common/eq_ensemble_kernel.cu:133-227.
struct CorrArgs {
  const float* stage;   // [k][chain][3]
  double* D;            // [((lvl*p + slot)*3 + comp)*nch + chain]
  double* A;            // [(lvl*3 + comp)*nch + chain]
  double* C;            // [(lvl*p + lag)*nch + chain]
  const int* stall;     // global stall flags
  int chain0, nch, p, m, s, nrows;
  const int* cnt;       // [3*s]: ins, macc, nins (clamped to p) at window start
  int type;             // 0: stress (block averages, products); 1: MSD (first value, squared differences)
};

// One value into level `lvl` and, through the block pushes, the levels above it
// (D, A and C in device memory).
__device__ __forceinline__ void corr_insert_from(const CorrArgs& a, int c, int lvl, double vx, double vy, double vz,
                                                 int* ins, int* macc, int* nins) {
  const int64_t nch = a.nch;
  const int p = a.p, m = a.m;
  for (;;) {
    if (lvl == a.s) break;
    const int in = ins[lvl];
    double* D = a.D + (int64_t)(lvl * p) * 3 * nch + c;
    D[(int64_t)(in * 3 + 0) * nch] = vx;
    D[(int64_t)(in * 3 + 1) * nch] = vy;
    D[(int64_t)(in * 3 + 2) * nch] = vz;
    double* A = a.A + (int64_t)(lvl * 3) * nch + c;
    // MSD carries the first value of each block up unaveraged
    // (common/eq_ensemble_kernel.cu:181-189)
    if (a.type == 0 || macc[lvl] == 0) { A[0] += vx; A[nch] += vy; A[2 * nch] += vz; }
    macc[lvl]++;
    const bool push = macc[lvl] == m;
    double ux = 0.0, uy = 0.0, uz = 0.0;
    if (push) {
      if (a.type == 0) { ux = A[0] / m; uy = A[nch] / m; uz = A[2 * nch] / m; }
      else { ux = A[0]; uy = A[nch]; uz = A[2 * nch]; }
      A[0] = 0.0; A[nch] = 0.0; A[2 * nch] = 0.0;
      macc[lvl] = 0;
    }
    const int jmin = (lvl == 0) ? 0 : p / m;
    double* Cc = a.C + (int64_t)(lvl * p) * nch + c;
    for (int j = jmin; j < p; ++j) {
      if (j > nins[lvl]) break;
      int idx = in - j;
      if (idx < 0) idx += p;
      const double dx = D[(int64_t)(idx * 3 + 0) * nch];
      const double dy = D[(int64_t)(idx * 3 + 1) * nch];
      const double dz = D[(int64_t)(idx * 3 + 2) * nch];
      if (a.type == 0) {
        Cc[(int64_t)j * nch] += vx * dx + vy * dy + vz * dz;
      } else {
        const double ex = vx - dx, ey = vy - dy, ez = vz - dz;
        Cc[(int64_t)j * nch] += ex * ex + ey * ey + ez * ez;
      }
    }
    ins[lvl] = (in + 1 == p) ? 0 : in + 1;
    nins[lvl] = nins[lvl] < p ? nins[lvl] + 1 : p;
    if (!push) break;
    ++lvl;
    vx = ux; vy = uy; vz = uz;
  }
}

// p too large for the kernel below: thread per chain, every level in device memory.
__global__ void __launch_bounds__(256) corr_update_serial_kernel(CorrArgs a) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.nch) return;
  int ins[40], macc[40], nins[40];
  for (int k = 0; k < a.s; ++k) { ins[k] = a.cnt[k]; macc[k] = a.cnt[a.s + k]; nins[k] = a.cnt[2 * a.s + k]; }
  const int64_t nch = a.nch;
  for (int row = 0; row < a.nrows; ++row) {
    const float* o = a.stage + ((int64_t)row * nch + c) * 3;
    corr_insert_from(a, c, 0, o[0], o[1], o[2], ins, macc, nins);
  }
}


// A window's samples into the correlator, level by level: kCorrChains chains per block
// (chain fastest in the thread index and in LDS, as in device memory) by up to 16 lag
// threads.  A level's values of a chunk of rows lie in LDS behind the last p before them,
// so every lag of every chain sums its products on its own, in row order as a sample by
// sample update does, and the accumulators and shift register of a level are read and
// written once per chunk.  The block averages (first values for MSD) handed up are the
// next level's values.
// One thread per chain with the lags in turn was bound by its serial chain of device-memory
// accesses: 64 rows of 20,011 chains with p = 64 took 2,909 us, of 1000 chains with p = 16
// 231 us.
template <int CH>
__global__ void __launch_bounds__(16 * CH) corr_update_kernel(CorrArgs a, int chunk) {
  extern __shared__ double corr_lds[];
  const int p = a.p, m = a.m, LT = blockDim.x / CH;
  double* cur = corr_lds;                            // [p older values, oldest first; chunk new ones][3][CH]
  double* nxt = cur + (int64_t)(p + chunk) * 3 * CH;  // [chunk / m + 1][3][CH]
  const int ch = threadIdx.x % CH, lt = threadIdx.x / CH;
  const int c0 = blockIdx.x * CH, c = c0 + ch;
  const bool on = c < a.nch;
  const int64_t nch = a.nch;
  for (int row0 = 0; row0 < a.nrows; row0 += chunk) {
    int n = min(chunk, a.nrows - row0);
    const int live = min(CH, a.nch - c0);
    for (int e = threadIdx.x; e < n * 3 * live; e += blockDim.x) {
      const int r = e / (3 * live), x = e - r * 3 * live;
      cur[((p + r) * 3 + x % 3) * CH + x / 3] = (double)a.stage[((int64_t)(row0 + r) * nch + c0) * 3 + x];
    }
    int done = row0;  // values this level took in earlier chunks of the window
    for (int lvl = 0; lvl < a.s && n > 0; ++lvl) {
      const int ins = (int)((a.cnt[lvl] + (int64_t)done) % p);
      const int macc = (int)((a.cnt[a.s + lvl] + (int64_t)done) % m);
      const int nins = min(p, a.cnt[2 * a.s + lvl] + done);
      double* D = a.D + (int64_t)(lvl * p) * 3 * nch + c;
      for (int i = lt; i < p; i += LT) {
        const int age = p - i;
        if (on && age <= nins) {
          const int slot = ins >= age ? ins - age : ins - age + p;
#pragma unroll
          for (int q = 0; q < 3; ++q) cur[(i * 3 + q) * CH + ch] = D[(int64_t)(slot * 3 + q) * nch];
        }
      }
      __syncthreads();
      // lag sums: four lags of a thread share the reads of the new value
      const int jmin = lvl == 0 ? 0 : p / m;
      for (int j0 = lt; j0 < p; j0 += 4 * LT) {
        double cs[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int j = j0 + k * LT;
          cs[k] = on && j >= jmin && j < p ? a.C[(int64_t)(lvl * p + j) * nch + c] : 0.0;
        }
        if (on) {
          for (int r = 0; r < n; ++r) {
            const double vx = cur[((p + r) * 3 + 0) * CH + ch], vy = cur[((p + r) * 3 + 1) * CH + ch],
                         vz = cur[((p + r) * 3 + 2) * CH + ch];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const int j = j0 + k * LT;
              if (j < p && nins + r >= j) {
                const double* d = cur + (p + r - j) * 3 * CH + ch;
                const double dx = d[0], dy = d[CH], dz = d[2 * CH];
                if (a.type == 0) {
                  cs[k] += vx * dx + vy * dy + vz * dz;
                } else {
                  const double ex = vx - dx, ey = vy - dy, ez = vz - dz;
                  cs[k] += ex * ex + ey * ey + ez * ez;
                }
              }
            }
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int j = j0 + k * LT;
          if (on && j >= jmin && j < p) a.C[(int64_t)(lvl * p + j) * nch + c] = cs[k];
        }
      }
      // block accumulators, one component a thread; MSD carries the first value of each
      // block up unaveraged (common/eq_ensemble_kernel.cu:181-189)
      if (on) {
        for (int q = lt; q < 3; q += LT) {
          double acc = a.A[(int64_t)(lvl * 3 + q) * nch + c];
          int mc = macc, k = 0;
          for (int r = 0; r < n; ++r) {
            const double v = cur[((p + r) * 3 + q) * CH + ch];
            if (a.type == 0 || mc == 0) acc += v;
            if (++mc == m) {
              nxt[(k * 3 + q) * CH + ch] = a.type == 0 ? acc / m : acc;
              acc = 0.0;
              mc = 0;
              ++k;
            }
          }
          a.A[(int64_t)(lvl * 3 + q) * nch + c] = acc;
        }
        for (int r = max(0, n - p) + lt; r < n; r += LT) {
          const int slot = (ins + r) % p;
#pragma unroll
          for (int q = 0; q < 3; ++q) D[(int64_t)(slot * 3 + q) * nch] = cur[((p + r) * 3 + q) * CH + ch];
        }
      }
      __syncthreads();
      const int up = (macc + n) / m;
      for (int e = threadIdx.x; e < up * 3 * CH; e += blockDim.x) cur[p * 3 * CH + e] = nxt[e];
      done = (int)((a.cnt[a.s + lvl] + (int64_t)done) / m);
      n = up;
      __syncthreads();
    }
  }
}

// G(level, lag) = sum over healthy chains of C / (3 * n_pairs * n_healthy); the chains are
// first .. first+count-1 of an ensemble of ld chains (C is [point][ld]).  Block (point,
// part) sums one of gridDim.y parts of the chains; points without a pair yet, and the lags
// below p/m of the upper levels, are left out.  The parts are added in order by
// corr_parts_kernel, so the result does not depend on timing.  Row npts counts the chains.
// (One block a point: 345 us for 192 points of 131,072 chains; 40 us in 32 parts.)
struct CorrPoints {
  int p, m, s;
  int nins[40];  // values each level has taken, clamped to p
};
__global__ void __launch_bounds__(256) corr_reduce_kernel(const double* C, int ld, const int* stall, int chain0,
                                                            int first, int count, CorrPoints P, double* part) {
  const int pt = blockIdx.x, npts = P.s * P.p;
  const int lvl = pt / P.p, lag = pt - lvl * P.p;
  if (pt < npts && (lag >= P.nins[lvl] || (lvl > 0 && lag < P.p / P.m))) {
    if (threadIdx.x == 0) part[(int64_t)pt * gridDim.y + blockIdx.y] = 0.0;
    return;
  }
  const int per = (count + gridDim.y - 1) / gridDim.y;
  const int lo = first + blockIdx.y * per, hi = min(first + count, lo + per);
  double acc = 0.0;
  for (int c = lo + threadIdx.x; c < hi; c += blockDim.x)
    if (stall[chain0 + c] == 0) acc += pt < npts ? C[(int64_t)pt * ld + c] : 1.0;
  __shared__ double red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[(int64_t)pt * gridDim.y + blockIdx.y] = red[0];
}
__global__ void __launch_bounds__(256) corr_parts_kernel(const double* part, int parts, int npts, double* out) {
  const int pt = blockIdx.x * blockDim.x + threadIdx.x;
  if (pt >= npts) return;
  double acc = 0.0;
  for (int k = 0; k < parts; ++k) acc += part[(int64_t)pt * parts + k];
  out[pt] = acc;
}

// ------------------------------------------------------------------ window parameters
// Head of a window pass: (t_end, k0, k_end) of every ensemble of the pass into its
// EnsParams, then the correlator level counters.  One block.  In a captured pass they come
// from a block of pinned host memory the host fills before each replay, so the graph itself
// never changes; so do those of many ensembles.  Otherwise they are the launch's argument
// (the pinned block costs an engine 0.25 ms to have and to give back).
__device__ __forceinline__ void stage_window(const WinParam* wp, int n_ens, EnsParams* P, const int* cnt_src,
                                             int* cnt_dst, int n_cnt) {
  for (int i = threadIdx.x; i < n_ens; i += blockDim.x) {
    const WinParam w = wp[i];
    P[w.ens].t_end = w.t_end;
    P[w.ens].k0 = w.k0;
    P[w.ens].k_end = w.k_end;
  }
  for (int i = threadIdx.x; i < n_cnt; i += blockDim.x) cnt_dst[i] = cnt_src[i];
}
__global__ void __launch_bounds__(256) stage_window_kernel(const WinParam* __restrict__ wp, int n_ens,
                                                           EnsParams* P, const int* __restrict__ cnt_src,
                                                           int* cnt_dst, int n_cnt) {
  stage_window(wp, n_ens, P, cnt_src, cnt_dst, n_cnt);
}
__global__ void __launch_bounds__(256) stage_args_kernel(WinArgs w, EnsParams* P, int* cnt_dst) {
  stage_window(w.win, w.n_ens, P, w.cnt, cnt_dst, w.n_cnt);
}

// ------------------------------------------------------------------ ensemble stress now
// Stress of the current state (common/ensemble_kernel.cu:504-538 per chain, averaged by
// common/ensemble.cu:210-221): per chain sigma_ab = -sum_i 3 Q_ia Q_ib / N_i, Lpp =
// sum_i |Q_i| and Z, in FP64 from the stored FP32 strands, after the deformation still
// pending from the chain's last jump (dt_prev; the reference applies it with olddt).
// Chains that have stalled are left out.  A fixed grid of kStressBlocks blocks strides
// over the chains, one wave a chain, one lane a strand (the arrays are read in whole
// lines; one thread a chain took 101 us for 20,011 chains of Z ~ 100, call included, this 42).
// A wave looks at 16 chains a turn (four lanes each; their headers' latency once) and does
// them together where none is longer than 16, else four at a time, 16 lanes a chain, where
// none of the four is longer than 64 (200,000 chains of Nk 6: 39 us a thread a chain, 98 a
// wave a chain, 38 so; 60,000 of Nk 12 31, 40, 31; 131,072 of Nk 100 281, 83, 59).  Block b writes
// its partial sums to part[9b .. 9b+8] (xx yy zz xy yz zx Lpp Z count), which the host adds in
// block order, so the result does not depend on timing.
constexpr int kStressWaves = 16;
struct StressSum {
  double v[9];
  __device__ __forceinline__ void add(const ChainArrays& ch, const KappaArg& K, int64_t s, double dt) {
    double x = ch.Qx[s], y = ch.Qy[s], z = ch.Qz[s];
    if (dt != 0.0) {
      const double x1 = x + dt * ((double)K.k[0] * x + (double)K.k[1] * y + (double)K.k[2] * z);
      const double y1 = y + dt * ((double)K.k[3] * x + (double)K.k[4] * y + (double)K.k[5] * z);
      const double z1 = z + dt * ((double)K.k[6] * x + (double)K.k[7] * y + (double)K.k[8] * z);
      x = x1; y = y1; z = z1;
    }
    const double t3 = 3.0 / (double)ch.N[s];
    v[0] -= t3 * x * x; v[1] -= t3 * y * y; v[2] -= t3 * z * z;
    v[3] -= t3 * x * y; v[4] -= t3 * y * z; v[5] -= t3 * x * z;
    v[6] += sqrt(x * x + y * y + z * z);
  }
};
__global__ void __launch_bounds__(64 * kStressWaves) chain_stress_kernel(ChainArrays ch, int chain0, int n, KappaArg K,
                                                                         double* part) {
  __shared__ double red[9][kStressWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4, rl = lane & 15, ql = lane & 3;
  if ((int)blockIdx.x * kStressWaves >= n) {  // no chain is left for it
    if (threadIdx.x < 9) part[blockIdx.x * 9 + threadIdx.x] = 0.0;
    return;
  }
  StressSum S;
  double (&acc)[9] = S.v;
#pragma unroll
  for (int q = 0; q < 9; ++q) acc[q] = 0.0;
  const int stride = gridDim.x * kStressWaves;
  for (int i0 = blockIdx.x * kStressWaves + wave; i0 < n; i0 += 16 * stride) {
    // lanes 4g .. 4g+3 have chain i0 + g * stride
    const int i = i0 + (lane >> 2) * stride, c = chain0 + i;
    int Z = 0;
    int64_t b = 0;
    float dt = 0.0f;
    if (i < n && ch.stall[c] == 0) {
      Z = ch.Z[c];
      b = ch.base[c];
      dt = ch.dt_prev[c];
      if (ql == 0) {
        acc[7] += (double)Z;
        acc[8] += 1.0;
      }
    }
    if (i0 + stride < n && !__ballot(Z > 16)) {
      for (int k = ql; k < Z; k += 4) S.add(ch, K, b + k, (double)dt);
      continue;
    }
    for (int h = 0; h < 4 && i0 + 4 * h * stride < n; ++h) {
      const int Zr = __shfl(Z, 16 * h + 4 * row);
      const int64_t br = __shfl(b, 16 * h + 4 * row);
      const float dr = __shfl(dt, 16 * h + 4 * row);
      if (i0 + (4 * h + 1) * stride < n && !__ballot(Zr > 64)) {
        for (int k = rl; k < Zr; k += 16) S.add(ch, K, br + k, (double)dr);
      } else {
        for (int r = 0; r < 4; ++r) {
          const int Zc = __shfl(Zr, 16 * r);
          if (Zc == 0) continue;
          const int64_t bc = __shfl(br, 16 * r);
          const double dc = (double)__shfl(dr, 16 * r);
          for (int k = lane; k < Zc; k += 64) S.add(ch, K, bc + k, dc);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    for (int d = 32; d > 0; d >>= 1) acc[q] += __shfl_down(acc[q], d, 64);
    if (lane == 0) red[q][wave] = acc[q];
  }
  __syncthreads();
  if (threadIdx.x < 9) {
    double s = 0.0;
    for (int w = 0; w < kStressWaves; ++w) s += red[threadIdx.x][w];
    part[blockIdx.x * 9 + threadIdx.x] = s;
  }
}

// ------------------------------------------------------------------ state invariants
// Counts, over chains chain0 .. chain0+n-1, the violations of the model's invariants
// (App. A.1 of the chain state): out[0] Z outside 1..Nk, out[1] a strand with N < 1,
// out[2] sum of N != Nk, out[3] an end strand (index 0 or Z-1, Z > 1) with Q != 0,
// out[4] a non-finite Q or CD rate, out[5] stalled chains, out[6] chains whose clock is
// below t_min.  The counters (7 x uint64) must be zero on entry.  One wave a chain, one lane
// a strand (one thread a chain took 130 us for 20,011 chains of Z ~ 100, call included, this
// 42), or 16 or four shorter chains at a time as above (200,000 of Nk 6: 41, 124, 41 us; 60,000
// of Nk 12 32, 53, 33; 131,072 of Nk 100 572, 97, 72).
struct StrandChecks {
  long long all;
  bool n, f, e;
  __device__ __forceinline__ void add(const ChainArrays& ch, int64_t b, int k, int Z) {
    const int N = ch.N[b + k];
    n = n || N < 1;
    all += N;
    const float x = ch.Qx[b + k], y = ch.Qy[b + k], z = ch.Qz[b + k];
    f = f || !isfinite(x) || !isfinite(y) || !isfinite(z) || (k < Z - 1 && !isfinite(ch.w[b + k]));
    if (Z > 1 && (k == 0 || k == Z - 1)) e = e || x != 0.f || y != 0.f || z != 0.f;
  }
  // the findings of the lanes of `mask` (all: their sum), to be counted by one of them
  __device__ __forceinline__ void count(uint64_t mask, bool mine, int nk, unsigned int (&v)[7]) const {
    const bool bn = (__ballot(n) & mask) != 0, bf = (__ballot(f) & mask) != 0, be = (__ballot(e) & mask) != 0;
    if (mine) {
      v[1] += bn;
      v[2] += all != nk;
      v[3] += be;
      v[4] += bf;
    }
  }
};
__global__ void __launch_bounds__(256) check_state_kernel(ChainArrays ch, int chain0, int n, double t_min,
                                                          unsigned long long* out) {
  __shared__ unsigned int tot[7];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4, rl = lane & 15, ql = lane & 3;
  if (threadIdx.x < 7) tot[threadIdx.x] = 0;
  __syncthreads();
  unsigned int v[7] = {0, 0, 0, 0, 0, 0, 0};  // on every fourth lane
  const int stride = gridDim.x * 4;
  for (int i0 = blockIdx.x * 4 + wave; i0 < n; i0 += 16 * stride) {
    const int i = i0 + (lane >> 2) * stride, c = chain0 + i;  // lanes 4g .. 4g+3: chain i0 + g * stride
    int Z = 0, nk = 0;
    int64_t b = 0;
    if (i < n) {
      Z = ch.Z[c];
      nk = ch.nk[c];
      b = ch.base[c];
      const bool in = Z >= 1 && Z <= nk && Z <= ch.cap[c];
      if (ql == 0) {
        v[0] += !in;
        v[5] += ch.stall[c] != 0;
        v[6] += !(ch.t[c] >= t_min);
      }
      Z = in ? Z : 0;
    }
    if (i0 + stride < n && !__ballot(Z > 16)) {
      StrandChecks s{0, false, false, false};
      for (int k = ql; k < Z; k += 4) s.add(ch, b, k, Z);
      for (int d = 2; d > 0; d >>= 1) s.all += __shfl_xor(s.all, d, 64);
      s.count(0xfull << (lane & ~3), ql == 0 && Z > 0, nk, v);
      continue;
    }
    for (int h = 0; h < 4 && i0 + 4 * h * stride < n; ++h) {
      const int Zr = __shfl(Z, 16 * h + 4 * row), nr = __shfl(nk, 16 * h + 4 * row);
      const int64_t br = __shfl(b, 16 * h + 4 * row);
      if (i0 + (4 * h + 1) * stride < n && !__ballot(Zr > 64)) {
        StrandChecks s{0, false, false, false};
        for (int k = rl; k < Zr; k += 16) s.add(ch, br, k, Zr);
        for (int d = 8; d > 0; d >>= 1) s.all += __shfl_xor(s.all, d, 64);
        s.count(0xffffull << (16 * row), rl == 0 && Zr > 0, nr, v);
      } else {
        for (int r = 0; r < 4; ++r) {
          const int Zc = __shfl(Zr, 16 * r);
          if (Zc == 0) continue;
          const int64_t bc = __shfl(br, 16 * r);
          StrandChecks s{0, false, false, false};
          for (int k = lane; k < Zc; k += 64) s.add(ch, bc, k, Zc);
          for (int d = 32; d > 0; d >>= 1) s.all += __shfl_xor(s.all, d, 64);
          s.count(~0ull, lane == 16 * r, nr, v);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 7; ++q)
    if (ql == 0 && v[q]) atomicAdd(tot + q, v[q]);
  __syncthreads();
  if (threadIdx.x < 7 && tot[threadIdx.x]) atomicAdd(out + threadIdx.x, (unsigned long long)tot[threadIdx.x]);
}

// ------------------------------------------------------------------ copy probe (bandwidth)
// Plain 16-byte copy, grid-stride: the reference point for HBM byte counters and the
// achievable copy bandwidth of the device.
__global__ void copy_probe_kernel(const float4* __restrict__ in, float4* __restrict__ out, size_t n4) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) out[i] = in[i];
}

// ------------------------------------------------------------------ scan probe (tests)
// Canonical scan tree of the KMC kernels.  form 1: one chain of n <= 1024 positions
// (wave form, four register groups): out[0..n) inclusive sums, out[n] total.
// form 0: four chains of n <= 64 positions (row form), form 2: two chains of n <= 128
// positions (pair form), form 3: two chains of n <= 256 positions (pair form with two
// register groups), form 4: four chains of n <= 128 positions (row form with two register
// groups): chain r reads in[r*n ..] and writes out[r*(n+1) ..].
// Centre-of-mass sample of one chain state in a chosen geometry (0 row form, 1 pair form,
// 2/3/4 wave form G = 1/2/4, 7 pair form with two groups): in[4i..4i+3] = Qx Qy Qz N of
// strand i, in[4n] = Nk; out = 3 floats.
template <int CPW, int G>
__device__ void com_probe(const float* in, float* out, int n, lds_f* buf) {
  static_assert(Geo<CPW, G>::STG <= 1024, "the strand lengths fit the probe's LDS buffer");
  const LaneC<CPW> L;
  const Stage<CPW, G> S{buf, L.srow * G};
  Strands<G> C;
  int nv[4 * G];
#pragma unroll
  for (int j = 0; j < 4 * G; ++j) {
    const int p = L.pos(j);
    const bool on = p < n;
    C.qx[j] = on ? in[4 * p] : 0.0f;
    C.qy[j] = on ? in[4 * p + 1] : 0.0f;
    C.qz[j] = on ? in[4 * p + 2] : 0.0f;
    nv[j] = on ? (int)in[4 * p + 3] : 0;
    C.w[j] = 0.0f;
  }
#pragma unroll
  for (int g = 0; g < G; ++g) S.put4i(kStN, g, L.pos0, nv[4 * g], nv[4 * g + 1], nv[4 * g + 2], nv[4 * g + 3]);
  wave_lds_sync();
  float sv[3];
  com_sample<CPW, G>(C, S, n, in[4 * n], L, sv);
  if (L.lane == 0) { out[0] = sv[0]; out[1] = sv[1]; out[2] = sv[2]; }
}
__global__ void __launch_bounds__(64) com_probe_kernel(const float* in, float* out, int n, int geom) {
  __shared__ float buf[1024];  // the kStN staging array of one wave (strand lengths)
  lds_f* b = (lds_f*)buf;
  if (geom == 0) com_probe<4, 1>(in, out, n, b);
  else if (geom == 1) com_probe<2, 1>(in, out, n, b);
  else if (geom == 2) com_probe<1, 1>(in, out, n, b);
  else if (geom == 3) com_probe<1, 2>(in, out, n, b);
  else if (geom == kGeomPair2) com_probe<2, 2>(in, out, n, b);
  else if (geom == kGeomRow2) com_probe<4, 2>(in, out, n, b);
  else com_probe<1, 4>(in, out, n, b);
}

__global__ void __launch_bounds__(64) scan_probe_kernel(const float* in, float* out, int n, int form) {
  if (form == 5) {
    const LaneC<1> L;
    float v[8], g[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = L.pos(j);
      v[j] = p < n ? in[p] : 0.0f;
    }
    const float tot = chain_scan<1, 2>(v, g, n, L);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = L.pos(j);
      if (p < n) out[p] = g[j];
    }
    if (L.lane == 0) out[n] = tot;
  } else if (form == 1) {
    const LaneC<1> L;
    float v[16], g[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int p = L.pos(j);
      v[j] = p < n ? in[p] : 0.0f;
    }
    const float tot = chain_scan<1, 4>(v, g, n, L);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int p = L.pos(j);
      if (p < n) out[p] = g[j];
    }
    if (L.lane == 0) out[n] = tot;
  } else if (form == 2) {
    const LaneC<2> L;
    const int r = L.lane >> 5;
    float v[4], g[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = L.pos(j);
      v[j] = p < n ? in[r * n + p] : 0.0f;
    }
    const float tot = chain_scan<2, 1>(v, g, n, L);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = L.pos(j);
      if (p < n) out[r * (n + 1) + p] = g[j];
    }
    if (L.sl == 0) out[r * (n + 1) + n] = tot;
  } else if (form == 4) {
    const LaneC<4> L;
    const int r = L.lane >> 4;
    float v[8], g[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = L.pos(j);
      v[j] = p < n ? in[r * n + p] : 0.0f;
    }
    const float tot = chain_scan<4, 2>(v, g, n, L);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = L.pos(j);
      if (p < n) out[r * (n + 1) + p] = g[j];
    }
    if (L.sl == 0) out[r * (n + 1) + n] = tot;
  } else if (form == 3) {
    const LaneC<2> L;
    const int r = L.lane >> 5;
    float v[8], g[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = L.pos(j);
      v[j] = p < n ? in[r * n + p] : 0.0f;
    }
    const float tot = chain_scan<2, 2>(v, g, n, L);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = L.pos(j);
      if (p < n) out[r * (n + 1) + p] = g[j];
    }
    if (L.sl == 0) out[r * (n + 1) + n] = tot;
  } else {
    const LaneC<4> L;
    const int r = L.lane >> 4;
    float v[4], g[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = L.pos(j);
      v[j] = p < n ? in[r * n + p] : 0.0f;
    }
    const float tot = chain_scan<4, 1>(v, g, n, L);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = L.pos(j);
      if (p < n) out[r * (n + 1) + p] = g[j];
    }
    if (L.sl == 0) out[r * (n + 1) + n] = tot;
  }
}

__global__ void math_probe_kernel(const float* in, float* out, int n, int which) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float x = in[i];
  float r = 0.0f;
  if (which == 0) r = dexpf(x);
  else if (which == 1) r = dlogf(x);
  else if (which == 2) { float s, c; dsincos2pif(x, s, c); r = s; }
  else if (which == 3) { float s, c; dsincos2pif(x, s, c); r = c; }
  out[i] = r;
}

__global__ void philox_probe_kernel(const uint32_t* ctr_key, uint32_t* out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t* q = ctr_key + 6 * i;
  const uint4 r = philox4x32_10(make_uint4(q[0], q[1], q[2], q[3]), q[4], q[5]);
  out[4 * i + 0] = r.x; out[4 * i + 1] = r.y; out[4 * i + 2] = r.z; out[4 * i + 3] = r.w;
}

}  // namespace dsm

// ------------------------------------------------------------------ launchers
#include "dsm_launch.h"

namespace dsm {

hipError_t launch_kmc(const KmcArgs& a, int geom, bool plain, int grid, hipStream_t st) {
  static_assert(kNumGeoms == 6, "one case per geometry below");
  switch (geom) {
    case 0: return launch_kmc_geom_0(a, plain, grid, st);
    case 1: return launch_kmc_geom_1(a, plain, grid, st);
    case 2: return launch_kmc_geom_2(a, plain, grid, st);
    case 3: return launch_kmc_geom_3(a, plain, grid, st);
    case 4: return launch_kmc_geom_4(a, plain, grid, st);
    case 5: return launch_kmc_geom_5(a, plain, grid, st);
    case kGeomPair2: return launch_kmc_geom_7(a, plain, grid, st);
    default: return hipErrorInvalidValue;
  }
}

int kmc_max_blocks_per_cu(int geom, bool plain, int lds_floats, bool ext) {
  switch (geom) {
    case 0: return kmc_occupancy_geom_0(plain, lds_floats, ext);
    case 1: return kmc_occupancy_geom_1(plain, lds_floats, ext);
    case 2: return kmc_occupancy_geom_2(plain, lds_floats, ext);
    case 3: return kmc_occupancy_geom_3(plain, lds_floats, ext);
    case 4: return kmc_occupancy_geom_4(plain, lds_floats, ext);
    case 5: return kmc_occupancy_geom_5(plain, lds_floats, ext);
    case kGeomPair2: return kmc_occupancy_geom_7(plain, lds_floats, ext);
    default: return 0;
  }
}


hipError_t launch_init_eq(const ChainArrays& ch, const EnsParams* ens, const float* tabs, int first, int n,
                          int lanes, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  if (lanes == 16)
    hipLaunchKernelGGL(init_eq_kernel<16>, dim3((n + 15) / 16), dim3(256), 0, st, ch, ens, tabs, first, n);
  else
    hipLaunchKernelGGL(init_eq_kernel<4>, dim3((n + 63) / 64), dim3(256), 0, st, ch, ens, tabs, first, n);
  return hipGetLastError();
}

hipError_t launch_fill_u32(void* p, uint32_t v, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (uint32_t*)p, v, n);
  return hipGetLastError();
}

hipError_t launch_set_ev_stop(const uint64_t* ev, uint64_t* ev_stop, int chain0, int n, uint64_t add,
                              hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(set_ev_stop_kernel, dim3((n + 255) / 256), dim3(256), 0, st, ev, ev_stop, chain0, n, add);
  return hipGetLastError();
}

hipError_t launch_sum_counters(const uint64_t* ev, const uint64_t* zsum, int chain0, int n, unsigned long long* out,
                               hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const int grid = n > 256 * 4096 ? 256 : (n + 4095) / 4096;  // integer sums: the order does not matter
  hipLaunchKernelGGL((sum_counters_kernel<false>), dim3(grid), dim3(1024), 0, st, ev, zsum, chain0, n, out, 0);
  return hipGetLastError();
}
hipError_t launch_set_counters(const uint64_t* ev, const uint64_t* zsum, int chain0, int n, unsigned long long* out,
                               int n_zero, hipStream_t st) {
  hipLaunchKernelGGL((sum_counters_kernel<true>), dim3(1), dim3(1024), 0, st, ev, zsum, chain0, n, out, n_zero);
  return hipGetLastError();
}

hipError_t launch_split_geoms(const int* src, int n, const ChainArrays& ch, const EnsParams* ens, int* lists, int cap,
                              int* counts, int margin_div, int lane_cap, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(split_geoms_kernel, dim3((n + 1023) / 1024), dim3(1024), 0, st, src, n, ch, ens, lists, cap,
                     counts, margin_div, lane_cap);
  return hipGetLastError();
}

hipError_t launch_init_counts(int* cnt, int n, int n0, hipStream_t st) {
  hipLaunchKernelGGL(init_counts_kernel, dim3((n + 255) / 256), dim3(256), 0, st, cnt, n, n0);
  return hipGetLastError();
}

hipError_t launch_z_order_block(const int* src, int first, int n, const int* Z, const int* stall, int width, int* cnt,
                                int n_cnt, int n0, int* dst, int* n_out, hipStream_t st) {
  hipLaunchKernelGGL(zorder_block_kernel, dim3(1), dim3(1024), 0, st, src, first, n, Z, stall, width, cnt, n_cnt, n0,
                     dst, n_out);
  return hipGetLastError();
}

hipError_t launch_z_order(const int* src, int first, int n, const int* Z, const int* stall, int width, int* scratch,
                          int* dst, int* n_out, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const int blocks = n > 64 * 1024 * 4 ? 256 : (n + 4095) / 4096 + 1;  // a few elements per thread
  hipLaunchKernelGGL(zhist_kernel, dim3(blocks), dim3(1024), 0, st, src, first, n, Z, stall, width, scratch);
  hipLaunchKernelGGL(zscan_kernel, dim3(1), dim3(64), 0, st, scratch, n_out);
  hipLaunchKernelGGL(zscatter_kernel, dim3(blocks), dim3(1024), 0, st, src, first, n, Z, stall, width, scratch, dst);
  return hipGetLastError();
}

hipError_t launch_iota(int* p, int start, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(iota_kernel, dim3((n + 255) / 256), dim3(256), 0, st, p, start, n);
  return hipGetLastError();
}

int flow_reduce_parts(int nch) {
  const int parts = (nch + 1023) / 1024;
  return parts < 1 ? 1 : parts > 64 ? 64 : parts;
}
hipError_t launch_flow_reduce(const float* stage, int nch, int nrows, double* part, double* out, hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  const int parts = flow_reduce_parts(nch);
  hipLaunchKernelGGL(flow_reduce_kernel, dim3(nrows, parts), dim3(256), 0, st, stage, nch, parts > 1 ? part : out);
  if (parts > 1)
    hipLaunchKernelGGL(flow_parts_kernel, dim3((nrows * 9 + 255) / 256), dim3(256), 0, st, part, parts, nrows, out);
  return hipGetLastError();
}

hipError_t launch_corr_update(const float* stage, double* D, double* A, double* C, const int* stall, int chain0,
                              int nch, int p, int m, int s, int nrows, const int* cnt, int type, hipStream_t st) {
  if (nrows <= 0 || nch <= 0) return hipSuccess;
  CorrArgs a{stage, D, A, C, stall, chain0, nch, p, m, s, nrows, cnt, type};
  // 16 chains a block: 128-byte rows of the [...][chain] arrays.  An ensemble of few chains
  // takes four, so that its blocks are not all on a few CUs.
  const int chunk = nrows < 64 ? nrows : 64, lt = p < 16 ? (p < 4 ? 4 : p) : 16;
  const size_t per_chain = sizeof(double) * 3 * (size_t)(p + chunk + chunk / m + 1);
  const int ch = nch <= 4096 || 16 * per_chain > 64 * 1024 ? 4 : 16;
  const size_t lds = per_chain * ch;
  if (lds <= 64 * 1024) {
    const dim3 grid((nch + ch - 1) / ch), block(ch * lt);
    if (ch == 4) hipLaunchKernelGGL(corr_update_kernel<4>, grid, block, lds, st, a, chunk);
    else hipLaunchKernelGGL(corr_update_kernel<16>, grid, block, lds, st, a, chunk);
  } else {
    hipLaunchKernelGGL(corr_update_serial_kernel, dim3((nch + 255) / 256), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

int corr_reduce_parts(int count) {
  const int parts = (count + 4095) / 4096;
  return parts < 1 ? 1 : parts > 64 ? 64 : parts;
}
hipError_t launch_corr_reduce(const double* C, int ld, const int* stall, int chain0, int first, int count, int p, int m,
                              int s, const int64_t* nins, double* part, double* out, hipStream_t st) {
  CorrPoints P{};
  P.p = p;
  P.m = m;
  P.s = s;
  for (int k = 0; k < s && k < 40; ++k) P.nins[k] = (int)(nins[k] < p ? nins[k] : p);
  const int parts = corr_reduce_parts(count), npts = s * p;
  hipLaunchKernelGGL(corr_reduce_kernel, dim3(npts + 1, parts), dim3(256), 0, st, C, ld, stall, chain0, first, count, P,
                     parts > 1 ? part : out);
  if (parts > 1)
    hipLaunchKernelGGL(corr_parts_kernel, dim3((npts + 256) / 256), dim3(256), 0, st, part, parts, npts + 1, out);
  return hipGetLastError();
}

hipError_t launch_stage_window(const WinParam* wp, int n_ens, EnsParams* P, const int* cnt_src, int* cnt_dst,
                               int n_cnt, hipStream_t st) {
  hipLaunchKernelGGL(stage_window_kernel, dim3(1), dim3(256), 0, st, wp, n_ens, P, cnt_src, cnt_dst, n_cnt);
  return hipGetLastError();
}

hipError_t launch_stage_args(const WinArgs& w, EnsParams* P, int* cnt_dst, hipStream_t st) {
  hipLaunchKernelGGL(stage_args_kernel, dim3(1), dim3(256), 0, st, w, P, cnt_dst);
  return hipGetLastError();
}

hipError_t launch_chain_stress(const ChainArrays& ch, int chain0, int n, const float kappa[9], double* part,
                               hipStream_t st) {
  KappaArg K;
  for (int i = 0; i < 9; ++i) K.k[i] = kappa[i];
  hipLaunchKernelGGL(chain_stress_kernel, dim3(kStressBlocks), dim3(64 * kStressWaves), 0, st, ch, chain0, n, K, part);
  return hipGetLastError();
}

hipError_t launch_check_state(const ChainArrays& ch, int chain0, int n, double t_min, unsigned long long* out,
                              hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const int grid = std::min(2048, (n + 3) / 4);
  hipLaunchKernelGGL(check_state_kernel, dim3(grid), dim3(256), 0, st, ch, chain0, n, t_min, out);
  return hipGetLastError();
}

hipError_t launch_copy_probe(const void* in, void* out, size_t n4, int grid, hipStream_t st) {
  hipLaunchKernelGGL(copy_probe_kernel, dim3(grid), dim3(256), 0, st, (const float4*)in, (float4*)out, n4);
  return hipGetLastError();
}
hipError_t launch_scan_probe(const float* in, float* out, int n, int form, hipStream_t st) {
  hipLaunchKernelGGL(scan_probe_kernel, dim3(1), dim3(64), 0, st, in, out, n, form);
  return hipGetLastError();
}
hipError_t launch_com_probe(const float* in, float* out, int n, int geom, hipStream_t st) {
  hipLaunchKernelGGL(com_probe_kernel, dim3(1), dim3(64), 0, st, in, out, n, geom);
  return hipGetLastError();
}
hipError_t launch_math_probe(const float* in, float* out, int n, int which, hipStream_t st) {
  hipLaunchKernelGGL(math_probe_kernel, dim3((n + 255) / 256), dim3(256), 0, st, in, out, n, which);
  return hipGetLastError();
}
hipError_t launch_philox_probe(const uint32_t* ck, uint32_t* out, int n, hipStream_t st) {
  hipLaunchKernelGGL(philox_probe_kernel, dim3((n + 255) / 256), dim3(256), 0, st, ck, out, n);
  return hipGetLastError();
}

}  // namespace dsm
