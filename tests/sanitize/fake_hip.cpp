// fake_hip.cpp -- a host-only stand-in for the HIP runtime calls and kernel launchers that
// the engine (dsm_engine.cpp) uses, so that its host code -- allocation, routes, launch
// shapes -- can be built with g++ and run under AddressSanitizer on a machine without a GPU.
// Test infrastructure only.  "Device" memory is host memory: a launcher touches the ends of
// every range that its kernel would use, so a range too small shows; a null pointer among
// them is counted.  The jump kernels record their launch and move no chain.
#include "fake_hip.h"

#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>

#include "dsm_launch.h"

namespace fake {
std::vector<Launch> launches;
int nulls = 0;
int64_t allocs = 0, fail_from = 0, fail_to = 0, live_bytes = 0, live_count = 0, pinned = 0;
size_t capacity = (size_t)1 << 33;
static std::map<void*, size_t> sizes;
static int handle;

template <typename T>
bool use(T* p, int64_t n) {  // the first and the last element
  if (n <= 0) return true;
  if (!p) { ++nulls; return false; }
  volatile char* c = (volatile char*)p;
  char x = c[0];
  c[0] = x;
  x = c[(size_t)n * sizeof(T) - 1];
  c[(size_t)n * sizeof(T) - 1] = x;
  return true;
}
template <typename T>
T* any() { return (T*)&handle; }
}  // namespace fake
using namespace fake;

extern "C" {
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "out of memory"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  ++allocs;
  *p = nullptr;
  if ((allocs >= fail_from && allocs <= fail_to) || (size_t)live_bytes + n > capacity) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  sizes[*p] = n;
  live_bytes += (int64_t)n;
  ++live_count;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  live_bytes -= (int64_t)sizes.at(p);
  --live_count;
  sizes.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { ++pinned; *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *t = capacity;
  *f = capacity > (size_t)live_bytes ? capacity - (size_t)live_bytes : 0;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  if (n && (!d || !s)) { ++nulls; return hipErrorInvalidValue; }
  if (n) std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n) {
  if (n && !d) { ++nulls; return hipErrorInvalidValue; }
  if (n) std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = any<std::remove_pointer_t<hipStream_t>>(); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = any<std::remove_pointer_t<hipGraph_t>>(); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *x = any<std::remove_pointer_t<hipGraphExec_t>>();
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = any<std::remove_pointer_t<hipEvent_t>>(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
}  // extern "C"

namespace dsm {

static void chains(const ChainArrays& c, int first, int n) {
  use(c.Z + first, n); use(c.nk + first, n); use(c.ens + first, n); use(c.cap + first, n); use(c.stall + first, n);
  use(c.cid + first, n); use(c.local + first, n); use(c.base + first, n); use(c.t + first, n); use(c.ev + first, n);
  use(c.dt_prev + first, n); use(c.next_sample + first, n); use(c.ev_stop + first, n); use(c.zsum + first, n);
  use(c.R1 + 3 * (int64_t)first, 3 * (int64_t)n);
}
// what every jump kernel uses; the chains' numbers and ensembles are looked up from the list
static void jumps(const KmcArgs& a, Launch l) {
  launches.push_back(l);
  chains(a.ch, 0, 1);
  const bool ok = use(a.n_work, 1) & use(a.queue, 1) & use(a.n_overflow, 1) & use(a.work, 1) & use(a.overflow, 1) &
                  use(a.ens, 1) & use(a.tabs, 1);
  if (!ok) return;
  for (int i = 0; i < *a.n_work; ++i) {
    const int c = a.work[i];
    if (c < 0) continue;
    use(a.ch.Z + c, 1);
    const EnsParams* P = a.ens + a.ch.ens[c];
    use(P, 1);
    use(a.tabs + P->tab_off, (int64_t)kNumTables * (P->nmax + 2) + 4 * P->nmax + 4);
    if (P->partner) use(a.tabs + P->pd_off, (int64_t)12 * kPartnerK);
    const int64_t b = a.ch.base[c], n = a.ch.cap[c];
    use(a.ch.Qx + b, n); use(a.ch.Qy + b, n); use(a.ch.Qz + b, n); use(a.ch.N + b, n); use(a.ch.w + b, n);
    if (l.name == "lane") use(a.rec + kLaneRecFloats * b, kLaneRecFloats * n);
    if (P->sample_mode != kSampleNone && P->k_end > P->k0)
      use(a.stage + P->stage_off, (P->k_end - P->k0) * P->nchains * (P->sample_mode == kSampleFlow ? 8 : 3));
  }
  if (l.name.rfind("lane", 0) == 0 || l.name.rfind("solo", 0) == 0) use(a.lane_tab, kLaneTabFloats);
}

hipError_t launch_kmc(const KmcArgs& a, int geom, bool plain, int grid, hipStream_t) {
  jumps(a, Launch{geom == 0 ? "row" : geom == 1 ? "pair" : geom == kGeomPair2 ? "pair2" : "wave", geom, grid, 0, plain, false});
  return hipSuccess;
}
int kmc_max_blocks_per_cu(int, bool, int, bool) { return 8; }
hipError_t launch_kmc_rowpair(const KmcArgs& row, const KmcArgs& pair, bool row2, int grid, hipStream_t) {
  jumps(row, Launch{"rowpair", 0, grid, 0, false, row2});
  jumps(pair, Launch{"rowpair", 1, grid, 0, false, row2});
  return hipSuccess;
}
int kmc_rowpair_occupancy(int, bool, bool) { return 8; }
hipError_t launch_kmc_lane(const KmcArgs& a, int quads, int grid, hipStream_t) {
  jumps(a, Launch{"lane", 4 * quads, grid, a.lanes, false, false});
  return a.lanes >= 1 && a.lanes <= lane_max_lanes(quads) ? hipSuccess : hipErrorInvalidValue;
}
hipError_t launch_kmc_lane_flow(const KmcArgs& a, int cap, int grid, hipStream_t) {
  jumps(a, Launch{"lane_flow", cap, grid, a.lanes, false, false});
  return a.lanes >= 1 && a.lanes <= flow_max_lanes(cap) ? hipSuccess : hipErrorInvalidValue;
}
int kmc_solo_occupancy(int) { return 16; }
hipError_t launch_kmc_solo(const KmcArgs& a, int cap, int grid, hipStream_t) {
  jumps(a, Launch{"solo", cap, grid, 0, false, false});
  return hipSuccess;
}
int kmc_solo_flow_occupancy(int) { return 8; }
hipError_t launch_kmc_solo_flow(const KmcArgs& a, int cap, int grid, hipStream_t) {
  jumps(a, Launch{"solo_flow", cap, grid, 0, false, false});
  return hipSuccess;
}
hipError_t launch_init_eq(const ChainArrays& ch, const EnsParams* ens, const float* tabs, int first, int n, int lanes,
                          hipStream_t) {
  if (lanes != 4 && lanes != 16) return hipErrorInvalidValue;
  chains(ch, first, n);
  for (int c = first; c < first + n; ++c) {
    const EnsParams* P = ens + ch.ens[c];
    if (!use(P, 1) || !use(tabs + P->tab_off, (int64_t)kNumTables * (P->nmax + 2) + 4 * P->nmax + 4)) return hipSuccess;
    if (P->partner) use(tabs + P->pd_off, (int64_t)12 * kPartnerK);
    const int64_t b = ch.base[c];
    use(ch.Qx + b, ch.cap[c]); use(ch.Qy + b, ch.cap[c]); use(ch.Qz + b, ch.cap[c]); use(ch.w + b, ch.cap[c]);
    ch.N[b] = ch.nk[c];
    ch.Z[c] = 1;
    ch.t[c] = 0.0;
    ch.stall[c] = 0;
  }
  return hipSuccess;
}
hipError_t launch_fill_u32(void* p, uint32_t v, int64_t n, hipStream_t) {
  if (use((uint32_t*)p, n)) for (int64_t i = 0; i < n; ++i) ((uint32_t*)p)[i] = v;
  return hipSuccess;
}
hipError_t launch_iota(int* p, int start, int n, hipStream_t) {
  if (use(p, n)) for (int i = 0; i < n; ++i) p[i] = start + i;
  return hipSuccess;
}
hipError_t launch_init_counts(int* cnt, int n, int n0, hipStream_t) {
  if (use(cnt, n)) for (int i = 0; i < n; ++i) cnt[i] = i ? 0 : n0;
  return hipSuccess;
}
hipError_t launch_z_order(const int* src, int first, int n, const int* Z, const int* stall, int, int* scratch, int* dst,
                          int* n_out, hipStream_t) {
  use(scratch, kZOrderScratch);
  int k = 0;
  if (!use(n_out, 1) || !use(dst, 1)) return hipSuccess;
  for (int i = 0; i < n; ++i) {
    const int c = src ? src[i] : first + i;
    if (c < 0) continue;
    use(Z + c, 1); use(stall + c, 1);
    dst[k++] = c;
  }
  *n_out = k;
  return hipSuccess;
}
hipError_t launch_z_order_block(const int* src, int first, int n, const int* Z, const int* stall, int width, int* cnt,
                                int n_cnt, int n0, int* dst, int* n_out, hipStream_t st) {
  launch_init_counts(cnt, n_cnt, n0, st);
  return launch_z_order(src, first, n, Z, stall, width, cnt, dst, n_out, st);
}
hipError_t launch_split_geoms(const int* src, int n, const ChainArrays& ch, const EnsParams* ens, int* lists, int cap,
                              int* counts, int, int lane_cap, hipStream_t) {
  if (!use(counts, kNumGeoms) || !use(lists, (int64_t)kNumGeoms * cap)) return hipSuccess;
  for (int i = 0; i < n; ++i) {
    if (src[i] < 0) continue;
    use(ens + ch.ens[src[i]], 1);
    const int b = lane_cap ? 0 : src[i] % kNumGeoms;
    lists[(int64_t)b * cap + counts[b]++] = src[i];
  }
  return hipSuccess;
}
hipError_t launch_sum_counters(const uint64_t* ev, const uint64_t* zsum, int chain0, int n, unsigned long long* out,
                               hipStream_t) {
  use(ev + chain0, n); use(zsum + chain0, n); use(out, 2);
  return hipSuccess;
}
hipError_t launch_set_counters(const uint64_t* ev, const uint64_t* zsum, int chain0, int n, unsigned long long* out,
                               int n_zero, hipStream_t st) {
  for (int i = 0; i < n_zero; ++i) out[i] = 0;
  return launch_sum_counters(ev, zsum, chain0, n, out, st);
}
hipError_t launch_set_ev_stop(const uint64_t* ev, uint64_t* ev_stop, int chain0, int n, uint64_t, hipStream_t) {
  use(ev + chain0, n); use(ev_stop + chain0, n);
  return hipSuccess;
}
int flow_reduce_parts(int nch) {
  const int parts = (nch + 1023) / 1024;
  return parts < 1 ? 1 : parts > 64 ? 64 : parts;
}
hipError_t launch_flow_reduce(const float* stage, int nch, int nrows, double* part, double* out, hipStream_t) {
  use(stage, (int64_t)nrows * nch * 8); use(part, (int64_t)nrows * flow_reduce_parts(nch) * 9);
  if (use(out, (int64_t)nrows * 9)) std::memset(out, 0, sizeof(double) * 9 * (size_t)nrows);
  return hipSuccess;
}
hipError_t launch_corr_update(const float* stage, double* D, double* A, double* C, const int* stall, int chain0, int nch,
                              int p, int, int s, int nrows, const int* cnt, int, hipStream_t) {
  use(stage, (int64_t)nrows * nch * 3); use(D, (int64_t)s * p * 3 * nch); use(A, (int64_t)s * 3 * nch);
  use(C, (int64_t)s * p * nch); use(stall + chain0, nch); use(cnt, 3 * s);
  return hipSuccess;
}
int corr_reduce_parts(int count) {
  const int parts = (count + 4095) / 4096;
  return parts < 1 ? 1 : parts > 64 ? 64 : parts;
}
hipError_t launch_corr_reduce(const double* C, int ld, const int* stall, int chain0, int first, int count, int p, int,
                              int s, const int64_t* nins, double* part, double* out, hipStream_t) {
  use(C, (int64_t)s * p * ld); use(stall + chain0 + first, count); use(nins, s);
  use(part, ((int64_t)s * p + 1) * corr_reduce_parts(count));
  if (use(out, (int64_t)s * p + 1)) std::memset(out, 0, sizeof(double) * ((size_t)s * p + 1));
  return hipSuccess;
}
hipError_t launch_chain_stress(const ChainArrays& ch, int chain0, int n, const float*, double* part, hipStream_t) {
  chains(ch, chain0, n);
  if (use(part, kStressBlocks * 9)) std::memset(part, 0, sizeof(double) * 9 * kStressBlocks);
  return hipSuccess;
}
hipError_t launch_check_state(const ChainArrays& ch, int chain0, int n, double, unsigned long long* out, hipStream_t) {
  chains(ch, chain0, n);
  use(out, 7);
  return hipSuccess;
}
hipError_t launch_stage_window(const WinParam* wp, int n_ens, EnsParams* P, const int* cnt_src, int* cnt_dst, int n_cnt,
                               hipStream_t) {
  for (int i = 0; i < n_ens; ++i) {
    if (!use(P + wp[i].ens, 1) || !P) return hipSuccess;
    P[wp[i].ens].t_end = wp[i].t_end;
    P[wp[i].ens].k0 = wp[i].k0;
    P[wp[i].ens].k_end = wp[i].k_end;
  }
  if (use(cnt_dst, n_cnt)) for (int i = 0; i < n_cnt; ++i) cnt_dst[i] = cnt_src[i];
  return hipSuccess;
}
hipError_t launch_stage_args(const WinArgs& w, EnsParams* P, int* cnt_dst, hipStream_t st) {
  return launch_stage_window(w.win, w.n_ens, P, w.cnt, cnt_dst, w.n_cnt, st);
}
hipError_t launch_copy_probe(const void*, void*, size_t, int, hipStream_t) { return hipSuccess; }
hipError_t launch_scan_probe(const float*, float*, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_com_probe(const float*, float*, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_math_probe(const float*, float*, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_philox_probe(const uint32_t*, uint32_t*, int, hipStream_t) { return hipSuccess; }

}  // namespace dsm
