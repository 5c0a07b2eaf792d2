// engine_checks.cpp -- drives the engine's host code over the host-only HIP stand-in.
// Usage: engine_checks <check>; exit code 0 when every check passes.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "dsm.h"
#include "fake_hip.h"

static int failures = 0;
#define CHECK(c)                                                           \
  do {                                                                     \
    if (!(c)) {                                                            \
      std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
      ++failures;                                                          \
    }                                                                      \
  } while (0)

static dsm_ensemble_desc desc(int n, int nk, int sample, float beta = 1.0f) {
  dsm_ensemble_desc d{};
  d.n_chains = n;
  d.nk = nk;
  d.beta = beta;
  d.cd = 1;
  d.seed = 1;
  d.sample_mode = sample;
  d.delta = 1.0;
  d.corr_p = 16;
  d.corr_m = 2;
  d.corr_levels = 3;
  d.window = 4;
  if (sample == DSM_SAMPLE_FLOW) d.kappa[1] = 0.01f;
  return d;
}

// ------------------------------------------------------------------ failed allocations
// The calls of a session, in order; each may fail for want of memory and is then repeated.
struct Session {
  dsm_engine* e = nullptr;
  int32_t id[4] = {-1, -1, -1, -1};
  std::vector<std::function<int()>> calls;
  Session() {
    auto add = [this](int k, int n, int nk, int sample, int partner = 0, int levels = 3) {
      calls.push_back([=] {
        dsm_ensemble_desc d = desc(n, nk, sample);
        d.corr_levels = levels;
        d.partner_mode = partner;
        return dsm_add_ensemble(e, &d, &id[k]);
      });
      calls.push_back([=] { return dsm_init_equilibrium(e, id[k]); });
    };
    auto run = [this](int k, double t) {
      calls.push_back([=] { return dsm_advance(e, id[k], t, DSM_MODE_BATCHED, nullptr, nullptr, nullptr); });
    };
    calls.push_back([this] { return dsm_create(0, &e); });
    add(0, 40, 30, DSM_SAMPLE_GT);
    run(0, 6.0);
    calls.push_back([this] {
      double lag[80], g[80];
      int32_t np = 0;
      return dsm_correlator(e, id[0], 80, lag, g, &np);
    });
    add(1, 3000, 20, DSM_SAMPLE_FLOW);
    run(1, 5.0);
    run(0, 9.0);
    add(2, 500, 300, DSM_SAMPLE_MSD, DSM_PARTNER_MELT, 9);
    calls.push_back([this] {
      const double t[3] = {12.0, 8.0, 6.0};
      return dsm_advance_many(e, id, t, 3, DSM_MODE_BATCHED, nullptr, nullptr);
    });
    calls.push_back([this] { return dsm_remove_ensemble(e, id[1]); });
    add(3, 5000, 60, DSM_SAMPLE_GT);
    run(3, 6.0);
    run(0, 20.0);
    calls.push_back([this] { return dsm_advance_events(e, id[2], 5, DSM_MODE_BATCHED, nullptr); });
    calls.push_back([this] { return dsm_advance_events(e, id[2], 2, DSM_MODE_PLAIN, nullptr); });
  }
  ~Session() { dsm_destroy(e); }
};

// What can run on the ensembles there are, while nothing can be allocated: it may be
// refused, but uses no pointer that a failed call left behind.
static void others(Session& s) {
  if (!s.e) return;
  for (int32_t id : s.id) {
    if (id < 0) continue;
    const int rc = dsm_advance(s.e, id, 2.0, DSM_MODE_BATCHED, nullptr, nullptr, nullptr);
    CHECK(rc == DSM_OK || rc == DSM_ERR_MEMORY || rc == DSM_ERR_ARG);  // (ARG: removed)
  }
}

static void check_alloc() {
  int64_t total = 0, bytes = 0;
  {
    Session s;
    const int64_t a0 = fake::allocs;
    for (auto& c : s.calls) CHECK(c() == DSM_OK);
    total = fake::allocs - a0;
    bytes = fake::live_bytes;
  }
  CHECK(fake::live_bytes == 0 && total > 60);
  // n failures in a row: one, or all until the call has been refused
  for (int64_t n : {(int64_t)1, (int64_t)1 << 40}) {
    for (int64_t k = 1; k <= total; ++k) {
      Session s;
      fake::nulls = 0;
      fake::fail_next(k, n);
      int refused = 0;
      for (auto& c : s.calls) {
        int rc = c();
        if (rc == DSM_ERR_MEMORY) {
          ++refused;
          others(s);
          fake::fail_none();
          others(s);
          rc = c();
        }
        CHECK(rc == DSM_OK);
      }
      fake::fail_none();
      CHECK(refused <= 1);
      if (fake::nulls) std::fprintf(stderr, "allocation %lld of %lld (%s)\n", (long long)k, (long long)total, n > 1 ? "all" : "one");
      CHECK(fake::nulls == 0);
      // a refused call leaves nothing behind (what stays allocated may have grown in other steps)
      CHECK(fake::live_bytes <= bytes + bytes / 4);
      if (failures > 20) return;
    }
  }
  CHECK(fake::live_bytes == 0);
}

// ------------------------------------------------------------------ the lane form's records give way
// With the records in memory, no single failed allocation is the caller's: they are given
// back for it, and the next pass takes them again or runs without.
static int64_t lanes_session(int64_t k, bool* ran) {
  dsm_engine* e = nullptr;
  CHECK(dsm_create(0, &e) == DSM_OK);
  CHECK(dsm_set_option(e, DSM_OPT_LANE, 2) == DSM_OK && dsm_set_option(e, DSM_OPT_SMALL_PER_CU, 0) == DSM_OK);
  int32_t id = -1, fl = -1, more = -1;
  dsm_ensemble_desc d = desc(100, 30, DSM_SAMPLE_GT), f = desc(5000, 40, DSM_SAMPLE_FLOW), x = desc(700, 50, DSM_SAMPLE_MSD);
  x.partner_mode = DSM_PARTNER_MELT;
  CHECK(dsm_add_ensemble(e, &d, &id) == DSM_OK && dsm_init_equilibrium(e, id) == DSM_OK);
  auto run = [&](int32_t i, double t) { CHECK(dsm_advance(e, i, t, DSM_MODE_BATCHED, nullptr, nullptr, nullptr) == DSM_OK); };
  fake::launches.clear();
  fake::nulls = 0;
  run(id, 3.0);
  *ran = fake::launches[0].name == "lane";
  const int64_t a0 = fake::allocs;
  if (k > 0) fake::fail_next(k);
  double lag[80], g[80];
  int32_t np = 0;
  CHECK(dsm_correlator(e, id, 80, lag, g, &np) == DSM_OK);
  CHECK(dsm_add_ensemble(e, &f, &fl) == DSM_OK && dsm_init_equilibrium(e, fl) == DSM_OK);
  run(fl, 6.0);
  CHECK(dsm_add_ensemble(e, &x, &more) == DSM_OK && dsm_init_equilibrium(e, more) == DSM_OK);
  run(more, 6.0);
  for (int i = 0; i < 16; ++i) {
    int32_t j = -1;
    d.salt = (uint32_t)i + 1;
    CHECK(dsm_add_ensemble(e, &d, &j) == DSM_OK && dsm_init_equilibrium(e, j) == DSM_OK);
    run(j, 3.0);
  }
  fake::fail_none();
  fake::launches.clear();
  run(id, 9.0);
  CHECK(fake::launches[0].name == "lane" && fake::nulls == 0);
  const int64_t n = fake::allocs - a0;
  dsm_destroy(e);
  CHECK(fake::live_bytes == 0);
  return n;
}
static void check_lanes() {
  bool ran = false;
  const int64_t n = lanes_session(0, &ran);
  CHECK(ran && n > 40);
  for (int64_t k = 1; k <= n && failures < 20; ++k) lanes_session(k, &ran);
  int without = 0;
  for (int64_t k = 1; k <= 6; ++k) {
    dsm_engine* e = nullptr;
    CHECK(dsm_create(0, &e) == DSM_OK);
    dsm_set_option(e, DSM_OPT_LANE, 2);
    dsm_set_option(e, DSM_OPT_SMALL_PER_CU, 0);
    int32_t id = -1;
    dsm_ensemble_desc d = desc(100, 30, DSM_SAMPLE_NONE);
    CHECK(dsm_add_ensemble(e, &d, &id) == DSM_OK && dsm_init_equilibrium(e, id) == DSM_OK);
    fake::launches.clear();
    fake::fail_next(k);
    CHECK(dsm_advance(e, id, 3.0, DSM_MODE_BATCHED, nullptr, nullptr, nullptr) == DSM_OK);
    without += fake::launches[0].name != "lane";
    fake::fail_none();
    dsm_destroy(e);
  }
  CHECK(without == 2);  // the tables or the records: the other forms run
}

// ------------------------------------------------------------------ options
struct Run {  // one pass of `n` chains a piece of the ensembles given, the options set
  std::vector<fake::Launch> l;
  Run(const std::vector<dsm_ensemble_desc>& ds, const std::vector<std::pair<int, int>>& opts, double t = 3.0) {
    dsm_engine* e = nullptr;
    CHECK(dsm_create(0, &e) == DSM_OK);
    for (auto& o : opts) CHECK(dsm_set_option(e, o.first, o.second) == DSM_OK);
    std::vector<int32_t> ids;
    for (auto& d : ds) {
      int32_t id = -1;
      CHECK(dsm_add_ensemble(e, &d, &id) == DSM_OK && dsm_init_equilibrium(e, id) == DSM_OK);
      ids.push_back(id);
    }
    fake::launches.clear();
    fake::nulls = 0;
    const std::vector<double> te(ids.size(), t);
    CHECK(dsm_advance_many(e, ids.data(), te.data(), (int32_t)ids.size(), DSM_MODE_BATCHED, nullptr, nullptr) == DSM_OK);
    CHECK(fake::nulls == 0 && !fake::launches.empty());
    l = fake::launches;
    dsm_destroy(e);
  }
  bool has(const char* name) const {
    for (auto& x : l)
      if (x.name == name) return true;
    return false;
  }
  const std::string& first() const { return l[0].name; }
};

static const int kCu = 256;

static void check_waves() {
  // DSM_OPT_BLOCKS_PER_CU bounds the waves of every form
  const std::vector<std::vector<dsm_ensemble_desc>> passes = {
      {desc(40000, 60, DSM_SAMPLE_GT)},                                   // lanes, then solo
      {desc(40000, 60, DSM_SAMPLE_FLOW)},                                 // row
      {desc(70000, 25, DSM_SAMPLE_FLOW)},                                 // lanes under flow
      {desc(2000, 100, DSM_SAMPLE_GT)},                                   // solo
      {desc(2000, 100, DSM_SAMPLE_FLOW)},                                 // solo under flow
      {desc(3500, 700, DSM_SAMPLE_GT)},                                   // concurrent
      {desc(3500, 700, DSM_SAMPLE_GT), desc(3500, 600, DSM_SAMPLE_FLOW)}  // concurrent with flow
  };
  std::string seen;
  for (auto& ds : passes)
    for (int cap : {1, 2, 3, 8, 12, 100}) {
      const Run r(ds, {{DSM_OPT_BLOCKS_PER_CU, cap}, {DSM_OPT_LANE, 2}});
      for (auto& x : r.l) {
        const int per = x.name.rfind("lane", 0) == 0 ? 8 : 1;
        if (x.grid * per > cap * kCu) std::fprintf(stderr, "%s %d: %d waves\n", x.name.c_str(), x.size, x.grid * per);
        CHECK(x.grid >= 1 && x.grid * per <= cap * kCu);
        seen += " " + x.name;
      }
    }
  for (const char* f : {"lane", "lane_flow", "solo", "solo_flow", "rowpair", "wave"}) CHECK(seen.find(f) != std::string::npos);
}

static void check_concurrent() {
  // DSM_OPT_CONCURRENT = 1: side by side wherever a chain can leave the row form, the short
  // ones in lanes first; 0: never
  for (int lane : {0, 1, 2}) {
    const std::vector<std::pair<int, int>> always = {{DSM_OPT_CONCURRENT, 1}, {DSM_OPT_LANE, lane}};
    const Run still({desc(50000, 100, DSM_SAMPLE_GT)}, always), flow({desc(20000, 70, DSM_SAMPLE_FLOW, 3.0f)}, always);
    CHECK(still.has("rowpair") && flow.has("rowpair"));
    CHECK(still.has("lane") == (lane > 0) && !flow.has("lane_flow"));
    const Run in_turn({desc(50000, 700, DSM_SAMPLE_GT)}, {{DSM_OPT_CONCURRENT, 0}, {DSM_OPT_LANE, lane}});
    CHECK(!in_turn.has("rowpair"));
  }
  const Run by_itself({desc(50000, 100, DSM_SAMPLE_GT)}, {});
  CHECK(by_itself.first() == "lane" && !by_itself.has("rowpair"));
}

// ------------------------------------------------------------------ routes
static dsm_ensemble_desc every(dsm_ensemble_desc d, double delta) {
  d.delta = delta;
  return d;
}
// Which form takes the chains of a pass; the times beside a case are its former route's and
// the lane form's, in ms.
static void check_lane_route() {
  const int GT = DSM_SAMPLE_GT, MSD = DSM_SAMPLE_MSD, NONE = DSM_SAMPLE_NONE;
  auto lanes = [](const std::vector<dsm_ensemble_desc>& ds) { return Run(ds, {}, 0.01).has("lane"); };
  CHECK(lanes({desc(131072, 100, GT)}));                  // 9.1 / 5.2
  CHECK(lanes({desc(131072, 100, MSD)}));                 // 8.0 / 4.8
  CHECK(lanes({desc(50021, 150, GT)}));                   // 5.7 / 2.7
  CHECK(lanes({desc(262144, 12, GT)}));                   // 16.5 / 10.2
  CHECK(lanes({desc(40000, 50, GT)}));                    // 1.07 times as fast
  CHECK(lanes({desc(131072, 100, NONE, 6.0f)}));
  CHECK(lanes({desc(70000, 100, GT), desc(70000, 60, GT)}));
  // a sample costs the lane form several times what it costs the others
  CHECK(!lanes({every(desc(131072, 100, GT), 0.03)}));    // 15.2 / 26.4
  CHECK(!lanes({every(desc(131072, 100, MSD), 0.1)}));    // 12.1 / 20.5
  CHECK(!lanes({every(desc(40000, 60, GT), 0.1)}));       // 12.8 / 15.7
  CHECK(!lanes({desc(131072, 100, GT, 30.0f)}));          // 2.3 / 4.0 (0.4 jumps a sample)
  // long strands
  CHECK(!lanes({desc(40000, 1000, GT, 30.0f)}));          // 2.7 / 5.2
  CHECK(!lanes({desc(40000, 60, GT, 6.0f)}));             // 2.4 / 3.4
  CHECK(!lanes({desc(40000, 60, GT, 12.0f)}));            // 1.4 / 2.4
  // of several ensembles, each counts by its own price
  CHECK(!lanes({desc(20000, 100, GT), desc(100000, 100, GT, 30.0f)}));
}
static void check_share_route() {
  // mixed lengths, the shorter chains in lanes first where they are many
  auto mixed = [](int n, int sample, float beta, double delta) {
    std::vector<int32_t> nk((size_t)n);
    for (int i = 0; i < n; ++i) nk[(size_t)i] = i % 50 == 0 ? 900 : 30 + i % 170;
    dsm_ensemble_desc d = every(desc(n, 900, sample, beta), delta);
    d.nk_per_chain = nk.data();
    return Run({d}, {}, 0.01).has("lane");
  };
  CHECK(mixed(200000, DSM_SAMPLE_GT, 1.0f, 1.0));         // the polydisperse melt's kind: 12.5 / 10.6
  CHECK(!mixed(90000, DSM_SAMPLE_GT, 3.0f, 1.0));         // 4.8 / 6.0
  CHECK(!mixed(200000, DSM_SAMPLE_MSD, 8.0f, 0.3));       // 5.3 / 8.4
  CHECK(!mixed(200000, DSM_SAMPLE_GT, 20.0f, 1.0));       // 3.7 / 4.6
}

static void check_flow_route() {
  auto lanes = [](int n, int nk, int ens, float beta, double delta) {
    return Run(std::vector<dsm_ensemble_desc>((size_t)ens, every(desc(n, nk, DSM_SAMPLE_FLOW, beta), delta)), {}, 0.01)
        .has("lane_flow");
  };
  CHECK(lanes(16384, 50, 16, 1.0f, 1.0));    // row 15.1, lanes 10.6
  CHECK(lanes(65536, 25, 1, 1.0f, 1.0));     // 4.2 / 2.7
  CHECK(lanes(262144, 12, 1, 1.0f, 1.0));    // 6.5 / 1.8
  CHECK(lanes(2000, 25, 16, 1.0f, 1.0));     // 1.6 times as fast
  CHECK(lanes(16384, 50, 16, 6.0f, 1.0));    // 5.1 / 1.6
  CHECK(!lanes(20000, 40, 2, 0.3f, 1.0));    // 3.1 / 3.6
  CHECK(!lanes(10000, 25, 2, 1.0f, 1.0));    // 0.73 times
  CHECK(!lanes(10000, 40, 2, 5.0f, 1.0));    // 0.65
  CHECK(!lanes(30000, 25, 1, 3.0f, 1.0));    // 0.72
  CHECK(!lanes(65536, 60, 1, 8.0f, 1.0));    // 0.86
  CHECK(!lanes(65536, 100, 1, 25.0f, 1.0));  // 0.6
  CHECK(!lanes(30000, 12, 1, 1.0f, 0.2));    // 0.89
}

static void check_solo_route() {
  const int GT = DSM_SAMPLE_GT, MSD = DSM_SAMPLE_MSD;
  auto first = [](const dsm_ensemble_desc& d) { return Run({d}, {}, 0.01).first(); };
  CHECK(first(desc(64, 16, GT)) == "solo");                  // wave 0.48, solo 0.46
  CHECK(first(desc(1000, 25, GT)) == "solo");                // 0.71 / 0.68
  CHECK(first(desc(3000, 100, GT)) == "solo");               // 1.57 / 1.48
  CHECK(first(desc(1500, 100, GT, 12.0f)) == "solo");        // 0.98 / 0.66
  CHECK(first(every(desc(64, 100, GT), 0.1)) == "solo");     // 1.08 times as fast
  CHECK(first(desc(3000, 8, GT)) == "wave");                 // 0.83
  CHECK(first(desc(2500, 25, GT)) == "wave");                // 0.81 / 0.90
  CHECK(first(every(desc(3000, 30, GT), 0.1)) == "wave");    // 0.71
  CHECK(first(every(desc(1000, 30, GT), 0.1)) == "wave");    // 0.90
  CHECK(first(every(desc(3000, 100, GT), 0.1)) == "wave");   // 0.80
  CHECK(first(every(desc(3000, 30, MSD), 0.1)) == "wave");
  // several ensembles count together; longer chains keep the form however few jumps a sample
  CHECK(Run({desc(1500, 10, GT), desc(1500, 12, GT)}, {}, 0.01).first() == "wave");
  CHECK(Run({every(desc(1500, 1000, GT), 0.03)}, {}, 0.01).has("solo"));
}

static void check_solo_flow_route() {
  auto first = [](int n, int nk, float beta) { return Run({desc(n, nk, DSM_SAMPLE_FLOW, beta)}, {}, 0.01).first(); };
  CHECK(first(3001, 30, 1.0f) == "solo_flow");   // wave 0.94, solo 0.82
  CHECK(first(300, 100, 1.0f) == "solo_flow");   // 1.58 times as fast
  CHECK(first(64, 100, 8.0f) == "solo_flow");    // 1.23
  CHECK(first(300, 30, 20.0f) == "solo_flow");   // 1.30: no strand can be long
  CHECK(first(3000, 100, 30.0f) == "wave");      // 0.85
  CHECK(first(300, 200, 20.0f) == "wave");       // 0.43 / 0.48
  CHECK(first(3000, 200, 30.0f) == "wave");      // 0.78
}

static void check_bin2_route() {
  auto two = [](int n, int nk, float beta) {
    const Run r({desc(n, nk, DSM_SAMPLE_GT, beta)}, {{DSM_OPT_LANE, 0}}, 0.01);
    CHECK(r.has("rowpair"));
    return r.has("pair2");
  };
  CHECK(two(100000, 168, 0.4f));   // two chains a wave 8.6, one 9.7 ms
  CHECK(two(40000, 239, 1.0f));    // 0.98
  CHECK(!two(16000, 168, 0.4f));   // 1.08
  CHECK(!two(100000, 154, 0.4f));  // 1.02
  CHECK(!two(100000, 189, 0.4f));  // 1.5
  CHECK(!two(40000, 300, 1.0f));   // 1.13
  CHECK(!two(20000, 600, 1.0f));
}

// ------------------------------------------------------------------ window parameters
static void check_window() {
  // a window's parameters travel with its launch: no pinned memory but for many ensembles or a
  // captured window
  const auto d = desc(40, 30, DSM_SAMPLE_GT);
  fake::pinned = 0;
  for (int k : {1, 2, 16}) Run(std::vector<dsm_ensemble_desc>((size_t)k, d), {});
  dsm_ensemble_desc big = d;
  big.corr_levels = 40;
  Run({big, big}, {});
  CHECK(fake::pinned == 0);
  Run(std::vector<dsm_ensemble_desc>(17, d), {});
  CHECK(fake::pinned == 1);
  Run({big, big, big}, {});
  CHECK(fake::pinned == 2);
  Run({d}, {{DSM_OPT_GRAPH, 1}}, 9.0);
  CHECK(fake::pinned == 3);
}

// ------------------------------------------------------------------ refused stays refused
static void check_refused() {
  dsm_engine* e = nullptr;
  CHECK(dsm_create(0, &e) == DSM_OK);
  int32_t id = -1;
  for (int k = 0; k < 3; ++k) {  // a background that has no quantiles
    dsm_ensemble_desc d = desc(20, 30, DSM_SAMPLE_GT);
    d.partner_mode = DSM_PARTNER_GEX;
    d.gex[0] = 1.0f;
    d.gex[1] = 0.0f;
    d.gex[2] = 40000.0f;
    d.gex[3] = 120.0f;
    CHECK(dsm_add_ensemble(e, &d, &id) == DSM_ERR_ARG);
  }
  dsm_ensemble_desc d = desc(20, 30, DSM_SAMPLE_GT);
  d.corr_m = 3;  // 16 points
  for (int k = 0; k < 3; ++k) CHECK(dsm_add_ensemble(e, &d, &id) == DSM_ERR_ARG);
  d.corr_m = 2;
  CHECK(dsm_add_ensemble(e, &d, &id) == DSM_OK && id == 0);
  dsm_destroy(e);
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  if (which == "alloc") check_alloc();
  else if (which == "refused") check_refused();
  else if (which == "lanes") check_lanes();
  else if (which == "waves") check_waves();
  else if (which == "concurrent") check_concurrent();
  else if (which == "route_lane") check_lane_route();
  else if (which == "route_share") check_share_route();
  else if (which == "route_flow") check_flow_route();
  else if (which == "route_solo") check_solo_route();
  else if (which == "route_solo_flow") check_solo_flow_route();
  else if (which == "route_bin2") check_bin2_route();
  else if (which == "window") check_window();
  else return 2;
  std::printf("engine checks (%s): %d failures\n", which.c_str(), failures);
  return failures ? 1 : 0;
}
