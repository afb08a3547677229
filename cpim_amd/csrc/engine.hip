// C-ABI implementation of include/cpim_gpu.h for MI355X (gfx950).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/cpim_gpu.h"
#include "kernels.h"

#define CPIM_VERSION "cpim_amd 0.1 (gfx950)"

namespace {

// ---------------------------------------------------------------------------
// Errors
// ---------------------------------------------------------------------------
thread_local std::string g_last_error;

struct CpimFailure {
  int code;
  std::string msg;
};

[[noreturn]] void fail(int code, const std::string& msg) { throw CpimFailure{code, msg}; }

#define HIPC(expr)                                                                        \
  do {                                                                                    \
    hipError_t e__ = (expr);                                                              \
    if (e__ != hipSuccess)                                                                \
      fail(e__ == hipErrorOutOfMemory ? CPIM_ERR_OUT_OF_MEMORY : CPIM_ERR_HIP,            \
           std::string(#expr) + ": " + hipGetErrorString(e__));                           \
  } while (0)

template <typename F>
int guarded(F&& f) {
  try {
    f();
    return CPIM_OK;
  } catch (const CpimFailure& e) {
    g_last_error = e.msg;
    return e.code;
  } catch (const std::bad_alloc&) {
    g_last_error = "host allocation failed";
    return CPIM_ERR_OUT_OF_MEMORY;
  } catch (const std::exception& e) {
    g_last_error = e.what();
    return CPIM_ERR_RUNTIME;
  }
}

#define REQUIRE(cond, msg) \
  do {                     \
    if (!(cond)) fail(CPIM_ERR_INVALID_ARGUMENT, msg); \
  } while (0)

// ---------------------------------------------------------------------------
// Device properties (cached)
// ---------------------------------------------------------------------------
struct DevProps {
  int cus = 0;
  int max_lds = 0;
  int coop = 0;
  long long wall_khz = 0;
  long long mem = 0;
  std::string arch;
};

DevProps props_of(int dev) {
  static std::mutex mu;
  static std::vector<std::unique_ptr<DevProps>> cache;
  std::lock_guard<std::mutex> lock(mu);
  if ((int)cache.size() <= dev) cache.resize(dev + 1);
  if (!cache[dev]) {
    auto p = std::make_unique<DevProps>();
    hipDeviceProp_t prop;
    HIPC(hipGetDeviceProperties(&prop, dev));
    p->cus = prop.multiProcessorCount;
    p->max_lds = (int)prop.sharedMemPerBlock;
    p->mem = (long long)prop.totalGlobalMem;
    p->arch = prop.gcnArchName;
    int coop = 0;
    HIPC(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    p->coop = coop;
    int khz = 0;
    HIPC(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    p->wall_khz = khz;
    cache[dev] = std::move(p);
  }
  return *cache[dev];
}

// LDS used by one workgroup-engine domain copy; kept below 64 KB so that
// several workgroups share a CU.
constexpr long long kLdsBudget = 60 * 1024;

// Device wall-clock budget of one asynchronous fixpoint launch (ms); a
// launch that exceeds it returns an error instead of running on.
constexpr long long kAsyncBudgetMs = 20000;
// Waves per CU of the asynchronous fixpoint's grid.
constexpr int kAsyncWavesPerCu = 2;

// MAC nodes one launch may run before it returns to the host.
constexpr long long kNodesPerLaunch = 1 << 14;

// ---------------------------------------------------------------------------
// Model image: validated host-side layout of one network
// ---------------------------------------------------------------------------
struct ModelImage {
  int n = 0, max_dom = 0, W = 0, dpad = 0;
  int num_cons = 0;       // given
  int num_active = 0;     // propagated
  std::vector<int> cap;
  std::vector<ConMeta> con;
  std::vector<int> adj_off;
  std::vector<int4> adj;
  std::vector<int> bin_cons;          // active indices of binary constraints (plane build order)
  std::vector<int> tabs;              // active indices of table constraints
  bool simple = true;                 // no two binary constraints have the same scope
  int max_deg = 0;                    // most constraints on one variable
  int big_tabs = 0;                   // tables that small_table (device.h) does not take
  double reach = 0.0;                 // arcs of a variable and of its neighbours, mean over the values
  double density = 0.0;               // allowed share of the binary tuples (sample_density)
  std::vector<u64> rel_dense;         // owned dense rows when the desc has none
  const u64* rel = nullptr;           // [nb][max_dom][rel_words]
  int rel_words = 0;
  std::vector<u64> tsup;
  long long sup_words = 0;
  std::vector<u64> init_dom;          // [n][W]
  std::vector<int> nbr;               // [n] distinct neighbours over the active constraints, then tabs
};

// Share of the tuples that the binary constraints allow, from at most 8 rows
// each of at most 32 constraints.
double sample_density(const ModelImage& im) {
  const size_t nb = im.bin_cons.size();
  long long ones = 0, all = 0;
  for (size_t i = 0; i < std::min<size_t>(nb, 32); ++i) {
    const size_t k = i * nb / std::min<size_t>(nb, 32);
    const ConMeta& m = im.con[im.bin_cons[k]];
    const int cx = im.cap[m.scope[0]], rows = std::min(cx, 8);
    for (int j = 0; j < rows; ++j) {
      const u64* row = im.rel + (k * im.max_dom + (size_t)j * cx / rows) * im.rel_words;
      for (int w = 0; w < im.W; ++w) ones += __builtin_popcountll(row[w]);
    }
    all += (long long)rows * im.cap[m.scope[1]];
  }
  return all ? std::min(1.0, (double)ones / (double)all) : 1.0;
}

// What tests_by_workgroup asks of a network.
void measure_network(ModelImage& im) {
  auto deg = [&](int v) { return im.adj_off[v + 1] - im.adj_off[v]; };
  double values = 0.0;
  for (int v = 0; v < im.n; ++v) {
    long long arcs = deg(v);
    for (int k = im.adj_off[v]; k < im.adj_off[v + 1]; ++k)
      if (im.adj[k].y >= 0) arcs += deg(im.adj[k].y);
    im.max_deg = std::max(im.max_deg, deg(v));
    im.reach += (double)std::min<long long>(arcs, (long long)im.adj.size()) * im.cap[v];
    values += im.cap[v];
  }
  im.reach /= values;
  im.density = sample_density(im);
}

ModelImage make_image(const cpim_model_desc* d, bool skip_non_binary, bool own_rel = false) {
  REQUIRE(d != nullptr, "model description is null");
  REQUIRE(d->num_vars >= 1, "model has no variables");
  REQUIRE(d->dom_size != nullptr, "dom_size is null");
  REQUIRE(d->num_cons >= 0, "negative constraint count");
  REQUIRE(d->num_cons == 0 || (d->con_arity && d->con_scope), "constraint arrays are null");
  ModelImage im;
  im.n = d->num_vars;
  im.cap.assign(d->dom_size, d->dom_size + im.n);
  for (int v = 0; v < im.n; ++v) {
    REQUIRE(im.cap[v] >= 1, "domain of variable " + std::to_string(v) + " is empty");
    REQUIRE(im.cap[v] <= 64 * CPIM_MAX_WORDS, "domain size above 1024 is not supported");
    im.max_dom = std::max(im.max_dom, im.cap[v]);
  }
  im.W = (im.max_dom + 63) / 64;
  im.dpad = 64 * im.W;
  im.num_cons = d->num_cons;
  const long long nw = (long long)im.n * im.W;
  // scopes
  std::vector<long long> scope_off(d->num_cons + 1, 0);
  int nbin_total = 0;
  for (int c = 0; c < d->num_cons; ++c) {
    const int ar = d->con_arity[c];
    REQUIRE(ar >= 2, "constraint " + std::to_string(c) + " has arity below 2");
    scope_off[c + 1] = scope_off[c] + ar;
    if (ar == 2) ++nbin_total;
  }
  for (long long i = 0; i < scope_off[d->num_cons]; ++i)
    REQUIRE(d->con_scope[i] >= 0 && d->con_scope[i] < im.n, "scope names an unknown variable");
  const bool any_nary = nbin_total != d->num_cons;
  if (any_nary && !skip_non_binary) REQUIRE(d->tup_off && d->tuples, "tables need tup_off/tuples");
  if (!d->bin_rel) REQUIRE(nbin_total == 0 || (d->tup_off && d->tuples), "binary relations missing");
  if (d->bin_rel) REQUIRE(d->rel_words >= im.W, "rel_words is below ceil(max_dom/64)");
  // active constraints
  long long sup_off = 0, tsup_off = 0;
  int bin_k = 0;
  std::vector<int> bin_ordinal_of_active;
  for (int c = 0; c < d->num_cons; ++c) {
    const int ar = d->con_arity[c];
    const int* sc = d->con_scope + scope_off[c];
    if (ar == 2) {
      REQUIRE(sc[0] != sc[1], "binary constraint " + std::to_string(c) + " repeats a variable");
      ConMeta m{};
      m.kind = 0;
      m.arity = 2;
      m.scope[0] = sc[0];
      m.scope[1] = sc[1];
      m.off = sup_off;
      sup_off += 2ll * im.W * im.dpad;
      im.bin_cons.push_back((int)im.con.size());
      bin_ordinal_of_active.push_back(bin_k);
      im.con.push_back(m);
      ++bin_k;
    } else {
      if (skip_non_binary) continue;
      REQUIRE(ar <= CPIM_MAX_ARITY, "tables of arity above 8 are not supported");
      const long long t0 = d->tup_off[c], t1 = d->tup_off[c + 1];
      REQUIRE(t1 >= t0 && (t1 - t0) % ar == 0, "tup_off does not delimit whole tuples");
      const long long T = (t1 - t0) / ar;
      REQUIRE(T < (1ll << 31), "tables of 2^31 tuples or more are not supported");
      for (int i = 0; i < ar; ++i)
        for (int j = i + 1; j < ar; ++j) REQUIRE(sc[i] != sc[j], "table scope repeats a variable");
      ConMeta m{};
      m.kind = 1;
      m.arity = ar;
      for (int i = 0; i < CPIM_MAX_ARITY; ++i) m.scope[i] = sc[i < ar ? i : 0];  // (wg_fixpoint reads all)
      m.tw = std::max<int>(1, (int)((T + 63) / 64));
      m.off = tsup_off;
      const long long words = (long long)ar * im.dpad * m.tw;
      REQUIRE(tsup_off + words <= (1ll << 32), "table supports above 32 GiB are not supported");
      im.tsup.resize(tsup_off + words, 0ull);
      for (long long t = 0; t < T; ++t) {
        const int32_t* tup = d->tuples + t0 + t * ar;
        bool ok = true;
        for (int i = 0; i < ar; ++i) ok = ok && tup[i] >= 0 && tup[i] < im.cap[sc[i]];
        REQUIRE(ok, "table tuple value outside its domain");
        for (int i = 0; i < ar; ++i)
          im.tsup[tsup_off + ((long long)i * im.dpad + tup[i]) * m.tw + (t >> 6)] |= 1ull << (t & 63);
      }
      tsup_off += words;
      bin_ordinal_of_active.push_back(-1);
      im.tabs.push_back((int)im.con.size());
      if (im.max_dom > 16 || ar > 4 || m.tw > 8) ++im.big_tabs;
      im.con.push_back(m);
    }
  }
  im.num_active = (int)im.con.size();
  im.sup_words = std::max<long long>(sup_off, 1);
  if (im.tsup.empty()) im.tsup.assign(1, 0ull);
  // dense binary rows
  if (d->bin_rel) {
    im.rel = reinterpret_cast<const u64*>(d->bin_rel);
    im.rel_words = d->rel_words;
    if (own_rel) {
      im.rel_dense.assign(im.rel, im.rel + (size_t)nbin_total * im.max_dom * d->rel_words);
      im.rel = im.rel_dense.data();
    }
  } else if (!im.bin_cons.empty()) {
    im.rel_words = im.W;
    im.rel_dense.assign((size_t)im.bin_cons.size() * im.max_dom * im.W, 0ull);
    int k = 0;
    for (int c = 0; c < d->num_cons; ++c) {
      if (d->con_arity[c] != 2) continue;
      const int* sc = d->con_scope + scope_off[c];
      REQUIRE(d->tup_off[c + 1] >= d->tup_off[c] && (d->tup_off[c + 1] - d->tup_off[c]) % 2 == 0,
              "tup_off does not delimit whole tuples");
      for (long long t = d->tup_off[c]; t < d->tup_off[c + 1]; t += 2) {
        const int a = d->tuples[t], b = d->tuples[t + 1];
        REQUIRE(a >= 0 && a < im.cap[sc[0]] && b >= 0 && b < im.cap[sc[1]],
                "binary tuple value outside its domain");
        im.rel_dense[((size_t)k * im.max_dom + a) * im.W + (b >> 6)] |= 1ull << (b & 63);
      }
      ++k;
    }
    im.rel = im.rel_dense.data();
  }
  // CSR (constraint order per variable, like Network's subscription lists)
  std::vector<int> deg(im.n, 0);
  for (const auto& m : im.con)
    for (int i = 0; i < m.arity; ++i) ++deg[m.scope[i]];
  im.adj_off.assign(im.n + 1, 0);
  for (int v = 0; v < im.n; ++v) im.adj_off[v + 1] = im.adj_off[v] + deg[v];
  im.adj.resize(im.adj_off[im.n]);
  std::vector<int> pos(im.adj_off.begin(), im.adj_off.end() - 1);
  for (int c = 0; c < im.num_active; ++c) {
    const auto& m = im.con[c];
    for (int i = 0; i < m.arity; ++i) {
      const int v = m.scope[i];
      const int other = m.kind == 0 ? m.scope[1 - i] : -1;
      // binary: index of the constraint's plane pair (sup offset / (2 W dpad))
      const int pair = m.kind == 0 ? (int)(m.off / (2ll * im.W * im.dpad)) : -1;
      im.adj[pos[v]++] = make_int4(c, other, i | v << 4, pair);
    }
  }
  // neighbour counts (Network::get_neighbor, src/Network.cpp:467-474)
  im.nbr.assign(im.n, 0);
  {
    std::vector<int> seen(im.n, -1), paired(im.n, -1);
    for (int v = 0; v < im.n; ++v)
      for (int k = im.adj_off[v]; k < im.adj_off[v + 1]; ++k) {
        const auto& m = im.con[im.adj[k].x];
        if (m.kind == 0) {
          const int y = im.adj[k].y;
          if (paired[y] == v) im.simple = false;
          paired[y] = v;
        }
        for (int i = 0; i < m.arity; ++i) {
          const int y = m.scope[i];
          if (y != v && seen[y] != v) {
            seen[y] = v;
            ++im.nbr[v];
          }
        }
      }
  }
  im.nbr.insert(im.nbr.end(), im.tabs.begin(), im.tabs.end());
  // level 0
  im.init_dom.assign(nw, 0ull);
  for (int v = 0; v < im.n; ++v)
    for (int a = 0; a < im.cap[v]; ++a) {
      const bool keep = d->init_dom == nullptr ||
                        ((d->init_dom[(long long)v * im.W + (a >> 6)] >> (a & 63)) & 1ull);
      if (keep) im.init_dom[(long long)v * im.W + (a >> 6)] |= 1ull << (a & 63);
    }
  return im;
}

// ---------------------------------------------------------------------------
// Device copy of a network
// ---------------------------------------------------------------------------
// Device memory: owned (freed on destruction) or a view into an Arena.
struct DevAlloc {
  void* p = nullptr;
  bool owned = true;
  DevAlloc() = default;
  explicit DevAlloc(size_t bytes) {
    if (bytes == 0) bytes = 16;
    HIPC(hipMalloc(&p, bytes));
  }
  static DevAlloc view(void* q) {
    DevAlloc d;
    d.p = q;
    d.owned = false;
    return d;
  }
  ~DevAlloc() {
    if (p && owned) (void)hipFree(p);
  }
  DevAlloc(const DevAlloc&) = delete;
  DevAlloc& operator=(const DevAlloc&) = delete;
  DevAlloc(DevAlloc&& o) noexcept : p(o.p), owned(o.owned) { o.p = nullptr; }
  DevAlloc& operator=(DevAlloc&& o) noexcept {
    if (this != &o) {
      if (p && owned) (void)hipFree(p);
      p = o.p;
      owned = o.owned;
      o.p = nullptr;
    }
    return *this;
  }
  template <typename T>
  T* as() const { return static_cast<T*>(p); }
};

// One device allocation carved into the arrays of one network (and its
// search state): a served request costs one hipMalloc instead of one per
// array.  plan mode (block == nullptr) only adds up the sizes.
struct Arena {
  DevAlloc block;
  long long cap = 0, used = 0;
  static long long round(long long b) { return (std::max<long long>(b, 16) + 255) & ~255ll; }
  void reserve(long long bytes) {
    block = DevAlloc((size_t)std::max<long long>(bytes, 256));
    cap = bytes;
    used = 0;
  }
  DevAlloc take(long long bytes) {
    const long long b = round(bytes);
    if (!block.p) {  // plan mode
      used += b;
      return DevAlloc();
    }
    if (used + b > cap) fail(CPIM_ERR_RUNTIME, "arena overflow (size plan and build disagree)");
    DevAlloc d = DevAlloc::view(static_cast<char*>(block.p) + used);
    used += b;
    return d;
  }
};

struct DevModel {
  int n = 0, W = 0, dpad = 0, max_dom = 0, num_active = 0;
  DevAlloc adj_off, adj, con, sup, tsup, cap, nbr;  // nbr: [n], then the table constraints
  int ntabs = 0, big_tabs = 0;
  bool simple = false;
  DevAlloc lnet_img;  // the network image for LDS (LdsNet), when small enough
  LdsNet lnet{};
  long long bytes = 0;
  DevNet net() const {
    DevNet d;
    d.n = n;
    d.W = W;
    d.dpad = dpad;
    d.ncons = num_active;
    d.adj_off = adj_off.as<int>();
    d.adj = adj.as<int4>();
    d.con = con.as<ConMeta>();
    d.sup = sup.as<u64>();
    d.tsup = tsup.as<u64>();
    d.tabs = nbr.as<int>() + n;
    d.ntabs = ntabs;
    d.big_tabs = big_tabs;
    d.cap = max_dom;
    d.simple = simple ? 1 : 0;
    return d;
  }
};

// One device array: a view of `arena` when given, else its own allocation.
DevAlloc dev_array(Arena* arena, long long bytes) {
  return arena ? arena->take(bytes) : DevAlloc((size_t)std::max<long long>(bytes, 16));
}

template <typename T>
void upload(DevAlloc& dst, const std::vector<T>& src, hipStream_t s, long long& bytes, Arena* arena = nullptr) {
  const size_t b = std::max<size_t>(sizeof(T) * src.size(), 16);
  dst = dev_array(arena, (long long)b);
  if (!src.empty()) HIPC(hipMemcpyAsync(dst.p, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice, s));
  bytes += (long long)b;
}

// Largest network image copied into LDS by the device MAC (LdsNet).
constexpr long long kLdsNetMax = 128 * 1024;

long long align16(long long b) { return (b + 15) & ~15ll; }

// The LdsNet image of a network: the arrays of DevNet in one block, planes
// and tables with value stride dc (LdsNet) instead of dpad.  Built after the
// planes (the plane rows are copied from the device planes); skipped when the
// image would exceed kLdsNetMax.  The copies are queued on s from `h`,
// which the caller keeps until s is synchronized.
struct LdsLayout {
  int dc;
  long long o_adj, o_con, o_sup, o_tsup, o_tabs, bytes;
};

LdsLayout lds_layout(const ModelImage& im, bool odd = true) {
  // an even stride only where the odd one alone keeps the image out of LDS.
  // The odd one can make the image too large for a unit's share of a CU; the
  // rows are then read from memory.  A batch at that line, 512 x n=60 d=8
  // e=355, takes 1.6 ms all the same.
  const int n = im.n, W = im.W, dc = odd ? im.max_dom | 1 : im.max_dom;
  const long long npairs = (long long)im.bin_cons.size();
  long long tsup_c = 0;
  for (const ConMeta& m : im.con)
    if (m.kind == 1) tsup_c += (long long)m.arity * dc * m.tw;
  LdsLayout L;
  L.dc = dc;
  L.o_adj = align16(4ll * (n + 1));
  L.o_con = L.o_adj + align16(16ll * (long long)im.adj.size());
  L.o_sup = L.o_con + align16((long long)sizeof(ConMeta) * (long long)im.con.size());
  const long long sup_words = npairs * 2 * W * dc + 64ll * W;
  L.o_tsup = L.o_sup + align16(8 * sup_words);
  // small tables read 16 rows a position, past the last one's end by up to 16 x 8 words
  L.o_tabs = L.o_tsup + align16(8 * std::max<long long>(1, tsup_c + (tsup_c ? 16 * 8 : 0)));
  L.bytes = L.o_tabs + align16(4 * (long long)im.tabs.size());
  if (odd && L.bytes > kLdsNetMax) return lds_layout(im, false);
  return L;
}

void build_lds_image(const ModelImage& im, DevModel& dm, hipStream_t s, std::vector<char>& h,
                     Arena* arena = nullptr) {
  const int n = im.n, W = im.W, dpad = im.dpad;
  const long long npairs = (long long)im.bin_cons.size();
  const LdsLayout L = lds_layout(im);
  const int dc = L.dc;
  const long long o_adj = L.o_adj, o_con = L.o_con, o_sup = L.o_sup, o_tsup = L.o_tsup, bytes = L.bytes;
  if (bytes > kLdsNetMax) return;
  h.assign((size_t)bytes, 0);
  std::memcpy(h.data(), im.adj_off.data(), 4 * (size_t)(n + 1));
  if (!im.adj.empty()) std::memcpy(h.data() + o_adj, im.adj.data(), 16 * im.adj.size());
  ConMeta* con = (ConMeta*)(h.data() + o_con);
  u64* ts = (u64*)(h.data() + o_tsup);
  long long toff = 0;
  for (size_t c = 0; c < im.con.size(); ++c) {
    ConMeta m = im.con[c];
    if (m.kind == 0) {
      m.off = m.off / (2ll * W * dpad) * (2ll * W * dc);
    } else {
      for (int q = 0; q < m.arity; ++q)
        for (int a = 0; a < im.max_dom; ++a)
          std::memcpy(ts + toff + ((long long)q * dc + a) * m.tw,
                      im.tsup.data() + m.off + ((long long)q * dpad + a) * m.tw, 8 * (size_t)m.tw);
      m.off = toff;
      toff += (long long)m.arity * dc * m.tw;
    }
    con[c] = m;
  }
  if (!im.tabs.empty()) std::memcpy(h.data() + L.o_tabs, im.tabs.data(), 4 * im.tabs.size());
  dm.lnet_img = dev_array(arena, bytes);
  HIPC(hipMemcpyAsync(dm.lnet_img.p, h.data(), (size_t)bytes, hipMemcpyHostToDevice, s));
  if (npairs > 0)
    HIPC(hipMemcpy2DAsync((char*)dm.lnet_img.p + o_sup, 8 * (size_t)dc, dm.sup.p, 8 * (size_t)dpad,
                          8 * (size_t)std::min(dc, dpad), (size_t)(npairs * 2 * W), hipMemcpyDeviceToDevice, s));
  dm.bytes += bytes;
  dm.lnet.src = dm.lnet_img.as<uint4>();
  dm.lnet.bytes = (int)bytes;
  dm.lnet.dc = dc;
  dm.lnet.o_adj = (int)o_adj;
  dm.lnet.o_con = (int)o_con;
  dm.lnet.o_sup = (int)o_sup;
  dm.lnet.o_tsup = (int)o_tsup;
  dm.lnet.o_tabs = (int)L.o_tabs;
  // wg_fixpoint_flat: a lane per variable, kFlatArcs arcs a lane (one if a
  // domain has more than 16 values), a wave per table
  const int arcs = (int)im.adj.size(), tabs = (int)im.tabs.size();
  auto waves = [](int lanes) { return 64 * ((lanes + 63) / 64); };
  const int per_lane = im.max_dom <= 16 ? kFlatArcs : 1;
  const int least = std::max(waves(n), std::max(64, waves((arcs + per_lane - 1) / per_lane)) + 64 * tabs);
  bool small = W == 1 && im.max_dom <= 32 && tabs <= kFlatTables && least <= 1024;
  for (const ConMeta& m : im.con) small = small && (m.kind == 0 || (im.max_dom <= 16 && m.arity <= 4 && m.tw <= 8));
  if (small) {
    dm.lnet.flat_min = least;
    dm.lnet.flat_threads = std::min(1024, std::max(least, waves(arcs) + 64 * tabs));
  }
}

// Whether the workgroup fixpoint looks at the tables first (wg_fixpoint's kTabs).
bool many_tables(const ModelImage& im, int threads) {
  return (int)im.tabs.size() > kTableTurns * (threads / 64);
}

// Whether a search takes the whole workgroup fixpoint (kTight and kTabs) when it
// has no network image.
//
// For the tables, more than kTableTurns a wave: 300 of arity 5 and 3,000 tuples,
// 60 nodes, 33 ms against 43; 900 of arity 3, 7.3 against 15.3 ms.
//
// For tight relations settled by the wave (wave_settle), domains of three words and more, and at least 12 turns of a
// 1024-lane workgroup over the arc words.  Where that is so, a lane's serial
// work is what a round waits for.  With it against without it, ms: n=300 d=250
// e=20000 t=0.963, 30 nodes 13.8 / 25.5, t=0.95 6.3 / 10.1; n=300 d=250 e=2000
// t=0.97 2.7 / 3.7; n=50 d=1000 e=600 t=0.97 2.7 / 3.2, t=0.5 2.24 / 2.17.
// Below that line, and for two words, the choice between the two sides costs
// more than it saves: n=30 d=1000 e=131 3.7 / 2.4; n=100 d=250 e=1000 t=0.9 5.9
// / 5.1; n=300 d=100 e=6000 t=0.84 1.66 / 1.39.  (Such a network's rows alone
// are more than 3 MB, far beyond an image.)
bool full_search(const ModelImage& im, int threads) {
  long long wp = 1;
  while (wp < im.W) wp *= 2;
  return many_tables(im, threads) || (im.W >= 3 && (long long)im.adj.size() * wp >= 12 * 1024);
}

// Device bytes build_device_model takes from an arena for im (the same
// arrays, each rounded as the arena rounds it).
long long model_arena_bytes(const ModelImage& im) {
  auto r = [](long long b) { return Arena::round(std::max<long long>(b, 16)); };
  long long b = r(4ll * (long long)im.adj_off.size()) + r(16ll * (long long)im.adj.size()) +
                r((long long)sizeof(ConMeta) * (long long)im.con.size()) + r(8ll * (long long)im.tsup.size()) +
                r(4ll * (long long)im.cap.size()) + r(4ll * (long long)im.nbr.size()) + r(8ll * im.sup_words);
  const long long img = lds_layout(im).bytes;
  if (img <= kLdsNetMax) b += r(img);
  return b;
}

// Staging of the dense rows on their way to the planes: bins (the binary
// constraints' indices) and slices of rows, reused across builds when the
// caller keeps it.
struct PlaneStaging {
  DevAlloc buf;
  long long bytes = 0;
  char* get(long long b) {
    if (b > bytes) {
      buf = DevAlloc((size_t)b);
      bytes = b;
    }
    return buf.as<char>();
  }
};

// The device arrays of a network; with an arena they are views into it (one
// allocation in all), with staging the row slices reuse its buffer.  Returns
// after the planes and the image are complete on stream s.
void build_device_model(const ModelImage& im, DevModel& dm, hipStream_t s, Arena* arena = nullptr,
                        PlaneStaging* staging = nullptr) {
  dm.n = im.n;
  dm.W = im.W;
  dm.dpad = im.dpad;
  dm.max_dom = im.max_dom;
  dm.num_active = im.num_active;
  upload(dm.adj_off, im.adj_off, s, dm.bytes, arena);
  upload(dm.adj, im.adj, s, dm.bytes, arena);
  upload(dm.con, im.con, s, dm.bytes, arena);
  upload(dm.tsup, im.tsup, s, dm.bytes, arena);
  upload(dm.cap, im.cap, s, dm.bytes, arena);
  upload(dm.nbr, im.nbr, s, dm.bytes, arena);
  dm.ntabs = (int)im.tabs.size();
  dm.big_tabs = im.big_tabs;
  dm.simple = im.simple;
  dm.sup = dev_array(arena, (long long)sizeof(u64) * im.sup_words);
  dm.bytes += sizeof(u64) * im.sup_words;
  const int nb = (int)im.bin_cons.size();
  if (nb > 0) {
    // Upload the dense rows in slices and build the planes on the device.
    const long long row_words = (long long)im.max_dom * im.rel_words;
    const int slice = (int)std::max<long long>(1, std::min<long long>(nb, (256ll << 20) / (8 * row_words)));
    const long long bins_bytes = Arena::round(4ll * nb);
    PlaneStaging local;
    PlaneStaging& st = staging ? *staging : local;
    char* base = st.get(bins_bytes + 8ll * row_words * slice);
    int* bins = reinterpret_cast<int*>(base);
    u64* rel_dev = reinterpret_cast<u64*>(base + bins_bytes);
    HIPC(hipMemcpyAsync(bins, im.bin_cons.data(), 4ll * nb, hipMemcpyHostToDevice, s));
    for (int k0 = 0; k0 < nb; k0 += slice) {
      const int k1 = std::min(nb, k0 + slice);
      HIPC(hipMemcpyAsync(rel_dev, im.rel + (long long)k0 * row_words,
                          sizeof(u64) * row_words * (k1 - k0), hipMemcpyHostToDevice, s));
      const long long waves = (long long)(k1 - k0) * im.W;
      const int threads = 256;
      const long long blocks = (waves * 64 + threads - 1) / threads;
      hipLaunchKernelGGL(k_build_planes, dim3((unsigned)blocks), dim3(threads), 0, s,
                         rel_dev, k1 - k0, im.max_dom, im.rel_words, im.W, im.dpad,
                         bins + k0, dm.con.as<ConMeta>(), dm.cap.as<int>(), dm.sup.as<u64>());
      HIPC(hipGetLastError());
      if (k1 < nb) HIPC(hipStreamSynchronize(s));  // the next slice overwrites rel_dev
    }
  }
  std::vector<char> lds_image;  // host side of the image copy, until the sync below
  build_lds_image(im, dm, s, lds_image, arena);
  HIPC(hipStreamSynchronize(s));
}

struct DeviceGuard {
  int prev = 0;
  explicit DeviceGuard(int dev) {
    HIPC(hipGetDevice(&prev));
    if (prev != dev) HIPC(hipSetDevice(dev));
  }
  ~DeviceGuard() { (void)hipSetDevice(prev); }
};

long long now_ns() {
  return std::chrono::duration_cast<std::chrono::nanoseconds>(
             std::chrono::steady_clock::now().time_since_epoch())
      .count();
}

}  // namespace

// Device buffers of the singleton-test paths, kept by the model between
// calls (grown on demand) so that a SAC pass allocates nothing once warm.
struct SacScratch {
  DevAlloc tests, fails, revs;
  long long cap = 0;
  DevAlloc stests, perm, gfirst, gorder;  // bit-sliced path: sorted tests, their order, group starts,
                                          // group of each workgroup slot
  long long scap = 0, gcap = 0;
  // removal slices of the wide bit-sliced kernel: zeroed when allocated, and
  // left all zero by every launch of that kernel
  DevAlloc dead;
  long long dead_bytes = 0;
  hipEvent_t ev[2] = {nullptr, nullptr};
  SacScratch() = default;
  SacScratch(const SacScratch&) = delete;
  SacScratch& operator=(const SacScratch&) = delete;
  ~SacScratch() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  void events() {
    for (hipEvent_t& e : ev)
      if (!e) HIPC(hipEventCreate(&e));
  }
};

// ---------------------------------------------------------------------------
// Host boxes: pinned memory that kernels answer in (HostBox in kernels.h), one
// per model from its first call on.  Pinning takes tens of microseconds, so
// models that come and go hand their boxes on through a pool of at most
// kBoxPool; every box returns to it, or is freed, with its model.
// ---------------------------------------------------------------------------
namespace {

constexpr long long kBoxDataBytes = 64 * 1024;
constexpr size_t kBoxPool = 8;
std::mutex g_box_mu;
std::vector<HostBox*> g_boxes;

HostBox* take_box() {
  {
    std::lock_guard<std::mutex> lock(g_box_mu);
    if (!g_boxes.empty()) {
      HostBox* b = g_boxes.back();
      g_boxes.pop_back();
      return b;
    }
  }
  void* p = nullptr;
  HIPC(hipHostMalloc(&p, sizeof(HostBox) + kBoxDataBytes, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
  HostBox* b = static_cast<HostBox*>(p);
  b->seq = 0;
  b->issued = 0;
  return b;
}

void give_box(HostBox* b) {
  if (!b) return;
  {
    std::lock_guard<std::mutex> lock(g_box_mu);
    if (g_boxes.size() < kBoxPool) {
      g_boxes.push_back(b);
      return;
    }
  }
  (void)hipHostFree(b);
}

}  // namespace

// ---------------------------------------------------------------------------
// GModel
// ---------------------------------------------------------------------------
// Words before the asynchronous frontier in `front`: the rounds' three bitmaps,
// up to the next 256 bytes (its waves read 64 words at a time).
constexpr long long async_front(int nvw) { return (3ll * nvw + 63) & ~63ll; }

struct cpim_gmodel {
  int device = 0;
  hipStream_t stream = nullptr;
  ModelImage im;  // host layout (rel pointer not kept beyond build)
  Arena arena;    // the device arrays below, in one allocation
  DevModel dm;
  int max_depth = 0;
  int current_level = 0;
  int assigned_size = 0;
  DevAlloc dom;    // [max_depth][n][W]
  DevAlloc size;   // [max_depth][n]
  DevAlloc front;  // three bitmaps of variables (grid rounds), then one of constraints (asynchronous)
  DevAlloc ctl;    // GacCtl
  bool ctl_ready = false;      // ctl and front are in their first state (k_gac_init, grid_finish)
  mutable HostBox* box_ = nullptr;  // answers of the model's kernels
  DevAlloc async_ctl;
  DevAlloc scratch;  // workgroup-engine scratch when a copy does not fit in LDS
  long long scratch_bytes = 0;
  int nfw = 0;     // words of a bitmap of the constraints
  int nvw = 0;     // words of a bitmap of the variables
  std::vector<int2> assigned;  // d_assigned mirror: (var, value) per level
  // per level: at its closure (a fixpoint ended consistent and nothing wrote
  // since), closed but for the domain of one variable (its id), or open
  enum : int { kOpen = -2, kClosed = -1 };
  std::vector<int> closure;
  void wrote(int level, int var) {
    int& c = closure[level];
    c = c == kClosed || c == var ? var : kOpen;
  }
  // the fixpoint over every constraint (var < 0) or from var ended
  void settled(int level, int before, int var, const cpim_gac_stats& st) {
    const bool all = var < 0 || before == kClosed || before == var;
    closure[level] = st.converged && !st.inconsistent && all ? kClosed : kOpen;
  }
  DevProps props;
  SacScratch sac;
  hipEvent_t gev[2] = {nullptr, nullptr};  // kernel timing of the fixpoint entry points
  // dom/wdeg bookkeeping of the network (Tabular::weight, Network.cpp:303):
  // weights start at 1 with the model and persist across solves, as the
  // reference's constraint weights do; the stamps order AC3's revisions
  // within a call (in LDS where they fit)
  DevAlloc wdeg_weight, wdeg_stamp;

  // the weights (and room for the stamps), allocated on first use, and the
  // weights set to 1, on first use or on reset
  void wdeg_init() {
    const int nc = std::max(1, dm.num_active);
    if (!wdeg_weight.p) {
      wdeg_weight = DevAlloc(sizeof(float) * nc);
      wdeg_stamp = DevAlloc(sizeof(int) * nc);
    }
    const std::vector<float> ones(nc, 1.0f);
    HIPC(hipMemcpyAsync(wdeg_weight.p, ones.data(), sizeof(float) * nc, hipMemcpyHostToDevice, stream));
    HIPC(hipStreamSynchronize(stream));  // `ones` is host stack memory
  }

  // The box and the number of the next call that answers in it (counted by the
  // host: a launch that failed may leave earlier ones queued, which still
  // store their numbers).
  HostBox* box() const {
    if (!box_) box_ = take_box();
    return box_;
  }
  unsigned long long next_seq() const { return ++box()->issued; }

  // Waits for call `seq` (its kernel is the last work queued on the stream):
  // the kernel's answer arrives a few microseconds before the runtime reports
  // the stream idle.  The stream is asked now and then, so that a launch that
  // failed ends the wait with its error.
  void wait_box(unsigned long long seq) const {
    const unsigned long long* at = &box_->seq;
    for (unsigned i = 1;; ++i) {
      if (__atomic_load_n(at, __ATOMIC_ACQUIRE) == seq) return;
      __builtin_ia32_pause();
      if ((i & 4095u) == 0u) {
        const hipError_t e = hipStreamQuery(stream);
        if (e == hipErrorNotReady) {
          (void)hipGetLastError();
          continue;
        }
        HIPC(e);
        if (__atomic_load_n(at, __ATOMIC_ACQUIRE) == seq) return;
        fail(CPIM_ERR_RUNTIME, "a kernel ended without its answer");
      }
    }
  }
  double ticks_ms(unsigned long long ticks) const { return (double)ticks / (double)std::max<long long>(props.wall_khz, 1); }

  // One k_level_op on a level, and its answer.
  int level_op(int op, int level, int var, int value) const {
    HostBox* b = box();
    const unsigned long long seq = next_seq();
    // more threads where the sizes are many: 20,000 of them 18.5 us with 256
    // threads, 12 with 1024 (copying them to the host 13.5); up to 2,048, 0.5 us more
    const bool many = (op == kOpMinVar || op == kOpAll) && dm.n > 2048;
    hipLaunchKernelGGL(many ? k_level_op<1024> : k_level_op<256>, dim3(1), dim3(many ? 1024 : 256), 0, stream, op,
                       level_dom(level), level_size(level), dm.n, dm.W, dm.max_dom, var, value, &b->scalar, &b->seq, seq);
    HIPC(hipGetLastError());
    wait_box(seq);
    return b->scalar;
  }

  void gac_events() {
    for (hipEvent_t& e : gev)
      if (!e) HIPC(hipEventCreate(&e));
  }
  // device time between gev[0] and gev[1] (both recorded, gev[1] complete)
  double gac_elapsed_ms() {
    float ms = 0.f;
    HIPC(hipEventElapsedTime(&ms, gev[0], gev[1]));
    return ms;
  }

  u64* level_dom(int level) const { return dom.as<u64>() + (long long)level * dm.n * dm.W; }
  int* level_size(int level) const { return size.as<int>() + (long long)level * dm.n; }
  long long level_words() const { return (long long)dm.n * dm.W; }

  char* get_scratch(long long bytes) {
    if (bytes > scratch_bytes) {
      scratch = DevAlloc((size_t)bytes);
      scratch_bytes = bytes;
    }
    return scratch.as<char>();
  }
  void sync() { HIPC(hipStreamSynchronize(stream)); }
  bool level_in_box() const { return 8 * level_words() <= kBoxDataBytes; }
};

extern "C" {

void cpim_gmodel_options_default(cpim_gmodel_options* o) {
  if (!o) return;
  o->device_id = 0;
  o->enable_prefetch = 0;
  o->skip_non_binary = 1;
  o->skip_conflicts = 0;
}

const char* cpim_last_error(void) { return g_last_error.c_str(); }
const char* cpim_version(void) { return CPIM_VERSION; }

int cpim_get_device_info(int32_t device_id, cpim_device_info* out) {
  return guarded([&] {
    REQUIRE(out != nullptr, "out is null");
    int count = 0;
    HIPC(hipGetDeviceCount(&count));
    REQUIRE(device_id >= 0 && device_id < count, "invalid device id");
    const DevProps p = props_of(device_id);
    out->compute_units = p.cus;
    out->lds_bytes_per_block = p.max_lds;
    out->cooperative_launch = p.coop;
    out->wavefront_size = 64;
    out->global_mem_bytes = p.mem;
    std::snprintf(out->arch, sizeof(out->arch), "%s", p.arch.c_str());
  });
}

int cpim_measure_copy_bandwidth(int32_t device_id, int64_t bytes, int32_t reps, double* gbps) {
  return guarded([&] {
    REQUIRE(gbps && bytes >= 16 && reps >= 1, "bad argument");
    DeviceGuard g(device_id);
    const DevProps p = props_of(device_id);
    const long long n16 = bytes / 16;
    DevAlloc a(16 * n16), b(16 * n16);
    hipStream_t s;
    HIPC(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    HIPC(hipMemsetAsync(a.p, 1, 16 * n16, s));
    hipEvent_t e0, e1;
    HIPC(hipEventCreate(&e0));
    HIPC(hipEventCreate(&e1));
    const int threads = 256;
    const long long blocks = std::min<long long>((n16 + threads - 1) / threads, 8ll * p.cus * 4);
    double best = 0;
    for (int r = 0; r < reps; ++r) {
      HIPC(hipEventRecord(e0, s));
      hipLaunchKernelGGL(k_stream_copy, dim3((unsigned)blocks), dim3(threads), 0, s, a.as<uint4>(), b.as<uint4>(), n16);
      HIPC(hipGetLastError());
      HIPC(hipEventRecord(e1, s));
      HIPC(hipEventSynchronize(e1));
      float ms = 0.f;
      HIPC(hipEventElapsedTime(&ms, e0, e1));
      if (ms > 0) best = std::max(best, 2.0 * 16 * n16 / (ms * 1e-3) / 1e9);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(s);
    *gbps = best;
  });
}

int cpim_gmodel_create(const cpim_model_desc* desc, const cpim_gmodel_options* opts,
                       cpim_gmodel** out) {
  return guarded([&] {
    REQUIRE(out != nullptr, "out is null");
    *out = nullptr;
    cpim_gmodel_options o;
    cpim_gmodel_options_default(&o);
    if (opts) o = *opts;
    // validate the model before touching the device
    ModelImage im = make_image(desc, o.skip_non_binary != 0);
    measure_network(im);
    int count = 0;
    HIPC(hipGetDeviceCount(&count));
    REQUIRE(o.device_id >= 0 && o.device_id < count, "invalid device id");
    DeviceGuard g(o.device_id);
    auto m = std::make_unique<cpim_gmodel>();
    m->device = o.device_id;
    m->props = props_of(o.device_id);
    HIPC(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    m->im = std::move(im);
    const int n = m->im.n;
    m->max_depth = n + 1;
    m->nfw = std::max(1, (m->im.num_active + 31) / 32);
    m->nvw = (n + 31) / 32;
    const long long lw = (long long)n * m->im.W;
    const long long dom_bytes = (long long)sizeof(u64) * lw * m->max_depth;
    const long long size_bytes = (long long)sizeof(int) * n * m->max_depth;
    const long long front_bytes = (long long)sizeof(unsigned) * (async_front(m->nvw) + m->nfw);
    m->arena.reserve(model_arena_bytes(m->im) + Arena::round(dom_bytes) + Arena::round(size_bytes) +
                     Arena::round(front_bytes) + Arena::round((long long)sizeof(GacCtl)));
    build_device_model(m->im, m->dm, m->stream, &m->arena);
    m->im.rel = nullptr;
    m->im.rel_dense.clear();
    m->im.rel_dense.shrink_to_fit();
    m->dom = m->arena.take(dom_bytes);
    m->size = m->arena.take(size_bytes);
    m->front = m->arena.take(front_bytes);
    m->ctl = m->arena.take((long long)sizeof(GacCtl));
    HIPC(hipMemcpyAsync(m->dom.p, m->im.init_dom.data(), sizeof(u64) * lw, hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(k_sizes, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->level_dom(0),
                       m->level_size(0), n, m->dm.W);
    HIPC(hipGetLastError());
    m->assigned.assign(m->max_depth, make_int2(-1, -1));
    m->closure.assign(m->max_depth, cpim_gmodel::kOpen);
    m->dm.bytes += dom_bytes + size_bytes + front_bytes + (long long)sizeof(GacCtl);
    m->sync();
    *out = m.release();
  });
}

int cpim_gmodel_destroy(cpim_gmodel* m) {
  return guarded([&] {
    if (!m) return;
    DeviceGuard g(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    hipStream_t s = m->stream;
    give_box(m->box_);
    for (hipEvent_t e : m->gev)
      if (e) (void)hipEventDestroy(e);
    delete m;
    if (s) (void)hipStreamDestroy(s);
  });
}

int cpim_gmodel_get_info(const cpim_gmodel* m, cpim_gmodel_info* out) {
  return guarded([&] {
    REQUIRE(m && out, "null argument");
    out->num_vars = m->dm.n;
    out->num_constraints = m->im.num_cons;
    out->num_active = m->dm.num_active;
    out->max_dom_size = m->dm.max_dom;
    out->dom_words = m->dm.W;
    out->bit_dom_int_size = (m->dm.max_dom + 31) / 32;
    out->max_depth = m->max_depth;
    out->subscription_size = m->im.adj_off.empty() ? 0 : m->im.adj_off.back();
    out->device_bytes = m->dm.bytes;
  });
}

}  // extern "C"

// ---------------------------------------------------------------------------
// GAC on the current level
// ---------------------------------------------------------------------------
namespace {

bool fits_lds(const cpim_gmodel* m) { return wg_mem_bytes(m->dm.n, m->dm.W) <= kLdsBudget; }


int knob(const char* name);

// Device wall-clock ticks a one-launch fixpoint (persistent or asynchronous)
// may run before it reports an error: the fixpoint_budget_us knob, or
// kAsyncBudgetMs.
unsigned long long fixpoint_budget_ticks(const cpim_gmodel* m) {
  const long long khz = std::max<long long>(m->props.wall_khz, 1);
  const long long us = knob("fixpoint_budget_us");
  return us > 0 ? (unsigned long long)std::max<long long>(1, khz * us / 1000)
                : (unsigned long long)(khz * kAsyncBudgetMs);
}

unsigned long long slot_sum(const unsigned long long (&v)[kStatSlots]) {
  unsigned long long t = 0;
  for (unsigned long long x : v) t += x;
  return t;
}

// Control block and changed bitmaps cleared.
void gac_start(cpim_gmodel* m, unsigned* F, GacCtl* ctl) {
  const int blocks = (int)std::max<long long>(1, std::min<long long>((3ll * m->nvw + 255) / 256, 1024));
  hipLaunchKernelGGL(k_gac_init, dim3(blocks), dim3(256), 0, m->stream, ctl, F, m->nvw);
  HIPC(hipGetLastError());
}

// Lanes of a grid round: one per word of every arc, words rounded up to a
// power of two, and a wave per table; beyond small tables, a workgroup each up to
// one per CU (30 tables of 20,000 tuples over 200 values, 7.9 ms on two CUs, 5.9
// spread).  With several words a wave takes fewer
// arcs than it has lanes for, down to 16 lanes, as long as there is at most one
// workgroup per CU (`later`: at most the two that a round launches): what a
// wave's arcs settle together is done one after the other (wave_settle).
// Against full waves, us: n=60 d=1024 e=60 t=0.995 785 -> 297, n=100 d=1024
// e=300 t=0.99 345 -> 149, n=300 d=250 e=4000 t=0.96 131 -> 73.  A full round of
// loose relations pays for a second workgroup per CU (n=500 d=250 e=20000 t=0.25
// 20 -> 26); a later round, of the changed variables' arcs only, does not (the
// same at t=0.963 252 -> 235, at t=0.9 after one assignment 330 -> 246).
long long grid_lanes(const cpim_gmodel* m, bool later) {
  const long long arcs = (long long)m->im.adj.size();
  const long long most = (later ? 2ll : 1ll) * std::max(1, m->props.cus) * kRoundThreads;
  long long wp = 1;
  while (wp < m->dm.W) wp *= 2;
  long long lanes = arcs * wp;
  for (int used = 32; wp > 1 && used >= 16 && (later ? lanes : 2 * lanes) <= most; used /= 2) lanes *= 2;
  return std::max({lanes, 64ll * m->dm.ntabs, std::min<long long>(m->im.big_tabs, m->props.cus) * kRoundThreads});
}

// Largest round copy of the persistent fixpoint in LDS: one workgroup per CU.
constexpr long long kPersistentLdsMax = 128 * 1024;

// The persistent fixpoint kernel on the current level, with ctl and F in their
// first state: a lane per arc word, at most one 1024-thread workgroup per CU.
// Every workgroup must be resident for the grid barrier; if some were not, the
// barrier's bounded wait turns that into the time-budget error the caller
// reports (out->err).
void persistent_launch(cpim_gmodel* m, int assigned_var, unsigned* F, GacCtl* ctl, GacResult* out,
                       unsigned long long* seq_at, unsigned long long seq) {
  const int L = m->current_level;
  const long long lanes = grid_lanes(m, false);
  const long long lds = persistent_lds_bytes(m->dm.n, m->dm.W);
  const bool staged = lds <= std::min<long long>(kPersistentLdsMax, m->props.max_lds - 1024);
  const long long want = (lanes + kPersistentThreads - 1) / kPersistentThreads;
  const int grid = (int)std::max<long long>(1, std::min<long long>(want, m->props.cus));
  const long long max_rounds = (long long)m->dm.n * m->dm.max_dom + 2;
  const int mr = (int)std::min<long long>(max_rounds, INT_MAX);
  const unsigned long long max_ticks = fixpoint_budget_ticks(m);
  hipLaunchKernelGGL(staged ? k_gac_persistent<true> : k_gac_persistent<false>, dim3(grid), dim3(kPersistentThreads),
                     staged ? (size_t)lds : 0, m->stream, m->dm.net(), m->level_dom(L), m->level_size(L), F, m->nvw,
                     ctl, mr, assigned_var, assigned_var >= 0 ? 1 : 0, (int)m->im.adj.size(), max_ticks, out, seq_at, seq);
  HIPC(hipGetLastError());
}

void fill_gac_stats(const GacResult& res, int rounds, bool converged, double kms, cpim_gac_stats* st) {
  st->iterations = rounds;
  st->deletions = (int32_t)res.deletions;
  st->inconsistent = res.wipe_round != INT_MAX;
  st->converged = st->inconsistent ? 0 : converged;
  st->revisions = (int64_t)res.revisions;
  st->kernel_ms = kms;
}

// Rounds of a host-driven fixpoint queued before the host looks at their
// outcome: one, then two, four, ... up to this many.  A look costs about 10 us,
// a launch that finds the fixpoint over about 2 us.
constexpr int kRoundsAhead = 8;

// changed: a bitmap of variables to go on from (NULL: starts from assigned_var).
void gac_async(cpim_gmodel* m, int assigned_var, cpim_gac_stats* st, const unsigned* changed = nullptr) {
  const int L = m->current_level;
  u64* dom = m->level_dom(L);
  int* size = m->level_size(L);
  unsigned* F = m->front.as<unsigned>() + async_front(m->nvw);
  const int nfw = m->nfw;
  if (!m->async_ctl.p) m->async_ctl = DevAlloc(sizeof(AsyncCtl));
  AsyncCtl* ctl = m->async_ctl.as<AsyncCtl>();
  m->gac_events();
  HIPC(hipEventRecord(m->gev[0], m->stream));
  // (cleared by a kernel: a copy from the host right after a call that answered
  // in the box first waits for the runtime to see that call's kernel end, some
  // 18 us)
  hipLaunchKernelGGL(k_async_init, dim3(std::min((nfw + 255) / 256, 1024)), dim3(256), 0, m->stream, F, nfw, ctl);
  const int seed_blocks = changed ? (m->dm.n + 255) / 256 : (assigned_var < 0 ? (nfw + 255) / 256 : 1);
  hipLaunchKernelGGL(k_seed_async, dim3(seed_blocks), dim3(256), 0, m->stream, F, nfw, m->dm.num_active,
                     m->dm.adj_off.as<int>(), m->dm.adj.as<int4>(), assigned_var, changed, m->dm.n, ctl);
  HIPC(hipGetLastError());
  // two waves per CU: on the C2 cascade 1024 waves took 5.0-6.0 ms, 512
  // waves 3.8-4.4 ms and 256 waves 4.4-4.9 ms (more waves, more contention on
  // the frontier words and the pending count)
  const int threads = 256;
  const int waves = std::max(1, std::min(nfw, kAsyncWavesPerCu * m->props.cus));
  const int blocks = (waves + threads / 64 - 1) / (threads / 64);
  const unsigned long long max_ticks = fixpoint_budget_ticks(m);
  DevNet net = m->dm.net();
  hipLaunchKernelGGL(k_gac_async, dim3(blocks), dim3(threads), 0, m->stream, net, dom, size, F, nfw, ctl, max_ticks);
  HIPC(hipGetLastError());
  HIPC(hipEventRecord(m->gev[1], m->stream));
  AsyncCtl res{};
  HIPC(hipMemcpyAsync(&res, ctl, sizeof(res), hipMemcpyDeviceToHost, m->stream));
  m->sync();
  st->kernel_ms = m->gac_elapsed_ms();
  if (res.err) fail(CPIM_ERR_RUNTIME, "asynchronous fixpoint exceeded its time budget");
  st->iterations = 1;
  st->deletions = (int32_t)slot_sum(res.deletions);
  st->inconsistent = res.wipe != 0;
  st->converged = !res.wipe && res.pending == 0;
  st->revisions = (int64_t)slot_sum(res.revisions);
}

void gac_block(cpim_gmodel* m, int assigned_var, cpim_gac_stats* st, const unsigned* changed = nullptr) {
  const int L = m->current_level;
  DevNet net = m->dm.net();
  const long long bytes = wg_mem_bytes(m->dm.n, m->dm.W);
  const int threads = 1024;
  const bool tabs = many_tables(m->im, threads);
  HostBox* box = m->box();
  const unsigned long long seq = m->next_seq();
  if (bytes <= kLdsBudget) {
    hipLaunchKernelGGL((tabs ? k_block_gac<true, true> : k_block_gac<true, false>), dim3(1), dim3(threads),
                       (size_t)bytes, m->stream, net, m->level_dom(L), m->level_size(L), assigned_var, changed,
                       (char*)nullptr, &box->gac, &box->seq, seq);
  } else {
    char* scratch = m->get_scratch(bytes);
    hipLaunchKernelGGL((tabs ? k_block_gac<false, true> : k_block_gac<false, false>), dim3(1), dim3(threads), 0,
                       m->stream, net, m->level_dom(L), m->level_size(L), assigned_var, changed, scratch,
                       &box->gac, &box->seq, seq);
  }
  HIPC(hipGetLastError());
  m->wait_box(seq);
  fill_gac_stats(box->gac, 1, box->gac.converged != 0, m->ticks_ms(box->gac.ticks), st);
}

// What AUTO does with a long, narrow cascade: rounds that look like a chain
// (kTailRounds of them, the last ones of at most kTailArcWords arc words) go on
// in one launch.  A round over the grid costs 8 us however little it does, one
// of the workgroup fixpoint 2.5 to 4 us, one of the asynchronous kernel 5 us:
// a path of 1,000 variables 7.6 ms by rounds alone and 2.7 with the workgroup
// fixpoint; of 4,200, seeded, 35 and 23 ms with the asynchronous kernel.
enum class Tail { kNone, kBlock, kAsync };
constexpr int kTailRounds = 31;
constexpr long long kTailArcWords = 1024;  // one turn of a 1024-thread workgroup

// by_variable: a seeded fixpoint keeps a frontier of variables, as the workgroup
// fixpoint does, instead of one of constraints (host-driven rounds only).
void gac_grid(cpim_gmodel* m, int assigned_var, bool persistent, cpim_gac_stats* st, bool by_variable = false,
              Tail tail = Tail::kNone) {
  const int L = m->current_level;
  unsigned* F = m->front.as<unsigned>();
  GacCtl* ctl = m->ctl.as<GacCtl>();
  HostBox* box = m->box();
  if (!m->ctl_ready) gac_start(m, F, ctl);
  m->ctl_ready = false;  // until this fixpoint has put it back
  unsigned long long seq = m->next_seq();
  double kms = 0.0;
  int rounds = 0;
  GacResult res{};
  bool converged = false;
  if (persistent) {
    persistent_launch(m, assigned_var, F, ctl, &box->gac, &box->seq, seq);
    m->wait_box(seq);
    res = box->gac;
    kms = m->ticks_ms(res.ticks);
    if (res.err) fail(CPIM_ERR_RUNTIME, "persistent fixpoint exceeded its time budget at a grid barrier");
    rounds = res.rounds;
    converged = res.converged != 0;
  } else {
    const DevNet net = m->dm.net();
    const long long max_rounds = (long long)m->dm.n * m->dm.max_dom + 2;
    auto blocks = [&](bool later) {
      const long long k = (grid_lanes(m, later) + kRoundThreads - 1) / kRoundThreads;
      return (int)std::max<long long>(1, std::min<long long>(k, 2ll * m->props.cus));
    };
    const int grid[2] = {blocks(false), blocks(true)};
    // each round of a batch answers in a result of its own
    GacResult* answers = reinterpret_cast<GacResult*>(box->data);
    bool over = false, narrow = false;
    for (int r0 = 0, ahead = 1; r0 < max_rounds && !over && !narrow; r0 += ahead, ahead = std::min(2 * ahead, kRoundsAhead)) {
      const int k = (int)std::min<long long>(ahead, max_rounds - r0);
      for (int i = 0; i < k; ++i) {
        if (r0 + i > 0) seq = m->next_seq();
        answers[i].rounds = 0;  // stays 0 if the fixpoint was over before
        hipLaunchKernelGGL(k_gac_round, dim3(grid[r0 + i > 0 ? 1 : 0]), dim3(kRoundThreads), 0, m->stream, net,
                           m->level_dom(L), m->level_size(L), F, m->nvw, ctl, r0 + i, assigned_var,
                           assigned_var >= 0 && !by_variable ? 1 : 0, (int)m->im.adj.size(), &answers[i], &box->seq,
                           seq);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) (void)hipStreamSynchronize(m->stream);  // the rounds queued before answer in the box
        HIPC(e);
      }
      m->wait_box(seq);
      const unsigned long long revisions = res.revisions;
      for (int i = 0; i < k && !over; ++i) {
        if (answers[i].rounds == 0) continue;
        res = answers[i];
        kms += m->ticks_ms(res.ticks);
        rounds = res.rounds;
        converged = res.last_push_round < rounds - 1;
        over = converged || res.wipe_round < rounds;
      }
      narrow = tail != Tail::kNone && !over && rounds >= kTailRounds &&
               (long long)(res.revisions - revisions) * m->dm.W <= kTailArcWords * k;
    }
    if (narrow) {
      cpim_gac_stats rest{};
      const unsigned* changed = F + (long long)(rounds % 3) * m->nvw;  // in the last round
      if (tail == Tail::kBlock) gac_block(m, assigned_var, &rest, changed);
      else gac_async(m, assigned_var, &rest, changed);
      gac_start(m, F, ctl);
      m->ctl_ready = true;
      fill_gac_stats(res, rounds, false, kms, st);
      st->iterations += rest.iterations;
      st->deletions += rest.deletions;
      st->revisions += rest.revisions;
      st->inconsistent = rest.inconsistent;
      st->converged = rest.converged;
      st->kernel_ms += rest.kernel_ms;
      return;
    }
    if (!over) {  // rounds bounded by the number of values: not reached
      m->sync();
      gac_start(m, F, ctl);
    }
  }
  m->ctl_ready = true;
  fill_gac_stats(res, rounds, converged, kms, st);
}

// Constraints times words a domain up to which AUTO takes one workgroup with
// the domains in LDS, and beyond which the host-driven rounds, each spread
// over the grid.  Measured (one workgroup against rounds, us; the root of a
// network whose revisions all find supports / of one that cascades / after
// one assignment): 300 constraints of 20 values 16/23/17 against 14/36/27;
// 1000 of 16 values 23/32/19 against 15/38/31; 1000 of 64 values 24/84/19
// against 15/58/29; 2500 of 16 values 36/57/21 against 16/57/33; 1000 of 200
// values (4 words) 42/708/24 against 16/133/35.  The asynchronous kernel takes
// 165 to 700 us after one assignment where the rounds take 31 to 46 (300 to
// 2000 variables); the persistent kernel is faster still (22 to 34), but needs
// every workgroup resident at once, which AUTO does not ask of a caller with
// several streams.
constexpr long long kAutoBlockWords = 800;
// Constraints up to which a fixpoint that AUTO seeds with one variable keeps a
// frontier of variables (domains that fit in LDS), and beyond which it keeps
// one of constraints.  On a level that is not at its closure the two answer
// differently, so this line stays, whichever kernel runs.
constexpr int kAutoByVariable = 4096;

int auto_gac_mode(const cpim_gmodel* m) {
  return fits_lds(m) && (long long)m->dm.num_active * m->dm.W <= kAutoBlockWords ? CPIM_GAC_BLOCK : CPIM_GAC_PLAIN;
}

void gac(cpim_gmodel* m, int assigned_var, int mode, cpim_gac_stats* st) {
  std::memset(st, 0, sizeof(*st));
  const bool by_variable = mode == CPIM_GAC_AUTO && fits_lds(m) && m->dm.num_active <= kAutoByVariable;
  Tail tail = Tail::kNone;
  if (by_variable) tail = Tail::kBlock;
  else if (mode == CPIM_GAC_AUTO && assigned_var >= 0) tail = Tail::kAsync;
  if (mode == CPIM_GAC_AUTO) mode = auto_gac_mode(m);
  if (m->dm.num_active == 0) {
    st->converged = 1;
    return;
  }
  const int L = m->current_level, before = m->closure[L];
  m->closure[L] = cpim_gmodel::kOpen;
  switch (mode) {
    case CPIM_GAC_PLAIN: gac_grid(m, assigned_var, false, st, by_variable, tail); break;
    case CPIM_GAC_PERSISTENT: gac_grid(m, assigned_var, true, st); break;
    case CPIM_GAC_BLOCK: gac_block(m, assigned_var, st); break;
    case CPIM_GAC_ASYNC: gac_async(m, assigned_var, st); break;
    default: fail(CPIM_ERR_INVALID_ARGUMENT, "unknown GAC mode " + std::to_string(mode));
  }
  m->settled(L, before, assigned_var, *st);
}

void check_var(const cpim_gmodel* m, int var, const char* fn) {
  if (var < 0 || var >= m->dm.n)
    fail(CPIM_ERR_RUNTIME, std::string("[GModel::") + fn + "] Invalid var: " + std::to_string(var));
}

void check_level(const cpim_gmodel* m, int level, const char* fn) {
  if (level < 0 || level >= m->max_depth)
    fail(CPIM_ERR_RUNTIME, std::string("[GModel::") + fn + "] Invalid level: " + std::to_string(level));
}

// Host copy of one level.  Levels that fit the box come through it with one
// launch (larger ones through the runtime's copies).
void read_level(const cpim_gmodel* m, int level, u64* out) {
  const size_t bytes = sizeof(u64) * (size_t)m->level_words();
  if (!m->level_in_box()) {
    HIPC(hipMemcpyAsync(out, m->level_dom(level), bytes, hipMemcpyDeviceToHost, m->stream));
    HIPC(hipStreamSynchronize(m->stream));
    return;
  }
  HostBox* box = m->box();
  const unsigned long long seq = m->next_seq();
  hipLaunchKernelGGL(k_level_get, dim3(1), dim3(1024), 0, m->stream, m->level_dom(level), box->data,
                     (int)m->level_words(), &box->seq, seq);
  HIPC(hipGetLastError());
  m->wait_box(seq);
  std::memcpy(out, box->data, bytes);
}

// Sets one level to the words that fill(words) writes, sizes included.
template <typename Fill>
void write_level(cpim_gmodel* m, int level, Fill&& fill) {
  const int n = m->dm.n, W = m->dm.W;
  m->closure[level] = cpim_gmodel::kOpen;
  if (!m->level_in_box()) {
    std::vector<u64> w((size_t)m->level_words());
    fill(w.data());
    HIPC(hipMemcpyAsync(m->level_dom(level), w.data(), sizeof(u64) * w.size(), hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(k_sizes, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->level_dom(level),
                       m->level_size(level), n, W);
    HIPC(hipGetLastError());
    m->sync();
    return;
  }
  HostBox* box = m->box();
  const unsigned long long seq = m->next_seq();
  fill(reinterpret_cast<u64*>(box->data));
  hipLaunchKernelGGL(k_level_put, dim3(1), dim3(1024), 0, m->stream, reinterpret_cast<const u64*>(box->data),
                     m->level_dom(level), m->level_size(level), n, W, &box->seq, seq);
  HIPC(hipGetLastError());
  m->wait_box(seq);
}

}  // namespace

extern "C" {

int cpim_gmodel_enforce_gac(cpim_gmodel* m, int32_t assigned_var, int32_t mode, cpim_gac_stats* st) {
  return guarded([&] {
    REQUIRE(m && st, "null argument");
    if (assigned_var >= 0) check_var(m, assigned_var, "EnforceGAC");
    DeviceGuard g(m->device);
    gac(m, assigned_var, mode, st);
  });
}


int cpim_gmodel_create_new_level(cpim_gmodel* m, int32_t* new_level) {
  return guarded([&] {
    REQUIRE(m && new_level, "null argument");
    if (m->current_level >= m->max_depth - 1)
      fail(CPIM_ERR_RUNTIME, "[GModel::CreateNewLevel] Max depth reached: " + std::to_string(m->max_depth));
    DeviceGuard g(m->device);
    const int L = ++m->current_level;
    m->closure[L] = m->closure[L - 1];
    if (m->level_in_box()) {
      const unsigned long long seq = m->next_seq();
      hipLaunchKernelGGL(k_level_copy, dim3(1), dim3(1024), 0, m->stream, m->level_dom(L - 1), m->level_dom(L),
                         m->level_size(L - 1), m->level_size(L), m->dm.n, m->dm.W, &m->box()->seq, seq);
      HIPC(hipGetLastError());
      m->wait_box(seq);
    } else {
      HIPC(hipMemcpyAsync(m->level_dom(L), m->level_dom(L - 1), sizeof(u64) * m->level_words(),
                          hipMemcpyDeviceToDevice, m->stream));
      HIPC(hipMemcpyAsync(m->level_size(L), m->level_size(L - 1), sizeof(int) * m->dm.n, hipMemcpyDeviceToDevice,
                          m->stream));
      m->sync();
    }
    *new_level = L;
  });
}

int cpim_gmodel_back_to_level(cpim_gmodel* m, int32_t level) {
  return guarded([&] {
    REQUIRE(m, "null argument");
    if (level < 0 || level >= m->max_depth)
      fail(CPIM_ERR_RUNTIME, "[GModel::BackToLevel] Invalid level: " + std::to_string(level));
    if (level > m->current_level)
      fail(CPIM_ERR_RUNTIME, "[GModel::BackToLevel] Cannot back to future level: " + std::to_string(level) +
                                 " (current=" + std::to_string(m->current_level) + ")");
    m->current_level = level;
    while (m->assigned_size > level) --m->assigned_size;
  });
}

int cpim_gmodel_current_level(const cpim_gmodel* m, int32_t* level) {
  return guarded([&] {
    REQUIRE(m && level, "null argument");
    *level = m->current_level;
  });
}

int cpim_gmodel_assign_value(cpim_gmodel* m, int32_t var, int32_t value, int32_t level, int32_t* ok) {
  return guarded([&] {
    REQUIRE(m && ok, "null argument");
    check_var(m, var, "AssignValue");
    check_level(m, level, "AssignValue");
    if (value < 0 || value >= m->dm.max_dom)
      fail(CPIM_ERR_RUNTIME, "[GModel::AssignValue] Invalid value: " + std::to_string(value));
    DeviceGuard g(m->device);
    m->wrote(level, var);
    m->level_op(kOpAssign, level, var, value);
    m->assigned[level] = make_int2(var, value);
    m->assigned_size = std::max(m->assigned_size, level + 1);
    *ok = 1;
  });
}

int cpim_gmodel_remove_value(cpim_gmodel* m, int32_t var, int32_t value, int32_t level, int32_t* ok) {
  return guarded([&] {
    REQUIRE(m && ok, "null argument");
    check_var(m, var, "RemoveValue");
    check_level(m, level, "RemoveValue");
    *ok = 0;
    if (value < 0 || value >= m->dm.max_dom) return;
    DeviceGuard g(m->device);
    m->wrote(level, var);
    *ok = m->level_op(kOpRemove, level, var, value) > 0;
  });
}

int cpim_gmodel_domain_size(const cpim_gmodel* m, int32_t var, int32_t level, int32_t* size) {
  return guarded([&] {
    REQUIRE(m && size, "null argument");
    check_var(m, var, "GetDomainSize");
    check_level(m, level, "GetDomainSize");
    DeviceGuard g(m->device);
    *size = m->level_op(kOpSize, level, var, 0);
  });
}

int cpim_gmodel_min_domain_var(const cpim_gmodel* m, int32_t level, int32_t* var) {
  return guarded([&] {
    REQUIRE(m && var, "null argument");
    check_level(m, level, "GetMinDomainVar");
    DeviceGuard g(m->device);
    *var = m->level_op(kOpMinVar, level, 0, 0);
  });
}

int cpim_gmodel_is_assigned(const cpim_gmodel* m, int32_t var, int32_t level, int32_t* res) {
  return guarded([&] {
    REQUIRE(m && res, "null argument");
    check_var(m, var, "IsAssigned");
    check_level(m, level, "IsAssigned");
    DeviceGuard g(m->device);
    *res = m->level_op(kOpSize, level, var, 0) == 1;
  });
}

int cpim_gmodel_is_fully_assigned(const cpim_gmodel* m, int32_t level, int32_t* res) {
  return guarded([&] {
    REQUIRE(m && res, "null argument");
    check_level(m, level, "IsFullyAssigned");
    DeviceGuard g(m->device);
    *res = m->level_op(kOpAll, level, 0, 0);
  });
}

int cpim_gmodel_assigned_value(const cpim_gmodel* m, int32_t var, int32_t level, int32_t* value) {
  return guarded([&] {
    REQUIRE(m && value, "null argument");
    check_var(m, var, "GetAssignedValue");
    check_level(m, level, "GetAssignedValue");
    DeviceGuard g(m->device);
    *value = m->level_op(kOpAssigned, level, var, 0);
  });
}

int cpim_gmodel_first_value(const cpim_gmodel* m, int32_t var, int32_t level, int32_t* value) {
  return guarded([&] {
    REQUIRE(m && value, "null argument");
    check_var(m, var, "GetFirstValue");
    check_level(m, level, "GetFirstValue");
    DeviceGuard g(m->device);
    *value = m->level_op(kOpFirst, level, var, 0);
  });
}

int cpim_gmodel_next_value(const cpim_gmodel* m, int32_t var, int32_t value, int32_t level, int32_t* next) {
  return guarded([&] {
    REQUIRE(m && next, "null argument");
    check_var(m, var, "GetNextValue");
    check_level(m, level, "GetNextValue");
    if (value < 0 || value >= m->dm.max_dom - 1) {
      *next = -1;
      return;
    }
    DeviceGuard g(m->device);
    *next = m->level_op(kOpFirst, level, var, value + 1);
  });
}

int cpim_gmodel_read_domains(const cpim_gmodel* m, int32_t level, uint64_t* out) {
  return guarded([&] {
    REQUIRE(m && out, "null argument");
    check_level(m, level, "ReadDomains");
    DeviceGuard g(m->device);
    read_level(m, level, reinterpret_cast<u64*>(out));
  });
}

int cpim_gmodel_weights(cpim_gmodel* m, float* out, int64_t capacity, int64_t* count, int32_t reset) {
  return guarded([&] {
    REQUIRE(m && count, "null argument");
    REQUIRE(capacity >= 0 && (capacity == 0 || out), "null argument");
    DeviceGuard g(m->device);
    const int nc = m->dm.num_active;
    *count = nc;
    if (out && capacity > 0 && nc > 0) {
      const long long k = std::min<long long>(capacity, nc);
      if (m->wdeg_weight.p) {
        HIPC(hipMemcpyAsync(out, m->wdeg_weight.p, sizeof(float) * k, hipMemcpyDeviceToHost, m->stream));
        HIPC(hipStreamSynchronize(m->stream));
      } else {
        for (long long i = 0; i < k; ++i) out[i] = 1.0f;  // no dom/wdeg solve yet
      }
    }
    if (reset && m->wdeg_weight.p) m->wdeg_init();
  });
}

int cpim_gmodel_write_domains(cpim_gmodel* m, int32_t level, const uint64_t* in) {
  return guarded([&] {
    REQUIRE(m && in, "null argument");
    check_level(m, level, "WriteDomains");
    DeviceGuard g(m->device);
    // mask to the domain capacities so that sizes stay exact
    const u64* inw = reinterpret_cast<const u64*>(in);
    write_level(m, level, [&](u64* w) {
      for (int v = 0; v < m->dm.n; ++v)
        for (int j = 0; j < m->dm.W; ++j) {
          const int k = m->im.cap[v] - 64 * j;
          const u64 mask = k >= 64 ? ~0ull : (k <= 0 ? 0ull : ((1ull << k) - 1ull));
          w[(long long)v * m->dm.W + j] = inw[(long long)v * m->dm.W + j] & mask;
        }
    });
  });
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Singleton tests and SAC
// ---------------------------------------------------------------------------
namespace {

// Launch k_singleton_tests over `count` tests: one workgroup per test.  With
// domains in LDS the whole list is one launch; with global scratch the list
// is cut into launches of kScratchBlocks workgroups.
constexpr long long kScratchBlocks = 2048;

void run_singleton_batched(cpim_gmodel* m, const int2* tests_host, long long count, unsigned char* fail_host,
                           cpim_sac_stats* st, SacScratch& S) {
  if (count == 0) return;
  if (count > S.cap) {
    S.tests = DevAlloc(sizeof(int2) * count);
    S.fails = DevAlloc(count);
    S.cap = count;
  }
  if (!S.revs.p) S.revs = DevAlloc(sizeof(unsigned long long) * kStatSlots);  // per-slot counters
  HIPC(hipMemcpyAsync(S.tests.p, tests_host, sizeof(int2) * count, hipMemcpyHostToDevice, m->stream));
  HIPC(hipMemsetAsync(S.revs.p, 0, sizeof(unsigned long long) * kStatSlots, m->stream));
  const int L = m->current_level;
  DevNet net = m->dm.net();
  const long long bytes = wg_mem_bytes(m->dm.n, m->dm.W);
  const int threads = 256;
  const bool tabs = many_tables(m->im, threads);
  S.events();
  HIPC(hipEventRecord(S.ev[0], m->stream));
  if (bytes <= kLdsBudget) {
    for (long long first = 0; first < count; first += INT_MAX) {
      const long long blocks = std::min<long long>(count - first, INT_MAX);
      hipLaunchKernelGGL((tabs ? k_singleton_tests<true, true> : k_singleton_tests<true, false>),
                         dim3((unsigned)blocks), dim3(threads), (size_t)bytes, m->stream, net, m->level_dom(L),
                         m->level_size(L), S.tests.as<int2>(), count, first,
                         S.fails.as<unsigned char>(), S.revs.as<unsigned long long>(), (char*)nullptr, 0ll);
      HIPC(hipGetLastError());
    }
  } else {
    char* scratch = m->get_scratch(bytes * kScratchBlocks);
    for (long long first = 0; first < count; first += kScratchBlocks) {
      const long long blocks = std::min<long long>(count - first, kScratchBlocks);
      hipLaunchKernelGGL((tabs ? k_singleton_tests<false, true> : k_singleton_tests<false, false>),
                         dim3((unsigned)blocks), dim3(threads), 0, m->stream, net,
                         m->level_dom(L), m->level_size(L), S.tests.as<int2>(), count, first,
                         S.fails.as<unsigned char>(), S.revs.as<unsigned long long>(), scratch, bytes);
      HIPC(hipGetLastError());
    }
  }
  HIPC(hipEventRecord(S.ev[1], m->stream));
  HIPC(hipMemcpyAsync(fail_host, S.fails.p, count, hipMemcpyDeviceToHost, m->stream));
  unsigned long long revs_slots[kStatSlots];
  HIPC(hipMemcpyAsync(revs_slots, S.revs.p, sizeof(revs_slots), hipMemcpyDeviceToHost, m->stream));
  m->sync();
  const unsigned long long revs = slot_sum(revs_slots);
  float ms = 0.f;
  HIPC(hipEventElapsedTime(&ms, S.ev[0], S.ev[1]));
  st->kernel_ms += ms;
  st->revisions += (int64_t)revs;
  st->singleton_tests += count;
}

// Bit-sliced path: tests sorted by variable and cut into groups of at most
// 64 (a variable with more values is split into balanced groups; small
// variables share a group), one workgroup per group.  The slices of the
// resident groups take n * dpad words each, within kSliceBudgetBytes.
// ---------------------------------------------------------------------------
// Tuning knobs (cpim_tune_set / cpim_tune_get), process-wide; 0 = automatic.
// Their first values come from the environment.
// ---------------------------------------------------------------------------
struct Knob {
  const char* name;
  const char* env;
  std::atomic<int> value;
  bool loaded;
};
Knob g_knobs[] = {
    {"sac_slice_masks", "CPIM_SLICE_MASKS", {0}, false},
    {"sac_slice_threads", "CPIM_SLICE_THREADS", {0}, false},
    {"sac_slice_kernel", "CPIM_SLICE_KERNEL", {0}, false},
    {"unit_threads", "CPIM_UNIT_THREADS", {0}, false},
    {"sac_slice_nibbles", "CPIM_SLICE_NIBBLES", {0}, false},
    {"mac_lds_net", "CPIM_MAC_LDS_NET", {0}, false},
    {"fixpoint_budget_us", "CPIM_FIXPOINT_BUDGET_US", {0}, false},
    {"sac_slice_bytes", "CPIM_SLICE_BYTES", {0}, false},
};
std::mutex g_knob_mu;

bool knob_valid(const char* name, long long v) {
  const std::string k(name);
  if (k == "sac_slice_masks") return v == 0 || v == 1 || v == 2 || v == 4;
  if (k == "sac_slice_kernel") return v == 0 || v == 1;
  if (k == "sac_slice_nibbles") return v == 0 || v == 1 || v == 2;
  if (k == "sac_slice_bytes") return v == 0 || v == 1 || v == 4 || v == 6;
  if (k == "mac_lds_net") return v == 0 || v == 1;
  if (k == "fixpoint_budget_us") return v >= 0 && v <= 600000000ll;
  return v == 0 || (v >= 64 && v <= 1024 && v % 64 == 0);
}

Knob* find_knob(const char* name) {
  for (Knob& k : g_knobs)
    if (std::strcmp(k.name, name) == 0) {
      std::lock_guard<std::mutex> lock(g_knob_mu);
      if (!k.loaded) {
        const char* e = std::getenv(k.env);
        const long long v = e ? std::atoll(e) : 0;
        k.value = knob_valid(name, v) ? (int)v : 0;
        k.loaded = true;
      }
      return &k;
    }
  return nullptr;
}

int knob(const char* name) { return find_knob(name)->value.load(); }

// Bit-sliced singleton tests.  Two kernels: k_sliced_wide<M> (default: 64 M
// tests per workgroup, one shared stage per changed variable) and
// k_sliced_tests (64 tests, one stage per wave; sac_slice_kernel = 1).
constexpr int kSliceThreads = 512;

int slice_threads() {
  const int t = knob("sac_slice_threads");
  return t ? t : kSliceThreads;
}
constexpr long long kSliceBudgetBytes = 4ll << 30;

// Threads per workgroup for this network: the configured size, halved while
// the per-wave staging areas exceed the LDS budget (0 if even one wave does not fit).
int slice_threads_for(const cpim_gmodel* m) {
  int t = slice_threads();
  while (t > 64 && slice_lds_bytes(m->dm.n, m->dm.dpad, t / 64) > kLdsBudget) t /= 2;
  return slice_lds_bytes(m->dm.n, m->dm.dpad, t / 64) <= kLdsBudget ? t : 0;
}

// Masks per (variable, value) of the wide kernel: sac_slice_masks, or 4 when
// the tests fill a workgroup of 256 per CU, 2 when 128 do, else 1; halved
// while the LDS image does not fit (0 if M = 1 does not).
int wide_masks_for(const cpim_gmodel* m, long long count) {
  int M = knob("sac_slice_masks");
  if (M == 0) {
    const long long cus = std::max(1, m->props.cus);
    M = count >= 256 * cus ? 4 : (count >= 128 * cus ? 2 : 1);
  }
  while (M > 1 && wide_lds_bytes(m->dm.n, m->dm.W, M) > kLdsBudget) M /= 2;
  return wide_lds_bytes(m->dm.n, m->dm.W, M) <= kLdsBudget ? M : 0;
}

bool use_wide_kernel() { return knob("sac_slice_kernel") == 0; }

// Nibble tables (sac_slice_nibbles: 0 auto = on when their LDS image stays
// within 80 KB, two workgroups per CU; 1 on when it fits; 2 off).
bool use_nibble_tables(const cpim_gmodel* m, int M) {
  const int k = knob("sac_slice_nibbles");
  if (k == 2) return false;
  const long long b = wide_lds_bytes(m->dm.n, m->dm.W, M, true);
  return b <= (k == 1 ? (long long)m->props.max_lds : std::min<long long>(m->props.max_lds, 80 * 1024));
}

// Byte tables in front of the nibble tables (sac_slice_bytes: 4 or 6 = that
// many whenever the single stage buffer fits; 0 and 1 = none).
int byte_tables_for(const cpim_gmodel* m, int M, bool nib) {
  const int k = knob("sac_slice_bytes");
  if (!nib || k <= 1) return 0;
  const long long limit = k ? (long long)m->props.max_lds : std::min<long long>(m->props.max_lds, 80 * 1024);
  for (int nb : {6, 4})
    if ((k == 0 || k == nb) && wide_lds_bytes(m->dm.n, m->dm.W, M, true, nb) <= limit) return nb;
  return 0;
}

bool sliced_eligible(const cpim_gmodel* m) {
  if ((int)m->im.bin_cons.size() != m->im.num_active) return false;
  return use_wide_kernel() ? wide_masks_for(m, 1) > 0 : slice_threads_for(m) > 0;
}

void run_singleton_sliced(cpim_gmodel* m, const int2* tests_host, long long count, unsigned char* fail_host,
                          cpim_sac_stats* st, SacScratch& S) {
  if (count == 0) return;
  REQUIRE(count <= INT_MAX, "too many singleton tests for one call");
  // Tests are grouped by variable: a list sorted by variable (every SAC pass)
  // needs no sort.  The check has no early exit, so that it vectorizes.
  int descents = 0;
  for (long long i = 1; i < count; ++i) descents |= tests_host[i].x < tests_host[i - 1].x;
  bool sorted_in = descents == 0;
  std::vector<int> order;
  std::vector<int2> sorted_buf;
  const int2* sorted = tests_host;
  if (!sorted_in) {
    order.resize((size_t)count);
    for (long long i = 0; i < count; ++i) order[(size_t)i] = (int)i;
    std::stable_sort(order.begin(), order.end(),
                     [&](int a, int b) { return tests_host[a].x < tests_host[b].x; });
    sorted_buf.resize((size_t)count);
    for (long long i = 0; i < count; ++i) sorted_buf[(size_t)i] = tests_host[order[(size_t)i]];
    sorted = sorted_buf.data();
  }
  const bool wide = use_wide_kernel();
  const int M = wide ? wide_masks_for(m, count) : 1;
  const bool nib = wide && use_nibble_tables(m, M);
  const int nb = wide ? byte_tables_for(m, M, nib) : 0;
  REQUIRE(M > 0, "bit-sliced singleton tests do not fit in LDS");
  const long long cap = 64ll * M;  // tests per workgroup
  std::vector<int> gfirst;
  std::vector<long long> w;  // expected work of each group: summed degree of its variables
  gfirst.reserve((size_t)(count / 32 + 2));
  w.reserve((size_t)(count / 32 + 2));
  int open = -1;  // start of the group being filled, -1 if none
  for (long long i = 0; i < count;) {
    // end j of the run of x: gallop, then bisect (the list is sorted)
    const int x = sorted[i].x;
    long long lo = i, step = 1;
    while (lo + step < count && sorted[lo + step].x == x) {
      lo += step;
      step *= 2;
    }
    long long hi = std::min(count, lo + step);  // sorted[hi].x != x, or hi == count
    while (hi - lo > 1) {
      const long long mid = lo + (hi - lo) / 2;
      if (sorted[mid].x == x) lo = mid;
      else hi = mid;
    }
    const long long j = hi;
    const long long len = j - i;
    const long long dx = m->im.adj_off[x + 1] - m->im.adj_off[x];
    if (len > cap) {
      open = -1;
      const long long k = (len + cap - 1) / cap;
      for (long long p = 0; p < k; ++p) {
        gfirst.push_back((int)(i + len * p / k));
        w.push_back(dx);
      }
    } else if (open < 0 || i + len - open > cap) {
      gfirst.push_back((int)i);
      w.push_back(dx);
      open = (int)i;
    } else {
      w.back() += dx;
    }
    i = j;
  }
  const long long groups = (long long)gfirst.size();
  gfirst.push_back((int)count);
  // Place the groups on workgroups by expected work.  The pass runs as one
  // wave of workgroups, two per CU; workgroups bid and bid + cus share a CU
  // (dispatch fills one slot per CU, then the second).  The heaviest groups
  // (by the summed degree of their variables) get the CUs that hold a single
  // workgroup, and every other heavy group shares its CU with a light one, so
  // that the kernel does not wait on two heavy groups sharing a CU.  With more
  // groups than slots, heavy groups go first.  (C3: 8.1 -> 7.1 ms per pass.)
  // The kernel reads the group of each slot from gorder; the test list keeps
  // its order.
  std::vector<int> gorder;
  if (wide && groups > 1 && groups <= kSliceBudgetBytes / (8ll * m->dm.n * m->dm.dpad * M)) {
    const int cus = std::max(1, m->props.cus);
    std::vector<int> rank((size_t)groups);
    for (long long g = 0; g < groups; ++g) rank[(size_t)g] = (int)g;
    std::stable_sort(rank.begin(), rank.end(), [&](int a, int b) { return w[(size_t)a] > w[(size_t)b]; });
    const int B = (int)groups;
    std::vector<int> at_bid(rank);  // more than two per CU, or one: heaviest first
    if (B > cus && B <= 2 * cus) {
      int next = 0;
      for (int k = B - cus; k < cus; ++k) at_bid[(size_t)k] = rank[(size_t)next++];
      for (int k = 0; k < B - cus; ++k) {
        at_bid[(size_t)k] = rank[(size_t)(next + k)];
        at_bid[(size_t)(k + cus)] = rank[(size_t)(B - 1 - k)];
      }
    }
    // the kernel takes slot gi = xcd * q + min(xcd, rem) + (bid >> 3) for bid
    const int q = B >> 3, rem = B & 7;
    gorder.resize((size_t)B);
    for (int bid = 0; bid < B; ++bid) {
      const int xcd = bid & 7;
      gorder[(size_t)(xcd * q + (xcd < rem ? xcd : rem) + (bid >> 3))] = at_bid[(size_t)bid];
    }
  }
  if (count > S.scap) {
    S.stests = DevAlloc(sizeof(int2) * count);
    S.perm = DevAlloc(sizeof(int) * count);
    S.scap = count;
  }
  if (count > S.cap) {
    S.fails = DevAlloc(count);
    S.tests = DevAlloc(sizeof(int2) * count);
    S.cap = count;
  }
  if (groups + 1 > S.gcap) {
    S.gfirst = DevAlloc(sizeof(int) * (groups + 1));
    S.gorder = DevAlloc(sizeof(int) * (groups + 1));
    S.gcap = groups + 1;
  }
  if (!S.revs.p) S.revs = DevAlloc(sizeof(unsigned long long) * kStatSlots);  // per-slot counters
  S.events();
  HIPC(hipMemcpyAsync(S.stests.p, sorted, sizeof(int2) * count, hipMemcpyHostToDevice, m->stream));
  if (!sorted_in)
    HIPC(hipMemcpyAsync(S.perm.p, order.data(), sizeof(int) * count, hipMemcpyHostToDevice, m->stream));
  HIPC(hipMemcpyAsync(S.gfirst.p, gfirst.data(), sizeof(int) * (groups + 1), hipMemcpyHostToDevice, m->stream));
  if (!gorder.empty())
    HIPC(hipMemcpyAsync(S.gorder.p, gorder.data(), sizeof(int) * gorder.size(), hipMemcpyHostToDevice, m->stream));
  const int* go = gorder.empty() ? nullptr : S.gorder.as<int>();
  HIPC(hipMemsetAsync(S.revs.p, 0, sizeof(unsigned long long) * kStatSlots, m->stream));
  const long long slice_bytes = 8ll * m->dm.n * m->dm.dpad * M;
  const long long per_launch = std::max<long long>(1, std::min<long long>(groups, kSliceBudgetBytes / slice_bytes));
  u64* slices = nullptr;
  if (wide) {
    if (slice_bytes * per_launch > S.dead_bytes) {
      S.dead = DevAlloc((size_t)(slice_bytes * per_launch));
      S.dead_bytes = slice_bytes * per_launch;
      HIPC(hipMemsetAsync(S.dead.p, 0, (size_t)S.dead_bytes, m->stream));
    }
    slices = S.dead.as<u64>();
  } else {
    slices = reinterpret_cast<u64*>(m->get_scratch(slice_bytes * per_launch));
  }
  const int L = m->current_level;
  DevNet net = m->dm.net();
  int threads = 0;
  size_t lds = 0;
  if (wide) {
    // 16 waves from 128 tests up, 8 below; at least one thread per test, at
    // most the kernel's launch bound
    threads = knob("sac_slice_threads") ? knob("sac_slice_threads") : (M >= 2 ? 1024 : 512);
    threads = std::min(std::max(threads, 64 * M), kWideMaxThreads);
    lds = (size_t)wide_lds_bytes(m->dm.n, m->dm.W, M, nib, nb);
  } else {
    threads = slice_threads_for(m);
    lds = (size_t)slice_lds_bytes(m->dm.n, m->dm.dpad, threads / 64);
  }
  const int* perm = sorted_in ? nullptr : S.perm.as<int>();
  HIPC(hipEventRecord(S.ev[0], m->stream));
  for (long long g0 = 0; g0 < groups; g0 += per_launch) {
    const long long blocks = std::min(per_launch, groups - g0);
    const dim3 grid((unsigned)blocks), block(threads);
    const u64* base = m->level_dom(L);
    const int2* tl = S.stests.as<int2>();
    const int* gf = S.gfirst.as<int>();
    unsigned char* fl = S.fails.as<unsigned char>();
    unsigned long long* rv = S.revs.as<unsigned long long>();
    if (!wide) hipLaunchKernelGGL(k_sliced_tests, grid, block, lds, m->stream, net, base, tl, gf, g0, perm, fl, rv, slices);
#define CPIM_WIDE(MM, NIB, NB) \
  hipLaunchKernelGGL((k_sliced_wide<MM, NIB, NB>), grid, block, lds, m->stream, net, base, tl, gf, go, g0, perm, fl, rv, slices)
#define CPIM_WIDE_M(MM)                                \
  {                                                    \
    if (nb == 6) CPIM_WIDE(MM, true, 6);               \
    else if (nb == 4) CPIM_WIDE(MM, true, 4);          \
    else if (nib) CPIM_WIDE(MM, true, 0);              \
    else CPIM_WIDE(MM, false, 0);                      \
  }
    else if (M == 1) CPIM_WIDE_M(1)
    else if (M == 2) CPIM_WIDE_M(2)
    else CPIM_WIDE_M(4)
#undef CPIM_WIDE_M
#undef CPIM_WIDE
    HIPC(hipGetLastError());
  }
  HIPC(hipEventRecord(S.ev[1], m->stream));
  HIPC(hipMemcpyAsync(fail_host, S.fails.p, count, hipMemcpyDeviceToHost, m->stream));
  unsigned long long revs_slots[kStatSlots];
  HIPC(hipMemcpyAsync(revs_slots, S.revs.p, sizeof(revs_slots), hipMemcpyDeviceToHost, m->stream));
  m->sync();
  const unsigned long long revs = slot_sum(revs_slots);
  float ms = 0.f;
  HIPC(hipEventElapsedTime(&ms, S.ev[0], S.ev[1]));
  st->kernel_ms += ms;
  st->revisions += (int64_t)revs;
  st->singleton_tests += count;
}

void run_singleton_plain(cpim_gmodel* m, const int2* tests, long long count, unsigned char* fail_host,
                         cpim_sac_stats* st);

// CPIM_SAC_BATCHED: one workgroup per test for networks with tables and where
// the estimates below say so, the bit-sliced kernels otherwise.  Both estimates
// are of a pass without cascades, in microseconds:
//  * workgroups: as many turns of the resident workgroups as the tests take,
//    each about 18 plus its arc words in two rounds (`reach`);
//  * bit-sliced: the variables that a group of 64 M tests changes, walked one
//    after another, about 8 each; where one variable has far more constraints
//    than the others (a star), the group that tests it walks that many.
// With cascades a bit-sliced group walks every variable that any of its tests
// changes, and workgroups win up to some 24 x 2^20 arc words (n=480 d=256 e=4800
// t=0.887, 215M: 276 against 30 ms; n=300 d=100 e=3000 t=0.826, 26M: 25.5
// against 33.5 ms).  A variable whose neighbour kept p d values loses a value to
// it with probability (1 - p)^(p d); 50 values lost to deg neighbours are the
// line (24 lost at n=300 d=64 e=1000 t=0.80, 965 against 631 us; 73 at t=0.84,
// 1350 against 4026 us); beyond 10 turns one loss a value is asked as well
// (n=150 d=200 e=300, 14.6 turns: 0.9 lost at t=0.916, 1396 against 947 us; 2.3
// at t=0.948, 6200 against 11868).
// A long chain (a path, a lattice) takes about as many rounds as it changes
// variables, and every turn of workgroups pays for all of them: there a group's
// variables, times the arcs within reach over a path's six (with cascades arc
// words over three), must outnumber the turns.  Measured, workgroups against bit-sliced, us:
//   n=60 d=37 e=500      88 / 173, cascading 330 / 2899
//   n=120 d=50 e=3570   309 / 761      n=200 d=64 e=4000   379 / 503
//   n=100 d=100 e=1500  347 / 421      n=500 d=16 e=3000   171 / 342
//   n=200 d=64 e=800    182 / 157, cascading 1572 / 5611
//   n=60 d=300 e=300    427 / 341, cascading 6686 / 26152
//   n=40 d=1000 e=100   cascading 44416 / 119273
//   n=100 d=128 e=600   215 / 199      n=200 d=128 e=2000  616 / 398
//   star n=600 d=64     684 / 1309     star n=2000 d=64    6977 / 5211
//   path n=60 d=37      495 / 355      path n=700 d=64     148098 / 8566
//   lattice 25x25 d=16  196 / 242      lattice 25x25 d=40  608 / 216
bool tests_by_workgroup(const cpim_gmodel* m, long long tests) {
  const long long bytes = wg_mem_bytes(m->dm.n, m->dm.W);
  if (bytes > kLdsBudget) return false;
  const double cus = std::max(1, m->props.cus), W = m->dm.W, d = m->dm.max_dom;
  const double per_cu = (double)std::min<long long>(8, std::max<long long>(1, m->props.max_lds / (bytes + 512)));
  const double turns = (double)tests / (cus * per_cu);
  const int M = std::max(1, wide_masks_for(m, tests));
  const double deg = (double)m->im.adj.size() / m->dm.n;
  const double vars = std::max(1.0, 64.0 * M / d);
  const double waves = std::max(1.0, std::ceil((double)tests / (64.0 * M * 2.0 * cus)));
  const double by_wg = turns * (18.0 + m->im.reach * W / 50.0);
  const double sliced = waves * (vars * (1.0 + deg) * (7.5 + 0.5 * W) + 2.5 * (m->im.max_deg - deg));
  const double p = m->im.density, lost = deg * std::pow(1.0 - p, p * d);  // of a value's chances, by all neighbours
  const bool cascades = (double)tests * m->im.reach * W <= (double)(24ll << 20) && d * lost >= 50.0 &&
                        (turns <= 10.0 || lost >= 1.0);
  const double spread = cascades ? m->im.reach * W / 3.0 : m->im.reach / 6.0;
  return (cascades || by_wg <= sliced) && 1.6 * turns <= vars * std::max(1.0, spread);
}

void run_singleton_device(cpim_gmodel* m, int mode, const int2* tests, long long count, unsigned char* fail_out,
                          cpim_sac_stats* st, SacScratch& S) {
  // (on an open level the two kernels answer differently: a bit-sliced test
  // sees what the other tests of its group revise, so it stays the choice there)
  const bool closed = m->closure[m->current_level] == cpim_gmodel::kClosed;
  if (mode == CPIM_SAC_BATCHED)
    mode = sliced_eligible(m) && !(closed && tests_by_workgroup(m, count)) ? CPIM_SAC_SLICED : CPIM_SAC_WORKGROUP;
  if (mode == CPIM_SAC_SLICED) {
    if (!sliced_eligible(m))
      fail(CPIM_ERR_UNSUPPORTED, "bit-sliced singleton tests need a binary network whose work lists fit in LDS");
    run_singleton_sliced(m, tests, count, fail_out, st, S);
  } else if (mode == CPIM_SAC_WORKGROUP) {
    run_singleton_batched(m, tests, count, fail_out, st, S);
  } else {
    run_singleton_plain(m, tests, count, fail_out, st);
  }
}

// One host-driven fixpoint per test on a scratch level: copy the level,
// reduce x to {a}, seed the constraints of x, rounds as in gac_grid.
void run_singleton_plain(cpim_gmodel* m, const int2* tests, long long count, unsigned char* fail_host,
                         cpim_sac_stats* st) {
  const int L = m->current_level;
  if (L + 1 >= m->max_depth) fail(CPIM_ERR_RUNTIME, "no free level for singleton tests");
  const int T = L + 1;
  m->closure[T] = cpim_gmodel::kOpen;
  const long long t0 = now_ns();
  std::vector<u64> word(m->dm.W);
  const int one = 1;
  for (long long i = 0; i < count; ++i) {
    const int x = tests[i].x, a = tests[i].y;
    HIPC(hipMemcpyAsync(m->level_dom(T), m->level_dom(L), sizeof(u64) * m->level_words(),
                        hipMemcpyDeviceToDevice, m->stream));
    HIPC(hipMemcpyAsync(m->level_size(T), m->level_size(L), sizeof(int) * m->dm.n, hipMemcpyDeviceToDevice,
                        m->stream));
    std::fill(word.begin(), word.end(), 0ull);
    word[a >> 6] = 1ull << (a & 63);
    HIPC(hipMemcpyAsync(m->level_dom(T) + (long long)x * m->dm.W, word.data(), sizeof(u64) * m->dm.W,
                        hipMemcpyHostToDevice, m->stream));
    HIPC(hipMemcpyAsync(m->level_size(T) + x, &one, sizeof(int), hipMemcpyHostToDevice, m->stream));
    m->current_level = T;
    cpim_gac_stats gs;
    std::memset(&gs, 0, sizeof(gs));
    try {
      gac_grid(m, x, false, &gs);
    } catch (...) {
      m->current_level = L;
      throw;
    }
    m->current_level = L;
    fail_host[i] = gs.inconsistent ? 1 : 0;
    st->revisions += gs.revisions;
  }
  st->kernel_ms += (now_ns() - t0) * 1e-6;
  st->singleton_tests += count;
}

std::vector<int2> all_tests(cpim_gmodel* m, const std::vector<u64>& dom) {
  std::vector<int2> t;
  for (int v = 0; v < m->dm.n; ++v)
    for (int a = 0; a < m->im.cap[v]; ++a)
      if ((dom[(long long)v * m->dm.W + (a >> 6)] >> (a & 63)) & 1ull) t.push_back(make_int2(v, a));
  return t;
}

}  // namespace

extern "C" {

int cpim_tune_set(const char* name, int64_t value) {
  return guarded([&] {
    REQUIRE(name, "null argument");
    Knob* k = find_knob(name);
    REQUIRE(k, "unknown tuning knob");
    REQUIRE(knob_valid(name, value), "value out of range for this knob");
    k->value = (int)value;
  });
}

int cpim_tune_get(const char* name, int64_t* value) {
  return guarded([&] {
    REQUIRE(name && value, "null argument");
    Knob* k = find_knob(name);
    REQUIRE(k, "unknown tuning knob");
    *value = k->value.load();
  });
}

int cpim_gmodel_singleton_tests(cpim_gmodel* m, const int32_t* tests, int64_t count, int32_t mode, uint8_t* fail_out,
                                cpim_sac_stats* st) {
  return guarded([&] {
    REQUIRE(m && st && (count == 0 || (tests && fail_out)), "null argument");
    REQUIRE(count >= 0, "negative test count");
    DeviceGuard g(m->device);
    std::memset(st, 0, sizeof(*st));
    const int2* t = reinterpret_cast<const int2*>(tests);
    for (long long i = 0; i < count; ++i) {
      REQUIRE(t[i].x >= 0 && t[i].x < m->dm.n, "test names an unknown variable");
      REQUIRE(t[i].y >= 0 && t[i].y < m->im.cap[t[i].x], "test value outside the domain");
    }
    REQUIRE(mode >= CPIM_SAC_BATCHED && mode <= CPIM_SAC_SLICED, "unknown singleton-test mode");
    SacScratch& S = m->sac;
    run_singleton_device(m, mode, t, count, fail_out, st, S);
    st->consistent = 1;
    st->passes = 1;
  });
}

// SAC closure by passes: every singleton test of the current domains (one
// batched launch), removal of the failed values, GAC from the variables that
// lost values, until a pass removes nothing.  The closure is unique, so the
// result equals SAC1::enforce (src/SAC1.cpp:57-103).
int cpim_gmodel_enforce_sac(cpim_gmodel* m, int32_t mode, cpim_sac_stats* st) {
  return guarded([&] {
    REQUIRE(m && st, "null argument");
    REQUIRE(mode >= CPIM_SAC_BATCHED && mode <= CPIM_SAC_SLICED, "unknown SAC mode");
    DeviceGuard g(m->device);
    std::memset(st, 0, sizeof(*st));
    const int L = m->current_level;
    cpim_gac_stats gs;
    gac(m, -1, CPIM_GAC_AUTO, &gs);
    st->revisions += gs.revisions;
    if (gs.inconsistent) {
      st->consistent = 0;
      return;
    }
    SacScratch& S = m->sac;
    while (true) {
      std::vector<u64> dom((size_t)m->level_words());
      read_level(m, L, dom.data());
      std::vector<int2> tests = all_tests(m, dom);
      std::vector<unsigned char> fl(tests.size(), 0);
      run_singleton_device(m, mode, tests.data(), (long long)tests.size(), fl.data(), st, S);
      ++st->passes;
      long long removed = 0;
      for (size_t i = 0; i < tests.size(); ++i)
        if (fl[i]) {
          dom[(long long)tests[i].x * m->dm.W + (tests[i].y >> 6)] &= ~(1ull << (tests[i].y & 63));
          ++removed;
        }
      if (removed == 0) break;
      st->removed += removed;
      // a variable whose every value failed its singleton test has an empty
      // domain: that is a wipe-out even if no constraint reaches it
      bool empty = false;
      for (int v = 0; v < m->dm.n && !empty; ++v) {
        u64 any = 0;
        for (int w = 0; w < m->dm.W; ++w) any |= dom[(long long)v * m->dm.W + w];
        empty = any == 0;
      }
      write_level(m, L, [&](u64* w) { std::memcpy(w, dom.data(), sizeof(u64) * dom.size()); });
      if (empty) {
        st->consistent = 0;
        return;
      }
      gac(m, -1, CPIM_GAC_AUTO, &gs);
      st->revisions += gs.revisions;
      if (gs.inconsistent) {
        st->consistent = 0;
        return;
      }
    }
    st->consistent = 1;
  });
}

// ---------------------------------------------------------------------------
// Device MAC
// ---------------------------------------------------------------------------
int cpim_gmodel_solve(cpim_gmodel* m, const cpim_solve_opts* opts, cpim_search_stats* st, int32_t* solution,
                      cpim_node_record* trace, int32_t* trace_len) {
  return guarded([&] {
    REQUIRE(m && st, "null argument");
    cpim_solve_opts o{};
    if (opts) o = *opts;
    REQUIRE(o.branching == CPIM_BRANCH_BINARY, "the device solver implements binary branching only");
    REQUIRE(o.var_heuristic == CPIM_VARH_DOM_MIN || o.var_heuristic == CPIM_VARH_DOM_DEG ||
                o.var_heuristic == CPIM_VARH_DOM_WDEG,
            "unknown variable heuristic");
    REQUIRE(o.reserved == 0, "cpim_solve_opts.reserved must be 0");
    REQUIRE(o.trace_capacity >= 0, "negative trace capacity");
    REQUIRE(o.trace_capacity == 0 || trace, "trace buffer is null");
    REQUIRE(o.max_solutions >= 0 && o.solution_capacity >= 0, "negative solution count");
    REQUIRE(m->current_level == 0, "the device solver starts from level 0");
    DeviceGuard g(m->device);
    std::memset(st, 0, sizeof(*st));
    m->closure[0] = cpim_gmodel::kOpen;  // until the root closure is back
    const int n = m->dm.n;
    const long long t0 = now_ns();
    const long long sol_cap = std::max<long long>(1, o.solution_capacity);
    DevAlloc state(sizeof(MacState)), stack(sizeof(int2) * n), sol(sizeof(int) * n * sol_cap);
    // the search keeps its depth-0 trail in level 0 and rewrites it when it
    // backtracks at the root; level 0 gets the root closure back afterwards,
    // as the reference leaves it (GModelSolver::Solve runs EnforceGAC on
    // level 0 and searches on the levels above)
    DevAlloc root(sizeof(u64) * m->level_words());
    DevAlloc tr(sizeof(NodeRec) * std::max(1, o.trace_capacity));
    MacState s0{};
    s0.status = MAC_INIT;
    HIPC(hipMemcpyAsync(state.p, &s0, sizeof(s0), hipMemcpyHostToDevice, m->stream));
    MacArgs A{};
    A.state = state.as<MacState>();
    A.trail = m->level_dom(0);
    A.stack = stack.as<int2>();
    A.solution = sol.as<int>();
    A.sol_cap = sol_cap;
    A.max_solutions = o.max_solutions;
    A.trace = o.trace_capacity > 0 ? tr.as<NodeRec>() : nullptr;
    A.trace_cap = o.trace_capacity;
    A.node_limit = o.node_limit;
    A.step_budget = 0;
    A.deadline = 0;
    A.root_out = root.as<u64>();
    A.nbr = o.var_heuristic == CPIM_VARH_DOM_DEG ? m->dm.nbr.as<int>() : nullptr;
    if (o.var_heuristic == CPIM_VARH_DOM_WDEG) {
      if (!m->wdeg_weight.p) m->wdeg_init();
      A.weight = m->wdeg_weight.as<float>();
      A.stamp_tab = m->wdeg_stamp.as<int>();
    }
    DevNet net = m->dm.net();
    const long long bytes = wg_mem_bytes(n, m->dm.W);
    hipEvent_t e0, e1;
    HIPC(hipEventCreate(&e0));
    HIPC(hipEventCreate(&e1));
    HIPC(hipEventRecord(e0, m->stream));
    // Every launch runs a bounded number of nodes (so no launch can run for
    // long); the search state stays on the device between launches and the
    // host checks the time limit in between.
    A.step_budget = kNodesPerLaunch;
    MacState s{};
    // The network image goes to LDS too when it fits beside the domains.
    LdsNet lnet{};
    if (knob("mac_lds_net") == 0 && m->dm.lnet.bytes > 0 &&
        bytes + m->dm.lnet.bytes <= (long long)m->props.max_lds - 2048)
      lnet = m->dm.lnet;
    const bool lds = bytes <= kLdsBudget;
    const int threads = lds && lnet.flat_min && !A.weight ? lnet.flat_threads : 1024;
    long long dyn = lds ? bytes + lnet.bytes : 0;
    if (A.weight && dyn + 16 + 4ll * m->dm.num_active <= (long long)m->props.max_lds - 2048) {
      A.stamp_off = (int)std::max(16ll, dyn);  // 0 means memory
      dyn = A.stamp_off + 4ll * m->dm.num_active;
    }
    while (true) {
      char* scratch = lds ? nullptr : m->get_scratch(bytes);
      auto* kernel = lds ? (A.weight ? k_mac<true, true, false> : k_mac<true, false, false>)
                         : (A.weight ? k_mac<false, true, false> : k_mac<false, false, false>);
      if ((!lds || lnet.bytes == 0) && full_search(m->im, threads))
        kernel = lds ? (A.weight ? k_mac<true, true, true> : k_mac<true, false, true>)
                     : (A.weight ? k_mac<false, true, true> : k_mac<false, false, true>);
      hipLaunchKernelGGL(kernel, dim3(1), dim3(threads), (size_t)dyn, m->stream, net, A, scratch, lds ? lnet : LdsNet{});
      HIPC(hipGetLastError());
      HIPC(hipMemcpyAsync(&s, state.p, sizeof(s), hipMemcpyDeviceToHost, m->stream));
      m->sync();
      if (s.status != MAC_RUNNING) break;
      if (o.time_limit_ms > 0 && (now_ns() - t0) / 1000000 > o.time_limit_ms) {
        st->time_out = 1;
        break;
      }
    }
    HIPC(hipEventRecord(e1, m->stream));
    HIPC(hipEventSynchronize(e1));
    float ms = 0.f;
    HIPC(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    st->num_positive = s.npos;
    st->num_negative = s.nneg;
    st->num_solutions = s.nsol;
    st->unsolvable = s.status == MAC_UNSAT && s.nsol == 0;
    if (s.status == MAC_LIMIT) st->time_out = 1;
    st->gac_iterations = s.npos + s.nneg + 1;
    st->solve_time = (now_ns() - t0) * 1e-9;
    st->gac_time = ms * 1e-3;
    if (solution) {
      const long long kept = std::min<long long>(s.nsol, sol_cap);
      if (kept > 0)
        HIPC(hipMemcpyAsync(solution, sol.p, sizeof(int) * n * kept, hipMemcpyDeviceToHost, m->stream));
      for (long long i = kept * n; i < n * (o.solution_capacity > 0 ? sol_cap : 1); ++i) solution[i] = -1;
    }
    const int tl = std::min(s.trace_len, o.trace_capacity);
    if (tl > 0) {
      std::vector<NodeRec> h(tl);
      HIPC(hipMemcpyAsync(h.data(), tr.p, sizeof(NodeRec) * tl, hipMemcpyDeviceToHost, m->stream));
      m->sync();
      for (int i = 0; i < tl; ++i) {
        trace[i].positive = h[i].positive;
        trace[i].var = h[i].var;
        trace[i].value = h[i].value;
        trace[i].consistent = h[i].consistent;
        trace[i].dom_hash = h[i].dom_hash;
      }
    }
    if (trace_len) *trace_len = s.trace_len;
    HIPC(hipMemcpyAsync(m->level_dom(0), root.p, sizeof(u64) * m->level_words(), hipMemcpyDeviceToDevice,
                        m->stream));
    hipLaunchKernelGGL(k_sizes, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->level_dom(0), m->level_size(0), n,
                       m->dm.W);
    HIPC(hipGetLastError());
    m->sync();
    if (!(s.status == MAC_UNSAT && s.npos + s.nneg == 0)) m->closure[0] = cpim_gmodel::kClosed;
  });
}

}  // extern "C"

#include "batch.inc"

#include "noalloc.inc"
