// ragged.hip -- many independent transforms of uneven lengths and kinds
// (complex c2c, real r2c / c2r) in a few launches.
//
// A batch is planned once (rfh_batch_create): every job gets the passes the
// per-call engine would run for it (direct LDS line, Bluestein in LDS, the
// four-step passes, or pre -> c2c -> post for real lengths without a fused
// plan), all sized to one LDS budget, with its temporaries carved out of one
// arena.  The passes are cut into tiles (a group of lines each), one workgroup
// per tile on the general line body (mixline.hpp), and grouped by level: level
// k holds the k-th pass of every job that has one, so a tile depends only on
// tiles of earlier levels.  A level runs as one launch per workgroup size (64
// to 1024 threads), the largest passes first: the hardware hands the next tile
// to whichever CU has room, a long line takes a whole CU's LDS and a short one
// a wave.  Kernel boundaries order the levels, so no workgroup ever waits on
// another and a large job's tiles spread over many CUs.  The LDS budget is
// picked by a small autotuner that times the candidates on scratch copies of
// the batch's buffers.
//
// Execution allocates nothing and calls no host synchronisation, so it can
// be captured in a HIP graph.
#include <fcntl.h>
#include <unistd.h>

#include <algorithm>
#include <cctype>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <set>
#include <sstream>
#include <string>
#include <tuple>

#include "../../include/rocket_fft_hip.h"
#include "passes.hpp"

namespace rfh {
namespace {
using namespace dev;

constexpr int OP_PRE = 9;   // one line: real / half-complex input -> complex work line
constexpr int OP_POST = 10; // one line: complex work line -> real / half-complex output
// elements of a pre / post line per tile: the elementwise real-transform
// steps are cut into tiles like the line passes, so that a long line's
// pre / post step spreads over many workgroups instead of one
constexpr int64_t kPrePostChunk = 2048;

// Workgroup sizes, and the LDS a tile may take in them: a launch reserves for
// every workgroup what its largest tile needs, and with these limits the CU's
// 160 KB hold the waves its registers do (four per SIMD).
struct TileClass {
  int threads;
  size_t lds;
};
constexpr TileClass kClass[] = {{64, 10240}, {256, 40960}, {512, 81920}, {1024, 163840}};
constexpr int kClasses = 4;
// A class with fewer threads than this in a level joins the next larger one
// there: half a round of the chip's waves costs less than a launch of its own.
constexpr int64_t kMergeThreads = 256 * 512;
constexpr int kXcds = 8;  // workgroup i of a launch runs on XCD i mod 8

template <typename T>
struct BatchPass {
  int op;
  LineArgs<T> a;
  MixGeom m;
};
struct UnitDev {  // tile `tile` of pass `pass`
  int pass;
  int tile;
};
struct Launch {  // units [first, first + count) in workgroups of `threads`
  int threads, first, count;
  size_t lds;
};

// elements [tile C, (tile + 1) C) of a pre / post line (C = kPrePostChunk)
template <typename T>
__device__ void pre_line(const LineArgs<T> &a, int tile) {
  C2<T> *t = reinterpret_cast<C2<T> *>(a.out);
  const int mode = a.sub & 0xff;
  const int64_t j0 = int64_t(tile) * kPrePostChunk;
  const int64_t j1 = min(j0 + kPrePostChunk, int64_t(a.f.n));
  for (int64_t j = j0 + threadIdx.x; j < j1; j += blockDim.x)
    t[j] = pre_elem<T, int64_t>(mode, a.in, a.esi, a.bign, a.f.n, j, false,
                                (a.sub & R2R_CONJ) != 0, false, ComputedRoot<T>{a.bign});
}

template <typename T>
__device__ void post_line(const LineArgs<T> &a, int tile) {
  const C2<T> *t = reinterpret_cast<const C2<T> *>(a.in);
  const int mode = (a.sub >> 8) & 0xff;
  const int64_t n = a.bign;
  const int64_t k0 = int64_t(tile) * kPrePostChunk;
  if (mode == kPostComplexHalf || mode == kPostHalfSpectrum) {
    const int64_t k1 = min(k0 + kPrePostChunk, n / 2 + 1);
    for (int64_t k = k0 + threadIdx.x; k < k1; k += blockDim.x) {
      C2<T> v = mode == kPostComplexHalf
                    ? t[k]
                    : half_spectrum_bin<T>([&](int64_t q) { return t[q]; }, n, k);
      if (a.sub & R2R_CONJ) v.y = -v.y;
      a.out[k * a.eso] = a.fct * v.x;
      a.out[k * a.eso + 1] = a.fct * v.y;
    }
  } else {
    const int64_t k1 = min(k0 + kPrePostChunk, n);
    for (int64_t k = k0 + threadIdx.x; k < k1; k += blockDim.x)
      a.out[k * a.eso] =
          a.fct * post_elem<T, int64_t>(mode, [&](int64_t q) { return t[q]; }, n, k, false, false,
                                        ComputedRoot<T>{n});
  }
}

// One tile per workgroup.  Bound by a tile's latency (about 20 us for 4096
// elements of a column pass: arguments, loads, two twiddled exchanges, stores,
// each waiting for the one before) times the 16 waves per CU that 128
// registers allow: 4096 jobs 1857 -> 865 us, 1.8 GB of traffic at 2.1 TB/s,
// against 256-thread workgroups that pulled units from a queue and ran every
// tile, long or short, with two line buffers.
template <typename T>
__global__ void __launch_bounds__(kMixThreads<T>)
    k_ragged(const UnitDev *__restrict__ units, const BatchPass<T> *__restrict__ passes) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const UnitDev u = units[blockIdx.x];
  const BatchPass<T> &p = passes[u.pass];
  if (p.op == OP_PRE) pre_line<T>(p.a, u.tile);
  else if (p.op == OP_POST) post_line<T>(p.a, u.tile);
  else mix_body<T, OP_ANY>(p.a, p.m, u.tile, smem_raw);
}

// ------------------------------------------------------------------ host

struct Built {
  size_t budget = 0;
  DevBuf units, passes, arena;
  std::vector<Launch> launches;  // in order
  std::vector<std::shared_ptr<C2CPlan>> c2c_keep;
  std::vector<std::shared_ptr<RealPlan>> real_keep;
  int njobs = 0;
  int lds_need = 0;  // of the launch that takes most
  int grid = 0;      // workgroups of the largest launch
};

struct Batch {
  bool dbl = false;
  std::vector<rfh_job_t> jobs;
  std::unique_ptr<Built> b;
  int autotuned = 0;
  double tuned_ms = 0;
};

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

LineSet one_line(const void *in, void *out, int64_t esi, int64_t eso) {
  LineSet g{};
  g.in = in;
  g.out = out;
  g.nlines = 1;
  g.nb = 0;
  g.esi = esi;
  g.eso = eso;
  return g;
}

// Geometry of a pass's tiles: 16 elements per thread whatever the number of
// lines (other jobs fill the CUs), short interleaved lines gathered to about
// 256 threads, and no more lines than there are.
template <typename T>
MixGeom batch_geom(const PassSpec &ps, const LineArgs<T> &a) {
  const bool inter = a.lfast_in || a.lfast_out;
  int want = ps.lines;
  if (inter) {
    want = std::max(want, sizeof(T) == 8 ? 4 : 8);
    while (want < 64 && want * 2 * ((a.f.n + 15) / 16) <= 256) want *= 2;
    while (want > 1 && want / 2 >= a.nlines) want /= 2;
  }
  // a prime stage's long sums are spread over as many threads as there are
  bool prime = false;
  for (int s = 0; s < a.f.nst; ++s) prime = prime || a.f.st[s].radix > 17;
  MixGeom m = mix_geometry(a.f, ps.d->pbo, sizeof(T) == 8,
                           prime && !inter ? 1 : int64_t(1) << 30, inter, want, lds_limit());
  if (m.L == 0) RFH_THROW(3, "ragged batch: a line does not fit in LDS");
  if (!inter) m.L = int(std::min<int64_t>(m.L, a.nlines));
  return m;
}

template <typename T>
std::unique_ptr<Built> build(const std::vector<rfh_job_t> &jobs, bool dbl, size_t budget) {
  auto B = std::make_unique<Built>();
  B->budget = budget;
  B->njobs = int(jobs.size());
  const size_t ce = 2 * sizeof(T);
  // pass 1: plans and temporaries
  std::vector<std::vector<PassLaunch>> per(jobs.size());
  std::vector<size_t> tmp_off(jobs.size()), work_off(jobs.size());
  size_t arena = 0;
  std::vector<std::shared_ptr<C2CPlan>> cplan(jobs.size());
  std::vector<std::shared_ptr<RealPlan>> rplan(jobs.size());
  for (size_t i = 0; i < jobs.size(); ++i) {
    const rfh_job_t &j = jobs[i];
    if (j.n == 0) continue;
    if (j.kind == RFH_JOB_C2C) {
      cplan[i] = get_c2c_plan(j.n, dbl, budget);
      tmp_off[i] = arena;
      arena = align_up(arena + c2c_tmp_bytes(*cplan[i], one_line(nullptr, nullptr, 2, 2)), 256);
    } else {
      rplan[i] = get_real_plan(j.n, dbl, budget);
      if (!rplan[i]->fused) {  // pre -> c2c(m) -> post through a work line of m
        const uint64_t m = rplan[i]->half ? j.n / 2 : j.n;
        cplan[i] = get_c2c_plan(m, dbl, budget);
        work_off[i] = arena;
        arena = align_up(arena + size_t(m) * ce, 256);
        tmp_off[i] = arena;
        arena = align_up(arena + c2c_tmp_bytes(*cplan[i], one_line(nullptr, nullptr, 2, 2)), 256);
      }
    }
  }
  B->arena.bytes = 0;
  if (arena) {
    HIP_CHECK(hipMalloc(&B->arena.p, arena));
    B->arena.bytes = arena;
  }
  char *ar = static_cast<char *>(B->arena.p);
  // pass 2: the passes of every job
  for (size_t i = 0; i < jobs.size(); ++i) {
    const rfh_job_t &j = jobs[i];
    if (j.n == 0) continue;
    const int dir = j.forward ? -1 : +1;
    if (j.kind == RFH_JOB_C2C) {
      per[i] = describe_c2c(*cplan[i], one_line(j.in, j.out, 2, 2), dir, j.fct, ar + tmp_off[i]);
      check_tmp_spans(per[i], ar + tmp_off[i],
                      c2c_tmp_bytes(*cplan[i], one_line(nullptr, nullptr, 2, 2)), dbl ? 8 : 4);
      continue;
    }
    const bool r2c = j.kind == RFH_JOB_R2C;
    if (rplan[i]->fused) {
      per[i].push_back(describe_real_fused(*rplan[i], r2c ? kR2C : kC2R,
                                           one_line(j.in, j.out, r2c ? 1 : 2, r2c ? 2 : 1),
                                           r2c ? !j.forward : j.forward, j.fct));
      continue;
    }
    // Real lengths without a fused plan: pre -> c2c -> post through the work
    // line.  Of an even length the pairs of reals are the complex line: r2c
    // transforms the input as it lies, c2r into the output.
    void *work = ar + work_off[i];
    const bool half = rplan[i]->half;
    const void *cin = work;
    void *cout = work;
    double cfct = 1.0;
    if (r2c && half) {
      cin = j.in;
    } else {
      PassSpec pre{};
      pre.d = &cplan[i]->main;  // only desc.n (= m) is read
      pre.op = OP_PRE;
      pre.bign = int64_t(j.n);
      const int mode = r2c ? kPreRealAsComplex : (half ? kPreHalfSpectrum : kPreHermitian);
      pre.sub = mode | (!r2c && j.forward ? R2R_CONJ : 0);
      per[i].push_back(PassLaunch{pre, one_line(j.in, work, r2c ? 1 : 2, 2)});
    }
    if (!r2c && half) {
      cout = j.out;
      cfct = j.fct;
    }
    const auto cp = describe_c2c(*cplan[i], one_line(cin, cout, 2, 2), r2c ? -1 : +1, cfct,
                                 ar + tmp_off[i]);
    check_tmp_spans(cp, ar + tmp_off[i],
                    c2c_tmp_bytes(*cplan[i], one_line(nullptr, nullptr, 2, 2)), dbl ? 8 : 4);
    for (const auto &pl : cp) per[i].push_back(pl);
    if (cout == work) {
      PassSpec post{};
      post.d = &cplan[i]->main;
      post.op = OP_POST;
      post.bign = int64_t(j.n);
      post.fct = j.fct;
      const int mode = r2c ? (half ? kPostHalfSpectrum : kPostComplexHalf) : kPostReal;
      post.sub = (mode << 8) | (r2c && !j.forward ? R2R_CONJ : 0);
      per[i].push_back(PassLaunch{post, one_line(work, j.out, 2, r2c ? 2 : 1)});
    }
  }
  // pass 3: device tables; tiles by level and workgroup size
  struct Item {  // one pass
    double cost;  // of all its tiles: elements x stages, a prime stage by its sums
    double time;  // of one tile, in the same units over its threads
    int pass, tiles, level, cls;
    size_t lds;
  };
  std::vector<BatchPass<T>> pd;
  std::vector<std::vector<Item>> job_items(jobs.size());
  int levels = 0;
  auto class_of = [](int threads, size_t lds) {
    int c = 0;
    while (c < kClasses - 1 && (kClass[c].threads < threads || kClass[c].lds < lds)) ++c;
    return c;
  };
  for (size_t i = 0; i < jobs.size(); ++i) {
    levels = std::max(levels, int(per[i].size()));
    for (const PassLaunch &pl : per[i]) {
      if (pl.ps.op == OP_BLUE_IN || pl.ps.op == OP_BLUE_MUL || pl.ps.op == OP_BLUE_OUT)
        RFH_THROW(3, "ragged batch: length " + std::to_string(jobs[i].n) +
                         " needs the multi-pass Bluestein form, which the batch kernel "
                         "does not run");
      BatchPass<T> p{};
      p.op = pl.ps.op;
      p.a = make_line_args<T>(pl.ps, pl.g);
      Item it{};
      if (p.op == OP_PRE || p.op == OP_POST) {
        p.a.f.n = int(cplan[i]->n);  // work-line length m
        // outputs of the step: the work line, or the half spectrum / real line
        const int post_mode = (p.a.sub >> 8) & 0xff;
        const int64_t count =
            p.op == OP_PRE ? int64_t(p.a.f.n)
            : (post_mode == kPostComplexHalf || post_mode == kPostHalfSpectrum) ? p.a.bign / 2 + 1
                                                                                : p.a.bign;
        it.tiles = int((count + kPrePostChunk - 1) / kPrePostChunk);
        it.cost = double(count);
        it.time = double(kPrePostChunk) / kThreads;
        it.cls = class_of(kThreads, 0);
      } else {
        p.m = batch_geom<T>(pl.ps, p.a);
        it.tiles = int((pl.g.nlines + p.m.L - 1) / p.m.L);
        double stages = 0;
        for (int s = 0; s < p.m.nst; ++s)
          stages += p.m.st[s].radix > 17 ? 0.3 * p.m.st[s].radix : 1.0;
        if (p.op == OP_BLUE || p.op == OP_BLUEROW) stages *= 2;
        it.cost = double(pl.g.nlines) * p.a.f.n * stages;
        it.time = double(p.a.f.n) * (stages + 4) / p.m.T;
        it.lds = size_t(p.m.L * p.m.ld + p.m.ngen) * ce;
        it.cls = class_of(p.m.L * p.m.T, it.lds);
        if (it.lds > lds_limit() || p.m.L * p.m.T > kMixThreads<T>)
          RFH_THROW(3, "ragged batch: a pass exceeds the workgroup");
      }
      it.pass = int(pd.size());
      pd.push_back(p);
      job_items[i].push_back(it);
    }
  }
  // Levels: a job of fewer passes than the longest starts where the least work
  // is, so that the one-pass jobs fill the levels that few long ones reach.
  std::vector<double> load(size_t(levels), 0.0);
  std::vector<size_t> order(jobs.size());
  for (size_t i = 0; i < jobs.size(); ++i) order[i] = i;
  auto job_cost = [&](size_t i) {
    double c = 0;
    for (const Item &it : job_items[i]) c += it.cost;
    return c;
  };
  std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) {
    const auto key = [&](size_t i) { return std::make_pair(job_items[i].size(), job_cost(i)); };
    return key(x) > key(y);
  });
  std::vector<std::vector<Item>> by_level(size_t(levels) * kClasses);
  for (size_t i : order) {
    const size_t np = job_items[i].size();
    size_t at = 0;
    double best = 1e300;
    for (size_t o = 0; o + np <= size_t(levels); ++o) {
      double most = 0;
      for (size_t k = 0; k < np; ++k) most = std::max(most, load[o + k] + job_items[i][k].cost);
      if (most < best) {
        best = most;
        at = o;
      }
    }
    for (size_t k = 0; k < np; ++k) {
      Item &it = job_items[i][k];
      load[at + k] += it.cost;
      by_level[(at + k) * kClasses + size_t(it.cls)].push_back(it);
    }
  }
  std::vector<UnitDev> units;
  for (int lv = 0; lv < levels; ++lv) {
    std::vector<Item> *cl = &by_level[size_t(lv) * kClasses];
    for (int c = 0; c < kClasses - 1; ++c) {
      int64_t threads = 0;
      for (const Item &it : cl[c]) threads += int64_t(it.tiles) * kClass[c].threads;
      int up = c + 1;
      while (up < kClasses && cl[up].empty()) ++up;
      if (threads && threads < kMergeThreads && up < kClasses) {
        cl[up].insert(cl[up].end(), cl[c].begin(), cl[c].end());
        cl[c].clear();
      }
    }
    for (int c = kClasses - 1; c >= 0; --c) {
      if (cl[c].empty()) continue;
      Launch L{std::min(kClass[c].threads, kMixThreads<T>), int(units.size()), 0, 0};
      // the longest tiles first; all tiles of a pass on one XCD, whose L2
      // then holds the pass's tables once
      std::stable_sort(cl[c].begin(), cl[c].end(), [](const Item &x, const Item &y) {
        return x.time > y.time;
      });
      std::vector<UnitDev> q[kXcds];
      for (const Item &it : cl[c]) {
        int x = 0;
        for (int k = 1; k < kXcds; ++k)
          if (q[k].size() < q[x].size()) x = k;
        for (int t = 0; t < it.tiles; ++t) q[x].push_back(UnitDev{it.pass, t});
        L.count += it.tiles;
        L.lds = std::max(L.lds, it.lds);
      }
      size_t head[kXcds] = {};
      for (int i = 0; i < L.count; ++i) {
        int x = i % kXcds;
        if (head[x] == q[x].size())  // this one is empty: the fullest gives a tile
          for (int k = 0; k < kXcds; ++k)
            if (q[k].size() - head[k] > q[x].size() - head[x]) x = k;
        units.push_back(q[x][head[x]++]);
      }
      B->launches.push_back(L);
    }
  }
  for (const Launch &L : B->launches) {
    B->lds_need = std::max(B->lds_need, int(L.lds));
    B->grid = std::max(B->grid, L.count);
  }
  B->units.upload(units.data(), units.size() * sizeof(UnitDev));
  B->passes.upload(pd.data(), pd.size() * sizeof(BatchPass<T>));
  for (auto &p : cplan)
    if (p) B->c2c_keep.push_back(p);
  for (auto &p : rplan)
    if (p) B->real_keep.push_back(p);
  return B;
}

std::mutex g_attr_mu;
std::set<std::pair<int, int>> g_attr_set;  // (device, double precision)

template <typename T>
void launch_batch(const Built &B, hipStream_t s) {
  if (B.njobs == 0) return;
  const void *fn = reinterpret_cast<const void *>(&k_ragged<T>);
  {
    std::lock_guard<std::mutex> lk(g_attr_mu);
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    if (!g_attr_set.count({dev, int(sizeof(T) == 8)})) {
      hipFuncAttributes fa;
      HIP_CHECK(hipFuncGetAttributes(&fa, fn));
      HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(lds_limit() - fa.sharedSizeBytes)));
      g_attr_set.insert({dev, int(sizeof(T) == 8)});
    }
  }
  for (const Launch &L : B.launches) {
    hipLaunchKernelGGL(k_ragged<T>, dim3(unsigned(L.count)), dim3(unsigned(L.threads)), L.lds, s,
                       static_cast<const UnitDev *>(B.units.p) + L.first,
                       static_cast<const BatchPass<T> *>(B.passes.p));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) RFH_THROW(2, std::string("ragged launch: ") + hipGetErrorString(e));
  }
}

int cu_count() {
  static int n = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      v = 256;
    return v > 0 ? v : 256;
  }();
  return n;
}

void run(Batch &bt, hipStream_t s) {
  if (bt.dbl)
    launch_batch<double>(*bt.b, s);
  else
    launch_batch<float>(*bt.b, s);
}

double time_ms(Batch &bt, hipStream_t s, int reps) {
  hipEvent_t e0, e1;
  HIP_CHECK(hipEventCreate(&e0));
  HIP_CHECK(hipEventCreate(&e1));
  run(bt, s);  // warm
  HIP_CHECK(hipEventRecord(e0, s));
  for (int r = 0; r < reps; ++r) run(bt, s);
  HIP_CHECK(hipEventRecord(e1, s));
  HIP_CHECK(hipEventSynchronize(e1));
  float ms = 0;
  HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return double(ms) / reps;
}

std::unique_ptr<Built> build_any(const Batch &bt, size_t budget) {
  return bt.dbl ? build<double>(bt.jobs, true, budget) : build<float>(bt.jobs, false, budget);
}

// Autotuner: the LDS budget, which sets how long a line runs in one pass
// (a long one has a CU to itself); each candidate is timed on the batch.
// Results are kept per batch signature (precision, then kind and length of
// every job) for the process and, when a cache directory is set, in a text
// file per GPU architecture and CU count that later processes read:
//   <dir>/ragged_tune_<arch>_<cus>cu.txt, one line per signature:
//   "rfh1 <fnv-1a hash> <second hash> <jobs> <lds budget> <largest grid>"
// Lines are appended with one write each; unreadable lines are ignored.
std::mutex g_tune_mu;
std::map<std::vector<uint64_t>, std::pair<size_t, int>> g_tuned;
std::string g_cache_dir;  // empty: no disk cache
struct DiskKey {
  uint64_t h1, h2, n;
  bool operator<(const DiskKey &o) const {
    return std::tie(h1, h2, n) < std::tie(o.h1, o.h2, o.n);
  }
};
std::map<DiskKey, std::pair<size_t, int>> g_disk;
std::string g_disk_loaded;  // file whose lines are in g_disk

std::vector<uint64_t> signature(const Batch &bt) {
  std::vector<uint64_t> sig{uint64_t(bt.dbl)};
  for (const auto &j : bt.jobs) sig.push_back((uint64_t(j.kind) << 60) ^ j.n);
  return sig;
}

// The version of the kernels and candidates that a tuning result holds for: one
// more with every change.  It is part of the key, so that lines of an earlier
// build are not found and their batches timed again.
constexpr uint64_t kTuneVersion = 2;

DiskKey disk_key(const std::vector<uint64_t> &sig) {
  uint64_t h1 = 1469598103934665603ull, h2 = 0x9e3779b97f4a7c15ull ^ kTuneVersion;
  for (uint64_t v : sig) {
    for (int b = 0; b < 8; ++b) {
      h1 = (h1 ^ ((v >> (8 * b)) & 0xff)) * 1099511628211ull;
    }
    h2 ^= v + 0x9e3779b97f4a7c15ull + (h2 << 6) + (h2 >> 2);
    h2 *= 0xff51afd7ed558ccdull;
  }
  return DiskKey{h1, h2, uint64_t(sig.size())};
}

// LDS budgets the autotuner tries: lines of up to 4096 / 8192 complex64
// elements in one pass, or all that fit a CU
std::vector<size_t> tune_budgets() { return {size_t(65536), size_t(131072), whole_line_budget()}; }

bool budget_ok(size_t b) {
  for (size_t c : tune_budgets())
    if (b == c) return true;
  return false;
}

std::string cache_file() {
  if (g_cache_dir.empty()) return {};
  int dev = 0;
  (void)hipGetDevice(&dev);
  hipDeviceProp_t pr;
  std::string arch = "gpu";
  if (hipGetDeviceProperties(&pr, dev) == hipSuccess) {
    arch.clear();
    for (const char *c = pr.gcnArchName; *c && *c != ':'; ++c)
      arch += std::isalnum(static_cast<unsigned char>(*c)) ? *c : '_';
  }
  return g_cache_dir + "/ragged_tune_" + arch + "_" + std::to_string(cu_count()) + "cu.txt";
}

// with g_tune_mu held
void load_disk(const std::string &path) {
  if (path == g_disk_loaded) return;
  g_disk.clear();
  g_disk_loaded = path;
  std::ifstream f(path);
  std::string line;
  while (std::getline(f, line)) {
    std::istringstream is(line);
    std::string tag;
    DiskKey k{};
    size_t budget = 0;
    int grid = 0;
    if (!(is >> tag >> std::hex >> k.h1 >> k.h2 >> std::dec >> k.n >> budget >> grid)) continue;
    if (tag != "rfh1" || !budget_ok(budget) || grid <= 0) continue;
    g_disk[k] = {budget, grid};
  }
}

void append_disk(const std::string &path, const DiskKey &k, size_t budget, int grid) {
  char buf[160];
  const int len = std::snprintf(buf, sizeof buf, "rfh1 %016llx %016llx %llu %zu %d\n",
                                (unsigned long long)k.h1, (unsigned long long)k.h2,
                                (unsigned long long)k.n, budget, grid);
  const int fd = ::open(path.c_str(), O_WRONLY | O_CREAT | O_APPEND, 0644);
  if (fd < 0) return;  // the cache is an optimisation: an unwritable directory is not an error
  const ssize_t w = ::write(fd, buf, size_t(len));
  (void)w;  // a short write leaves a line that later reads ignore
  ::close(fd);
}

void autotune(Batch &bt, hipStream_t s) {
  const auto sig = signature(bt);
  const DiskKey dk = disk_key(sig);
  std::string path;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(sig);
    if (it != g_tuned.end()) {
      bt.b = build_any(bt, it->second.first);
      bt.autotuned = 2;
      return;
    }
    path = cache_file();
    if (!path.empty()) {
      load_disk(path);
      auto d = g_disk.find(dk);
      if (d != g_disk.end()) {
        std::unique_ptr<Built> b;
        try {
          b = build_any(bt, d->second.first);
        } catch (const Error &) {
          // a cached budget that no longer plans (another build): tune again
        }
        if (b) {
          bt.b = std::move(b);
          bt.autotuned = 3;
          g_tuned[sig] = d->second;
          return;
        }
      }
    }
  }
  // The candidates run on scratch copies of the job buffers, never on the
  // caller's: a job may be in place or read another job's output, and
  // creating a batch must not transform anything.
  Batch tb;
  tb.dbl = bt.dbl;
  tb.jobs = bt.jobs;
  DevBuf scratch;
  {
    const size_t rs = bt.dbl ? 8 : 4, cs = 2 * rs;
    size_t total = 0;
    std::vector<std::pair<size_t, size_t>> off(tb.jobs.size());
    for (size_t i = 0; i < tb.jobs.size(); ++i) {
      const rfh_job_t &j = tb.jobs[i];
      const size_t h = size_t(j.n / 2 + 1);
      const size_t in_b = j.kind == RFH_JOB_C2C ? j.n * cs : (j.kind == RFH_JOB_R2C ? j.n * rs : h * cs);
      const size_t out_b = j.kind == RFH_JOB_C2C ? j.n * cs : (j.kind == RFH_JOB_R2C ? h * cs : j.n * rs);
      off[i].first = total;
      total = align_up(total + in_b, 256);
      off[i].second = total;
      total = align_up(total + out_b, 256);
    }
    if (total) {
      HIP_CHECK(hipMalloc(&scratch.p, total));
      scratch.bytes = total;
      HIP_CHECK(hipMemsetAsync(scratch.p, 0, total, s));
    }
    char *base = static_cast<char *>(scratch.p);
    for (size_t i = 0; i < tb.jobs.size(); ++i) {
      tb.jobs[i].in = base + off[i].first;
      tb.jobs[i].out = base + off[i].second;
    }
  }
  double best = 1e300;
  size_t best_budget = 0;
  for (size_t budget : tune_budgets()) {
    try {
      tb.b = build_any(tb, budget);
    } catch (const Error &) {
      continue;
    }
    const double ms = time_ms(tb, s, 3);
    if (ms < best) {
      best = ms;
      best_budget = budget;
    }
  }
  HIP_CHECK(hipStreamSynchronize(s));  // the timing runs are done with the scratch copies
  tb.b.reset();
  if (!best_budget) RFH_THROW(3, "ragged batch: no LDS budget fits every job");
  bt.b = build_any(bt, best_budget);
  bt.autotuned = 1;
  bt.tuned_ms = best;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tuned[sig] = {best_budget, bt.b->grid};
  if (!path.empty() && path == cache_file()) {
    append_disk(path, dk, best_budget, bt.b->grid);
    g_disk[dk] = {best_budget, bt.b->grid};
  }
}

// device or managed memory (the kernel dereferences job pointers
// directly; host memory would fault)
bool device_memory(const void *p) {
  if (!p) return false;
  hipPointerAttribute_t at;
  std::memset(&at, 0, sizeof(at));
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged;
}

template <typename F>
int guarded_int(F &&f) {
  try {
    fork_guard();
    f();
    return 0;
  } catch (const Error &e) {
    set_error(e.code, e.msg);
    return e.code;
  } catch (const std::exception &e) {
    set_error(1, e.what());
    return 1;
  }
}

}  // namespace
}  // namespace rfh

using namespace rfh;

extern "C" {

int rfh_batch_create(const rfh_job_t *jobs, int64_t njobs, bool double_precision, bool tune,
                     void *stream, void **handle) {
  return guarded_int([&] {
    auto *bt = new Batch();
    bt->dbl = double_precision;
    bt->jobs.assign(jobs, jobs + njobs);
    const size_t al = double_precision ? 16 : 8;
    for (const auto &j : bt->jobs) {
      if (j.kind < RFH_JOB_C2C || j.kind > RFH_JOB_C2R) {
        delete bt;
        RFH_THROW(3, "ragged batch: unknown job kind");
      }
      if ((reinterpret_cast<uintptr_t>(j.in) | reinterpret_cast<uintptr_t>(j.out)) % al) {
        delete bt;
        RFH_THROW(3, "ragged batch: job buffers must be aligned to the complex element size");
      }
      if (j.n > 0 && (!device_memory(j.in) || !device_memory(j.out))) {
        delete bt;
        RFH_THROW(3, "ragged batch: job buffers must be device (or managed) memory");
      }
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    try {
      if (tune) {
        autotune(*bt, s);
      } else {
        bt->b = build_any(*bt, 65536);
      }
    } catch (...) {
      delete bt;
      throw;
    }
    *handle = bt;
  });
}

int rfh_batch_execute(void *handle, void *stream) {
  return guarded_int([&] {
    Batch *bt = static_cast<Batch *>(handle);
    run(*bt, static_cast<hipStream_t>(stream));
  });
}

int rfh_batch_execute_serial(void *handle, void *stream) {
  // one drop-in call per transform, as a caller of numba_c2c / numba_r2c /
  // numba_c2r would make them, enqueued on the same stream
  hipStream_t prev_s;
  bool prev_b;
  thread_stream(&prev_s, &prev_b);
  rfh_set_stream(stream, false);
  const int rc = guarded_int([&] {
    Batch *bt = static_cast<Batch *>(handle);
    const int64_t rs = bt->dbl ? 8 : 4, cs = 2 * rs;
    struct Arr1 {
      arystruct_t s;
      int64_t ss[2];
    };
    uint64_t axis0 = 0;
    Arr1 ax{};
    ax.s.nitems = 1;
    ax.s.itemsize = 8;
    ax.s.data = &axis0;
    ax.s.shape_and_strides[0] = 1;
    ax.s.shape_and_strides[1] = 8;
    for (const rfh_job_t &j : bt->jobs) {
      if (j.n == 0) continue;
      Arr1 ai{}, ao{};
      const bool c2c = j.kind == RFH_JOB_C2C, r2c = j.kind == RFH_JOB_R2C;
      const int64_t h = int64_t(j.n / 2 + 1);
      ai.s.itemsize = (c2c || !r2c) ? cs : rs;
      ai.s.shape_and_strides[0] = (c2c || r2c) ? int64_t(j.n) : h;
      ai.s.shape_and_strides[1] = ai.s.itemsize;
      ai.s.data = const_cast<void *>(j.in);
      ao.s.itemsize = (c2c || r2c) ? cs : rs;
      ao.s.shape_and_strides[0] = (c2c || !r2c) ? int64_t(j.n) : h;
      ao.s.shape_and_strides[1] = ao.s.itemsize;
      ao.s.data = j.out;
      if (c2c)
        numba_c2c(1, &ai.s, &ao.s, &ax.s, j.forward != 0, j.fct, 1);
      else if (r2c)
        numba_r2c(1, &ai.s, &ao.s, &ax.s, j.forward != 0, j.fct, 1);
      else
        numba_c2r(1, &ai.s, &ao.s, &ax.s, j.forward != 0, j.fct, 1);
      char msg[256];
      if (rfh_last_error(msg, sizeof msg)) RFH_THROW(3, std::string("per-transform call: ") + msg);
    }
  });
  rfh_set_stream(prev_s, prev_b);
  return rc;
}

int rfh_tune_cache(const char *dir, bool clear_memory) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  if (clear_memory) g_tuned.clear();
  g_cache_dir = dir ? std::string(dir) : std::string();
  while (g_cache_dir.size() > 1 && g_cache_dir.back() == '/') g_cache_dir.pop_back();
  g_disk.clear();
  g_disk_loaded.clear();
  return 0;
}

int rfh_batch_info(void *handle, int *grid, int *lds_bytes, int *autotuned, double *tuned_ms) {
  Batch *bt = static_cast<Batch *>(handle);
  *grid = bt->b ? bt->b->grid : 0;
  *lds_bytes = bt->b ? bt->b->lds_need : 0;
  *autotuned = bt->autotuned;
  *tuned_ms = bt->tuned_ms;
  return 0;
}

int rfh_batch_destroy(void *handle) {
  return guarded_int([&] { delete static_cast<Batch *>(handle); });
}

}  // extern "C"
