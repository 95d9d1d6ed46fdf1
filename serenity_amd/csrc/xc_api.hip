// C ABI of the XC Fock build (include/serenity_xc.h): resident handles, the
// screening/AO setup of a basis-functions-on-grid controller, and the
// density -> functional -> Fock pipeline on one HIP stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <deque>
#include <initializer_list>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/serenity_xc.h"
#include "host/host.h"
#include "kernels/xc_internal.h"

using namespace sxc;

namespace {

/* Work items of one block are consecutive in a list.  Workgroups of a launch are
 * dealt to the 8 XCDs round-robin (workgroup w runs on XCD w mod 8, from some
 * starting XCD), each with its own L2.  Cut the list into 8 contiguous ranges of
 * whole blocks (about a fair share of the items' cost each; the blocks are in grid order,
 * so a range is a region of the molecule) and interleave them: one XCD runs a
 * block's items one after another, its re-reads of the block's tiles hit its L2,
 * and the density-matrix rows its region reads stay in that L2 too (density stage
 * at (H2O)64/def2-TZVP: 4.46 -> 4.36 ms FP32 against dealing blocks to the
 * shortest queue). */
template <typename Item, typename Cost>
void xcd_order(std::vector<Item>& v, Cost&& cost) {
  constexpr int kXcd = 8;
  double total = 0.0;
  for (const Item& x : v) total += cost(x);
  size_t begin[kXcd + 1] = {};
  size_t i = 0;
  double sum = 0.0;
  for (int x = 0; x < kXcd; ++x) {
    begin[x] = i;
    const double end = total * (x + 1) / kXcd;
    while (i < v.size() && (x + 1 == kXcd || sum < end)) {  // whole blocks
      const int block = v[i].block;
      for (; i < v.size() && v[i].block == block; ++i) sum += cost(v[i]);
    }
  }
  begin[kXcd] = v.size();
  size_t len = 0;
  for (int x = 0; x < kXcd; ++x) len = std::max(len, begin[x + 1] - begin[x]);
  std::vector<Item> out;
  out.reserve(v.size());
  for (size_t k = 0; k < len; ++k)
    for (int x = 0; x < kXcd; ++x)
      if (begin[x] + k < begin[x + 1]) out.push_back(v[begin[x] + k]);
  v.swap(out);
}

thread_local std::string g_last_error;

struct XcError : std::runtime_error {
  int code;
  XcError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define HIPX(expr)                                                                                    \
  do {                                                                                                \
    hipError_t e_ = (expr);                                                                           \
    if (e_ != hipSuccess)                                                                             \
      throw XcError(XC_ERR_DEVICE, std::string(#expr) + " failed: " + hipGetErrorString(e_));         \
  } while (0)

void require(bool cond, int code, const std::string& msg) {
  if (!cond) throw XcError(code, msg);
}

template <typename F>
int guarded(F&& f) {
  try {
    f();
    return XC_OK;
  } catch (const XcError& e) {
    g_last_error = e.what();
    return e.code;
  } catch (const std::exception& e) {
    g_last_error = e.what();
    return XC_ERR_INPUT;
  } catch (...) {
    g_last_error = "unknown error";
    return XC_ERR_STATE;
  }
}

}  // namespace

// Workspace of xc_functional_device_noalloc: the per-block energies and their sum live in this
// file-scope device array instead of a per-call allocation.  Each device holds its own copy;
// host code never uses the array's name as an address, only the pointer that
// hipGetSymbolAddress returns for the current device (kept per device in g_noalloc_ptr).
constexpr int kNoallocBlocks = 131072;  // 1 MiB of per-block energies + the sum
static __device__ __align__(256) double scratch[kNoallocBlocks + 1];

namespace {
std::mutex g_noalloc_mu;
std::map<int, double*> g_noalloc_ptr;  // device -> address of that device's scratch

// Called once per device with that device current (context creation).
void noalloc_setup_current_device(int device) {
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (g_noalloc_ptr.count(device)) return;
  void* p = nullptr;
  HIPX(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  require(p != nullptr, XC_ERR_DEVICE, "hipGetSymbolAddress(scratch) returned no address");
  g_noalloc_ptr[device] = static_cast<double*>(p);
}

double* noalloc_scratch(int device) {
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  auto it = g_noalloc_ptr.find(device);
  require(it != g_noalloc_ptr.end(), XC_ERR_STATE, "no-allocation workspace not set up on this device");
  return it->second;
}
}  // namespace

// Execution lanes of a build: its stream plus kAux helper streams.  The launches
// of one stage (the Fock shapes, the J engine's classes) are independent, so they are spread over
// the lanes after a fork and joined before the next stage.
constexpr int kAux = 3;
struct Lanes {
  int n = 1;  // lanes in use: 1 (the build's stream only) or kAux + 1
  hipStream_t main = nullptr;
  hipStream_t aux[kAux] = {};
  hipEvent_t fork = nullptr;
  hipEvent_t join[kAux] = {};
  void create(hipStream_t m, bool helpers) {
    main = m;
    n = helpers ? kAux + 1 : 1;
    if (!helpers) return;
    for (int i = 0; i < kAux; ++i) {
      HIPX(hipStreamCreateWithFlags(&aux[i], hipStreamNonBlocking));
      HIPX(hipEventCreateWithFlags(&join[i], hipEventDisableTiming));
    }
    HIPX(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
  }
  void destroy() {
    for (int i = 0; i < kAux; ++i) {
      if (aux[i]) (void)hipStreamDestroy(aux[i]);
      if (join[i]) (void)hipEventDestroy(join[i]);
      aux[i] = nullptr;
      join[i] = nullptr;
    }
    if (fork) (void)hipEventDestroy(fork);
    fork = nullptr;
  }
  hipStream_t lane(int i) const { return i % (kAux + 1) == 0 ? main : aux[i % (kAux + 1) - 1]; }
  void fork_all() const {
    HIPX(hipEventRecord(fork, main));
    for (int i = 0; i < kAux; ++i) HIPX(hipStreamWaitEvent(aux[i], fork, 0));
  }
  void join_all() const {
    for (int i = 0; i < kAux; ++i) {
      HIPX(hipEventRecord(join[i], aux[i]));
      HIPX(hipStreamWaitEvent(main, join[i], 0));
    }
  }
};

struct PackWork;

// Pinned memory that host matrices and tables pass through on their way to and from the device: a
// ring of pieces, so that a long copy's pieces are moved on the host and over the link at once.
// Pageable memory copied directly goes through the runtime's own staging: 4.6 KB, 2.65 MB and 15 MB to
// the host take 22, 160 and 907 us, to the device 15, 88 and 416; to and from pinned memory they take 12, 55
// and 273 us, and the host's share (34 and 190 us) overlaps.  A kernel of the build's stream as the mover
// measured the same.  Used under the context's lock and on its stream only.
struct HostStage {
  static constexpr size_t kPiece = size_t(1) << 20;
  static constexpr int kPieces = 4;
  char* p = nullptr;
  hipEvent_t ev[kPieces] = {};
  bool pending[kPieces] = {};
  int piece = 0;
  size_t off = 0;
  void create() {
    HIPX(hipHostMalloc((void**)&p, kPiece * kPieces, hipHostMallocMapped | hipHostMallocCoherent));
    for (auto& e : ev) HIPX(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  void destroy() {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (p) (void)hipHostFree(p);
  }
  // Room for len <= kPiece bytes; enter(i) is called with piece i free before it is used again.
  template <typename Enter>
  char* take(hipStream_t s, size_t len, Enter&& enter) {
    if (off + len > kPiece) {
      HIPX(hipEventRecord(ev[piece], s));
      pending[piece] = true;
      piece = (piece + 1) % kPieces;
      off = 0;
      if (pending[piece]) HIPX(hipEventSynchronize(ev[piece]));
      pending[piece] = false;
      enter(piece);
    }
    char* q = p + (size_t)piece * kPiece + off;
    off += (len + 63) / 64 * 64;
    return q;
  }
  // Host -> device; the host memory is free again on return.
  void up(hipStream_t s, void* dst, const void* src, size_t bytes) {
    for (size_t o = 0; o < bytes; o += kPiece) {
      const size_t len = std::min(kPiece, bytes - o);
      char* q = take(s, len, [](int) {});
      std::memcpy(q, (const char*)src + o, len);
      HIPX(hipMemcpyAsync((char*)dst + o, q, len, hipMemcpyHostToDevice, s));
    }
  }
  struct Out {
    void* host;
    const void* dev;
    size_t bytes;
  };
  // Device -> host; what the stream held is done and everything is in place on return.
  void down(hipStream_t s, std::initializer_list<Out> outs) {
    struct Part {
      int piece;
      char *host, *q;
      size_t len;
    };
    std::deque<Part> parts;
    const auto deliver = [&](int i) {
      while (!parts.empty() && parts.front().piece == i) {
        std::memcpy(parts.front().host, parts.front().q, parts.front().len);
        parts.pop_front();
      }
    };
    for (const Out& o : outs)
      for (size_t k = 0; o.host && k < o.bytes; k += kPiece) {
        const size_t len = std::min(kPiece, o.bytes - k);
        char* q = take(s, len, deliver);
        HIPX(hipMemcpyAsync(q, (const char*)o.dev + k, len, hipMemcpyDeviceToHost, s));
        parts.push_back({piece, (char*)o.host + k, q, len});
      }
    while (!parts.empty() && parts.front().piece != piece) {
      const int i = parts.front().piece;
      HIPX(hipEventSynchronize(ev[i]));
      deliver(i);
    }
    HIPX(hipStreamSynchronize(s));
    deliver(piece);
    std::fill(pending, pending + kPieces, false);
    off = 0;
  }
};

struct xc_ctx {
  int device = 0;
  PackWork* pack = nullptr;  // device lists of packed builds (allocated on first use)
  // packed-build compositions seen before (controllers, functional, precision, threshold):
  // their own lists and, from the second build on, a captured graph
  std::map<std::vector<uint64_t>, PackWork*> pack_graphs;
  uint64_t pack_calls = 0;  // packed builds so far (recency of the cached compositions)
  hipStream_t stream = nullptr;
  Lanes lanes;  // helper lanes of builds on the context stream
  std::recursive_mutex mu;
  int64_t bytes = 0;
  // E_xc of the last build: pinned host memory that the kernels write (a copy of 8 bytes back to the
  // host costs 15 us more than the wait for the stream)
  double* energy = nullptr;
  int* flag = nullptr;  // likewise, for a kernel's report
  double* pack_energy = nullptr;  // likewise of a packed build's systems (grown on demand)
  size_t pack_energies = 0;
  HostStage stage;
  std::map<void*, size_t> user_allocs;  // buffers handed out by xc_device_alloc
  int live_handles = 0;                 // bases, grids and controllers not yet destroyed
  // stage timing: XC_NSTAGES + 1 events per profiled build
  bool profile = false;
  // every row reduce sums in 64-bit integers (F the same bit for bit on every run); set while no
  // basis, grid or controller exists
  bool deterministic = false;
  std::vector<hipEvent_t> ev_pool;
  size_t ev_used = 0;
  hipEvent_t next_event() {
    if (ev_used == ev_pool.size()) {
      hipEvent_t e;
      HIPX(hipEventCreate(&e));
      ev_pool.push_back(e);
    }
    return ev_pool[ev_used++];
  }
  void mark() {
    if (profile) HIPX(hipEventRecord(next_event(), stream));
  }

  // Device blocks are kept for reuse when released: a serving loop builds and evicts controllers
  // again and again, and hipMalloc / hipFree of their multi-GB buffers cost milliseconds each and
  // now and then stall.  Blocks are sized in 2 MiB steps (256 bytes below 1 MiB); an allocation
  // takes the smallest cached block that fits within 1/8 + 2 MiB of its size, else a new one.
  // The cache is given back to the device when a hipMalloc fails and when the context ends; where
  // that is not enough, so are the controllers' spare scratches.
  // `bytes` counts the blocks in use.
  std::multimap<size_t, void*> cache;            // block size -> released block
  std::unordered_map<void*, size_t> block_size;  // every block of this context -> size
  size_t cached = 0;
  static size_t block_round(size_t b) {
    constexpr size_t kBig = size_t(1) << 20, kStep = size_t(2) << 20;
    return b >= kBig ? (b + kStep - 1) / kStep * kStep : (b + 255) / 256 * 256;
  }
  void trim() {
    (void)hipDeviceSynchronize();
    for (auto& kv : cache) {
      (void)hipFree(kv.second);
      block_size.erase(kv.second);
    }
    cache.clear();
    cached = 0;
  }
  // Controllers whose second spin scratch no recorded graph holds: reclaim releases it (the controller
  // then runs one spin after the other), so that it never keeps memory from what has to have it.
  std::vector<xc_bfogc*> spare;
  void reclaim();
  // spare_too: false for what the caller can do without
  void* alloc(size_t bytes_, bool spare_too = true) {
    if (bytes_ == 0) return nullptr;
    HIPX(hipSetDevice(device));
    const size_t need = block_round(bytes_);
    auto it = cache.lower_bound(need);
    if (it != cache.end() && it->first <= need + need / 8 + (size_t(2) << 20)) {
      void* p = it->second;
      const size_t sz = it->first;
      cache.erase(it);
      cached -= sz;
      bytes += (int64_t)sz;
      return p;
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, need);
    if (e == hipErrorOutOfMemory && cached) {
      (void)hipGetLastError();
      trim();
      e = hipMalloc(&p, need);
    }
    if (e == hipErrorOutOfMemory && spare_too && !spare.empty()) {
      (void)hipGetLastError();
      reclaim();
      trim();
      e = hipMalloc(&p, need);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      throw XcError(e == hipErrorOutOfMemory ? XC_ERR_MEMORY : XC_ERR_DEVICE,
                    "hipMalloc of " + std::to_string(bytes_) + " bytes failed: " + hipGetErrorString(e));
    }
    block_size[p] = need;
    bytes += (int64_t)need;
    return p;
  }
  void release(void* p, size_t) {
    if (!p) return;
    auto it = block_size.find(p);
    if (it == block_size.end()) {
      (void)hipFree(p);
      return;
    }
    // enqueued work may still use the block: wait for the device, as hipFree does
    (void)hipDeviceSynchronize();
    bytes -= (int64_t)it->second;
    cache.emplace(it->second, p);
    cached += it->second;
  }
};

namespace {

// Device allocation owned by a handle.
template <typename T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  xc_ctx* ctx = nullptr;
  void alloc(xc_ctx* c, size_t count, bool spare_too = true) {
    free_();
    ctx = c;
    n = count;
    p = (T*)c->alloc(count * sizeof(T), spare_too);
  }
  void upload(xc_ctx* c, const T* host, size_t count) {
    alloc(c, count);
    c->stage.up(c->stream, p, host, count * sizeof(T));
  }
  void free_() {
    if (p && ctx) ctx->release(p, n * sizeof(T));
    p = nullptr;
    n = 0;
  }
  ~DBuf() { free_(); }
};


}  // namespace

// Merged lists and per-system table of packed builds, grown on demand; a packed build
// synchronises before it returns, so they are free again for the next one.
struct PackWork {
  DBuf<DevBlock> blocks;
  DBuf<PackSys> sys;
  DBuf<WorkItem> dens[2];  // [1: of the systems whose density is the quadratic form]
  DBuf<FockItem> fock[kFockShapes];
  DBuf<double> round;
  hipGraphExec_t exec = nullptr;  // captured build of a repeated composition
  uint64_t last_use = 0;          // packed-build counter at its last use (least recently used is evicted)
  ~PackWork() {
    if (exec) (void)hipGraphExecDestroy(exec);
  }
};

// drop every cached packed composition that names bf (its buffers are going away)
void forget_packs_of(xc_ctx* ctx, const void* bf) {
  for (auto it = ctx->pack_graphs.begin(); it != ctx->pack_graphs.end();) {
    bool uses = false;
    for (size_t i = 0; i + 3 < it->first.size(); ++i) uses = uses || it->first[i] == (uint64_t)(uintptr_t)bf;
    if (uses) {
      delete it->second;
      it = ctx->pack_graphs.erase(it);
    } else {
      ++it;
    }
  }
}

template <typename T>
void upload_grow(xc_ctx* ctx, DBuf<T>& b, const std::vector<T>& v) {
  if (v.empty()) return;
  if (b.n < v.size()) b.alloc(ctx, std::max(v.size(), 2 * b.n));
  ctx->stage.up(ctx->stream, b.p, v.data(), v.size() * sizeof(T));
}

struct xc_basis {
  xc_ctx* ctx = nullptr;
  int nshell = 0, nao = 0, maxl = 0;
  std::vector<DevShell> shells;
  std::vector<double> alpha, coef, ang;
  DBuf<DevShell> d_shells;
  DBuf<double> d_alpha, d_coef, d_ang;
};

// Density-fitted Coulomb matrix of an orbital basis over an auxiliary basis (the J engine).
struct xc_coulomb {
  xc_ctx* ctx = nullptr;
  xc_basis* basis = nullptr;
  xc_basis* aux = nullptr;
  std::vector<JPair> pairs;
  int64_t herm_total = 0;
  int ncart_aux = 0;
  std::vector<int> cart_off;  // first Cartesian function of every auxiliary shell
  int naux = 0;               // auxiliary primitives
  int64_t aherm_total = 0;
  JView view{};               // class offsets; its arrays are d_pair, d_aux and d_boys
  DBuf<JPair> d_pairs;
  DBuf<int> d_cart_off, d_prim_shell, d_shell_prim;
  DBuf<double> d_pair, d_aux, d_prim_coef, d_boys;
  // work items of [0: the right-hand side, 1: the potential]
  std::vector<JItem> items[2][kJClasses];
  DBuf<JItem> d_items[2][kJClasses];
  std::vector<JPairItem> pair_items[kJPairClasses];
  DBuf<JPairItem> d_pair_items[kJPairClasses];
  DBuf<double> d_D, d_V, d_U, d_bc, d_cc, d_P, d_J;
  // the metric's Cholesky factor (lower, row-major), the inverses of its diagonal blocks, and the solves' vectors
  DBuf<double> d_L, d_dinv, d_b, d_y;
  void plan_items();
};

namespace {

// Boys functions at the table's nodes: the confluent series in extended precision.
std::vector<double> boys_table() {
  std::vector<double> tab((size_t)kBoysRows * kBoysCols);
  for (int i = 0; i < kBoysRows; ++i) {
    const long double T = (long double)i / kBoysPerUnit, e = expl(-T);
    tab[(size_t)i * kBoysCols] = (double)e;
    for (int m = 0; m + 1 < kBoysCols; ++m) {
      long double term = 1.0L / (2 * m + 1), sum = term;
      for (int k = 1; term > 1e-22L * sum; ++k) {
        term *= 2.0L * T / (2 * m + 2 * k + 1);
        sum += term;
      }
      tab[(size_t)i * kBoysCols + 1 + m] = (double)(e * sum);
    }
  }
  return tab;
}

}  // namespace

// Items of the meetings, the largest L + l first.  An item is one wavefront.  Its length is set by
// the operations of a meeting, so that the items take about the same time and there are about
// kTarget of them (the chip holds 1024 to 4096 of these wavefronts at once), but at most 64
// (potential) or 512 (right-hand side) meetings per lane, where the atomic additions at an item's
// end no longer show, and at least 2.  With one length for all classes the few pairs of f and d
// shells made a few long items: 32.6 of 51 ms of (H2O)32/def2-TZVP went to 0.4 % of the meetings.
void xc_coulomb::plan_items() {
  // steps 1 and 5: runs of at most 64 pairs of one kind of shells
  const auto& sh = basis->shells;
  const auto kind = [&](const JPair& q) {
    return ((sh[q.A].l * 2 + sh[q.A].pure) * (kJMaxLPrim + 1) + sh[q.B].l) * 2 + sh[q.B].pure;
  };
  for (size_t q = 0; q < pairs.size();) {
    size_t e = q + 1;
    while (e < pairs.size() && e < q + 64 && kind(pairs[e]) == kind(pairs[q])) ++e;
    const DevShell &A = sh[pairs[q].A], &B = sh[pairs[q].B];
    pair_items[A.l + B.l > kJPairTop].push_back(
        JPairItem{A.l, B.l, (int)q, (int)(e - q), A.nfunc, B.nfunc, A.ang_off, B.ang_off});
    q = e;
  }
  constexpr int kTarget = 16384, kMaxLab = 2 * kJMaxLPrim;
  const auto hcount = [](int L) { return (L + 1) * (L + 2) * (L + 3) / 6; };
  const auto cost = [&](int L, int l) {
    double c = 60.0 + 2.0 * hcount(L) * hcount(l);
    for (int i = 0; i <= L + l; ++i) c += 3.0 * hcount(i);
    return L + l > kJClassTop[1] ? 4.0 * c : c;  // these spill registers
  };
  const auto width_of = [&](int l, int na) {  // lanes per pair in the right-hand side
    if (l < kJGroupL) return 64;
    int w = 1;
    while (w < na && w < 64) w *= 2;
    return w;
  };
  double pot = 0.0, rhs = 0.0;
  for (int L = 0; L <= kMaxLab; ++L) {
    const int64_t nq = view.pair0[L + 1] - view.pair0[L];
    for (int l = 0; l <= kJMaxLAux; ++l) {
      const int64_t na = view.aux0[l + 1] - view.aux0[l];
      if (!na || !nq) continue;
      const int w = width_of(l, (int)na);
      pot += cost(L, l) * (double)((nq + 63) / 64 * na);
      rhs += cost(L, l) * (double)((na + w - 1) / w * ((nq * w + 63) / 64));
    }
  }
  const auto length = [&](double total, int L, int l, double hi) {
    return (int)std::min(std::max(std::round(total / kTarget / cost(L, l)), 2.0), hi);
  };
  for (int M = kMaxLab + kJMaxLAux; M >= 0; --M) {
    const int cls = M <= kJClassTop[0] ? 0 : M <= kJClassTop[1] ? 1 : 2;
    for (int L = std::max(0, M - kJMaxLAux); L <= std::min(M, kMaxLab); ++L) {
      const int l = M - L;
      const int q0 = view.pair0[L], q1 = view.pair0[L + 1], a0 = view.aux0[l], a1 = view.aux0[l + 1];
      if (q0 == q1 || a0 == a1) continue;
      const int pot_len = length(pot, L, l, 64.0);
      for (int q = q0; q < q1; q += 64)
        for (int a = a0; a < a1; a += pot_len)
          items[1][cls].push_back(JItem{L, l, q, std::min(64, q1 - q), a, std::min(pot_len, a1 - a)});
      const int w = width_of(l, a1 - a0), nq = length(rhs, L, l, 512.0) * (64 / w);
      for (int a = a0; a < a1; a += w)
        for (int q = q0; q < q1; q += nq) items[0][cls].push_back(JItem{L, l, q, std::min(nq, q1 - q), a, w});
    }
  }
}

struct xc_grid {
  xc_ctx* ctx = nullptr;
  int64_t npts = 0;
  DBuf<double> d_pts, d_w;
};

struct xc_bfogc {
  xc_ctx* ctx = nullptr;
  xc_basis* basis = nullptr;
  xc_grid* grid = nullptr;
  int bs = 128;
  double radial_thr = 1e-9;
  int deriv = 1, ncomp = 4, nblocks = 0;
  std::vector<DevBlock> blocks;
  int64_t tile_elems = 0;
  int64_t sum_nb = 0;
  double sum_B_nb2 = 0.0;
  DBuf<DevBlock> d_blocks;
  DBuf<int> d_ao_idx, d_sig_shell, d_sig_pos;
  DBuf<double> d_t64;
  DBuf<float> d_t32;
  // contraction work lists
  int npass_max = 0;
  std::vector<WorkItem> dens_work;
  std::vector<FockItem> fock_items[kFockShapes];  // by workgroup shape
  DBuf<WorkItem> d_dens_work;
  // mixed precision: every block's density items contiguously (from dens_item0[b]); the device lists
  // of the dense blocks refined in FP64 and their counts; the FP32-rounded density matrix in FP64
  std::vector<WorkItem> dens_by_block;
  std::vector<int> dens_item0;
  DBuf<WorkItem> d_dens_by_block, d_dense_list, d_carry_list;
  DBuf<int> d_dens_item0, d_dense_cnt, d_carry_cnt;
  // mixed precision: the blocks contracted in FP64 by the last mixed build that were still dense
  // (one byte per block); the next mixed build's FP32 pass skips them
  DBuf<unsigned char> d_dense_mask;
  DBuf<double> d_P32d;
  DBuf<FockItem> d_fock_items[kFockShapes];
  // per-build work buffers
  DBuf<double> d_part, d_rho, d_grad, d_vs, d_gw, d_eblk, d_U, d_P, d_F, d_v, d_g;
  // Fock sub-tile scratch (FP64 size when FP64 tiles are kept, else FP32) and the row entries of
  // the reduce (sorted by AO row, then block)
  int64_t t_elems = 0;
  DBuf<double> d_T;
  DBuf<RowEnt> d_rowent;
  DBuf<int> d_rowptr;
  DBuf<float> d_P32;
  DBuf<double> d_round;  // row or finalize-block partials of the FP32 rounding term, per spin
  // supersystem density of a non-additive build with this controller active (allocated on first use)
  DBuf<double> d_rho_sup, d_grad_sup, d_rho_sup_b, d_grad_sup_b;
  // cached grid density (xc_bfogc_update_density) and the energies of it per functional
  DBuf<double> d_rho_c, d_grad_c, d_ecache;
  bool rho_c_valid = false, rho_c_grad = false;
  // nuclear gradient (allocated on first use): per-AO partials, atom map, result
  DBuf<double> d_gacc, d_gout;
  DBuf<int> d_ao_atom;
  // unrestricted builds (allocated on first use): beta density, potential, P and F
  DBuf<double> d_rho_b, d_grad_b, d_vs_b, d_gw_b, d_Pb, d_Fb;
  // the other spin's scratch of a build that runs both spins at once (kPairUnknown until first asked for)
  DBuf<double> d_part_b, d_T_b, d_U_b;
  DBuf<PackSys> d_pair;
  enum { kPairUnknown, kPairYes, kPairNo } pair = kPairUnknown;
  DBuf<float> d_P32b;
  bool ecache_valid[kNumFunctionals] = {};
  // serving: a build of this controller is in flight on a server slot; captured builds
  bool in_flight = false;
  std::map<std::pair<int, double>, hipGraphExec_t> graphs;  // (functional + 16 precision, threshold)
  ~xc_bfogc() {
    for (auto& kv : graphs) (void)hipGraphExecDestroy(kv.second);
    keep_pair();
  }
  // no longer among the context's spare scratches
  void keep_pair() {
    if (!ctx) return;
    auto& v = ctx->spare;
    v.erase(std::remove(v.begin(), v.end(), this), v.end());
  }
  void drop_pair() {
    d_part_b.free_();
    d_T_b.free_();
    d_U_b.free_();
  }
};

void xc_ctx::reclaim() {
  for (xc_bfogc* bf : spare) {
    bf->drop_pair();
    bf->pair = xc_bfogc::kPairNo;
  }
  spare.clear();
}

namespace {

// Launch order and lanes of a stage's work classes: the non-empty classes, the
// largest first, dealt round-robin over the lanes (fork / join only when more
// than one class has work).
template <typename F>
void over_lanes(const Lanes& L, int nclass, const std::function<int(int)>& count, F&& launch) {
  int nz = 0;
  for (int c = nclass - 1; c >= 0; --c) nz += count(c) > 0 ? 1 : 0;
  const bool par = nz > 1 && L.n > 1;
  if (par) L.fork_all();
  int k = 0;
  for (int c = nclass - 1; c >= 0; --c)
    if (count(c) > 0) launch(c, par ? L.lane(k++) : L.main);
  if (par) L.join_all();
}

// A density without its gradient as the quadratic form over half of the folded matrix: where a
// block can have more than one column pass (a pass contracts everything up to its last column, so one
// pass saves nothing and the fold's launch costs 4 us).
bool use_form(bool gga, int n) { return !gga && n > 16 * kDensMaxS; }

template <typename T>
void run_density(xc_bfogc* bf, const T* tiles, const T* P, int want_grad, const Lanes& L, bool form = false) {
  launch_density_sub<T>(L.main, bf->d_dens_work.p, (int)bf->dens_work.size(), bf->d_blocks.p, bf->d_ao_idx.p, tiles,
                        P, bf->basis->nao, want_grad, bf->d_part.p, bf->grid->npts, nullptr, nullptr, nullptr, form);
}

// Mixed precision: the FP32 density pass, and FP64 density items (FP64 tiles, the FP32-rounded P
// in FP64) for the blocks whose largest density exceeds kMixedRhoThreshold.  The controller's mask
// holds the blocks the last mixed build found dense: their FP64 items run beside the FP32 pass over
// the other blocks (on a helper lane), then the blocks outside
// the mask that the FP32 pass finds dense get theirs, and the mask keeps the blocks whose FP64
// density exceeds the threshold.  The lists are filled on the device, so those launches cover the
// lists' capacity and run only the filled part.
void run_density_mixed(xc_bfogc* bf, int want_grad, const Lanes& L) {
  const DenseList carry = {bf->d_carry_list.p, bf->d_carry_cnt.p}, late = {bf->d_dense_list.p, bf->d_dense_cnt.p};
  const int n = bf->basis->nao, nwork = (int)bf->dens_work.size();
  const int64_t N = bf->grid->npts;
  auto fp64_pass = [&](hipStream_t s, const DenseList& list) {
    launch_density_sub<double>(s, list.item, nwork, bf->d_blocks.p, bf->d_ao_idx.p, bf->d_t64.p, bf->d_P32d.p, n,
                               want_grad, bf->d_part.p, N, nullptr, list.count);
  };
  launch_list_masked(L.main, bf->d_blocks.p, bf->nblocks, bf->d_dens_by_block.p, bf->d_dens_item0.p, carry,
                     bf->d_dense_mask.p);
  over_lanes(L, 2, [&](int) { return nwork; }, [&](int c, hipStream_t s) {
    if (c == 1)
      launch_density_sub<float>(s, bf->d_dens_work.p, nwork, bf->d_blocks.p, bf->d_ao_idx.p, bf->d_t32.p, bf->d_P32.p,
                                n, want_grad, bf->d_part.p, N, nullptr, nullptr, bf->d_dense_mask.p);
    else
      fp64_pass(s, carry);
  });
  launch_mark_dense(L.main, bf->d_blocks.p, bf->nblocks, N, bf->d_part.p, kMixedRhoThreshold, bf->d_dens_by_block.p,
                    bf->d_dens_item0.p, late, bf->d_dense_mask.p);
  fp64_pass(L.main, late);
  launch_refresh_dense(L.main, bf->d_blocks.p, bf->nblocks, N, bf->d_part.p, kMixedRhoThreshold,
                       bf->d_dense_mask.p);
}

// A controller whose server build is still running owns its work buffers (P, partial
// densities, potentials, U) until the build completes: refuse any other use first.
void require_idle(const xc_bfogc* bf, const char* who) {
  require(!bf->in_flight, XC_ERR_STATE, std::string(who) + ": a server build of this controller is in flight");
}

void require_idle(const xc_bfogc* act, int nenv, xc_bfogc* const* env, const char* who) {
  require_idle(act, who);
  for (int i = 0; i < nenv; ++i)
    if (env && env[i]) require_idle(env[i], who);
}

// The Fock stage in two steps: the blocks' sub-tiles into the scratch (run_fock_tiles), then the
// row reduce into the lower triangle of U (run_fock_reduce; every element of that triangle is
// written, so U needs no clearing).  run_fock does both.
template <typename T>
void run_fock_tiles(xc_bfogc* bf, const T* tiles, int gga, double thr, const Lanes& L, const double* vs = nullptr,
                    const double* gw = nullptr) {
  if (!vs) vs = bf->d_vs.p;
  if (!gw) gw = bf->d_gw.p;
  T* Tscr = reinterpret_cast<T*>(bf->d_T.p);
  over_lanes(L, kFockShapes, [&](int c) { return (int)bf->fock_items[c].size(); }, [&](int c, hipStream_t s) {
    launch_fock_sub<T>(s, c, bf->d_fock_items[c].p, (int)bf->fock_items[c].size(), bf->d_blocks.p, tiles, vs, gw, gga,
                       thr, Tscr, bf->grid->npts);
  });
}

template <typename T>
void run_fock_reduce(xc_bfogc* bf, const Lanes& L, const ReduceOut& out = ReduceOut{},
                     const EnvEnergies& env = EnvEnergies{}) {
  launch_fock_reduce<T>(L.main, bf->d_rowent.p, bf->d_rowptr.p, reinterpret_cast<const T*>(bf->d_T.p),
                        bf->d_ao_idx.p, bf->d_U.p, bf->basis->nao, nullptr, 1, bf->ctx->deterministic,
                        bf->sum_nb > 256 * (int64_t)bf->nblocks, out, env);
}

// The reduce and what follows it: F (overwritten), the FP32 rounding partials of one spin (P32 given;
// the spin's slot of d_round), and E = the sum of the block energies (E given) plus the rounding
// partials of nspin slots (less the environment's energies: small matrices only).  Small matrices get
// their rows and the energy from the reduce itself.
template <typename T>
void run_fock_finish(xc_bfogc* bf, const Lanes& L, double* dF, const double* P, const float* P32, int spin, int nspin,
                     double* E, const EnvEnergies& env = EnvEnergies{}) {
  hipStream_t s = L.main;
  const int n = bf->basis->nao;
  const int nxc = (int)((bf->grid->npts + kTile - 1) / kTile);
  const bool direct = n <= kDirectRows;
  const int nround = direct ? n : finalize_blocks(n);
  double* round = P32 ? bf->d_round.p + (size_t)spin * nround : nullptr;
  if (direct) {
    run_fock_reduce<T>(bf, L, ReduceOut{true, dF, P, P32, round, bf->d_eblk.p, nxc, P32 ? nullptr : E}, env);
  } else {
    run_fock_reduce<T>(bf, L);
    if (s == bf->ctx->stream && nspin == 1) bf->ctx->mark();
    launch_finalize(s, bf->d_U.p, dF, n, 0, P32 ? P : nullptr, P32, round);
  }
  if (s == bf->ctx->stream && nspin == 1 && direct) bf->ctx->mark();
  if (E && (P32 || !direct))
    launch_sum(s, bf->d_eblk.p, nxc, E, 0, P32 ? bf->d_round.p : nullptr, P32 ? (int64_t)nspin * nround : 0);
}

// Whether an unrestricted build runs both spins in each launch.  A spin's density and Fock kernels leave a
// tail of idle compute units and read the same tiles: (H2O)5/def2-TZVP (215 AOs, 63 392
// points) 600 us one after the other, 482 at once (densities 197 -> 166, Fock stages 200 -> 160).
// For matrices that take the direct reduce and 128-point blocks; it needs a second scratch of each kind,
// and a controller that has no room for it, or had to give it back, keeps one spin after the other.
bool pair_buffers(xc_bfogc* bf) {
  if (bf->pair == xc_bfogc::kPairNo) return false;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  HIPX(hipStreamIsCapturing(bf->ctx->stream, &st));
  if (st != hipStreamCaptureStatusNone) {
    // a build that is recorded into a graph allocates nothing: undecided, it runs one spin after the
    // other; the scratch that a graph holds stays for the controller's life
    if (bf->pair == xc_bfogc::kPairYes) bf->keep_pair();
    return bf->pair == xc_bfogc::kPairYes;
  }
  if (bf->pair == xc_bfogc::kPairYes) return true;
  const size_t n = (size_t)bf->basis->nao;
  auto found = xc_bfogc::kPairNo;
  if (n <= kDirectRows && bf->bs == kTile) {
    try {
      bf->d_part_b.alloc(bf->ctx, bf->d_part.n, false);
      bf->d_T_b.alloc(bf->ctx, bf->d_T.n, false);
      bf->d_U_b.alloc(bf->ctx, n * n, false);
      bf->d_pair.alloc(bf->ctx, 2, false);
      bf->ctx->spare.push_back(bf);
      found = xc_bfogc::kPairYes;
    } catch (const XcError& e) {
      bf->drop_pair();
      if (e.code != XC_ERR_MEMORY) throw;
    }
  }
  bf->pair = found;
  return found == xc_bfogc::kPairYes;
}

// Both spins of an unrestricted build in each launch.
template <typename T>
void enqueue_build_pair(xc_bfogc* bf, int functional, double thr, const double* const* Ps, double* const* Fs,
                               const Lanes& L, double* d_energy) {
  constexpr bool fp32 = sizeof(T) == 4;
  hipStream_t s = L.main;
  const int n = bf->basis->nao;
  const int64_t N = bf->grid->npts;
  const int nxc = (int)((N + kTile - 1) / kTile);
  const int g = functional_is_gga(functional) ? 1 : 0;
  const bool form = !fp32 && use_form(g, n);
  PackPair pair{};
  for (int sp = 0; sp < 2; ++sp) {
    PackSys& ps = pair.s[sp];
    ps.tiles = fp32 ? (const void*)bf->d_t32.p : (const void*)bf->d_t64.p;
    ps.P64 = Ps[sp];
    ps.P32 = fp32 ? (sp ? bf->d_P32b.p : bf->d_P32.p) : nullptr;
    ps.U = sp ? bf->d_U_b.p : bf->d_U.p;
    ps.P = fp32 ? (const void*)ps.P32 : form ? (const void*)ps.U : (const void*)Ps[sp];
    ps.ao_idx = bf->d_ao_idx.p;
    ps.part = sp ? bf->d_part_b.p : bf->d_part.p;
    ps.w = bf->grid->d_w.p;
    ps.vs = sp ? bf->d_vs_b.p : bf->d_vs.p;
    ps.gw = sp ? bf->d_gw_b.p : bf->d_gw.p;
    ps.T = sp ? bf->d_T_b.p : bf->d_T.p;
    ps.ent = bf->d_rowent.p;
    ps.row_ptr = bf->d_rowptr.p;
    ps.F = Fs[sp];
    ps.eblk = bf->d_eblk.p;
    ps.round = bf->d_round.p + (size_t)sp * (fp32 ? n : 0);
    ps.E = sp == 1 && !fp32 ? d_energy : nullptr;  // (FP32: with the rounding term below)
    ps.npts = N;
    ps.n = n;
    ps.nxc = nxc;
  }
  const PackSys* sys = bf->d_pair.p;
  launch_set_pair(s, pair, bf->d_pair.p);
  if (fp32) launch_pack_to_float(s, sys, 2, (int64_t)n * n);
  if (form) launch_fold(s, nullptr, nullptr, n, sys, 2);
  launch_density_sub<T>(s, bf->d_dens_work.p, (int)bf->dens_work.size(), bf->d_blocks.p, nullptr, nullptr, nullptr, 0, g,
                        nullptr, 0, sys, nullptr, nullptr, form, true);
  launch_functional_pol(s, functional, N, kTile, nullptr, nullptr, nullptr, nullptr, bf->grid->d_w.p, bf->d_vs.p,
                        bf->d_gw.p, bf->d_vs_b.p, bf->d_gw_b.p, bf->d_eblk.p, nullptr, nullptr, nullptr, nullptr,
                        bf->d_blocks.p, bf->d_part.p, bf->d_part_b.p);
  over_lanes(L, kFockShapes, [&](int c) { return (int)bf->fock_items[c].size(); }, [&](int c, hipStream_t st) {
    launch_fock_sub<T>(st, c, bf->d_fock_items[c].p, (int)bf->fock_items[c].size(), bf->d_blocks.p, nullptr, nullptr,
                       nullptr, g, thr, nullptr, 0, sys, true);
  });
  ReduceOut out{};
  out.direct = true;
  out.round = fp32 ? bf->d_round.p : nullptr;
  launch_fock_reduce<T>(s, nullptr, nullptr, nullptr, nullptr, nullptr, n, sys, 2, bf->ctx->deterministic,
                        bf->sum_nb > 256 * (int64_t)bf->nblocks, out);
  // with the first-order FP32 rounding term of each spin density matrix (dE_xc/dP_s = F_s)
  if (fp32) launch_sum(s, bf->d_eblk.p, nxc, d_energy, 0, bf->d_round.p, 2 * (int64_t)n);
  HIPX(hipGetLastError());
}

template <typename T>
void run_fock(xc_bfogc* bf, const T* tiles, int gga, double thr, const Lanes& L, const double* vs = nullptr,
              const double* gw = nullptr) {
  run_fock_tiles<T>(bf, tiles, gga, thr, L, vs, gw);
  run_fock_reduce<T>(bf, L);
}

}  // namespace

namespace {
// Shell list of the host integral entry points (flat arrays as in xc_basis_create).
std::vector<Shell> host_shells(const char* who, int nshell, const int* shell_l, const int* shell_pure,
                               const int* shell_nprim, const double* shell_center, const double* alpha,
                               const double* coef, int lmax) {
  require(nshell > 0 && shell_l && shell_pure && shell_nprim && shell_center && alpha && coef, XC_ERR_ARG,
          std::string(who) + ": bad shell arguments");
  std::vector<Shell> sh(nshell);
  int k = 0;
  for (int s = 0; s < nshell; ++s) {
    sh[s].l = shell_l[s];
    sh[s].pure = shell_pure[s] != 0;
    require(sh[s].l >= 0 && sh[s].l <= lmax, XC_ERR_INPUT,
            std::string(who) + ": angular momentum above " + std::to_string(lmax));
    require(shell_nprim[s] > 0, XC_ERR_INPUT, std::string(who) + ": shell without primitives");
    sh[s].center = {shell_center[3 * s], shell_center[3 * s + 1], shell_center[3 * s + 2]};
    for (int q = 0; q < shell_nprim[s]; ++q, ++k) {
      sh[s].alpha.push_back(alpha[k]);
      sh[s].coef.push_back(coef[k]);
    }
  }
  return sh;
}
int nao_of(const std::vector<Shell>& sh) {
  int n = 0;
  for (const auto& s : sh) n += s.nfunc();
  return n;
}
}  // namespace

extern "C" {

const char* xc_last_error(void) { return g_last_error.c_str(); }

int xc_version(void) { return 1; }

int xc_ctx_create(int device, xc_ctx** out) {
  return guarded([&] {
    require(out != nullptr, XC_ERR_ARG, "xc_ctx_create: null output");
    int ndev = 0;
    HIPX(hipGetDeviceCount(&ndev));
    require(device >= 0 && device < ndev, XC_ERR_ARG, "xc_ctx_create: no HIP device " + std::to_string(device));
    auto* c = new xc_ctx();
    c->device = device;
    HIPX(hipSetDevice(device));
    noalloc_setup_current_device(device);
    HIPX(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    c->lanes.create(c->stream, true);
    HIPX(hipHostMalloc((void**)&c->energy, 2 * sizeof(double), hipHostMallocMapped | hipHostMallocCoherent));
    c->energy[0] = c->energy[1] = 0.0;
    c->flag = reinterpret_cast<int*>(c->energy + 1);
    c->stage.create();
    *out = c;
  });
}

int xc_ctx_destroy(xc_ctx* ctx) {
  return guarded([&] {
    if (!ctx) return;
    require(ctx->live_handles == 0, XC_ERR_STATE,
            "xc_ctx_destroy: " + std::to_string(ctx->live_handles) + " basis/grid/controller handles still alive");
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (auto e : ctx->ev_pool) (void)hipEventDestroy(e);
    ctx->stage.destroy();
    (void)hipHostFree(ctx->energy);
    if (ctx->pack_energy) (void)hipHostFree(ctx->pack_energy);
    delete ctx->pack;
    ctx->pack = nullptr;
    for (auto& kv : ctx->pack_graphs) delete kv.second;
    ctx->pack_graphs.clear();
    ctx->lanes.destroy();
    (void)hipStreamDestroy(ctx->stream);
    ctx->trim();
    delete ctx;
  });
}

int xc_ctx_synchronize(xc_ctx* ctx) {
  return guarded([&] {
    require(ctx, XC_ERR_ARG, "null context");
    HIPX(hipStreamSynchronize(ctx->stream));
  });
}

void* xc_ctx_stream(xc_ctx* ctx) { return ctx ? (void*)ctx->stream : nullptr; }

int xc_ctx_memory(xc_ctx* ctx, int64_t* bytes_in_use) {
  return guarded([&] {
    require(ctx && bytes_in_use, XC_ERR_ARG, "null argument");
    *bytes_in_use = ctx->bytes;
  });
}

void xc_free_host(void* p) { std::free(p); }

int xc_normalize_contraction(int l, int nprim, const double* alpha, double* coef) {
  return guarded([&] {
    require(l >= 0 && nprim > 0 && alpha && coef, XC_ERR_ARG, "xc_normalize_contraction: bad arguments");
    std::vector<double> a(alpha, alpha + nprim), c(coef, coef + nprim);
    renormalize_contraction(l, a, c);
    std::copy(c.begin(), c.end(), coef);
  });
}

int xc_load_basis(const char* path, int natoms, const int* Z, const double* coords, int pure, int* nshell,
                  int** shell_l, int** shell_nprim, int** shell_atom, double** shell_center, double** alpha,
                  double** coef) {
  return guarded([&] {
    require(path && natoms > 0 && Z && coords && nshell && shell_l && shell_nprim && shell_atom && shell_center &&
                alpha && coef,
            XC_ERR_ARG, "xc_load_basis: bad arguments");
    static const char* symbols[] = {"",  "h",  "he", "li", "be", "b",  "c",  "n",  "o",  "f",  "ne", "na", "mg",
                                    "al", "si", "p",  "s",  "cl", "ar", "k",  "ca", "sc", "ti", "v",  "cr", "mn",
                                    "fe", "co", "ni", "cu", "zn", "ga", "ge", "as", "se", "br", "kr"};
    std::vector<Shell> all;
    for (int a = 0; a < natoms; ++a) {
      require(Z[a] >= 1 && Z[a] <= 36, XC_ERR_INPUT, "xc_load_basis: element out of range");
      auto sh = parse_turbomole_basis(path, symbols[Z[a]], pure != 0);
      for (auto& s : sh) {
        s.center = {coords[3 * a], coords[3 * a + 1], coords[3 * a + 2]};
        s.atom = a;
        all.push_back(s);
      }
    }
    const int ns = (int)all.size();
    int np = 0;
    for (auto& s : all) np += (int)s.alpha.size();
    *nshell = ns;
    *shell_l = (int*)std::malloc(sizeof(int) * ns);
    *shell_nprim = (int*)std::malloc(sizeof(int) * ns);
    *shell_atom = (int*)std::malloc(sizeof(int) * ns);
    *shell_center = (double*)std::malloc(sizeof(double) * 3 * ns);
    *alpha = (double*)std::malloc(sizeof(double) * np);
    *coef = (double*)std::malloc(sizeof(double) * np);
    int k = 0;
    for (int s = 0; s < ns; ++s) {
      (*shell_l)[s] = all[s].l;
      (*shell_nprim)[s] = (int)all[s].alpha.size();
      (*shell_atom)[s] = all[s].atom;
      for (int d = 0; d < 3; ++d) (*shell_center)[3 * s + d] = all[s].center[d];
      for (size_t q = 0; q < all[s].alpha.size(); ++q, ++k) {
        (*alpha)[k] = all[s].alpha[q];
        (*coef)[k] = all[s].coef[q];
      }
    }
  });
}

int xc_molecular_grid(int natoms, const int* Z, const double* coords, int grid_type, int radial_type, int accuracy,
                      int smoothing, double weight_threshold, int sort, int64_t* npoints, double** points,
                      double** weights, int64_t* npoints_before_cut) {
  return guarded([&] {
    require(natoms > 0 && Z && coords && npoints && points && weights, XC_ERR_ARG, "xc_molecular_grid: bad arguments");
    require(grid_type >= 0 && grid_type <= 2 && radial_type >= 0 && radial_type <= 4, XC_ERR_ARG,
            "xc_molecular_grid: unknown grid or radial type");
    GridSettings s;
    s.type = (GridType)grid_type;
    s.radial = (RadialType)radial_type;
    s.accuracy = accuracy;
    s.smoothing = (unsigned)smoothing;
    s.weight_threshold = weight_threshold;
    s.sort = sort != 0;
    MolecularGrid g = build_molecular_grid(std::vector<int>(Z, Z + natoms), std::vector<double>(coords, coords + 3 * natoms), s);
    const int64_t n = (int64_t)g.weights.size();
    *npoints = n;
    *points = (double*)std::malloc(sizeof(double) * 3 * std::max<int64_t>(n, 1));
    *weights = (double*)std::malloc(sizeof(double) * std::max<int64_t>(n, 1));
    std::memcpy(*points, g.points.data(), sizeof(double) * 3 * n);
    std::memcpy(*weights, g.weights.data(), sizeof(double) * n);
    if (npoints_before_cut) *npoints_before_cut = g.n_before_cut;
  });
}

int xc_molecular_grid_device(xc_ctx* ctx, int natoms, const int* Z, const double* coords, int grid_type,
                             int radial_type, int accuracy, int smoothing, double weight_threshold, int sort,
                             int64_t* npoints, double** points, double** weights, int64_t* npoints_before_cut) {
  return guarded([&] {
    require(ctx && natoms > 0 && Z && coords && npoints && points && weights, XC_ERR_ARG,
            "xc_molecular_grid_device: bad arguments");
    require(grid_type >= 0 && grid_type <= 2 && radial_type >= 0 && radial_type <= 4, XC_ERR_ARG,
            "xc_molecular_grid_device: unknown grid or radial type");
    GridSettings s;
    s.type = (GridType)grid_type;
    s.radial = (RadialType)radial_type;
    s.accuracy = accuracy;
    s.smoothing = (unsigned)smoothing;
    s.weight_threshold = weight_threshold;
    s.sort = sort != 0;
    // everything after the per-element reference grids runs on the device: candidates, partition,
    // weight cut, Hilbert order
    const GridProblem P = grid_problem(std::vector<int>(Z, Z + natoms),
                                       std::vector<double>(coords, coords + 3 * natoms), s, false);
    const int64_t nc = P.cand_off.back();
    require(nc < (int64_t)1 << 31, XC_ERR_ARG, "xc_molecular_grid_device: too many candidate points");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    DBuf<double> d_xyz, d_dist, d_apair, d_min, d_ref_xyz, d_ref_w, d_w, d_pts, d_pw, d_part, d_box, d_opts, d_ow;
    DBuf<int64_t> d_ref_off, d_cand_off, d_key, d_key2, d_idx, d_order;
    DBuf<int> d_keep, d_pos;
    DBuf<unsigned char> d_temp;
    d_xyz.upload(ctx, P.xyz.data(), P.xyz.size());
    d_dist.upload(ctx, P.dist.data(), P.dist.size());
    d_apair.upload(ctx, P.apair.data(), P.apair.size());
    d_min.upload(ctx, P.min_dist.data(), P.min_dist.size());
    d_ref_xyz.upload(ctx, P.ref_xyz.data(), P.ref_xyz.size());
    d_ref_w.upload(ctx, P.ref_w.data(), P.ref_w.size());
    d_ref_off.upload(ctx, P.ref_off.data(), P.ref_off.size());
    d_cand_off.upload(ctx, P.cand_off.data(), P.cand_off.size());
    const size_t ncs = (size_t)std::max<int64_t>(nc, 1);
    d_w.alloc(ctx, ncs);
    d_keep.alloc(ctx, ncs);
    d_pos.alloc(ctx, ncs);
    d_pts.alloc(ctx, 3 * ncs);
    d_pw.alloc(ctx, ncs);
    launch_partition_gen(st, P.type, P.smoothing, P.natoms, d_xyz.p, d_dist.p, d_apair.p, d_min.p, nc, d_ref_xyz.p,
                         d_ref_w.p, d_ref_off.p, d_cand_off.p, weight_threshold, d_w.p, d_keep.p);
    const size_t scan_bytes = grid_scan_temp_bytes(nc);
    d_temp.alloc(ctx, std::max<size_t>(scan_bytes, 1));
    launch_cut(st, P.natoms, d_xyz.p, nc, d_ref_xyz.p, d_ref_off.p, d_cand_off.p, d_w.p, d_keep.p, d_pos.p, d_temp.p,
               scan_bytes, d_pts.p, d_pw.p);
    HIPX(hipGetLastError());
    int last[2] = {0, 0};
    if (nc)
      ctx->stage.down(st, {{&last[0], d_pos.p + nc - 1, sizeof(int)}, {&last[1], d_keep.p + nc - 1, sizeof(int)}});
    const int64_t n = (int64_t)last[0] + last[1];
    const double* res_pts = d_pts.p;
    const double* res_w = d_pw.p;
    if (s.sort && n >= 2) {
      const int64_t length = hilbert_length(n);
      d_part.alloc(ctx, 6 * (size_t)bbox_part_count());
      d_box.alloc(ctx, 6);
      launch_bbox(st, d_pts.p, n, length, d_part.p, d_box.p);
      const size_t sort_bytes = grid_sort_temp_bytes(n);
      if (sort_bytes > d_temp.n) d_temp.alloc(ctx, sort_bytes);
      d_key.alloc(ctx, n);
      d_key2.alloc(ctx, n);
      d_idx.alloc(ctx, n);
      d_order.alloc(ctx, n);
      d_opts.alloc(ctx, 3 * (size_t)n);
      d_ow.alloc(ctx, n);
      launch_hilbert_order(st, d_pts.p, d_pw.p, n, d_box.p, length, d_key.p, d_key2.p, d_idx.p, d_order.p, d_temp.p,
                           sort_bytes, d_opts.p, d_ow.p);
      HIPX(hipGetLastError());
      res_pts = d_opts.p;
      res_w = d_ow.p;
    }
    *npoints = n;
    *points = (double*)std::malloc(sizeof(double) * 3 * std::max<int64_t>(n, 1));
    *weights = (double*)std::malloc(sizeof(double) * std::max<int64_t>(n, 1));
    ctx->stage.down(st, {{*points, res_pts, sizeof(double) * 3 * n}, {*weights, res_w, sizeof(double) * n}});
    if (npoints_before_cut) *npoints_before_cut = nc;
  });
}

int xc_hilbert_sort(int64_t npoints, double* points, double* weights) {
  return guarded([&] {
    require(npoints >= 0 && (npoints == 0 || (points && weights)), XC_ERR_ARG, "xc_hilbert_sort: bad arguments");
    std::vector<double> p(points, points + 3 * npoints), w(weights, weights + npoints);
    hilbert_sort(p, w);
    std::copy(p.begin(), p.end(), points);
    std::copy(w.begin(), w.end(), weights);
  });
}

int xc_lebedev(int npoints, double* x, double* y, double* z, double* w) {
  return guarded([&] {
    require(x && y && z && w, XC_ERR_ARG, "xc_lebedev: null output");
    std::vector<double> vx, vy, vz, vw;
    lebedev_rule(npoints, vx, vy, vz, vw);
    std::copy(vx.begin(), vx.end(), x);
    std::copy(vy.begin(), vy.end(), y);
    std::copy(vz.begin(), vz.end(), z);
    std::copy(vw.begin(), vw.end(), w);
  });
}


int xc_overlap(int nshell, const int* shell_l, const int* shell_pure, const int* shell_nprim, const double* shell_center,
               const double* alpha, const double* coef, double* S) {
  return guarded([&] {
    require(S, XC_ERR_ARG, "xc_overlap: null output");
    auto sh = host_shells("xc_overlap", nshell, shell_l, shell_pure, shell_nprim, shell_center, alpha, coef, 6);
    std::vector<double> out;
    overlap_matrix(sh, out);
    std::copy(out.begin(), out.end(), S);
  });
}

int xc_boys(int m, double T, double* F) {
  return guarded([&] {
    require(F && m >= 0 && m <= 17 && T >= 0.0, XC_ERR_ARG, "xc_boys: bad arguments");
    *F = boys_function(m, T);
  });
}

int xc_one_electron(int nshell, const int* shell_l, const int* shell_pure, const int* shell_nprim,
                    const double* shell_center, const double* alpha, const double* coef, int natoms, const int* Z,
                    const double* coords, double* T, double* V) {
  return guarded([&] {
    require(natoms >= 0 && (natoms == 0 || (Z && coords)) && T && V, XC_ERR_ARG, "xc_one_electron: bad arguments");
    auto sh = host_shells("xc_one_electron", nshell, shell_l, shell_pure, shell_nprim, shell_center, alpha, coef, 4);
    std::vector<int> z(Z, Z + natoms);
    std::vector<double> x(coords, coords + 3 * natoms), t, v;
    one_electron_matrices(sh, z, x, t, v);
    std::copy(t.begin(), t.end(), T);
    std::copy(v.begin(), v.end(), V);
  });
}

int xc_eri_packed(int nshell, const int* shell_l, const int* shell_pure, const int* shell_nprim,
                  const double* shell_center, const double* alpha, const double* coef, double schwarz_threshold,
                  double* eri) {
  return guarded([&] {
    require(eri && schwarz_threshold >= 0.0, XC_ERR_ARG, "xc_eri_packed: bad arguments");
    auto sh = host_shells("xc_eri_packed", nshell, shell_l, shell_pure, shell_nprim, shell_center, alpha, coef, 4);
    const int64_t n = nao_of(sh), np = n * (n + 1) / 2;
    require(np * np <= (int64_t)1 << 31, XC_ERR_INPUT, "xc_eri_packed: more than 2^31 integrals; use density fitting");
    std::vector<double> out;
    eri_packed(sh, schwarz_threshold, out);
    std::copy(out.begin(), out.end(), eri);
  });
}

int xc_ri_j_integrals(int nshell, const int* shell_l, const int* shell_pure, const int* shell_nprim,
                      const double* shell_center, const double* alpha, const double* coef, int naux_shell,
                      const int* aux_l, const int* aux_pure, const int* aux_nprim, const double* aux_center,
                      const double* aux_alpha, const double* aux_coef, double schwarz_threshold, double* B3,
                      double* M) {
  return guarded([&] {
    require(B3 && M && schwarz_threshold >= 0.0, XC_ERR_ARG, "xc_ri_j_integrals: bad arguments");
    auto sh = host_shells("xc_ri_j_integrals", nshell, shell_l, shell_pure, shell_nprim, shell_center, alpha, coef, 4);
    auto ax = host_shells("xc_ri_j_integrals (auxiliary)", naux_shell, aux_l, aux_pure, aux_nprim, aux_center,
                          aux_alpha, aux_coef, 4);
    std::vector<double> b, m;
    ri_j_integrals(sh, ax, schwarz_threshold, b, m);
    std::copy(b.begin(), b.end(), B3);
    std::copy(m.begin(), m.end(), M);
  });
}

int xc_basis_create(xc_ctx* ctx, int nshell, const int* shell_l, const int* shell_pure, const int* shell_nprim,
                    const double* shell_center, const double* alpha, const double* coef, xc_basis** out) {
  return guarded([&] {
    require(ctx && out && nshell > 0 && shell_l && shell_pure && shell_nprim && shell_center && alpha && coef,
            XC_ERR_ARG, "xc_basis_create: bad arguments");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    auto* b = new xc_basis();
    b->ctx = ctx;
    b->nshell = nshell;
    int prim = 0, ao = 0;
    for (int s = 0; s < nshell; ++s) {
      const int l = shell_l[s];
      if (l < 0 || l > kMaxL) {
        delete b;
        throw XcError(XC_ERR_INPUT, "xc_basis_create: angular momentum above " + std::to_string(kMaxL));
      }
      DevShell d{};
      d.cx = shell_center[3 * s];
      d.cy = shell_center[3 * s + 1];
      d.cz = shell_center[3 * s + 2];
      d.l = l;
      d.pure = shell_pure[s] != 0;
      d.nprim = shell_nprim[s];
      d.prim_off = prim;
      d.ao_off = ao;
      d.ncart = (l + 1) * (l + 2) / 2;
      d.nfunc = d.pure ? 2 * l + 1 : d.ncart;
      d.ang_off = (int)b->ang.size();
      if (d.pure) {
        auto T = solid_harmonic_coefficients(l);
        b->ang.insert(b->ang.end(), T.begin(), T.end());
      } else {
        auto f = cartesian_norm_factors(l);
        for (int i = 0; i < d.ncart; ++i)
          for (int j = 0; j < d.ncart; ++j) b->ang.push_back(i == j ? f[i] : 0.0);
      }
      for (int q = 0; q < d.nprim; ++q) {
        b->alpha.push_back(alpha[prim + q]);
        b->coef.push_back(coef[prim + q]);
      }
      prim += d.nprim;
      ao += d.nfunc;
      b->maxl = std::max(b->maxl, l);
      b->shells.push_back(d);
    }
    b->nao = ao;
    b->d_shells.upload(ctx, b->shells.data(), b->shells.size());
    b->d_alpha.upload(ctx, b->alpha.data(), b->alpha.size());
    b->d_coef.upload(ctx, b->coef.data(), b->coef.size());
    b->d_ang.upload(ctx, b->ang.data(), b->ang.size());
    HIPX(hipStreamSynchronize(ctx->stream));
    ++ctx->live_handles;
    *out = b;
  });
}

int xc_basis_destroy(xc_basis* basis) {
  return guarded([&] {
    if (!basis) return;
    --basis->ctx->live_handles;
    delete basis;
  });
}

int xc_basis_nao(const xc_basis* basis, int* nao) {
  return guarded([&] {
    require(basis && nao, XC_ERR_ARG, "null argument");
    *nao = basis->nao;
  });
}

int xc_grid_create(xc_ctx* ctx, int64_t npoints, const double* points, const double* weights, xc_grid** out) {
  return guarded([&] {
    require(ctx && out && npoints > 0 && points && weights, XC_ERR_ARG, "xc_grid_create: bad arguments");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    auto* g = new xc_grid();
    g->ctx = ctx;
    g->npts = npoints;
    g->d_pts.upload(ctx, points, (size_t)(3 * npoints));
    g->d_w.upload(ctx, weights, (size_t)npoints);
    HIPX(hipStreamSynchronize(ctx->stream));
    ++ctx->live_handles;
    *out = g;
  });
}

int xc_grid_destroy(xc_grid* grid) {
  return guarded([&] {
    if (!grid) return;
    --grid->ctx->live_handles;
    delete grid;
  });
}

int xc_bfogc_create(xc_basis* basis, xc_grid* grid, int max_block_size, double radial_threshold,
                    int highest_derivative, int keep_fp32, xc_bfogc** out) {
  return guarded([&] {
    require(basis && grid && out, XC_ERR_ARG, "xc_bfogc_create: null argument");
    require(basis->ctx == grid->ctx, XC_ERR_ARG, "xc_bfogc_create: basis and grid live on different contexts");
    require(max_block_size >= 1 && max_block_size <= kTile, XC_ERR_ARG,
            "xc_bfogc_create: max block size must be in [1, 128]");
    require(highest_derivative >= 0 && highest_derivative <= 2, XC_ERR_ARG,
            "xc_bfogc_create: highest derivative must be 0, 1 or 2");
    require(radial_threshold >= 0.0, XC_ERR_ARG, "xc_bfogc_create: radial threshold must not be negative");
    require(keep_fp32 >= 0 && keep_fp32 <= 2, XC_ERR_ARG, "xc_bfogc_create: keep_fp32 must be 0, 1 or 2");
    xc_ctx* ctx = basis->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipSetDevice(ctx->device));
    auto* bf = new xc_bfogc();
    try {
      bf->ctx = ctx;
      bf->basis = basis;
      bf->grid = grid;
      bf->bs = max_block_size;
      bf->radial_thr = radial_threshold;
      bf->deriv = highest_derivative;
      bf->ncomp = highest_derivative >= 2 ? 10 : highest_derivative == 1 ? 4 : 1;
      const int64_t N = grid->npts;
      const int64_t nb64 = (N + max_block_size - 1) / max_block_size;
      require(nb64 < (1LL << 31), XC_ERR_ARG, "xc_bfogc_create: too many blocks");
      const int nb = (int)nb64;
      bf->nblocks = nb;
      const int ns = basis->nshell;
      // 1. shell screening per block on the device
      DBuf<int> d_pos, d_count;
      d_pos.alloc(ctx, (size_t)nb * ns);
      d_count.alloc(ctx, 2 * (size_t)nb);
      launch_screen(ctx->stream, grid->d_pts.p, N, max_block_size, nb, basis->d_shells.p, ns, basis->d_alpha.p,
                    basis->d_coef.p, radial_threshold, d_pos.p, d_count.p);
      HIPX(hipGetLastError());
      std::vector<int> count(2 * (size_t)nb);
      ctx->stage.down(ctx->stream, {{count.data(), d_count.p, sizeof(int) * count.size()}});
      // 2. the blocks' offsets and work items; their lists (compact AO indices padded to kAoPad,
      // significant shells, row entries) are filled on the device
      bf->blocks.resize(nb);
      bf->dens_item0.assign(nb, 0);
      int64_t tile_off = 0, idx_off = 0, shell_off = 0;
      for (int b = 0; b < nb; ++b) {
        DevBlock& bk = bf->blocks[b];
        bk.first = (int64_t)b * max_block_size;
        bk.npts = (int)std::min<int64_t>(max_block_size, N - bk.first);
        const int cnt = count[2 * b], nsh = count[2 * b + 1];
        bk.idx_off = (int)idx_off;
        bk.shell_off = (int)shell_off;
        bk.nb = cnt;
        bk.nshell = nsh;
        bk.npad = (cnt + kAoPad - 1) / kAoPad * kAoPad;
        idx_off += bk.npad;
        shell_off += nsh;
        bk.tile_off = tile_off;
        tile_off += (int64_t)bk.npad * kTile * bf->ncomp;
        bk.toff = bf->t_elems;
        bf->t_elems += fock_subtile_elems(bk.npad);
        bf->sum_nb += cnt;
        bf->sum_B_nb2 += (double)bk.npts * cnt * cnt;
        bk.npass = 0;
        if (cnt > 0) {
          // what is computed ends with the 16 columns of the last AO (the padding goes to 32)
          const int nc = (cnt + 15) / 16 * 16;
          // density: balanced passes of at most 16 kDensMaxS columns, 16-column granularity
          const int npass = (nc + 16 * kDensMaxS - 1) / (16 * kDensMaxS);
          const int width = ((nc + npass - 1) / npass + 15) / 16 * 16;
          int s = 0;
          bf->dens_item0[b] = (int)bf->dens_by_block.size();
          for (int c0 = 0; c0 < nc; c0 += width, ++s)
            bf->dens_by_block.push_back(WorkItem{b, c0, std::min(width, nc - c0), s});
          bk.npass = s;
          bf->npass_max = std::max(bf->npass_max, s);
          // Fock: the whole upper triangle of 16 x 16 sub-tiles as one item of the smallest workgroup
          // shape that holds it, else pairs of 128-row panels
          int shape = 0;
          while (shape < kFockShapes && nc > kFockShape[shape].npad) ++shape;
          auto add = [&](int k, int a0, int na, int b0, int nbr) {
            const int ta = na / 16, tb = nbr / 16;
            bf->fock_items[k].push_back(FockItem{b, a0, na, b0, nbr, nbr == 0 ? ta * (ta + 1) / 2 : ta * tb});
          };
          if (shape < kFockShapes) {
            add(shape, 0, nc, 0, 0);
          } else {
            const int np = (nc + kFockPanel - 1) / kFockPanel;
            for (int P = 0; P < np; ++P) {
              const int a0 = P * kFockPanel, na = std::min(kFockPanel, nc - a0);
              add(kFockPanelShape, a0, na, 0, 0);
              for (int Q = P + 1; Q < np; ++Q) {
                const int b0 = Q * kFockPanel;
                add(kFockPanelShape, a0, na, b0, std::min(kFockPanel, nc - b0));
              }
            }
          }
        }
      }
      bf->dens_work = bf->dens_by_block;
      xcd_order(bf->dens_work, [&](const WorkItem& w) { return (double)w.b * bf->blocks[w.block].npad; });
      for (auto& items : bf->fock_items) xcd_order(items, [](const FockItem& f) { return (double)f.nsub; });
      bf->tile_elems = tile_off;
      require(idx_off < (1LL << 31), XC_ERR_ARG, "xc_bfogc_create: too many AOs over the blocks");
      const int nao = basis->nao;
      // 3. admission by footprint (the context's cached blocks count as free; where it does not fit, so
      // do the spare scratches and the positions, given back before the tiles are allocated)
      size_t free_b = 0, total_b = 0;
      HIPX(hipMemGetInfo(&free_b, &total_b));
      free_b += ctx->cached;
      const double need =
          (double)tile_off * ((keep_fp32 != 2 ? sizeof(double) : 0) + (keep_fp32 ? sizeof(float) : 0)) +
          (double)bf->t_elems * (keep_fp32 != 2 ? sizeof(double) : sizeof(float));
      const bool tight = !(need < 0.9 * (double)free_b);
      if (tight) {
        ctx->reclaim();
        HIPX(hipMemGetInfo(&free_b, &total_b));
        free_b += ctx->cached + sizeof(int) * d_pos.n;
      }
      require(need < 0.9 * (double)free_b, XC_ERR_MEMORY,
              "xc_bfogc_create: AO tiles and Fock scratch need " + std::to_string(need / 1e9) + " GB, " +
                  std::to_string(free_b / 1e9) + " GB free");
      // 4. upload lists, evaluate AO tiles
      bf->d_blocks.upload(ctx, bf->blocks.data(), bf->blocks.size());
      bf->d_rowptr.alloc(ctx, (size_t)nao + 1);
      bf->d_rowent.alloc(ctx, (size_t)std::max<int64_t>(bf->sum_nb, 1));
      bf->d_ao_idx.alloc(ctx, (size_t)std::max<int64_t>(idx_off, 1));
      bf->d_sig_shell.alloc(ctx, (size_t)std::max<int64_t>(shell_off, 1));
      bf->d_sig_pos.alloc(ctx, (size_t)std::max<int64_t>(shell_off, 1));
      DBuf<int> d_rowcnt;
      d_rowcnt.alloc(ctx, (size_t)row_chunks(nb) * ns);
      launch_block_lists(ctx->stream, bf->d_blocks.p, nb, basis->d_shells.p, ns, nao, d_pos.p, bf->d_sig_shell.p,
                         bf->d_sig_pos.p, bf->d_ao_idx.p, d_rowcnt.p, bf->d_rowptr.p, bf->d_rowent.p);
      if (tight) {
        d_pos.free_();
        d_rowcnt.free_();
      }
      bf->d_dens_work.upload(ctx, bf->dens_work.data(), bf->dens_work.size());
      if (keep_fp32 == 1) {  // both tile sets: the mixed-precision build is available
        bf->d_dens_by_block.upload(ctx, bf->dens_by_block.data(), bf->dens_by_block.size());
        bf->d_dens_item0.upload(ctx, bf->dens_item0.data(), bf->dens_item0.size());
        bf->d_dense_list.alloc(ctx, std::max<size_t>(bf->dens_work.size(), 1));
        bf->d_carry_list.alloc(ctx, std::max<size_t>(bf->dens_work.size(), 1));
        bf->d_dense_cnt.alloc(ctx, 1);
        bf->d_carry_cnt.alloc(ctx, 1);
        bf->d_dense_mask.alloc(ctx, std::max(bf->nblocks, 1));
        HIPX(hipMemsetAsync(bf->d_dense_mask.p, 0, std::max(bf->nblocks, 1), ctx->stream));
      }
      for (int c = 0; c < kFockShapes; ++c)
        bf->d_fock_items[c].upload(ctx, bf->fock_items[c].data(), bf->fock_items[c].size());
      const size_t nt_el = (size_t)std::max<int64_t>(tile_off, 1);
      if (keep_fp32 != 2) bf->d_t64.alloc(ctx, nt_el);
      if (keep_fp32) bf->d_t32.alloc(ctx, nt_el);
      int max_nshell = 0;
      for (const DevBlock& bk : bf->blocks) max_nshell = std::max(max_nshell, bk.nshell);
      launch_ao_eval(ctx->stream, bf->d_blocks.p, nb, max_nshell, bf->d_sig_shell.p, bf->d_sig_pos.p, basis->d_shells.p,
                     basis->d_alpha.p, basis->d_coef.p, basis->d_ang.p, grid->d_pts.p, radial_threshold,
                     radial_threshold > 0.0 ? -std::log(radial_threshold) : HUGE_VAL, bf->ncomp, bf->d_t64.p,
                     keep_fp32 ? bf->d_t32.p : nullptr);
      HIPX(hipGetLastError());
      // 5. work buffers of a build
      const int n = basis->nao;
      const int nxc = (int)((N + kTile - 1) / kTile);
      bf->d_part.alloc(ctx, (size_t)std::max(bf->npass_max, 1) * 4 * N);
      bf->d_rho.alloc(ctx, N);
      bf->d_grad.alloc(ctx, 3 * N);
      bf->d_vs.alloc(ctx, N);
      bf->d_gw.alloc(ctx, 3 * N);
      bf->d_v.alloc(ctx, N);
      bf->d_g.alloc(ctx, 3 * N);
      bf->d_eblk.alloc(ctx, std::max(nxc, 1));
      bf->d_U.alloc(ctx, (size_t)n * n);
      // sub-tile scratch in the widest contraction precision the controller supports
      const int64_t t_doubles = keep_fp32 != 2 ? bf->t_elems : (bf->t_elems + 1) / 2;
      bf->d_T.alloc(ctx, (size_t)std::max<int64_t>(t_doubles, 1));
      bf->d_P.alloc(ctx, (size_t)n * n);
      bf->d_F.alloc(ctx, (size_t)n * n + 1);  // a server build's E_xc behind it
      if (keep_fp32) {
        bf->d_P32.alloc(ctx, (size_t)n * n);
        bf->d_round.alloc(ctx, 2 * (size_t)std::max(finalize_blocks(n), n));
      }
      if (keep_fp32 == 1) bf->d_P32d.alloc(ctx, (size_t)n * n);
      HIPX(hipStreamSynchronize(ctx->stream));
    } catch (...) {
      delete bf;
      throw;
    }
    ++ctx->live_handles;
    *out = bf;
  });
}

int xc_bfogc_destroy(xc_bfogc* bfogc) {
  return guarded([&] {
    if (!bfogc) return;
    std::lock_guard<std::recursive_mutex> lk(bfogc->ctx->mu);
    require(!bfogc->in_flight, XC_ERR_STATE, "xc_bfogc_destroy: a server build of this controller is in flight");
    (void)hipStreamSynchronize(bfogc->ctx->stream);
    forget_packs_of(bfogc->ctx, bfogc);
    --bfogc->ctx->live_handles;
    delete bfogc;
  });
}

int xc_bfogc_info(const xc_bfogc* bf, int* nblocks, int64_t* npoints, int* nao, int* max_block_size) {
  return guarded([&] {
    require(bf, XC_ERR_ARG, "null bfogc");
    if (nblocks) *nblocks = bf->nblocks;
    if (npoints) *npoints = bf->grid->npts;
    if (nao) *nao = bf->basis->nao;
    if (max_block_size) *max_block_size = bf->bs;
  });
}

int xc_bfogc_stats(const xc_bfogc* bf, int64_t* sum_nb, double* sum_B_nb2, int64_t* tile_bytes) {
  return guarded([&] {
    require(bf, XC_ERR_ARG, "null bfogc");
    if (sum_nb) *sum_nb = bf->sum_nb;
    if (sum_B_nb2) *sum_B_nb2 = bf->sum_B_nb2;
    if (tile_bytes)
      *tile_bytes = bf->tile_elems * (int64_t)((bf->d_t64.p ? sizeof(double) : 0) + (bf->d_t32.p ? sizeof(float) : 0));
  });
}

int xc_bfogc_block_data(const xc_bfogc* bf, int block, double* values, double* gx, double* gy, double* gz,
                        int* negligible, int* block_size) {
  return guarded([&] {
    require(bf, XC_ERR_ARG, "null bfogc");
    require(block >= 0 && block < bf->nblocks, XC_ERR_ARG, "block index out of range");
    require(!(gx || gy || gz) || bf->deriv >= 1, XC_ERR_STATE, "gradients were not evaluated (highest derivative 0)");
    require(bf->d_t64.p, XC_ERR_STATE, "xc_bfogc_block_data: the controller keeps FP32 tiles only");
    std::lock_guard<std::recursive_mutex> lk(bf->ctx->mu);
    const DevBlock& bk = bf->blocks[block];
    const int n = bf->basis->nao;
    const int64_t cnt = (int64_t)bk.npad * kTile * bf->ncomp;
    std::vector<double> t((size_t)std::max<int64_t>(cnt, 1));
    std::vector<int> idx((size_t)bk.npad);
    if (cnt) {
      HIPX(hipMemcpyAsync(idx.data(), bf->d_ao_idx.p + bk.idx_off, sizeof(int) * idx.size(), hipMemcpyDeviceToHost,
                          bf->ctx->stream));
      HIPX(hipMemcpyAsync(t.data(), bf->d_t64.p + bk.tile_off, sizeof(double) * cnt, hipMemcpyDeviceToHost,
                          bf->ctx->stream));
      HIPX(hipStreamSynchronize(bf->ctx->stream));
    }
    const int B = bk.npts;
    if (block_size) *block_size = B;
    double* outs[4] = {values, gx, gy, gz};
    for (int c = 0; c < 4; ++c)
      if (outs[c]) std::fill(outs[c], outs[c] + (size_t)B * n, 0.0);
    if (negligible) std::fill(negligible, negligible + n, 1);
    for (int i = 0; i < bk.nb; ++i) {
      const int mu = idx[i];
      if (negligible) negligible[mu] = 0;
      for (int c = 0; c < std::min(bf->ncomp, 4); ++c) {
        if (!outs[c]) continue;
        for (int p = 0; p < B; ++p)
          outs[c][(size_t)mu * B + p] = t[((size_t)c * bk.npad + i) * kTile + p];
      }
    }
  });
}

int xc_bfogc_block_hessian(const xc_bfogc* bf, int block, double* hess) {
  return guarded([&] {
    require(bf && hess, XC_ERR_ARG, "xc_bfogc_block_hessian: null argument");
    require(block >= 0 && block < bf->nblocks, XC_ERR_ARG, "block index out of range");
    require(bf->deriv >= 2, XC_ERR_STATE, "second derivatives were not evaluated (highest derivative < 2)");
    require(bf->d_t64.p, XC_ERR_STATE, "xc_bfogc_block_hessian: the controller keeps FP32 tiles only");
    std::lock_guard<std::recursive_mutex> lk(bf->ctx->mu);
    const DevBlock& bk = bf->blocks[block];
    const int n = bf->basis->nao;
    const int B = bk.npts;
    const int64_t cnt = (int64_t)bk.npad * kTile * 6;
    std::vector<double> t((size_t)std::max<int64_t>(cnt, 1));
    std::vector<int> idx((size_t)bk.npad);
    if (cnt) {
      HIPX(hipMemcpyAsync(idx.data(), bf->d_ao_idx.p + bk.idx_off, sizeof(int) * idx.size(), hipMemcpyDeviceToHost,
                          bf->ctx->stream));
      HIPX(hipMemcpyAsync(t.data(), bf->d_t64.p + bk.tile_off + (int64_t)4 * bk.npad * kTile, sizeof(double) * cnt,
                          hipMemcpyDeviceToHost, bf->ctx->stream));
      HIPX(hipStreamSynchronize(bf->ctx->stream));
    }
    std::fill(hess, hess + (size_t)6 * B * n, 0.0);
    for (int i = 0; i < bk.nb; ++i) {
      const int mu = idx[i];
      for (int c = 0; c < 6; ++c)
        for (int p = 0; p < B; ++p)
          hess[((size_t)c * n + mu) * B + p] = t[((size_t)c * bk.npad + i) * kTile + p];
    }
  });
}

int xc_density(xc_bfogc* bf, const double* P, double* rho, double* grad, int* nonneg) {
  return guarded([&] {
    require(bf && P && rho, XC_ERR_ARG, "xc_density: null argument");
    require(!bf->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
    require(!grad || bf->deriv >= 1, XC_ERR_STATE, "xc_density: gradient requested but AO gradients not evaluated");
    require(bf->d_t64.p, XC_ERR_STATE, "xc_density: the controller keeps FP32 tiles only");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    const int n = bf->basis->nao;
    const int64_t N = bf->grid->npts;
    ctx->stage.up(ctx->stream, bf->d_P.p, P, sizeof(double) * n * n);
    run_density<double>(bf, bf->d_t64.p, bf->d_P.p, grad ? 1 : 0, ctx->lanes);
    launch_reduce_partials(ctx->stream, bf->d_blocks.p, bf->bs, N, bf->d_part.p, grad ? 1 : 0, bf->d_rho.p,
                           bf->d_grad.p);
    HIPX(hipGetLastError());
    ctx->stage.down(ctx->stream, {{rho, bf->d_rho.p, sizeof(double) * N}, {grad, bf->d_grad.p, sizeof(double) * 3 * N}});
    if (nonneg)
      for (int b = 0; b < bf->nblocks; ++b) nonneg[b] = bf->blocks[b].nb > 0 ? 1 : 0;
  });
}

int xc_functional(xc_ctx* ctx, int functional, int64_t npts, int block_size, const double* rho, const double* grad,
                  const double* weights, double* eps, double* v, double* g, double* energy) {
  return guarded([&] {
    require(ctx && rho && weights && npts > 0, XC_ERR_ARG, "xc_functional: bad arguments");
    require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "xc_functional: unknown functional");
    require(block_size >= 1 && block_size <= kTile, XC_ERR_ARG, "xc_functional: block size must be in [1,128]");
    const bool gga = functional_is_gga(functional);
    require(!gga || grad, XC_ERR_ARG, "xc_functional: GGA functional needs the density gradient");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    DBuf<double> d_rho, d_grad, d_w, d_eps, d_v, d_g, d_eblk, d_E;
    const int nxc = (int)((npts + block_size - 1) / block_size);
    d_rho.upload(ctx, rho, npts);
    if (gga) d_grad.upload(ctx, grad, 3 * npts);
    d_w.upload(ctx, weights, npts);
    d_eps.alloc(ctx, npts);
    d_v.alloc(ctx, npts);
    if (gga) d_g.alloc(ctx, 3 * npts);
    d_eblk.alloc(ctx, nxc);
    d_E.alloc(ctx, 1);
    launch_functional(ctx->stream, functional, npts, block_size, d_rho.p, d_grad.p, nullptr, nullptr, d_w.p,
                      d_eps.p, d_v.p, d_g.p, nullptr, nullptr, d_eblk.p);
    launch_sum(ctx->stream, d_eblk.p, nxc, d_E.p);
    HIPX(hipGetLastError());
    if (g && !gga) std::fill(g, g + 3 * npts, 0.0);
    double E = 0.0;
    ctx->stage.down(ctx->stream, {{eps, d_eps.p, sizeof(double) * npts},
                                  {v, d_v.p, sizeof(double) * npts},
                                  {gga ? g : nullptr, d_g.p, sizeof(double) * 3 * npts},
                                  {&E, d_E.p, sizeof(double)}});
    if (energy) *energy = E;
  });
}

int xc_functional_device_noalloc(xc_ctx* ctx, int functional, int64_t npts, int block_size, const double* d_rho,
                                 const double* d_grad, const double* d_weights, double* d_eps, double* d_v,
                                 double* d_g, double* energy) {
  return guarded([&] {
    require(ctx && d_rho && d_weights && npts > 0, XC_ERR_ARG, "xc_functional_device_noalloc: bad arguments");
    require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG,
            "xc_functional_device_noalloc: unknown functional");
    require(block_size >= 1 && block_size <= kTile, XC_ERR_ARG,
            "xc_functional_device_noalloc: block size must be in [1,128]");
    const bool gga = functional_is_gga(functional);
    require(!gga || d_grad, XC_ERR_ARG, "xc_functional_device_noalloc: GGA functional needs the density gradient");
    const int64_t nxc = (npts + block_size - 1) / block_size;
    require(nxc <= kNoallocBlocks, XC_ERR_ARG,
            "xc_functional_device_noalloc: " + std::to_string(nxc) + " blocks of " + std::to_string(block_size) +
                " points exceed the workspace of at most " + std::to_string(kNoallocBlocks) + " blocks");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipSetDevice(ctx->device));
    double* scr = noalloc_scratch(ctx->device);
    // every per-block slot [0, nxc) is written by the functional kernel and the sum slot by the
    // sum kernel, so nothing left from an earlier call is read
    launch_functional(ctx->stream, functional, npts, block_size, d_rho, gga ? d_grad : nullptr, nullptr,
                      nullptr, d_weights, d_eps, d_v, gga ? d_g : nullptr, nullptr, nullptr, scr);
    if (!gga && d_g) launch_fill(ctx->stream, d_g, 3 * npts, 0.0);
    launch_sum(ctx->stream, scr, nxc, scr + kNoallocBlocks);
    HIPX(hipGetLastError());
    if (energy) {
      ctx->stage.down(ctx->stream, {{energy, scr + kNoallocBlocks, sizeof(double)}});
    }
  });
}

int xc_fock_add(xc_bfogc* bf, double thr, const double* v, const double* g, double* F) {
  return guarded([&] {
    require(bf && v && F, XC_ERR_ARG, "xc_fock_add: null argument");
    require(!bf->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
    require(!g || bf->deriv >= 1, XC_ERR_STATE, "xc_fock_add: gradient potential needs AO gradients");
    require(bf->d_t64.p, XC_ERR_STATE, "xc_fock_add: the controller keeps FP32 tiles only");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    const int n = bf->basis->nao;
    const int64_t N = bf->grid->npts;
    ctx->stage.up(ctx->stream, bf->d_v.p, v, sizeof(double) * N);
    if (g) ctx->stage.up(ctx->stream, bf->d_g.p, g, sizeof(double) * 3 * N);
    launch_weight_potential(ctx->stream, N, bf->grid->d_w.p, bf->d_v.p, g ? bf->d_g.p : nullptr, bf->d_vs.p,
                            bf->d_gw.p);
    run_fock<double>(bf, bf->d_t64.p, g ? 1 : 0, thr, ctx->lanes);
    ctx->stage.up(ctx->stream, bf->d_F.p, F, sizeof(double) * n * n);
    launch_finalize(ctx->stream, bf->d_U.p, bf->d_F.p, n, 1);
    HIPX(hipGetLastError());
    ctx->stage.down(ctx->stream, {{F, bf->d_F.p, sizeof(double) * n * n}});
  });
}

// One build enqueued on stream s, E_xc left in d_energy (device).  Stage
// events are recorded only on the context stream.
static void enqueue_build(xc_bfogc* bf, int functional, int precision, double thr, const double* dP, double* dF,
                          const Lanes& L, double* d_energy) {
  xc_ctx* ctx = bf->ctx;
  hipStream_t s = L.main;
  require(!bf->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
  require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32 || precision == XC_PREC_MIXED, XC_ERR_ARG,
          "unknown precision");
  const bool gga = functional_is_gga(functional);
  const bool mixed = precision == XC_PREC_MIXED;
  const bool lowp = precision != XC_PREC_FP64;  // FP32 contractions (mixed: plus the FP64 refinement)
  require(!gga || bf->deriv >= 1, XC_ERR_STATE, "GGA functional needs AO gradients (highest derivative 1)");
  require(!lowp || bf->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
  require(lowp || bf->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
  require(!mixed || (bf->d_t64.p && bf->d_P32d.p), XC_ERR_STATE,
          "mixed precision needs both tile sets (keep_fp32 = 1)");
  const int n = bf->basis->nao;
  const int64_t N = bf->grid->npts;
  if (s == ctx->stream) ctx->mark();
  if (lowp) launch_to_float(s, dP, bf->d_P32.p, (int64_t)n * n);
  if (mixed) launch_to_double(s, bf->d_P32.p, bf->d_P32d.p, (int64_t)n * n);
  if (s == ctx->stream) ctx->mark();
  if (!lowp) {
    const bool form = use_form(gga, n);  // U is free until the reduce
    if (form) launch_fold(s, dP, bf->d_U.p, n);
    run_density<double>(bf, bf->d_t64.p, form ? bf->d_U.p : dP, gga ? 1 : 0, L, form);
  } else {
    if (mixed)
      run_density_mixed(bf, gga ? 1 : 0, L);
    else
      run_density<float>(bf, bf->d_t32.p, bf->d_P32.p, gga ? 1 : 0, L);
  }
  if (s == ctx->stream) ctx->mark();
  if (bf->bs == kTile) {
    launch_functional(s, functional, N, kTile, nullptr, nullptr, bf->d_blocks.p, bf->d_part.p,
                      bf->grid->d_w.p, nullptr, nullptr, nullptr, bf->d_vs.p, bf->d_gw.p, bf->d_eblk.p);
  } else {
    launch_reduce_partials(s, bf->d_blocks.p, bf->bs, N, bf->d_part.p, gga ? 1 : 0, bf->d_rho.p, bf->d_grad.p);
    launch_functional(s, functional, N, kTile, bf->d_rho.p, gga ? bf->d_grad.p : nullptr, nullptr,
                      nullptr, bf->grid->d_w.p, nullptr, nullptr, nullptr, bf->d_vs.p, bf->d_gw.p, bf->d_eblk.p);
  }
  if (s == ctx->stream) ctx->mark();
  if (!lowp)
    run_fock_tiles<double>(bf, bf->d_t64.p, gga ? 1 : 0, thr, L);
  else
    run_fock_tiles<float>(bf, bf->d_t32.p, gga ? 1 : 0, thr, L);
  if (s == ctx->stream) ctx->mark();
  // FP32 contractions see fl32(P): E_xc[P] = E_xc[fl32(P)] + tr(F (P - fl32(P))) to first order,
  // the trace formed with F and added with the energy sum (the mixed form's FP64
  // refinement also contracts fl32(P), so the same term applies to every block)
  if (!lowp)
    run_fock_finish<double>(bf, L, dF, nullptr, nullptr, 0, 1, d_energy);
  else
    run_fock_finish<float>(bf, L, dF, dP, bf->d_P32.p, 0, 1, d_energy);
  if (s == ctx->stream) ctx->mark();
  HIPX(hipGetLastError());
}

/* Buffers of unrestricted builds, each allocated once (never reallocated: pointers to
 * them may already be in enqueued work). */
static void ensure_pol_buffers(xc_bfogc* bf, bool fp32) {
  xc_ctx* ctx = bf->ctx;
  const int n = bf->basis->nao;
  const int64_t N = bf->grid->npts;
  if (!bf->d_rho_b.p) bf->d_rho_b.alloc(ctx, N);
  if (!bf->d_grad_b.p) bf->d_grad_b.alloc(ctx, 3 * N);
  if (!bf->d_vs_b.p) bf->d_vs_b.alloc(ctx, N);
  if (!bf->d_gw_b.p) bf->d_gw_b.alloc(ctx, 3 * N);
  if (!bf->d_Pb.p) bf->d_Pb.alloc(ctx, (size_t)n * n);
  if (!bf->d_Fb.p) bf->d_Fb.alloc(ctx, (size_t)n * n);
  if (fp32 && !bf->d_P32b.p) bf->d_P32b.alloc(ctx, (size_t)n * n);
}

/* Unrestricted build (FuncPotential<UNRESTRICTED>): spin densities from P_a and P_b,
 * the spin-polarised functional, and F_a, F_b from w v_s, w g_s (one Fock pass per
 * spin, each with its own block skip); E_xc left in d_energy. */
static void enqueue_build_pol(xc_bfogc* bf, int functional, int precision, double thr, const double* dPa,
                              const double* dPb, double* dFa, double* dFb, const Lanes& L, double* d_energy) {
  hipStream_t s = L.main;
  require(!bf->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
  require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
  require(precision != XC_PREC_MIXED, XC_ERR_ARG,
          "mixed precision is available for restricted single-system builds only");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32, XC_ERR_ARG, "unknown precision");
  const bool gga = functional_is_gga(functional);
  require(!gga || bf->deriv >= 1, XC_ERR_STATE, "GGA functional needs AO gradients (highest derivative 1)");
  require(precision == XC_PREC_FP64 || bf->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
  require(precision == XC_PREC_FP32 || bf->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
  const int n = bf->basis->nao;
  const int64_t N = bf->grid->npts;
  ensure_pol_buffers(bf, precision == XC_PREC_FP32);
  const double* Ps[2] = {dPa, dPb};
  double* Fs[2] = {dFa, dFb};
  if (pair_buffers(bf)) {
    if (precision == XC_PREC_FP64)
      enqueue_build_pair<double>(bf, functional, thr, Ps, Fs, L, d_energy);
    else
      enqueue_build_pair<float>(bf, functional, thr, Ps, Fs, L, d_energy);
    return;
  }
  // spin densities: one density pass per spin through the shared partial buffer
  double* rho[2] = {bf->d_rho.p, bf->d_rho_b.p};
  double* grad[2] = {bf->d_grad.p, bf->d_grad_b.p};
  float* P32[2] = {bf->d_P32.p, bf->d_P32b.p};
  for (int sp = 0; sp < 2; ++sp) {
    if (precision == XC_PREC_FP64) {
      const bool form = use_form(gga, n);
      if (form) launch_fold(s, Ps[sp], bf->d_U.p, n);
      run_density<double>(bf, bf->d_t64.p, form ? bf->d_U.p : Ps[sp], gga ? 1 : 0, L, form);
    } else {
      launch_to_float(s, Ps[sp], P32[sp], (int64_t)n * n);
      run_density<float>(bf, bf->d_t32.p, P32[sp], gga ? 1 : 0, L);
    }
    launch_reduce_partials(s, bf->d_blocks.p, bf->bs, N, bf->d_part.p, gga ? 1 : 0, rho[sp], grad[sp]);
  }
  launch_functional_pol(s, functional, N, kTile, bf->d_rho.p, bf->d_grad.p, bf->d_rho_b.p,
                        bf->d_grad_b.p, bf->grid->d_w.p, bf->d_vs.p, bf->d_gw.p, bf->d_vs_b.p, bf->d_gw_b.p,
                        bf->d_eblk.p);
  const double* vs[2] = {bf->d_vs.p, bf->d_vs_b.p};
  const double* gw[2] = {bf->d_gw.p, bf->d_gw_b.p};
  for (int sp = 0; sp < 2; ++sp) {
    // with the first-order FP32 rounding term of each spin density matrix (dE_xc/dP_s = F_s)
    double* E = sp == 1 ? d_energy : nullptr;
    if (precision == XC_PREC_FP64) {
      run_fock_tiles<double>(bf, bf->d_t64.p, gga ? 1 : 0, thr, L, vs[sp], gw[sp]);
      run_fock_finish<double>(bf, L, Fs[sp], nullptr, nullptr, sp, 2, E);
    } else {
      run_fock_tiles<float>(bf, bf->d_t32.p, gga ? 1 : 0, thr, L, vs[sp], gw[sp]);
      run_fock_finish<float>(bf, L, Fs[sp], Ps[sp], P32[sp], sp, 2, E);
    }
  }
  HIPX(hipGetLastError());
}

/* Non-additive build: rho_sup = rho_act + sum_env rho_env on the shared grid,
 * v = v[rho_sup] - v[rho_act] integrated with the active basis,
 * E = E[rho_sup] - E[rho_act] - sum_env E[rho_env] (left in ctx->energy). */
// The functional stage of a non-additive build of sub[0] among sub[1..]: w v and w g of v[rho_sup] -
// v[rho_act] into sub[0].  E[rho_sup] - E[rho_act] - E[rho_env] ... goes into the context's energy, here or
// (small matrices) with the returned list in run_nadd_fock.  cached: on the cached densities, keeping
// each E[rho_env] until its density changes.
static EnvEnergies run_nadd_functional(const std::vector<xc_bfogc*>& sub, int functional, bool cached) {
  xc_bfogc* act = sub[0];
  xc_ctx* ctx = act->ctx;
  hipStream_t s = ctx->stream;
  const bool gga = functional_is_gga(functional);
  const int64_t N = act->grid->npts;
  const int nxc = (int)((N + kTile - 1) / kTile);
  const double* w = act->grid->d_w.p;
  // rho_sup = rho_act + rho_env[0] + ... in list order, inside the functional's launch (what exceeds
  // its list is summed before it)
  DensityList sup{};
  const auto append = [](DensityList& L, const DBuf<double>& rho, const DBuf<double>& grad) {
    L.rho[L.n] = rho.p;
    L.grad[L.n++] = grad.p;
  };
  if (sub.size() > (size_t)kListMax && !act->d_rho_sup.p) {
    act->d_rho_sup.alloc(ctx, N);
    act->d_grad_sup.alloc(ctx, 3 * N);
  }
  for (xc_bfogc* b : sub) {
    if (sup.n == kListMax) {
      launch_sum_densities(s, sup, N, gga ? 1 : 0, act->d_rho_sup.p, act->d_grad_sup.p);
      sup.n = 0;
      append(sup, act->d_rho_sup, act->d_grad_sup);
    }
    append(sup, cached ? b->d_rho_c : b->d_rho, cached ? b->d_grad_c : b->d_grad);
  }
  // the environment's energies that are missing, beside the functional (kListMax of them per launch)
  std::vector<xc_bfogc*> missing;
  for (size_t i = 1; i < sub.size(); ++i)
    if (!cached || !sub[i]->ecache_valid[functional]) missing.push_back(sub[i]);
  for (size_t i0 = 0; i0 == 0 || i0 < missing.size(); i0 += kListMax) {
    DensityList pending{};
    double* eblk[kListMax] = {};
    for (size_t i = i0; i < std::min(missing.size(), i0 + kListMax); ++i) {
      eblk[pending.n] = missing[i]->d_eblk.p;
      append(pending, cached ? missing[i]->d_rho_c : missing[i]->d_rho,
             cached ? missing[i]->d_grad_c : missing[i]->d_grad);
    }
    launch_nadd_functional(s, functional, N, i0 == 0, sup, cached ? act->d_rho_c.p : act->d_rho.p,
                           cached ? act->d_grad_c.p : act->d_grad.p, pending, eblk, w, act->d_vs.p, act->d_gw.p,
                           act->d_eblk.p);
  }
  EnvEnergies env_e{};
  for (size_t i0 = 1; i0 == 1 || i0 < sub.size(); i0 += kListMax) {
    env_e.n = 0;
    for (size_t i = i0; i < std::min(sub.size(), i0 + kListMax); ++i) {
      xc_bfogc* b = sub[i];
      const bool valid = cached && b->ecache_valid[functional];
      env_e.e[env_e.n] = cached ? b->d_ecache.p + functional : nullptr;
      env_e.eblk[env_e.n++] = valid ? nullptr : b->d_eblk.p;
    }
    // one list of a small matrix goes with its row reduce, in the workgroup that sums the energy
    if (sub.size() > (size_t)kListMax + 1 || act->basis->nao > kDirectRows)
      launch_nadd_energy(s, i0 == 1 ? act->d_eblk.p : nullptr, nxc, env_e, ctx->energy);
  }
  return env_e;
}

// The Fock stage of a non-additive build, with the energy where the functional stage left its sum.
static void run_nadd_fock(const std::vector<xc_bfogc*>& sub, int functional, int precision, double thr,
                          const EnvEnergies& env, bool cached, double* dF) {
  xc_bfogc* act = sub[0];
  xc_ctx* ctx = act->ctx;
  const int g = functional_is_gga(functional) ? 1 : 0;
  const bool with_energy = act->basis->nao <= kDirectRows && sub.size() <= (size_t)kListMax + 1;
  double* E = with_energy ? ctx->energy : nullptr;
  if (precision == XC_PREC_FP32)
    run_fock_tiles<float>(act, act->d_t32.p, g, thr, ctx->lanes);
  else
    run_fock_tiles<double>(act, act->d_t64.p, g, thr, ctx->lanes);
  ctx->mark();
  if (precision == XC_PREC_FP32)
    run_fock_finish<float>(act, ctx->lanes, dF, nullptr, nullptr, 0, 1, E, env);
  else
    run_fock_finish<double>(act, ctx->lanes, dF, nullptr, nullptr, 0, 1, E, env);
  if (cached)
    for (size_t i = 1; i < sub.size(); ++i) sub[i]->ecache_valid[functional] = true;
}

static void enqueue_nadd(xc_bfogc* act, int nenv, xc_bfogc* const* env, int functional, int precision, double thr,
                         const double* dP_act, const double* const* dP_env, double* dF) {
  xc_ctx* ctx = act->ctx;
  require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
  require(precision != XC_PREC_MIXED, XC_ERR_ARG,
          "mixed precision is available for restricted single-system builds only");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32, XC_ERR_ARG, "unknown precision");
  require(nenv >= 0 && (nenv == 0 || (env && dP_env)), XC_ERR_ARG, "non-additive build: null environment list");
  const bool gga = functional_is_gga(functional);
  const bool fp32 = precision == XC_PREC_FP32;
  std::vector<xc_bfogc*> sub(1, act);
  std::vector<const double*> Ps(1, dP_act);
  for (int i = 0; i < nenv; ++i) {
    require(env[i] && dP_env[i], XC_ERR_ARG, "non-additive build: null environment controller or density");
    require(env[i] != act, XC_ERR_ARG, "non-additive build: the active controller is also listed as environment");
    for (int j = 0; j < i; ++j)
      require(env[j] != env[i], XC_ERR_ARG, "non-additive build: an environment controller is listed twice");
    sub.push_back(env[i]);
    Ps.push_back(dP_env[i]);
  }
  for (xc_bfogc* b : sub) {
    require(b->ctx == ctx, XC_ERR_ARG, "non-additive build: controllers live on different contexts");
    require(b->grid == act->grid, XC_ERR_ARG,
            "non-additive build: all subsystem controllers must be defined on the same (supersystem) grid");
    require(b->bs == act->bs, XC_ERR_ARG, "non-additive build: controllers differ in block size");
    require_idle(b, "non-additive build");
    require(!gga || b->deriv >= 1, XC_ERR_STATE, "GGA functional needs AO gradients (highest derivative 1)");
    require(!fp32 || b->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
    require(fp32 || b->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
  }
  const int64_t N = act->grid->npts;
  hipStream_t s = ctx->stream;
  ctx->mark();
  if (fp32)
    for (size_t i = 0; i < sub.size(); ++i)
      launch_to_float(s, Ps[i], sub[i]->d_P32.p, (int64_t)sub[i]->basis->nao * sub[i]->basis->nao);
  ctx->mark();
  for (size_t i = 0; i < sub.size(); ++i) {
    xc_bfogc* b = sub[i];
    if (fp32)
      run_density<float>(b, b->d_t32.p, b->d_P32.p, gga ? 1 : 0, ctx->lanes);
    else
      run_density<double>(b, b->d_t64.p, Ps[i], gga ? 1 : 0, ctx->lanes);
    launch_reduce_partials(s, b->d_blocks.p, b->bs, N, b->d_part.p, gga ? 1 : 0, b->d_rho.p, b->d_grad.p, 0);
  }
  ctx->mark();
  const EnvEnergies env_e = run_nadd_functional(sub, functional, false);
  ctx->mark();
  run_nadd_fock(sub, functional, precision, thr, env_e, false, dF);
  ctx->mark();
  HIPX(hipGetLastError());
}

/* Unrestricted non-additive build (NAddFuncPotential<UNRESTRICTED>::getMatrix): spin
 * densities of every subsystem on the shared grid, rho_sup^s = sum of them,
 * v^s = v^s[rho_sup] - v^s[rho_act] integrated with the active basis per spin,
 * E = E[sup] - E[act] - sum_env E[env] (left in ctx->energy). */
static void enqueue_nadd_pol(xc_bfogc* act, int nenv, xc_bfogc* const* env, int functional, int precision,
                             double thr, const double* dPa_act, const double* dPb_act, const double* const* dPa_env,
                             const double* const* dPb_env, double* dFa, double* dFb) {
  xc_ctx* ctx = act->ctx;
  require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
  require(precision != XC_PREC_MIXED, XC_ERR_ARG,
          "mixed precision is available for restricted single-system builds only");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32, XC_ERR_ARG, "unknown precision");
  require(nenv >= 0 && (nenv == 0 || (env && dPa_env && dPb_env)), XC_ERR_ARG,
          "non-additive build: null environment list");
  const bool gga = functional_is_gga(functional);
  const bool fp32 = precision == XC_PREC_FP32;
  std::vector<xc_bfogc*> sub(1, act);
  std::vector<const double*> Pa(1, dPa_act), Pb(1, dPb_act);
  for (int i = 0; i < nenv; ++i) {
    require(env[i] && dPa_env[i] && dPb_env[i], XC_ERR_ARG,
            "non-additive build: null environment controller or density");
    require(env[i] != act, XC_ERR_ARG, "non-additive build: the active controller is also listed as environment");
    for (int j = 0; j < i; ++j)
      require(env[j] != env[i], XC_ERR_ARG, "non-additive build: an environment controller is listed twice");
    sub.push_back(env[i]);
    Pa.push_back(dPa_env[i]);
    Pb.push_back(dPb_env[i]);
  }
  for (xc_bfogc* b : sub) {
    require(b->ctx == ctx, XC_ERR_ARG, "non-additive build: controllers live on different contexts");
    require(b->grid == act->grid, XC_ERR_ARG,
            "non-additive build: all subsystem controllers must be defined on the same (supersystem) grid");
    require(b->bs == act->bs, XC_ERR_ARG, "non-additive build: controllers differ in block size");
    require(!b->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
    require(!gga || b->deriv >= 1, XC_ERR_STATE, "GGA functional needs AO gradients (highest derivative 1)");
    require(!fp32 || b->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
    require(fp32 || b->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
    ensure_pol_buffers(b, fp32);
  }
  const int64_t N = act->grid->npts;
  const int nxc = (int)((N + kTile - 1) / kTile);
  if (!act->d_rho_sup.p) {
    act->d_rho_sup.alloc(ctx, N);
    act->d_grad_sup.alloc(ctx, 3 * N);
  }
  if (!act->d_rho_sup_b.p) {
    act->d_rho_sup_b.alloc(ctx, N);
    act->d_grad_sup_b.alloc(ctx, 3 * N);
  }
  hipStream_t s = ctx->stream;
  const double* w = act->grid->d_w.p;
  const int g = gga ? 1 : 0;
  double* sup_r[2] = {act->d_rho_sup.p, act->d_rho_sup_b.p};
  double* sup_g[2] = {act->d_grad_sup.p, act->d_grad_sup_b.p};
  for (size_t i = 0; i < sub.size(); ++i) {
    xc_bfogc* b = sub[i];
    const double* P[2] = {Pa[i], Pb[i]};
    float* P32[2] = {b->d_P32.p, b->d_P32b.p};
    double* rho[2] = {b->d_rho.p, b->d_rho_b.p};
    double* grd[2] = {b->d_grad.p, b->d_grad_b.p};
    for (int sp = 0; sp < 2; ++sp) {
      if (fp32) {
        launch_to_float(s, P[sp], P32[sp], (int64_t)b->basis->nao * b->basis->nao);
        run_density<float>(b, b->d_t32.p, P32[sp], g, ctx->lanes);
      } else {
        run_density<double>(b, b->d_t64.p, P[sp], g, ctx->lanes);
      }
      launch_reduce_partials(s, b->d_blocks.p, b->bs, N, b->d_part.p, g, rho[sp], grd[sp], 0);
      launch_reduce_partials(s, b->d_blocks.p, b->bs, N, b->d_part.p, g, sup_r[sp], sup_g[sp], i == 0 ? 0 : 1);
    }
  }
  // v^s[sup] - v^s[act] and E[sup] - E[act]
  launch_functional_pol(s, functional, N, kTile, sup_r[0], sup_g[0], sup_r[1], sup_g[1], w, act->d_vs.p,
                        act->d_gw.p, act->d_vs_b.p, act->d_gw_b.p, act->d_eblk.p, act->d_rho.p, act->d_grad.p,
                        act->d_rho_b.p, act->d_grad_b.p);
  launch_sum(s, act->d_eblk.p, nxc, ctx->energy, 0);
  for (size_t i = 1; i < sub.size(); ++i) {
    xc_bfogc* b = sub[i];
    launch_functional_pol(s, functional, N, kTile, b->d_rho.p, b->d_grad.p, b->d_rho_b.p, b->d_grad_b.p, w,
                          nullptr, nullptr, nullptr, nullptr, b->d_eblk.p);
    launch_sum(s, b->d_eblk.p, nxc, ctx->energy, 1);
  }
  const double* vs[2] = {act->d_vs.p, act->d_vs_b.p};
  const double* gw[2] = {act->d_gw.p, act->d_gw_b.p};
  double* Fs[2] = {dFa, dFb};
  for (int sp = 0; sp < 2; ++sp) {
    if (fp32) {
      run_fock_tiles<float>(act, act->d_t32.p, g, thr, ctx->lanes, vs[sp], gw[sp]);
      run_fock_finish<float>(act, ctx->lanes, Fs[sp], nullptr, nullptr, sp, 2, nullptr);
    } else {
      run_fock_tiles<double>(act, act->d_t64.p, g, thr, ctx->lanes, vs[sp], gw[sp]);
      run_fock_finish<double>(act, ctx->lanes, Fs[sp], nullptr, nullptr, sp, 2, nullptr);
    }
  }
  HIPX(hipGetLastError());
}

int xc_nadd_fock_build_unrestricted(xc_bfogc* active, int nenv, xc_bfogc* const* env, int functional, int precision,
                                    double thr, const double* Pa_active, const double* Pb_active,
                                    const double* const* Pa_env, const double* const* Pb_env, double* Fa, double* Fb,
                                    double* energy) {
  return guarded([&] {
    require(active && Pa_active && Pb_active && Fa && Fb, XC_ERR_ARG, "xc_nadd_fock_build_unrestricted: null argument");
    require(nenv >= 0 && (nenv == 0 || (env && Pa_env && Pb_env)), XC_ERR_ARG,
            "xc_nadd_fock_build_unrestricted: null environment list");
    xc_ctx* ctx = active->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require_idle(active, nenv, env, "xc_nadd_fock_build_unrestricted");
    std::vector<xc_bfogc*> sub(1, active);
    for (int i = 0; i < nenv; ++i) {
      require(env[i] && Pa_env[i] && Pb_env[i], XC_ERR_ARG,
              "xc_nadd_fock_build_unrestricted: null environment controller or density");
      require(env[i]->ctx == ctx, XC_ERR_ARG, "xc_nadd_fock_build_unrestricted: controllers live on different contexts");
      sub.push_back(env[i]);
    }
    // host spin densities into each controller's P (alpha) and Pb (beta) buffers
    std::vector<const double*> dPa(nenv), dPb(nenv);
    for (size_t i = 0; i < sub.size(); ++i) {
      xc_bfogc* b = sub[i];
      ensure_pol_buffers(b, precision == XC_PREC_FP32);
      const int m = b->basis->nao;
      const double* ha = i == 0 ? Pa_active : Pa_env[i - 1];
      const double* hb = i == 0 ? Pb_active : Pb_env[i - 1];
      ctx->stage.up(ctx->stream, b->d_P.p, ha, sizeof(double) * m * m);
      ctx->stage.up(ctx->stream, b->d_Pb.p, hb, sizeof(double) * m * m);
      if (i > 0) {
        dPa[i - 1] = b->d_P.p;
        dPb[i - 1] = b->d_Pb.p;
      }
    }
    enqueue_nadd_pol(active, nenv, env, functional, precision, thr, active->d_P.p, active->d_Pb.p, dPa.data(),
                     dPb.data(), active->d_F.p, active->d_Fb.p);
    const int n = active->basis->nao;
    ctx->stage.down(ctx->stream, {{Fa, active->d_F.p, sizeof(double) * n * n}, {Fb, active->d_Fb.p, sizeof(double) * n * n}});
    if (energy) *energy = *ctx->energy;
  });
}

int xc_bfogc_update_density(xc_bfogc* bf, int precision, const double* dP, int with_gradient) {
  return guarded([&] {
    require(bf && dP, XC_ERR_ARG, "xc_bfogc_update_density: null argument");
    require(precision != XC_PREC_MIXED, XC_ERR_ARG,
          "mixed precision is available for restricted single-system builds only");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32, XC_ERR_ARG, "unknown precision");
    require(!with_gradient || bf->deriv >= 1, XC_ERR_STATE,
            "xc_bfogc_update_density: gradient requested but AO gradients not evaluated");
    require(precision == XC_PREC_FP64 || bf->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
    require(precision == XC_PREC_FP32 || bf->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require_idle(bf, "xc_bfogc_update_density");
    const int n = bf->basis->nao;
    const int64_t N = bf->grid->npts;
    if (!bf->d_rho_c.p) {
      bf->d_rho_c.alloc(ctx, N);
      bf->d_grad_c.alloc(ctx, 3 * N);
      bf->d_ecache.alloc(ctx, kNumFunctionals);
    }
    const int g = with_gradient ? 1 : 0;
    if (precision == XC_PREC_FP32) {
      launch_to_float(ctx->stream, dP, bf->d_P32.p, (int64_t)n * n);
      run_density<float>(bf, bf->d_t32.p, bf->d_P32.p, g, ctx->lanes);
    } else {
      run_density<double>(bf, bf->d_t64.p, dP, g, ctx->lanes);
    }
    launch_reduce_partials(ctx->stream, bf->d_blocks.p, bf->bs, N, bf->d_part.p, g, bf->d_rho_c.p, bf->d_grad_c.p,
                           0);
    HIPX(hipGetLastError());
    bf->rho_c_valid = true;
    bf->rho_c_grad = with_gradient != 0;
    for (bool& v : bf->ecache_valid) v = false;
  });
}

int xc_nadd_fock_build_cached(xc_bfogc* act, int nenv, xc_bfogc* const* env, int functional, int precision,
                              double thr, double* dF, double* energy) {
  return guarded([&] {
    require(act && dF, XC_ERR_ARG, "xc_nadd_fock_build_cached: null argument");
    require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
    require(precision != XC_PREC_MIXED, XC_ERR_ARG,
          "mixed precision is available for restricted single-system builds only");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32, XC_ERR_ARG, "unknown precision");
    require(nenv >= 0 && (nenv == 0 || env), XC_ERR_ARG, "non-additive build: null environment list");
    xc_ctx* ctx = act->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    const bool gga = functional_is_gga(functional);
    require(!gga || act->deriv >= 1, XC_ERR_STATE, "GGA functional needs AO gradients (highest derivative 1)");
    require(precision == XC_PREC_FP64 || act->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
    require(precision == XC_PREC_FP32 || act->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
    std::vector<xc_bfogc*> sub(1, act);
    for (int i = 0; i < nenv; ++i) {
      require(env[i], XC_ERR_ARG, "non-additive build: null environment controller");
      require(env[i] != act, XC_ERR_ARG, "non-additive build: the active controller is also listed as environment");
      for (int j = 0; j < i; ++j)
        require(env[j] != env[i], XC_ERR_ARG, "non-additive build: an environment controller is listed twice");
      sub.push_back(env[i]);
    }
    for (xc_bfogc* b : sub) {
      require(b->ctx == ctx, XC_ERR_ARG, "non-additive build: controllers live on different contexts");
      require(b->grid == act->grid, XC_ERR_ARG,
              "non-additive build: all subsystem controllers must be defined on the same (supersystem) grid");
      require_idle(b, "xc_nadd_fock_build_cached");
      require(b->rho_c_valid, XC_ERR_STATE,
              "xc_nadd_fock_build_cached: a subsystem has no cached density (call xc_bfogc_update_density)");
      require(!gga || b->rho_c_grad, XC_ERR_STATE,
              "xc_nadd_fock_build_cached: GGA functional needs cached density gradients");
    }
    hipStream_t s = ctx->stream;
    ctx->mark();
    ctx->mark();
    ctx->mark();
    const EnvEnergies env_e = run_nadd_functional(sub, functional, true);
    ctx->mark();
    run_nadd_fock(sub, functional, precision, thr, env_e, true, dF);
    ctx->mark();
    HIPX(hipGetLastError());
    if (energy) {
      HIPX(hipStreamSynchronize(s));
      *energy = *ctx->energy;
    }
  });
}

int xc_nadd_fock_build_device(xc_bfogc* active, int nenv, xc_bfogc* const* env, int functional, int precision,
                              double thr, const double* dP_active, const double* const* dP_env, double* dF,
                              double* energy) {
  return guarded([&] {
    require(active && dP_active && dF, XC_ERR_ARG, "xc_nadd_fock_build_device: null argument");
    xc_ctx* ctx = active->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require_idle(active, nenv, env, "xc_nadd_fock_build_device");
    enqueue_nadd(active, nenv, env, functional, precision, thr, dP_active, dP_env, dF);
    if (energy) {
      HIPX(hipStreamSynchronize(ctx->stream));
      *energy = *ctx->energy;
    }
  });
}

int xc_nadd_fock_build(xc_bfogc* active, int nenv, xc_bfogc* const* env, int functional, int precision, double thr,
                       const double* P_active, const double* const* P_env, double* F, double* energy) {
  return guarded([&] {
    require(active && P_active && F, XC_ERR_ARG, "xc_nadd_fock_build: null argument");
    require(nenv >= 0 && (nenv == 0 || (env && P_env)), XC_ERR_ARG, "xc_nadd_fock_build: null environment list");
    xc_ctx* ctx = active->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require_idle(active, nenv, env, "xc_nadd_fock_build");
    const int n = active->basis->nao;
    ctx->stage.up(ctx->stream, active->d_P.p, P_active, sizeof(double) * n * n);
    std::vector<const double*> dP(nenv);
    for (int i = 0; i < nenv; ++i) {
      require(env[i] && P_env[i], XC_ERR_ARG, "xc_nadd_fock_build: null environment controller or density");
      require(env[i]->ctx == ctx, XC_ERR_ARG, "xc_nadd_fock_build: controllers live on different contexts");
      const int m = env[i]->basis->nao;
      ctx->stage.up(ctx->stream, env[i]->d_P.p, P_env[i], sizeof(double) * m * m);
      dP[i] = env[i]->d_P.p;
    }
    enqueue_nadd(active, nenv, env, functional, precision, thr, active->d_P.p, dP.data(), active->d_F.p);
    ctx->stage.down(ctx->stream, {{F, active->d_F.p, sizeof(double) * n * n}});
    if (energy) *energy = *ctx->energy;
  });
}

int xc_fock_build_device(xc_bfogc* bf, int functional, int precision, double thr, const double* dP, double* dF,
                         double* energy) {
  return guarded([&] {
    require(bf && dP && dF, XC_ERR_ARG, "xc_fock_build_device: null argument");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    enqueue_build(bf, functional, precision, thr, dP, dF, ctx->lanes, ctx->energy);
    if (energy) {
      HIPX(hipStreamSynchronize(ctx->stream));
      *energy = *ctx->energy;
    }
  });
}

int xc_fock_build_packed(int nsys, xc_bfogc* const* bfs, int functional, int precision, double thr,
                         const double* const* dP, double* const* dF, double* energies) {
  return guarded([&] {
    require(nsys >= 1 && bfs && dP && dF && energies, XC_ERR_ARG, "xc_fock_build_packed: bad arguments");
    xc_ctx* ctx = bfs[0] ? bfs[0]->ctx : nullptr;
    require(ctx != nullptr, XC_ERR_ARG, "xc_fock_build_packed: null controller");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
    require(precision != XC_PREC_MIXED, XC_ERR_ARG,
          "mixed precision is available for restricted single-system builds only");
  require(precision == XC_PREC_FP64 || precision == XC_PREC_FP32, XC_ERR_ARG, "unknown precision");
    const bool gga = functional_is_gga(functional);
    const bool fp32 = precision == XC_PREC_FP32;
    std::vector<DevBlock> blocks;
    std::vector<PackSys> sys(nsys);
    std::vector<WorkItem> dens[2];
    std::vector<FockItem> fock[kFockShapes];
    int64_t maxnn = 0;
    int maxn = 0;
    for (int i = 0; i < nsys; ++i) {
      xc_bfogc* bf = bfs[i];
      require(bf && dP[i] && dF[i], XC_ERR_ARG, "xc_fock_build_packed: null controller or matrix");
      require(bf->ctx == ctx, XC_ERR_ARG, "xc_fock_build_packed: controllers of different contexts");
      for (int j = 0; j < i; ++j)
        require(bfs[j] != bf, XC_ERR_ARG, "xc_fock_build_packed: a controller appears twice (shared scratch)");
      require(!bf->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
      require(bf->bs == kTile, XC_ERR_STATE, "xc_fock_build_packed: controllers need 128-point blocks");
      require(!gga || bf->deriv >= 1, XC_ERR_STATE, "GGA functional needs AO gradients (highest derivative 1)");
      require(!fp32 || bf->d_t32.p, XC_ERR_STATE, "FP32 contractions need keep_fp32 tiles");
      require(fp32 || bf->d_t64.p, XC_ERR_STATE, "FP64 contractions need FP64 tiles");
      const int n = bf->basis->nao;
      const int blk0 = (int)blocks.size();
      for (DevBlock b : bf->blocks) {
        b.sys = i;
        blocks.push_back(b);
      }
      // each system's density as in its build alone: the form sums in another order, and a
      // deterministic context's F is the same packed and alone
      const bool form = !fp32 && use_form(gga, n);
      for (WorkItem w : bf->dens_work) {
        w.block += blk0;
        dens[form].push_back(w);
      }
      for (int c = 0; c < kFockShapes; ++c)
        for (FockItem f : bf->fock_items[c]) {
          f.block += blk0;
          fock[c].push_back(f);
        }
      PackSys& ps = sys[i];
      ps.tiles = fp32 ? (const void*)bf->d_t32.p : (const void*)bf->d_t64.p;
      ps.P = fp32 ? (const void*)bf->d_P32.p : form ? (const void*)bf->d_U.p : (const void*)dP[i];
      ps.P64 = dP[i];
      ps.P32 = fp32 ? bf->d_P32.p : nullptr;
      ps.ao_idx = bf->d_ao_idx.p;
      ps.part = bf->d_part.p;
      ps.w = bf->grid->d_w.p;
      ps.vs = bf->d_vs.p;
      ps.gw = bf->d_gw.p;
      ps.U = bf->d_U.p;
      ps.T = bf->d_T.p;
      ps.ent = bf->d_rowent.p;
      ps.row_ptr = bf->d_rowptr.p;
      ps.F = dF[i];
      ps.eblk = bf->d_eblk.p;
      ps.npts = bf->grid->npts;
      ps.n = n;
      ps.blk0 = blk0;
      ps.nxc = (int)((bf->grid->npts + kTile - 1) / kTile);
      maxnn = std::max(maxnn, (int64_t)n * n);
      maxn = std::max(maxn, n);
    }
    // a composition seen once before runs as a captured graph; the first build is eager
    std::vector<uint64_t> key;
    for (int i = 0; i < nsys; ++i) key.push_back((uint64_t)(uintptr_t)bfs[i]);
    uint64_t thr_bits = 0;
    std::memcpy(&thr_bits, &thr, sizeof(thr_bits));
    key.push_back((uint64_t)functional);
    key.push_back((uint64_t)precision);
    key.push_back(thr_bits);
    // graphs pay where launches are short (many small systems: 4.1 vs 4.3 ms for 32 small
    // molecules); a graph runs the class launches of a stage one after another instead of on
    // the four lanes, which costs more than it saves for packs of large grids (25 FDE subsystems
    // on a 353 701-point grid: 3.5 vs 2.7 ms), so large packs stay eager
    const bool graphable = blocks.size() <= 32768;
    auto hit = graphable ? ctx->pack_graphs.find(key) : ctx->pack_graphs.end();
    bool capture = false;
    PackWork* pwp = nullptr;
    if (!graphable) {
      if (!ctx->pack) ctx->pack = new PackWork();
      pwp = ctx->pack;
    } else if (hit == ctx->pack_graphs.end()) {
      if (ctx->pack_graphs.size() >= 16) {  // bounded cache: forget the least recently used composition
        auto lru = ctx->pack_graphs.begin();
        for (auto it = ctx->pack_graphs.begin(); it != ctx->pack_graphs.end(); ++it)
          if (it->second->last_use < lru->second->last_use) lru = it;
        delete lru->second;
        ctx->pack_graphs.erase(lru);
      }
      ctx->pack_graphs.emplace(key, new PackWork()).first->second->last_use = ++ctx->pack_calls;
      if (!ctx->pack) ctx->pack = new PackWork();
      pwp = ctx->pack;
    } else {
      pwp = hit->second;
      pwp->last_use = ++ctx->pack_calls;
      capture = pwp->exec == nullptr;
    }
    PackWork& pw = *pwp;
    if (pw.round.n < (size_t)nsys * kPackRoundBlocks) pw.round.alloc(ctx, (size_t)2 * nsys * kPackRoundBlocks);
    if (ctx->pack_energies < (size_t)nsys) {
      HIPX(hipStreamSynchronize(ctx->stream));
      if (ctx->pack_energy) (void)hipHostFree(ctx->pack_energy);
      ctx->pack_energy = nullptr;
      ctx->pack_energies = 0;
      const size_t want = std::max<size_t>(2 * (size_t)nsys, 64);
      HIPX(hipHostMalloc((void**)&ctx->pack_energy, sizeof(double) * want, hipHostMallocMapped | hipHostMallocCoherent));
      ctx->pack_energies = want;
    }
    for (int i = 0; i < nsys; ++i) {
      sys[i].round = pw.round.p + (size_t)i * kPackRoundBlocks;
      sys[i].E = ctx->pack_energy + i;
    }
    hipStream_t s = ctx->stream;
    const Lanes& L = ctx->lanes;
    const int g = gga ? 1 : 0;
    // the per-system table (matrices of this call) is uploaded every time; a replayed graph reads it
    upload_grow(ctx, pw.sys, sys);
    if (pw.exec) {
      HIPX(hipGraphLaunch(pw.exec, s));
    } else {
      upload_grow(ctx, pw.blocks, blocks);
      for (int k = 0; k < 2; ++k) upload_grow(ctx, pw.dens[k], dens[k]);
      for (int c = 0; c < kFockShapes; ++c) upload_grow(ctx, pw.fock[c], fock[c]);
      const PackSys* dsys = pw.sys.p;
      // one launch per stage (and Fock shape) for every system of the pack
      auto enqueue = [&]() {
        if (fp32) launch_pack_to_float(s, dsys, nsys, maxnn);
        if (!dens[1].empty()) launch_fold(s, nullptr, nullptr, maxn, dsys, nsys);
        over_lanes(L, 2, [&](int k) { return (int)dens[k].size(); }, [&](int k, hipStream_t st) {
          if (fp32)
            launch_density_sub<float>(st, pw.dens[k].p, (int)dens[k].size(), pw.blocks.p, nullptr, nullptr, nullptr, 0,
                                      g, nullptr, 0, dsys);
          else
            launch_density_sub<double>(st, pw.dens[k].p, (int)dens[k].size(), pw.blocks.p, nullptr, nullptr, nullptr, 0,
                                       g, nullptr, 0, dsys, nullptr, nullptr, k == 1);
        });
        launch_functional_packed(s, functional, (int)blocks.size(), pw.blocks.p, dsys);
        over_lanes(L, kFockShapes, [&](int c) { return (int)fock[c].size(); }, [&](int c, hipStream_t st) {
          if (fp32)
            launch_fock_sub<float>(st, c, pw.fock[c].p, (int)fock[c].size(), pw.blocks.p, nullptr, nullptr, nullptr, g,
                                   thr, nullptr, 0, dsys);
          else
            launch_fock_sub<double>(st, c, pw.fock[c].p, (int)fock[c].size(), pw.blocks.p, nullptr, nullptr, nullptr, g,
                                    thr, nullptr, 0, dsys);
        });
        const bool direct = maxn <= kDirectRows;
        static_assert(kDirectRows <= kPackRoundBlocks, "a system's rounding partials fit its slots");
        ReduceOut out{};
        out.direct = direct;
        out.round = fp32 ? pw.round.p : nullptr;  // (each system's own slots from the table)
        if (fp32)
          launch_fock_reduce<float>(s, nullptr, nullptr, nullptr, nullptr, nullptr, maxn, dsys, nsys,
                                    ctx->deterministic, false, out);
        else
          launch_fock_reduce<double>(s, nullptr, nullptr, nullptr, nullptr, nullptr, maxn, dsys, nsys,
                                     ctx->deterministic, false, out);
        if (!direct) launch_pack_finalize(s, dsys, nsys, fp32 ? 1 : 0);
        if (fp32 || !direct) launch_pack_sum(s, dsys, nsys, !fp32 ? 0 : direct ? -1 : kPackRoundBlocks);
      };
      if (capture) {
        // second build of this composition: capture it (kernel nodes only, no memsets) into its own lists
        hipGraph_t graph = nullptr;
        HIPX(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        try {
          enqueue();
        } catch (...) {
          (void)hipStreamEndCapture(s, &graph);
          if (graph) (void)hipGraphDestroy(graph);
          throw;
        }
        HIPX(hipStreamEndCapture(s, &graph));
        hipGraphExec_t exec = nullptr;
        const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        HIPX(e);
        pw.exec = exec;
        HIPX(hipGraphLaunch(pw.exec, s));
      } else {
        enqueue();
      }
    }
    HIPX(hipGetLastError());
    HIPX(hipStreamSynchronize(s));
    std::copy(ctx->pack_energy, ctx->pack_energy + nsys, energies);
  });
}

namespace {
// XC gradient of one (restricted: Pb == nullptr) or two spin density matrices (host).
void geom_gradient(xc_bfogc* bf, int functional, const double* Pa, const double* Pb, int natoms, const int* ao_atom,
                   double* grad, double* energy) {
  require(bf && Pa && grad && ao_atom && natoms > 0, XC_ERR_ARG, "xc_geom_gradient: bad arguments");
  require(!bf->in_flight, XC_ERR_STATE, "a server build of this controller is in flight");
  require(functional >= 0 && functional < kNumFunctionals, XC_ERR_ARG, "unknown functional");
  const bool gga = functional_is_gga(functional);
  require(bf->deriv >= (gga ? 2 : 1), XC_ERR_STATE,
          gga ? "xc_geom_gradient: a GGA gradient needs AO second derivatives (highest derivative 2)"
              : "xc_geom_gradient: needs AO gradients (highest derivative 1)");
  require(bf->d_t64.p, XC_ERR_STATE, "xc_geom_gradient: needs FP64 tiles");
  xc_ctx* ctx = bf->ctx;
  std::lock_guard<std::recursive_mutex> lk(ctx->mu);
  hipStream_t s = ctx->stream;
  const int n = bf->basis->nao;
  const int64_t N = bf->grid->npts;
  const int nxc = (int)((N + kTile - 1) / kTile);
  for (int i = 0; i < n; ++i)
    require(ao_atom[i] >= 0 && ao_atom[i] < natoms, XC_ERR_INPUT, "xc_geom_gradient: AO atom index out of range");
  if (!bf->d_gacc.p) {
    bf->d_gacc.alloc(ctx, (size_t)3 * std::max(n, 1));
    bf->d_ao_atom.alloc(ctx, (size_t)std::max(n, 1));
  }
  if ((int64_t)bf->d_gout.n < 3 * (int64_t)natoms) bf->d_gout.alloc(ctx, (size_t)3 * natoms);
  if (Pb) ensure_pol_buffers(bf, false);
  ctx->stage.up(s, bf->d_ao_atom.p, ao_atom, sizeof(int) * n);
  ctx->stage.up(s, bf->d_P.p, Pa, sizeof(double) * n * n);
  if (Pb) ctx->stage.up(s, bf->d_Pb.p, Pb, sizeof(double) * n * n);
  // density and functional as in a Fock build (FP64), then the gradient contractions
  if (!Pb) {
    run_density<double>(bf, bf->d_t64.p, bf->d_P.p, gga ? 1 : 0, ctx->lanes);
    if (bf->bs == kTile) {
      launch_functional(s, functional, N, kTile, nullptr, nullptr, bf->d_blocks.p, bf->d_part.p,
                        bf->grid->d_w.p, nullptr, nullptr, nullptr, bf->d_vs.p, bf->d_gw.p, bf->d_eblk.p);
    } else {
      launch_reduce_partials(s, bf->d_blocks.p, bf->bs, N, bf->d_part.p, gga ? 1 : 0, bf->d_rho.p, bf->d_grad.p);
      launch_functional(s, functional, N, kTile, bf->d_rho.p, gga ? bf->d_grad.p : nullptr, nullptr,
                        nullptr, bf->grid->d_w.p, nullptr, nullptr, nullptr, bf->d_vs.p, bf->d_gw.p, bf->d_eblk.p);
    }
  } else {
    const double* Ps[2] = {bf->d_P.p, bf->d_Pb.p};
    double* rho[2] = {bf->d_rho.p, bf->d_rho_b.p};
    double* grd[2] = {bf->d_grad.p, bf->d_grad_b.p};
    for (int sp = 0; sp < 2; ++sp) {
      run_density<double>(bf, bf->d_t64.p, Ps[sp], gga ? 1 : 0, ctx->lanes);
      launch_reduce_partials(s, bf->d_blocks.p, bf->bs, N, bf->d_part.p, gga ? 1 : 0, rho[sp], grd[sp]);
    }
    launch_functional_pol(s, functional, N, kTile, bf->d_rho.p, bf->d_grad.p, bf->d_rho_b.p,
                          bf->d_grad_b.p, bf->grid->d_w.p, bf->d_vs.p, bf->d_gw.p, bf->d_vs_b.p, bf->d_gw_b.p,
                          bf->d_eblk.p);
  }
  launch_fill(s, bf->d_gacc.p, (int64_t)3 * n, 0.0);
  // restricted: -2 P_mu,nu with the total-density potential; unrestricted: the same per spin
  launch_gradient(s, bf->d_dens_work.p, (int)bf->dens_work.size(), bf->d_blocks.p, bf->d_ao_idx.p, bf->d_t64.p,
                  bf->d_P.p, n, bf->d_vs.p, bf->d_gw.p, gga ? 1 : 0, N, bf->d_gacc.p);
  if (Pb)
    launch_gradient(s, bf->d_dens_work.p, (int)bf->dens_work.size(), bf->d_blocks.p, bf->d_ao_idx.p, bf->d_t64.p,
                    bf->d_Pb.p, n, bf->d_vs_b.p, bf->d_gw_b.p, gga ? 1 : 0, N, bf->d_gacc.p);
  launch_gradient_atoms(s, bf->d_gacc.p, bf->d_ao_atom.p, n, natoms, bf->d_gout.p);
  launch_sum(s, bf->d_eblk.p, nxc, ctx->energy);
  HIPX(hipGetLastError());
  ctx->stage.down(s, {{grad, bf->d_gout.p, sizeof(double) * 3 * natoms}});
  if (energy) *energy = *ctx->energy;
}
}  // namespace

int xc_geom_gradient(xc_bfogc* bf, int functional, const double* P, int natoms, const int* ao_atom, double* grad,
                     double* energy) {
  return guarded([&] { geom_gradient(bf, functional, P, nullptr, natoms, ao_atom, grad, energy); });
}

int xc_geom_gradient_unrestricted(xc_bfogc* bf, int functional, const double* Pa, const double* Pb, int natoms,
                                  const int* ao_atom, double* grad, double* energy) {
  return guarded([&] {
    require(Pb, XC_ERR_ARG, "xc_geom_gradient_unrestricted: null beta density");
    geom_gradient(bf, functional, Pa, Pb, natoms, ao_atom, grad, energy);
  });
}

int xc_fock_build_unrestricted(xc_bfogc* bf, int functional, int precision, double thr, const double* Pa,
                               const double* Pb, double* Fa, double* Fb, double* energy) {
  return guarded([&] {
    require(bf && Pa && Pb && Fa && Fb, XC_ERR_ARG, "xc_fock_build_unrestricted: null argument");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require_idle(bf, "xc_fock_build_unrestricted");
    const int n = bf->basis->nao;
    ensure_pol_buffers(bf, precision == XC_PREC_FP32);
    ctx->stage.up(ctx->stream, bf->d_P.p, Pa, sizeof(double) * n * n);
    ctx->stage.up(ctx->stream, bf->d_Pb.p, Pb, sizeof(double) * n * n);
    enqueue_build_pol(bf, functional, precision, thr, bf->d_P.p, bf->d_Pb.p, bf->d_F.p, bf->d_Fb.p, ctx->lanes,
                      ctx->energy);
    ctx->stage.down(ctx->stream, {{Fa, bf->d_F.p, sizeof(double) * n * n}, {Fb, bf->d_Fb.p, sizeof(double) * n * n}});
    if (energy) *energy = *ctx->energy;
  });
}

int xc_fock_build_unrestricted_device(xc_bfogc* bf, int functional, int precision, double thr, const double* dPa,
                                      const double* dPb, double* dFa, double* dFb, double* energy) {
  return guarded([&] {
    require(bf && dPa && dPb && dFa && dFb, XC_ERR_ARG, "xc_fock_build_unrestricted_device: null argument");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    enqueue_build_pol(bf, functional, precision, thr, dPa, dPb, dFa, dFb, ctx->lanes, ctx->energy);
    if (energy) {
      HIPX(hipStreamSynchronize(ctx->stream));
      *energy = *ctx->energy;
    }
  });
}

int xc_ri_metric(int naux_shell, const int* aux_l, const int* aux_pure, const int* aux_nprim,
                 const double* aux_center, const double* aux_alpha, const double* aux_coef, double* M) {
  return guarded([&] {
    require(M, XC_ERR_ARG, "xc_ri_metric: null output");
    auto ax = host_shells("xc_ri_metric", naux_shell, aux_l, aux_pure, aux_nprim, aux_center, aux_alpha, aux_coef, 4);
    std::vector<double> m;
    ri_metric(ax, m);
    std::copy(m.begin(), m.end(), M);
  });
}

int xc_coulomb_create(xc_basis* basis, xc_basis* aux, double threshold, xc_coulomb** out) {
  return guarded([&] {
    require(basis && aux && out && threshold >= 0.0, XC_ERR_ARG, "xc_coulomb_create: bad arguments");
    require(basis->ctx == aux->ctx, XC_ERR_ARG, "xc_coulomb_create: bases live on different contexts");
    require(basis->maxl <= kJMaxLPrim, XC_ERR_INPUT,
            "xc_coulomb_create: orbital shells above l = " + std::to_string(kJMaxLPrim));
    require(aux->maxl <= kJMaxLAux, XC_ERR_INPUT,
            "xc_coulomb_create: auxiliary shells above l = " + std::to_string(kJMaxLAux));
    xc_ctx* ctx = basis->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipSetDevice(ctx->device));
    auto* jc = new xc_coulomb();
    try {
      jc->ctx = ctx;
      jc->basis = basis;
      jc->aux = aux;
      // significant primitive pairs, grouped by angular momentum
      const auto& sh = basis->shells;
      const int ns = (int)sh.size();
      for (int A = 0; A < ns; ++A)
        for (int B = 0; B <= A; ++B) {
          const DevShell& a = sh[A];
          const DevShell& b = sh[B];
          const double dx = a.cx - b.cx, dy = a.cy - b.cy, dz = a.cz - b.cz, ab2 = dx * dx + dy * dy + dz * dz;
          for (int i = 0; i < a.nprim; ++i)
            for (int j = 0; j < b.nprim; ++j) {
              const double ea = basis->alpha[a.prim_off + i], eb = basis->alpha[b.prim_off + j];
              const double p = ea + eb;
              const double K = basis->coef[a.prim_off + i] * basis->coef[b.prim_off + j] * std::exp(-ea * eb / p * ab2);
              if (std::fabs(K) * std::pow(M_PI / p, 1.5) < threshold) continue;
              JPair q{};
              q.A = A;
              q.B = B;
              q.L = a.l + b.l;
              q.sym = A == B ? 1.0 : 2.0;
              q.p = p;
              q.K = K;
              const double ac[3] = {a.cx, a.cy, a.cz}, bc[3] = {b.cx, b.cy, b.cz};
              for (int d = 0; d < 3; ++d) {
                q.P[d] = (ea * ac[d] + eb * bc[d]) / p;
                q.PA[d] = q.P[d] - ac[d];
                q.PB[d] = q.P[d] - bc[d];
              }
              jc->pairs.push_back(q);
            }
        }
      // by L, then l_A and the kinds of the shells, otherwise in order (a counting sort)
      const auto key = [&](const JPair& q) {
        return ((q.L * (kJMaxLPrim + 1) + sh[q.A].l) * 2 + sh[q.A].pure) * 2 + sh[q.B].pure;
      };
      {
        std::vector<size_t> at((2 * kJMaxLPrim + 1) * (kJMaxLPrim + 1) * 4 + 1, 0);
        for (const auto& q : jc->pairs) ++at[key(q) + 1];
        for (size_t k = 1; k < at.size(); ++k) at[k] += at[k - 1];
        std::vector<JPair> sorted(jc->pairs.size());
        for (const auto& q : jc->pairs) sorted[at[key(q)]++] = q;
        jc->pairs.swap(sorted);
      }
      const auto hcount = [](int L) { return (L + 1) * (L + 2) * (L + 3) / 6; };
      constexpr int kMaxLab = 2 * kJMaxLPrim;
      JView& view = jc->view;
      int64_t off = 0;
      int count[kMaxLab + 1] = {};
      for (auto& q : jc->pairs) {
        q.herm_off = (int)off;
        off += hcount(q.L);
        ++count[q.L];
      }
      require(off < (1LL << 31), XC_ERR_INPUT, "xc_coulomb_create: too many primitive pairs");
      jc->herm_total = off;
      int64_t h0 = 0;
      for (int L = 0; L <= kMaxLab; ++L) {
        view.pair0[L + 1] = view.pair0[L] + count[L];
        view.herm0[L] = (int)h0;
        h0 += (int64_t)count[L] * hcount(L);
      }
      for (const auto& s : aux->shells) {
        jc->cart_off.push_back(jc->ncart_aux);
        jc->ncart_aux += s.ncart;
      }
      // auxiliary primitives by angular momentum
      std::vector<double> apos, acoef;
      std::vector<int> prim_shell, shell_prim(aux->shells.size(), 0);
      int64_t ah = 0;
      for (int l = 0; l <= kJMaxLAux; ++l) {
        view.aux0[l] = (int)prim_shell.size();
        view.aherm0[l] = (int)ah;
        for (size_t k = 0; k < aux->shells.size(); ++k) {
          const DevShell& s = aux->shells[k];
          if (s.l != l) continue;
          shell_prim[k] = (int)prim_shell.size();
          for (int i = 0; i < s.nprim; ++i) {
            apos.insert(apos.end(), {s.cx, s.cy, s.cz, aux->alpha[s.prim_off + i]});
            acoef.push_back(aux->coef[s.prim_off + i]);
            prim_shell.push_back((int)k);
          }
        }
        ah += (int64_t)(prim_shell.size() - view.aux0[l]) * hcount(l);
      }
      view.aux0[kJMaxLAux + 1] = jc->naux = (int)prim_shell.size();
      require(ah < (1LL << 31), XC_ERR_INPUT, "xc_coulomb_create: too many auxiliary primitives");
      jc->aherm_total = ah;
      jc->plan_items();
      const int n = basis->nao;
      jc->d_pairs.upload(ctx, jc->pairs.data(), jc->pairs.size());
      jc->d_cart_off.upload(ctx, jc->cart_off.data(), jc->cart_off.size());
      std::vector<double> ppos(4 * jc->pairs.size());
      for (size_t q = 0; q < jc->pairs.size(); ++q) {
        const JPair& pr = jc->pairs[q];
        const double x[4] = {pr.P[0], pr.P[1], pr.P[2], pr.p};
        std::copy(x, x + 4, ppos.begin() + 4 * q);
      }
      static const std::vector<double> boys = boys_table();
      jc->d_pair.upload(ctx, ppos.data(), ppos.size());
      jc->d_aux.upload(ctx, apos.data(), apos.size());
      jc->d_prim_coef.upload(ctx, acoef.data(), acoef.size());
      jc->d_prim_shell.upload(ctx, prim_shell.data(), prim_shell.size());
      jc->d_shell_prim.upload(ctx, shell_prim.data(), shell_prim.size());
      jc->d_boys.upload(ctx, boys.data(), boys.size());
      view.pair = jc->d_pair.p;
      view.aux = jc->d_aux.p;
      view.boys = jc->d_boys.p;
      for (int k = 0; k < 2; ++k)
        for (int c = 0; c < kJClasses; ++c)
          jc->d_items[k][c].upload(ctx, jc->items[k][c].data(), jc->items[k][c].size());
      for (int c = 0; c < kJPairClasses; ++c)
        jc->d_pair_items[c].upload(ctx, jc->pair_items[c].data(), jc->pair_items[c].size());
      jc->d_U.alloc(ctx, std::max<int64_t>(jc->aherm_total, 1));  // U of step 4, W of step 2
      jc->d_D.alloc(ctx, std::max<int64_t>(off, 1));
      jc->d_V.alloc(ctx, std::max<int64_t>(off, 1));
      jc->d_bc.alloc(ctx, std::max(jc->ncart_aux, 1));
      jc->d_cc.alloc(ctx, std::max(jc->ncart_aux, 1));
      jc->d_P.alloc(ctx, (size_t)n * n);
      jc->d_J.alloc(ctx, (size_t)n * n);
      HIPX(hipStreamSynchronize(ctx->stream));
    } catch (...) {
      delete jc;
      throw;
    }
    ++ctx->live_handles;
    *out = jc;
  });
}

int xc_coulomb_info(const xc_coulomb* jc, int64_t* npairs, int64_t* hermite_terms) {
  return guarded([&] {
    require(jc, XC_ERR_ARG, "xc_coulomb_info: null handle");
    if (npairs) *npairs = (int64_t)jc->pairs.size();
    if (hermite_terms) *hermite_terms = jc->herm_total;
  });
}

int xc_coulomb_destroy(xc_coulomb* jc) {
  return guarded([&] {
    if (!jc) return;
    (void)hipStreamSynchronize(jc->ctx->stream);
    --jc->ctx->live_handles;
    delete jc;
  });
}

// b in Cartesian auxiliary functions (d_bc) from the density in d_P.
static void enqueue_coulomb_rhs(xc_coulomb* jc) {
  xc_ctx* ctx = jc->ctx;
  hipStream_t s = ctx->stream;
  const int n = jc->basis->nao;
  over_lanes(ctx->lanes, kJPairClasses, [&](int c) { return (int)jc->pair_items[c].size(); },
             [&](int c, hipStream_t st) {
    launch_jdens(st, c, jc->d_pair_items[c].p, (int)jc->pair_items[c].size(), jc->d_pairs.p, jc->basis->d_shells.p,
                 jc->basis->d_ang.p, jc->view, jc->d_P.p, n, jc->d_D.p);
  });
  launch_fill(s, jc->d_U.p, jc->aherm_total, 0.0);
  // the widest classes (the longest items, few of them) beside the others
  over_lanes(ctx->lanes, kJClasses, [&](int c) { return (int)jc->items[0][c].size(); }, [&](int c, hipStream_t st) {
    launch_jrhs(st, c, jc->d_items[0][c].p, (int)jc->items[0][c].size(), jc->view, jc->d_D.p, jc->d_U.p);
  });
  launch_jaux_out(s, jc->view, jc->aux->d_shells.p, jc->aux->nshell, jc->d_shell_prim.p, jc->d_prim_coef.p,
                  jc->d_cart_off.p, jc->d_U.p, jc->d_bc.p);
  HIPX(hipGetLastError());
}

// J (d_J) from the Cartesian auxiliary coefficients in d_cc.
static void enqueue_coulomb_matrix(xc_coulomb* jc) {
  xc_ctx* ctx = jc->ctx;
  hipStream_t s = ctx->stream;
  const int n = jc->basis->nao;
  launch_jaux_in(s, jc->view, jc->naux, jc->d_prim_shell.p, jc->aux->d_shells.p, jc->d_prim_coef.p, jc->d_cart_off.p,
                 jc->d_cc.p, jc->d_U.p);
  launch_fill(s, jc->d_V.p, jc->herm_total, 0.0);
  over_lanes(ctx->lanes, kJClasses, [&](int c) { return (int)jc->items[1][c].size(); }, [&](int c, hipStream_t st) {
    launch_jpot(st, c, jc->d_items[1][c].p, (int)jc->items[1][c].size(), jc->view, jc->d_U.p, jc->d_V.p);
  });
  launch_fill(s, jc->d_J.p, (int64_t)n * n, 0.0);
  over_lanes(ctx->lanes, kJPairClasses, [&](int c) { return (int)jc->pair_items[c].size(); },
             [&](int c, hipStream_t st) {
    launch_jassemble(st, c, jc->d_pair_items[c].p, (int)jc->pair_items[c].size(), jc->d_pairs.p,
                     jc->basis->d_shells.p, jc->basis->d_ang.p, jc->view, jc->d_V.p, n, jc->d_J.p);
  });
  HIPX(hipGetLastError());
}

int xc_coulomb_rhs(xc_coulomb* jc, const double* P, double* b) {
  return guarded([&] {
    require(jc && P && b, XC_ERR_ARG, "xc_coulomb_rhs: null argument");
    xc_ctx* ctx = jc->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    hipStream_t s = ctx->stream;
    const int n = jc->basis->nao;
    ctx->stage.up(s, jc->d_P.p, P, sizeof(double) * n * n);
    enqueue_coulomb_rhs(jc);
    std::vector<double> bc(jc->ncart_aux);
    ctx->stage.down(s, {{bc.data(), jc->d_bc.p, sizeof(double) * bc.size()}});
    // Cartesian -> auxiliary AO: b_f = sum_c M[f][c] b_c
    for (int k = 0; k < jc->aux->nshell; ++k) {
      const DevShell& S = jc->aux->shells[k];
      for (int f = 0; f < S.nfunc; ++f) {
        double v = 0.0;
        for (int c = 0; c < S.ncart; ++c) v += jc->aux->ang[S.ang_off + f * S.ncart + c] * bc[jc->cart_off[k] + c];
        b[S.ao_off + f] = v;
      }
    }
  });
}

int xc_coulomb_matrix(xc_coulomb* jc, const double* c, double* J) {
  return guarded([&] {
    require(jc && c && J, XC_ERR_ARG, "xc_coulomb_matrix: null argument");
    xc_ctx* ctx = jc->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    hipStream_t s = ctx->stream;
    const int n = jc->basis->nao;
    // auxiliary AO -> Cartesian: cc_c = sum_f c_f M[f][c]
    std::vector<double> cc(std::max(jc->ncart_aux, 1), 0.0);
    for (int k = 0; k < jc->aux->nshell; ++k) {
      const DevShell& S = jc->aux->shells[k];
      for (int f = 0; f < S.nfunc; ++f)
        for (int q = 0; q < S.ncart; ++q)
          cc[jc->cart_off[k] + q] += c[S.ao_off + f] * jc->aux->ang[S.ang_off + f * S.ncart + q];
    }
    ctx->stage.up(s, jc->d_cc.p, cc.data(), sizeof(double) * jc->ncart_aux);
    enqueue_coulomb_matrix(jc);
    ctx->stage.down(s, {{J, jc->d_J.p, sizeof(double) * n * n}});
  });
}

int xc_coulomb_set_metric(xc_coulomb* jc, const double* L) {
  return guarded([&] {
    require(jc && L, XC_ERR_ARG, "xc_coulomb_set_metric: null argument");
    xc_ctx* ctx = jc->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    const int n = jc->aux->nao, B = kSolveBlock, nblk = (n + B - 1) / B;
    // the diagonal blocks' inverses, column by column (rows and columns beyond n: zero)
    std::vector<double> inv((size_t)nblk * B * B, 0.0);
    for (int k = 0; k < nblk; ++k) {
      const int m = std::min(B, n - k * B);
      const double* Lk = L + (size_t)k * B * n + (size_t)k * B;
      double* D = inv.data() + (size_t)k * B * B;
      for (int j = 0; j < m; ++j)
        for (int i = j; i < m; ++i) {
          double v = i == j ? 1.0 : 0.0;
          for (int q = j; q < i; ++q) v -= Lk[(size_t)i * n + q] * D[q * B + j];
          D[i * B + j] = v / Lk[(size_t)i * n + i];
        }
    }
    try {
      jc->d_dinv.upload(ctx, inv.data(), inv.size());
      jc->d_b.alloc(ctx, (size_t)std::max(n, 1));
      jc->d_y.alloc(ctx, (size_t)std::max(n, 1));
      jc->d_L.upload(ctx, L, (size_t)n * n);
    } catch (...) {
      jc->d_L.free_();
      throw;
    }
    HIPX(hipStreamSynchronize(ctx->stream));
  });
}

int xc_coulomb_build(xc_coulomb* jc, const double* P, double* J) {
  return guarded([&] {
    require(jc && P && J, XC_ERR_ARG, "xc_coulomb_build: null argument");
    require(jc->d_L.p, XC_ERR_STATE, "xc_coulomb_build: no metric (call xc_coulomb_set_metric)");
    xc_ctx* ctx = jc->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    hipStream_t s = ctx->stream;
    const int n = jc->basis->nao;
    ctx->stage.up(s, jc->d_P.p, P, sizeof(double) * n * n);
    enqueue_coulomb_rhs(jc);
    *ctx->flag = 0;  // (nothing that writes it is in flight: every call that does waits for it)
    launch_metric_solve(s, jc->d_L.p, jc->aux->nao, jc->d_dinv.p, jc->aux->d_shells.p, jc->aux->nshell,
                        jc->aux->d_ang.p, jc->d_cart_off.p, jc->d_bc.p, jc->d_b.p, jc->d_y.p, jc->d_cc.p, ctx->flag);
    enqueue_coulomb_matrix(jc);
    ctx->stage.down(s, {{J, jc->d_J.p, sizeof(double) * n * n}});
    require(*ctx->flag == 0, XC_ERR_INPUT, "array must not contain infs or NaNs");
  });
}

int xc_last_energy(xc_ctx* ctx, double* energy) {
  return guarded([&] {
    require(ctx && energy, XC_ERR_ARG, "null argument");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipStreamSynchronize(ctx->stream));
    *energy = *ctx->energy;
  });
}

int xc_fock_build(xc_bfogc* bf, int functional, int precision, double thr, const double* P, double* F,
                  double* energy) {
  return guarded([&] {
    require(bf && P && F, XC_ERR_ARG, "xc_fock_build: null argument");
    xc_ctx* ctx = bf->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require_idle(bf, "xc_fock_build");  // a server build reads d_P on its slot's stream to its end
    const int n = bf->basis->nao;
    ctx->stage.up(ctx->stream, bf->d_P.p, P, sizeof(double) * n * n);
    enqueue_build(bf, functional, precision, thr, bf->d_P.p, bf->d_F.p, ctx->lanes, ctx->energy);
    ctx->stage.down(ctx->stream, {{F, bf->d_F.p, sizeof(double) * n * n}});
    if (energy) *energy = *ctx->energy;
  });
}

int xc_ctx_set_deterministic(xc_ctx* ctx, int enable) {
  return guarded([&] {
    require(ctx, XC_ERR_ARG, "null context");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    require(ctx->live_handles == 0, XC_ERR_STATE,
            "xc_ctx_set_deterministic: set before any basis, grid or controller of the context exists");
    ctx->deterministic = enable != 0;
  });
}

int xc_profile(xc_ctx* ctx, int enable) {
  return guarded([&] {
    require(ctx, XC_ERR_ARG, "null context");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    ctx->profile = enable != 0;
  });
}

int xc_profile_collect(xc_ctx* ctx, double* stage_ms, int* nbuilds) {
  return guarded([&] {
    require(ctx && stage_ms, XC_ERR_ARG, "null argument");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipStreamSynchronize(ctx->stream));
    const size_t per = XC_NSTAGES + 1;
    for (int k = 0; k < XC_NSTAGES; ++k) stage_ms[k] = 0.0;
    const size_t nb = ctx->ev_used / per;
    for (size_t b = 0; b < nb; ++b)
      for (int k = 0; k < XC_NSTAGES; ++k) {
        float ms = 0.0f;
        HIPX(hipEventElapsedTime(&ms, ctx->ev_pool[b * per + k], ctx->ev_pool[b * per + k + 1]));
        stage_ms[k] += ms;
      }
    if (nbuilds) *nbuilds = (int)nb;
    ctx->ev_used = 0;
  });
}

int xc_device_alloc(xc_ctx* ctx, size_t bytes, void** dptr) {
  return guarded([&] {
    require(ctx && dptr, XC_ERR_ARG, "null argument");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    *dptr = ctx->alloc(bytes);
    if (*dptr) ctx->user_allocs[*dptr] = bytes;
  });
}

int xc_device_free(xc_ctx* ctx, void* dptr) {
  return guarded([&] {
    require(ctx, XC_ERR_ARG, "null context");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipStreamSynchronize(ctx->stream));
    if (dptr) {
      auto it = ctx->user_allocs.find(dptr);
      require(it != ctx->user_allocs.end(), XC_ERR_ARG, "xc_device_free: pointer not from xc_device_alloc");
      ctx->release(dptr, it->second);
      ctx->user_allocs.erase(it);
    }
  });
}

int xc_memcpy_h2d(xc_ctx* ctx, void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    require(ctx && dst && src, XC_ERR_ARG, "null argument");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    HIPX(hipStreamSynchronize(ctx->stream));
  });
}

int xc_device_copy(xc_ctx* ctx, void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    require(ctx && dst && src, XC_ERR_ARG, "null argument");
    require(bytes % 32 == 0, XC_ERR_ARG, "xc_device_copy: size must be a multiple of 32 bytes");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipSetDevice(ctx->device));
    launch_copy(ctx->stream, src, dst, (int64_t)(bytes / 32));
    HIPX(hipGetLastError());
    HIPX(hipStreamSynchronize(ctx->stream));
  });
}

// ---- serving ----------------------------------------------------------------
struct xc_server {
  struct Slot {
    hipStream_t stream = nullptr;
    Lanes lanes;
    hipEvent_t done = nullptr;
    double* h_P = nullptr;  // pinned staging of P, and of F with E behind it
    double* h_F = nullptr;
    size_t cap = 0;
    bool busy = false;
    int64_t ticket = -1;
    xc_bfogc* bf = nullptr;
    double* user_F = nullptr;
    double* user_E = nullptr;
  };
  xc_ctx* ctx = nullptr;
  std::vector<Slot> slots;
  bool graphs = true;
  int64_t next_ticket = 1;
  int64_t submitted = 0, graph_launches = 0;
};

namespace {

void server_slot_release(xc_server::Slot& sl) {
  if (sl.h_P) (void)hipHostFree(sl.h_P);
  if (sl.h_F) (void)hipHostFree(sl.h_F);
  sl.h_P = sl.h_F = nullptr;
  sl.cap = 0;
}

void server_finish(xc_server::Slot& sl, int n) {
  std::memcpy(sl.user_F, sl.h_F, sizeof(double) * (size_t)n * n);
  if (sl.user_E) *sl.user_E = sl.h_F[(size_t)n * n];
  sl.bf->in_flight = false;
  sl.busy = false;
  sl.bf = nullptr;
  sl.ticket = -1;
}

xc_server::Slot* server_slot_of(xc_server* srv, int64_t ticket) {
  for (auto& sl : srv->slots)
    if (sl.busy && sl.ticket == ticket) return &sl;
  return nullptr;
}

}  // namespace

int xc_server_create(xc_ctx* ctx, int nslots, int use_graphs, xc_server** out) {
  return guarded([&] {
    require(ctx && out, XC_ERR_ARG, "xc_server_create: null argument");
    require(nslots >= 1 && nslots <= 16, XC_ERR_ARG, "xc_server_create: slots must be in [1, 16]");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipSetDevice(ctx->device));
    auto* srv = new xc_server();
    srv->ctx = ctx;
    srv->graphs = use_graphs != 0;
    srv->slots.resize(nslots);
    try {
      for (auto& sl : srv->slots) {
        HIPX(hipStreamCreateWithFlags(&sl.stream, hipStreamNonBlocking));
        // concurrency comes from the slots: a slot's build stays on its own stream
        sl.lanes.create(sl.stream, false);
        HIPX(hipEventCreateWithFlags(&sl.done, hipEventDisableTiming));
      }
    } catch (...) {
      for (auto& sl : srv->slots) {
        sl.lanes.destroy();
        if (sl.stream) (void)hipStreamDestroy(sl.stream);
        if (sl.done) (void)hipEventDestroy(sl.done);
      }
      delete srv;
      throw;
    }
    ++ctx->live_handles;
    *out = srv;
  });
}

int xc_server_destroy(xc_server* srv) {
  return guarded([&] {
    if (!srv) return;
    std::lock_guard<std::recursive_mutex> lk(srv->ctx->mu);
    for (auto& sl : srv->slots) {
      (void)hipStreamSynchronize(sl.stream);
      if (sl.busy) {
        sl.bf->in_flight = false;
        sl.busy = false;
      }
      server_slot_release(sl);
      (void)hipEventDestroy(sl.done);
      sl.lanes.destroy();
      (void)hipStreamDestroy(sl.stream);
    }
    --srv->ctx->live_handles;
    delete srv;
  });
}

int xc_server_submit(xc_server* srv, xc_bfogc* bf, int functional, int precision, double thr, const double* P,
                     double* F, double* energy, int64_t* ticket) {
  return guarded([&] {
    require(srv && bf && P && F && ticket, XC_ERR_ARG, "xc_server_submit: null argument");
    require(bf->ctx == srv->ctx, XC_ERR_ARG, "xc_server_submit: controller of another context");
    xc_ctx* ctx = srv->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    *ticket = 0;
    if (bf->in_flight) throw XcError(XC_BUSY, "xc_server_submit: a build of this controller is in flight");
    xc_server::Slot* sl = nullptr;
    for (auto& c : srv->slots)
      if (!c.busy) {
        sl = &c;
        break;
      }
    if (!sl) throw XcError(XC_BUSY, "xc_server_submit: every slot is busy");
    const int n = bf->basis->nao;
    const size_t nn = (size_t)n * n;
    if (sl->cap < nn) {
      server_slot_release(*sl);
      HIPX(hipHostMalloc((void**)&sl->h_P, sizeof(double) * nn, hipHostMallocDefault));
      HIPX(hipHostMalloc((void**)&sl->h_F, sizeof(double) * (nn + 1), hipHostMallocDefault));
      sl->cap = nn;
    }
    std::memcpy(sl->h_P, P, sizeof(double) * nn);
    hipStream_t s = sl->stream;
    HIPX(hipMemcpyAsync(bf->d_P.p, sl->h_P, sizeof(double) * nn, hipMemcpyHostToDevice, s));
    if (srv->graphs) {
      const auto key = std::make_pair(functional + 16 * precision, thr);
      auto it = bf->graphs.find(key);
      if (it == bf->graphs.end()) {
        // capture one build on this controller's resident buffers (kernel nodes only, no memsets)
        hipGraph_t graph = nullptr;
        HIPX(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        try {
          enqueue_build(bf, functional, precision, thr, bf->d_P.p, bf->d_F.p, sl->lanes, bf->d_F.p + nn);
        } catch (...) {
          (void)hipStreamEndCapture(s, &graph);
          if (graph) (void)hipGraphDestroy(graph);
          throw;
        }
        HIPX(hipStreamEndCapture(s, &graph));
        hipGraphExec_t exec = nullptr;
        const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        HIPX(e);
        it = bf->graphs.emplace(key, exec).first;
      }
      HIPX(hipGraphLaunch(it->second, s));
      ++srv->graph_launches;
    } else {
      enqueue_build(bf, functional, precision, thr, bf->d_P.p, bf->d_F.p, sl->lanes, bf->d_F.p + nn);
    }
    HIPX(hipMemcpyAsync(sl->h_F, bf->d_F.p, sizeof(double) * (nn + 1), hipMemcpyDeviceToHost, s));
    HIPX(hipEventRecord(sl->done, s));
    sl->busy = true;
    sl->bf = bf;
    sl->user_F = F;
    sl->user_E = energy;
    sl->ticket = srv->next_ticket++;
    bf->in_flight = true;
    ++srv->submitted;
    *ticket = sl->ticket;
  });
}

int xc_server_poll(xc_server* srv, int64_t ticket, int* done) {
  return guarded([&] {
    require(srv && done, XC_ERR_ARG, "xc_server_poll: null argument");
    std::lock_guard<std::recursive_mutex> lk(srv->ctx->mu);
    xc_server::Slot* sl = server_slot_of(srv, ticket);
    require(sl != nullptr, XC_ERR_ARG, "xc_server_poll: unknown or finished ticket");
    const hipError_t q = hipEventQuery(sl->done);
    if (q == hipErrorNotReady) {
      *done = 0;
      return;
    }
    HIPX(q);
    server_finish(*sl, sl->bf->basis->nao);
    *done = 1;
  });
}

int xc_server_wait(xc_server* srv, int64_t ticket) {
  return guarded([&] {
    require(srv, XC_ERR_ARG, "xc_server_wait: null argument");
    std::lock_guard<std::recursive_mutex> lk(srv->ctx->mu);
    xc_server::Slot* sl = server_slot_of(srv, ticket);
    require(sl != nullptr, XC_ERR_ARG, "xc_server_wait: unknown or finished ticket");
    HIPX(hipEventSynchronize(sl->done));
    server_finish(*sl, sl->bf->basis->nao);
  });
}

int xc_server_stats(const xc_server* srv, int* busy_slots, int64_t* submitted, int64_t* graph_launches) {
  return guarded([&] {
    require(srv, XC_ERR_ARG, "xc_server_stats: null argument");
    std::lock_guard<std::recursive_mutex> lk(srv->ctx->mu);
    if (busy_slots) {
      int b = 0;
      for (const auto& sl : srv->slots) b += sl.busy ? 1 : 0;
      *busy_slots = b;
    }
    if (submitted) *submitted = srv->submitted;
    if (graph_launches) *graph_launches = srv->graph_launches;
  });
}

int xc_memcpy_d2h(xc_ctx* ctx, void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    require(ctx && dst && src, XC_ERR_ARG, "null argument");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    HIPX(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    HIPX(hipStreamSynchronize(ctx->stream));
  });
}

}  // extern "C"
