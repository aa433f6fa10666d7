// Solves in one launch while device allocations fail or the launch is refused,
// and large downloads while host allocations fail.  The driver's own hipMalloc stands before the runtime's and lets the k-th allocation of a call
// fail, for every k there is: the call has to end like one that had the memory
// (the sweeps, whose storage exists by then, need none of it), and so has the
// next call, whatever the failed one had allocated.  Nothing stays allocated
// that the sweeps do not read, nor anything once the handles are gone.
// Exit status 0 on success.
#include <dlfcn.h>

#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <random>
#include <thread>
#include <unordered_map>
#include <vector>

#include "lfgpu.h"

namespace {
long g_calls = 0, g_fail_at = -1;
size_t g_live = 0;  // bytes allocated
std::unordered_map<void *, size_t> g_size;
}  // namespace

extern "C" int hipMalloc(void **p, size_t bytes) {
  static auto *real = reinterpret_cast<int (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
  if (g_calls++ == g_fail_at) {
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  const int e = real(p, bytes);
  if (e == 0) g_live += g_size[*p] = bytes;
  return e;
}
struct Grid {
  uint32_t x, y, z;
};
int g_refuse = 0;  // what cooperative launches return
extern "C" int hipLaunchCooperativeKernel(const void *fn, Grid grid, Grid block, void **args,
                                          unsigned lds, void *stream) {
  static auto *real =
      reinterpret_cast<int (*)(const void *, Grid, Grid, void **, unsigned, void *)>(
          dlsym(RTLD_NEXT, "hipLaunchCooperativeKernel"));
  return g_refuse ? g_refuse : real(fn, grid, block, args, lds, stream);
}
long g_events = 0;
extern "C" int hipEventCreateWithFlags(void **ev, unsigned flags) {
  static auto *real = reinterpret_cast<int (*)(void **, unsigned)>(
      dlsym(RTLD_NEXT, "hipEventCreateWithFlags"));
  ++g_events;
  return real(ev, flags);
}
// this thread's host allocations in the library (the runtime's go as they
// are), of which the k-th fails
thread_local long g_news = 0, g_news_fail = -1;
static bool from_library(void *caller) {
  Dl_info info;
  return dladdr(caller, &info) != 0 && info.dli_fname && std::strstr(info.dli_fname, "liblfgpu.so");
}
void *operator new(size_t bytes) {
  void *p = nullptr;
  if (g_news_fail < 0 || !from_library(__builtin_return_address(0)) || g_news++ != g_news_fail)
    p = std::malloc(bytes);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" int hipFree(void *p) {
  static auto *real = reinterpret_cast<int (*)(void *)>(dlsym(RTLD_NEXT, "hipFree"));
  const auto it = g_size.find(p);
  if (it != g_size.end()) {
    g_live -= it->second;
    g_size.erase(it);
  }
  return real(p);
}

extern "C" int hipHostMalloc(void **p, size_t bytes, unsigned flags);
extern "C" int hipHostFree(void *p);
extern "C" int hipMemcpy(void *to, const void *from, size_t bytes, int kind);

namespace {
int fails = 0;
bool g_resident = true;  // solves run in one launch where the system fits
#define EXPECT(cond, ...)                 \
  do {                                    \
    if (!(cond)) {                        \
      std::printf("FAIL: " __VA_ARGS__);  \
      std::printf("\n");                  \
      ++fails;                            \
    }                                     \
  } while (0)
#define OK(call) EXPECT((call) == LFGPU_OK, "%s: %s", #call, lfgpu_last_error())

struct System {
  std::vector<int32_t> row, col, off{0};
  std::vector<double> val, rhs;
  int32_t n = 0;
};

// Adds a lattice Laplacian plus 0.01 (S x L vertices, every square cut along a
// diagonal, the other one in `turned` of ten squares of the first `lines`
// lines) as a problem.
void add_lattice(System &s, int S, int L, int turned, unsigned seed, int lines = 1 << 20) {
  std::mt19937 gen(seed);
  const int32_t base = s.n;
  std::vector<double> diag((size_t)S * L, 0.01);
  auto couple = [&](int a, int b) {
    const double w = 0.5 + gen() % 1000 * 0.002;
    s.row.insert(s.row.end(), {base + a, base + b});
    s.col.insert(s.col.end(), {base + b, base + a});
    s.val.insert(s.val.end(), {-w, -w});
    diag[a] += w;
    diag[b] += w;
  };
  for (int y = 0; y < L; ++y)
    for (int x = 0; x < S; ++x) {
      const int i = y * S + x;
      if (x + 1 < S) couple(i, i + 1);
      if (y + 1 < L) couple(i, i + S);
      if (x + 1 < S && y + 1 < L) {
        if (y < lines && (int)(gen() % 10) < turned) couple(i + 1, i + S);
        else couple(i, i + S + 1);
      }
    }
  for (int i = 0; i < S * L; ++i) {
    s.row.push_back(base + i);
    s.col.push_back(base + i);
    s.val.push_back(diag[i]);
    s.rhs.push_back(gen() % 1000 * 0.002 - 1.0);
  }
  s.n += S * L;
  s.off.push_back(s.n);
}

double norm(const std::vector<double> &a, const std::vector<double> *less = nullptr) {
  double s = 0.0;
  for (size_t i = 0; i < a.size(); ++i) {
    const double v = a[i] - (less ? (*less)[i] : 0.0);
    s += v * v;
  }
  return std::sqrt(s);
}

void run(const char *name, lfgpu_ctx *ctx, const System &s, int mode, bool batch) {
  std::vector<double> want((size_t)s.n), got((size_t)s.n);
  lfgpu_pcg_opts opts{};
  opts.rtol = 1e-11;
  opts.maxit = 20000;
  opts.mode = mode;
  // two solutions of residuals below rtol ||b||, no eigenvalue below 0.01, and
  // a tenth for the recurrence residual's distance from the true one
  const double bound = 2.2 * opts.rtol * norm(s.rhs) / 0.01;
  for (long k = 0;; ++k) {
    const size_t before = g_live;
    lfgpu_csr *A = nullptr;
    lfgpu_vec *b = nullptr, *x = nullptr;
    lfgpu_batch *bt = nullptr;
    OK(lfgpu_coo_to_csr(ctx, (int64_t)s.val.size(), s.row.data(), s.col.data(), s.val.data(), s.n,
                        s.n, &A));
    OK(lfgpu_vec_create(ctx, s.n, s.rhs.data(), &b));
    OK(lfgpu_vec_create(ctx, s.n, nullptr, &x));
    if (batch) OK(lfgpu_batch_create(ctx, A, (int)s.off.size() - 1, s.off.data(), &bt));
    lfgpu_pcg_info info{};
    auto solve = [&](int graph, std::vector<double> &to) {
      OK(lfgpu_vec_fill(x, 0.0));
      opts.graph = graph;
      if (batch) OK(lfgpu_batch_pcg(ctx, bt, b, x, &opts, nullptr, &info));
      else OK(lfgpu_pcg(ctx, A, b, x, &opts, &info));
      EXPECT(info.converged, "%s, allocation %ld: not converged", name, k);
      OK(lfgpu_vec_download(x, to.data(), s.n));
    };
    solve(1, want);
    const size_t swept = g_live;
    g_calls = 0;
    g_fail_at = k;
    solve(0, got);
    const bool failed = g_calls > k;
    g_fail_at = -1;
    EXPECT(norm(got, &want) <= bound, "%s, allocation %ld: %g off", name, k, norm(got, &want));
    EXPECT(failed || info.syncs == 1 || !g_resident, "%s: not in one launch", name);
    EXPECT(!failed || g_live == swept, "%s, allocation %ld: %ld bytes kept", name, k,
           (long)(g_live - swept));
    solve(0, got);
    EXPECT(norm(got, &want) <= bound, "%s, after allocation %ld: %g off", name, k,
           norm(got, &want));
    OK(lfgpu_batch_destroy(bt));
    OK(lfgpu_vec_destroy(x));
    OK(lfgpu_vec_destroy(b));
    OK(lfgpu_csr_destroy(A));
    EXPECT(g_live == before, "%s, allocation %ld: %ld bytes lost", name, k,
           (long)(g_live - before));
    if (!failed) {
      std::printf("%s: %ld allocations\n", name, k);
      std::fflush(stdout);
      return;
    }
  }
}

// The device's cooperative queue may belong to another process: its launches
// then fail with "the operation cannot be performed in the present state".
void refused(const char *name, lfgpu_ctx *ctx, const System &s, int mode, bool batch) {
  std::vector<double> want((size_t)s.n), got((size_t)s.n);
  lfgpu_csr *A = nullptr;
  lfgpu_vec *b = nullptr, *x = nullptr;
  lfgpu_batch *bt = nullptr;
  OK(lfgpu_coo_to_csr(ctx, (int64_t)s.val.size(), s.row.data(), s.col.data(), s.val.data(), s.n,
                      s.n, &A));
  OK(lfgpu_vec_create(ctx, s.n, s.rhs.data(), &b));
  OK(lfgpu_vec_create(ctx, s.n, nullptr, &x));
  if (batch) OK(lfgpu_batch_create(ctx, A, (int)s.off.size() - 1, s.off.data(), &bt));
  lfgpu_pcg_opts opts{};
  opts.rtol = 1e-11;
  opts.maxit = 20000;
  opts.mode = mode;
  const double bound = 2.2 * opts.rtol * norm(s.rhs) / 0.01;  // as in run()
  for (int turn = 0; turn < 4; ++turn) {  // the sweeps, refused twice, then not
    lfgpu_pcg_info info{};
    opts.graph = turn == 0 ? 1 : 0;
    g_refuse = turn < 3 ? 401 : 0;
    if (turn == 3) std::this_thread::sleep_for(std::chrono::milliseconds(600));
    OK(lfgpu_vec_fill(x, 0.0));
    if (batch) OK(lfgpu_batch_pcg(ctx, bt, b, x, &opts, nullptr, &info));
    else OK(lfgpu_pcg(ctx, A, b, x, &opts, &info));
    g_refuse = 0;
    EXPECT(info.converged, "%s, turn %d: not converged", name, turn);
    EXPECT(turn < 3 || info.syncs == 1 || !g_resident, "%s: not in one launch", name);
    OK(lfgpu_vec_download(x, got.data(), s.n));
    if (turn == 0) want = got;
    EXPECT(norm(got, &want) <= bound, "%s, turn %d: %g off", name, turn, norm(got, &want));
  }
  OK(lfgpu_batch_destroy(bt));
  OK(lfgpu_vec_destroy(x));
  OK(lfgpu_vec_destroy(b));
  OK(lfgpu_csr_destroy(A));
}

// Whether solves run in one launch here: another process may hold the queue.
bool resident(lfgpu_ctx *ctx, const System &s) {
  lfgpu_csr *A = nullptr;
  lfgpu_vec *b = nullptr, *x = nullptr;
  OK(lfgpu_coo_to_csr(ctx, (int64_t)s.val.size(), s.row.data(), s.col.data(), s.val.data(), s.n,
                      s.n, &A));
  OK(lfgpu_vec_create(ctx, s.n, s.rhs.data(), &b));
  OK(lfgpu_vec_create(ctx, s.n, nullptr, &x));
  lfgpu_pcg_opts opts{};
  opts.rtol = 1e-11;
  opts.maxit = 20000;
  lfgpu_pcg_info info{};
  OK(lfgpu_pcg(ctx, A, b, x, &opts, &info));
  OK(lfgpu_vec_destroy(x));
  OK(lfgpu_vec_destroy(b));
  OK(lfgpu_csr_destroy(A));
  return info.syncs == 1;
}

// A download through the staging ring creates no event (the context's device
// need not be current), and any of its host allocations may fail: the list of
// chunks, and what a copying thread takes to start.
void download(lfgpu_ctx *ctx) {
  const int64_t n = 3 << 20;
  std::vector<double> in((size_t)n), out((size_t)n);
  for (int64_t i = 0; i < n; ++i) in[i] = 1.0 / (1.0 + (double)i);
  lfgpu_vec *v = nullptr;
  OK(lfgpu_vec_create(ctx, n, in.data(), &v));
  const long events = g_events;
  OK(lfgpu_vec_download(v, out.data(), n));
  EXPECT(out == in, "download");
  EXPECT(g_events == events, "the download creates %ld events", g_events - events);
  long k = 0;
  for (bool failed = true; failed; ++k) {
    std::fill(out.begin(), out.end(), 0.0);
    g_news = 0;
    g_news_fail = k;
    const int rc = lfgpu_vec_download(v, out.data(), n);
    failed = g_news > k;
    g_news_fail = -1;
    EXPECT(rc == LFGPU_OK && out == in, "download, host allocation %ld", k);
  }
  std::printf("download: %ld host allocations\n", k - 1);
  OK(lfgpu_vec_destroy(v));
}

// The arrays of a matrix may go to different kinds of memory.
void scattered(lfgpu_ctx *ctx) {
  System s;
  add_lattice(s, 500, 400, 0, 1);
  lfgpu_csr *A = nullptr;
  OK(lfgpu_coo_to_csr(ctx, (int64_t)s.val.size(), s.row.data(), s.col.data(), s.val.data(), s.n,
                      s.n, &A));
  int64_t nnz = 0;
  OK(lfgpu_csr_info(A, nullptr, nullptr, &nnz));
  std::vector<int32_t> rp((size_t)s.n + 1), col((size_t)nnz), got((size_t)nnz);
  std::vector<double> val((size_t)nnz), val2((size_t)nnz);
  OK(lfgpu_csr_download(A, rp.data(), col.data(), val.data()));
  void *dev = nullptr, *pinned = nullptr;
  EXPECT(hipMalloc(&dev, 4 * (size_t)nnz) == 0 && hipHostMalloc(&pinned, 4 * (size_t)nnz, 0) == 0,
         "memory");
  for (void *to : {dev, pinned}) {
    OK(lfgpu_csr_download(A, rp.data(), static_cast<int32_t *>(to), val2.data()));
    EXPECT(hipMemcpy(got.data(), to, 4 * (size_t)nnz, 4) == 0, "hipMemcpy");
    EXPECT(got == col && val2 == val, "download to scattered arrays");
    std::fill(got.begin(), got.end(), 0);
    std::fill(val2.begin(), val2.end(), 0.0);
  }
  hipHostFree(pinned);
  hipFree(dev);
  OK(lfgpu_csr_destroy(A));
}

// Asking for the storage allocates nothing (the calling thread's device need
// not be the matrix's), also where the answer takes the symmetry test first.
void storage(lfgpu_ctx *ctx, const System &s) {
  lfgpu_csr *A = nullptr;
  lfgpu_vec *b = nullptr, *x = nullptr;
  OK(lfgpu_coo_to_csr(ctx, (int64_t)s.val.size(), s.row.data(), s.col.data(), s.val.data(), s.n,
                      s.n, &A));
  OK(lfgpu_vec_create(ctx, s.n, s.rhs.data(), &b));
  OK(lfgpu_vec_create(ctx, s.n, nullptr, &x));
  OK(lfgpu_spmv(ctx, A, b, x));
  const long calls = g_calls;
  int kind = -1, ndiag = 0, sym = 0;
  OK(lfgpu_solver_storage(A, &kind, &ndiag, &sym));
  EXPECT(kind == LFGPU_STORAGE_DIA && ndiag == 6 && sym == 1, "storage %d, %d diagonals, %d", kind,
         ndiag, sym);
  EXPECT(g_calls == calls, "lfgpu_solver_storage allocates");
  OK(lfgpu_vec_destroy(x));
  OK(lfgpu_vec_destroy(b));
  OK(lfgpu_csr_destroy(A));
}
}  // namespace

int main() {
  lfgpu_ctx *ctx = nullptr;
  OK(lfgpu_ctx_create(0, &ctx));
  if (!ctx) return 1;
  System lattice, ell, equal, bands, both, mixed;
  add_lattice(lattice, 90, 70, 0, 1);
  add_lattice(ell, 90, 70, 5, 2);
  for (int k = 0; k < 4; ++k) add_lattice(equal, 24, 30, 0, 3 + k);
  for (int k = 0; k < 4; ++k) add_lattice(bands, 24 + k, 30, 0, 7 + k);
  for (int k = 0; k < 6; ++k) add_lattice(both, 40 + k, 50, k % 2 ? 5 : 0, 11 + k);
  // (what the middle of the turned ones shows does not cover them: no diagonals
  // for the sweeps, which run on sliced ELL, but for the others' tiles)
  for (int k = 0; k < 6; ++k) add_lattice(mixed, 70 + k, 50, k % 2 ? 5 : 0, 21 + k, 10);
  g_resident = resident(ctx, lattice);
  std::printf("solves run in one launch: %s\n", g_resident ? "yes" : "no");
  for (int mode : {LFGPU_PCG_FP64, LFGPU_PCG_MIXED, LFGPU_PCG_MIXED_MATRIX}) {
    run("lattice", ctx, lattice, mode, false);
    run("sliced ELL", ctx, ell, mode, false);
    run("batch of equal lattices", ctx, equal, mode, true);
    run("batch of lattices", ctx, bands, mode, true);
    run("batch of both", ctx, both, mode, true);
    run("batch of both, swept on ELL", ctx, mixed, mode, true);
    refused("lattice", ctx, lattice, mode, false);
    refused("sliced ELL", ctx, ell, mode, false);
    refused("batch of both", ctx, both, mode, true);
  }
  storage(ctx, lattice);
  download(ctx);
  scattered(ctx);
  OK(lfgpu_ctx_destroy(ctx));
  if (fails) return 1;
  std::printf("OK\n");
  return 0;
}
