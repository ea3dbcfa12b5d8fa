// The parts of the CPU's HIP runtime with state: guarded memory and launches.
#include <hip/hip_runtime.h>
#include <mutex>
#include <sys/mman.h>
#include <ucontext.h>
#include <unordered_map>
#include <vector>

cpu_index threadIdx, blockIdx, blockDim, gridDim;

static std::mutex g_mu;
static std::unordered_map<void *, std::pair<void *, size_t>> g_maps;
static constexpr size_t PAGE = 4096;

hipError_t cpu_malloc(void **p, size_t n)
{
  const size_t body = (n + PAGE - 1) / PAGE * PAGE, all = body + 2 * PAGE;
  char *m = (char *)mmap(nullptr, all, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == (char *)MAP_FAILED) return hipErrorCpu;
  mprotect(m, PAGE, PROT_NONE);
  mprotect(m + PAGE + body, PAGE, PROT_NONE);
  *p = m + PAGE + (body - n) / 16 * 16;
  memset(m + PAGE, 0xC3, body);  // (callers clear what they rely on)
  std::lock_guard<std::mutex> lk(g_mu);
  g_maps[*p] = {m, all};
  return hipSuccess;
}

hipError_t hipFree(void *p)
{
  if (!p) return hipSuccess;
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_maps.find(p);
  if (it == g_maps.end()) return hipErrorCpu;
  munmap(it->second.first, it->second.second);
  g_maps.erase(it);
  return hipSuccess;
}

namespace {
struct NeedsThreads {};
struct Fiber { ucontext_t ctx; bool done; std::vector<char> stack; };
std::vector<Fiber> g_fibers;
ucontext_t g_main;
bool g_threads = false;  // the block's threads have contexts of their own
int g_current = 0;
void (*g_run)(void *);
void *g_arg;

void set_thread(unsigned t, dim3 b) { threadIdx = {t % b.x, t / b.x % b.y, t / (b.x * b.y)}; }

void entry()
{
  g_run(g_arg);
  g_fibers[g_current].done = true;
  swapcontext(&g_fibers[g_current].ctx, &g_main);
}

// Every thread to its next barrier, in turn, until all have ended.
void run_threads(unsigned n, dim3 b, bool reverse)
{
  if (g_fibers.size() < n) g_fibers.resize(n);
  for (unsigned t = 0; t < n; ++t) {
    Fiber &f = g_fibers[t];
    if (f.stack.empty()) f.stack.resize(1 << 16);
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack.data();
    f.ctx.uc_stack.ss_size = f.stack.size();
    f.ctx.uc_link = nullptr;
    f.done = false;
    makecontext(&f.ctx, entry, 0);
  }
  g_threads = true;
  for (unsigned left = n; left;) {
    left = 0;
    for (unsigned q = 0; q < n; ++q) {
      const unsigned t = reverse ? n - 1 - q : q;
      if (g_fibers[t].done) continue;
      g_current = (int)t;
      set_thread(t, b);
      swapcontext(&g_main, &g_fibers[t].ctx);
      left += !g_fibers[t].done;
    }
  }
  g_threads = false;
}
}  // namespace

void __syncthreads()
{
  if (!g_threads) throw NeedsThreads();
  swapcontext(&g_fibers[g_current].ctx, &g_main);
}

void cpu_launch(dim3 g, dim3 b, void (*run)(void *), void *arg)
{
  static std::mutex launch;
  std::lock_guard<std::mutex> lk(launch);
  const char *o = getenv("CPU_HIP_ORDER");
  const bool reverse = o && strcmp(o, "reverse") == 0;
  g_run = run;
  g_arg = arg;
  blockDim = {b.x, b.y, b.z};
  gridDim = {g.x, g.y, g.z};
  const unsigned n = b.x * b.y * b.z;
  const unsigned long long nb = (unsigned long long)g.x * g.y * g.z;
  if (!nb || !n || n > 1024) {
    fprintf(stderr, "launch of %llu blocks of %u threads\n", nb, n);
    abort();
  }
  for (unsigned long long q = 0; q < nb; ++q) {
    const unsigned long long i = reverse ? nb - 1 - q : q;
    blockIdx = {(unsigned)(i % g.x), (unsigned)(i / g.x % g.y), (unsigned)(i / ((unsigned long long)g.x * g.y))};
    try {
      for (unsigned t = 0; t < n; ++t) {
        set_thread(reverse ? n - 1 - t : t, b);
        run(arg);
      }
    } catch (const NeedsThreads &) {
      run_threads(n, b, reverse);
    }
  }
}
