// The runtime of hip/hip_runtime.h: device memory with guard pages, and kernels
// run one workgroup at a time, every work-item a coroutine that is switched
// where the work-items of a wavefront or workgroup meet.
//
// Checked, with a message and exit(3): a barrier that some work-items of the
// workgroup have left behind, lanes of one wavefront that meet in different
// places.  Reads and writes past an allocation fault (SIGSEGV), fixed arrays are
// compiled with bounds checks (SIGILL).  A launch with more dynamic LDS than
// 64 KiB, or than hipFuncSetAttribute allowed it, fails.
//
// IMSRG_EMU_CHECK: launches are checked, kernels not run.
// IMSRG_EMU_SPLIT=w: wavefront w of workgroup 1 of every launch starts before
// workgroup 0, which then runs whole before the rest of workgroup 1 (LDS kept
// apart), as two workgroups on two compute units may.
#include <link.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "hip/hip_runtime.h"

namespace imsrg {  // dynamic LDS of the kernels in this namespace
thread_local double lds[20480], pan_lds[20480], S6[20480], WS[20480];
}

namespace emu {
Index tid, bid, bdim, gdim;
namespace {
std::mutex mu;
constexpr size_t kStack = 128 << 10, kMaxItems = 1024;
struct Item {
  void *sp = nullptr;
  Index id{};
  bool live = false;
  const void *at = nullptr;  // where it waits (return address), null: running
  bool block = false;        // of the workgroup (else of its wavefront)
  unsigned phase = 0;
};
Item items[kMaxItems];
int nitem = 0, cur = -1;
char *stacks = nullptr;
void *main_sp = nullptr;
const std::function<void()> *body = nullptr;
alignas(16) double xchg[kMaxItems / 64][2][64 * 16];

extern "C" void emu_switch(void **save, void *to);
asm(R"(
.text
.globl emu_switch
emu_switch:
  pushq %rbp
  pushq %rbx
  pushq %r12
  pushq %r13
  pushq %r14
  pushq %r15
  movq %rsp, (%rdi)
  movq %rsi, %rsp
  popq %r15
  popq %r14
  popq %r13
  popq %r12
  popq %rbx
  popq %rbp
  ret
)");
[[noreturn]] void die(const char *what) {
  std::fprintf(stderr, "emulated kernel: %s (workgroup %u,%u work-item %u)\n", what, bid.x, bid.y, tid.x);
  std::fflush(stderr);
  std::_Exit(3);
}
void entry() {
  (*body)();
  items[cur].live = false;
  emu_switch(&items[cur].sp, main_sp);
}
void resume(int i) {
  cur = i;
  tid = items[i].id;
  emu_switch(&main_sp, items[i].sp);
}
void wait(const void *at, bool block) {
  Item &it = items[cur];
  it.at = at;
  it.block = block;
  emu_switch(&it.sp, main_sp);
}
void start(int i) {
  Item &it = items[i];
  it.live = true;
  it.at = nullptr;
  it.phase = 0;
  it.id = Index{(unsigned)i, 0, 0};
  void **s = (void **)(stacks + (i + 1) * kStack - 64);
  *--s = nullptr;  // alignment: the entry sees a stack as after a call
  *--s = (void *)entry;
  for (int k = 0; k < 6; k++) *--s = nullptr;
  it.sp = s;
}
// runs the items of [a, b) that can go on until they wait or end
bool step(int a, int b) {
  bool any = false;
  for (int i = a; i < b; i++)
    if (items[i].live && !items[i].at) {
      resume(i);
      any = true;
    }
  return any;
}
// releases wavefronts and the workgroup where everyone has arrived
void release() {
  for (int w = 0; w < nitem; w += 64) {
    const void *at = nullptr;
    bool all = true, some = false;
    for (int i = w; i < std::min(w + 64, nitem); i++)
      if (items[i].live) {
        some = true;
        if (!items[i].at || items[i].block) all = false;
        else if (!at) at = items[i].at;
      }
    if (!some || !all) continue;
    for (int i = w; i < std::min(w + 64, nitem); i++)
      if (items[i].live) {
        if (items[i].at != at) bid.z = 0, tid = items[i].id, die("lanes of a wavefront meet in different places");
        items[i].at = nullptr;
      }
  }
  bool all = nitem > 0, gone = false, some = false;
  for (int i = 0; i < nitem; i++) {
    if (!items[i].live) gone = true;
    else some = true, all = all && items[i].at && items[i].block;
  }
  if (!some || !all) return;
  if (gone) die("a barrier that some work-items of the workgroup do not reach");
  for (int i = 0; i < nitem; i++) items[i].at = nullptr;
}
bool done() {
  for (int i = 0; i < nitem; i++)
    if (items[i].live) return false;
  return true;
}
void finish() {
  while (!done()) {
    release();
    if (!step(0, nitem) && !done()) {
      for (int i = 0; i < nitem; i++)
        if (items[i].live) tid = items[i].id;
      die("work-items wait for each other");
    }
  }
}
// LDS: this module's thread-local storage
struct Tls {
  char *p = nullptr;
  size_t n = 0;
};
int find_tls(dl_phdr_info *info, size_t, void *out) {
  const char *me = (const char *)&imsrg::lds;
  if (!info->dlpi_tls_data) return 0;
  for (int k = 0; k < info->dlpi_phnum; k++)
    if (info->dlpi_phdr[k].p_type == PT_TLS) {
      char *p = (char *)info->dlpi_tls_data;
      const size_t n = info->dlpi_phdr[k].p_memsz;
      if (me >= p && me < p + n) *(Tls *)out = Tls{p, n};
    }
  return 0;
}
int split_wave() {
  const char *s = std::getenv("IMSRG_EMU_SPLIT");
  return s ? std::atoi(s) : -1;
}
std::map<const void *, int> lds_limit;
hipError_t last = hipSuccess;
long long clock_blocks = 0;
}  // namespace

__attribute__((noinline)) void barrier() { wait(__builtin_return_address(0), true); }
__attribute__((noinline)) const double *exchange(const void *mine, size_t n) {
  Item &it = items[cur];
  double *buf = xchg[cur >> 6][it.phase ^= 1];
  std::memcpy(buf + 16 * (cur & 63), mine, n);
  wait((const void *)n, false);  // (callers are inlined: the size stands for the place)
  return buf;
}

void run(const void *kernel, dim3 g, dim3 b, size_t lds, const std::function<void()> &f) {
  std::lock_guard<std::mutex> lock(mu);
  const int limit = lds_limit.count(kernel) ? std::max(lds_limit[kernel], 65536) : 65536;
  if ((int)lds > limit || g.x == 0 || g.y == 0 || g.z == 0 || b.x * b.y * b.z > kMaxItems) {
    std::fprintf(stderr, "emulated launch refused: grid %u,%u,%u block %u LDS %zu (limit %d)\n", g.x, g.y, g.z, b.x, lds,
                 limit);
    last = hipErrorInvalidValue;
    return;
  }
  if (std::getenv("IMSRG_EMU_CHECK")) return;
  if (!stacks) stacks = (char *)mmap(nullptr, kStack * kMaxItems, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  body = &f;
  bdim = Index{b.x, b.y, b.z};
  gdim = Index{g.x, g.y, g.z};
  nitem = (int)b.x;
  clock_blocks += (long long)g.x * g.y * g.z;
  const int sw = split_wave();
  Tls tls;
  dl_iterate_phdr(find_tls, &tls);
  // (the host's own thread-local variables are there too)
  const std::vector<char> host(tls.p, tls.p + tls.n);
  auto fresh = [&] {
    std::memset(tls.p, 0x7f, tls.n);  // what an LDS word holds before it is written: a large number
    for (int i = 0; i < nitem; i++) start(i);
  };
  for (unsigned z = 0; z < g.z; z++)
    for (unsigned y = 0; y < g.y; y++) {
      unsigned x = 0;
      if (sw >= 0 && g.x > 1 && 64 * sw < nitem) {
        // wavefront sw of workgroup 1 up to where it first waits
        bid = Index{1, y, z};
        fresh();
        step(64 * sw, std::min(64 * sw + 64, nitem));
        std::vector<char> keep(tls.p, tls.p + tls.n), st(stacks, stacks + kStack * nitem);
        std::vector<Item> it(items, items + nitem);
        std::vector<double> xc((double *)xchg, (double *)xchg + sizeof(xchg) / 8);
        bid.x = 0;
        fresh();
        finish();
        std::memcpy(tls.p, keep.data(), tls.n);
        std::memcpy(stacks, st.data(), st.size());
        std::copy(it.begin(), it.end(), items);
        std::memcpy(xchg, xc.data(), sizeof(xchg));
        bid.x = 1;
        finish();
        x = 2;
      }
      for (; x < g.x; x++) {
        bid = Index{x, y, z};
        fresh();
        finish();
      }
    }
  std::memcpy(tls.p, host.data(), tls.n);
}
}  // namespace emu

unsigned long long __ballot(bool p) {
  const double v = p ? 1.0 : 0.0;
  const double *all = emu::exchange(&v, sizeof(double));
  unsigned long long m = 0;
  for (int k = 0; k < 64; k++) m |= (unsigned long long)(all[16 * k] != 0.0) << k;
  return m;
}
emu_double4 emu_mfma_f64(double a, double b, emu_double4 c) {
  const double ab[2] = {a, b};
  const double *all = emu::exchange(ab, sizeof(ab));
  const int l = emu::lane();
  for (int v = 0; v < 4; v++) {
    const int row = (l >> 4) + 4 * v, col = l & 15;
    for (int k = 0; k < 4; k++) c[v] = std::fma(all[16 * (16 * k + row)], all[16 * (16 * k + col) + 1], c[v]);
  }
  return c;
}

// ---------------------------------------------------------------- runtime
struct emu_event {
  long long t = 0;
};
namespace {
struct Alloc {
  void *map;
  size_t len, n;
  int host;
};
std::mutex amu;
std::map<void *, Alloc> allocs;
size_t in_use = 0, limit = SIZE_MAX;
}  // namespace
extern "C" {
void emu_set_limit(size_t n) { limit = n; }  // device bytes in use at most
size_t emu_in_use() { return in_use; }
hipError_t emu_malloc(void **p, size_t n, int host) {
  std::lock_guard<std::mutex> lock(amu);
  if (!host && (n > limit || in_use + n > limit)) return emu::last = hipErrorOutOfMemory;
  const size_t page = 4096, body = (n + page - 1) / page * page, len = body + 2 * page;
  char *m = (char *)mmap(nullptr, len, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (m == MAP_FAILED) return emu::last = hipErrorOutOfMemory;
  mprotect(m, page, PROT_NONE);
  mprotect(m + page + body, page, PROT_NONE);
  *p = m + page + body - (n + 15) / 16 * 16;  // ends at the guard page, 16-byte aligned
  std::memset(*p, 0xff, n);
  allocs[*p] = Alloc{m, len, n, host};
  if (!host) in_use += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  std::lock_guard<std::mutex> lock(amu);
  auto it = allocs.find(p);
  if (it == allocs.end()) std::fprintf(stderr, "emulated free of an unknown address\n"), std::_Exit(3);
  if (!it->second.host) in_use -= it->second.n;
  munmap(it->second.map, it->second.len);
  allocs.erase(it);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memmove(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipGetLastError() {
  const hipError_t e = emu::last;
  emu::last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "emulated error"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 163840, hipSuccess; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v) { return emu::lds_limit[f] = v, hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return *s = (hipStream_t) new int(0), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return delete (int *)s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = new emu_event, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
// time runs in workgroups launched
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e->t = emu::clock_blocks, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { return *ms = (float)(b->t - a->t), hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, void *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
