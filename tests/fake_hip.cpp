// Stand-in for the HIP runtime, for tests of the library's host code without a
// device: memory is host memory, streams and events are tokens, kernels do
// nothing, except that k_screen marks every shell on every tile.  Freed memory
// is kept mapped and remembered, so that a table which still names it can be
// found: fake_stale() counts the words of the launched plans' tables that point
// into freed memory.  fake_fail_in(n): the n-th allocation from now on fails.
// fake_engine() counts the copies of pinned memory large enough for the runtime
// to give them to a copy engine.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

namespace {
typedef int err_t;  // hipError_t
constexpr err_t kOk = 0, kInvalid = 1, kNoMem = 2;
std::map<uintptr_t, size_t> live, dead;
std::map<const void *, std::string> names;
std::set<uintptr_t> captured, pinned;
long fail_in = 0, stale = 0, engine = 0;
bool capturing = false;
err_t last = kOk;
int token;

uintptr_t owner(const std::map<uintptr_t, size_t> &m, uintptr_t a) {
  auto it = m.upper_bound(a);
  if (it == m.begin()) return 0;
  --it;
  return a < it->first + it->second ? it->first : 0;
}
void check(uintptr_t block) {
  if (!live.count(block)) {  // the table itself is gone
    ++stale;
    return;
  }
  const uintptr_t *w = (const uintptr_t *)block;
  for (size_t i = 0; i < live[block] / 8; ++i) stale += owner(dead, w[i]) != 0;
}
err_t set(err_t e) {
  if (e) last = e;
  return e;
}
}  // namespace

extern "C" {
long fake_stale() { return stale; }
long fake_engine() { return engine; }
long fake_live() { return (long)live.size(); }
void fake_fail_in(long n) { fail_in = n; }

void **__hipRegisterFatBinary(const void *) { return (void **)&token; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
struct dim3_ {
  uint32_t x, y, z;
};
static dim3_ cfg_g, cfg_b;
err_t __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t, void *) {
  cfg_g = g;
  cfg_b = b;
  return kOk;
}
err_t __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *s, void **st) {
  *g = cfg_g;
  *b = cfg_b;
  *s = 0;
  *st = nullptr;
  return kOk;
}
err_t hipLaunchKernel(const void *f, dim3_, dim3_, void **args, size_t, void *) {
  const std::string &n = names[f];
  if (n.find("k_screen") != std::string::npos) {
    const long nt = *(long *)args[0];
    const int ns = *(int *)args[6], n8 = *(int *)args[8], nw = (n8 + 31) / 32, nws = (ns + 31) / 32;
    int *nb = *(int **)args[9];
    uint32_t *sig = *(uint32_t **)args[10], *sm = *(uint32_t **)args[11];
    for (long t = 0; t < nt; ++t) {
      nb[t] = 8 * n8;
      for (int q = 0; q < 4; ++q)
        for (int r = 0; r < n8; ++r) sig[(4 * t + q) * nw + r / 32] |= 1u << (r % 32);
      for (int s = 0; s < ns; ++s) sm[t * nws + s / 32] |= 1u << (s % 32);
    }
  }
  if (n.find("k_functional") != std::string::npos || n.find("k_bracket_sum") != std::string::npos) {
    const uintptr_t block = owner(live, *(uintptr_t *)args[0]);  // the units' table
    if (capturing) captured.insert(block);
    check(block);
  }
  return kOk;
}

err_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (fail_in > 0 && --fail_in == 0) return set(kNoMem);
  *p = calloc(1, n ? n : 1);
  live[(uintptr_t)*p] = n;
  return kOk;
}
err_t hipFree(void *p) {
  if (!p) return kOk;
  auto it = live.find((uintptr_t)p);
  if (it == live.end()) return set(kInvalid);
  dead[it->first] = it->second;
  live.erase(it);
  return kOk;
}
err_t hipHostMalloc(void **p, size_t n, unsigned) {
  const err_t e = hipMalloc(p, n);
  if (e == kOk) pinned.insert((uintptr_t)*p);
  return e;
}
err_t hipHostFree(void *p) { return hipFree(p); }
err_t hipMemcpy(void *d, const void *s, size_t n, int) {
  if (n && (!d || !s)) return set(kInvalid);
  memcpy(d, s, n);
  return kOk;
}
err_t hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *) {
  for (const void *p : {(const void *)d, s}) engine += n > 16384 && pinned.count(owner(live, (uintptr_t)p));
  return hipMemcpy(d, s, n, k);
}
err_t hipMemset(void *d, int v, size_t n) {
  if (n && !d) return set(kInvalid);
  if (v || owner(live, (uintptr_t)d) != (uintptr_t)d) memset(d, v, n);
  return kOk;  // a whole fresh block is zero already
}
err_t hipMemsetAsync(void *d, int v, size_t n, void *) { return hipMemset(d, v, n); }
err_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = 288ull << 30;
  return kOk;
}
err_t hipDeviceGetAttribute(int *v, int, int) {
  *v = 100000;
  return kOk;
}
err_t hipGetDevice(int *d) {
  *d = 0;
  return kOk;
}
err_t hipGetLastError() {
  const err_t e = last;
  last = kOk;
  return e;
}
const char *hipGetErrorString(err_t) { return "stand-in error"; }
err_t hipGetSymbolAddress(void **, const void *) { return kInvalid; }
static err_t tok(void **p) {
  *p = &token;
  return kOk;
}
err_t hipStreamCreateWithFlags(void **s, unsigned) { return tok(s); }
err_t hipStreamDestroy(void *) { return kOk; }
err_t hipStreamSynchronize(void *) { return kOk; }
err_t hipStreamWaitEvent(void *, void *, unsigned) { return kOk; }
err_t hipEventCreate(void **e) { return tok(e); }
err_t hipEventCreateWithFlags(void **e, unsigned) { return tok(e); }
err_t hipEventDestroy(void *) { return kOk; }
err_t hipEventRecord(void *, void *) { return kOk; }
err_t hipEventSynchronize(void *) { return kOk; }
err_t hipEventElapsedTime(float *t, void *, void *) {
  *t = 0.0f;
  return kOk;
}
err_t hipStreamBeginCapture(void *, int) {
  captured.clear();
  capturing = true;
  return kOk;
}
err_t hipStreamEndCapture(void *, void **g) {
  capturing = false;
  return tok(g);
}
err_t hipGraphInstantiate(void **x, void *, void **, char *, size_t) { return tok(x); }
err_t hipGraphLaunch(void *, void *) {
  for (uintptr_t b : captured) check(b);
  return kOk;
}
err_t hipGraphExecDestroy(void *) { return kOk; }
err_t hipGraphDestroy(void *) { return kOk; }
}
