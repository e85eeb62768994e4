// Memory rules of the served form (pk_server.cpp), on the host: the device is
// a number of bytes, and each step of a job takes as many of them as the job
// says.  Usage: server_memory_test CASE; prints "ok" or what is wrong.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

#include "pakhip.h"

static constexpr uint64_t MB = 1ull << 20;

// ---- the device -------------------------------------------------------------
static std::mutex dev_mu;
static uint64_t dev_cap = 1000 * MB, dev_used = 0;
static std::map<void*, uint64_t> dev_blocks;
static uintptr_t dev_next = 0x10000;

static hipError_t dev_alloc(void** p, uint64_t n) {
  std::lock_guard<std::mutex> lk(dev_mu);
  if (dev_used + n > dev_cap) return hipErrorOutOfMemory;
  dev_used += n;
  dev_next += 0x1000;
  *p = reinterpret_cast<void*>(dev_next);
  dev_blocks[*p] = n;
  return hipSuccess;
}
static hipError_t dev_free(void* p) {
  std::lock_guard<std::mutex> lk(dev_mu);
  auto it = dev_blocks.find(p);
  if (it == dev_blocks.end()) {
    std::printf("freed twice or never allocated\n");
    std::_Exit(1);
  }
  dev_used -= it->second;
  dev_blocks.erase(it);
  return hipSuccess;
}

// Host allocations fail in a thread while its flag is set.
static thread_local bool no_host_memory = false;
void* operator new(std::size_t n) {
  if (no_host_memory) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* fr, size_t* tot) {
  *fr = dev_cap - dev_used;
  *tot = dev_cap;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t*, int) { return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return dev_alloc(p, n); }
hipError_t hipMalloc(void** p, size_t n) { return dev_alloc(p, n); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return dev_free(p); }
hipError_t hipFree(void* p) { return dev_free(p); }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "out of memory"; }

// ---- the context: a job's input is the sizes of its steps ---------------------
struct Steps {
  uint64_t count, cutoff, nodes;  // device bytes
  uint64_t n;                     // k-mers of the table
};
struct pk_ctx {
  void* buf[3] = {};
  uint64_t held[3] = {};
  Steps s{};
};
static int step(pk_ctx* c, int i, uint64_t bytes) {
  if (c->held[i] >= bytes) return PK_OK;
  if (c->buf[i]) dev_free(c->buf[i]);
  c->buf[i] = nullptr;
  c->held[i] = 0;
  if (dev_alloc(&c->buf[i], bytes) != hipSuccess) return PK_ENOMEM;
  c->held[i] = bytes;
  return PK_OK;
}
int pk_ctx_create(pk_ctx** out, int, uint64_t) {
  *out = new pk_ctx();
  return PK_OK;
}
void pk_ctx_destroy(pk_ctx* c) {
  for (void* p : c->buf)
    if (p) dev_free(p);
  delete c;
}
const char* pk_last_error(const pk_ctx*) { return "out of memory"; }
void* pk_ctx_stream(pk_ctx*) { return nullptr; }
uint64_t pk_ctx_device_bytes(const pk_ctx* c) { return c->held[0] + c->held[1] + c->held[2]; }
int pk_ctx_release_buffers(pk_ctx* c) {
  for (int i = 0; i < 3; i++) {
    if (c->buf[i]) dev_free(c->buf[i]);
    c->buf[i] = nullptr;
    c->held[i] = 0;
  }
  return PK_OK;
}
int pk_ctx_set_tuning(pk_ctx*, const pk_tuning*) { return PK_OK; }
int pk_ctx_set_alloc_mode(pk_ctx*, int) { return PK_OK; }
int pk_count(pk_ctx* c, const char* fasta, uint64_t, int k, int, pk_table* out) {
  std::memcpy(&c->s, fasta, sizeof(c->s));
  const int rc = step(c, 0, c->s.count);
  if (rc == PK_OK) *out = pk_table{c->s.n, k <= 32 ? 1 : 2, k, nullptr, nullptr};
  return rc;
}
int pk_last_timing(const pk_ctx*, pk_timing* t) {
  *t = pk_timing{};
  return PK_OK;
}
int pk_cutoff(pk_ctx* c, int, uint64_t*, int* mb, uint64_t* nk) {
  *mb = 1;
  *nk = 1;
  return step(c, 1, c->s.cutoff);
}
int pk_kept_table(pk_ctx*, pk_table* out) {
  *out = pk_table{1, 1, 31, nullptr, nullptr};
  return PK_OK;
}
int pk_macro_nodes(pk_ctx* c, pk_mn_table* out) {
  *out = pk_mn_table{1, 31, nullptr};
  return step(c, 2, c->s.nodes);
}
}  // extern "C"

// ---- the cases ----------------------------------------------------------------
static int run_job(pk_server* s, const Steps& st, int t, int nodes, uint64_t* ticket) {
  pk_job j{};
  j.fasta = reinterpret_cast<const char*>(&st);
  j.nbytes = sizeof(st);
  j.k = 31;
  j.t = t;
  j.fasta_on_device = 1;
  j.want_nodes = nodes;
  if (pk_server_submit(s, &j, ticket)) return -100;
  pk_job_result r{};
  if (pk_server_wait(s, *ticket, &r)) return -101;
  return r.status;
}

static int fail(const char* what) {
  std::printf("%s\n", what);
  return 1;
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  pk_server* s = nullptr;
  // (spare result blocks up to an eighth of the budget)
  if (pk_server_create(&s, 0, 1, 1600 * MB)) return fail("create");
  uint64_t a = 0, b = 0;
  const Steps first{500 * MB, 0, 0, 12 * MB};  // a result block of 144 MB
  if (run_job(s, first, -1, 0, &a)) return fail("first job");
  if (which == "cutoff" || which == "nodes") {
    // the second job's later steps fit only without the first one's block
    if (pk_server_release(s, a)) return fail("release");
    if (dev_used < 640 * MB) return fail("no block was kept");
    const Steps second = which == "cutoff" ? Steps{500 * MB, 400 * MB, 1 * MB, MB}
                                           : Steps{500 * MB, 1 * MB, 400 * MB, MB};
    if (run_job(s, second, 21, 1, &b)) return fail("second job refused");
    if (pk_server_release(s, b)) return fail("release");
  } else if (which == "release") {
    // the second block is kept and the first, beyond what is kept, given back,
    // without a host allocation and without an exception
    if (run_job(s, first, -1, 0, &b)) return fail("second job");
    if (pk_server_release(s, a)) return fail("release");
    const uint64_t used = dev_used;
    no_host_memory = true;
    int rc = -200;
    try {
      rc = pk_server_release(s, b);
    } catch (...) {
    }
    no_host_memory = false;
    if (rc) return fail("release without host memory");
    pk_job_result r{};
    if (pk_server_poll(s, b, &r) != PK_EINVAL) return fail("still known");
    if (dev_used >= used) return fail("nothing given back");
    if (run_job(s, first, -1, 0, &a)) return fail("third job");
  } else {
    return fail("unknown case");
  }
  pk_server_destroy(s);
  if (dev_used) return fail("device memory left");
  std::printf("ok\n");
  return 0;
}
