// rh_align.cpp on a stand-in for the HIP runtime and its kernels: streams,
// events and a memory pool that only keep books, and a call that can be made
// to fail. Usage: align_host <scenario>; prints what went wrong, exits 1.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "align_types.hpp"
#include "racon_hip.h"

namespace {

typedef std::set<int> Kernels;
int next_kernel = 0;
Kernels running;                            // launched, not waited for
std::map<hipStream_t, Kernels> before;      // kernels that a stream's next work follows
std::map<hipEvent_t, Kernels> recorded;
std::map<void*, size_t> held;
size_t pool = size_t(1) << 30, in_use = 0;
int frees = 0;
int fail_in = -1;  // calls until the one that fails (-1: none)
std::string problem;

bool failing() { return fail_in >= 0 && fail_in-- == 0; }
void finish(const Kernels& done) {
  for (int k : done) running.erase(k);
}
// A copy or a clear on `s`: nothing may still run that it does not follow.
void touch(hipStream_t s, const char* what) {
  for (int k : running) {
    if (before[s].count(k) == 0) problem = std::string(what) + " beside a running kernel";
  }
}
hipStream_t new_stream() {
  static uintptr_t n = 0x1000;
  return reinterpret_cast<hipStream_t>(n += 16);
}
}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 4; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipStreamCreate(hipStream_t* s) { *s = new_stream(); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (failing()) return hipErrorUnknown;
  finish(before[s]);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(new_stream());
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (failing()) return hipErrorUnknown;
  recorded[e] = before[s];
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (failing()) return hipErrorUnknown;
  before[s].insert(recorded[e].begin(), recorded[e].end());
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (failing()) return hipErrorUnknown;
  finish(recorded[e]);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = pool - in_use;
  *t = pool;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  static uintptr_t at = 1 << 20;
  if (n > pool - in_use) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void*>(at += (n + 4095) / 4096 * 4096);
  held[*p] = n;
  in_use += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (p == nullptr) return hipSuccess;
  ++frees;
  finish(Kernels(running));  // (waits for the whole device)
  in_use -= held[p];
  held.erase(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t s) {
  if (failing()) return hipErrorUnknown;
  touch(s, "a copy");
  return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t s) {
  if (failing()) return hipErrorUnknown;
  touch(s, "a clear");
  return hipSuccess;
}
}  // extern "C"

namespace rh {
void set_error(const std::string&) {}
void clear_error() {}
hipError_t align_occupancy(int* blocks, uint32_t waves) {
  *blocks = waves == 1 ? 20 : 2;
  return hipSuccess;
}
hipError_t launch_align_batch(const AlignParams& p, uint32_t grid, hipStream_t s) {
  if (failing()) return hipErrorUnknown;
  const size_t room = held[p.scratch];
  if (room < grid * p.slot_bytes) problem = "slots outgrow their buffer";
  before[s].insert(next_kernel);
  running.insert(next_kernel++);
  return hipSuccess;
}
hipError_t launch_breaking_points(const AlignPair*, const AlignResult*, const uint8_t*,
                                  const BreakSpan*, uint32_t, uint32_t, uint32_t*, uint32_t*,
                                  hipStream_t) {
  return hipSuccess;
}
}  // namespace rh

namespace {
const std::string bases(1 << 20, 'A');

// n pairs of `length` bases
void add(std::vector<rh_pair>& pairs, uint32_t n, uint32_t length) {
  const char* s = bases.data();
  for (uint32_t i = 0; i < n; ++i) pairs.push_back(rh_pair{s, length, s, length});
}
int bad(const std::string& what) {
  std::printf("%s\n", what.c_str());
  return 1;
}

// A failure after the first launch leaves no kernel that the next upload
// could overwrite the inputs of.
int errors() {
  std::vector<rh_pair> pairs;
  add(pairs, 2, 20000);
  add(pairs, 400, 500);
  int failed = 0;
  for (int at = 0; at < 40; ++at) {
    rh_align_batch* b = nullptr;
    if (rh_align_create(0, &b) != RH_OK) return bad("create");
    if (rh_align_upload(b, pairs.size(), pairs.data()) != RH_OK) return bad("upload");
    const int launched = next_kernel;
    fail_in = at;
    const int32_t rc = rh_align_run(b);
    fail_in = -1;
    if (rc == RH_OK) {
      if (next_kernel - launched != 2) return bad("not the two kernels of a mixed batch");
      if (failed < 5) return bad("few calls failed");
      rh_align_destroy(b);
      return 0;
    }
    failed += next_kernel > launched;
    if (rh_align_upload(b, pairs.size(), pairs.data()) != RH_OK) return bad("second upload");
    if (rh_align_run(b) != RH_OK) return bad("second run");
    if (!problem.empty()) return bad("call " + std::to_string(at) + ": " + problem);
    rh_align_destroy(b);
  }
  return bad("no run without a failure");
}

// Batches of few long, many short and both kinds of pairs on one object, in
// every order: what a batch kept for the last one never refuses the next.
int memory() {
  std::vector<rh_pair> kinds[3];
  add(kinds[0], 40, 8000);    // one wave each
  add(kinds[1], 8, 40000);    // teams
  add(kinds[2], 8, 40000);
  add(kinds[2], 200, 8000);   // both
  for (size_t mb : {48u, 64u, 96u, 160u, 400u}) {
    pool = mb << 20;
    for (int order = 0; order < 27; ++order) {
      rh_align_batch* b = nullptr;
      if (rh_align_create(0, &b) != RH_OK) return bad("create");
      for (int at = order, k = 0; k < 3; ++k, at /= 3) {
        const std::vector<rh_pair>& pairs = kinds[at % 3];
        if (rh_align_upload(b, pairs.size(), pairs.data()) != RH_OK) return bad("upload");
        if (rh_align_run(b) != RH_OK) {
          return bad("order " + std::to_string(order) + " batch " + std::to_string(k) + " of " +
                     std::to_string(mb) + " MB refused");
        }
      }
      rh_align_destroy(b);
      if (in_use != 0 || !problem.empty()) return bad("left: " + problem);
    }
  }
  return 0;
}

// A team's slot that outgrows the memory: its pairs run one wave each, as
// long as one such slot fits.
int small() {
  std::vector<rh_pair> pairs;
  add(pairs, 4, 100000);
  pool = 16u << 20;
  rh_align_batch* b = nullptr;
  if (rh_align_create(0, &b) != RH_OK) return bad("create");
  if (rh_align_upload(b, pairs.size(), pairs.data()) != RH_OK) return bad("upload");
  if (rh_align_run(b) != RH_OK) return bad("refused");
  rh_align_destroy(b);
  return problem.empty() ? 0 : bad(problem);
}
}  // namespace

int main(int argc, char** argv) {
  const std::string scenario = argc > 1 ? argv[1] : "";
  if (scenario == "errors") return errors();
  if (scenario == "memory") return memory();
  if (scenario == "small") return small();
  return bad("unknown scenario " + scenario);
}
