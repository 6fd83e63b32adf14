// load_failures.cpp -- mmp_fiber_load with each of its runtime calls failing in turn, on the host: this program's
// own definitions of the HIP runtime calls stand in for the library's (device memory is host memory, kernels do
// nothing, a graph is a token), and the k-th copy or synchronisation of a load returns an error. Until a load has
// gone through whole, a solver whose lines and coupling blocks are only partly those of the new plan must refuse to
// step; a load repeated after the failure must leave device memory as an undisturbed load does.
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "mmprop.h"

namespace {

struct Block {
  char* p;
  size_t n;
};
std::vector<Block> g_blocks;
long g_fail_at = -1, g_calls = 0;  // the fallible call to fail (-1: none), and how many there were
int g_token;

hipError_t fallible() { return g_calls++ == g_fail_at ? hipErrorUnknown : hipSuccess; }

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "forced"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = &g_token, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  g_blocks.push_back({static_cast<char*>(std::calloc(n ? n : 1, 1)), n});
  *p = g_blocks.back().p;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  for (size_t i = 0; i < g_blocks.size(); i++)
    if (g_blocks[i].p == p) {
      std::free(p);
      g_blocks.erase(g_blocks.begin() + i);
      break;
    }
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  const hipError_t e = fallible();
  if (e == hipSuccess) std::memcpy(d, s, n);
  return e;
}
hipError_t hipStreamSynchronize(hipStream_t) { return fallible(); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(&g_token), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = reinterpret_cast<hipGraph_t>(&g_token), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return *e = reinterpret_cast<hipGraphExec_t>(&g_token), hipSuccess;
}
hipError_t hipGraphUpload(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(&g_token), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
  return hipSuccess;
}
// the library's kernels are not registered anywhere
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(&g_token); }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}

namespace {

int g_bad = 0;
void expect(bool ok, const char* what, long k) {
  if (ok) return;
  std::fprintf(stderr, "FAILED: %s (call %ld; last error: %s)\n", what, k, mmp_last_error());
  g_bad++;
}

// Every (k, l, m) with k + l - m - p even; symmetric: equal values at (l, m) and (m, l).
struct Fiber {
  std::vector<double> beta, qv, fields, hr;
  std::vector<uint32_t> off, klm;
  mmp_params p{};
  Fiber(uint32_t M, uint32_t nt, bool symmetric, double length) {
    for (uint32_t q = 0; q < M; q++) beta.insert(beta.end(), {-1.5e3 * q, 5e-4 * q, 0.02, 3e-5});
    off.push_back(0);
    for (uint32_t q = 0; q < M; q++) {
      for (uint32_t k = 0; k < M; k++)
        for (uint32_t l = 0; l < M; l++)
          for (uint32_t m = 0; m < M; m++)
            if ((k + l + m + q) % 2 == 0) {
              klm.insert(klm.end(), {k, l, m});
              qv.push_back(6e12 * (1. + q + 2. * k + 3. * (l + m) + (symmetric ? 0. : 0.5 * l)));
            }
      off.push_back((uint32_t)qv.size());
    }
    fields.assign(2 * (size_t)M * nt, 0.);
    for (size_t j = 0; j < fields.size(); j++) fields[j] = 1. + 1e-3 * (j % 97);
    hr.assign(nt, 0.);
    for (uint32_t j = 0; j < nt; j++) hr[j] = std::exp(-0.01 * j);
    p.n_modes = M;
    p.fiber_length = length;
    p.n_beta = 4;
    p.dispersion_coefficients = beta.data();
    p.coupling_offsets = off.data();
    p.coupling_klm = klm.data();
    p.coupling_values = qv.data();
    p.nt = nt;
    p.time_window = 20.;
    p.pulse_width = 0.1;
    p.initial_fields = fields.data();
    p.n_steps = 1000;
    p.method_order = 4;
    p.nonlinearity_const = 1.4e-13;
    p.raman_proportion = 0.18;
    p.raman_response = hr.data();
    p.raman = 1;
  }
};

std::vector<std::vector<char>> memory() {
  std::vector<std::vector<char>> out;
  for (const Block& b : g_blocks) out.emplace_back(b.p, b.p + b.n);
  return out;
}

mmp_solver* batch(mmp_ctx* ctx, const std::vector<mmp_params>& ps) {
  const mmp_options o{MMP_PRECISION_FP64, MMP_PAIRS_PHYSICAL, 0, 0};
  mmp_solver* s = nullptr;
  expect(mmp_batch_create(ctx, (uint32_t)ps.size(), ps.data(), &o, &s) == MMP_OK, "mmp_batch_create", -1);
  return s;
}

}  // namespace

int main() {
  mmp_ctx* ctx = nullptr;
  if (mmp_ctx_create(0, &ctx) != MMP_OK) return 2;
  Fiber a(6, 4096, true, 0.5), c(6, 4096, true, 0.6), general(6, 4096, false, 0.7);
  // an undisturbed load: the runtime calls of one that changes the plan, and of one that does not
  mmp_solver* s = batch(ctx, {a.p, a.p, c.p});
  g_calls = 0;
  expect(mmp_fiber_load(s, 1, &general.p) == MMP_OK, "load", -1);
  const long all = g_calls;
  const auto want = memory();
  g_calls = 0;
  expect(mmp_fiber_load(s, 1, &general.p) == MMP_OK, "second load", -1);
  const long change = all - g_calls;
  mmp_solver_destroy(s);
  expect(change > 4, "the load changes the plan", -1);
  for (long k = 0; k < all; k++) {
    s = batch(ctx, {a.p, a.p, c.p});
    g_calls = 0;
    g_fail_at = k;
    expect(mmp_fiber_load(s, 1, &general.p) != MMP_OK, "a load with a failing call reports it", k);
    g_fail_at = -1;
    if (k >= 1 && k <= change)  // (call 0 waits for the queued work)
      expect(mmp_advance(s, 1) != MMP_OK, "no step on a plan that is only partly there", k);
    expect(mmp_fiber_load(s, 1, &general.p) == MMP_OK, "the load repeated", k);
    expect(memory() == want, "device memory after the repeated load", k);
    expect(mmp_advance(s, 17) == MMP_OK, "steps after the repeated load", k);
    mmp_solver_destroy(s);
  }
  mmp_ctx_destroy(ctx);
  std::printf("%ld calls, %ld of the change of plan\n%s\n", all, change, g_bad ? "FAILED" : "load failure checks passed");
  return g_bad ? 1 : 0;
}
