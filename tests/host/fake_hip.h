// A HIP runtime and launch functions that run nothing, for tests of the host side (csrc/engine.cpp) without a GPU: every call of
// interest is written to `calls`, device memory is host memory, and an allocation above `limit` bytes fails.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <set>
#include <string>
#include <vector>

#include "ha.h"
#include "ha_kernels.h"

static std::vector<std::string> calls;
static size_t limit = ~(size_t)0;
static std::vector<void*> state_out;  // where each gated-delta launch writes its state
static std::vector<ha::GqaArgs> gqa_calls;
static hipError_t last_error = hipSuccess;

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t* p, int) { memset(p, 0, sizeof *p); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t n) {
  calls.push_back("malloc");
  if (n > limit) { *p = nullptr; return last_error = hipErrorOutOfMemory; }
  *p = calloc(1, n);
  return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { if (v || n < (1 << 26)) memset(p, v, n); return hipSuccess; }  // (new memory is zero)
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { calls.push_back("copy"); memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
  calls.push_back("copy2d");
  for (size_t i = 0; i < h; i++) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)malloc(8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free((void*)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)malloc(8); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { calls.push_back("event"); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
}

namespace ha {
static hipError_t gdn(const GdnArgs& a, float mark) {
  calls.push_back("launch");
  state_out.push_back(a.S_out);
  for (size_t i = 0; i < (size_t)a.B * a.H * a.DK * a.DV; i++) a.S_out[i] = mark + (float)state_out.size();
  return hipSuccess;
}
hipError_t launch_gdn_sequential(const GdnArgs& a, hipStream_t) { return gdn(a, 100); }
hipError_t launch_gdn_chunked(const GdnArgs& a, hipStream_t) { return gdn(a, 200); }
hipError_t launch_gdn_split(const GdnArgs& a, hipStream_t) { return gdn(a, 300); }
hipError_t launch_gdn_duo(const GdnArgs& a, hipStream_t) { return gdn(a, 400); }
bool gdn_duo_fits(int B, int H) { return B * H % 8 == 0 && B * H <= 128; }
size_t gdn_split_image_bytes() { return 1024; }
hipError_t launch_tail_update(const TailArgs& a, hipStream_t) {
  calls.push_back("tails");
  for (int i = 0; i < a.n; i++) memset(a.tail_out[i], 7, 64);
  for (int i = 0; i < a.n && a.state_bytes; i++) memcpy(a.state_out[i], a.state[i], a.state_bytes);
  return hipSuccess;
}
hipError_t launch_gqa(const GqaArgs& a, hipStream_t) { calls.push_back("gqa"); gqa_calls.push_back(a); return hipSuccess; }
hipError_t launch_gqa_rows(const GqaArgs& a, hipStream_t) { calls.push_back("gqa_rows"); gqa_calls.push_back(a); return hipSuccess; }
size_t gqa_part_slots(int pairs, int, int) { return (size_t)pairs; }
size_t gqa_part_slot_bytes() { return 64; }
hipError_t mnb_check(const MnbArgs&) { return hipSuccess; }
MnbShape mnb_shape(const MnbArgs& a) { return MnbShape{a.M, a.N, a.K, a.bits, a.group, a.asym != 0, true}; }
hipError_t launch_mnb_strip(const MnbArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_mnb_tiles(const MnbArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_mnb_gemv(const MnbArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_mnb_gemm(const MnbArgs&, hipStream_t) { return hipSuccess; }
hipError_t mnb_scratch_setup(int) { return hipSuccess; }
float* mnb_scratch(int) { return nullptr; }
hipError_t launch_fwht(void*, long, int, hipStream_t) { return hipSuccess; }
hipError_t launch_embed(const EmbedArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_add_norm(const AddNormArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_silu_mul(const void*, void*, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_add_bias(void*, const float*, int, int, hipStream_t) { return hipSuccess; }
}  // namespace ha

static int fails = 0;
#define CHECK(x) \
  do { \
    if (!(x)) { fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #x, ha_last_error()); fails++; } \
  } while (0)

static long where(const char* what, size_t from = 0) {
  for (size_t i = from; i < calls.size(); i++)
    if (calls[i] == what) return (long)i;
  return -1;
}

static ha_config config(const unsigned char* kinds, int n, int batch, int max_ctx) {
  ha_config c;
  memset(&c, 0, sizeof c);
  c.n_layers = n; c.layer_kind = kinds; c.batch = batch; c.max_ctx = max_ctx;
  c.H = 16; c.DK = 128; c.DV = 128; c.conv_k = 4; c.lin_stride = 8256; c.lin_dtype = HA_F32; c.lin_gnorm = 1;
  c.HQ = 8; c.HK = 2; c.HD = 256; c.rot_dim = 64; c.full_stride = 5120; c.full_dtype = HA_F16; c.rope_theta = 1e7f; c.eps = 1e-6f;
  return c;
}
