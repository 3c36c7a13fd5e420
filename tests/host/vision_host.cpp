// vision_host.cpp -- the vision tower's host side (api_vision.hip as built for the library) over
// stand-ins for the device: memory that is never touched, kernels that note their call.  A tensor's
// facts are what the caller says; a kernel fails when told to.  Loaded by test_vision_host.py.
#include "../../ex-nihilo_amd/csrc/api_host.h"
#include <cstdlib>

static std::string g_err, g_log;
static float g_max = 1.f;   // what vis_stats finds in the next tensors
static double g_sumsq = 1.0;
static uint32_t g_inexact = 0;             // and vis_pack
static int g_fail = 0;                     // the step that fails: 1 vis_stats, 2 vis_pack, 3 the flags' way back, 4 vis_rows
static int g_rows = 0, g_cols = 0;         // the product (its W's shape) of spread g_spread; the others' is 1
static double g_spread = 1.0, g_qk = 1.0;  // and q's and k's mean squares
static exn_ctx g_ctx;

namespace exn {
void set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
}
static hipError_t note(const char* what) {
  g_log += what;
  g_log += ' ';
  return hipSuccess;
}
hipError_t tensor_stats_clear(hipStream_t, uint32_t* rec, int64_t n) {
  memset(rec, 0, (size_t)n * 16);
  return hipSuccess;
}
hipError_t vis_stats(hipStream_t, int64_t, int64_t, const float*, uint32_t* rec) {
  if (g_fail == 1) return hipErrorUnknown;
  memcpy(rec, &g_max, 4);
  memcpy(rec + 2, &g_sumsq, 8);
  return hipSuccess;
}
hipError_t vis_pack(hipStream_t, int64_t, int, int, float, const float*, uint16_t*, uint32_t* inexact) {
  *inexact = g_inexact;
  if (g_fail == 3) g_fail = -1;
  return g_fail == 2 ? hipErrorUnknown : hipSuccess;
}
hipError_t vis_square(hipStream_t, int, const float*, const float*, double*) { return hipSuccess; }
hipError_t vis_rows(hipStream_t, int rows, int cols, const float*, const double*, int, const float*, int, double* t2, double* spread) {
  for (int i = 0; i < rows; ++i) t2[i] = g_qk;
  if (g_fail == 4) return hipErrorUnknown;
  *spread = rows == g_rows && cols == g_cols ? g_spread * g_spread : 1.0;
  return hipSuccess;
}
hipError_t vis_widen(hipStream_t, int64_t, const uint16_t*, int, float*) { return hipSuccess; }
hipError_t round_f16(hipStream_t, int64_t, float*) { return hipSuccess; }
hipError_t synth_normal(hipStream_t, uint64_t, int64_t, float, float, int, float*) { return hipSuccess; }
hipError_t vis_sum(hipStream_t, int64_t, const float*, const float*, float*) { return hipSuccess; }
hipError_t vis_prep(hipStream_t, const float*, int, int, int, const float*, int, int, float*, float*, float*) { return hipSuccess; }
hipError_t vis_ln_s(hipStream_t, int64_t, int, int, float*, int, const float*, const float*, const float*, const float*, float,
                    uint16_t* ys, float*) {
  return note(ys ? "ln/s" : "ln/f");
}
hipError_t vis_gemm(hipStream_t, const float*, const float*, const float*, const float*, float*, int64_t, int64_t, int64_t, int) {
  return note("mm/f");
}
hipError_t vis_gemm_s(hipStream_t, const uint16_t*, const uint16_t*, const float*, const float*, float*, uint16_t*, int64_t,
                      int64_t, int64_t, float, float, int64_t, int) {
  return note("mm/s");
}
int vis_split(int64_t, int64_t, int64_t) { return 2; }
int vis_tile(int64_t, int64_t, int64_t, int) { return 0; }
hipError_t vis_gemm_part(hipStream_t, const uint16_t*, const uint16_t*, float*, int64_t, int64_t, int64_t, float, int) {
  return note("mm/s");
}
hipError_t vis_heads(hipStream_t, int, int, const float*, const float*, float, float*, float*, float*) { return note("heads/f"); }
hipError_t vis_heads_s(hipStream_t, int, int, int, const float*, const float*, float, float, float, uint16_t*, uint16_t*, uint16_t*) {
  return note("heads/s");
}
hipError_t vis_attend(hipStream_t, int, int, const float*, const float*, const float*, float*) { return note("attend/f"); }
hipError_t vis_attend_s(hipStream_t, int, int, int, const uint16_t*, const uint16_t*, const uint16_t*, float, float, int,
                        uint16_t*, float*) {
  return note("attend/s");
}
}  // namespace exn

int use(exn_ctx*) { return EXN_OK; }
uint64_t gen_key(uint64_t s, uint64_t t) { return s + t; }
int dev_alloc(void** p, size_t n) {
  *p = malloc(n ? n : 1);
  return *p ? EXN_OK : EXN_ENOMEM;
}
void dev_free(void* p) { free(p); }
int ctx_tmp(exn_ctx* c, size_t n, void** out) {
  if (c->tmp_bytes < n) {
    free(c->tmp);
    c->tmp = malloc(n);
    c->tmp_bytes = n;
  }
  *out = c->tmp;
  return EXN_OK;
}

extern "C" {
// only what comes back to the host is looked at
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
  if (g_fail == -1) return hipErrorUnknown;
  if (kind == hipMemcpyDeviceToHost) memcpy(dst, src, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "a planted failure"; }

exn_ctx* vh_ctx() { return &g_ctx; }
void vh_facts(float mx, double sumsq, int inexact, int fail) {
  g_max = mx;
  g_sumsq = sumsq;
  g_inexact = (uint32_t)inexact;
  g_fail = fail;
}
void vh_spread(int rows, int cols, double spread, double qk) {
  g_rows = rows;
  g_cols = cols;
  g_spread = spread;
  g_qk = qk;
}
// the kernels an encode of a 64 x 64 picture launches, in order
const char* vh_encode(exn_vision* v) {
  static float px[64 * 64 * 4], out[4 * 4 * 4096];
  g_log.clear();
  if (exn_vision_encode_dev(v, px, 64, 64, out, out + 4 * 4096) != EXN_OK) g_log = "error " + g_err;
  return g_log.c_str();
}
}
