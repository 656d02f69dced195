// The library's host side over a device of a stated memory size, without a GPU:
// the runtime calls below count what is allocated and fail past the limit, the
// launches do nothing.  Exit status 0 and "ok" when every check holds.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <vector>

#include "../../include/rstr_hip.h"
#include "../../pretrained-rstr_amd/csrc/kernels.h"

static size_t g_limit = SIZE_MAX, g_used = 0;
static std::map<void*, size_t> g_blocks;
static hipError_t g_last = hipSuccess;
static std::function<void()> g_on_sync;

static hipError_t take(void** p, size_t n) {
  if (g_used + n > g_limit) return g_last = hipErrorOutOfMemory;
  *p = calloc(1, n ? n : 1);
  g_blocks[*p] = n;
  g_used += n;
  return hipSuccess;
}
static hipError_t give(void* p) {
  if (!p) return hipSuccess;
  if (!g_blocks.count(p)) {
    printf("a free of memory that is not allocated\n");
    exit(1);
  }
  g_used -= g_blocks[p];
  g_blocks.erase(p);
  free(p);
  return hipSuccess;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memmove(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return memmove(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = reinterpret_cast<hipStream_t>(&g_limit), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  if (g_on_sync) {
    auto f = std::move(g_on_sync);
    g_on_sync = nullptr;
    f();
  }
  return hipSuccess;
}
}

namespace rstr {
static char g_scratch[64];
hipError_t static_scratch_address(void** p) { return *p = g_scratch, hipSuccess; }
hipError_t launch_gen_linear(hipStream_t, const QTensor&, int, int, int, uint64_t, const float*) { return hipSuccess; }
hipError_t launch_gen_f32(hipStream_t, float*, int64_t, uint64_t, double, double, double) { return hipSuccess; }
hipError_t launch_prescale(hipStream_t, float*, const float*, int64_t, double) { return hipSuccess; }
size_t attn_tab_words(const AttnGeom& g, int max_items) { return 8 * (size_t)g.batch + 4 * (size_t)max_items; }
hipError_t launch_attn_lists(hipStream_t, const AttnGeom*, int, const int32_t*, int32_t*, size_t, int) {
  return hipGetLastError();
}
hipError_t launch_attn_split(hipStream_t, const AttnGeom&, const float*, const uint16_t*, const uint16_t*, const int32_t*,
                             int32_t*, float*, int, const AttnOut*) {
  return hipGetLastError();
}
hipError_t launch_attn_merge(hipStream_t, const AttnGeom&, const int32_t*, int32_t*, const float*, float*, ActBuf*) {
  return hipGetLastError();
}
}  // namespace rstr

static rstr_session* g_s;
#define CHECK(x)                                                                 \
  do {                                                                           \
    if (!(x)) {                                                                  \
      printf("line %d: %s (%s)\n", __LINE__, #x, g_s ? rstr_last_error(g_s) : ""); \
      return 1;                                                                  \
    }                                                                            \
  } while (0)

static int attend(rstr_pool* p, int lanes) {
  const int n_q = 8, hd = 128, pps = 4;
  std::vector<float> q((size_t)lanes * n_q * hd, 1.0f), out(q.size());
  std::vector<int32_t> rows, pos(lanes, 63), table((size_t)lanes * pps), len(lanes, 64), start(lanes, 0);
  for (int b = 0; b <= lanes; b++) rows.push_back(b);
  for (size_t i = 0; i < table.size(); i++) table[i] = (int)(i % 4);
  return rstr_attention_run(p, 0, lanes, n_q, 16, 0, 0.1f, q.data(), rows.data(), pos.data(), table.data(), pps,
                            len.data(), start.data(), out.data());
}

int main() {
  rstr_model_desc d{};
  d.n_layers = 1;
  d.d_model = d.d_ff = 128;
  d.n_q = 8;
  d.n_kv = 1;
  d.head_dim = 128;
  d.vocab = 512;
  d.weight_bits = 4;
  d.eps = 1e-6f;
  d.attn_scale = 0.1f;
  d.rope_global = d.rope_local = 1e4;
  rstr_model* m = nullptr;
  rstr_pool *a = nullptr, *b = nullptr, *c = nullptr;
  CHECK(rstr_session_open(0, &g_s) == RSTR_OK);
  CHECK(rstr_model_bind_synthetic(g_s, &d, 1, &m) == RSTR_OK);
  CHECK(rstr_pool_open(m, 16, 8, &a) == RSTR_OK);
  const size_t idle = g_used;
  CHECK(attend(a, 64) == RSTR_OK);
  const size_t kept = g_used - idle;
  CHECK(kept > 0);

  // a pool that fits only without what is kept: 100 pages are 819 200 bytes
  CHECK(rstr_pool_open(m, 16, 100, &b) == RSTR_OK);
  const size_t pool_bytes = g_used - idle - kept;
  CHECK(rstr_pool_close(b) == RSTR_OK);
  g_limit = g_used + pool_bytes - 1;
  CHECK(kept > 1 && rstr_pool_open(m, 16, 100, &b) == RSTR_OK);
  CHECK(g_used == idle + pool_bytes);
  // the refused first attempt is no launch's error, and the next call asks anew
  g_limit = SIZE_MAX;
  CHECK(attend(b, 8) == RSTR_OK && attend(a, 64) == RSTR_OK);

  // blocks in use stay: an allocation beside the running call fails, the call does not
  size_t before = 0, after = 0;
  int rc = RSTR_OK;
  CHECK(rstr_pool_close(b) == RSTR_OK);
  g_limit = g_used + pool_bytes - 1;
  g_on_sync = [&] {
    before = g_used;
    rc = rstr_pool_open(m, 16, 100, &c);
    after = g_used;
  };
  CHECK(attend(a, 64) == RSTR_OK);
  CHECK(rc == RSTR_E_OOM && c == nullptr && before == after);
  // a second pool's call takes the first one's idle blocks, never its own
  g_limit = SIZE_MAX;
  CHECK(rstr_pool_open(m, 16, 8, &b) == RSTR_OK);
  g_limit = g_used + kept - 1;
  CHECK(attend(b, 64) == RSTR_OK);
  CHECK(g_used <= g_limit);

  CHECK(rstr_pool_close(a) == RSTR_OK && rstr_pool_close(b) == RSTR_OK);
  CHECK(rstr_model_close(m) == RSTR_OK && rstr_session_close(g_s) == RSTR_OK);
  g_s = nullptr;
  CHECK(g_used == 0);
  printf("ok\n");
  return 0;
}
