/*
 * A device on the CPU for the host side of gq_runtime.hip: the HIP calls it
 * makes (device memory as malloc with a capacity and failures on request) and
 * the launchers it calls, which follow the workspaces instead of computing.
 * tests/test_runtime_host.py links it with gq_runtime.hip in place of the HIP
 * runtime and the kernels.
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <string>
#include <utility>

#include "gq_internal.h"

namespace {

struct Block {
  size_t bytes;
};
std::map<char *, Block> live; /* device memory */
size_t used, capacity = (size_t)288 << 30, refuse_from = ~(size_t)0;
long refuse_after = -1; /* allocations granted before all are refused; -1: no such limit */
bool refuse_pinned;
hipError_t last = hipSuccess; /* the last call that failed, until it is asked for */
std::map<std::string, long> counts;
std::string errors;

void error(const std::string &s) { errors += s + "\n"; }

/* [p, p + n) lies in one live allocation */
bool in_bounds(const void *p, size_t n) {
  auto it = live.upper_bound((char *)p);
  if (it == live.begin()) return false;
  --it;
  return (char *)p + n <= it->first + it->second.bytes;
}

void need(const char *what, const void *p, size_t n) {
  if (!in_bounds(p, n)) error(std::string(what) + " outside device memory");
}

/* K-part sums that a launch left to a later one: the workspace and the stamp
 * written there */
struct Owed {
  const float *part = nullptr;
  float stamp = 0;
  int n = 0;
} owed_qkv, owed_x;
float serial;
const int *captured_tokens; /* the token log of the captured step */

/* a launch whose sums its caller adds; n parts of tokens x rows */
void leave(Owed &o, float *part, int n, size_t floats) {
  need("K parts", part, sizeof(float) * n * floats);
  o.part = part, o.n = n, o.stamp = ++serial;
  for (int k = 0; k < n; k++) part[k * floats] = o.stamp;
}

void take(Owed &o, const char *what, const float *part, int n, size_t floats) {
  if (!o.n) {
    if (part) error(std::string(what) + ": parts that no launch left");
    return;
  }
  if (!part || part != o.part || n != o.n) {
    error(std::string(what) + ": parts lost");
  } else if (!in_bounds(part, sizeof(float) * n * floats)) {
    error(std::string(what) + ": parts freed");
  } else {
    for (int k = 0; k < n; k++)
      if (part[k * floats] != o.stamp) error(std::string(what) + ": parts overwritten");
  }
  o = Owed();
}

} // namespace

extern "C" {
/* what the tests ask for and see */
void fake_reset(size_t total) { capacity = total, refuse_from = ~(size_t)0, refuse_after = -1, refuse_pinned = false, last = hipSuccess, counts.clear(), errors.clear(), owed_qkv = owed_x = Owed(); }
void fake_refuse_from(size_t bytes) { refuse_from = bytes; } /* allocations of so many bytes and more fail */
void fake_refuse_after(long n) { refuse_after = n; }
void fake_refuse_pinned(int on) { refuse_pinned = on != 0; }
const char *fake_errors() { return errors.c_str(); }
long fake_count(const char *what) { return counts[what]; }
size_t fake_used() { return used; }

/* ---- the HIP runtime ---- */
hipError_t hipMalloc(void **p, size_t n) {
  counts["malloc"]++;
  if (refuse_after > 0) refuse_after--;
  else if (refuse_after == 0) n = ~(size_t)0;
  if (n >= refuse_from || n > capacity - used) {
    counts["refused"]++;
    return last = hipErrorOutOfMemory;
  }
  /* a large block holds no more host memory than its start: nothing here
   * writes past the first floats of a part */
  char *b = (char *)malloc(n);
  if (!b) return hipErrorOutOfMemory;
  live[b] = Block{n}, used += n, *p = b;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = live.find((char *)p);
  if (it == live.end()) {
    error("free of what is not allocated");
    return hipErrorInvalidValue;
  }
  used -= it->second.bytes;
  free(it->first);
  live.erase(it);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = capacity - used, *t = capacity, hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  counts["host_malloc"]++;
  if (refuse_pinned) return last = hipErrorOutOfMemory;
  return (*p = calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k != hipMemcpyDeviceToHost) need("copy to", d, n);
  if (k != hipMemcpyHostToDevice) need("copy from", s, n);
  return memmove(d, s, n), hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int, size_t n, hipStream_t) { return need("memset", p, n), hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }
hipError_t hipGetLastError() { return std::exchange(last, hipSuccess); }
const char *hipGetErrorString(hipError_t) { return "fake device"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)&live, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = (hipGraph_t)&live, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return *e = (hipGraphExec_t)&live, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  counts["graph"]++;
  need("captured token log", captured_tokens, sizeof(int));
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)&live, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)&live, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
void **__hipRegisterFatBinary(void *) { return nullptr; }
void __hipRegisterVar(void *, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void *) {}
}

/* ---- the launchers ----
 * each asks for the last error, as the real ones do after their launch */
static int launched() { return hipGetLastError() == hipSuccess ? 0 : -4; }
int gq_attn_nch(int, int max_seq) { return (max_seq + 31) / 32; }
int gq_attn_smax(int, int) { return 32; }
int gq_argmax_blocks(int n) { return (n + 1023) / 1024; }
size_t gq_dense_bytes(int rows, int K, bool swiglu) { return (size_t)rows * K * (swiglu ? 4 : 2); }
size_t gq_mm_tile_bytes(int, int rows, int cols, bool swiglu) { return (size_t)rows * cols * (swiglu ? 2 : 1); }
size_t gq_q6k_units_bytes(int rows, int cols) { return (size_t)rows * cols; }
size_t gq_sample_ws_bytes(int vocab) { return 16 * (size_t)vocab; }
size_t gq_sample_topk_bytes(int vocab, int k) { return k <= 256 ? 12 * (size_t)vocab : 0; }
bool gq_flash_takes(int n_heads, int n_kv, int hd) { return (hd == 64 || hd == 128) && n_heads / n_kv <= 8; }
size_t gq_flash_parts(int ntok, int pos, int n_heads, int, int, int) { return pos ? (size_t)2 * ntok * n_heads : 0; }
bool gq_matvec_mm_forced() { return false; }
bool gq_matvec_q6k_ref() { return false; }
void gq_matvec_set_cus(int) {}

static int pgemm_parts(int mode, int T, size_t rows, float *part, size_t cap, int *out, int n) {
  if (out) *out = 0;
  if (mode == MV_SWIGLU || !out || !part) return launched();
  if ((size_t)n * T * rows > cap) return launched();
  leave(mode == MV_RESID ? owed_x : owed_qkv, part, n, (size_t)T * rows);
  *out = n;
  return launched();
}
int gq_launch_pgemm(int mode, const PgArgs &a, hipStream_t) {
  counts["pgemm"]++;
  size_t rows = 0;
  for (int i = 0; i < a.nseg; i++) rows += a.seg[i].rows;
  return pgemm_parts(mode, a.T, rows, a.part, a.part_cap, a.kparts_out, 2);
}
int gq_launch_dense(int mode, const DnArgs &a, int, hipStream_t) {
  counts["dense"]++;
  size_t rows = 0;
  for (int i = 0; i < a.nseg; i++) rows += a.rows[i];
  need("bf16 copy", a.w, gq_dense_bytes((int)rows, a.K, mode == MV_SWIGLU));
  if (mode == MV_RESID && (!a.part || (size_t)a.T * rows > a.part_cap)) return -1;
  return pgemm_parts(mode, a.T, rows, a.part, a.part_cap, a.kparts_out, mode == MV_RESID ? 1 : 4);
}
int gq_launch_dense_tile(void *dst, int, const void *w0, const void *w1, int rows, int K, hipStream_t) {
  counts["dense_tile"]++;
  need("bf16 copy", dst, gq_dense_bytes(rows, K, w1 != nullptr));
  need("weights", w0, 1);
  return launched();
}
int gq_launch_rmsnorm_rows(const float *x, const float *, float *, int dim, int rows, float, hipStream_t, __bf16 *,
                           const float *parts, int nparts, float *) {
  need("norm", x, sizeof(float) * dim * rows);
  take(owed_x, "norm", parts, parts ? nparts : 0, (size_t)rows * dim);
  return launched();
}
int gq_launch_rope_append(const RopeArgs &a, hipStream_t) {
  counts["rope_append"]++;
  take(owed_qkv, "rope", a.parts, a.parts ? a.kparts : 0, (size_t)a.ntok * a.prow);
  return launched();
}
int gq_launch_flash_prefill(const AttnArgs &a, int, hipStream_t) {
  counts["flash"]++;
  if (a.part_o) need("attention parts", a.part_o, sizeof(float) * 2 * a.ntok * a.n_heads * (a.hd + 2));
  return launched();
}
int gq_launch_argmax(const float *x, int n, float *, int, int *out, int *tokens, int *, int *, hipStream_t, int, const void *, int,
                     float *, const ArgmaxHost &h) {
  need("logits", x, sizeof(float) * n);
  if (tokens) need("token log", captured_tokens = tokens, sizeof(int));
  if (h.token) *h.token = 3;
  else *out = 3;
  return launched();
}
int gq_launch_sample(const float *, int, float temperature, int, float, int, const SampleWs &w, int *out, hipStream_t) {
  if (temperature <= 0.f) return 1;
  counts[w.topk ? "topk_fast" : "topk_replay"]++;
  *out = 5;
  return launched();
}
int gq_launch_attention(const AttnArgs &a, hipStream_t, hipEvent_t) {
  need("attention parts", a.part_o, sizeof(float) * a.n_heads * a.nch * a.hd);
  need("attention sums", a.part_ml, sizeof(float) * a.n_heads * a.nch * 2);
  return launched();
}
int gq_launch_matvec(int, int, const MvArgs &, hipStream_t) { return launched(); }
int gq_launch_matvec_pair(int, const MvArgs &, int, const MvArgs &, hipStream_t) { return 1; }
int gq_launch_mm_tile(void *, int, const void *, const void *, int, int, hipStream_t) { return launched(); }
int gq_launch_q6k_units(void *, const void *, int, int, hipStream_t) { return launched(); }
int gq_launch_rmsnorm(const float *, const float *, float *, int, float, hipStream_t) { return launched(); }
int gq_launch_embed(int, const void *, int, const int *, int, float *out, hipStream_t, int *, int, int) { return need("embedding", out, 4), launched(); }
int gq_launch_embed_rows(int, const void *, int, const int *tokens, int n, float *, hipStream_t) {
  counts["chunk"]++;
  for (int i = 0; i < n; i++) counts["token_sum"] += tokens[i];
  return launched();
}
int gq_launch_to_bf16(const float *, __bf16 *, size_t, hipStream_t) { return launched(); }
int gq_launch_silu_mul(float *, const float *, int, hipStream_t) { return launched(); }
int gq_launch_copy(void *, const void *, size_t, int, hipStream_t) { return launched(); }
int gq_launch_stream_read(const void *, size_t, uint32_t *, size_t, hipStream_t) { return launched(); }
int gq_launch_synth_quant(void *, int, int, int, uint64_t, hipStream_t) { return launched(); }
int gq_launch_synth_normal(float *, size_t, uint64_t, int, hipStream_t) { return launched(); }
int gq_launch_synth_kv(float *, int, int, int, int, int, uint64_t, hipStream_t) { return launched(); }
