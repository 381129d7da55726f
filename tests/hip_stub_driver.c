/* Drives the host code of libseoulkv4_hip without a GPU: this program defines
 * the HIP runtime calls that the library makes (its definitions come before
 * the runtime's), so device memory is counted host memory, a launch runs
 * nothing, and one can be made to fail.  tests/test_hip_stub.py builds it and
 * runs one scenario per test: hip_stub_driver NAME.  Exit status 0: every
 * expectation held. */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#include "seoulkv4_hip.h"

#define CHECK(cond, ...)                                       \
  do {                                                         \
    if (!(cond)) {                                             \
      fprintf(stderr, "FAILED %s:%d: ", __FILE__, __LINE__);   \
      fprintf(stderr, __VA_ARGS__);                            \
      fprintf(stderr, "\n");                                   \
      exit(2);                                                 \
    }                                                          \
  } while (0)

/* ------------------------------------------------------- the counted runtime */
static struct { char *at; size_t bytes; } blocks[64];
static int live;              /* device allocations not freed yet */
static int launches;          /* kernel launches so far */
static int fail_launch = -1;  /* this launch (counted from 0) fails */
static hipError_t last_error = hipSuccess;

hipError_t hipMalloc(void **p, size_t n) {
  for (int i = 0; i < 64; ++i)
    if (!blocks[i].at) {
      *p = blocks[i].at = aligned_alloc(256, (n + 255) & ~(size_t)255);
      blocks[i].bytes = n;
      ++live;
      return hipSuccess;
    }
  return hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  for (int i = 0; i < 64; ++i)
    if (blocks[i].at == p) {
      free(p);
      blocks[i].at = NULL;
      --live;
      return hipSuccess;
    }
  CHECK(0, "hipFree of memory that is not allocated");
  return hipErrorInvalidValue;
}
/* bytes of the live allocation that holds [p, p + n), or 0 */
static size_t block_of(const void *p, size_t n) {
  const char *c = p;
  for (int i = 0; i < 64; ++i)
    if (blocks[i].at && c >= blocks[i].at && c + n <= blocks[i].at + blocks[i].bytes)
      return blocks[i].bytes;
  return 0;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned f) { (void)f; *d = h; return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { (void)st; return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
  (void)st;
  CHECK(block_of(d, n), "memset of %zu bytes past its allocation", n);
  return hipMemset(d, v, n);
}
hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : hipErrorInvalidDevice; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = 160 * 1024; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) { (void)d; memset(p, 0, sizeof *p); return hipSuccess; }
hipError_t hipFuncGetAttributes(struct hipFuncAttributes *a, const void *f) { (void)f; memset(a, 0, sizeof *a); return hipSuccess; }
static int an_object;
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)&an_object; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { (void)s; (void)e; (void)f; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; *e = (hipEvent_t)&an_object; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) { (void)g; (void)b; (void)sh; (void)s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s) {
  memset(g, 0, sizeof *g);
  memset(b, 0, sizeof *b);
  *sh = 0;
  *s = NULL;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t sh, hipStream_t s) {
  (void)f; (void)g; (void)b; (void)a; (void)sh; (void)s;
  if (launches++ == fail_launch) return last_error = hipErrorLaunchFailure;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}

/* -------------------------------------------------------------- a tiny index */
enum { T = 512, NC = 32, SINK = 16, LOCAL = 48 };
static uint16_t kv[4 * T * 256], query[16 * 256];

static void *create(void) {
  static uint8_t plane[NC * 64];
  static float scale[NC];
  static uint16_t resid[NC], gfs[NC / 32];
  static int32_t offsets[NC + 1], values[T];
  int n = 0;
  for (int c = 0; c < NC; ++c) {  /* token t of the retrieval zone in list t % NC */
    offsets[c] = n;
    for (int t = SINK; t < T - LOCAL; ++t)
      if (t % NC == c) values[n++] = t;
  }
  offsets[NC] = n;
  skv_index_desc ix;
  memset(&ix, 0, sizeof ix);
  ix.context = T;
  ix.sink = SINK;
  ix.local = LOCAL;
  ix.n_centroids = NC;
  for (int g = 0; g < 4; ++g) {
    skv_cell_desc *c = &ix.cells[g];
    c->upper = c->lower = plane;
    c->scale = scale;
    c->resid_f16 = resid;
    c->gfs_f16 = gfs;
    c->offsets = offsets;
    c->values = values;
    c->nprobe = 8;
  }
  void *h = NULL;
  const int code = skv_create(&ix, kv, kv, 0, NULL, &h);
  CHECK(code == SKV_OK && h, "create: code %d '%s'", code, skv_last_error(NULL));
  return h;
}

/* ------------------------------------------------------------------ scenarios */
/* The outputs live until the handle and every hold on them are gone, and a
 * hold keeps nothing else of the handle. */
static void output_lifetime(void) {
  void *h = create(), *out, *tiles, *dense, *a = NULL, *b = NULL;
  const int all = live;
  CHECK(skv_output_hold(NULL, &a) == SKV_EINVAL && skv_output_hold(h, NULL) == SKV_EINVAL, "NULL");
  CHECK(skv_output_device(h, &out) == SKV_OK && skv_output_tiles_device(h, &tiles) == SKV_OK &&
            skv_dense_output_device(h, &dense) == SKV_OK, "pointers");
  CHECK(skv_output_hold(h, &a) == SKV_OK && skv_output_hold(h, &b) == SKV_OK, "hold");
  CHECK(live == all, "a hold allocates nothing");
  CHECK(skv_run(h, query) == SKV_OK && skv_sync(h, NULL) == SKV_OK, "step");
  memset(out, 7, 16 * 256 * 2);
  skv_output_release(b);
  skv_destroy(h);
  CHECK(live == 1, "%d allocations left under a hold, the outputs are one", live);
  const size_t bytes = block_of(out, 16 * 256 * 2);
  CHECK(bytes && bytes < 1 << 20, "outputs held in %zu bytes", bytes);
  CHECK(block_of(tiles, 4 * 32 * 4 * 256 * 2) && block_of(dense, 16 * 256 * 2), "all outputs held");
  CHECK(((unsigned char *)out)[16 * 256 * 2 - 1] == 7, "the last output is kept");
  skv_output_release(a);
  CHECK(live == 0, "%d allocations left after the last hold", live);
  skv_output_release(NULL);
  h = create();
  skv_destroy(h);
  CHECK(live == 0, "%d allocations left without a hold", live);
  h = create();
  CHECK(skv_output_hold(h, &a) == SKV_OK, "hold");
  skv_output_release(a);
  CHECK(live == all && skv_run(h, query) == SKV_OK, "a released hold frees nothing of the handle");
  skv_destroy(h);
  CHECK(live == 0, "%d allocations left", live);
}

/* A run whose launch fails binds nothing: neither its own query, which no
 * kernel stored, nor the one before it. */
static void failed_run(void) {
  void *h = create();
  CHECK(skv_enqueue(h) == SKV_ESTATE, "enqueue without a query");
  CHECK(skv_run(h, NULL) == SKV_EINVAL, "NULL query");
  for (int good = 0; good < 2; ++good) {  /* on the first call, and after a good one */
    if (good) CHECK(skv_run(h, query) == SKV_OK && skv_enqueue(h) == SKV_OK, "good run");
    fail_launch = launches;
    CHECK(skv_run(h, query) == SKV_EHIP, "failing run");
    CHECK(skv_enqueue(h) == SKV_ESTATE, "enqueue after a failed run");
    CHECK(skv_dense_decode(h) == SKV_ESTATE, "dense decode after a failed run");
  }
  CHECK(skv_bind_query(h, query) == SKV_OK && skv_enqueue(h) == SKV_OK &&
            skv_dense_decode(h) == SKV_OK, "bound again");
  skv_destroy(h);
}

int main(int argc, char **argv) {
  static const struct { const char *name; void (*fn)(void); } scenarios[] = {
      {"output_lifetime", output_lifetime},
      {"failed_run", failed_run},
  };
  for (size_t i = 0; i < sizeof scenarios / sizeof scenarios[0]; ++i)
    if (argc == 2 && !strcmp(argv[1], scenarios[i].name)) {
      scenarios[i].fn();
      printf("hip stub driver ok: %s\n", argv[1]);
      fflush(stdout);
      _Exit(0);  /* the runtime underneath never saw a device */
    }
  CHECK(0, "usage: %s SCENARIO", argv[0]);
  return 1;
}
