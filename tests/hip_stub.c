/*
 * hip_stub.c -- the HIP runtime and kernel launchers that host/bf_plan.c,
 * host/bf_batch.c and host/xc_plan.c call, without a GPU: device memory is host
 * memory, launches and stream operations are lines of a log.  Linked with those
 * files by tests/test_plan_host.py in place of libamdhip64 and the kernels.
 */
#define _GNU_SOURCE
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include "../dsa110-xengine_amd/csrc/bf_launch.h"

/* ---- what a test sets and reads ------------------------------------------- */
size_t stub_psum_bytes, stub_packed_bytes;   /* of every shape */
int stub_fused_slices;
int stub_fail_launch;                        /* the next beamforming launch fails */
int stub_slow_copies;                        /* host-to-device copies give other threads time */
void *stub_capturing;                        /* the stream that is being captured */
long stub_live;                              /* bytes allocated */
char *stub_psum;                             /* where the last launch was given its sums */
int stub_torn;                               /* weight launches whose arguments were of two calls */

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static char text[1 << 16];
static size_t at;
static int id_of(const void *p, int *n, const void *seen[64]) {
  for (int i = 0; i < *n; i++)
    if (seen[i] == p) return i;
  seen[*n] = p;
  return (*n)++;
}
static const void *streams[64], *events[64];
static int nstream, nevent;
static int sid(const void *s) { return id_of(s, &nstream, streams); }
static int eid(const void *e) { return id_of(e, &nevent, events); }
static void put(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  at += vsnprintf(text + at, sizeof(text) - at, fmt, ap);
  va_end(ap);
}
const char *stub_log(void) { return text; }
void stub_reset(void) { at = 0; text[0] = 0; }

/* ---- runtime ---------------------------------------------------------------- */
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipSetDevice(int d) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return "stub"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
  size_t *m = calloc(1, n + 64);
  m[0] = n;
  __atomic_fetch_add(&stub_live, (long)n, __ATOMIC_SEQ_CST);
  memset((char *)m + 64, 0xA5, n);           /* device memory holds anything */
  *p = (char *)m + 64;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  size_t *m = (size_t *)((char *)p - 64);
  __atomic_fetch_sub(&stub_live, (long)m[0], __ATOMIC_SEQ_CST);
  free(m);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  for (size_t i = 0; i < n; i += 4096) {
    memcpy((char *)d + i, (const char *)s + i, n - i < 4096 ? n - i : 4096);
    if (stub_slow_copies && k == hipMemcpyHostToDevice) usleep(200);
  }
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t s) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { *s = malloc(8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
  *c = (void *)s == stub_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) { *g = malloc(8); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *n, char *b, size_t z) {
  *e = malloc(8);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { free(e); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { free(g); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = malloc(8); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { *ms = 1.f; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  pthread_mutex_lock(&lock);
  put("record %d %d\n", sid(s), eid(e));
  pthread_mutex_unlock(&lock);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) {
  pthread_mutex_lock(&lock);
  put("wait %d %d\n", sid(s), eid(e));
  pthread_mutex_unlock(&lock);
  return hipSuccess;
}

/* ---- launchers ---------------------------------------------------------------- */
static char scratch[64];
size_t bfk_scratch_bytes(void) { return 8u << 20; }
int bfk_scratch_init(int device, void **p) { *p = scratch; return 0; }
const char *bfk_last_error(void) { return "stub"; }
size_t bfk_wfrag_bytes(const bfk_dims *d) { return 64; }
size_t bfk_wscale_bytes(const bfk_dims *d) { return 64; }
size_t bfk_bpart_bytes(const bfk_dims *d) { return 64; }
size_t bfk_psum_bytes(const bfk_dims *d) { return stub_psum_bytes; }
size_t bfk_packed_bytes(const bfk_dims *d) { return stub_packed_bytes; }
int bfk_pack_block(const bfk_dims *d) { return stub_packed_bytes && !d->pinned; }
int bfk_variant_supported(const bfk_dims *d, int v) { return v != 1; }
int bfk_spread_tiles(const bfk_dims *d) { return stub_psum_bytes != 0; }
int bfk_unset_differs(const bfk_dims *d) { return stub_psum_bytes != 0; }
int bfk_weights(const bfk_dims *d, const float *pos, const float *cal, const double *freqs, const double *theta, void *wf,
                float *ws, void *s) {
  /* a test's call holds one value everywhere */
  const float v = cal[0];
  int torn = 0;
  for (long i = 0; i < (long)d->nant * d->ncal * 4; i++) torn |= cal[i] != v;
  for (int i = 0; i < d->nchan; i++) torn |= (float)freqs[i] != v;
  for (int i = 0; i < d->nbeam; i++) torn |= (float)theta[i] != v;
  for (int i = 0; i < d->nant; i++) torn |= pos[i] != v;
  __atomic_fetch_add(&stub_torn, torn, __ATOMIC_SEQ_CST);
  return 0;
}
int bfk_beamform(const bfk_dims *d, const uint8_t *in, const void *wf, const float *ws, const float *sc, uint8_t *out,
                 float *power, float *bpart, float *beam_power, void *psum, int *summed, void *packed, void *s) {
  const int fused = !packed && !d->pinned && beam_power && psum && stub_psum_bytes;
  pthread_mutex_lock(&lock);
  stub_psum = psum;
  put("launch %d %s\n", sid(s), packed ? "packed" : fused ? "sums" : "plain");
  const int fail = stub_fail_launch;
  stub_fail_launch = 0;
  pthread_mutex_unlock(&lock);
  *summed = fused;
  return fail ? -3 : 0;
}
int bfk_stuff(const bfk_dims *d, const uint8_t *in, const float *sc, uint8_t *out, float *power, float *bpart, void *s) {
  return 0;
}
int bfk_beam_power(const bfk_dims *d, const float *bpart, float *bp, void *s) {
  pthread_mutex_lock(&lock);
  put("power %d\n", sid(s));
  pthread_mutex_unlock(&lock);
  return 0;
}
int bfk_batch_prepare(const bfk_dims *d, const bfk_batch_bufs *b, int n, void **h) { *h = malloc(8); return 0; }
int bfk_batch_launch(void *h, void *s) { return 0; }
int bfk_batch_launches(void *h) { return 2; }
void bfk_batch_free(void *h) { free(h); }

size_t bfk_xcorr_vis_bytes(int nant, int nchan) { return 64; }
size_t bfk_xcorr_part_bytes(int nant, int nchan, int nslice) { return nslice > 1 ? 64 * (size_t)nslice : 0; }
int bfk_xcorr_default_slices(int nchan, int npkt) { return 1; }
int bfk_xcorr_use_fused(int nant, int nchan, int npkt, int order) { return stub_fused_slices; }
int bfk_xcorr(int nant, int nchan, int npkt, int order, const uint8_t *in, uint8_t *turn, float *part, int nslice,
              int nfused, float *vis, void *s) {
  pthread_mutex_lock(&lock);
  put("xcorr %s\n", nfused ? "fused" : turn ? "turned" : "no turned copy");
  pthread_mutex_unlock(&lock);
  return nfused || turn ? 0 : -1;
}
