/*
 * A call that fails between its forks and joins: the program defines the HIP
 * runtime's hipEventRecord and lets one call of it fail (on the host, the
 * kernels already launched run on), and hipStreamSynchronize, which it logs.
 * For the k-th record of a batch over two pipelines, every k: the failing call
 * returns FOF_E_HIP and waits for every stream that it launched on before it
 * does; the next call on the context gives the outputs of the first.  A line
 * each: "<k> <streams waited for>".
 */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "fof_gpu.h"

static int records, fail_at;
static void *waited[64];
static int nwaited;

int hipEventRecord(void *e, void *s) {
  if (++records == fail_at) return 1;
  return ((int (*)(void *, void *))dlsym(RTLD_NEXT, "hipEventRecord"))(e, s);
}
int hipStreamSynchronize(void *s) {
  int k = 0;
  while (k < nwaited && waited[k] != s) k++;
  if (k == nwaited && nwaited < 64) waited[nwaited++] = s;
  return ((int (*)(void *))dlsym(RTLD_NEXT, "hipStreamSynchronize"))(s);
}
int hipMalloc(void **, size_t);
int hipMemcpy(void *, const void *, size_t, int);

#define CHECK(x)                                           \
  do {                                                     \
    int rc_ = (x);                                         \
    if (rc_) return printf("%s: %d\n", #x, rc_), 1;        \
  } while (0)

int main(void) {
  const uint64_t n = 20000;
  const double box = 27.2;
  void *host = malloc(64 * n), *in, *next, *label;
  for (int v = 0; v < 2; v++) {
    fof_gen_v1 g = {3 + v, n, box, 40, 0.5, 20.0, 2000.0, 1.9, 0.05, 300.0, 0.99, 0.0, 0.0, 0.0};
    CHECK(fof_gen_host(&g, (char *)host + 32 * n * v));
  }
  fof_volume_v1 vols[2];
  memset(vols, 0, sizeof vols);
  for (int v = 0; v < 2; v++) {
    vols[v].offset = n * v, vols[v].n = n;
    for (int d = 0; d < 3; d++) {
      vols[v].domain.rmax[d] = vols[v].domain.rmax_buff[d] = box;
      vols[v].domain.lcell[d] = 1.0;
    }
    vols[v].domain.linklength = 0.2;
    vols[v].domain.nphalomin = 20;
  }
  CHECK(hipMalloc(&in, 64 * n));
  CHECK(hipMalloc(&next, 8 * n));
  CHECK(hipMalloc(&label, 8 * n));
  CHECK(hipMemcpy(in, host, 64 * n, 1));
  fof_particles_v1 P;
  memset(&P, 0, sizeof P);
  P.version = FOF_ABI_VERSION;
  P.location = FOF_MEM_DEVICE;
  P.n = 2 * n;
  P.base = in;
  P.stride = 32, P.off_id = 0, P.off_pos = 8, P.off_vel = 20;
  fof_opts_v1 o;
  memset(&o, 0, sizeof o);
  o.version = FOF_ABI_VERSION;
  o.flags = FOF_OPT_NO_HALOS;
  o.pipelines = 2;
  fof_outputs_v1 out;
  memset(&out, 0, sizeof out);
  out.version = FOF_ABI_VERSION;
  out.location = FOF_MEM_DEVICE;
  out.next = next, out.label = label;
  fof_ctx *ctx;
  CHECK(fof_ctx_create(0, &ctx));
  CHECK(fof_link_gpu_ex(ctx, &P, vols, 2, &o, &out));
  uint32_t *first = malloc(16 * n), *again = malloc(16 * n);
  CHECK(hipMemcpy(first, next, 8 * n, 2));
  CHECK(hipMemcpy(first + 2 * n, label, 8 * n, 2));
  records = 0;
  CHECK(fof_link_gpu_ex(ctx, &P, vols, 2, &o, &out));
  const int all = records;
  for (int k = 1; k <= all; k++) {
    records = nwaited = 0, fail_at = k;
    if (fof_link_gpu_ex(ctx, &P, vols, 2, &o, &out) != FOF_E_HIP) return printf("%d: no error\n", k), 1;
    printf("%d %d\n", k, nwaited);
    fail_at = 0;
    CHECK(fof_link_gpu_ex(ctx, &P, vols, 2, &o, &out));
    CHECK(hipMemcpy(again, next, 8 * n, 2));
    CHECK(hipMemcpy(again + 2 * n, label, 8 * n, 2));
    if (memcmp(first, again, 16 * n)) return printf("%d: outputs differ\n", k), 1;
  }
  fof_ctx_destroy(ctx);
  return 0;
}
