/*
 * Which calls overlap the link kernels of a pipeline: the program defines the
 * HIP runtime's hipStreamWaitEvent, counts the library's calls to it and goes
 * on to the runtime.  With one volume and one pipeline a call makes none
 * unless it forks the link kernels to the pipeline's side stream.  Each line:
 * "<options> <count>", every call on a context of its own.
 */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "fof_gpu.h"

static int count;

int hipStreamWaitEvent(void *s, void *e, unsigned f) {
  count++;
  return ((int (*)(void *, void *, unsigned))dlsym(RTLD_NEXT, "hipStreamWaitEvent"))(s, e, f);
}
int hipMalloc(void **, size_t);
int hipMemcpy(void *, const void *, size_t, int);

#define CHECK(x)                                           \
  do {                                                     \
    int rc_ = (x);                                         \
    if (rc_) return printf("%s: %d\n", #x, rc_), 1;        \
  } while (0)

int main(void) {
  const uint64_t n = 24389;
  const double box = 29.0;
  fof_gen_v1 g = {3, n, box, 40, 0.5, 20.0, 2000.0, 1.9, 0.05, 300.0, 0.99, 0.0, 0.0, 0.0};
  void *host = malloc(32 * n), *in, *next, *label;
  CHECK(fof_gen_host(&g, host));
  fof_volume_v1 vol;
  memset(&vol, 0, sizeof vol);
  vol.n = n;
  for (int d = 0; d < 3; d++) {
    vol.domain.rmax[d] = vol.domain.rmax_buff[d] = box;
    vol.domain.lcell[d] = 1.0;
  }
  vol.domain.linklength = 0.2;
  vol.domain.nphalomin = 20;
  CHECK(hipMalloc(&in, 32 * n));
  CHECK(hipMalloc(&next, 4 * n));
  CHECK(hipMalloc(&label, 4 * n));
  CHECK(hipMemcpy(in, host, 32 * n, 1));
  fof_particles_v1 P;
  memset(&P, 0, sizeof P);
  P.version = FOF_ABI_VERSION;
  P.location = FOF_MEM_DEVICE;
  P.n = n;
  P.base = in;
  P.stride = 32, P.off_id = 0, P.off_pos = 8, P.off_vel = 20;
  const struct {
    const char *name;
    uint32_t flags;
  } calls[] = {{"eager", 0},
               {"timed", FOF_OPT_TIMING},
               {"graph", FOF_OPT_GRAPH},
               {"tuned", FOF_OPT_AUTOTUNE},
               {"tuned+graph", FOF_OPT_AUTOTUNE | FOF_OPT_GRAPH},
               {"tuned+timed", FOF_OPT_AUTOTUNE | FOF_OPT_TIMING}};
  for (int k = 0; k < 6; k++) {
    fof_ctx *ctx;
    CHECK(fof_ctx_create(0, &ctx));
    fof_opts_v1 o;
    memset(&o, 0, sizeof o);
    o.version = FOF_ABI_VERSION;
    o.flags = calls[k].flags;
    fof_outputs_v1 out;
    memset(&out, 0, sizeof out);
    out.version = FOF_ABI_VERSION;
    out.location = FOF_MEM_DEVICE;
    out.next = next, out.label = label;
    fof_stats_v1 st;
    out.stats = &st;
    count = 0;
    CHECK(fof_link_gpu_ex(ctx, &P, &vol, 1, &o, &out));
    printf("%s %d\n", calls[k].name, count);
    fof_ctx_destroy(ctx);
  }
  return 0;
}
