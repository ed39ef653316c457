/*
 * A caller of fof_link_gpu_noalloc that counts what the library asks the HIP
 * runtime to make.  The program defines the runtime's entry points that
 * allocate or create; the library's calls resolve to these (the executable
 * comes first in symbol lookup), which count while `counting` is set and go
 * on to the runtime.  On a fresh context: one fof_link_gpu_noalloc call, its
 * count, then a fof_link_gpu_ex call on the same input, whose outputs must be
 * the same and which allocates (so the counting works).  Output, a line each:
 * "noalloc <count> <names>" and "ex <count> <names>".
 */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "fof_gpu.h"

static int counting, count;
static char names[4096];

static void *made(const char *name) {
  if (counting) {
    count++;
    if (strlen(names) + strlen(name) + 2 < sizeof names) strcat(strcat(names, " "), name);
  }
  return dlsym(RTLD_NEXT, name);
}

#define WRAP(name, args, pass) \
  int name args { return ((int(*) args)made(#name)) pass; }
WRAP(hipMalloc, (void **p, size_t n), (p, n))
WRAP(hipExtMallocWithFlags, (void **p, size_t n, unsigned f), (p, n, f))
WRAP(hipMallocAsync, (void **p, size_t n, void *s), (p, n, s))
WRAP(hipMallocManaged, (void **p, size_t n, unsigned f), (p, n, f))
WRAP(hipHostMalloc, (void **p, size_t n, unsigned f), (p, n, f))
WRAP(hipHostRegister, (void *p, size_t n, unsigned f), (p, n, f))
WRAP(hipFree, (void *p), (p))
WRAP(hipHostFree, (void *p), (p))
WRAP(hipStreamCreate, (void **s), (s))
WRAP(hipStreamCreateWithFlags, (void **s, unsigned f), (s, f))
WRAP(hipEventCreate, (void **e), (e))
WRAP(hipEventCreateWithFlags, (void **e, unsigned f), (e, f))
WRAP(hipStreamBeginCapture, (void *s, int m), (s, m))
WRAP(hipGraphInstantiate, (void **e, void *g, void **n, char *b, size_t z), (e, g, n, b, z))
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
  void *host = malloc(32 * n);
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

  fof_ctx *ctx;
  CHECK(fof_ctx_create(0, &ctx));
  fof_particles_v1 P;
  memset(&P, 0, sizeof P);
  P.version = FOF_ABI_VERSION;
  P.location = FOF_MEM_DEVICE;
  P.n = n;
  P.stride = 32, P.off_id = 0, P.off_pos = 8, P.off_vel = 20;
  void *in;
  CHECK(hipMalloc(&in, 32 * n));
  CHECK(hipMemcpy(in, host, 32 * n, 1));
  P.base = in;

  uint32_t *out[2];
  uint64_t nh[2];
  for (int k = 0; k < 2; k++) {
    void *next, *label, *minid, *halos, *moments;
    CHECK(hipMalloc(&next, 4 * n));
    CHECK(hipMalloc(&label, 4 * n));
    CHECK(hipMalloc(&minid, 8 * n));
    CHECK(hipMalloc(&halos, sizeof(fof_halo_v1) * n));
    CHECK(hipMalloc(&moments, sizeof(fof_moments_v1) * n));
    fof_outputs_v1 o;
    memset(&o, 0, sizeof o);
    o.version = FOF_ABI_VERSION;
    o.location = FOF_MEM_DEVICE;
    o.next = next, o.label = label, o.minid = minid, o.halos = halos, o.moments = moments;
    o.halo_cap = n;
    count = 0, names[0] = 0, counting = 1;
    int rc = k ? fof_link_gpu_ex(ctx, &P, &vol, 1, NULL, &o)
               : fof_link_gpu_noalloc(ctx, &P, &vol.domain, NULL, &o);
    counting = 0;
    CHECK(rc);
    printf("%s %d%s\n", k ? "ex" : "noalloc", count, names);
    nh[k] = o.nhalos;
    out[k] = malloc(16 * n);
    CHECK(hipMemcpy(out[k], next, 4 * n, 2));
    CHECK(hipMemcpy(out[k] + n, label, 4 * n, 2));
    CHECK(hipMemcpy(out[k] + 2 * n, minid, 8 * n, 2));
  }
  if (nh[0] != nh[1] || nh[0] == 0) return printf("halos %d %d\n", (int)nh[0], (int)nh[1]), 1;
  if (memcmp(out[0], out[1], 16 * n)) return printf("outputs differ\n"), 1;
  fof_ctx_destroy(ctx);
  return 0;
}
