/*
 * test_routes.c -- which kernels the host runtime launches, on the CPU fake of
 * the HIP layer (xg_hip_fake.c), built with AddressSanitizer and UBSan.  TEST
 * INFRASTRUCTURE ONLY.
 *
 * One scenario per run, named on the command line; the trace log (XGPU_TRACE)
 * shows the launches, which tests/test_routes.py checks:
 *   tuning DIR   a tuning that is read and set again, an autotuner's, a cached
 *                one: the library's choice of tiles stays or goes as it should
 *   slices       blocks cut into slices, plain and swizzled, int8 and FP32: results,
 *                and every launch of a block failing in turn
 *   replay       a long FP32 block (two X-engine launches) captured and replayed
 *   shapes       one block that starts an integration and one that adds to it, by shape
 * Prints "ok <scenario>"; exits nonzero on the first failure.
 */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "xgpu_amd.h"

void xgh_fake_fail(const char *category, int after);
void xgh_fake_reset(void);
long long xgh_fake_live_allocations(void);
long long xgh_fake_calls(const char *category);

#define CHECK(cond, ...)                                                   \
  do {                                                                     \
    if (!(cond)) {                                                         \
      fprintf(stderr, "FAIL %s:%d: %s: ", __FILE__, __LINE__, #cond);      \
      fprintf(stderr, __VA_ARGS__);                                        \
      fprintf(stderr, "\n");                                               \
      exit(1);                                                             \
    }                                                                      \
  } while (0)
#define OK(call) CHECK((call) == XGPU_OK, "%s", xgpuAmdLastError())

static XGPUAmdEngine *engine(unsigned ns, unsigned nf, unsigned compute, unsigned swizzle, unsigned ntime) {
  XGPUAmdConfig c;
  memset(&c, 0, sizeof c);
  c.npol = 2;
  c.nstation = ns;
  c.nfrequency = nf;
  c.ntime = ntime;
  c.compute_type = compute;
  c.matrix_order = REAL_IMAG_TRIANGULAR_ORDER;
  c.time_swizzle = swizzle;
  XGPUAmdEngine *e = NULL;
  OK(xgpuAmdCreate(&e, &c));
  return e;
}

static int8_t *bytes(size_t n, unsigned seed, int range) {
  int8_t *x = malloc(n);
  uint64_t s = 0x9E3779B97F4A7C15ull * (seed + 1);
  for (size_t i = 0; i < n; ++i) {
    s ^= s << 13, s ^= s >> 7, s ^= s << 17;
    x[i] = (int8_t)((int)(s % (2 * (unsigned)range + 1)) - range);
  }
  return x;
}

static void *upload(const void *x, size_t n) {
  void *d = NULL;
  OK(xgpuAmdMalloc(&d, n));
  OK(xgpuAmdMemcpy(d, x, n, XGPU_H2D));
  return d;
}

static void step(XGPUAmdEngine *e, const void *d, unsigned nt) {
  OK(xgpuAmdClear(e));
  OK(xgpuAmdCorrelate(e, d, nt));
}

static void reread(XGPUAmdEngine *e) {
  XGPUAmdTuning t;
  OK(xgpuAmdGetTuning(e, &t));
  t.wg_per_cu = 1;
  t.graph = 2;
  OK(xgpuAmdSetTuning(e, &t));
}

static void tuning(const char *dir) {
  enum { NS = 4, NF = 1, NT = 6000, HOST = 128 }; /* HOST: samples of a host-path call */
  int8_t *x = bytes(NT * NF * NS * 4, 1, 20);
  void *d = upload(x, NT * NF * NS * 4);
  char path[512];
  XGPUAmdTuning t, best;
  for (int swizzle = 0; swizzle <= 4; swizzle += 4) {
    XGPUAmdEngine *e = engine(NS, NF, XGPU_INT8, swizzle, 0);
    step(e, d, NT); /* the library's choice */
    reread(e);
    step(e, d, NT); /* the same */
    memset(&t, 0, sizeof t);
    t.kernel = 2, t.staging = 2, t.stage = 32;
    OK(xgpuAmdSetTuning(e, &t));
    step(e, d, NT); /* asked for: square tiles */
    reread(e);
    step(e, d, NT); /* the same */
    xgpuAmdDestroy(e);
  }
  /* the autotuners' results, set again and on another engine */
  XGPUAmdEngine *e = engine(NS, NF, XGPU_INT8, 0, HOST), *f = engine(NS, NF, XGPU_INT8, 0, HOST);
  OK(xgpuAmdAutotuneHost(e, x, 0, 1, NULL, &best, NULL));
  reread(e); /* graph replay off, whichever was faster */
  step(e, d, NT); /* the library's choice: the time pipe is all that was tuned */
  best.graph = 2;
  OK(xgpuAmdSetTuning(f, &best));
  step(f, d, NT);
  xgpuAmdDestroy(f);
  memset(&t, 0, sizeof t);
  t.kernel = 2, t.staging = 2, t.stage = 32;
  OK(xgpuAmdSetTuning(e, &t));
  OK(xgpuAmdAutotuneHost(e, x, 0, 1, NULL, NULL, NULL));
  reread(e);
  step(e, d, NT); /* square tiles as before */
  xgpuAmdDestroy(e);
  /* cached lines: one that names square tiles, one that leaves them to the library */
  for (int kernel = 2; kernel >= 0; kernel -= 2) {
    snprintf(path, sizeof path, "%s/tuning%d.txt", dir, kernel);
    FILE *o = fopen(path, "w");
    CHECK(o, "%s", path);
    fprintf(o, "cpu fake of gfx950|%d|%d|%d|%d|2|2|%d|32|2|%d|1|2|0.01\n", NS, NF, NT, XGPU_INT8, kernel, HOST);
    fclose(o);
    e = engine(NS, NF, XGPU_INT8, 0, HOST);
    OK(xgpuAmdLoadTuning(e, path, NT));
    step(e, d, NT);
    xgpuAmdDestroy(e);
  }
  xgpuAmdFree(d);
  free(x);
}

/* Sums of blocks x (plain layout), taken by an engine that names the general kernel. */
static void *general(unsigned ns, unsigned nf, unsigned compute, const void *x, unsigned nt, int blocks,
                     size_t bytes) {
  XGPUAmdEngine *e = engine(ns, nf, compute, 0, 0);
  XGPUAmdTuning t;
  memset(&t, 0, sizeof t);
  t.kernel = 1;
  OK(xgpuAmdSetTuning(e, &t));
  for (int b = 0; b < blocks; ++b) OK(xgpuAmdCorrelate(e, x, nt));
  void *v = malloc(bytes);
  OK(xgpuAmdDump(e, v, 0));
  xgpuAmdDestroy(e);
  return v;
}

static void slices(void) {
  enum { NS = 4, NF = 1, BYTES = NF * NS * (NS + 1) / 2 * 8 * 4 };
  static const struct {
    unsigned compute, swizzle, nt;
    int launches, adds; /* of a block that starts an integration; of one that adds */
  } cases[] = {{XGPU_INT8, 0, 6001, 2, 2}, {XGPU_INT8, 4, 6000, 2, 2}, {XGPU_FLOAT32, 0, 6000, 3, 1}};
  for (size_t c = 0; c < sizeof cases / sizeof cases[0]; ++c) {
    const unsigned nt = cases[c].nt;
    const size_t nb = (size_t)nt * NF * NS * 4;
    int8_t *x = bytes(nb, 7 + (unsigned)c, 100);
    void *d = upload(x, nb), *in = d;
    if (cases[c].swizzle) {
      OK(xgpuAmdMalloc(&in, nb));
      OK(xgpuAmdSwizzleInput(in, d, NS, NF, nt, 0, NULL));
    }
    void *ref[3], *got = malloc(BYTES);
    for (int b = 1; b <= 2; ++b) ref[b] = general(NS, NF, cases[c].compute, d, nt, b, BYTES);
    XGPUAmdEngine *e = engine(NS, NF, cases[c].compute, cases[c].swizzle, 0);
    for (int b = 1; b <= 2; ++b) {
      const int n = b == 1 ? cases[c].launches : cases[c].adds;
      for (int fail = 0; fail < n; ++fail) {
        xgh_fake_reset();
        xgh_fake_fail("launch", fail);
        CHECK(xgpuAmdCorrelate(e, in, nt) == XGPU_CUDA_ERROR, "case %zu block %d launch %d", c, b, fail);
        CHECK(xgpuAmdSamples(e) == (unsigned long long)(b - 1) * nt, "case %zu: samples", c);
        xgh_fake_reset();
        if (b == 1) continue;
        OK(xgpuAmdDump(e, got, 0));
        CHECK(!memcmp(got, ref[1], BYTES), "case %zu: launch %d left something behind", c, fail);
      }
      xgh_fake_reset();
      OK(xgpuAmdCorrelate(e, in, nt));
      CHECK(xgh_fake_calls("launch") == n, "case %zu block %d: %lld launches", c, b, xgh_fake_calls("launch"));
      OK(xgpuAmdDump(e, got, 0));
      CHECK(!memcmp(got, ref[b], BYTES), "case %zu: %d blocks", c, b);
    }
    xgpuAmdDestroy(e);
    if (in != d) xgpuAmdFree(in);
    xgpuAmdFree(d);
    free(x);
    free(got);
    free(ref[1]);
    free(ref[2]);
  }
}

static void replay(void) {
  enum { NS = 4, NF = 1, NT = 600 };
  int8_t *x = bytes(NT * NF * NS * 4, 3, 20);
  void *d = upload(x, NT * NF * NS * 4);
  XGPUAmdEngine *e = engine(NS, NF, XGPU_FLOAT32, 0, 0);
  XGPUAmdTuning t;
  memset(&t, 0, sizeof t);
  t.graph = 1;
  OK(xgpuAmdSetTuning(e, &t));
  step(e, d, NT);
  step(e, d, NT);
  xgpuAmdDestroy(e);
  xgpuAmdFree(d);
  free(x);
}

static void shapes(void) {
  static const struct {
    unsigned ns, nf, nt, compute;
  } s[] = {
      /* complex-plane kernel or sub-tiles: stations, samples, channels */
      {2, 520, 4, XGPU_INT8}, {6, 520, 64, XGPU_INT8}, {6, 520, 130, XGPU_INT8}, {14, 520, 4, XGPU_INT8},
      {16, 520, 65, XGPU_INT8}, {18, 520, 4, XGPU_INT8}, {14, 512, 4, XGPU_INT8}, {66, 512, 1, XGPU_INT8},
      {74, 512, 1, XGPU_INT8}, {6, 256, 4, XGPU_INT8},
      {6, 520, 4, XGPU_FLOAT32},
      /* square tiles or sub-tiles */
      {16, 2, 64, XGPU_INT8}, {64, 8, 200, XGPU_INT8}, {256, 10, 8, XGPU_INT8}, {130, 130, 1, XGPU_INT8},
      {130, 45, 257, XGPU_INT8},
      /* FP32: exact sums, past them, adding past them */
      {16, 2, 64, XGPU_FLOAT32}, {4, 1, 513, XGPU_FLOAT32}, {4, 1, 512, XGPU_FLOAT32}};
  for (size_t i = 0; i < sizeof s / sizeof s[0]; ++i) {
    const size_t nb = (size_t)s[i].nt * s[i].nf * s[i].ns * 4;
    int8_t *x = bytes(nb, (unsigned)i, 20);
    void *d = upload(x, nb);
    XGPUAmdEngine *e = engine(s[i].ns, s[i].nf, s[i].compute, 0, 0);
    step(e, d, s[i].nt);
    OK(xgpuAmdCorrelate(e, d, s[i].nt));
    xgpuAmdDestroy(e);
    xgpuAmdFree(d);
    free(x);
  }
  /* batches: small arrays of few samples only, and one with a larger array too */
  XGPUAmdEngine *e[3] = {engine(2, 300, XGPU_INT8, 0, 0), engine(6, 300, XGPU_INT8, 0, 0),
                         engine(34, 3, XGPU_INT8, 0, 0)};
  int8_t *x = bytes(4 * 300 * 6 * 4, 1, 20);
  void *d = upload(x, 4 * 300 * 6 * 4);
  XGPUAmdBatchItem items[3] = {{e[0], d, 4}, {e[1], d, 4}, {e[2], d, 4}};
  OK(xgpuAmdCorrelateBatch(items, 2, NULL));
  OK(xgpuAmdCorrelateBatch(items, 3, NULL));
  for (int i = 0; i < 3; ++i) xgpuAmdDestroy(e[i]);
  xgpuAmdFree(d);
  free(x);
}

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  if (!strcmp(argv[1], "tuning") && argc == 3) tuning(argv[2]);
  else if (!strcmp(argv[1], "slices")) slices();
  else if (!strcmp(argv[1], "replay")) replay();
  else if (!strcmp(argv[1], "shapes")) shapes();
  else return 2;
  CHECK(xgh_fake_live_allocations() == 0, "leaked %lld", xgh_fake_live_allocations());
  printf("ok %s\n", argv[1]);
  return 0;
}
