/*
 * test_batches.c -- batches of jobs in square tiles and in sub-tiles on the
 * CPU fake of the HIP layer (xg_hip_fake.c), built with AddressSanitizer and
 * UBSan.  TEST INFRASTRUCTURE ONLY.
 *
 * Scenarios, named on the command line:
 *   retry   a batch whose launch or graph fails leaves every integration as
 *           it was, and the same batch again is exact; a batch is one launch
 *   cycle   a graph-knob batch over three input buffers, storing and adding,
 *           is captured once per buffer and state and replayed after that
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

static void fill(int8_t *x, size_t n, unsigned seed) {
  uint64_t s = 0x9E3779B97F4A7C15ull * (seed + 1);
  for (size_t i = 0; i < n; ++i) {
    s ^= s << 13, s ^= s >> 7, s ^= s << 17;
    x[i] = (int8_t)((int)(s % 41) - 20);
  }
}

static XGPUAmdEngine *engine(unsigned ns, unsigned nf) {
  XGPUAmdConfig c;
  memset(&c, 0, sizeof c);
  c.npol = 2;
  c.nstation = ns;
  c.nfrequency = nf;
  c.compute_type = XGPU_INT8;
  c.matrix_order = REGISTER_TILE_TRIANGULAR_ORDER;
  XGPUAmdEngine *e = NULL;
  CHECK(xgpuAmdCreate(&e, &c) == XGPU_OK, "create");
  return e;
}

/* Many channels of few stations (faster in sub-tiles) and stations that fill
 * square tiles: a batch of both kinds. */
enum { NE = 2, NT = 1 };
static const unsigned NS[NE] = {32, 128}, NF[NE] = {1600, 80};

static void graph_knob(XGPUAmdEngine *e, int on) {
  XGPUAmdTuning t;
  memset(&t, 0, sizeof t);
  t.graph = on ? 1 : 2;
  CHECK(xgpuAmdSetTuning(e, &t) == XGPU_OK, "graph knob");
}

static int32_t *dump(XGPUAmdEngine *e, unsigned ns, unsigned nf) {
  int32_t *v = malloc(sizeof(int32_t) * nf * ns * (ns + 1) / 2 * 8);
  CHECK(xgpuAmdDump(e, v, XGPU_DUMP_TRIANGULAR) == XGPU_OK, "dump");
  return v;
}

static void retry(void) {
  static const struct {
    const char *category;
    int after, graph, own_stream;
  } cases[] = {{"launch", 0, 0, 1}, {"launch", 1, 0, 1}, {"launch", 1, 0, 0},
               {"graph", 0, 1, 1}, {"graph", 1, 1, 0}, {"graph", 3, 1, 1}, {"launch", 1, 1, 1}};
  XGPUAmdEngine *e[NE], *other = engine(4, 1);
  void *d[NE];
  int32_t *one[NE];
  XGPUAmdBatchItem items[NE];
  for (int i = 0; i < NE; ++i) {
    const size_t nb = (size_t)NT * NF[i] * NS[i] * 4;
    int8_t *x = malloc(nb);
    fill(x, nb, (unsigned)i);
    e[i] = engine(NS[i], NF[i]);
    CHECK(xgpuAmdMalloc(&d[i], nb) == XGPU_OK && xgpuAmdMemcpy(d[i], x, nb, XGPU_H2D) == XGPU_OK, "upload");
    free(x);
    CHECK(xgpuAmdCorrelate(e[i], d[i], NT) == XGPU_OK, "one block");
    one[i] = dump(e[i], NS[i], NF[i]);
    items[i] = (XGPUAmdBatchItem){e[i], d[i], NT};
  }
  xgh_fake_reset();
  CHECK(xgpuAmdCorrelateBatch(items, NE, NULL) == XGPU_OK, "batch");
  CHECK(xgh_fake_calls("launch") == 1, "%lld launches of a batch", xgh_fake_calls("launch"));
  int failed = 0;
  for (size_t c = 0; c < sizeof cases / sizeof cases[0]; ++c) {
    void *stream = cases[c].own_stream ? NULL : xgpuAmdStream(other);
    graph_knob(e[0], cases[c].graph);
    for (int i = 0; i < NE; ++i) xgpuAmdClear(e[i]);
    CHECK(xgpuAmdCorrelateBatch(items, NE, stream) == XGPU_OK, "first batch");
    xgh_fake_reset();
    xgh_fake_fail(cases[c].category, cases[c].after);
    int blocks = 2;
    if (xgpuAmdCorrelateBatch(items, NE, stream) != XGPU_OK) {
      ++failed;
      for (int i = 0; i < NE; ++i)
        CHECK(xgpuAmdSamples(e[i]) == NT, "case %zu: engine %d counts %llu samples", c, i,
              xgpuAmdSamples(e[i]));
      xgh_fake_reset();
      CHECK(xgpuAmdCorrelateBatch(items, NE, stream) == XGPU_OK, "retry");
    }
    xgh_fake_reset();
    for (int i = 0; i < NE; ++i) {
      int32_t *v = dump(e[i], NS[i], NF[i]);
      const size_t n = (size_t)NF[i] * NS[i] * (NS[i] + 1) / 2 * 8;
      for (size_t k = 0; k < n; ++k)
        CHECK(v[k] == blocks * one[i][k], "case %zu (%s #%d) engine %d value %zu: %d, one block %d", c,
              cases[c].category, cases[c].after, i, k, v[k], one[i][k]);
      free(v);
    }
  }
  CHECK(failed >= 3, "%d faults reached the batch", failed);
  for (int i = 0; i < NE; ++i) {
    xgpuAmdDestroy(e[i]);
    xgpuAmdFree(d[i]);
    free(one[i]);
  }
  xgpuAmdDestroy(other);
  CHECK(xgh_fake_live_allocations() == 0, "leaked %lld", xgh_fake_live_allocations());
  printf("ok retry\n");
}

static void cycle(void) {
  enum { BUFS = 3, PASSES = 3 };
  XGPUAmdEngine *e[NE];
  void *d[NE][BUFS];
  for (int i = 0; i < NE; ++i) {
    const size_t nb = (size_t)NT * NF[i] * NS[i] * 4;
    e[i] = engine(NS[i], NF[i]);
    for (int b = 0; b < BUFS; ++b) {
      CHECK(xgpuAmdMalloc(&d[i][b], nb) == XGPU_OK, "malloc");
      memset(d[i][b], b + 1, nb);
    }
  }
  graph_knob(e[0], 1);
  for (int p = 0; p < PASSES; ++p) {
    xgh_fake_reset();
    for (int b = 0; b < BUFS; ++b) {
      XGPUAmdBatchItem items[NE];
      for (int i = 0; i < NE; ++i) {
        items[i] = (XGPUAmdBatchItem){e[i], d[i][b], NT};
        xgpuAmdClear(e[i]);
      }
      for (int k = 0; k < 2; ++k) CHECK(xgpuAmdCorrelateBatch(items, NE, NULL) == XGPU_OK, "batch");
    }
    /* one replay a batch; the first pass begins and ends one capture each too */
    const long long want = 2 * BUFS * (p == 0 ? 3 : 1);
    CHECK(xgh_fake_calls("graph") == want, "pass %d: %lld graph calls, expected %lld", p,
          xgh_fake_calls("graph"), want);
  }
  for (int i = 0; i < NE; ++i) {
    xgpuAmdDestroy(e[i]);
    for (int b = 0; b < BUFS; ++b) xgpuAmdFree(d[i][b]);
  }
  CHECK(xgh_fake_live_allocations() == 0, "leaked %lld", xgh_fake_live_allocations());
  printf("ok cycle\n");
}

int main(int argc, char **argv) {
  for (int i = 1; i < argc; ++i) {
    if (!strcmp(argv[i], "retry")) retry();
    else if (!strcmp(argv[i], "cycle")) cycle();
    else return 2;
  }
  return 0;
}
