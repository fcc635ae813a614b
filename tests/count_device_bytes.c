/* Stands in for the HIP runtime calls that creating a context makes, where
 * there is no GPU: hands out addresses that nothing dereferences, adds up the
 * bytes asked for, and does nothing else.  Preloaded by test_footprint.py. */
#include <stdlib.h>

static long long total;
static int count;
static long long sizes[4096];

long long counted_bytes(void) { return total; }
int counted_of_size(long long bytes) {
  int n = 0;
  for (int i = 0; i < count; ++i) n += sizes[i] == bytes;
  return n;
}
void counted_clear(void) { total = count = 0; }

int hipMalloc(void **p, size_t n) {
  *p = (void *)(0x100000000LL + 256LL * count);
  total += (long long)n;
  if (count < 4096) sizes[count++] = (long long)n;
  return 0;
}
int hipFree(void *p) { return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) {
  *p = calloc(1, n);
  return *p ? 0 : 2;
}
int hipHostFree(void *p) {
  free(p);
  return 0;
}
int hipMemset(void *p, int v, size_t n) { return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { return 0; }
int hipGetDevice(int *d) {
  *d = 0;
  return 0;
}
int hipGetLastError(void) { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) {
  *s = (void *)1;
  return 0;
}
int hipStreamSynchronize(void *s) { return 0; }
int hipStreamDestroy(void *s) { return 0; }
int hipEventDestroy(void *e) { return 0; }

typedef struct { unsigned x, y, z; } dim3_t;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void *s) { return 0; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *lds, void **s) {
  g->x = g->y = g->z = b->x = b->y = b->z = 1;
  *lds = 0;
  *s = 0;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t lds, void *s) { return 0; }
