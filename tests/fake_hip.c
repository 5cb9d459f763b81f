/* A stand-in for the HIP runtime, with which the library's host code runs
 * where there is no GPU: device memory is host memory, every call is done
 * when it returns, a wait takes 0.2 ms, and no kernel does anything but the
 * copies to and from pinned memory.  A launch is refused as HIP refuses it:
 * dynamic LDS above the function's maximum (64 KB until it is set), more than
 * 65536 blocks along y or z, or a name that contains $FAKE_HIP_REFUSE.  Copies
 * and fills of more than 256 MB are not made.  Of k_levels the order of work and
 * barriers is gone through on the tables it is given.  Loaded with RTLD_GLOBAL before
 * libusg.so. */
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

enum { kOk = 0, kInvalid = 1, kUnsupported = 801, kFunctions = 4096 };
typedef struct {
  unsigned x, y, z;
} dim3;

static struct {
  const void *f;
  const char *name;
  size_t lds;
} fn[kFunctions];
static int nfn;
static __thread int last;
static __thread struct {
  dim3 grid, block;
  size_t lds;
  void *stream;
} call;

static int find(const void *f) {
  for (int i = 0; i < nfn; i++)
    if (fn[i].f == f) return i;
  return -1;
}

void **__hipRegisterFatBinary(const void *p) {
  static void *handle;
  (void)p;
  return &handle;
}
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterVar(void) {}
void __hipRegisterFunction(void **h, const void *f, char *dev, const char *name) {
  (void)h, (void)dev;
  if (nfn == kFunctions) abort();
  fn[nfn].f = f;
  fn[nfn].name = name;
  fn[nfn++].lds = 65536;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream) {
  call.grid = grid, call.block = block, call.lds = lds, call.stream = stream;
  return kOk;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream) {
  *grid = call.grid, *block = call.block, *lds = call.lds, *stream = call.stream;
  return kOk;
}

/* place of value k of item c of n (components in pairs, or one array each) */
static size_t place(int k, int n, int c, int paired) {
  return paired ? (size_t)(k / 2) * 2 * n + 2 * (size_t)c + k % 2 : (size_t)k * n + c;
}
static void copy_fields(const char *name, void **a) {
  const size_t first = *(size_t *)a[2];
  const int total = *(int *)a[3], lv = *(int *)a[4], n = *(int *)a[5], paired = *(_Bool *)a[6];
  const int to = strstr(name, "k_to_host") != NULL, single = strstr(name, "k_to_hostIf") != NULL;
  for (int e = 0; e < total; e++) {
    const size_t g = first + e, p = place((int)(g & ((1u << lv) - 1)), n, (int)(g >> lv), paired);
    if (!to)
      (*(double **)a[1])[p] = (*(double **)a[0])[e];
    else
      (*(double **)a[1])[e] = single ? (*(float **)a[0])[p] : (*(double **)a[0])[p];
  }
}
/* k_levels: its groups take the chunks of a case in turn and meet at barriers.
 * Every group has to execute as many as there are levels, and to be past the
 * barrier of a chunk's level, and not past the next one, when it works on it. */
enum { kGroups = 4 };
typedef struct {
  int n;
  const int *pos, *cell, *code, (*chunk)[4], *coff;
  void *rec, *base, *diag, *tbase, *tdiag, *off;
} levels;
static void check(int ok, const char *what) {
  if (ok) return;
  fprintf(stderr, "k_levels: %s\n", what);
  exit(3);
}
static void check_levels(const levels *w, int ncase) {
  for (int c = 0; c < ncase; c++) {
    const int n0 = w->coff[c], n1 = w->coff[c + 1];
    int begun = 0;
    check((n1 - n0) % kGroups == 0, "a case's chunks are no whole rounds");
    for (int i = n0; i < n1; i++) begun += w->chunk[i][3] & 1;
    for (int g = 0; g < kGroups && n0 < n1; g++) {
      int waits = 0;
      for (int i = 0; i < g; i++) waits += w->chunk[n0][3] >> i & 1;
      for (int n = n0 + g; n < n1; n += kGroups) {
        int level = 0;
        for (int i = n0; i <= n; i++) level += w->chunk[i][3] & 1;
        waits += w->chunk[n][3] & 1;
        check(waits == level, "a group works on a chunk of another level");
        for (int i = 1; i < kGroups; i++) waits += w->chunk[n][3] >> i & 1;
      }
      check(waits == begun, "groups meet different numbers of barriers");
    }
  }
}
int hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **a, size_t lds, void *stream) {
  const int i = find(f);
  const char *refuse = getenv("FAKE_HIP_REFUSE");
  (void)block, (void)stream;
  if (i < 0 || lds > fn[i].lds || grid.y > 65536 || grid.z > 65536 || (refuse && *refuse && strstr(fn[i].name, refuse))) return last = kInvalid;
  if (strstr(fn[i].name, "k_to_host") || strstr(fn[i].name, "k_from_host")) copy_fields(fn[i].name, a);
  if (strstr(fn[i].name, "k_levels")) check_levels((const levels *)a[1] + !strstr(fn[i].name, "ELb1E"), grid.x);
  if (strstr(fn[i].name, "k_err_host")) memcpy(*(void **)a[1], *(void **)a[0], 2 * sizeof(int));
  return kOk;
}
int hipFuncSetAttribute(const void *f, int attr, int value) {
  const int i = find(f);
  (void)attr;
  if (i < 0 || value < 0 || value > 163840) return last = kInvalid;
  fn[i].lds = value;
  return kOk;
}

int hipGetLastError(void) {
  const int e = last;
  last = kOk;
  return e;
}
const char *hipGetErrorString(int e) { return e == kInvalid ? "invalid argument" : "error"; }
int hipGetDeviceCount(int *n) { return *n = 1, kOk; }
int hipGetDevice(int *d) { return *d = 0, kOk; }
int hipDeviceGetAttribute(int *v, int attr, int dev) {
  (void)attr, (void)dev;
  return *v = 163840, kOk;
}
int hipDeviceSynchronize(void) { return kOk; }

int hipMalloc(void **p, size_t n) { return *p = calloc(n ? n : 1, 1), *p ? kOk : 2; }
int hipFree(void *p) { return free(p), kOk; }
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  (void)flags;
  *p = malloc(n);
  if (*p) memset(*p, 0xff, n); /* nothing says that new memory is clear */
  return *p ? kOk : 2;
}
int hipHostFree(void *p) { return free(p), kOk; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
  (void)kind;
  if (n && n <= 1u << 28) memcpy(d, s, n);
  return kOk;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
  (void)stream;
  return hipMemcpy(d, s, n, kind);
}
int hipMemsetAsync(void *d, int v, size_t n, void *stream) {
  (void)stream;
  if (n <= 1u << 28) memset(d, v, n);
  return kOk;
}

int hipStreamCreate(void **s) { return *s = malloc(1), kOk; }
int hipStreamDestroy(void *s) { return free(s), kOk; }
int hipStreamSynchronize(void *s) {
  (void)s;
  return usleep(200), kOk;
}
int hipStreamBeginCapture(void *s, int mode) {
  (void)s, (void)mode;
  return last = kUnsupported;
}
int hipEventCreate(void **e) { return *e = malloc(1), kOk; }
int hipEventCreateWithFlags(void **e, unsigned flags) {
  (void)flags;
  return hipEventCreate(e);
}
int hipEventDestroy(void *e) { return free(e), kOk; }
int hipEventRecord(void *e, void *s) {
  (void)e, (void)s;
  return kOk;
}
int hipEventSynchronize(void *e) {
  (void)e;
  return usleep(200), kOk;
}
