/* Stand-in for the HIP runtime, for tests of host code without a GPU: two
 * "devices" whose memory is host memory.  Kernels do nothing, except that
 * k_put_counters copies the counters and puts in the values a test set.
 * Every allocation, launch, fill, stream or event creation and device
 * synchronisation made while another device than fake_expect()'s is current
 * is noted; so is a launch onto a stream of another device. */
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
  unsigned x, y, z;
} dim3_t;
typedef struct {
  int device;
} handle_t;

static _Thread_local int current = 0;
static int expected = -1;
static char notes[65536];
static int n_notes = 0;
static long long allocations[2];

static struct {
  const void* fn;
  char name[256];
} kernels[1024];
static int n_kernels = 0;

static struct {
  long long value;
  int reads;
} forced[64];

void fake_expect(int device) { expected = device; }
int fake_current(void) { return current; }
int fake_notes(char* out, int cap) {
  snprintf(out, (size_t)cap, "%s", notes);
  const int n = n_notes;
  n_notes = 0;
  notes[0] = 0;
  return n;
}
long long fake_allocations(int device) { return allocations[device]; }
/* Counter `slot` reads as `value` for the next `reads` reads. */
void fake_counter(int slot, long long value, int reads) {
  forced[slot].value = value;
  forced[slot].reads = reads;
}

static void note(const char* what, const char* name, int device) {
  if (expected < 0 || device == expected) return;
  const size_t at = strlen(notes);
  snprintf(notes + at, sizeof(notes) - at, "%s%s on device %d, expected %d\n", what, name, device, expected);
  ++n_notes;
}
static handle_t* make(const char* what) {
  note(what, "", current);
  handle_t* h = malloc(sizeof(*h));
  h->device = current;
  return h;
}

int hipSetDevice(int d) {
  current = d;
  return 0;
}
int hipGetDeviceCount(int* n) {
  *n = 2;
  return 0;
}
int hipDeviceGetAttribute(int* v, int attr, int d) {
  (void)attr;
  (void)d;
  *v = 100000;
  return 0;
}
int hipDeviceSynchronize(void) {
  note("hipDeviceSynchronize", "", current);
  return 0;
}
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) {
  (void)e;
  return "fake";
}

int hipMalloc(void** p, size_t n) {
  note("hipMalloc", "", current);
  ++allocations[current];
  *p = calloc(1, n ? n : 1);
  return *p ? 0 : 2;
}
int hipFree(void* p) {
  free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  (void)flags;
  note("hipHostMalloc", "", current);
  *p = calloc(1, n);
  return *p ? 0 : 2;
}
int hipHostFree(void* p) {
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  (void)kind;
  memmove(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) {
  (void)stream;
  return hipMemcpy(d, s, n, kind);
}
int hipMemset(void* d, int v, size_t n) {
  note("hipMemset", "", current);
  memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* stream) {
  (void)stream;
  return hipMemset(d, v, n);
}

int hipStreamCreateWithFlags(void** s, unsigned flags) {
  (void)flags;
  *s = make("hipStreamCreateWithFlags");
  return 0;
}
int hipStreamDestroy(void* s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void* s) {
  (void)s;
  return 0;
}
int hipStreamWaitEvent(void* s, void* e, unsigned flags) {
  (void)s;
  (void)e;
  (void)flags;
  return 0;
}
int hipStreamBeginCapture(void* s, int mode) {
  (void)s;
  (void)mode;
  return 0;
}
int hipStreamEndCapture(void* s, void** g) {
  (void)s;
  *g = make("hipStreamEndCapture");
  return 0;
}
int hipGraphInstantiate(void** x, void* g, void* node, char* log, size_t n) {
  (void)g;
  (void)node;
  (void)log;
  (void)n;
  *x = make("hipGraphInstantiate");
  return 0;
}
int hipGraphLaunch(void* x, void* s) {
  (void)x;
  (void)s;
  note("hipGraphLaunch", "", current);
  return 0;
}
int hipGraphDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphExecDestroy(void* x) {
  free(x);
  return 0;
}
int hipEventCreate(void** e) {
  *e = make("hipEventCreate");
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned flags) {
  (void)flags;
  *e = make("hipEventCreateWithFlags");
  return 0;
}
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void* e, void* s) {
  (void)e;
  (void)s;
  return 0;
}
int hipEventSynchronize(void* e) {
  (void)e;
  return 0;
}
int hipEventElapsedTime(float* ms, void* a, void* b) {
  (void)a;
  (void)b;
  *ms = 1.0f;
  return 0;
}

/* ---- kernels ---------------------------------------------------------------- */
void** __hipRegisterFatBinary(const void* data) {
  (void)data;
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* fn, char* device_fn, const char* name, unsigned limit, void* t, void* b,
                           void* bd, void* gd, int* ws) {
  (void)m;
  (void)device_fn;
  (void)limit;
  (void)t;
  (void)b;
  (void)bd;
  (void)gd;
  (void)ws;
  if (n_kernels < 1024) {
    kernels[n_kernels].fn = fn;
    snprintf(kernels[n_kernels++].name, sizeof(kernels[0].name), "%s", name);
  }
}
void __hipRegisterVar(void** m, void* var, char* host, char* device, int ext, size_t n, int constant, int global) {
  (void)m;
  (void)var;
  (void)host;
  (void)device;
  (void)ext;
  (void)n;
  (void)constant;
  (void)global;
}
int hipGetSymbolAddress(void** p, const void* sym) {
  (void)sym;
  *p = calloc(1, 1 << 20);
  return 0;
}

static _Thread_local struct {
  dim3_t grid, block;
  size_t lds;
  void* stream;
} call;
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void* stream) {
  call.grid = grid;
  call.block = block;
  call.lds = lds;
  call.stream = stream;
  return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, void** stream) {
  *grid = call.grid;
  *block = call.block;
  *lds = call.lds;
  *stream = call.stream;
  return 0;
}
int hipLaunchKernel(const void* fn, dim3_t grid, dim3_t block, void** args, size_t lds, void* stream) {
  (void)grid;
  (void)block;
  (void)lds;
  const char* name = "?";
  for (int k = 0; k < n_kernels; ++k)
    if (kernels[k].fn == fn) name = kernels[k].name;
  note("launch of ", name, current);
  if (stream) note("stream of ", name, ((handle_t*)stream)->device);
  if (strstr(name, "k_put_counters")) {
    const long long* from = *(const long long**)args[0];
    const int n = *(int*)args[1];
    long long* to = *(long long**)args[2];
    for (int k = 0; k < n; ++k) {
      to[k] = from[k];
      if (k < 64 && forced[k].reads > 0) {
        --forced[k].reads;
        to[k] = forced[k].value;
      }
    }
  }
  return 0;
}
