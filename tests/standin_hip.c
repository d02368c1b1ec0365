/* A stand-in for the HIP runtime calls that libdrawhip.so makes, so that tests can run its host code without a
 * device: device memory is host memory, every stream is the calling thread, and a launch is recorded instead of
 * run -- except the canvas-read kernel, which is done here on the host.  Loaded with RTLD_GLOBAL before the
 * library, whose calls then bind to these.  Allocations can be made to fail, and a page-fault handler can hold
 * the library's helper threads where they first touch an array. */
#define _GNU_SOURCE
#include <signal.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include <sys/syscall.h>
#include <time.h>
#include <unistd.h>

typedef struct {
  uint32_t x, y, z;
} Dim3;

/* ------------------------------------------------------------------ memory */
enum { kMaxBlocks = 4096 };
static struct {
  char* p;
  size_t n;
} g_block[kMaxBlocks];
static long g_fail_in = -1; /* device allocations until the one that fails; -1: none */

static long g_host_left = -1; /* host allocations that succeed; -1: all */

void standin_fail_alloc(long n) { g_fail_in = n; }
void standin_host_allocs(long n) { g_host_left = n; }

/* bytes from p to the end of its block, -1 if it is in none */
int64_t standin_room(uint64_t p) {
  for (int i = 0; i < kMaxBlocks; i++)
    if (g_block[i].p && p >= (uint64_t)g_block[i].p && p < (uint64_t)g_block[i].p + g_block[i].n)
      return (int64_t)((uint64_t)g_block[i].p + g_block[i].n - p);
  return -1;
}

static int new_block(void** out, size_t n) {
  for (int i = 0; i < kMaxBlocks; i++)
    if (!g_block[i].p) {
      g_block[i].p = calloc(1, n); /* untouched pages take no memory */
      g_block[i].n = n;
      *out = g_block[i].p;
      return g_block[i].p ? 0 : 2;
    }
  return 2;
}
int hipMalloc(void** out, size_t n) {
  if (g_fail_in >= 0 && g_fail_in-- == 0) return 2; /* hipErrorOutOfMemory */
  return new_block(out, n);
}
int hipHostMalloc(void** out, size_t n, unsigned flags) {
  (void)flags;
  if (g_host_left == 0) return 2;
  if (g_host_left > 0) g_host_left--;
  return new_block(out, n);
}
int hipFree(void* p) {
  for (int i = 0; i < kMaxBlocks; i++)
    if (p && g_block[i].p == p) {
      free(p);
      g_block[i].p = NULL;
    }
  return 0;
}
int hipHostFree(void* p) { return hipFree(p); }
int hipHostGetDevicePointer(void** out, void* p, unsigned flags) {
  (void)flags;
  *out = p;
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  (void)kind;
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) {
  (void)stream;
  return hipMemcpy(d, s, n, kind);
}
int hipMemsetAsync(void* d, int v, size_t n, void* stream) {
  (void)stream;
  memset(d, v, n);
  return 0;
}
int hipPointerGetAttributes(void* at, const void* p) {
  (void)at;
  (void)p;
  return 1; /* not the runtime's memory */
}
int hipGetSymbolAddress(void** out, const void* symbol) {
  (void)out;
  (void)symbol;
  return 1;
}

/* ------------------------------------------- device, streams, events, graphs */
static uint64_t g_queries;
uint64_t standin_queries(void) { return __atomic_load_n(&g_queries, __ATOMIC_RELAXED); }

int hipGetDevice(int* d) { return *d = 0; }
int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipSetDevice(int d) { return d ? 101 : 0; }
const char* hipGetErrorString(int e) { return e ? "stand-in error" : "no error"; }
int hipGetLastError(void) { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned flags) {
  (void)flags;
  *s = (void*)1;
  return 0;
}
int hipStreamDestroy(void* s) { return s ? 0 : 1; }
int hipStreamSynchronize(void* s) { return s ? 0 : 1; }
int hipStreamQuery(void* s) {
  __atomic_add_fetch(&g_queries, 1, __ATOMIC_RELAXED);
  return s ? 0 : 1;
}
int hipStreamBeginCapture(void* s, int mode) { return (void)mode, s ? 0 : 1; } /* launches are recorded twice */
int hipStreamEndCapture(void* s, void** g) { return *g = (void*)1, s ? 0 : 1; }
int hipEventCreate(void** e) { return *e = (void*)1, 0; }
int hipEventDestroy(void* e) { return e ? 0 : 1; }
int hipEventRecord(void* e, void* s) { return e && s ? 0 : 1; }
int hipEventElapsedTime(float* ms, void* a, void* b) { return *ms = 0.0f, a && b ? 0 : 1; }
int hipGraphDestroy(void* g) { return g ? 0 : 1; }
int hipGraphExecDestroy(void* g) { return g ? 0 : 1; }
int hipGraphInstantiate(void** x, void* g, void* a, void* b, size_t n) {
  (void)g, (void)a, (void)b, (void)n;
  return *x = (void*)1, 0;
}
int hipGraphLaunch(void* x, void* s) { return x && s ? 0 : 1; }

/* ----------------------------------------------------------------- launches */
enum { kMaxKernels = 512, kMaxLaunches = 65536, kMaxArgs = 16 };
static struct {
  const void* host;
  const char* name;
} g_kernel[kMaxKernels];
static int g_kernels;
static struct {
  const char* name;
  uint64_t arg[kMaxArgs]; /* of kernels with an entry in kArgs */
} g_launch[kMaxLaunches];
static long g_launches;

/* Kernels whose arguments are recorded, with how many they have (none by value of more than 8 bytes). */
static const struct {
  const char* name;
  int n;
} kArgs[] = {{"k_geom_emit", 15}, {"k_pair_hist", 8},     {"k_pair_scatter", 11}, {"k_pair_sort", 7},
             {"k_bin_small", 10}, {"k_bin_emitILb", 12},  {"k_bin_emit_wide", 11}, {"k_radix_hist", 5},
             {"k_radix_scatter", 10}};

void** __hipRegisterFatBinary(const void* data) {
  static void* handle;
  (void)data;
  return &handle;
}
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* host, char* f, const char* name, unsigned limit, void* tid, void* bid,
                           Dim3* bd, Dim3* gd, int* ws) {
  (void)h, (void)f, (void)limit, (void)tid, (void)bid, (void)bd, (void)gd, (void)ws;
  if (g_kernels < kMaxKernels) {
    g_kernel[g_kernels].host = host;
    g_kernel[g_kernels++].name = strdup(name);
  }
}
void __hipRegisterVar(void** h, void* var, char* a, char* b, int c, size_t d, int e, int f) {
  (void)h, (void)var, (void)a, (void)b, (void)c, (void)d, (void)e, (void)f;
}

static __thread struct {
  Dim3 grid, block;
  size_t lds;
  void* stream;
} t_config;
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
  t_config.grid = grid;
  t_config.block = block;
  t_config.lds = lds;
  t_config.stream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = t_config.grid;
  *block = t_config.block;
  *lds = t_config.lds;
  *stream = t_config.stream;
  return 0;
}

static int g_no_reads; /* k_read_out does nothing, as on a device that stopped */
void standin_no_reads(int on) { g_no_reads = on; }

/* k_read_out: see its definition for the arguments */
static void read_out(void** a) {
  const struct {
    const uint32_t* src[3];
    uint32_t n_seg, n_words4, n_words16;
  }* g = a[0];
  const struct {
    uint32_t *stage[2], *flags[2], ticket;
  }* parts = a[3];
  const uint64_t w0 = *(uint64_t*)a[1];
  const uint32_t n = *(uint32_t*)a[2], chunk = 4096, part = 15 * chunk;
  for (uint32_t i = 0; i < n; i++)
    for (uint32_t k = 0; k < 4; k++) {
      const uint64_t e = 4 * ((w0 + i) % g->n_words16) + k;
      parts->stage[i / part][4 * (i % part) + k] = e < g->n_words4 ? g->src[(w0 + i) / g->n_words16][e] : 0;
    }
  for (uint32_t i = 0; i < n; i += chunk)
    __atomic_store_n(&parts->flags[i / part][i % part / chunk], parts->ticket + i / part, __ATOMIC_RELEASE);
}

int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t lds, void* stream) {
  (void)grid, (void)block, (void)lds, (void)stream;
  const char* name = "?";
  for (int i = 0; i < g_kernels; i++)
    if (g_kernel[i].host == f) name = g_kernel[i].name;
  if (strstr(name, "k_read_out") && !g_no_reads) read_out(args);
  if (g_launches < kMaxLaunches) {
    g_launch[g_launches].name = name;
    for (size_t k = 0; k < sizeof kArgs / sizeof *kArgs; k++)
      if (strstr(name, kArgs[k].name))
        for (int i = 0; i < kArgs[k].n; i++) memcpy(&g_launch[g_launches].arg[i], args[i], 8);
    g_launches++;
  }
  return 0;
}
long standin_launches(int clear) {
  const long n = g_launches;
  if (clear) g_launches = 0;
  return n;
}
const char* standin_launch_name(long i) { return g_launch[i].name; }
uint64_t standin_launch_arg(long i, int k) { return g_launch[i].arg[k]; }

/* -------------------------------------------------- threads held at an array */
static char* g_held;
static size_t g_held_n;
static double g_hold_s;
static int g_holds;

static void on_fault(int sig, siginfo_t* si, void* u) {
  (void)u;
  char* const at = si->si_addr;
  if (!g_held || at < g_held || at >= g_held + g_held_n) {
    signal(sig, SIG_DFL);
    return;
  }
  static __thread int held;
  if (syscall(SYS_gettid) != getpid() && !held) {
    held = 1;
    const double s = g_hold_s;
    const struct timespec t = {(time_t)s, (long)((s - (double)(time_t)s) * 1e9)};
    __atomic_add_fetch(&g_holds, 1, __ATOMIC_RELAXED);
    nanosleep(&t, NULL);
  }
  mprotect((char*)((uintptr_t)at & ~(uintptr_t)4095), 4096, PROT_READ | PROT_WRITE);
}
/* n bytes of memory at which every thread but the main one stops once, for `seconds`, when it touches a new page */
void* standin_hold_array(size_t n, double seconds) {
  struct sigaction sa;
  memset(&sa, 0, sizeof sa);
  sa.sa_sigaction = on_fault;
  sa.sa_flags = SA_SIGINFO;
  sigaction(SIGSEGV, &sa, NULL);
  g_hold_s = seconds;
  g_held_n = (n + 4095) & ~(size_t)4095;
  g_held = mmap(NULL, g_held_n, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  return g_held;
}
int standin_holds(void) { return __atomic_load_n(&g_holds, __ATOMIC_RELAXED); }
