/* Stand-in for the HIP runtime: loaded globally before libmythos_oil.so it
 * takes the place of the runtime's functions, so that the library's host side
 * (checks, routes, workspace, locks) runs on a machine without a GPU.
 * Kernels are not run: each launch is recorded with its kernel's name, grid
 * and stream.  Device memory is addresses only, never touched. */
#include <pthread.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef void* stream_t;

enum { kMaxFns = 4096, kMaxLaunches = 65536 };
static struct { const void* host; const char* name; } fns[kMaxFns];
static int nfns;
static struct { const char* name; dim3 grid; stream_t stream; int thread; } launches[kMaxLaunches];
static int nlaunches, nmallocs, capture_mode;
static uint64_t malloc_bytes, next_address = 0x700000000000ull;
static stream_t capturing = (stream_t)-1, held = (stream_t)-1;
static int released = 1, waiting;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static pthread_cond_t cv = PTHREAD_COND_INITIALIZER;
static __thread struct { dim3 grid, block; size_t shmem; stream_t stream; } config;
static __thread int thread_mode, thread_id;

/* ---- what a test sets and reads ---- */
void rec_reset(void) { nlaunches = nmallocs = 0; malloc_bytes = 0; capturing = held = (stream_t)-1; }
int rec_launches(void) { return nlaunches; }
const char* rec_name(int i) { return launches[i].name; }
uint32_t rec_grid(int i, int d) { return d == 0 ? launches[i].grid.x : d == 1 ? launches[i].grid.y : launches[i].grid.z; }
int rec_thread(int i) { return launches[i].thread; }
int rec_mallocs(void) { return nmallocs; }
uint64_t rec_malloc_bytes(void) { return malloc_bytes; }
int rec_malloc_mode(void) { return capture_mode; } /* the capture mode of the thread that allocated last */
void rec_capture(stream_t s) { capturing = s; }    /* s is capturing ((void*)-1: none) */
void rec_thread_id(int id) { thread_id = id; }
/* a launch on stream s waits until rec_release (a full queue) */
void rec_hold(stream_t s) { pthread_mutex_lock(&mu); held = s; released = 0; waiting = 0; pthread_mutex_unlock(&mu); }
int rec_waiting(void) { pthread_mutex_lock(&mu); const int w = waiting; pthread_mutex_unlock(&mu); return w; }
void rec_release(void) {
    pthread_mutex_lock(&mu);
    released = 1;
    pthread_cond_broadcast(&cv);
    pthread_mutex_unlock(&mu);
}

/* ---- the runtime's functions that the library calls ---- */
void** __hipRegisterFatBinary(const void* data) { static void* h; (void)data; return &h; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned t, void* a, void* b, void* c,
                           void* d, int* w) {
    (void)m, (void)dev, (void)t, (void)a, (void)b, (void)c, (void)d, (void)w;
    if (nfns < kMaxFns) fns[nfns].host = host, fns[nfns++].name = name;
}
void __hipRegisterVar(void** m, void* v, char* h, const char* n, int e, size_t s, int c, int g) {
    (void)m, (void)v, (void)h, (void)n, (void)e, (void)s, (void)c, (void)g;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, stream_t st) {
    config.grid = g, config.block = b, config.shmem = s, config.stream = st;
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, stream_t* st) {
    *g = config.grid, *b = config.block, *s = config.shmem, *st = config.stream;
    return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t shmem, stream_t s) {
    (void)b, (void)args, (void)shmem;
    const char* name = "?";
    for (int i = 0; i < nfns; ++i)
        if (fns[i].host == f) name = fns[i].name;
    pthread_mutex_lock(&mu);
    if (nlaunches < kMaxLaunches) {
        launches[nlaunches].name = name;
        launches[nlaunches].grid = g;
        launches[nlaunches].stream = s;
        launches[nlaunches++].thread = thread_id;
    }
    if (s == held)
        while (!released) {
            waiting = 1;
            pthread_cond_wait(&cv, &mu);
        }
    pthread_mutex_unlock(&mu);
    return 0;
}
int hipMalloc(void** p, size_t n) {
    pthread_mutex_lock(&mu);
    *p = (void*)next_address;
    next_address += (n + 4095) / 4096 * 4096;
    ++nmallocs;
    malloc_bytes += n;
    capture_mode = thread_mode;
    pthread_mutex_unlock(&mu);
    return 0;
}
int hipFree(void* p) { (void)p; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
const char* hipGetErrorString(int e) { (void)e; return "recorded"; }
int hipGetLastError(void) { return 0; }
int hipGetSymbolAddress(void** p, const void* s) { (void)s; *p = (void*)0x600000000000ull; return 0; }
int hipStreamIsCapturing(stream_t s, int* st) { *st = s == capturing ? 1 : 0; return 0; }
int hipThreadExchangeStreamCaptureMode(int* m) { const int old = thread_mode; thread_mode = *m; *m = old; return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { (void)d, (void)s, (void)n, (void)k; return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, stream_t st) { (void)d, (void)s, (void)n, (void)k, (void)st; return 0; }
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int k, stream_t st) {
    (void)d, (void)dp, (void)s, (void)sp, (void)w, (void)h, (void)k, (void)st;
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, stream_t s) { (void)d, (void)v, (void)n, (void)s; return 0; }
int hipMemsetD32Async(void* d, int v, size_t n, stream_t s) { (void)d, (void)v, (void)n, (void)s; return 0; }
int hipStreamCreateWithFlags(stream_t* s, unsigned f) { static char one; (void)f; *s = &one; return 0; }
int hipStreamDestroy(stream_t s) { (void)s; return 0; }
int hipStreamSynchronize(stream_t s) { (void)s; return 0; }
int hipStreamBeginCapture(stream_t s, int m) { (void)s, (void)m; return 0; }
int hipStreamEndCapture(stream_t s, void** g) { (void)s; *g = (void*)1; return 0; }
int hipGraphInstantiate(void** e, void* g, void** n, char* l, size_t z) { (void)g, (void)n, (void)l, (void)z; *e = (void*)1; return 0; }
int hipGraphLaunch(void* e, stream_t s) { (void)e, (void)s; return 0; }
int hipGraphDestroy(void* g) { (void)g; return 0; }
int hipGraphExecDestroy(void* e) { (void)e; return 0; }
int hipGraphGetNodes(void* g, void** n, size_t* c) { (void)g, (void)n; *c = 0; return 0; }
