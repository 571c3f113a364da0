/* The runtime calls that libcuvdia.so and cuv_amd/_native.so make, without a GPU: memory is host memory, a launch is
 * counted and runs nothing, and each call that can fail does so when a test says so.  Loaded with RTLD_GLOBAL ahead of
 * torch (tests/_fake_hip.py), so that both libraries' own calls end here. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

enum { SUCCESS = 0, OUT_OF_MEMORY = 2, UNKNOWN = 999 };
typedef struct { uint32_t x, y, z; } dim3_;

int fake_device = 0, fake_devices = 2;
int fake_launches = 0;                   /* kernels launched so far */
int fake_fail_launch = 0, fake_fail_event_create = 0, fake_fail_wait = 0, fake_fail_capturing = 0;
int fake_grid = 0;                       /* workgroups of the last launch */
void *fake_last_event = NULL;            /* the event of the last launch, and ... */
void *fake_waited_event = NULL;          /* ... the one waited for last */
volatile int fake_hold_launch = 0;       /* launches and waits stay in their call until it is 0, at most 10 s */
volatile int fake_held = 0;              /* calls that ran into those 10 s */
int fake_news = 0;                       /* calls of C++'s operator new; ... */
int fake_fail_new = 0;                   /* ... n > 0: the n-th from now throws std::bad_alloc, and this is 0 */

static int s_error = 0;
static int result(int fail) { return fail ? (s_error = UNKNOWN) : SUCCESS; }
static void hold(void)
{
    for (int i = 0; i < 10000 && fake_hold_launch; ++i) usleep(1000);
    if (fake_hold_launch) ++fake_held;
}

void _ZSt17__throw_bad_allocv(void);
void *_Znwm(size_t n)                    /* operator new(size_t) */
{
    ++fake_news;
    if (fake_fail_new > 0 && --fake_fail_new == 0) _ZSt17__throw_bad_allocv();
    void *p = malloc(n ? n : 1);
    if (!p) _ZSt17__throw_bad_allocv();
    return p;
}

int hipGetDeviceCount(int *n) { *n = fake_devices; return SUCCESS; }
int hipGetDevice(int *d) { *d = fake_device; return SUCCESS; }
int hipMalloc(void **p, size_t n) { return (*p = malloc(n)) ? SUCCESS : OUT_OF_MEMORY; }
int hipFree(void *p) { free(p); return SUCCESS; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) { memcpy(d, s, n); return SUCCESS; }
int hipDeviceSynchronize(void) { return SUCCESS; }
int hipGetLastError(void) { const int e = s_error; s_error = 0; return e; }
const char *hipGetErrorString(int e) { return e ? "a failure asked for" : "no error"; }
int hipGetSymbolAddress(void **p, const void *symbol) { static char block[1 << 16]; *p = block; return SUCCESS; }
int hipEventCreateWithFlags(void **e, unsigned flags)
{
    if (fake_fail_event_create) return result(1);
    *e = malloc(1);
    return SUCCESS;
}
int hipEventDestroy(void *e) { free(e); return SUCCESS; }
int hipEventSynchronize(void *e) { hold(); fake_waited_event = e; return result(fake_fail_wait || !e); }
int hipStreamSynchronize(void *s) { hold(); return result(fake_fail_wait); }
int hipStreamIsCapturing(void *s, int *status) { *status = 0; return result(fake_fail_capturing); }
int hipExtLaunchKernel(const void *f, dim3_ grid, dim3_ block, void **args, size_t lds, void *stream, void *start, void *stop, int flags)
{
    hold();
    ++fake_launches;
    fake_grid = grid.x;
    fake_last_event = stop;
    return result(fake_fail_launch);
}
int hipLaunchKernel(const void *f, dim3_ grid, dim3_ block, void **args, size_t lds, void *stream)
{
    return hipExtLaunchKernel(f, grid, block, args, lds, stream, NULL, NULL, 0);
}
static __thread struct { dim3_ grid, block; size_t lds; void *stream; } s_config;
int __hipPushCallConfiguration(dim3_ grid, dim3_ block, size_t lds, void *stream)
{
    s_config.grid = grid, s_config.block = block, s_config.lds = lds, s_config.stream = stream;
    return SUCCESS;
}
int __hipPopCallConfiguration(dim3_ *grid, dim3_ *block, size_t *lds, void **stream)
{
    *grid = s_config.grid, *block = s_config.block, *lds = s_config.lds, *stream = s_config.stream;
    return SUCCESS;
}

/* torch's current stream: the default one (c10::hip::getCurrentHIPStream and HIPStream::stream) */
typedef struct { int64_t a, b; } stream_;
stream_ _ZN3c103hip19getCurrentHIPStreamEa(signed char device) { const stream_ s = {0, 0}; return s; }
void *_ZNK3c103hip9HIPStream6streamEv(const stream_ *s) { return NULL; }
