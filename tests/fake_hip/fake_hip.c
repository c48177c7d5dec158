/* The HIP calls of a plan's creation, on host memory and with a limit: preloaded before
 * libpgrav it lets a test run out of device memory without a device. */
#include <malloc.h>
#include <stdlib.h>
#include <string.h>

static size_t used, limit = (size_t)-1;
static int last;

size_t fake_used(void) { return used; }
void fake_limit(size_t bytes) { limit = bytes; }

int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevice(int *d) { return *d = 0; }
int hipDeviceGetAttribute(int *v, int attr, int d) { return (void)attr, (void)d, *v = 256, 0; }
int hipGetLastError(void) {
    const int e = last;
    last = 0;
    return e;
}
int hipMalloc(void **p, size_t bytes) {
    *p = malloc(bytes ? bytes : 1);
    if (!*p || used + malloc_usable_size(*p) > limit) {
        free(*p);
        *p = NULL;
        return last = 2;
    }
    used += malloc_usable_size(*p);
    return 0;
}
int hipFree(void *p) {
    if (p)
        used -= malloc_usable_size(p);
    free(p);
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return (void)kind, memcpy(d, s, n), 0; }
int hipMemset(void *d, int c, size_t n) { return memset(d, c, n), 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { return (void)f, *s = &used, 0; }
int hipStreamSynchronize(void *s) { return (void)s, 0; }
int hipStreamDestroy(void *s) { return (void)s, 0; }
int hipEventCreate(void **e) { return *e = &used, 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { return (void)f, *e = &used, 0; }
int hipEventRecord(void *e, void *s) { return (void)e, (void)s, 0; }
int hipEventDestroy(void *e) { return (void)e, 0; }
