/* Failing allocations and copies of the HIP runtime, from the host: loaded
 * before libvfps.so with global symbols, its functions stand in front of the
 * runtime's, count, and refuse the calls they are told to refuse.  Nothing
 * reaches the device from a refused call. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <stdlib.h>

enum { SUCCESS = 0, OUT_OF_MEMORY = 2 };

static int countdown;          /* hipMalloc/hipMemcpy calls up to a failing one */
static size_t pinned_limit;    /* hipHostMalloc from this size on fails, 0: none */
static int live;               /* device allocations not yet freed */
static int refused;

void hip_faults_at(int call) { countdown = call; }
void hip_faults_pinned(size_t bytes) { pinned_limit = bytes; }
int hip_faults_live(void) { return live; }
int hip_faults_refused(void) { return refused; }

static void *real(const char *name)
{
    void *h = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD);
    void *f = h ? dlsym(h, name) : NULL;
    if (!f) abort();
    return f;
}

static int refuse(void)
{
    if (countdown > 0 && --countdown == 0) {
        refused++;
        return 1;
    }
    return 0;
}

int hipMalloc(void **p, size_t bytes)
{
    int rc;
    if (refuse()) return OUT_OF_MEMORY;
    rc = ((int (*)(void **, size_t))real("hipMalloc"))(p, bytes);
    if (rc == SUCCESS) live++;
    return rc;
}

int hipFree(void *p)
{
    if (p) live--;
    return ((int (*)(void *))real("hipFree"))(p);
}

int hipMemcpy(void *dst, const void *src, size_t bytes, int kind)
{
    if (refuse()) return OUT_OF_MEMORY;
    return ((int (*)(void *, const void *, size_t, int))real("hipMemcpy"))(
        dst, src, bytes, kind);
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    if (pinned_limit && bytes >= pinned_limit) {
        refused++;
        return OUT_OF_MEMORY;
    }
    return ((int (*)(void **, size_t, unsigned))real("hipHostMalloc"))(p, bytes,
                                                                        flags);
}
