/* Stands before the HIP runtime in a test process: counts hipSetDevice, bounds
 * what hipMalloc hands out, as a card of `shim_budget` bytes would (and refuses
 * requests of just `shim_unwanted` bytes), keeps the last allocations' addresses
 * and calls `shim_before_graph` before a graph is launched. */
#include <pthread.h>
#include <stddef.h>

int (*shim_malloc)(void **, size_t), (*shim_free)(void *), (*shim_set_device)(int); /* the runtime's own */
int (*shim_graph_launch)(void *, void *), (*shim_mem_info)(size_t *, size_t *);
void (*shim_before_graph)(void);
size_t shim_budget = (size_t)-1, shim_unwanted, shim_used, shim_peak;
int shim_refused, shim_set_device_calls;
int shim_n_recent;
struct { void *p; size_t n; } shim_recent[256]; /* ring, in order of allocation */

#define SLOTS 65536
static struct { void *p; size_t n; } held[SLOTS];
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;

int hipMalloc(void **p, size_t n)
{
    int e = 2; /* hipErrorOutOfMemory */
    pthread_mutex_lock(&mu);
    if (n == shim_unwanted || n > shim_budget || shim_used > shim_budget - n) {
        shim_refused++;
    } else if ((e = shim_malloc(p, n)) == 0) {
        int k = 0;
        while (k < SLOTS - 1 && held[k].p) k++;
        held[k].p = *p;
        held[k].n = n;
        shim_recent[shim_n_recent % 256].p = *p;
        shim_recent[shim_n_recent++ % 256].n = n;
        shim_used += n;
        if (shim_used > shim_peak) shim_peak = shim_used;
    }
    pthread_mutex_unlock(&mu);
    return e;
}

int hipFree(void *p)
{
    pthread_mutex_lock(&mu);
    for (int k = 0; p && k < SLOTS; k++)
        if (held[k].p == p) {
            shim_used -= held[k].n;
            held[k].p = NULL;
            break;
        }
    pthread_mutex_unlock(&mu);
    return shim_free(p);
}

int hipMemGetInfo(size_t *free_bytes, size_t *total)
{
    const int e = shim_mem_info(free_bytes, total);
    const size_t left = shim_budget > shim_used ? shim_budget - shim_used : 0;
    if (e == 0 && *free_bytes > left) *free_bytes = left;
    return e;
}

int hipGraphLaunch(void *exec, void *stream)
{
    if (shim_before_graph) shim_before_graph();
    return shim_graph_launch(exec, stream);
}

int hipSetDevice(int device)
{
    shim_set_device_calls++;
    return shim_set_device(device);
}
