/* HIP's memory calls with limits, for tests of what the library does when an
 * allocation fails: loaded for all to see before the library, these take the
 * place of HIP's own, which they call. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>

enum { kOutOfMemory = 2, kBlocks = 1 << 16 }; /* hipErrorOutOfMemory */

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static struct { void *p; size_t n; } blocks[kBlocks];
static size_t device_used, device_peak;
static size_t device_limit = (size_t)-1, pin_limit = (size_t)-1, pins;

static void *hip(const char *name) {
    static void *lib;
    if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
    void *f = lib ? dlsym(lib, name) : NULL;
    if (!f) {
        fprintf(stderr, "limits: no %s\n", name);
        abort();
    }
    return f;
}

/* Bytes of device memory in use, the most since the last call, and new limits:
 * on those bytes, and on one allocation of pinned memory. */
size_t limits_used(void) { return device_used; }
size_t limits_peak(void) {
    const size_t n = device_peak;
    device_peak = device_used;
    return n;
}
/* Allocations of pinned memory so far. */
size_t limits_pins(void) { return pins; }
void limits_set(size_t device, size_t pin) {
    device_limit = device;
    pin_limit = pin;
}

int hipMalloc(void **p, size_t n) {
    pthread_mutex_lock(&lock);
    int rc = kOutOfMemory;
    if (device_used + n <= device_limit) {
        rc = ((int (*)(void **, size_t))hip("hipMalloc"))(p, n);
        for (int i = 0; rc == 0 && i < kBlocks; ++i)
            if (!blocks[i].p) {
                blocks[i].p = *p;
                blocks[i].n = n;
                device_used += n;
                if (device_used > device_peak) device_peak = device_used;
                break;
            }
    }
    pthread_mutex_unlock(&lock);
    return rc;
}

int hipFree(void *p) {
    pthread_mutex_lock(&lock);
    const int rc = ((int (*)(void *))hip("hipFree"))(p);
    for (int i = 0; p && i < kBlocks; ++i)
        if (blocks[i].p == p) {
            device_used -= blocks[i].n;
            blocks[i].p = NULL;
            break;
        }
    pthread_mutex_unlock(&lock);
    return rc;
}

int hipHostMalloc(void **p, size_t n, unsigned flags) {
    if (n > pin_limit) return kOutOfMemory;
    ++pins;
    return ((int (*)(void **, size_t, unsigned))hip("hipHostMalloc"))(p, n, flags);
}
