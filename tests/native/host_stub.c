/* For tests of the library's host code without a GPU, preloaded into a process of its own: the memory calls of the HIP
 * runtime on ordinary memory, and thread creation, each of which can be told to fail. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>

/* how many more calls succeed; negative: all of them */
int stub_threads_left = -1, stub_host_mallocs_left = -1, stub_mallocs_left = -1, stub_copies_left = -1;
int stub_allocations = 0; /* allocations not freed yet */

static int take(int* left) {
    if (*left == 0) return 0;
    if (*left > 0) --*left;
    return 1;
}

int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
    static int (*real)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    if (real == NULL) *(void**)&real = dlsym(RTLD_NEXT, "pthread_create");
    return take(&stub_threads_left) ? real(t, a, f, arg) : EAGAIN;
}

static int get(void** p, size_t n, int* left) {
    *p = NULL;
    if (!take(left)) return 2; /* hipErrorOutOfMemory */
    if (posix_memalign(p, 4096, n) != 0) return 2;
    __sync_fetch_and_add(&stub_allocations, 1);
    return 0;
}
static int put(void* p) {
    if (p != NULL) __sync_fetch_and_sub(&stub_allocations, 1);
    free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned flags) { (void)flags; return get(p, n, &stub_host_mallocs_left); }
int hipMalloc(void** p, size_t n) { return get(p, n, &stub_mallocs_left); }
int hipHostFree(void* p) { return put(p); }
int hipFree(void* p) { return put(p); }
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
    (void)kind;
    if (!take(&stub_copies_left)) return 1;
    memcpy(d, s, n);
    return 0;
}
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) { (void)stream; return hipMemcpy(d, s, n, kind); }
int hipStreamSynchronize(void* stream) { (void)stream; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }
