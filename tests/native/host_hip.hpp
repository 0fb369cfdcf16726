// The HIP calls of libkunhip.so answered by host memory: a program that
// includes this (linked with -rdynamic) drives the library on the CPU, its own
// symbols coming before the HIP runtime's. Copies are made at once, streams
// and events do nothing. The program says what device allocations and kernel
// launches do.
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

typedef void *P;
struct Dim {
    unsigned x, y, z;
};

P host_alloc(size_t bytes); // null: out of memory
void host_free(P p);
int host_launch(const void *func, Dim grid, Dim block, P *args);

#define FAKE extern "C" __attribute__((visibility("default"))) int
FAKE hipMalloc(P *p, size_t n) { return (*p = host_alloc(n)) ? 0 : 2; }
FAKE hipFree(P p) {
    host_free(p);
    return 0;
}
FAKE hipHostMalloc(P *p, size_t n, unsigned) { return (*p = calloc(1, n + 1)) ? 0 : 2; }
FAKE hipHostFree(P p) {
    free(p);
    return 0;
}
FAKE hipMemcpy(P d, const void *s, size_t n, int) {
    memcpy(d, s, n);
    return 0;
}
FAKE hipMemcpyAsync(P d, const void *s, size_t n, int, P) {
    memcpy(d, s, n);
    return 0;
}
FAKE hipSetDevice(int) { return 0; }
FAKE hipGetDevice(int *d) {
    *d = 0;
    return 0;
}
FAKE hipGetLastError() { return 0; }
FAKE hipDeviceSynchronize() { return 0; }
FAKE hipStreamCreateWithFlags(P *s, unsigned) {
    *s = malloc(1);
    return 0;
}
FAKE hipStreamDestroy(P s) {
    free(s);
    return 0;
}
FAKE hipStreamSynchronize(P) { return 0; }
FAKE hipStreamWaitEvent(P, P, unsigned) { return 0; }
FAKE hipEventCreate(P *e) {
    *e = malloc(1);
    return 0;
}
FAKE hipEventCreateWithFlags(P *e, unsigned) {
    *e = malloc(1);
    return 0;
}
FAKE hipEventDestroy(P e) {
    free(e);
    return 0;
}
FAKE hipEventRecord(P, P) { return 0; }
FAKE hipEventSynchronize(P) { return 0; }

static thread_local struct {
    Dim g, b;
    size_t sh;
    P st;
} launch_config;
FAKE __hipPushCallConfiguration(Dim g, Dim b, size_t sh, P st) {
    launch_config = {g, b, sh, st};
    return 0;
}
FAKE __hipPopCallConfiguration(Dim *g, Dim *b, size_t *sh, P *st) {
    *g = launch_config.g;
    *b = launch_config.b;
    *sh = launch_config.sh;
    *st = launch_config.st;
    return 0;
}
FAKE hipLaunchKernel(const void *func, Dim grid, Dim block, P *args, size_t, P) {
    return host_launch(func, grid, block, args);
}
