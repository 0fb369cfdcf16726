// Device memory of corrWith: with little of it free, the inputs are taken in
// smaller groups; over calls of many shapes, what the executor keeps is
// bounded. The HIP calls of libkunhip.so are answered by host memory (kernels
// do nothing); the launches say how many rows of how many inputs were ranked
// and summed. Exits 1 where a call fails, an input or row is left out, a launch
// has more threads than a grid may have or too much is kept.
#include <stdio.h>

#include <map>
#include <vector>

#include "../../include/kun_capi.h"
#include "host_hip.hpp"

static std::map<P, size_t> live;
static size_t held = 0, limit = ~(size_t)0;
static long ranked = 0, summed = 0, groups = 0, wide = 0;

P host_alloc(size_t n) {
    if (held + n > limit) return nullptr;
    P p = malloc(16); // never touched: no kernel runs, device calls copy nothing
    live[p] = n;
    held += n;
    return p;
}
void host_free(P p) {
    if (!p) return;
    held -= live[p];
    live.erase(p);
    free(p);
}
int host_launch(const void *, Dim grid, Dim block, P *) {
    if ((size_t)grid.x * block.x >> 32) wide++;
    if (block.x == 320) { // the sums: a wavefront of chains and four that load
        summed += grid.y;
        groups += (long)grid.x * grid.y;
    } else {
        ranked += grid.x;
    }
    return 0;
}

int main() {
    P ex = kunCreateSingleThreadExecutor();
    const int n = 40;
    std::vector<const float *> x(n, (const float *)&x);
    std::vector<float *> o(n, (float *)&o);
    const float *y = (const float *)&y;
    int bad = 0;
    auto call = [&](size_t S, size_t T, const char *what) {
        ranked = summed = 0;
        if (kunCorrWithDevice(ex, 1, 1, n, x.data(), y, o.data(), S, T, 0, T, nullptr)) {
            printf("%s: %s\n", what, kunGetLastError());
            bad++;
        } else if (ranked != (long)(n * T) || summed != n) {
            printf("%s: %ld rows ranked, %ld inputs summed\n", what, ranked, summed);
            bad++;
        }
    };
    const size_t panel = 1000 * 500 * sizeof(float);
    for (size_t panels : {1, 2, 3, 7, 16}) {
        limit = held + panels * panel + 65536;
        call(1000, 500, "little memory");
        limit = ~(size_t)0;
    }
    for (size_t S = 100; S < 8000; S += 100) call(S, 900, "many shapes");
    if (held > (size_t)1 << 30) {
        printf("%zu bytes kept\n", held);
        bad++;
    }
    call(8000, 20000, "panels of 640 MB");
    if (held > (size_t)1 << 30) {
        printf("%zu bytes kept\n", held);
        bad++;
    }
    groups = 0; // of 8 rows
    const size_t rows = (size_t)1 << 28;
    if (kunCorrWithDevice(ex, 1, 0, 3, x.data(), y, o.data(), 1, rows + 5, 0, rows + 5, nullptr) || wide ||
        groups != 3 * (long)(rows / 8 + 1)) {
        printf("2^28 rows: %ld groups, %ld launches too wide\n", groups, wide);
        bad++;
    }
    kunDestoryExecutor(ex);
    if (held) {
        printf("%zu bytes never freed\n", held);
        bad++;
    }
    printf("%d faults\n", bad);
    return bad ? 1 : 0;
}
