// Rows read by one thread while another runs ticks: every row returned is one
// tick's. The HIP calls of libkunhip.so are answered by host memory, so that a
// tick's parts can be slowed down: a launch of the tick's kernels sets every output row to the
// tick's number; the launch that copies rows to the host, and the reader's own
// copies of a row, take it in two halves with a pause between them.
// Arguments: module name, its library. Exits 1 on a row of two ticks or one
// older than the last tick that had ended before the read began.
#include <stdio.h>
#include <unistd.h>

#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/kun_capi.h"
#include "host_hip.hpp"
#include "kun_module_abi.h"

static const size_t S = 512;
static std::mutex alloc_mu;
static std::vector<P> device_rows; // hipMalloc of one row, in order: the module's buffers
static std::vector<int> outputs;
static std::atomic<int> tick{0}, copies{0};

static thread_local bool slow = false;
extern "C" __attribute__((visibility("default"))) void *memcpy(void *d, const void *s, size_t n) {
    volatile char *to = (volatile char *)d;
    const volatile char *from = (const volatile char *)s;
    for (size_t i = 0; i < n; i++) {
        if (slow && n == S * sizeof(double) && i == n / 2) usleep(3000);
        to[i] = from[i];
    }
    return d;
}

P host_alloc(size_t n) {
    P p = calloc(1, n + 1);
    std::lock_guard<std::mutex> g(alloc_mu);
    if (n == S * sizeof(double)) device_rows.push_back(p);
    return p;
}
void host_free(P p) { free(p); }

static const void *copy_kernel = nullptr; // the one launched for several rows at once
int host_launch(const void *func, Dim grid, Dim, P *args) {
    if (grid.y >= 2) copy_kernel = func;
    if (func == copy_kernel) { // rows to the host: {sources[64], destinations[64]}
        P *rows = (P *)args[0];
        for (int half = 0; half < 2; half++) {
            for (unsigned r = 0; r < grid.y; r++)
                memcpy((char *)rows[64 + r] + half * S * 4, (char *)rows[r] + half * S * 4, S * 4);
            if (!half) usleep(2000);
        }
        copies++;
        return 0;
    }
    for (int b : outputs)
        for (size_t s = 0; s < S; s++) ((double *)device_rows[b])[s] = tick;
    return 0;
}

int main(int, char **argv) {
    P lib = kunLoadLibrary(argv[2]);
    P mod = lib ? kunGetModuleFromLibrary(lib, argv[1]) : nullptr;
    if (!mod) return 2;
    const auto *m = (const KunModuleDesc *)mod;
    if (m->dtype != KUN_DTYPE_DOUBLE) return 2;
    P ex = kunCreateSingleThreadExecutor();
    P c = kunCreateStream(ex, mod, S);
    if (!c) return 2;
    for (int b = 0; b < m->nbuf; b++)
        if (m->bufs[b].kind == KUN_BUF_OUTPUT) outputs.push_back(b);
    if (outputs.size() < 2 || device_rows.size() < (size_t)m->nbuf) return 2;
    for (int t = 0; t < 2; t++) {
        kunStreamRun(c);
        for (int b : outputs) kunStreamGetCurrentBuffer(c, (size_t)b);
    }
    if (!copy_kernel) return 2;
    std::atomic<bool> stop{false};
    std::atomic<int> ended{0}, reads{0}, bad{0};
    std::thread reader([&] {
        for (unsigned pass = 0; !stop; usleep(100 * (pass++ % 7)))
            for (int b : outputs) {
                const int before = ended;
                slow = true;
                const double *row = (const double *)kunStreamGetCurrentBuffer(c, (size_t)b);
                slow = false;
                for (size_t s = 0; s < S; s++)
                    if (row[s] != row[0] || row[s] < before) {
                        bad++;
                        break;
                    }
                reads++;
            }
    });
    for (int t = 1; t <= 400; t++) {
        tick = t;
        kunStreamRun(c);
        ended = t;
        usleep(200 * (t % 20));
    }
    stop = true;
    reader.join();
    printf("%d reads, %d ticks with copies, %d wrong rows\n", (int)reads, (int)copies, (int)bad);
    kunDestoryStream(c);
    return bad || reads < 100 || copies < 50 ? 1 : 0;
}
