// Row and column reductions after the factors: corrWith (per-day
// correlation of each factor with a target, e.g. forward returns) and
// aggregrate (per-stock reductions over runs of equal labels, e.g. bars into
// days).
//
// corrWith restates cpp/Kun/CorrWith.hpp:11-121: per row, sums over the
// stocks in stock order of x, y, x*x, y*y and x*y (no NaN skipping), each
// divided by the stock count, then (XY - X*Y) / (sqrt(X2 - X*X) *
// sqrt(Y2 - Y*Y)). The five sums are sequential chains in stock order (bit
// parity). With rank inputs, x is the row's rank, computed by the Rank row
// kernel first.
//
// aggregrate restates cpp/Kun/Aggregration.cpp:11-105: one lane per stock
// walks the rows in order; a change of label closes a group and stores its
// sum (kahanAdd), min and max (NaN if any NaN), first, last, count (every
// row) and mean (sum / count) at the group's index.
#include <hip/hip_runtime.h>

#include "kun_cs.hpp"
#include "kun_device.hpp"

namespace {

__device__ __forceinline__ size_t rr_at(int sts, long t, long s, long S, long T, int blk) {
    return sts ? ((size_t)(s / blk) * T + t) * blk + s % blk : (size_t)t * S + s;
}

// Bound by the chains' latency: an add that waits for the one before it
// takes 8.9 clocks, 5000 stocks 19 us, however little of the GPU they fill.
// So each lane of a workgroup's first wavefront runs one chain of one row
// (CORR_ROWS rows x 5 chains) and does nothing but read the next terms and
// add; the other wavefronts load the rows a tile ahead and leave the terms --
// a, b, a*a, b*b, a*b, each rounded as the chain would -- in LDS; and the
// inputs of a call share a launch, so that their chains run side by side.
// Rows are padded with -0, which leaves every sum as it is.
//
// 4 inputs of 1000 rows of 5000 stocks: 39 us; a lane that walked all five
// chains of its own row, a launch per input, took 1910.
constexpr int CORR_ROWS = 8, CORR_TILE = 128, CORR_STAGE = 256, CORR_CHAINS = 5;
constexpr int CORR_BLOCK = 64 + CORR_STAGE;
constexpr int CORR_STRIDE = CORR_TILE + 4; // chains of 16-byte reads start four banks apart
constexpr int CORR_STEP = 16;              // terms read ahead of their adds
constexpr int CORR_INPUTS = 16;            // inputs of one launch

// rows [start, start + L) of the inputs (layout `xsts`, rows of T) and y
// (`ysts`); x may instead be [L][S] TS arrays of ranks (xrows = L, xrow0 = 0)
struct CorrArgs {
    const float *x[CORR_INPUTS], *y;
    float *out[CORR_INPUTS];
    int xsts, ysts, blk;
    long xT, xrow0, yT, S, start, L;
};

__global__ __launch_bounds__(CORR_BLOCK) void corr_rows(const CorrArgs A) {
    __shared__ __attribute__((aligned(16))) float term[2][CORR_CHAINS * CORR_ROWS * CORR_STRIDE];
    __shared__ float total[CORR_CHAINS][CORR_ROWS];
    const float *x = A.x[blockIdx.y];
    const long r0 = (long)blockIdx.x * CORR_ROWS;
    const int nr = (int)(A.L - r0 < CORR_ROWS ? A.L - r0 : CORR_ROWS);
    const int ntile = (int)((A.S + CORR_TILE - 1) / CORR_TILE);
    constexpr int PER = CORR_ROWS * CORR_TILE / CORR_STAGE;
    if (threadIdx.x >= 64) {
        const int id = threadIdx.x - 64;
        float a[PER], b[PER];
        auto load = [&](int tile) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int e = id + q * CORR_STAGE, r = e / CORR_TILE;
                const long s = (long)tile * CORR_TILE + e % CORR_TILE;
                a[q] = b[q] = -0.f;
                if (r < nr && s < A.S) {
                    a[q] = x[rr_at(A.xsts, r0 + r + A.xrow0, s, A.S, A.xT, A.blk)];
                    b[q] = A.y[rr_at(A.ysts, r0 + r + A.start, s, A.S, A.yT, A.blk)];
                }
            }
        };
        auto store = [&](int tile) {
            float *t = term[tile & 1];
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int e = id + q * CORR_STAGE;
                const bool in = (long)tile * CORR_TILE + e % CORR_TILE < A.S;
                float *at = t + e / CORR_TILE * CORR_STRIDE + e % CORR_TILE;
                constexpr int C = CORR_ROWS * CORR_STRIDE;
                at[0] = a[q];
                at[C] = b[q];
                at[2 * C] = in ? a[q] * a[q] : -0.f; // (-0) * (-0) is +0
                at[3 * C] = in ? b[q] * b[q] : -0.f;
                at[4 * C] = in ? a[q] * b[q] : -0.f;
            }
        };
        load(0);
        store(0);
        load(1);
        for (int t = 0; t < ntile; t++) {
            __syncthreads(); // tile t is stored, tile t - 1 summed
            if (t + 1 < ntile) {
                store(t + 1);
                load(t + 2);
            }
        }
    } else {
        const int chain = threadIdx.x / CORR_ROWS, r = threadIdx.x % CORR_ROWS;
        const int at = (chain < CORR_CHAINS ? chain : 0) * CORR_ROWS * CORR_STRIDE + r * CORR_STRIDE;
        float sum = 0.f;
        for (int t = 0; t < ntile; t++) {
            __syncthreads();
            const float *v = term[t & 1] + at;
            float g[CORR_STEP], h[CORR_STEP];
#pragma unroll
            for (int u = 0; u < CORR_STEP; u++) g[u] = v[u];
#pragma unroll
            for (int k = 0; k < CORR_TILE; k += 2 * CORR_STEP) {
#pragma unroll
                for (int u = 0; u < CORR_STEP; u++) h[u] = v[k + CORR_STEP + u];
                __builtin_amdgcn_sched_barrier(0); // the reads stay ahead of the adds
#pragma unroll
                for (int u = 0; u < CORR_STEP; u++) sum = sum + g[u];
                if (k + 2 * CORR_STEP < CORR_TILE)
#pragma unroll
                    for (int u = 0; u < CORR_STEP; u++) g[u] = v[k + 2 * CORR_STEP + u];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < CORR_STEP; u++) sum = sum + h[u];
            }
        }
        if (chain < CORR_CHAINS) total[chain][r] = sum;
    }
    __syncthreads();
    if ((int)threadIdx.x < nr) {
        const float n = (float)A.S;
        const int r = threadIdx.x;
        const float X = total[0][r] / n, Y = total[1][r] / n, X2 = total[2][r] / n, Y2 = total[3][r] / n;
        const float XY = total[4][r] / n;
        A.out[blockIdx.y][r0 + r] = (XY - X * Y) / (sqrtf(X2 - X * X) * sqrtf(Y2 - Y * Y));
    }
}

struct AggOut {
    void *p[7]; // sum, min, max, first, last, count, mean (null: not wanted)
};

template <typename T>
__global__ __launch_bounds__(64) void aggregate_cols(const T *in, const T *labels, AggOut o, long S, long start,
                                                     long L) {
    const long s = (long)blockIdx.x * 64 + threadIdx.x;
    if (s >= S || L <= 0) return;
    const T inf = kun::inf<T>();
    T sum = 0, comp = 0, mn = inf, mx = -inf, last = 0, count = 0;
    T first = in[(size_t)start * S + s];
    T last_label = labels[start];
    long g = 0;
    auto flush = [&]() {
        const T vals[7] = {sum, mn, mx, first, last, count, sum / count};
#pragma unroll
        for (int k = 0; k < 7; k++)
            if (o.p[k]) ((T *)o.p[k])[(size_t)g * S + s] = vals[k];
    };
    for (long i = 0; i < L; i++) {
        const T label = labels[start + i];
        const T cur = in[(size_t)(start + i) * S + s];
        if (label != last_label) {
            flush();
            g++;
            first = cur;
            sum = 0;
            comp = 0;
            mn = inf;
            mx = -inf;
            count = 0;
        }
        count = count + T(1);
        last = cur;
        last_label = label;
        mx = (mx != mx || cur != cur) ? kun::qnan<T>() : (mx > cur ? mx : cur);
        mn = (mn != mn || cur != cur) ? kun::qnan<T>() : (mn < cur ? mn : cur);
        const T y = cur - comp;
        const T t = sum + y;
        comp = (t - sum) - y;
        sum = t;
    }
    flush();
}

} // namespace

namespace kun_cs {

int corr_inputs() { return CORR_INPUTS; }

hipError_t launch_corr(int n, const float *const *x, int xsts, long xT, long xrow0, const float *y, int ysts, long yT,
                       float *const *out, long S, long start, long L, int blk, hipStream_t st) {
    if (L <= 0 || n <= 0) return hipSuccess;
    if (n > CORR_INPUTS) return hipErrorInvalidValue;
    // a grid has fewer than 2^32 threads
    const long per = 1L << 24;
    for (long l0 = 0; l0 < L; l0 += per) {
        CorrArgs a;
        for (int i = 0; i < CORR_INPUTS; i++) {
            a.x[i] = x[i < n ? i : 0];
            a.out[i] = out[i < n ? i : 0] + l0;
        }
        a.y = y;
        a.xsts = xsts;
        a.ysts = ysts;
        a.blk = blk;
        a.xT = xT;
        a.xrow0 = xrow0 + l0;
        a.yT = yT;
        a.S = S;
        a.start = start + l0;
        a.L = L - l0 < per ? L - l0 : per;
        hipLaunchKernelGGL(corr_rows, dim3((unsigned)((a.L + CORR_ROWS - 1) / CORR_ROWS), (unsigned)n),
                           dim3(CORR_BLOCK), 0, st, a);
    }
    return hipGetLastError();
}

hipError_t launch_aggregate(int dtype, const void *in, const void *labels, void *const *outs, long S, long start,
                            long L, hipStream_t st) {
    if (L <= 0 || S <= 0) return hipSuccess;
    AggOut o;
    for (int k = 0; k < 7; k++) o.p[k] = outs[k];
    const dim3 grid((unsigned)((S + 63) / 64));
    if (dtype)
        hipLaunchKernelGGL(aggregate_cols<double>, grid, dim3(64), 0, st, (const double *)in, (const double *)labels, o,
                           S, start, L);
    else
        hipLaunchKernelGGL(aggregate_cols<float>, grid, dim3(64), 0, st, (const float *)in, (const float *)labels, o, S,
                           start, L);
    return hipGetLastError();
}

} // namespace kun_cs

// ---- host drivers -----------------------------------------------------------
#include <string.h>

#include <algorithm>
#include <memory>
#include <string>
#include <vector>

#include "kun_rt.hpp"

namespace kunrt {

namespace {

struct DevBuf {
    Executor &ex;
    void *p = nullptr;
    size_t n = 0;
    DevBuf(Executor &e, size_t bytes) : ex(e), p(e.pool.get(bytes)), n(bytes) {}
    ~DevBuf() { ex.pool.put(p, n); }
};

size_t count_groups(const char *labels, size_t esz, size_t start, size_t L) {
    if (L == 0) return 0;
    size_t g = 1;
    for (size_t i = start + 1; i < start + L; i++) {
        const bool diff = esz == 8 ? ((const double *)labels)[i] != ((const double *)labels)[i - 1]
                                   : ((const float *)labels)[i] != ((const float *)labels)[i - 1];
        g += diff ? 1 : 0;
    }
    return g;
}

} // namespace

void corr_with(Executor &ex, bool device, int sts, bool rank_inputs, int n, const float *const *inputs,
               const float *target, float *const *outs, size_t S, size_t T, size_t start, size_t L, int blk,
               hipStream_t st) {
    if (start + L > T) throw Error("Bad parameter: cur_time + length exceeds total_time");
    if (n < 0) throw Error("bad number of inputs");
    if (rank_inputs && (long)S > kun_cs::max_rank_stocks(0))
        throw Error("Rank over more than " + std::to_string(kun_cs::max_rank_stocks(0)) + " stocks is not supported");
    std::lock_guard<std::mutex> g(ex.mu);
    HIPCHECK(hipSetDevice(ex.device));
    if (!st) st = ex.stream;
    const size_t in_bytes = (sts ? (S + blk - 1) / blk * blk : S) * T * sizeof(float);
    // a launch takes a group of inputs: as many as it can, device copies and
    // ranks together within a gigabyte, or fewer where the device has less
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t x_bytes = device ? 0 : up(in_bytes), o_bytes = device ? 0 : up(L * sizeof(float) + 4);
    const size_t r_bytes = rank_inputs ? up(S * L * sizeof(float) + 4) : 0;
    const size_t each = x_bytes + o_bytes + r_bytes, most = (size_t)1 << 30;
    size_t fit = (size_t)kun_cs::corr_inputs();
    if (each) fit = std::min(fit, std::max<size_t>(1, most > x_bytes ? (most - x_bytes) / each : 0));
    int group = (int)std::min<size_t>(fit, (size_t)n);
    while (group > 1 && each && !ex.corr.reserve(x_bytes + group * each, ex.pool)) group /= 2;
    if (group && each && !ex.corr.reserve(x_bytes + group * each, ex.pool))
        throw Error("hipMalloc of " + std::to_string(x_bytes + group * each) + " bytes for corrWith failed");
    // the workspace is free again when the call returns, also by an error
    struct Wait {
        hipStream_t st;
        bool on;
        ~Wait() {
            if (on) hipStreamSynchronize(st);
        }
    } wait{st, each != 0};
    const float *y = target;
    char *at = ex.corr.p;
    if (!device && n) {
        HIPCHECK(hipMemcpyAsync(at, target, in_bytes, hipMemcpyHostToDevice, st));
        y = (const float *)at;
        at += x_bytes;
    }
    std::vector<char *> dx, dout, ranks;
    for (int k = 0; k < group; k++, at += each) {
        dx.push_back(at);
        dout.push_back(at + x_bytes);
        ranks.push_back(at + x_bytes + o_bytes);
    }
    for (int i0 = 0; i0 < n; i0 += group) {
        const int m = std::min(group, n - i0);
        std::vector<const float *> x(m);
        std::vector<float *> o(m);
        hipError_t e = hipSuccess;
        for (int k = 0; k < m; k++) {
            x[k] = inputs[i0 + k];
            o[k] = outs[i0 + k];
            if (!device) {
                HIPCHECK(hipMemcpyAsync(dx[k], x[k], in_bytes, hipMemcpyHostToDevice, st));
                x[k] = (const float *)dx[k];
                o[k] = (float *)dout[k];
            }
            if (rank_inputs && e == hipSuccess) {
                kun_cs::View vi{(void *)x[k], sts ? 0 : 1, (long)T, (long)start}, vo{ranks[k], 1, (long)L, 0};
                e = kun_cs::launch_rank(0, vi, vo, (long)S, (long)L, blk, st);
                x[k] = (const float *)ranks[k];
            }
        }
        if (e == hipSuccess)
            e = rank_inputs ? kun_cs::launch_corr(m, x.data(), 0, (long)L, 0, y, sts, (long)T, o.data(), (long)S,
                                                  (long)start, (long)L, blk, st)
                            : kun_cs::launch_corr(m, x.data(), sts, (long)T, (long)start, y, sts, (long)T, o.data(),
                                                  (long)S, (long)start, (long)L, blk, st);
        if (e != hipSuccess) throw Error(std::string("corrWith kernel: ") + hipGetErrorString(e));
        if (!device)
            for (int k = 0; k < m; k++)
                HIPCHECK(hipMemcpyAsync(outs[i0 + k], o[k], L * sizeof(float), hipMemcpyDeviceToHost, st));
    }
    // host buffers are copied back, the workspace is free
    wait.on = false;
    if (!device || rank_inputs) HIPCHECK(hipStreamSynchronize(st));
}

void aggregate(Executor &ex, bool device, int n, const void *const *inputs, const void *const *labels, int dtype,
               void *const *outs, size_t S, size_t T, size_t start, size_t L, size_t out_rows, hipStream_t st) {
    if (start + L > T) throw Error("Bad parameter: cur_time + length exceeds total_time");
    if (n < 0) throw Error("bad number of aggregrations");
    const size_t esz = dtype ? 8 : 4;
    std::lock_guard<std::mutex> g(ex.mu);
    HIPCHECK(hipSetDevice(ex.device));
    if (!st) st = ex.stream;
    std::vector<char> hl;
    for (int i = 0; i < n; i++) {
        // group count from the labels (copied back when they live on the device)
        const char *lab = (const char *)labels[i];
        if (device) {
            hl.resize(T * esz);
            HIPCHECK(hipMemcpyAsync(hl.data(), labels[i], T * esz, hipMemcpyDeviceToHost, st));
            HIPCHECK(hipStreamSynchronize(st));
            lab = hl.data();
        }
        const size_t groups = count_groups(lab, esz, start, L);
        if (device && groups > out_rows)
            throw Error("aggregrate: " + std::to_string(groups) + " label groups exceed the " +
                        std::to_string(out_rows) + " output rows");
        void *dev_outs[7];
        std::unique_ptr<DevBuf> din, dlab, douts[7];
        const void *x = inputs[i], *lb = labels[i];
        if (!device) {
            din.reset(new DevBuf(ex, S * T * esz + 8));
            dlab.reset(new DevBuf(ex, T * esz + 8));
            HIPCHECK(hipMemcpyAsync(din->p, inputs[i], S * T * esz, hipMemcpyHostToDevice, st));
            HIPCHECK(hipMemcpyAsync(dlab->p, labels[i], T * esz, hipMemcpyHostToDevice, st));
            x = din->p;
            lb = dlab->p;
        }
        for (int k = 0; k < 7; k++) {
            void *o = outs[(size_t)i * 7 + k];
            dev_outs[k] = o;
            if (o && !device) {
                douts[k].reset(new DevBuf(ex, groups * S * esz + 8));
                dev_outs[k] = douts[k]->p;
            }
        }
        hipError_t e = kun_cs::launch_aggregate(dtype, x, lb, dev_outs, (long)S, (long)start, (long)L, st);
        if (e != hipSuccess) throw Error(std::string("aggregrate kernel: ") + hipGetErrorString(e));
        if (!device) {
            for (int k = 0; k < 7; k++)
                if (outs[(size_t)i * 7 + k])
                    HIPCHECK(hipMemcpyAsync(outs[(size_t)i * 7 + k], dev_outs[k], groups * S * esz,
                                            hipMemcpyDeviceToHost, st));
            HIPCHECK(hipStreamSynchronize(st));
        }
    }
}

} // namespace kunrt
