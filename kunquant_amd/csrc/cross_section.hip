// Cross-sectional row kernels: Rank and Scale over the stocks of one row.
//
// Rank (restates cpp/Kun/Rank.hpp:11-57): per row, the non-NaN values are
// sorted; a value's rank is the average 1-based position of its tie group
// [lo, hi): sum = (lo + hi + 1) * (hi - lo) / 2 in integers, then
// T(sum) / T(hi - lo) / T(n). -0 and +0 tie (std::sort / equal_range use
// operator<). On the device a row's values become order-preserving integer
// keys (-0 canonicalised to +0, NaN to the largest key) and are cut into
// buckets of a key or two in LDS; a key's tie group is counted within its
// bucket (BucketRank, below). Rows whose buckets stay crowded are sorted, by
// an LSD radix sort with 4-bit digits counted per lane (CountRank).
//
// Scale (restates cpp/Kun/Scale.hpp:13-46): sum of |x| over non-NaN values
// accumulated sequentially in stock order (bit-exact order), then
// x / sum, or NaN when x == 0 and sum == 0.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "kun_cs.hpp"
#include "kun_device.hpp"

namespace {

template <typename T> struct KeyOf;
template <> struct KeyOf<float> { using K = uint32_t; };
template <> struct KeyOf<double> { using K = uint64_t; };

template <typename T> __device__ __forceinline__ typename KeyOf<T>::K rank_key(T x) {
    using K = typename KeyOf<T>::K;
    constexpr int NB = sizeof(K) * 8;
    if (x != x) return ~K(0);
    if (x == T(0)) x = T(0);
    K u = kun::to_bits(x);
    return (u >> (NB - 1)) ? ~u : (u | (K(1) << (NB - 1)));
}

__device__ __forceinline__ size_t cs_at(int layout, long row, long s, long S, long rows, int blk) {
    if (layout == 1) return (size_t)row * S + s;
    if (layout == 2) return (size_t)s;
    return ((size_t)(s / blk) * rows + row) * blk + s % blk;
}

// LAY: the view's layout fixed at compile time (-1: read from the view)
template <int LAY> __device__ __forceinline__ size_t lay_at(const kun_cs::View &v, long row, long s, long S, int blk) {
    if (LAY == 1) return (size_t)row * S + s;
    if (LAY == 2) return (size_t)s;
    return cs_at(v.layout, row, s, S, v.rows, blk);
}

// cell (row, s0 + i), s0 the same on every lane: for rows whose cells are
// consecutive the address is a scalar one plus the lane's i, and no lane
// keeps an index per cell
template <int LAY, typename T>
__device__ __forceinline__ T *cell_at(T *p, const kun_cs::View &v, long row, int s0, int i, long S, int blk) {
    if (LAY == -1) return p + lay_at<LAY>(v, row, s0 + i, S, blk);
    return p + lay_at<LAY>(v, row, s0, S, blk) + (unsigned)i;
}

// A kernel launch through a sink: the arguments converted to the kernel's
// parameter types, one pointer to each.
template <typename... P, size_t... I>
hipError_t sink_launch_impl(kun_cs::Sink &sink, const void *k, dim3 g, dim3 b, std::index_sequence<I...>,
                            std::tuple<P...> vals) {
    void *ptrs[] = {(void *)&std::get<I>(vals)...};
    return sink.launch(k, g, b, ptrs);
}
template <typename... P, typename... A>
hipError_t sink_launch(kun_cs::Sink &sink, void (*k)(P...), dim3 g, dim3 b, A... a) {
    static_assert(sizeof...(P) == sizeof...(A), "kernel argument count");
    return sink_launch_impl<P...>(sink, (const void *)k, g, b, std::index_sequence_for<P...>{},
                                  std::tuple<P...>((P)a...));
}

// ---- wavefront primitives (64 lanes) ------------------------------------

// number of lanes below this one whose bit is set in `mask`
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// lanes of the wavefront holding the same 8-bit digit as this lane: one
// ballot per digit bit; a lane disagrees with the lanes whose ballot bit
// differs from its own bit (m: all ones when this lane's bit is set), and
// the peers are the lanes that never disagree
// (bits on which the row's keys differ, `vary`, uniform: the others tell no
// lanes apart and are skipped)
__device__ __forceinline__ uint64_t same_digit(uint32_t d, uint32_t vary) {
    uint32_t miss_lo = 0, miss_hi = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        if (!((vary >> b) & 1u)) continue;
        const uint32_t m = (uint32_t)((int32_t)(d << (31 - b)) >> 31);
        const uint64_t bal = __ballot(m != 0u);
        miss_lo |= (uint32_t)bal ^ m;
        miss_hi |= (uint32_t)(bal >> 32) ^ m;
    }
    return ~(((uint64_t)miss_hi << 32) | miss_lo);
}

template <typename V> __device__ __forceinline__ V wave_incl_sum(V v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const V u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}

template <typename V> __device__ __forceinline__ V wave_incl_max(V v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const V u = __shfl_up(v, o, 64);
        if (lane >= o && u > v) v = u;
    }
    return v;
}

template <typename V> __device__ __forceinline__ V wave_sum(V v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
template <typename V> __device__ __forceinline__ V wave_and(V v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v &= __shfl_xor(v, o, 64);
    return v;
}
template <typename V> __device__ __forceinline__ V wave_or(V v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, 64);
    return v;
}

// rank of every member of the tie group at sorted positions [a, b) among n
// non-NaN values; rn = RN(1 / n) in double
template <typename T> __device__ __forceinline__ T group_rank(int a, int b, int n, double rn) {
    // rows of at most 16384 stocks: (a + b + 1) * (b - a) < 2^31, so the
    // reference's integer sum fits 32 bits and converts to T the same way
    const int32_t sum = (a + b + 1) * (b - a) / 2;
    // where the sum converts exactly, its quotient by b - a is (a + b + 1) / 2
    // exactly; only the largest tie groups of float rows need the division
    T q = (T)(a + b + 1) * T(0.5);
    if (sizeof(T) == 4 && sum >= 1 << 24) q = (T)sum / (T)(b - a);
    // q >= 1, so the float quotient is normal and the double product exact
    // (kun::div_rc)
    if constexpr (sizeof(T) == 4) return kun::div_const(q, rn, (float)n);
    else return q / (T)n;
}

// ---- Rank of long 64-bit rows: keys-only LSD radix sort -------------------
//
// For 64-bit keys of rows above 8192 stocks, whose (key, stock) pairs would
// not fit in LDS. A workgroup of BLOCK lanes (NW = BLOCK / 64 wavefronts)
// holds N = BLOCK x ITEMS keys in registers, wavefront w owning positions
// [w*64*ITEMS, (w+1)*64*ITEMS): item j of lane l is position
// w*64*ITEMS + j*64 + l (loads and stores of consecutive lanes are
// consecutive). Each pass sorts stably by one 8-bit digit:
//  1. ranking: per item, the lanes with the same digit are found by ballots
//     (same_digit); the lowest such lane adds their count to the wavefront's
//     own LDS histogram row, every lane's rank within its digit being the
//     row's previous count plus its lanes_below;
//  2. a block scan turns the histograms into starting positions, digit by
//     digit and within a digit wavefront by wavefront -- the order the
//     positions held -- so the pass is stable;
//  3. keys are scattered to LDS and read back.
// Digit positions on which every key of the row agrees are skipped (their
// stable pass would keep the order); the row's AND and OR of keys tell.
// Each lane then finds its own keys' tie groups by binary search in the
// sorted keys.
template <typename T, int BLOCK, int ITEMS> struct KeysRank {
    using K = typename KeyOf<T>::K;
    static constexpr int N = BLOCK * ITEMS;
    static constexpr int NW = BLOCK / 64;
    static_assert(NW % 4 == 0 && NW <= 16, "BLOCK must be 256, 512 or 1024");
    struct Smem {
        K key[N];                        // keys in sorted order
        uint32_t hist[NW][256];          // per wavefront digit counts, then starting positions
        uint32_t wv[NW];                 // per wavefront totals of the scans
        K wand[NW], wor[NW];
    };

    // hist := exclusive prefix in (digit, wavefront) order. Thread t owns
    // digit t / (NW/4) of wavefronts 4g .. 4g+3 (g = t % (NW/4)): thread
    // order is that order, so one block scan of per-thread sums does it.
    static __device__ __forceinline__ void scan_hist(Smem &sm) {
        constexpr int G = NW / 4;
        const int t = threadIdx.x, d = t / G, g = t % G, lane = t & 63, w = t >> 6;
        uint32_t v[4], s = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = sm.hist[4 * g + i][d];
            s += v[i];
        }
        const uint32_t incl = wave_incl_sum(s);
        if (lane == 63) sm.wv[w] = incl;
        __syncthreads();
        uint32_t run = incl - s;
        for (int q = 0; q < w; q++) run += sm.wv[q];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sm.hist[4 * g + i][d] = run;
            run += v[i];
        }
    }

    static __device__ __forceinline__ void row(Smem &sm, const kun_cs::View &in, const kun_cs::View &out, long S,
                                               int blk, long t) {
        if (S <= 0) return; // uniform: nothing to rank
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        const int base = w * 64 * ITEMS + lane;
        const T *src = (const T *)in.ptr;
        T *dst = (T *)out.ptr;
        const long rin = t + in.row0;
        K key[ITEMS];
        int cnt = 0;
        K kand = ~K(0), kor = K(0);
        // every load issued before any is used (stocks past S read the last
        // stock's cell and are then replaced by padding keys)
        T xs[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const long s = base + j * 64;
            xs[j] = src[cs_at(in.layout, rin, s < S ? s : S - 1, S, in.rows, blk)];
        }
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const long s = base + j * 64;
            const bool live = s < S;
            const K k = live ? rank_key(xs[j]) : ~K(0);
            cnt += (live && xs[j] == xs[j]) ? 1 : 0;
            key[j] = k;
            kand &= k;
            kor |= k;
        }
        cnt = wave_sum(cnt);
        kand = wave_and(kand);
        kor = wave_or(kor);
        if (lane == 0) {
            sm.wv[w] = (uint32_t)cnt;
            sm.wand[w] = kand;
            sm.wor[w] = kor;
        }
        __syncthreads();
        int n = 0;
#pragma unroll
        for (int q = 0; q < NW; q++) {
            n += (int)sm.wv[q];
            kand &= sm.wand[q];
            kor |= sm.wor[q];
        }
        const K diff = kand ^ kor; // bits on which the row's keys differ
        __syncthreads();           // sm.wv is the scans' from here on
        bool moved = false;
        for (int p = 0; p < (int)sizeof(K); p++) {
            const int sh = 8 * p;
            if (((diff >> sh) & K(0xff)) == K(0)) continue; // uniform over the workgroup
            moved = true;
            uint32_t *hw = sm.hist[w];
            // this wavefront's row only: its reads of the row in the
            // previous pass ended before the last barrier
            for (int q = lane; q < 256; q += 64) hw[q] = 0;
            // rank of each key within its digit among this wavefront's keys
            // before it, two 16-bit ranks per register
            uint32_t loc2[(ITEMS + 1) / 2];
            const uint32_t vary = (uint32_t)(diff >> sh) & 0xffu;
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const uint32_t d = (uint32_t)(key[j] >> sh) & 0xffu;
                const uint64_t peers = same_digit(d, vary);
                const uint32_t below = lanes_below(peers);
                const uint32_t prior = hw[d];
                if (below == 0) hw[d] = prior + (uint32_t)__popcll(peers);
                if (j % 2 == 0) loc2[j / 2] = prior + below;
                else loc2[j / 2] |= (prior + below) << 16;
                // one key at a time: interleaving the keys' ballot chains
                // buys no speed and costs the registers of a second
                // resident workgroup
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
            scan_hist(sm);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const uint32_t pos = hw[(uint32_t)(key[j] >> sh) & 0xffu] + ((loc2[j / 2] >> (16 * (j % 2))) & 0xffffu);
                sm.key[pos] = key[j];
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < ITEMS; j++) key[j] = sm.key[base + j * 64];
        }
        if (!moved) {
            // every key equal: the order is sorted as it stands
#pragma unroll
            for (int j = 0; j < ITEMS; j++) sm.key[base + j * 64] = key[j];
        }
        __syncthreads(); // the sorted keys are in sm.key
        // this lane's own keys again (the registers now hold sorted ones)
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const long s = base + j * 64;
            key[j] = rank_key(src[cs_at(in.layout, rin, s < S ? s : S - 1, S, in.rows, blk)]);
        }
#pragma unroll
        for (int j = 0; j < ITEMS; j++)
            if (base + j * 64 >= S) key[j] = ~K(0);
        rank_by_search(sm, key, n, dst, out, S, blk, t, base);
    }

    static __device__ __forceinline__ T rank_of(int a, int b, int n, double rn) { return group_rank<T>(a, b, n, rn); }

    static __device__ __forceinline__ void rank_by_search(Smem &sm, const K (&mine)[ITEMS], int n, T *dst,
                                                          const kun_cs::View &out, long S, int blk, long t,
                                                          int base) {
        const double rn = 1.0 / (double)n;
        // groups of G keys at a time, their searches interleaved
        constexpr int G = ITEMS < 4 ? ITEMS : 4;
#pragma unroll
        for (int j0 = 0; j0 < ITEMS; j0 += G) {
            // lower bounds
            int lo[G], len[G];
#pragma unroll
            for (int j = 0; j < G; j++) {
                lo[j] = 0;
                len[j] = n;
            }
            for (int step = 0; step < 32; step++) {
                bool any = false;
#pragma unroll
                for (int j = 0; j < G; j++) {
                    if (len[j] > 0) {
                        const int half = len[j] >> 1;
                        if (sm.key[lo[j] + half] < mine[j0 + j]) {
                            lo[j] += half + 1;
                            len[j] -= half + 1;
                        } else {
                            len[j] = half;
                        }
                        any = true;
                    }
                }
                if (!any) break;
            }
            // upper bounds, searched only for keys with ties
            int hi[G];
#pragma unroll
            for (int j = 0; j < G; j++) {
                hi[j] = lo[j] + 1;
                len[j] = (mine[j0 + j] != ~K(0) && hi[j] < n && sm.key[hi[j]] == mine[j0 + j]) ? n - hi[j] : 0;
            }
            for (int step = 0; step < 32; step++) {
                bool any = false;
#pragma unroll
                for (int j = 0; j < G; j++) {
                    if (len[j] > 0) {
                        const int half = len[j] >> 1;
                        if (!(mine[j0 + j] < sm.key[hi[j] + half])) {
                            hi[j] += half + 1;
                            len[j] -= half + 1;
                        } else {
                            len[j] = half;
                        }
                        any = true;
                    }
                }
                if (!any) break;
            }
#pragma unroll
            for (int j = 0; j < G; j++) {
                const long s = base + (j0 + j) * 64;
                if (s >= S) continue;
                const T r = (mine[j0 + j] != ~K(0) && lo[j] < n) ? rank_of(lo[j], hi[j], n, rn) : kun::qnan<T>();
                dst[cs_at(out.layout, t + out.row0, s, S, out.rows, blk)] = r;
            }
        }
    }
};

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ uint64_t lane_value(uint64_t v, int l) {
    return (uint64_t)lane_value((uint32_t)(v >> 32), l) << 32 | lane_value((uint32_t)v, l);
}

// the value CTRL brings from a lane before this one, 0 where there is none
template <int CTRL, int ROWS> __device__ __forceinline__ uint32_t dpp_before(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> __device__ __forceinline__ uint64_t dpp_before(uint64_t v) {
    return (uint64_t)dpp_before<CTRL, ROWS>((uint32_t)(v >> 32)) << 32 | dpp_before<CTRL, ROWS>((uint32_t)v);
}

// inclusive prefix sum / max over the 64 lanes by DPP row shifts and row
// broadcasts (rows of 16 lanes, then across rows); max assumes values >= 0
__device__ __forceinline__ uint32_t dpp_incl_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false); // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false); // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false); // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false); // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false); // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false); // row_bcast:31
    return v;
}
// inclusive prefix sum within each row of 16 lanes
__device__ __forceinline__ uint32_t dpp_row_incl_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false); // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false); // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false); // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false); // row_shr:8
    return v;
}
__device__ __forceinline__ int dpp_incl_max(int v) {
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
    return v;
}

// ---- Rank: LSD radix sort with per-lane digit counters -------------------
//
// The (key, stock) form for rows whose pairs fit in LDS. A workgroup of
// BLOCK lanes holds N = BLOCK x ITEMS keys in registers, lane t owning
// positions [t*ITEMS, (t+1)*ITEMS) (blocked; the first pass may start from
// any order, the loads are striped for coalescing). Each pass sorts stably by
// one 4-bit digit:
//  1. each lane counts its own keys' digits in registers, sixteen 4-bit
//     fields per 8 keys: a key's rank among the lane's earlier keys of its
//     digit is the fields' value before its increment. The counts go to the
//     lane's own column of the LDS table cnt[8][BLOCK], digit d in half
//     d >> 3 of word cnt[d & 7][t] -- no atomics, no ballots;
//  2. one block scan of the table in memory order (word-major, lane-minor:
//     digits 0-7 in the low halves, 8-15 in the high halves; adding the low
//     digits' total to every high half puts digits 8-15 after them) gives
//     each (digit, lane) the position of its first key;
//  3. keys and stocks are scattered to their positions in LDS and read back
//     blocked.
// Within a digit, positions go lane by lane and within a lane key by key --
// the order the positions held -- so each pass is stable. Digit positions
// on which every key of the row agrees are skipped (the row's AND and OR of
// keys tell). Tie groups come from a max-scan of group starts over the
// sorted positions.
template <typename T, int BLOCK, int ITEMS> struct CountRank {
    using K = typename KeyOf<T>::K;
    static constexpr int N = BLOCK * ITEMS;
    static constexpr int NW = BLOCK / 64;
    static constexpr int NG = (ITEMS + 7) / 8; // groups of up to 8 keys, one field register each
    static constexpr int NB = (int)sizeof(K) * 8;
    static_assert(BLOCK % 64 == 0 && NW <= 16, "BLOCK: 64..1024 lanes");
    static_assert(N <= 16384, "positions and counts are 16-bit");
    struct alignas(16) Smem {
        K key[N];                // sorted keys; scratch of the block scans; then group ends, ranks by stock
        uint16_t idx[N];         // stock at each position
        uint32_t cnt[8 * BLOCK]; // digit counts, then first positions; scratch of the group scan
    };

    static __device__ __forceinline__ uint32_t digit(K k, int sh) { return (uint32_t)(k >> sh) & 15u; }

    template <int LIN, int LOUT>
    static __device__ __forceinline__ void row(Smem &sm, const kun_cs::View &in, const kun_cs::View &out, long S,
                                               int blk, long t) {
        if (S <= 0) return; // uniform: nothing to rank
        const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
        const int wu = __builtin_amdgcn_readfirstlane(w); // w, known uniform
        const T *src = (const T *)in.ptr;
        T *dst = (T *)out.ptr;
        const long rin = t + in.row0;
        T xs[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const long s = w * 64 * ITEMS + j * 64 + lane;
            xs[j] = src[lay_at<LIN>(in, rin, s < S ? s : S - 1, S, blk)];
        }
        K key[ITEMS];
        uint32_t id2[(ITEMS + 1) / 2]; // stock of each key, two 16-bit ids per register
        int cnt = 0;
        K kand = ~K(0), kor = K(0);
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const long s = w * 64 * ITEMS + j * 64 + lane;
            const bool live = s < S;
            const K k = live ? rank_key(xs[j]) : ~K(0);
            cnt += (live && xs[j] == xs[j]) ? 1 : 0;
            key[j] = k;
            if (j % 2 == 0) id2[j / 2] = (uint32_t)s;
            else id2[j / 2] |= (uint32_t)s << 16;
            kand &= k;
            kor |= k;
        }
        cnt = wave_sum(cnt);
        kand = wave_and(kand);
        kor = wave_or(kor);
        // wavefront partials in the key area (its next writer, the first
        // pass's scan, comes after a barrier)
        K *xa = sm.key, *xo = sm.key + NW;
        uint32_t *xc = (uint32_t *)(sm.key + 2 * NW);
        if (lane == 0) {
            xa[w] = kand;
            xo[w] = kor;
            xc[w] = (uint32_t)cnt;
        }
        __syncthreads();
        // lane q < NW holds wavefront q's partials
        const int n = wave_sum(lane < NW ? (int)xc[lane] : 0);
        kand = wave_and(lane < NW ? xa[lane] : ~K(0));
        kor = wave_or(lane < NW ? xo[lane] : K(0));
        const K diff = kand ^ kor; // bits on which the row's keys differ
        const uint16_t *first16 = (const uint16_t *)sm.cnt;
        uint32_t *xs32 = (uint32_t *)sm.key; // scan scratch
        bool moved = false;
        for (int sh = 0; sh < NB; sh += 4) {
            if (digit(diff, sh) == 0u) continue; // uniform over the workgroup
            moved = true;
            // 1. per-lane counts; pre[j]: the earlier keys of this lane with
            // key j's digit
            uint64_t f[NG];
            uint32_t pre[ITEMS];
#pragma unroll
            for (int g = 0; g < NG; g++) f[g] = 0;
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const uint32_t d4 = digit(key[j], sh) * 4u;
                uint32_t p = 0;
#pragma unroll
                for (int g = 0; g < j / 8; g++) p += (uint32_t)(f[g] >> d4) & 15u;
                pre[j] = p + ((uint32_t)(f[j / 8] >> d4) & 15u);
                f[j / 8] += (uint64_t)1 << d4;
            }
            // kept as computed here rather than recomputed at the scatter
            // from eight 64-bit partial counts
#pragma unroll
            for (int j = 0; j < ITEMS; j++) asm volatile("" : "+v"(pre[j]));
#pragma unroll
            for (int k = 0; k < 8; k++) {
                uint32_t word = 0;
#pragma unroll
                for (int g = 0; g < NG; g++)
                    word += (((uint32_t)f[g] >> (4 * k)) & 15u) | ((((uint32_t)(f[g] >> 32) >> (4 * k)) & 15u) << 16);
                sm.cnt[k * BLOCK + tid] = word;
            }
            __syncthreads();
            // 2. exclusive scan of the table in memory order; lane t owns words [8t, 8t+8)
            uint4 *c4 = (uint4 *)sm.cnt;
            const uint4 lo = c4[2 * tid], hi = c4[2 * tid + 1];
            const uint32_t v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            uint32_t s = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) s += v[i];
            const uint32_t incl = dpp_incl_sum(s);
            if (lane == 63) xs32[w] = incl;
            __syncthreads();
            // wavefront totals: lane q of every wavefront holds the sum of
            // totals 0..q (prefix over the first 16 lanes)
            const uint32_t wp = dpp_row_incl_sum(lane < NW ? xs32[lane] : 0u);
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)wp, NW - 1);
            const uint32_t before = wu ? (uint32_t)__builtin_amdgcn_readlane((int)wp, wu - 1) : 0u;
            uint32_t run = before + incl - s + ((total & 0xffffu) << 16);
            uint32_t o[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                o[i] = run;
                run += v[i];
            }
            c4[2 * tid] = make_uint4(o[0], o[1], o[2], o[3]);
            c4[2 * tid + 1] = make_uint4(o[4], o[5], o[6], o[7]);
            __syncthreads();
            // 3. scatter to the sorted positions (every lookup issued before
            // the first store), read back blocked
            uint32_t pos[ITEMS];
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const uint32_t d = digit(key[j], sh);
                pos[j] = first16[((d & 7u) * BLOCK + tid) * 2 + (d >> 3)];
            }
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const uint32_t at = pos[j] + pre[j];
                sm.key[at] = key[j];
                sm.idx[at] = (uint16_t)(id2[j / 2] >> (16 * (j % 2)));
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < ITEMS; j++) key[j] = sm.key[tid * ITEMS + j];
            if constexpr (ITEMS % 2 == 0) {
                // stock pairs (2j, 2j+1) are adjacent: one word each
#pragma unroll
                for (int j = 0; j < ITEMS / 2; j++) id2[j] = ((const uint32_t *)sm.idx)[tid * ITEMS / 2 + j];
            } else {
                id2[0] = sm.idx[tid];
            }
        }
        if (!moved) {
            // every key equal: any order is sorted
            __syncthreads(); // the partials' readers are done
#pragma unroll
            for (int j = 0; j < ITEMS; j++) sm.key[tid * ITEMS + j] = key[j];
            __syncthreads();
        }
        ties<LOUT>(sm, key, id2, n, dst, out, S, blk, t);
    }

    static __device__ __forceinline__ T rank_of(int a, int b, int n, double rn) { return group_rank<T>(a, b, n, rn); }

    // sorted keys at positions P = tid*ITEMS + j (registers and sm.key)
    template <int LOUT>
    static __device__ __forceinline__ void ties(Smem &sm, const K (&key)[ITEMS], const uint32_t (&id2)[(ITEMS + 1) / 2],
                                                int n, T *dst, const kun_cs::View &out, long S, int blk, long t) {
        const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
        const int P0 = tid * ITEMS;
        // a[j]: start of key j's group (the last position <= P0 + j that starts one)
        int a[ITEMS];
        bool last[ITEMS];
        int cur = -1;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const bool first = j > 0 ? key[j - 1] != key[j] : (P0 == 0 || sm.key[P0 - 1] != key[0]);
            last[j] = j + 1 < ITEMS ? key[j] != key[j + 1] : (P0 + ITEMS == N || sm.key[P0 + ITEMS] != key[j]);
            if (first) cur = P0 + j;
            a[j] = cur;
        }
        // group start carried in from earlier lanes: exclusive max-scan of
        // (cur + 1), 0 meaning none
        const int incl = dpp_incl_max(cur + 1);
        int prev = __shfl_up(incl, 1, 64);
        if (lane == 0) prev = 0;
        int *xm = (int *)sm.cnt;
        if (lane == 63) xm[w] = incl;
        __syncthreads(); // also: every read of sm.key above is done
        int carry = prev;
#pragma unroll
        for (int q = 0; q < NW; q++) carry = q < w && xm[q] > carry ? xm[q] : carry;
        carry -= 1;
        int *endof = (int *)sm.key;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (a[j] < 0) a[j] = carry;
            const int P = P0 + j;
            if (P < n && last[j]) endof[a[j]] = P + 1;
        }
        __syncthreads();
        const double rn = 1.0 / (double)n;
        T r[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; j++) r[j] = P0 + j < n ? rank_of(a[j], endof[a[j]], n, rn) : kun::qnan<T>();
        __syncthreads();
        T *res = (T *)sm.key;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const int id = (int)((id2[j / 2] >> (16 * (j % 2))) & 0xffffu);
            if (id < S) res[id] = r[j];
        }
        __syncthreads();
        for (long s = tid; s < S; s += BLOCK) dst[lay_at<LOUT>(out, t + out.row0, s, S, blk)] = res[s];
    }
};

// ---- Rank: buckets that follow the row's distribution ----------------------
//
// Ranks need no sorted order, only how many keys lie below each key and how
// many equal it. The row is cut into buckets by a monotone map of the keys,
// fine enough that a bucket holds a key or two whatever the distribution:
//  1. a histogram of NC coarse buckets, the leading bits of key - smallest
//     key;
//  2. its prefix sum gives every coarse bucket as many position pairs as it
//     has keys, split evenly over its range: position = 2 * first + (fraction
//     within the bucket) * 2 * count. Within a coarse bucket (at most a
//     fraction of an octave where the row spans several) values are near
//     enough to evenly spread;
//  3. a histogram over the positions (16-bit counts, two to a word); a key's
//     turn in its bucket is the value its count had before it;
//  4. the prefix sum of that histogram gives each bucket its place, and the
//     keys are written there (sorted up to the order inside a bucket);
//  5. every lane, which still holds the keys it loaded, counts the smaller
//     and equal keys of each one's bucket, four at a time. Reading past a
//     bucket's end is harmless: later buckets hold larger keys, and the keys
//     end with four of the largest pattern.
// Buckets of more than DEEP keys are whole tie groups as a rule (discrete
// values): a lane whose key differs from its bucket's first one raises a
// flag, and unless some bucket of the row is both deep and mixed, a deep
// bucket's bounds are the tie group's. A row with such a bucket (values close
// together beside distant ones) is cut once more:
//  6. every bucket's range is divided evenly by two positions for each of its
//     keys, as coarse buckets were, and 3. to 5. follow.
// Where a bucket is deep and mixed after that too (clusters within clusters),
// nothing has been written and the row is sorted.
//
// 2 N positions (FSH = 0), or N / 2 (FSH = 2) where 64-bit keys leave less
// LDS.
//
// 1024 rows of 8192 floats: 37 us a launch, 92 by the sort (floor 13 us at
// the card's copy rate); 750 rows of 5003 doubles: 43 against 191, the sort
// needing 16 passes; one row of 5000 doubles: 12 against 54; a pool cycle's
// Rank segments of about 2200 stocks: 7.9 against 15. Rows of values within
// 1e-4 of each other and one of 1e30: 97 us for 1024 of 8192 floats (142 when
// such rows were sorted after the first cut, 92 by the sort alone), 69 for 750
// of 5003 doubles (227, 191). Within 1e-9, doubles end in the sort: 273 us, 246
// after one cut. Bound by LDS accesses
// and the instructions around them (about ten accesses a key, most of them
// to random banks). Two workgroups a CU are worth 43 -> 37 us for float rows
// of 8192 and take 64 registers, so values are packed and taken apart again
// rather than kept.
template <typename T, int BLOCK, int ITEMS, int FSH> struct BucketRank {
    using K = typename KeyOf<T>::K;
    static constexpr int N = BLOCK * ITEMS;
    static constexpr int NW = BLOCK / 64;
    static constexpr int NC = BLOCK * (FSH == 0 && ITEMS >= 4 ? ITEMS / 4 : 1);
    static constexpr int CW = NC / BLOCK;          // coarse buckets per lane
    static constexpr int FWORDS = N >> FSH;        // words of two positions
    static constexpr int FW = FWORDS / BLOCK;      // of them per lane
    static constexpr int DEEP = 64;
    static_assert(FW >= 1 && N <= 16384, "positions and counts are 16-bit");
    struct alignas(16) Smem {
        uint32_t fine[FWORDS + 4]; // counts, then first places, of the positions 2w and 2w + 1
        K key[N + 4];              // keys by bucket
        uint32_t coarse[NC + 1];   // counts, then first keys
        K wmax[NW], wmin[NW];
        uint32_t wn[NW], wc[NW], wf[NW];
        uint32_t mixed[2], n;
        int sh;
        K kmin;
    };

    static __device__ __forceinline__ uint32_t wave_max(uint32_t v) {
        v = max(v, dpp_before<0x111, 0xf>(v));
        v = max(v, dpp_before<0x112, 0xf>(v));
        v = max(v, dpp_before<0x114, 0xf>(v));
        v = max(v, dpp_before<0x118, 0xf>(v));
        v = max(v, dpp_before<0x142, 0xa>(v));
        v = max(v, dpp_before<0x143, 0xc>(v));
        return lane_value(v, 63);
    }
    static __device__ __forceinline__ uint64_t wave_max(uint64_t v) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const uint64_t u = __shfl_xor(v, o, 64);
            v = u > v ? u : v;
        }
        return v;
    }
    // sum of the wavefronts' totals before wavefront w
    static __device__ __forceinline__ uint32_t before(const uint32_t (&tot)[NW], int w, int lane) {
        const uint32_t p = dpp_row_incl_sum(lane < NW ? tot[lane] : 0u);
        return w ? lane_value(p, w - 1) : 0u;
    }

    // AGAIN: the row that this function left before with deep mixed buckets
    template <int LIN, int LOUT, bool AGAIN>
    static __device__ __forceinline__ bool row(Smem &sm, const kun_cs::View &in, const kun_cs::View &out, long S,
                                               int blk, long t) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
        const T *src = (const T *)in.ptr;
        T *dst = (T *)out.ptr;
        const long rin = t + in.row0;
        const int n_all = (int)S;
        K key[ITEMS]; // ~0: missing
        K kmin;
        uint32_t n = 0;
        int sh = 0;         // bits of key - kmin below the coarse bucket's
        uint32_t at[ITEMS]; // position, turn in the high half
        if constexpr (!AGAIN) {
            T xs[ITEMS];
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const int left = n_all - j * BLOCK;
                if (left > 0) xs[j] = *cell_at<LIN>(src, in, rin, j * BLOCK, min(tid, left - 1), S, blk);
            }
#pragma unroll
            for (int i = 0; i < CW; i++) sm.coarse[i * BLOCK + tid] = 0;
#pragma unroll
            for (int i = 0; i < FW; i++) sm.fine[i * BLOCK + tid] = 0;
            if (tid < 2) sm.mixed[tid] = 0;
            K kmax = 0, kinv = 0;
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                key[j] = tid < n_all - j * BLOCK ? rank_key(xs[j]) : ~K(0);
                const bool live = key[j] != ~K(0);
                n += (uint32_t)__popcll(__ballot(live));
                const K a = live ? key[j] : K(0), b = ~key[j];
                kmax = a > kmax ? a : kmax;
                kinv = b > kinv ? b : kinv; // a missing cell's is 0
            }
            kmax = wave_max(kmax);
            kinv = wave_max(kinv);
            if (lane == 0) {
                sm.wmax[w] = kmax;
                sm.wmin[w] = kinv;
                sm.wn[w] = n;
            }
            __syncthreads();
            // lane q < NW holds wavefront q's
            n = lane_value(dpp_row_incl_sum(lane < NW ? sm.wn[lane] : 0u), NW - 1);
            kmax = wave_max(lane < NW ? sm.wmax[lane] : K(0));
            kinv = wave_max(lane < NW ? sm.wmin[lane] : K(0));
            kmin = ~kinv;
            if (n && kmax != kmin) {
                const K range = kmax - kmin;
                const int bits = sizeof(K) == 8 ? 64 - __builtin_clzll((uint64_t)range) : 32 - __builtin_clz((uint32_t)range);
                constexpr int CB = __builtin_ctz(NC);
                sh = bits > CB ? bits - CB : 0;
            }
            sh = __builtin_amdgcn_readfirstlane(sh);
            // Missing cells go through the same instructions, adding nothing to a
            // count of their lane's own and storing the largest pattern where the
            // keys end with it anyway: no branch per cell.
            // 1. coarse counts
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const bool live = key[j] != ~K(0);
                atomicAdd(&sm.coarse[live ? (uint32_t)((key[j] - kmin) >> sh) : (uint32_t)tid], live ? 1u : 0u);
            }
            __syncthreads();
            // 2. first keys of the coarse buckets
            {
                uint32_t c[CW], s = 0;
#pragma unroll
                for (int i = 0; i < CW; i++) {
                    c[i] = sm.coarse[tid * CW + i];
                    s += c[i];
                }
                const uint32_t incl = dpp_incl_sum(s);
                if (lane == 63) sm.wc[w] = incl;
                __syncthreads();
                uint32_t run = before(sm.wc, w, lane) + incl - s;
#pragma unroll
                for (int i = 0; i < CW; i++) {
                    sm.coarse[tid * CW + i] = run;
                    run += c[i];
                }
                if (tid == 0) sm.coarse[NC] = n;
            }
            __syncthreads();
            // 3. positions, and each key's turn in its bucket
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const K r = key[j] != ~K(0) ? key[j] - kmin : K(0);
                const uint32_t b = (uint32_t)(r >> sh);
                const uint32_t c0 = sm.coarse[b], c1 = sm.coarse[b + 1];
                // the bits below the bucket's, as a 32-bit fraction of its range
                constexpr int TOP = (int)sizeof(K) * 8 - 1;
                const uint32_t frac = (uint32_t)(((r << 1) << (TOP - sh)) >> (TOP - 31));
                at[j] = (2 * c0 + __umulhi(frac, 2 * (c1 - c0))) >> FSH;
            }
        } else {
            // 6. What the first time left in LDS: the coarse buckets' first keys
            // and the positions' first places. A bucket's positions, two for
            // each of its keys, divide what was one position before. The keys
            // are loaded again, so that the first time keeps no register for it.
            n = lane_value(sm.n, 0);
            sh = __builtin_amdgcn_readfirstlane(sm.sh);
            kmin = lane_value(sm.kmin, 0);
#pragma unroll
            for (int j = 0; j < ITEMS; j++)
                key[j] = tid < n_all - j * BLOCK ? rank_key(*cell_at<LIN>(src, in, rin, j * BLOCK, tid, S, blk)) : ~K(0);
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const K r = key[j] != ~K(0) ? key[j] - kmin : K(0);
                const uint32_t b = (uint32_t)(r >> sh);
                const uint32_t c0 = sm.coarse[b], c1 = sm.coarse[b + 1];
                // the bits below the bucket's, as a 32-bit fraction of its range
                constexpr int TOP = (int)sizeof(K) * 8 - 1;
                const uint32_t frac = (uint32_t)(((r << 1) << (TOP - sh)) >> (TOP - 31));
                // the position, the key's fraction of it, and its bucket
                const uint32_t full = 2 * c0 + __umulhi(frac, 2 * (c1 - c0)), p = full >> FSH;
                uint32_t f = frac * (2 * (c1 - c0));
                if (FSH) f = __builtin_amdgcn_alignbit(full, f, FSH);
                const uint32_t sp = __builtin_amdgcn_alignbit(sm.fine[(p >> 1) + 1], sm.fine[p >> 1], (p & 1) * 16);
                at[j] = (2 * (sp & 0xffffu) + __umulhi(f, 2 * ((sp >> 16) - (sp & 0xffffu)))) >> FSH;
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < FW; i++) sm.fine[i * BLOCK + tid] = 0;
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const bool live = key[j] != ~K(0);
            at[j] = live ? at[j] : 2u * (uint32_t)tid;
            const uint32_t half = (at[j] & 1) * 16;
            const uint32_t old = atomicAdd(&sm.fine[at[j] >> 1], (live ? 1u : 0u) << half);
            at[j] |= (old >> half) << 16;
            // one register a key from here on, not the three it is made of
            asm volatile("" : "+v"(at[j]));
        }
        __syncthreads();
        // 4. first places of the buckets
        {
            uint32_t c[FW], s = 0;
#pragma unroll
            for (int i = 0; i < FW; i++) {
                c[i] = sm.fine[tid * FW + i];
                s += (c[i] & 0xffffu) + (c[i] >> 16);
            }
            const uint32_t incl = dpp_incl_sum(s);
            if (lane == 63) sm.wf[w] = incl;
            __syncthreads();
            uint32_t run = before(sm.wf, w, lane) + incl - s;
#pragma unroll
            for (int i = 0; i < FW; i++) {
                const uint32_t mid = run + (c[i] & 0xffffu);
                sm.fine[tid * FW + i] = run | mid << 16;
                run = mid + (c[i] >> 16);
            }
            if (tid == 0) sm.fine[FWORDS] = n;
            if (tid < 4) sm.key[n + tid] = ~K(0);
        }
        __syncthreads();
        uint32_t span[ITEMS]; // first place of the bucket, end in the high half
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const uint32_t p = at[j] & 0xffffu;
            span[j] = __builtin_amdgcn_alignbit(sm.fine[(p >> 1) + 1], sm.fine[p >> 1], (p & 1) * 16);
            sm.key[key[j] != ~K(0) ? (span[j] & 0xffffu) + (at[j] >> 16) : n] = key[j];
            asm volatile("" : "+v"(span[j]));
        }
        __syncthreads();
        // 5. deep buckets must be tie groups
        auto size = [&](int j) { return (int)(span[j] >> 16) - (int)(span[j] & 0xffffu); };
        bool deep = false;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) deep = deep || (key[j] != ~K(0) && size(j) > DEEP);
        if (__ballot(deep)) {
            bool mixed = false;
#pragma unroll
            for (int j = 0; j < ITEMS; j++) asm volatile("" : "+v"(span[j]));
#pragma unroll
            for (int j = 0; j < ITEMS; j++)
                if (key[j] != ~K(0) && size(j) > DEEP) mixed = mixed || sm.key[span[j] & 0xffffu] != key[j];
            if (__ballot(mixed) && lane == 0) sm.mixed[AGAIN] = 1;
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane((int)sm.mixed[AGAIN])) { // the same on every lane
            if (!AGAIN && tid == 0) {
                sm.kmin = kmin;
                sm.sh = sh;
                sm.n = n;
            }
            return false;
        }
        const double rn = 1.0 / (double)(int)n;
        constexpr int G = ITEMS < 16 / (int)sizeof(K) ? ITEMS : 16 / (int)sizeof(K); // keys counted side by side
#pragma unroll
        for (int j0 = 0; j0 < ITEMS; j0 += G) {
            K q[G][4];
            int lt[G], le[G];
            // bounds and sizes taken from the packed word again for every
            // group, rather than kept for all keys at once
#pragma unroll
            for (int g = 0; g < G; g++) asm volatile("" : "+v"(span[j0 + g]));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int u = 0; u < 4; u++) q[g][u] = sm.key[(span[j0 + g] & 0xffffu) + u];
#pragma unroll
            for (int g = 0; g < G; g++) {
                lt[g] = le[g] = 0;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    lt[g] += q[g][u] < key[j0 + g] ? 1 : 0;
                    le[g] += q[g][u] <= key[j0 + g] ? 1 : 0;
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                const int j = j0 + g, sz = size(j);
                const bool live = key[j] != ~K(0);
                const int a = (int)(span[j] & 0xffffu);
                if (live && sz > 4 && sz <= DEEP)
                    for (int i = a + 4; i < a + sz; i++) {
                        const K k = sm.key[i];
                        lt[g] += k < key[j] ? 1 : 0;
                        le[g] += k <= key[j] ? 1 : 0;
                    }
                if (sz > DEEP) le[g] = sz;
                const T r = live ? group_rank<T>(a + lt[g], a + le[g], (int)n, rn) : kun::qnan<T>();
                if (tid < n_all - j * BLOCK) *cell_at<LOUT>(dst, out, t + out.row0, j * BLOCK, tid, S, blk) = r;
            }
        }
        return true;
    }
};

// KIND 0: CountRank (pairs); 1: KeysRank (64-bit keys beyond 8192 stocks):
// how a row is sorted whose buckets are deep and mixed. LAY: both views'
// layout (-1: read from the views)
template <typename T, int BLOCK, int ITEMS, int KIND, int LAY>
__device__ __forceinline__ void rank_row_k(const kun_cs::View &in, const kun_cs::View &out, long S, int blk,
                                           const long t) {
    if (S <= 0) return; // uniform: nothing to rank
    using B = BucketRank<T, BLOCK, ITEMS, KIND == 0 ? 0 : 2>;
    using R = std::conditional_t<KIND == 0, CountRank<T, BLOCK, ITEMS>, KeysRank<T, BLOCK, ITEMS>>;
    __shared__ union Smem {
        typename B::Smem b;
        typename R::Smem r;
        __device__ Smem() {}
    } sm;
    if (B::template row<LAY, LAY, false>(sm.b, in, out, S, blk, t)) return;
    __syncthreads(); // what it left in the shared memory is there
    if (B::template row<LAY, LAY, true>(sm.b, in, out, S, blk, t)) return;
    __syncthreads(); // the flag's readers are done with the shared memory
    if constexpr (KIND == 0) R::template row<LAY, LAY>(sm.r, in, out, S, blk, t);
    else R::row(sm.r, in, out, S, blk, t);
}

// Wavefronts per SIMD the registers leave room for: two workgroups of 1024
// lanes share a CU where their LDS allows it (float rows up to 8192)
template <typename T, int BLOCK, int ITEMS> constexpr int rank_waves() {
    return BLOCK * ITEMS * (int)sizeof(T) <= 32768 ? 8 : 4;
}

// one workgroup per row of the views
template <typename T, int BLOCK, int ITEMS, int KIND, int LAY>
__global__ __launch_bounds__(BLOCK, (rank_waves<T, BLOCK, ITEMS>())) void rank_rows(kun_cs::View in, kun_cs::View out, long S, int blk) {
    rank_row_k<T, BLOCK, ITEMS, KIND, LAY>(in, out, S, blk, blockIdx.x);
}

// one workgroup per segment (a contiguous run of stocks of one row)
template <typename T, int BLOCK, int ITEMS, int KIND>
__global__ __launch_bounds__(BLOCK, (rank_waves<T, BLOCK, ITEMS>())) void rank_segs(const kun_cs::Seg *segs) {
    const kun_cs::Seg g = segs[blockIdx.x];
    const kun_cs::View in{const_cast<void *>(g.in), 2, 1, 0}, out{g.out, 2, 1, 0};
    rank_row_k<T, BLOCK, ITEMS, KIND, 2>(in, out, g.n, 1, 0);
}

// ---- Scale: row sums in stock order, a tile at a time ---------------------
//
// The reference adds |x| cell by cell, so the rounding of every add is part
// of the result and the plain form is one dependent add per stock: 8.9 clocks
// each on one wavefront, whatever else the GPU does. The sum of non-negative
// terms has more structure. While the running sum s stays inside one binade
// it is a multiple of one unit u, and adding x moves it by a whole number of
// units that depends on s only through whether s / u is odd (round to nearest
// even breaks a tie by that bit, and nothing else of s enters the rounding).
// A run of consecutive cells is therefore a function of that one bit, found
// by adding the run to the binade's first value and to the one after it, and
// such functions compose. So:
//  * a wavefront takes a tile of 64 x CHAIN_K cells, each lane CHAIN_K
//    consecutive ones, and every lane adds its cells to both starting values;
//  * a scan over the lanes composes the runs (a plain integer prefix sum
//    unless some lane met a tie);
//  * where the sum leaves the binade, the lanes before are taken, that lane's
//    cells are added one by one, and the rest of the tile starts over in the
//    new binade. The sum never falls, so a row leaves at most as many
//    binades as the type has, and about 13 for 8192 cells of like size.
// The result is the sequential sum bit for bit, infinities and subnormals
// included (a subnormal sum's unit is the smallest subnormal).
//
// 1024 rows of 8192 floats: 15.3 us a launch (2.2 TB/s), bound by the tiles'
// adds and scans on the one wavefront a SIMD has; the chain on one lane per
// row took 49.5 us. 750 rows of 5003 doubles: 13.0 us against 34.6; one row
// per session of a pool, about 2200 stocks, summed and divided: 10.3 us
// against 24.5.
constexpr int CHAIN_K = 16;
constexpr int CHAIN_TILE = 64 * CHAIN_K;
// Lanes' cells of a row's first tile that are added one by one. The sum leaves
// a binade with about every doubling of the cells it holds, which costs a scan
// and a start over, some 700 clocks, where an add takes nine: short rows were
// slower than by the chain. 1000 rows of 200 floats 9.0 us (10.7 by tiles
// from the first cell on, 8.9 by the chain alone), of 500 9.5 (11.5, 10.6), of
// 1000 10.8 (12.9, 13.7), of 3000 16.2 (17.9, 27.4); 20000 rows of 50 doubles
// 31 (44, 29). 16 lanes are as good for short rows and slower for 500 to 3000
// cells, 32 slower from 500 on.
constexpr int CHAIN_HEAD = 8;

// inclusive scan over the lanes of the runs' moves from an even (i0) and an
// odd (i1) sum, in units
template <int CTRL, int ROWS, typename U> __device__ __forceinline__ void compose_step(U &i0, U &i1) {
    const U l0 = dpp_before<CTRL, ROWS>(i0), l1 = dpp_before<CTRL, ROWS>(i1);
    const U r0 = l0 + ((l0 & 1) ? i1 : i0), r1 = l1 + ((l1 & 1) ? i0 : i1);
    i0 = r0;
    i1 = r1;
}
template <typename U> __device__ __forceinline__ void scan_runs(U &i0, U &i1) {
    compose_step<0x111, 0xf>(i0, i1); // row_shr:1, 2, 4, 8, then row_bcast:15, 31
    compose_step<0x112, 0xf>(i0, i1);
    compose_step<0x114, 0xf>(i0, i1);
    compose_step<0x118, 0xf>(i0, i1);
    compose_step<0x142, 0xa>(i0, i1);
    compose_step<0x143, 0xc>(i0, i1);
}
template <typename U> __device__ __forceinline__ U scan_units(U v) {
    v += dpp_before<0x111, 0xf>(v);
    v += dpp_before<0x112, 0xf>(v);
    v += dpp_before<0x114, 0xf>(v);
    v += dpp_before<0x118, 0xf>(v);
    v += dpp_before<0x142, 0xa>(v);
    v += dpp_before<0x143, 0xc>(v);
    return v;
}

// s plus the cells of a tile from lane `first` on, added in order (lane l holds
// cells l * CHAIN_K .. in v); v >= +0, not NaN; s is the same on every lane
template <typename T> __device__ __forceinline__ T add_in_order(T s, const T (&v)[CHAIN_K], int first) {
    using U = typename kun::Bits<T>::U;
    constexpr U LIM = U(1) << kun::Bits<T>::MANT; // units in a binade
    const int lane = threadIdx.x & 63;
    for (;;) {
        const U sb = kun::to_bits(s);
        if ((sb >> kun::Bits<T>::MANT) == (U(1) << kun::Bits<T>::EXPB) - 1) return s; // infinite: stays
        const U b0 = sb & ~(LIM - 1);
        T s0 = kun::from_bits<T>(b0), s1 = kun::from_bits<T>(b0 | 1);
#pragma unroll
        for (int k = 0; k < CHAIN_K; k++) {
            s0 = s0 + v[k];
            s1 = s1 + v[k];
        }
        // consecutive bit patterns are one unit apart; a run that leaves
        // the binade counts as LIM, which no sum takes
        U i0 = kun::to_bits(s0) - b0, i1 = kun::to_bits(s1) - (b0 | 1);
        i0 = i0 < LIM ? i0 : LIM;
        i1 = i1 < LIM ? i1 : LIM;
        if (lane < first) i0 = i1 = 0;
        U move;
        if (__ballot(i0 != i1)) {
            scan_runs(i0, i1);
            move = (sb & 1) ? i1 : i0;
        } else {
            move = scan_units(i0);
        }
        const uint64_t leaves = __ballot((sb & (LIM - 1)) + move >= LIM);
        if (!leaves) return kun::from_bits<T>(sb + lane_value(move, 63));
        const int l = __builtin_ctzll(leaves);
        T t = kun::from_bits<T>(l ? sb + lane_value(move, l - 1) : sb);
#pragma unroll
        for (int k = 0; k < CHAIN_K; k++) t = t + v[k];
        s = kun::from_bits<T>(lane_value(kun::to_bits(t), l));
        first = l + 1;
        if (first == 64) return s;
    }
}

// |x|, or +0 for a missing cell: adding +0 leaves the sum as it is
template <typename T> __device__ __forceinline__ T scale_term(T x) { return x == x ? kun::vabs(x) : T(0); }

// Sum of row `row` of the view, by one wavefront. Tiles are loaded two ahead
// (coalesced) and turned lane by lane through LDS; the four cells of padding
// per lane keep the reads of 16 bytes off each other's banks.
template <typename T> struct ChainTile {
    static constexpr int STRIDE = CHAIN_K + 16 / (int)sizeof(T);
    alignas(16) T cell[64 * STRIDE];
};
template <typename T, int LIN>
__device__ __forceinline__ T row_sum(ChainTile<T> &tile, const kun_cs::View &in, long row, long S, int blk) {
    const int lane = threadIdx.x & 63;
    const T *src = (const T *)in.ptr;
    auto load = [&](T (&x)[CHAIN_K], long c0) {
#pragma unroll
        for (int j = 0; j < CHAIN_K; j++) {
            const long s = c0 + j * 64 + lane;
            x[j] = s < S ? src[lay_at<LIN>(in, row, s, S, blk)] : T(0);
        }
    };
    T sum = T(0);
    auto add = [&](const T (&x)[CHAIN_K], auto head) {
#pragma unroll
        for (int j = 0; j < CHAIN_K; j++) {
            const int e = j * 64 + lane;
            tile.cell[e / CHAIN_K * ChainTile<T>::STRIDE + e % CHAIN_K] = scale_term(x[j]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        int first = 0;
        if constexpr (decltype(head)::value) {
            const int n = (int)(S < CHAIN_HEAD * CHAIN_K ? (S + CHAIN_K - 1) / CHAIN_K : CHAIN_HEAD);
            T g[CHAIN_K];
#pragma unroll
            for (int k = 0; k < CHAIN_K; k++) g[k] = tile.cell[k];
            for (; first < n; first++) {
                T h[CHAIN_K]; // (the last turn's is not used)
#pragma unroll
                for (int k = 0; k < CHAIN_K; k++) h[k] = tile.cell[(first + 1) * ChainTile<T>::STRIDE + k];
#pragma unroll
                for (int k = 0; k < CHAIN_K; k++) {
                    sum = sum + g[k];
                    g[k] = h[k];
                }
            }
            if (S <= CHAIN_HEAD * CHAIN_K) return;
        }
        T v[CHAIN_K];
#pragma unroll
        for (int k = 0; k < CHAIN_K; k++) v[k] = tile.cell[lane * ChainTile<T>::STRIDE + k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        sum = add_in_order(sum, v, first);
    };
    T x[CHAIN_K], y[CHAIN_K];
    load(x, 0);
    load(y, CHAIN_TILE);
    add(x, std::true_type{});
    for (long c0 = CHAIN_TILE; c0 < S; c0 += 2 * CHAIN_TILE) {
        load(x, c0 + CHAIN_TILE);
        add(y, std::false_type{});
        load(y, c0 + 2 * CHAIN_TILE);
        if (c0 + CHAIN_TILE < S) add(x, std::false_type{});
    }
    return sum;
}

// Many rows (batch runs): one wavefront per row leaves the sums in scratch
// and a second kernel divides every cell on all CUs; one row (stream ticks,
// pool segments): a workgroup whose first wavefront sums and which then
// divides. LIN / LOUT are the layouts (-1: read from the view at run time).
constexpr int SCALE_BLOCK = 256;

// Scratch of the split form: the rows' sums, then (float rows) RN(1/sum) in
// double at the next multiple of 8 bytes
template <typename T> __device__ __forceinline__ double *scale_rcs(T *sums, long rows) {
    return (double *)((char *)sums + ((size_t)rows * sizeof(T) + 7) / 8 * 8);
}

// x / tot, exactly as IEEE division, or NaN where x == 0 and tot == 0; float
// rows multiply by rc = RN(1/tot) in double (kun::div_rc)
__device__ __forceinline__ float scale_q(float x, float tot, double rc) {
    const float q = kun::div_rc(x, rc, tot);
    return (x == 0.f && tot == 0.f) ? kun::qnan<float>() : q;
}
__device__ __forceinline__ double scale_q(double x, double tot, double) {
    return (x == 0.0 && tot == 0.0) ? kun::qnan<double>() : x / tot;
}

template <typename T, int LIN>
__global__ __launch_bounds__(64) void scale_sums(kun_cs::View in, long S, long rows, int blk, T *sums) {
    __shared__ ChainTile<T> tile;
    const long r = blockIdx.x;
    const T sum = row_sum<T, LIN>(tile, in, r + in.row0, S, blk);
    if (threadIdx.x == 0) {
        sums[r] = sum;
        if (sizeof(T) == 4) scale_rcs(sums, rows)[r] = 1.0 / (double)sum;
    }
}

// one row per workgroup, summed and divided
template <typename T, int LIN, int LOUT>
__device__ __forceinline__ void scale_row(const kun_cs::View &in, const kun_cs::View &out, long S, int blk, long r) {
    __shared__ ChainTile<T> tile;
    __shared__ T total;
    if (threadIdx.x < 64) {
        const T sum = row_sum<T, LIN>(tile, in, r + in.row0, S, blk);
        if (threadIdx.x == 0) total = sum;
    }
    __syncthreads();
    const T *src = (const T *)in.ptr;
    T *dst = (T *)out.ptr;
    const T tot = total;
    const double rc = sizeof(T) == 4 ? 1.0 / (double)tot : 0.0;
    for (long s = threadIdx.x; s < S; s += SCALE_BLOCK) {
        const T x = src[lay_at<LIN>(in, r + in.row0, s, S, blk)];
        dst[lay_at<LOUT>(out, r + out.row0, s, S, blk)] = scale_q(x, tot, rc);
    }
}

template <typename T, int LIN, int LOUT>
__global__ __launch_bounds__(SCALE_BLOCK) void scale_rows(kun_cs::View in, kun_cs::View out, long S, int blk) {
    scale_row<T, LIN, LOUT>(in, out, S, blk, blockIdx.x);
}

// out = x / sum of its row, or NaN where x == 0 and the sum is 0: workgroup
// (x, y) takes SCALE_DIV_ITEMS x 256 stocks of rows y, y + gridDim.y, ...
constexpr int SCALE_DIV_ITEMS = 4;
template <typename T, int LIN, int LOUT>
__global__ __launch_bounds__(256) void scale_div(kun_cs::View in, kun_cs::View out, long S, long rows, int blk,
                                                 T *sums) {
    const long s0 = (long)blockIdx.x * (256 * SCALE_DIV_ITEMS) + threadIdx.x;
    const T *src = (const T *)in.ptr;
    T *dst = (T *)out.ptr;
    auto rows_of = [&](auto full) {
        for (long r = blockIdx.y; r < rows; r += gridDim.y) {
            const T tot = sums[r];
            const double rc = sizeof(T) == 4 ? scale_rcs(sums, rows)[r] : 0.0;
            T x[SCALE_DIV_ITEMS];
#pragma unroll
            for (int q = 0; q < SCALE_DIV_ITEMS; q++) {
                const long s = s0 + q * 256;
                x[q] = (full || s < S) ? src[lay_at<LIN>(in, r + in.row0, s, S, blk)] : T(0);
            }
#pragma unroll
            for (int q = 0; q < SCALE_DIV_ITEMS; q++) {
                const long s = s0 + q * 256;
                if (full || s < S) dst[lay_at<LOUT>(out, r + out.row0, s, S, blk)] = scale_q(x[q], tot, rc);
            }
        }
    };
    // whole workgroups of stocks take the unguarded copy
    if ((long)(blockIdx.x + 1) * (256 * SCALE_DIV_ITEMS) <= S)
        rows_of(std::true_type{});
    else
        rows_of(std::false_type{});
}

template <typename T> __global__ __launch_bounds__(SCALE_BLOCK) void scale_segs(const kun_cs::Seg *segs) {
    const kun_cs::Seg g = segs[blockIdx.x];
    const kun_cs::View in{const_cast<void *>(g.in), 2, 1, 0}, out{g.out, 2, 1, 0};
    scale_row<T, 2, 2>(in, out, g.n, 1, 0);
}

template <typename T, int LIN, int LOUT>
hipError_t launch_scale_split(const kun_cs::View &in, const kun_cs::View &out, long S, long rows, int blk,
                              kun_cs::Sink &sink, T *sums) {
    hipError_t e = sink_launch(sink, scale_sums<T, LIN>, dim3((unsigned)rows), dim3(64), in, S, rows, blk, sums);
    if (e != hipSuccess) return e;
    const long per = 256L * SCALE_DIV_ITEMS;
    return sink_launch(sink, scale_div<T, LIN, LOUT>,
                       dim3((unsigned)((S + per - 1) / per), (unsigned)(rows < 65535 ? rows : 65535)), dim3(256), in,
                       out, S, rows, blk, sums);
}

template <typename T>
hipError_t launch_scale_t(const kun_cs::View &in, const kun_cs::View &out, long S, long rows, int blk,
                          kun_cs::Sink &sink, void *scratch) {
    if (scratch && rows > 1) {
        T *sums = (T *)scratch;
        if (in.layout == 1 && out.layout == 1) return launch_scale_split<T, 1, 1>(in, out, S, rows, blk, sink, sums);
        return launch_scale_split<T, -1, -1>(in, out, S, rows, blk, sink, sums);
    }
    const dim3 grid((unsigned)rows);
    if (in.layout == 1 && out.layout == 1)
        return sink_launch(sink, scale_rows<T, 1, 1>, grid, dim3(SCALE_BLOCK), in, out, S, blk);
    if (in.layout == 2 && out.layout == 2)
        return sink_launch(sink, scale_rows<T, 2, 2>, grid, dim3(SCALE_BLOCK), in, out, S, blk);
    return sink_launch(sink, scale_rows<T, -1, -1>, grid, dim3(SCALE_BLOCK), in, out, S, blk);
}

template <typename T, int BLOCK, int ITEMS, int KIND>
hipError_t launch_rank_n(const kun_cs::View &in, const kun_cs::View &out, long S, long rows, int blk,
                         kun_cs::Sink &sink) {
    // rows of TS buffers (every batch run's temporaries) and single rows with
    // their addressing fixed at compile time; other layouts read the views'
    const dim3 grid((unsigned)rows), block(BLOCK);
    if (in.layout == 1 && out.layout == 1)
        return sink_launch(sink, rank_rows<T, BLOCK, ITEMS, KIND, 1>, grid, block, in, out, S, blk);
    if (in.layout == 2 && out.layout == 2)
        return sink_launch(sink, rank_rows<T, BLOCK, ITEMS, KIND, 2>, grid, block, in, out, S, blk);
    return sink_launch(sink, rank_rows<T, BLOCK, ITEMS, KIND, -1>, grid, block, in, out, S, blk);
}

// Workgroup shape by row length: at most 1024 lanes, up to 16 keys per lane;
// 64-bit keys of more than 8192 stocks sort without payloads (their pairs
// would not fit in LDS).
template <typename T>
hipError_t launch_rank_t(const kun_cs::View &in, const kun_cs::View &out, long S, long rows, int blk,
                         kun_cs::Sink &sink) {
    if (S <= 256) return launch_rank_n<T, 256, 1, 0>(in, out, S, rows, blk, sink);
    if (S <= 512) return launch_rank_n<T, 256, 2, 0>(in, out, S, rows, blk, sink);
    if (S <= 1024) return launch_rank_n<T, 256, 4, 0>(in, out, S, rows, blk, sink);
    if (S <= 2048) return launch_rank_n<T, 512, 4, 0>(in, out, S, rows, blk, sink);
    if (S <= 4096) return launch_rank_n<T, 1024, 4, 0>(in, out, S, rows, blk, sink);
    if (S <= 8192) return launch_rank_n<T, 1024, 8, 0>(in, out, S, rows, blk, sink);
    if (S <= 16384) return launch_rank_n<T, 1024, 16, sizeof(T) == 8 ? 1 : 0>(in, out, S, rows, blk, sink);
    return hipErrorInvalidValue;
}

template <typename T, int BLOCK, int ITEMS, int KIND>
hipError_t launch_rank_segs_n(const kun_cs::Seg *segs, int nseg, hipStream_t st) {
    hipLaunchKernelGGL((rank_segs<T, BLOCK, ITEMS, KIND>), dim3((unsigned)nseg), dim3(BLOCK), 0, st, segs);
    return hipGetLastError();
}

template <typename T> hipError_t launch_rank_segs_t(const kun_cs::Seg *segs, int nseg, long maxS, hipStream_t st) {
    if (maxS <= 256) return launch_rank_segs_n<T, 256, 1, 0>(segs, nseg, st);
    if (maxS <= 512) return launch_rank_segs_n<T, 256, 2, 0>(segs, nseg, st);
    if (maxS <= 1024) return launch_rank_segs_n<T, 256, 4, 0>(segs, nseg, st);
    if (maxS <= 2048) return launch_rank_segs_n<T, 512, 4, 0>(segs, nseg, st);
    if (maxS <= 4096) return launch_rank_segs_n<T, 1024, 4, 0>(segs, nseg, st);
    if (maxS <= 8192) return launch_rank_segs_n<T, 1024, 8, 0>(segs, nseg, st);
    if (maxS <= 16384) return launch_rank_segs_n<T, 1024, 16, sizeof(T) == 8 ? 1 : 0>(segs, nseg, st);
    return hipErrorInvalidValue;
}

} // namespace

namespace kun_cs {

hipError_t launch_rank_segs(int dtype, const Seg *segs, int nseg, long maxS, hipStream_t st) {
    if (nseg <= 0) return hipSuccess;
    return dtype ? launch_rank_segs_t<double>(segs, nseg, maxS, st) : launch_rank_segs_t<float>(segs, nseg, maxS, st);
}

hipError_t launch_scale_segs(int dtype, const Seg *segs, int nseg, hipStream_t st) {
    if (nseg <= 0) return hipSuccess;
    if (dtype)
        hipLaunchKernelGGL((scale_segs<double>), dim3((unsigned)nseg), dim3(SCALE_BLOCK), 0, st, segs);
    else
        hipLaunchKernelGGL((scale_segs<float>), dim3((unsigned)nseg), dim3(SCALE_BLOCK), 0, st, segs);
    return hipGetLastError();
}


long max_rank_stocks(int dtype) { return 16384; }

hipError_t launch_rank(int dtype, const View &in, const View &out, long S, long rows, int blk, Sink &sink) {
    if (rows <= 0) return hipSuccess;
    return dtype ? launch_rank_t<double>(in, out, S, rows, blk, sink)
                 : launch_rank_t<float>(in, out, S, rows, blk, sink);
}

hipError_t launch_rank(int dtype, const View &in, const View &out, long S, long rows, int blk, hipStream_t st) {
    StreamSink sink(st);
    return launch_rank(dtype, in, out, S, rows, blk, sink);
}

size_t scale_scratch_bytes(int dtype, long rows) {
    const size_t n = (size_t)(rows > 1 ? rows : 1);
    return dtype ? n * 8 : (n * 4 + 7) / 8 * 8 + n * 8;
}

hipError_t launch_scale(int dtype, const View &in, const View &out, long S, long rows, int blk, Sink &sink,
                        void *scratch) {
    if (rows <= 0) return hipSuccess;
    return dtype ? launch_scale_t<double>(in, out, S, rows, blk, sink, scratch)
                 : launch_scale_t<float>(in, out, S, rows, blk, sink, scratch);
}

hipError_t launch_scale(int dtype, const View &in, const View &out, long S, long rows, int blk, hipStream_t st,
                        void *scratch) {
    StreamSink sink(st);
    return launch_scale(dtype, in, out, S, rows, blk, sink, scratch);
}

} // namespace kun_cs
