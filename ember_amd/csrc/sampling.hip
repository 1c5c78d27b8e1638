// Token sampling on gfx950, one work-group (16 waves) per row of logits.
//
// Replaces the reference's sample_kernel / prob_kernel
// (src/backend/cuda/k_sampling.cu:149-198) with the distribution its host
// sampler defines (src/backend/sampling_host.cpp:20-66), in that order:
// temperature, top-k, top-p over the top-k set's mass, then min-p relative to
// the most likely token. Each cut keeps a prefix of the order the host sorts
// by (scaled logit v = x / temperature descending, token id ascending): a
// threshold theta and the last id kept at it (kept iff v > theta, or v ==
// theta and id <= id_cut), so tokens tied at a boundary are kept lowest id
// first, as many as the count or mass asks for. Min-p keeps exp(v - max) >=
// min_p. The token is argmax over the kept set of v + Gumbel noise (the Gumbel-max trick,
// sampling_rng.hpp:20-33: the noise depends only on (seed, counter, token id),
// so a row draws the same token in any batch). Greedy rows (temperature <=
// 1e-5) take the first largest logit. Rows whose largest v is not finite have no
// masses to cut by; they take the first largest v, as the host's draw does (a
// +inf logit wins over any noise; token 0 when all are -inf or NaN).
//
// What bounds it: passes of one CU over the row (608 KB at 151,936 logits, 6 to
// 10 us each), so the cuts are found in few of them. All sums are integers
// (counts, and exp(v - max) in 2^-40 fixed point), so they are the same
// whatever order the LDS atomics land in, and the kept set is a deterministic
// function of the logits (float atomics would make it depend on scheduling at
// the boundary). Two ways, the first that applies:
//  - candidates: a lower bound of the k-th largest logit from the threads'
//    maxima (one pass), then the few elements at or above it are collected,
//    sorted in LDS, and every cut, the mass and the draw come from that list;
//  - bins: a histogram over 1/64-wide steps below the maximum (one pass), then
//    the elements of the one bin that the cut falls in are collected and sorted.
//    While they are more than the list holds and differ, their range of keys
//    (order-preserving uint32 of v) is split into as many bins again; a tie's
//    cut is then found by radix over the ids.
// 16 rows of 151,936, top-k 40 and top-p 0.9: sample 27 us (303 by radix alone),
// token_probs 25 us (276); top-p 0.95 alone, by bins: 133 us (289) and 92 (248).
// Sample, masked to 30 tokens, top-k 40 and top-p 0.9: 107 us (1042); 80 distinct
// logits, top-p 0.95: 303 (523); all equal: 485 (1046), most of it in passes
// whose atomics all go to one bin.
#include <cstdint>
#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"

namespace ember::hip {
namespace {

constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / kWave;
constexpr double kFix = 1099511627776.0;  // 2^40: exp weights in (0, 1] as fixed point, V * 2^40 < 2^64

__device__ __forceinline__ uint32_t order_key(float f) {  // ascending floats -> ascending keys
    const uint32_t b = __float_as_uint(f + 0.0f);  // -0 orders as +0
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// SplitMix64's output function (sampling_rng.hpp:22-27) and the Gumbel(0, 1)
// noise of token `id` at draw `counter` (:30-33).
__device__ __forceinline__ uint64_t rng_mix(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ float gumbel_noise(uint64_t seed, uint64_t counter, uint32_t id) {
    const uint64_t h = rng_mix(seed ^ rng_mix(counter * 0x632BE59BD9B4E019ull + id));
    const float u = (static_cast<float>(h >> 40) + 0.5f) * (1.0f / 16777216.0f);  // in (0, 1)
    return -logf(-logf(u));
}

constexpr int kList = 2 * kSampleThreads;  // elements a cut's list holds
constexpr int kBins = 2 * kSampleThreads;  // of 1 / kBinsPerUnit each, below the largest scaled logit
constexpr float kBinsPerUnit = 64.0f;
// The largest top-k whose candidates are looked for: 512, where a pass over the row costs more than sorting the 1000 or
// so that they are (16 rows of 151,936, top-k 512: 45 us, by bins 115); in short rows less (token_probs of 4 rows of
// 8192, top-k 512: 19 to 23 us, by bins 19, before either 20; top-k 200: 16.4, 18.5).
__device__ __forceinline__ int most_candidates(int V) { return max(128, min(512, V / 32)); }

struct SampleLds {
    unsigned long long hist[256];
    unsigned long long wsum[kSampleWaves];
    float wmax[kSampleWaves];
    int widx[kSampleWaves];
    uint32_t prefix, mask;
    unsigned long long above;  // after a selection: the weight (or count) before what it found
    unsigned long long bins[kBins];
    unsigned long long list[kList];  // elements as (key of v, ~id): descending is the order of the cuts
    int listed;
    uint32_t low, high;  // the keys of a bin's last and first elements
};

// A prefix of the (v descending, id ascending) order.
struct Cut {
    float theta = -INFINITY;
    int id_cut = 0x7fffffff;
    __device__ __forceinline__ bool keeps(float v, int i) const { return v > theta || (v == theta && i <= id_cut); }
};

__device__ __forceinline__ float scaled(const float *x, int i, float t) { return x[i] / t; }

// Calls f(i, x[i]) for this thread's elements of a row (i = tid, tid + 1024,
// ..., ascending), with the loads of kRowBatch elements issued together: one
// memory round trip per batch instead of one per element (a 151,936-logit row
// is 148 elements per thread).
constexpr int kRowBatch = 16;
// In passes that few rows take (a bin of thousands, a tie's ids): the same time there within 1%, and less code, whose
// fetching the short launches feel (top-k 40, 16 rows of 151,936: with 81 KB of code 29.5 us, with 71 KB 28.9).
constexpr int kRareBatch = 8;
template <int B = kRowBatch, class F>
__device__ __forceinline__ void for_row(const float *x, int V, F f) {
    int i = static_cast<int>(threadIdx.x);
    for (; i + (B - 1) * kSampleThreads < V; i += B * kSampleThreads) {
        float v[B];
#pragma unroll
        for (int u = 0; u < B; u++) v[u] = x[i + u * kSampleThreads];
#pragma unroll
        for (int u = 0; u < B; u++) f(i + u * kSampleThreads, v[u]);
    }
    for (; i < V; i += kSampleThreads) f(i, x[i]);
}

__device__ __forceinline__ float block_max(float v, SampleLds &sh) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    const int wave = static_cast<int>(threadIdx.x) / kWave;
    __syncthreads();
    if (threadIdx.x % kWave == 0) sh.wmax[wave] = v;
    __syncthreads();
    float m = sh.wmax[0];
    for (int w = 1; w < kSampleWaves; w++) m = fmaxf(m, sh.wmax[w]);
    return m;
}

__device__ __forceinline__ unsigned long long block_sum_u64(unsigned long long v, SampleLds &sh) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    const int wave = static_cast<int>(threadIdx.x) / kWave;
    __syncthreads();
    if (threadIdx.x % kWave == 0) sh.wsum[wave] = v;
    __syncthreads();
    unsigned long long s = 0;
    for (int w = 0; w < kSampleWaves; w++) s += sh.wsum[w];
    return s;
}

// The sum of v over the threads before this one (and, in total, over all).
__device__ __forceinline__ unsigned long long block_scan_u64(unsigned long long v, SampleLds &sh, unsigned long long &total) {
    const int lane = static_cast<int>(threadIdx.x) % kWave, wave = static_cast<int>(threadIdx.x) / kWave;
    unsigned long long incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned long long up = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += up;
    }
    __syncthreads();
    if (lane == kWave - 1) sh.wsum[wave] = incl;
    __syncthreads();
    unsigned long long before = 0;
    total = 0;
    for (int w = 0; w < kSampleWaves; w++) {
        if (w < wave) before += sh.wsum[w];
        total += sh.wsum[w];
    }
    return before + incl - v;
}

// The weight exp(v - mx) in (0, 1] as fixed point, rounded down: the f32
// value's 24 significand bits, shifted (the same integer as through double).
__device__ __forceinline__ unsigned long long fixed_weight(float v, float mx) {
    const uint32_t b = __float_as_uint(expf(v - mx));
    const int e = static_cast<int>(b >> 23);  // 0 (zero, subnormal) to 127; 255 for a NaN
    const unsigned long long m = (b & 0x7fffffu) | 0x800000u;
    const int up = e - (127 + 23 - 40);
    return up >= 0 ? (e > 127 ? 0ull : m << up) : up > -24 && e > 0 ? m >> -up : 0ull;
}

__device__ __forceinline__ unsigned long long list_entry(float v, int i) {
    return static_cast<unsigned long long>(order_key(v)) << 32 | static_cast<uint32_t>(~i);
}
__device__ __forceinline__ float entry_value(unsigned long long e) { return key_value(static_cast<uint32_t>(e >> 32)); }
__device__ __forceinline__ int entry_id(unsigned long long e) { return static_cast<int>(~static_cast<uint32_t>(e)); }

// Sorts sh.list[0, n) descending, n <= kList; every thread calls it. Entries
// past n are overwritten with 0, which orders after every entry.
__device__ __forceinline__ void sort_list(int n, SampleLds &sh) {
    const int tid = static_cast<int>(threadIdx.x);
    int size = 2;
    while (size < n) size *= 2;
    __syncthreads();
    for (int i = n + tid; i < size; i += kSampleThreads) sh.list[i] = 0;
    __syncthreads();
    // Up to j = 64 a wave's pairs lie within its own 128 entries, and its LDS operations run in order: those steps need no
    // barrier, and waves without entries no part in them. (A barrier after each of the 66 steps of 2048 entries: 3 us more.)
    auto step = [&](int k, int j) {
        if (tid < size / 2) {  // pair (i, i + j); kList / 2 threads at most
            const int i = 2 * tid - (tid & (j - 1));
            const unsigned long long a = sh.list[i], b = sh.list[i + j];
            if (((i & k) == 0) == (a < b)) {
                sh.list[i] = b;
                sh.list[i + j] = a;
            }
        }
    };
    auto narrow = [&](int k, int j) {
        if (tid - tid % kWave >= size / 2) return;
        for (; j > 0; j /= 2) {
            step(k, j);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
        }
    };
    for (int k = 2; k <= min(size, 2 * kWave); k *= 2) narrow(k, k / 2);
    for (int k = 4 * kWave; k <= size; k *= 2) {
        __syncthreads();
        for (int j = k / 2; j > kWave; j /= 2) {
            step(k, j);
            __syncthreads();
        }
        narrow(k, kWave);
    }
    __syncthreads();
}

// The index of the threads' largest best (ties to the lowest; 0 if none is above -inf).
__device__ __forceinline__ int block_first_largest(float best, int idx, SampleLds &sh) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, kWave);
        const int oi = __shfl_xor(idx, o, kWave);
        if (ob > best || (ob == best && oi < idx)) {
            best = ob;
            idx = oi;
        }
    }
    const int wave = static_cast<int>(threadIdx.x) / kWave;
    __syncthreads();
    if (threadIdx.x % kWave == 0) {
        sh.wmax[wave] = best;
        sh.widx[wave] = idx;
    }
    __syncthreads();
    best = sh.wmax[0];
    idx = sh.widx[0];
    for (int w = 1; w < kSampleWaves; w++)
        if (sh.wmax[w] > best || (sh.wmax[w] == best && sh.widx[w] < idx)) {
            best = sh.wmax[w];
            idx = sh.widx[w];
        }
    return idx == 0x7fffffff ? 0 : idx;
}

// First largest score(i, x[i]) over i < V (ties to the lowest index).
template <int B = kRowBatch, class F>
__device__ __forceinline__ int block_argmax(const float *x, int V, F score, SampleLds &sh) {
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for_row<B>(x, V, [&](int i, float xi) {
        const float v = score(i, xi);
        if (v > best) {  // i ascends per thread: the first of equal values is kept
            best = v;
            idx = i;
        }
    });
    return block_first_largest(best, idx, sh);
}

// The r-th lowest id (r >= 1) among the elements `within` keeps whose v equals
// theta: a radix selection over the ids, 8 bits per pass from the top, counting
// from the lowest bin up.
__device__ __forceinline__ int kth_tied_id(const float *x, int V, float t, const Cut within, float theta, unsigned long long r,
                           SampleLds &sh) {
    const int tid = static_cast<int>(threadIdx.x);
    if (tid == 0) {
        sh.prefix = 0;
        sh.mask = 0;
        sh.above = 0;  // here: the count below the bins looked at so far
    }
    for (int shift = V > 1 ? (31 - __clz(V - 1)) / 8 * 8 : 0; shift >= 0; shift -= 8) {  // ids below V have no higher bytes
        for (int i = tid; i < 256; i += kSampleThreads) sh.hist[i] = 0;
        __syncthreads();
        const uint32_t prefix = sh.prefix, mask = sh.mask;
        for_row<kRareBatch>(x, V, [&](int i, float xi) {
            const float v = xi / t;
            if (v != theta || !within.keeps(v, i) || (static_cast<uint32_t>(i) & mask) != prefix) return;
            atomicAdd(&sh.hist[(static_cast<uint32_t>(i) >> shift) & 255u], 1ull);
        });
        __syncthreads();
        if (tid < kWave) {  // wave 0 finds the digit: lane l holds bins 4l .. 4l + 3
            unsigned long long mine = 0;
            for (int j = 0; j < 4; j++) mine += sh.hist[4 * tid + j];
            unsigned long long incl = mine;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const unsigned long long up = __shfl_up(incl, o, kWave);
                if (tid >= o) incl += up;
            }
            const unsigned long long below = sh.above;
            const bool hit = below + incl >= r;
            const unsigned long long ballot = __ballot(hit);
            const int first = ballot ? __ffsll(static_cast<long long>(ballot)) - 1 : kWave - 1;
            if (tid == first) {
                unsigned long long cum = below + (incl - mine);
                int d = 4 * tid;
                for (int j = 0; j < 3; j++, d++) {
                    if (cum + sh.hist[d] >= r) break;
                    cum += sh.hist[d];
                }
                sh.above = cum;
                sh.prefix = prefix | (static_cast<uint32_t>(d) << shift);
                sh.mask = mask | (255u << shift);
            }
        }
        __syncthreads();
    }
    return static_cast<int>(sh.prefix);
}

__device__ __forceinline__ unsigned long long top_p_target(float top_p, unsigned long long mass) {
    const double want = ceil(static_cast<double>(top_p) * static_cast<double>(mass));
    return want < 1.0 ? 1ull : static_cast<unsigned long long>(want);
}

// The first bin, from 0 up, at which the sums of sh.bins and `above` reach the
// target (set from the sum of all where target_of says so): true, with sh.prefix
// the bin and sh.above the weight before it, or false if they never do.
template <class F>
__device__ __forceinline__ bool find_bin(unsigned long long above, F target_of, unsigned long long &total, SampleLds &sh) {
    const int tid = static_cast<int>(threadIdx.x);
    const unsigned long long b0 = sh.bins[2 * tid], b1 = sh.bins[2 * tid + 1];
    const unsigned long long before = above + block_scan_u64(b0 + b1, sh, total), target = target_of(total);
    if (before < target && before + b0 + b1 >= target) {  // one thread at most
        sh.prefix = static_cast<uint32_t>(2 * tid + (before + b0 >= target ? 0 : 1));
        sh.above = before + (before + b0 >= target ? 0 : b0);
    }
    __syncthreads();
    return above + total >= target;
}

// The prefix of `within` (in the cuts' order) whose weight first reaches the
// target: `top_k` elements (top_p < 0), or top_p of the mass of `within`; all of
// it if it holds less. `kept`: the prefix's weight. Elements of -inf, which have
// no mass and are never drawn, are not counted: a row masked to fewer than top_k
// tokens keeps them all and looks for no cut among the rest.
__device__ __forceinline__ Cut prefix_cut(const float *x, int V, float t, const Cut within, float mx, int top_k,
                                          float top_p, unsigned long long &kept, SampleLds &sh) {
    const int tid = static_cast<int>(threadIdx.x);
    const bool prob = top_p >= 0.0f;
    using Batch = std::integral_constant<int, kRowBatch>;
    using Rare = std::integral_constant<int, kRareBatch>;
    auto weight = [&](float v) { return prob ? fixed_weight(v, mx) : 1ull; };
    // The sums of bin_of(v)'s bins over the elements of `within` above -inf (bin < 0: left out).
    auto fill_bins = [&](auto batch, auto bin_of) {
        __syncthreads();
        for (int i = tid; i < kBins; i += kSampleThreads) sh.bins[i] = 0;
        __syncthreads();
        for_row<decltype(batch)::value>(x, V, [&](int i, float xi) {
            const float v = xi / t;
            if (!(v > -INFINITY)) return;
            const int b = bin_of(v);
            if (b < 0 || !within.keeps(v, i)) return;
            const unsigned long long w = weight(v);
            if (w) atomicAdd(&sh.bins[b], w);
        });
        __syncthreads();
    };
    // The elements of `within` above -inf that in(v) takes, into sh.list: how many they are and, where the list does not
    // hold them, their lowest and highest key.
    uint32_t low = 0, high = 0;
    auto collect = [&](auto batch, auto in) {
        if (tid == 0) {
            sh.listed = 0;
            sh.low = ~0u;
            sh.high = 0;
        }
        __syncthreads();
        low = ~0u;
        high = 0;
        for_row<decltype(batch)::value>(x, V, [&](int i, float xi) {
            const float v = xi / t;
            if (!(v > -INFINITY) || !in(v) || !within.keeps(v, i)) return;
            const int at = atomicAdd(&sh.listed, 1);
            if (at < kList) sh.list[at] = list_entry(v, i);
            low = min(low, order_key(v));
            high = max(high, order_key(v));
        });
        __syncthreads();
        const int found = sh.listed;
        if (found > kList) {
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) {
                low = min(low, static_cast<uint32_t>(__shfl_xor(static_cast<int>(low), o, kWave)));
                high = max(high, static_cast<uint32_t>(__shfl_xor(static_cast<int>(high), o, kWave)));
            }
            if (tid % kWave == 0) {
                atomicMin(&sh.low, low);
                atomicMax(&sh.high, high);
            }
            __syncthreads();
            low = sh.low;
            high = sh.high;
        }
        return found;
    };

    // (mx - v) rounds the same way for equal v and never orders two v the other way round, so bins follow the order.
    auto step_of = [&](float v) {
        const float d = (mx - v) * kBinsPerUnit;
        return d < static_cast<float>(kBins - 1) ? static_cast<int>(d) : kBins - 1;
    };
    fill_bins(Batch{}, step_of);
    unsigned long long target = 0;
    auto set_target = [&](unsigned long long total) {
        return target = prob ? top_p_target(top_p, total) : static_cast<unsigned long long>(top_k);
    };
    if (!find_bin(0, set_target, kept, sh)) return within;
    const int step = static_cast<int>(sh.prefix);
    unsigned long long above = sh.above;
    int n = collect(Batch{}, [&](float v) { return step_of(v) == step; });
#pragma unroll 1
    while (n > kList && low < high) {  // at most three times: 32 bits of key, 11 of them a time
        const int shift = max(0, 32 - __clz(static_cast<int>(high - low)) - 11);  // (high - low) >> shift < kBins
        const uint32_t lo = low, hi = high;
        fill_bins(Rare{}, [&](float v) {
            const uint32_t k = order_key(v) - lo;
            return k > hi - lo ? -1 : kBins - 1 - static_cast<int>(k >> shift);
        });
        unsigned long long sum;
        find_bin(above, [&](unsigned long long) { return target; }, sum, sh);
        const uint32_t part = static_cast<uint32_t>(kBins - 1) - sh.prefix;
        above = sh.above;
        __syncthreads();  // every thread has read sh before it is reused
        n = collect(Rare{}, [&](float v) {
            const uint32_t k = order_key(v) - lo;
            return k <= hi - lo && k >> shift == part;
        });
    }
    Cut c;
    if (n <= kList) {
        sort_list(n, sh);
        const unsigned long long e0 = 2 * tid < n ? sh.list[2 * tid] : 0, e1 = 2 * tid + 1 < n ? sh.list[2 * tid + 1] : 0;
        const unsigned long long w0 = 2 * tid < n ? weight(entry_value(e0)) : 0;
        const unsigned long long w1 = 2 * tid + 1 < n ? weight(entry_value(e1)) : 0;
        unsigned long long all;
        const unsigned long long pre = above + block_scan_u64(w0 + w1, sh, all);
        __syncthreads();
        if (pre < target && pre + w0 + w1 >= target) {
            const bool first = pre + w0 >= target;
            sh.list[0] = first ? e0 : e1;  // every thread has read its entries
            sh.above = pre + (first ? w0 : w0 + w1);
        }
        __syncthreads();
        c.theta = entry_value(sh.list[0]);
        c.id_cut = entry_id(sh.list[0]);
        kept = sh.above;
        return c;
    }
    // One value, more often than the list holds: the lowest ids of the tie, as many as reach the target.
    const unsigned long long each = weight(key_value(high)), need = (target - above + each - 1) / each;
    c.theta = key_value(high);
    if (need < static_cast<unsigned long long>(n)) c.id_cut = kth_tied_id(x, V, t, within, c.theta, need, sh);
    kept = above + min(need, static_cast<unsigned long long>(n)) * each;
    return c;
}

struct Dist {
    bool greedy;
    bool certain;  // the largest v is not finite: nothing below it is settled
    float t, mx, min_w;
    float least;           // every logit that min_w keeps is above it
    Cut k, p;              // the top-k and top-p cuts (the top-p one lies inside the top-k one)
    unsigned long long z;  // fixed-point mass of the kept set (where asked for)
    int listed;            // the kept set is within sh.list[0, listed), sorted; 0: not listed
    __device__ __forceinline__ bool keeps(float v, int i) const { return k.keeps(v, i) && p.keeps(v, i) && expf(v - mx) >= min_w; }
};

// Rows whose kept set is among few elements: those at or above a bound that
// the threads' maxima give. top-k: at least top_k threads (ceil(top_k / 16) of
// each wave's) have a maximum at or above it, so the top_k first elements do.
// Without cuts: min-p, by its own bound; that list needs no order. Returns
// false, with nothing settled, when the bound lets too many through.
__device__ __forceinline__ bool few_candidates(const float *x, int V, const EmberSampleParams &p, float thread_max, bool cuts,
                                               Dist &d, SampleLds &sh) {
    const int tid = static_cast<int>(threadIdx.x), lane = tid % kWave;
    const bool by_k = p.top_k > 0 && p.top_k <= most_candidates(V) && p.top_k < V;
    if (!by_k && (cuts || !(d.least > -INFINITY))) return false;
    float bound;
    if (by_k) {
        float m = thread_max;  // the wave's maxima, sorted descending over its lanes
        for (int k = 2; k <= kWave; k *= 2)
            for (int j = k / 2; j > 0; j /= 2) {
                const float o = __shfl_xor(m, j, kWave);
                const bool larger = ((lane & j) == 0) == ((lane & k) == 0);  // this lane keeps the larger of the two
                m = larger ? fmaxf(m, o) : fminf(m, o);
            }
        const float mine = __shfl(m, (p.top_k + kSampleWaves - 1) / kSampleWaves - 1, kWave);
        bound = -block_max(-mine, sh);
        // Quotients of nearby logits can be equal: elements within rounding of the bound count too.
        bound -= fabsf(bound) * 0x1p-20f + 1e-30f;
    } else {
        bound = d.least;
    }
    if (!(bound / d.t > -INFINITY)) return false;  // quotients that overflow are all equal
    __syncthreads();
    if (tid == 0) sh.listed = 0;
    __syncthreads();
    for_row(x, V, [&](int i, float xi) {
        if (!(xi >= bound)) return;
        const int at = atomicAdd(&sh.listed, 1);
        if (at < kList) sh.list[at] = list_entry(xi / d.t, i);
    });
    __syncthreads();
    const int n = sh.listed;
    if (n > kList || n == 0) return false;
    if (by_k) sort_list(n, sh);
    const int kk = by_k ? min(p.top_k, n) : n;  // the top-k set: list[0, kk)
    // Each thread's two entries, their weights, and the mass before them.
    const int i0 = 2 * tid, i1 = 2 * tid + 1;
    const float v0 = i0 < kk ? entry_value(sh.list[i0]) : 0.0f, v1 = i1 < kk ? entry_value(sh.list[i1]) : 0.0f;
    const unsigned long long w0 = i0 < kk ? fixed_weight(v0, d.mx) : 0, w1 = i1 < kk ? fixed_weight(v1, d.mx) : 0;
    unsigned long long zk;
    const unsigned long long before = block_scan_u64(w0 + w1, sh, zk);
    int keep = kk;  // the top-p set: list[0, keep)
    if (p.top_p < 1.0f) {
        const unsigned long long target = top_p_target(p.top_p, zk);
        __syncthreads();
        if (before < target && before + w0 + w1 >= target)  // one thread
            sh.prefix = static_cast<uint32_t>(before + w0 >= target ? i0 + 1 : i1 + 1);
        __syncthreads();
        keep = static_cast<int>(sh.prefix);
    }
    if (by_k) {
        d.k.theta = entry_value(sh.list[kk - 1]);
        d.k.id_cut = entry_id(sh.list[kk - 1]);
    }
    if (p.top_p < 1.0f) {
        d.p.theta = entry_value(sh.list[keep - 1]);
        d.p.id_cut = entry_id(sh.list[keep - 1]);
    }
    d.listed = keep;
    d.z = block_sum_u64((i0 < keep && expf(v0 - d.mx) >= d.min_w ? w0 : 0) + (i1 < keep && expf(v1 - d.mx) >= d.min_w ? w1 : 0), sh);
    return true;
}

// The kept set of one row, in the host sampler's order; its mass if `mass`.
__device__ __forceinline__ Dist distribution(const float *x, int V, const EmberSampleParams &p, bool mass, SampleLds &sh) {
    Dist d{};
    d.greedy = !(p.temperature > 1e-5f);
    if (d.greedy) return d;
    d.t = p.temperature;
    float m = -INFINITY;
    for_row(x, V, [&](int, float xi) { m = fmaxf(m, xi); });
    d.mx = block_max(m, sh) / d.t;  // the largest quotient: division by t > 0 keeps the order
    d.certain = !(fabsf(d.mx) < INFINITY);
    if (d.certain) return d;
    d.min_w = p.min_p > 0.0f ? p.min_p : 0.0f;
    const Cut all;
    d.k = all;
    d.p = all;
    const bool cuts = (p.top_k > 0 && p.top_k < V) || p.top_p < 1.0f;
    // (ln(min_w) and the quotient's rounding, with room: the comparison that decides is on the weight)
    d.least = d.min_w > 0.0f ? (d.mx + logf(d.min_w) - 0.01f - fabsf(d.mx) * 0x1p-20f) * d.t : -INFINITY;
    if (mass && !cuts) {
        // No order to find: one pass, its weights through double (the same integers as fixed_weight's, in fewer
        // instructions where nothing else is done). token_probs of 16 rows of 151,936: 51 us, by the general pass below
        // 66; with min-p 0.02, 51 at most, collecting and sorting the candidates first 88 (4 rows of 8192: 8.4, 24.5).
        unsigned long long s = 0;
        for_row(x, V, [&](int, float xi) {
            if (!(xi >= d.least)) return;
            const float w = expf(xi / d.t - d.mx);
            if (w >= d.min_w) s += static_cast<unsigned long long>(static_cast<double>(w) * kFix);
        });
        d.z = block_sum_u64(s, sh);
        return d;
    }
    if (d.t < 1e5f && few_candidates(x, V, p, m, cuts, d, sh)) return d;
    unsigned long long kept = 0;  // weight of the set so far
    bool known = false;           // and it is the kept set's mass
#pragma unroll 1
    for (int which = 0; which < 2; which++) {
        if (which == 0 ? !(p.top_k > 0 && p.top_k < V) : !(p.top_p < 1.0f)) continue;
        const Cut c = prefix_cut(x, V, d.t, which == 0 ? all : d.k, d.mx, p.top_k, which == 0 ? -1.0f : fmaxf(p.top_p, 0.0f),
                                 kept, sh);
        if (which == 0) {
            d.k = c;
        } else {
            d.p = c;
            known = d.min_w == 0.0f;
        }
    }
    if (known || !mass) {
        d.z = kept;
        return d;
    }
    // the kept set's mass (min-p applied), for token probabilities
    unsigned long long s = 0;
    for_row(x, V, [&](int i, float xi) {
        const float v = xi / d.t;
        if (d.keeps(v, i)) s += fixed_weight(v, d.mx);
    });
    d.z = block_sum_u64(s, sh);
    return d;
}

__global__ void __launch_bounds__(kSampleThreads) sample_kernel(const float *__restrict__ logits, int V,
                                                                const EmberSampleParams *__restrict__ params,
                                                                int32_t *__restrict__ out) {
    __shared__ SampleLds sh;
    const int r = static_cast<int>(blockIdx.x);
    const float *x = logits + static_cast<int64_t>(r) * V;
    const EmberSampleParams p = params[r];
    const Dist d = distribution(x, V, p, false, sh);
    int tok;
    if (d.greedy) {
        tok = block_argmax(x, V, [](int, float xi) { return xi; }, sh);
    } else if (d.certain) {
        tok = block_argmax<kRareBatch>(x, V, [&](int, float xi) { return xi / d.t; }, sh);
    } else if (d.listed) {
        float best = -INFINITY;
        int idx = 0x7fffffff;
        for (int j = static_cast<int>(threadIdx.x); j < d.listed; j += kSampleThreads) {
            const float v = entry_value(sh.list[j]);
            const int i = entry_id(sh.list[j]);
            const float s = expf(v - d.mx) >= d.min_w ? v + gumbel_noise(p.seed, p.counter, static_cast<uint32_t>(i)) : -INFINITY;
            if (s > best || (s == best && s > -INFINITY && i < idx)) {
                best = s;
                idx = i;
            }
        }
        tok = block_first_largest(best, idx, sh);
    } else {
        tok = block_argmax(x, V, [&](int i, float xi) {
            const float v = xi / d.t;
            return d.keeps(v, i) ? v + gumbel_noise(p.seed, p.counter, static_cast<uint32_t>(i)) : -INFINITY;
        }, sh);
    }
    if (threadIdx.x == 0) out[r] = tok;
}

__global__ void __launch_bounds__(kSampleThreads) prob_kernel(const float *__restrict__ logits, int V, int R,
                                                              const EmberSampleParams *__restrict__ params,
                                                              const int32_t *__restrict__ rows,
                                                              const int32_t *__restrict__ tokens,
                                                              float *__restrict__ out) {
    __shared__ SampleLds sh;
    const int q = static_cast<int>(blockIdx.x), r = rows[q], tok = tokens[q];
    if (r < 0 || r >= R || tok < 0 || tok >= V) {  // uniform per work-group
        if (threadIdx.x == 0) out[q] = 0.0f;
        return;
    }
    const float *x = logits + static_cast<int64_t>(r) * V;
    const EmberSampleParams p = params[r];
    const Dist d = distribution(x, V, p, true, sh);
    float prob;
    if (d.greedy) {
        prob = block_argmax(x, V, [](int, float xi) { return xi; }, sh) == tok ? 1.0f : 0.0f;
    } else if (d.certain) {  // 0 for every token of a row with nothing above -inf
        prob = block_argmax<kRareBatch>(x, V, [&](int, float xi) { return xi / d.t; }, sh) == tok && d.mx > 0.0f ? 1.0f : 0.0f;
    } else {
        const float v = scaled(x, tok, d.t);
        const float w = expf(v - d.mx);
        prob = d.keeps(v, tok) && d.z ? static_cast<float>(static_cast<double>(w) * kFix / static_cast<double>(d.z)) : 0.0f;
    }
    if (threadIdx.x == 0) out[q] = prob;
}

constexpr int kEmbedThreads = 256;

// out[t] = the f16 embedding row of tokens[t], as f32 (k_elementwise.cu's embed_tokens).
__global__ void __launch_bounds__(kEmbedThreads) embed_kernel(const int32_t *__restrict__ tokens, int vocab,
                                                              const f16 *__restrict__ table, int hidden,
                                                              float *__restrict__ out) {
    const int t = static_cast<int>(blockIdx.x);
    const int tok = tokens[t];
    float *o = out + static_cast<int64_t>(t) * hidden;
    if (tok < 0 || tok >= vocab) {  // an id outside the table embeds as zeros (checked on the host)
        for (int i = static_cast<int>(threadIdx.x); i < hidden; i += kEmbedThreads) o[i] = 0.0f;
        return;
    }
    const f16 *row = table + static_cast<int64_t>(tok) * hidden;
    for (int i = 8 * static_cast<int>(threadIdx.x); i < hidden; i += 8 * kEmbedThreads) {
        const f16x8 v = *reinterpret_cast<const f16x8 *>(row + i);
#pragma unroll
        for (int j = 0; j < 8; j++) o[i + j] = static_cast<float>(v[j]);
    }
}

}  // namespace

hipError_t launch_sample(const EmberSampleArgs &a, hipStream_t stream) {
    hipLaunchKernelGGL(sample_kernel, dim3(static_cast<unsigned>(a.R)), dim3(kSampleThreads), 0, stream, a.logits,
                       a.vocab, a.params, a.out);
    return hipGetLastError();
}

hipError_t launch_token_probs(const EmberProbArgs &a, hipStream_t stream) {
    hipLaunchKernelGGL(prob_kernel, dim3(static_cast<unsigned>(a.n)), dim3(kSampleThreads), 0, stream, a.logits,
                       a.vocab, a.R, a.params, a.rows, a.tokens, a.out);
    return hipGetLastError();
}

hipError_t launch_embed(const EmberEmbedArgs &a, hipStream_t stream) {
    hipLaunchKernelGGL(embed_kernel, dim3(static_cast<unsigned>(a.T)), dim3(kEmbedThreads), 0, stream, a.tokens,
                       a.vocab, static_cast<const f16 *>(a.table), a.hidden, a.out);
    return hipGetLastError();
}

}  // namespace ember::hip
