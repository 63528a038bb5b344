// Token sampling on the device: temperature softmax, nucleus (top-p) filtering and the
// categorical draw of AutoregressiveModel.sampleToken (engine/ml/.../AutoregressiveModel.java:323-386),
// and the sample function AutoregressiveModel.of installs (:413-425: logits / temperature, the
// DistributionFeatures.softmax of compute/stats/.../DistributionFeatures.java:129-141, then
// sampleToken(probabilities, V, 1.0, 1.0, random)), with java.util.Random's generator
// (48-bit LCG, nextDouble = ((next(26) << 27) + next(27)) * 2^-53) kept per sequence on the device.
//
// Everything after the fp32 logits is double, the reference's precision.  A row of V values is cut
// into kBlocks chunks; each pass is one grid of (kBlocks, rows) 1024-thread blocks whose per-block
// maxima / sums go to the workspace and are combined by the next kernel in a fixed order (a
// wavefront butterfly over the 64 chunk values), so every result is deterministic.
//
// Nucleus filtering does not sort.  The reference keeps the shortest prefix of the probabilities
// sorted in descending order (ties in index order: Arrays.sort is stable) whose running sum
// reaches top_p.  With p* the smallest kept value, that is every value > p* plus the first c
// (by index) of the values == p*; p* is the largest key t with sum(p >= t) >= top_p.  It is found
// on the 64-bit patterns of the probabilities (non-negative doubles order as their bit patterns):
//  * one pass over the row adds the values into 1,024 buckets of equal width in the bit pattern between the
//    row's least and largest value, or by exponent and the first four mantissa bits where they lie further
//    apart than that covers (64 octaves below 1; what lies lower is below the fixed point's unit and never
//    holds p*), LDS per chunk, then the row's buckets with device-scope atomics; the last chunk to finish
//    (an arrival counter) picks the bucket whose range holds p* and clears the row's buckets for the next
//    draw;
//  * one pass copies that bucket's values, in index order, and sums what lies above it per chunk;
//  * the block that draws finishes the search on the copied values alone (a radix descent over the bucket's
//    bits, at most 48 and 8 at a time, ending early once one value is left).
// 8 x 151,936 values: 56 us a draw, against 124 with eight 8-bit passes over the whole row, whose first
// digits separate next to nothing.  Buckets by exponent and mantissa alone put a whole row of equal or
// nearly equal logits into one bucket, for the drawing block to go over digit by digit: one row of 151,936
// equal logits took 1,662 us (deviation 0.001: 256; rounded to whole numbers: 468), 33, 40 and 62 now, and 97,
// 76 and 77 with the eight passes.  Bucket sums are 2^-60 fixed point in u64, so the atomics are exact and
// associative (the result does not depend on arrival order); the kept set agrees with the reference's
// sequential double sums except when top_p lies within ~1e-13 of a partial sum.
//
// The draw mirrors the reference's loop `cumulative += probs[i]; if (r < cumulative) return i`:
// chunk masses locate the chunk whose interval holds r, then per-thread sums of contiguous index
// ranges and a walk of the crossing thread's elements locate the index.  Partial sums group
// differently from the reference's single running sum (rounding ~1e-16), so a draw within that
// distance of a boundary may pick the neighbour.
#include "ar_hip_internal.h"

namespace {

constexpr int kBlocks = 64;   // chunks per row (one wavefront of partials)
constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kBins = 1024;   // buckets of the nucleus search (one per thread of the block that picks)
constexpr int kCandLds = 4096;  // bucket values the drawing block holds in LDS
constexpr double kFix = 1152921504606846976.0;     // 2^60
constexpr double kEps64 = 2.220446049250313e-16;   // FP64 machine epsilon (Precision.java:110-121)

struct Ws {
    double* buf;                // [rows][V] exp values; probabilities once the nucleus search began
    double* pmax;               // [rows][kBlocks]
    double* psum;
    double* pemax;
    double* pemin;
    double* psum2;
    double* pmass;
    unsigned long long* gsum;   // [rows][kBins] fixed-point bucket sums of the row (zero between draws)
    unsigned* arrived;          // [rows] chunks done with the bucket pass (zero between draws)
    unsigned long long* sel;    // [rows][4]: the bucket of p*: least key (or -1: everything is kept), fixed-
                                // point sum above it, bits of its width
    unsigned long long* cand;   // [rows][V] bit patterns of the bucket's values, each chunk's at its own start
    unsigned* ncand;            // [rows][kBlocks]
};

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// The zero-initialised part (gsum, arrived) comes first so that it can be cleared once.
Ws carve(void* base, int rows, int V, size_t* total, size_t* zero_bytes) {
    Ws w{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const uintptr_t p = reinterpret_cast<uintptr_t>(base) + off;
        off += align256(bytes);
        return reinterpret_cast<void*>(p);
    };
    w.gsum = (unsigned long long*)take((size_t)rows * kBins * 8);
    w.arrived = (unsigned*)take((size_t)rows * 4);
    if (zero_bytes) *zero_bytes = off;
    w.buf = (double*)take((size_t)rows * V * 8);
    w.pmax = (double*)take((size_t)rows * kBlocks * 8);
    w.psum = (double*)take((size_t)rows * kBlocks * 8);
    w.pemax = (double*)take((size_t)rows * kBlocks * 8);
    w.pemin = (double*)take((size_t)rows * kBlocks * 8);
    w.psum2 = (double*)take((size_t)rows * kBlocks * 8);
    w.pmass = (double*)take((size_t)rows * kBlocks * 8);
    w.sel = (unsigned long long*)take((size_t)rows * 4 * 8);
    w.cand = (unsigned long long*)take((size_t)rows * V * 8);
    w.ncand = (unsigned*)take((size_t)rows * kBlocks * 4);
    if (total) *total = off;
    return w;
}

struct Args {
    const float* logits;
    int ls, V, mode;
    double T;
    bool topp;
    unsigned long long target;  // top_p in 2^-60 fixed point, rounded up
    Ws w;
    unsigned long long* rng;
    const int* state;
    unsigned long long* keys;
    int keys_stride;
    int* out;
};

__device__ inline double wave_max_d(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline double wave_sum_d(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// inclusive prefix over the lanes of a wavefront (Hillis-Steele; a fixed order of additions)
template <typename T>
__device__ inline T wave_incl_scan(T v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}
// block reductions: butterfly per wavefront, then the wavefront values in order
__device__ inline double block_max_d(double v, double* red) {
    v = wave_max_d(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = red[0];
    for (int w = 1; w < kWaves; w++) r = fmax(r, red[w]);
    __syncthreads();
    return r;
}
__device__ inline double block_sum_d(double v, double* red) {
    v = wave_sum_d(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = red[0];
    for (int w = 1; w < kWaves; w++) r += red[w];
    __syncthreads();
    return r;
}
// inclusive prefix over the block's threads in thread order (wavefront scans + the wavefront
// totals in order)
template <typename T>
__device__ inline T block_incl_scan(T v, T* red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    v = wave_incl_scan(v);
    if (lane == 63) red[w] = v;
    __syncthreads();
    T base = 0;
    for (int k = 0; k < w; k++) base += red[k];
    __syncthreads();
    return base + v;
}
// combine one row's 64 chunk partials (every thread gets the value; same order in every block)
__device__ inline double row_max(const double* p) { return wave_max_d(p[threadIdx.x & 63]); }
__device__ inline double row_max_neg(const double* p) { return wave_max_d(-p[threadIdx.x & 63]); }
__device__ inline double row_sum(const double* p) { return wave_sum_d(p[threadIdx.x & 63]); }

__device__ inline void chunk_of(int V, int blk, int* c0, int* c1) {
    const int per = (V + kBlocks - 1) / kBlocks;
    *c0 = min(V, blk * per);
    *c1 = min(V, *c0 + per);
}

__device__ inline double scaled(const Args& a, int b, int i) { return (double)a.logits[(size_t)b * a.ls + i] / a.T; }

// 1. maximum of logits / temperature per chunk
__global__ __launch_bounds__(kThreads) void smp_max_kernel(Args a) {
    __shared__ double red[kWaves];
    const int blk = blockIdx.x, b = blockIdx.y;
    int c0, c1;
    chunk_of(a.V, blk, &c0, &c1);
    double m = -INFINITY;
    for (int i = c0 + threadIdx.x; i < c1; i += kThreads) m = fmax(m, scaled(a, b, i));
    m = block_max_d(m, red);
    if (threadIdx.x == 0) a.w.pmax[b * kBlocks + blk] = m;
}

// 2. exponentials: sampleToken's exp(x - max), or the softmax-ignoring-zero of the model's sample
//    function (a value equal to 0 stays 0; the maximum itself gets exp(epsilon))
__global__ __launch_bounds__(kThreads) void smp_exp_kernel(Args a) {
    __shared__ double red[3 * kWaves];
    const int blk = blockIdx.x, b = blockIdx.y;
    int c0, c1;
    chunk_of(a.V, blk, &c0, &c1);
    const double M = row_max(a.w.pmax + b * kBlocks);
    double s = 0.0, emax = 0.0, emin = INFINITY;
    double* buf = a.w.buf + (size_t)b * a.V;
    for (int i = c0 + threadIdx.x; i < c1; i += kThreads) {
        const double y = scaled(a, b, i);
        double e;
        if (a.mode == AR_SAMPLE_TOKEN) {
            e = exp(y - M);
        } else {
            const double d = (y == 0.0) ? 0.0 : ((y == M) ? kEps64 : y - M);
            e = (d == 0.0) ? 0.0 : exp(d);
        }
        buf[i] = e;
        s += e;
        emax = fmax(emax, e);
        emin = fmin(emin, e);
    }
    // the three block reductions under one barrier, for thread 0 alone
    s = wave_sum_d(s);
    emax = wave_max_d(emax);
    emin = -wave_max_d(-emin);
    if ((threadIdx.x & 63) == 0) {
        const int w = threadIdx.x >> 6;
        red[w] = s;
        red[kWaves + w] = emax;
        red[2 * kWaves + w] = emin;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kWaves; w++) {
            s += red[w];
            emax = fmax(emax, red[kWaves + w]);
            emin = fmin(emin, red[2 * kWaves + w]);
        }
        a.w.pemin[b * kBlocks + blk] = emin;
        a.w.psum[b * kBlocks + blk] = s;
        a.w.pemax[b * kBlocks + blk] = emax;
    }
}

// 3. (model sample function) sampleToken's own softmax of the probabilities p = e / S1 at
//    temperature 1: f = exp(p - max p); max p = fl(max e / S1), division being monotone
__global__ __launch_bounds__(kThreads) void smp_exp2_kernel(Args a) {
    __shared__ double red[kWaves];
    const int blk = blockIdx.x, b = blockIdx.y;
    int c0, c1;
    chunk_of(a.V, blk, &c0, &c1);
    const double S1 = row_sum(a.w.psum + b * kBlocks);
    const double m2 = row_max(a.w.pemax + b * kBlocks) / S1;
    double* buf = a.w.buf + (size_t)b * a.V;
    double s = 0.0;
    for (int i = c0 + threadIdx.x; i < c1; i += kThreads) {
        const double f = exp(buf[i] / S1 - m2);
        buf[i] = f;
        s += f;
    }
    s = block_sum_d(s, red);
    if (threadIdx.x == 0) a.w.psum2[b * kBlocks + blk] = s;
}

__device__ inline double denom(const Args& a, int b) {
    return row_sum((a.mode == AR_SAMPLE_TOKEN ? a.w.psum : a.w.psum2) + b * kBlocks);
}

// Buckets of a row's probabilities: (key - base) >> bits, keys under base in the first.
struct Buckets {
    unsigned long long base;
    int bits;
    __device__ int of(unsigned long long key) const {
        return key <= base ? 0 : (int)min((key - base) >> bits, (unsigned long long)(kBins - 1));
    }
};

// Width 2^bits and first key, from the row's least and largest probability (e / D is monotone in e).
__device__ inline Buckets buckets_of(const Args& a, int b, double D) {
    const double* const pe = a.w.pemin + b * kBlocks;
    const unsigned long long lo = (unsigned long long)__double_as_longlong(-row_max_neg(pe) / D),
                             hi = (unsigned long long)__double_as_longlong(row_max(a.w.pemax + b * kBlocks) / D);
    const int bits = hi > lo ? max(0, 54 - __clzll((long long)(hi - lo))) : 0;
    if (bits > 48) return Buckets{(unsigned long long)(0x3FF0 - (kBins - 1)) << 48, 48};  // (1.0 in the last)
    return Buckets{lo, bits};
}

// 4. nucleus search, the whole row: probabilities (written back over the exponentials) into the buckets;
//    the last chunk to arrive picks the highest bucket d with sum(buckets >= d) >= target
__global__ __launch_bounds__(kThreads) void smp_bucket_kernel(Args a) {
    __shared__ unsigned long long sm[kBins], red[kWaves];
    __shared__ int last_s;
    static_assert(kBins == kThreads, "one bucket per thread");
    const int blk = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
    sm[t] = 0;
    __syncthreads();
    int c0, c1;
    chunk_of(a.V, blk, &c0, &c1);
    const double D = denom(a, b);
    const Buckets bk = buckets_of(a, b, D);
    double* buf = a.w.buf + (size_t)b * a.V;
    for (int i = c0 + t; i < c1; i += kThreads) {
        const double p = buf[i] / D;
        buf[i] = p;
        const unsigned long long f = (unsigned long long)(p * kFix);
        if (f) atomicAdd(&sm[bk.of((unsigned long long)__double_as_longlong(p))], f);
    }
    __syncthreads();
    unsigned long long* g = a.w.gsum + (size_t)b * kBins + t;
    if (sm[t]) __hip_atomic_fetch_add(g, sm[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // this thread's atomics have completed
    __syncthreads();
    if (t == 0) {
        unsigned* c = a.w.arrived + b;
        const unsigned prev = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = prev == (unsigned)(kBlocks - 1);
        if (last) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_s = last;
    }
    __syncthreads();
    if (!last_s) return;
    // thread t takes bucket kBins - 1 - t: an inclusive scan in thread order sums the buckets from the top
    g = a.w.gsum + (size_t)b * kBins + (kBins - 1 - t);
    const unsigned long long mine = __hip_atomic_load(g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(g, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long incl = block_incl_scan(mine, red);
    unsigned long long* sel = a.w.sel + b * 4;
    // the whole row may sum to less than top_p (the reference then keeps every value): no bucket
    if (t == kThreads - 1 && (incl < a.target || incl == 0)) sel[0] = ~0ull;
    const unsigned long long before = incl - mine;
    if (mine && incl >= a.target && (before < a.target || before == 0)) {
        sel[0] = bk.base + ((unsigned long long)(kBins - 1 - t) << bk.bits);
        sel[1] = before;
        sel[2] = bk.bits;
    }
}

// 5. nucleus search, the bucket of p*: its values' bit patterns in index order, and the mass above it
__global__ __launch_bounds__(kThreads) void smp_cand_kernel(Args a) {
    __shared__ double red[kWaves];
    __shared__ int wcnt[kWaves];
    const int blk = blockIdx.x, b = blockIdx.y, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int c0, c1;
    chunk_of(a.V, blk, &c0, &c1);
    const unsigned long long base = a.w.sel[b * 4];
    const bool cut = base != ~0ull;
    const int bits = cut ? (int)a.w.sel[b * 4 + 2] : 0;
    const double* buf = a.w.buf + (size_t)b * a.V;
    unsigned long long* cand = a.w.cand + (size_t)b * a.V + c0;
    double s = 0.0;
    int n = 0;  // values copied so far (the same in every thread)
    for (int i0 = c0; i0 < c1; i0 += kThreads) {
        const int i = i0 + t;
        const double p = i < c1 ? buf[i] : 0.0;
        const unsigned long long key = (unsigned long long)__double_as_longlong(p);
        const bool in = i < c1 && cut && key >= base && (key - base) >> bits == 0;
        if (i < c1 && (!cut || (key >= base && !in))) s += p;  // (no cut: everything lies above)
        const unsigned long long hits = __ballot(in);
        if (lane == 0) wcnt[wave] = __popcll(hits);
        __syncthreads();
        int at = n;
        for (int w = 0; w < kWaves; w++) {
            if (w < wave) at += wcnt[w];
            n += wcnt[w];
        }
        if (in) cand[at + __popcll(hits & ((1ull << lane) - 1))] = key;
        __syncthreads();
    }
    s = block_sum_d(s, red);
    if (t == 0) {
        a.w.pmass[b * kBlocks + blk] = s;
        a.w.ncand[b * kBlocks + blk] = (unsigned)n;
    }
}

__device__ inline void thread_range(int c0, int c1, int* r0, int* r1) {
    const int per = (c1 - c0 + kThreads - 1) / kThreads;
    *r0 = min(c1, c0 + (int)threadIdx.x * per);
    *r1 = min(c1, *r0 + per);
}

// 5'. (no nucleus) probability mass per chunk
__global__ __launch_bounds__(kThreads) void smp_mass_kernel(Args a) {
    __shared__ double red[kWaves];
    const int blk = blockIdx.x, b = blockIdx.y;
    int c0, c1, r0, r1;
    chunk_of(a.V, blk, &c0, &c1);
    thread_range(c0, c1, &r0, &r1);
    const double D = denom(a, b);
    const double* buf = a.w.buf + (size_t)b * a.V;
    double s = 0.0;
    for (int i = r0; i < r1; i++) s += buf[i] / D;
    s = block_sum_d(s, red);
    if (threadIdx.x == 0) a.w.pmass[b * kBlocks + blk] = s;
}

// The nucleus: values > p*, and the first `take` (by index) of the values == p*.
struct Nucleus {
    bool cut;  // false: every value is kept
    unsigned long long pstar, take;
};

__device__ inline double kept(const Nucleus& n, double q, unsigned long long* rank) {
    if (!n.cut) return q;
    const unsigned long long key = (unsigned long long)__double_as_longlong(q);
    if (key > n.pstar) return q;
    if (key == n.pstar) return (*rank)++ < n.take ? q : 0.0;
    return 0.0;
}

// LDS of the drawing block's end of the nucleus search
struct SearchLds {
    union {
        unsigned long long key[kCandLds];  // the bucket's values (when they fit), in index order
        struct {                           // ranges of a bucket that does not fit
            unsigned long long sum[kBins], lo[kBins], hi[kBins];
            unsigned cnt[kBins];
        } range;
    };
    unsigned long long sum[256];
    unsigned cnt[256];
    unsigned off[kBlocks + 1];         // first value of each chunk in that order
    unsigned long long ties[kBlocks];  // values == p* in the chunks before each chunk
    double mass[kBlocks];              // kept mass of each chunk
    unsigned long long prefix, above, pstar, take;  // prefix: p* - the bucket's least key, as far as known
    unsigned long long lo, hi;
    unsigned left;
    int pick;
};

// A bucket of more than kCandLds values, L.lo .. L.hi and not all equal (many equal values among others): cut
// down to the values that may be p*, its surroundings added to the chunks' mass.  Each round spreads the keys
// over 1,024 ranges of equal width and goes on with the span (least to largest key) of the one that holds p*,
// until its values are equal or fit L.key.  A thread adds up its run of values of one range before it touches
// LDS: atomics of a wavefront on one address go one after another.  Then one pass sums the keys above per
// chunk and moves the rest to the front of the chunk's copies (equal values: counts them).  L.ties: what
// is left of each chunk.  Bound by one CU's read of the copies: some 30 us a pass over 151,936 values.
__device__ void thin_bucket(const Args& a, int b, SearchLds& L, unsigned long long* red) {
    constexpr int U = 8;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    unsigned long long* const cand = a.w.cand + (size_t)b * a.V;
    // every value of this wavefront's chunks, in index order, in groups of 64 (0 past the end: below every
    // key), eight of them loaded together
    auto each = [&](auto&& group, auto&& chunk_end) {
        for (int c = wave; c < kBlocks; c += kWaves) {
            int c0, c1;
            chunk_of(a.V, c, &c0, &c1);
            const unsigned m = L.off[c + 1] - L.off[c];
            for (unsigned i0 = 0; i0 < m; i0 += 64 * U) {
                unsigned long long k[U];
#pragma unroll
                for (int u = 0; u < U; u++) k[u] = cand[c0 + min(i0 + 64 * u + lane, m - 1)];
#pragma unroll
                for (int u = 0; u < U; u++) group(c0, i0 + 64 * u + lane < m ? k[u] : 0ull);
            }
            chunk_end(c);
        }
    };
    unsigned long long lo = L.lo, hi = L.hi;
    for (int round = 0; round < 5; round++) {  // (48 bits, ten with every round)
        const int sh = max(0, 54 - __clzll((long long)(hi - lo)));
        __syncthreads();
        L.range.sum[t] = 0;
        L.range.lo[t] = ~0ull;
        L.range.hi[t] = 0;
        L.range.cnt[t] = 0;
        if (t == 0) L.pick = kBins;
        __syncthreads();
        int run = -1;
        unsigned n = 0;
        unsigned long long s = 0, mn = ~0ull, mx = 0;
        auto flush = [&]() {
            if (run < 0) return;
            atomicAdd(&L.range.cnt[run], n);
            atomicAdd(&L.range.sum[run], s);
            atomicMin(&L.range.lo[run], mn);
            atomicMax(&L.range.hi[run], mx);
        };
        each([&](int, unsigned long long key) {
            if (key < lo || key > hi) return;
            const int d = (int)((key - lo) >> sh);
            if (d != run) {
                flush();
                run = d;
                n = 0;
                s = 0;
                mn = ~0ull;
                mx = 0;
            }
            n++;
            s += (unsigned long long)(__longlong_as_double((long long)key) * kFix);
            mn = min(mn, key);
            mx = max(mx, key);
        }, [](int) {});
        flush();
        __syncthreads();
        const int d = kBins - 1 - t;  // an inclusive scan in thread order sums the ranges from the top
        const unsigned long long mine = L.range.sum[d], incl = block_incl_scan(mine, red);
        if (L.range.cnt[d] && L.above + incl >= a.target) atomicMin(&L.pick, t);
        __syncthreads();
        if (t == L.pick) {  // (the bucket holds p*: one does)
            L.lo = L.range.lo[d];
            L.hi = L.range.hi[d];
            L.left = L.range.cnt[d];
            L.above += incl - mine;
        }
        __syncthreads();
        lo = L.lo;
        hi = L.hi;
        if (lo >= hi || L.left <= (unsigned)kCandLds) break;
    }
    const bool equal = L.left > (unsigned)kCandLds;
    double s = 0.0;
    unsigned n = 0;
    each([&](int c0, unsigned long long key) {
        if (key > hi) s += __longlong_as_double((long long)key);
        const bool in = key >= lo && key <= hi;
        const unsigned long long hits = __ballot(in);
        // (at or before the place it was read from, and behind what is still to be read)
        if (!equal && in) cand[c0 + n + __popcll(hits & ((1ull << lane) - 1))] = key;
        n += __popcll(hits);
    }, [&](int c) {
        const double total = wave_sum_d(s);
        if (lane == 0) {
            L.mass[c] += total;
            L.ties[c] = n;
        }
        s = 0.0;
        n = 0;
    });
    __syncthreads();
    if (!equal && t < kBlocks) L.off[t + 1] = (unsigned)wave_incl_scan(L.ties[t]);
    __syncthreads();
}

// p*, the ties kept, and the kept mass of every chunk (L.mass), by the whole block.
__device__ Nucleus finish_search(const Args& a, int b, SearchLds& L, unsigned long long* red) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    unsigned long long base = a.w.sel[b * 4];
    if (t < kBlocks) L.mass[t] = a.w.pmass[b * kBlocks + t];
    if (base == ~0ull) {
        __syncthreads();
        return Nucleus{false, 0, 0};
    }
    int bits = (int)a.w.sel[b * 4 + 2];  // keys base .. base + 2^bits - 1
    if (t < kBlocks) {
        const unsigned c = a.w.ncand[b * kBlocks + t], incl = wave_incl_scan(c);
        L.off[t + 1] = incl;
        L.ties[t] = c;
        if (t == 0) L.off[0] = 0;
        if (t == kBlocks - 1) L.left = incl;
    }
    if (t == 0) {
        L.prefix = 0;
        L.above = a.w.sel[b * 4 + 1];
        L.lo = base;
        L.hi = base + ((1ull << bits) - 1);
    }
    __syncthreads();
    // values == p* kept, of the L.left there are
    auto set_take = [&]() {
        const unsigned long long pf = (unsigned long long)(__longlong_as_double((long long)L.pstar) * kFix);
        unsigned long long take = 1;
        if (a.target > L.above) take = pf ? (a.target - L.above + pf - 1) / pf : L.left;
        L.take = take < 1 ? 1 : (take > L.left ? L.left : take);
    };
    if (bits && L.left > (unsigned)kCandLds) thin_bucket(a, b, L, red);
    base = L.lo;
    bits = 64 - (L.hi > base ? __clzll((long long)(L.hi - base)) : 64);
    if (L.left > (unsigned)kCandLds) {
        // equal values: the first `take` by index, chunk by chunk
        if (t == 0) {
            L.pstar = base;
            set_take();
        }
        __syncthreads();
        const Nucleus nu{true, L.pstar, L.take};
        if (t < kBlocks) {
            const unsigned long long v = L.ties[t], before = wave_incl_scan(v) - v;
            const unsigned long long k = nu.take > before ? min(nu.take - before, v) : 0ull;
            L.ties[t] = before;
            L.mass[t] += (double)k * __longlong_as_double((long long)nu.pstar);
        }
        __syncthreads();
        return nu;
    }
    // chunk by chunk, a wavefront each: f(chunk, key, live) for every copied value
    auto each = [&](auto&& f) {
        for (int c = wave; c < kBlocks; c += kWaves) {
            const unsigned o = L.off[c], m = L.off[c + 1] - o;
            for (unsigned i0 = 0; i0 < m; i0 += 64) {
                const bool live = i0 + lane < m;
                f(c, live ? L.key[o + i0 + lane] : 0ull, live);
            }
        }
    };
    {  // 16 lanes a chunk: usually one load each
        int c0, c1;
        const int c = t / (kThreads / kBlocks);
        chunk_of(a.V, c, &c0, &c1);
        const unsigned o = L.off[c], m = L.off[c + 1] - o;
        for (unsigned i = t % (kThreads / kBlocks); i < m; i += kThreads / kBlocks)
            L.key[o + i] = a.w.cand[(size_t)b * a.V + c0 + i];
    }
    // radix descent over key - base: the highest digit d with above + sum(digits >= d) >= target at each level
    for (int left = bits;;) {  // bits that are still open
        if (left == 0 || L.left == 1) {
            // every value left has the prefix's bits: one value, or equal ones
            __syncthreads();
            const unsigned long long pre = L.prefix >> left;
            each([&](int, unsigned long long key, bool live) {
                if (live && (key - base) >> left == pre) L.pstar = key;
            });
            break;
        }
        const int width = min(left, 8), shift = left - width;
        if (t < 256) {
            L.cnt[t] = 0;
            L.sum[t] = 0;
        }
        __syncthreads();
        const unsigned long long want = L.prefix >> left, above = L.above;
        each([&](int, unsigned long long key, bool live) {
            if (live && (key - base) >> left == want) {
                const int d = (int)(((key - base) >> shift) & ((1u << width) - 1));
                atomicAdd(&L.cnt[d], 1u);
                atomicAdd(&L.sum[d], (unsigned long long)(__longlong_as_double((long long)key) * kFix));
            }
        });
        __syncthreads();
        if (t < 64) {
            unsigned long long lsum = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) lsum += L.sum[255 - 4 * lane - k];
            unsigned long long acc = above + wave_incl_scan(lsum) - lsum;  // the digits above this lane's four
            int hit = -1;
            unsigned long long acc_hit = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int d = 255 - 4 * lane - k;
                if (hit < 0 && L.cnt[d] && acc + L.sum[d] >= a.target) {
                    hit = d;
                    acc_hit = acc;
                }
                acc += L.sum[d];
            }
            const unsigned long long hits = __ballot(hit >= 0);  // (the bucket holds p*: never empty)
            if (hits && lane == __builtin_ctzll(hits)) {
                L.prefix |= (unsigned long long)hit << shift;
                L.above = acc_hit;
                L.left = L.cnt[hit];
            }
        }
        __syncthreads();
        left = shift;
    }
    __syncthreads();
    if (t == 0) set_take();
    __syncthreads();
    const Nucleus nu{true, L.pstar, L.take};
    // ties before each chunk, then the kept mass of the bucket's values per chunk (lane sums in index
    // order, then the lanes): added to the mass above the bucket
    for (int c = wave; c < kBlocks; c += kWaves)
        if (lane == 0) L.ties[c] = 0;
    each([&](int c, unsigned long long key, bool live) {
        const unsigned long long hits = __ballot(live && key == nu.pstar);
        if (lane == 0) L.ties[c] += __popcll(hits);
    });
    __syncthreads();
    if (t < kBlocks) {
        const unsigned long long v = L.ties[t], incl = wave_incl_scan(v);
        L.ties[t] = incl - v;
    }
    __syncthreads();
    double s = 0.0;
    int cur = -1;
    unsigned long long rank = 0;
    auto flush = [&]() {
        if (cur < 0) return;
        const double total = wave_sum_d(s);
        if (lane == 0) L.mass[cur] += total;
        s = 0.0;
    };
    each([&](int c, unsigned long long key, bool live) {
        if (c != cur) {
            flush();
            cur = c;
            rank = L.ties[c];
        }
        const unsigned long long hits = __ballot(live && key == nu.pstar);
        const bool tie = live && key == nu.pstar && rank + __popcll(hits & ((1ull << lane) - 1)) < nu.take;
        if (live && (key > nu.pstar || tie)) s += __longlong_as_double((long long)key);
        rank += __popcll(hits);
    });
    flush();
    __syncthreads();
    return nu;
}

__device__ inline double java_next_double(unsigned long long* s) {
    constexpr unsigned long long mult = 0x5DEECE66DULL, add = 0xBULL, mask = (1ULL << 48) - 1;
    unsigned long long x = *s;
    x = (x * mult + add) & mask;
    const long long hi = (long long)(x >> 22);  // next(26)
    x = (x * mult + add) & mask;
    const long long lo = (long long)(x >> 21);  // next(27)
    *s = x;
    return (double)((hi << 27) + lo) * 0x1.0p-53;
}

// 6. one block per row: the end of the nucleus search, the uniform draw and the index whose cumulative
//    interval holds it
__global__ __launch_bounds__(kThreads) void smp_draw_kernel(Args a) {
    __shared__ SearchLds L;
    __shared__ unsigned long long ured[kWaves];
    __shared__ double dred[kWaves];
    __shared__ int ifirst[kWaves], ilast[kWaves];
    __shared__ double sh_r, sh_c, sh_Z;
    __shared__ int sh_blk, sh_idx;
    const int b = blockIdx.x, t = threadIdx.x, lane = t & 63;
    // The model draws only when the next step feeds a sampled token (past the prompt), as
    // AutoregressiveModel.next applies its sample function (AutoregressiveModel.java:295-308).
    if (a.state && a.state[kStateNext] < a.state[kStatePrompt]) return;
    const double D = a.topp ? 1.0 : denom(a, b);  // (the nucleus search left probabilities in buf)
    const Nucleus n = a.topp ? finish_search(a, b, L, ured) : Nucleus{false, 0, 0};
    if (t < 64) {
        // chunk masses in index order; the first chunk whose running total exceeds r
        const double pm = a.topp ? L.mass[lane] : a.w.pmass[b * kBlocks + lane];
        const double Z = a.topp ? wave_sum_d(pm) : 1.0;
        const double m = a.topp ? pm / Z : pm;
        const double incl = wave_incl_scan(m);
        const double excl = __shfl_up(incl, 1, 64);
        double r = 0.0;
        if (lane == 0) r = java_next_double(a.rng + b);
        r = __shfl(r, 0, 64);
        const unsigned long long hits = __ballot(r < incl);
        if (lane == 0) {
            sh_r = r;
            sh_Z = Z;
            sh_blk = hits ? __builtin_ctzll(hits) : -1;
            sh_idx = a.V - 1;  // the reference's result when no running sum exceeds r
        }
        if (hits && lane == __builtin_ctzll(hits)) sh_c = lane ? excl : 0.0;
    }
    __syncthreads();
    const int blk = sh_blk;
    if (blk >= 0) {
        int c0, c1, r0, r1;
        chunk_of(a.V, blk, &c0, &c1);
        thread_range(c0, c1, &r0, &r1);
        const double* buf = a.w.buf + (size_t)b * a.V;
        // values == p* before this thread's contiguous range: earlier chunks, earlier threads
        unsigned long long ties = 0;
        if (n.cut)
            for (int i = r0; i < r1; i++) ties += (unsigned long long)__double_as_longlong(buf[i]) == n.pstar;
        const unsigned long long rank0 = n.cut ? L.ties[blk] + block_incl_scan(ties, ured) - ties : 0;
        const double Z = sh_Z, r = sh_r, c = sh_c;
        double s = 0.0;
        int last = -1;
        unsigned long long rank = rank0;
        for (int i = r0; i < r1; i++) {
            double q = kept(n, buf[i] / D, &rank);
            if (a.topp) q /= Z;
            s += q;
            if (q > 0.0) last = i;
        }
        const double incl = block_incl_scan(s, dred);
        // first thread whose running total exceeds r (thread order = index order), and the last
        // positive value of the chunk: the fallback when rounding of the grouped sums leaves r
        // past the chunk's total
        const unsigned long long wh = __ballot(r < c + incl);
        int wl = last;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) wl = max(wl, __shfl_xor(wl, o, 64));
        if (lane == 0) {
            ifirst[t >> 6] = wh ? (t & ~63) + __builtin_ctzll(wh) : 0x7FFFFFFF;
            ilast[t >> 6] = wl;
        }
        __syncthreads();
        int first = 0x7FFFFFFF, lastpos = -1;
        for (int w = 0; w < kWaves; w++) {
            first = min(first, ifirst[w]);
            lastpos = max(lastpos, ilast[w]);
        }
        if (first == 0x7FFFFFFF) {
            if (t == 0) sh_idx = lastpos >= 0 ? lastpos : c1 - 1;
        } else if (t == first) {
            double cc = c + (incl - s);
            rank = rank0;
            int idx = last >= 0 ? last : r1 - 1;
            for (int i = r0; i < r1; i++) {
                double q = kept(n, buf[i] / D, &rank);
                if (a.topp) q /= Z;
                cc += q;
                if (r < cc) {
                    idx = i;
                    break;
                }
            }
            sh_idx = idx;
        }
    }
    __syncthreads();
    if (t == 0) {
        const int idx = sh_idx;
        if (a.out) a.out[b] = idx;
        if (a.keys)  // beats every value key of the greedy epilogue: the next step feeds idx
            a.keys[(size_t)b * a.keys_stride] = (0xFFFFFFFFull << 32) | (unsigned long long)(0xFFFFFFFFu - (unsigned)idx);
    }
}

}  // namespace

bool sample_is_greedy(int mode, double temperature) {
    // sampleToken: temperature <= 0 is greedy; the model's sample function: temperature == 0
    return mode == AR_SAMPLE_TOKEN ? !(temperature > 0.0) : temperature == 0.0;
}

size_t sample_workspace_bytes(int rows, int vocab) {
    size_t total = 0;
    carve(nullptr, rows, vocab, &total, nullptr);
    return total;
}

int sample_workspace_clear(void* work, int rows, int vocab, hipStream_t st) {
    size_t zero = 0;
    carve(work, rows, vocab, nullptr, &zero);
    return launch_fill_i32((int*)work, 0, zero / 4, st);  // a kernel: safe inside a captured graph
}

int launch_sample(const SampleLaunch& s, hipStream_t st) {
    AR_CHECK_ARG(s.logits && s.work && s.rng && s.rows > 0 && s.vocab > 0 && s.logits_stride >= s.vocab,
                 "sample: bad arguments");
    AR_CHECK_ARG(s.mode == AR_SAMPLE_TOKEN || s.mode == AR_SAMPLE_MODEL, "sample: unknown mode %d", s.mode);
    AR_CHECK_ARG(!sample_is_greedy(s.mode, s.temperature), "sample: temperature %g selects the greedy path",
                 s.temperature);
    Args a{};
    a.logits = s.logits;
    a.ls = s.logits_stride;
    a.V = s.vocab;
    a.mode = s.mode;
    a.T = s.temperature;
    a.topp = s.mode == AR_SAMPLE_TOKEN && s.top_p < 1.0;
    a.w = carve(s.work, s.rows, s.vocab, nullptr, nullptr);
    a.rng = s.rng;
    a.state = s.state;
    a.keys = s.keys;
    a.keys_stride = s.keys_stride;
    a.out = s.out;
    const dim3 grid(kBlocks, s.rows), block(kThreads);
    hipLaunchKernelGGL(smp_max_kernel, grid, block, 0, st, a);
    AR_LAUNCH_CHECK();
    hipLaunchKernelGGL(smp_exp_kernel, grid, block, 0, st, a);
    AR_LAUNCH_CHECK();
    if (s.mode == AR_SAMPLE_MODEL) {
        hipLaunchKernelGGL(smp_exp2_kernel, grid, block, 0, st, a);
        AR_LAUNCH_CHECK();
    }
    if (a.topp) {
        // cumulative >= top_p in 2^-60 fixed point (top_p <= 0 keeps the single largest value)
        a.target = (unsigned long long)(s.top_p > 0.0 ? ceil(s.top_p * kFix) : 0.0);
        hipLaunchKernelGGL(smp_bucket_kernel, grid, block, 0, st, a);
        AR_LAUNCH_CHECK();
        hipLaunchKernelGGL(smp_cand_kernel, grid, block, 0, st, a);
        AR_LAUNCH_CHECK();
    } else {
        hipLaunchKernelGGL(smp_mass_kernel, grid, block, 0, st, a);
        AR_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(smp_draw_kernel, dim3(s.rows), block, 0, st, a);
    AR_LAUNCH_CHECK();
    return AR_HIP_OK;
}
