// Batched decode GEMV on the MFMA units: bf16 weights, 3..8 sequences.
//
// Same contract as the batch-1/2 GEMV (gemv_impl.h): the reference's dense -> matmul/weightedSum
// (domain/graph/.../LayerFeatures.java:785-830, compute/algebra/.../MatrixFeatures.java:182-337)
// with the RMSNorm prologue (NormalizationLayerFeatures.java:584-595) and the store / residual /
// SwiGLU / greedy-argmax epilogues.  With 8 sequences each weight element feeds 8 multiply-adds,
// which on the vector ALUs (fp32, 16 FMA lanes per SIMD per clock) costs about as much time as
// streaming the weight from HBM; the matrix cores take that work off the critical path.
//
// Product: one v_mfma_f32_16x16x32_bf16 per operand plane and 32-wide k-step.  A = 16 weight rows
// (lane l supplies row l%16, k = (l/16)*8 .. +7: one 16-byte load straight from the row-major bf16
// matrix); B = the batch as 16 columns (lane l supplies sequence l%16 at the same k; columns past
// the batch are 0).  The fp32 input is gain-scaled and split into bf16 planes hi = bf16(v),
// lo = bf16(v - hi), so hi + lo keeps 16 significant bits and the products accumulate in fp32.
// RMSNorm's 1/sqrt(mean(x^2) + eps) is a per-sequence scalar: the lanes accumulate sum(x^2) from
// the same loads and the factor scales the finished dot products.
//
// A block's wavefronts split the k-steps of a tile of weight rows and sum their 16 x 16 partial tiles
// through LDS in a fixed order.  Two forms:
//  * packed (up to 16 k-steps per wavefront: cols <= 4096, and at least as many tiles as CUs): one block per CU loops over
//    tiles with the input planes in registers (see gemv_mfma_pack_kernel);
//  * streaming (the rest): one tile per 16-wavefront block; each
//    chunk of k-steps issues its weight and input loads together, and the next chunk's loads are in
//    flight while the current chunk is converted and multiplied.
#include <algorithm>

#include "gemv_impl.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kPackWaves = 8;
constexpr int kPackSteps = 16;   // k-steps of a wavefront whose planes stay in registers
constexpr int kStreamWaves = 16;
constexpr int kStreamChunk = 2;  // k-steps per load chunk (two chunks in flight)
constexpr int kMaxKSplit = 4;    // k-slices per tile in the split streaming form

__device__ inline unsigned bf16_bits(float f) {  // round to nearest even (v_cvt_pk_bf16_f32); NaN stays NaN
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}

// 8 consecutive inputs of one sequence: gain applied when gp is given (sum of squares of the raw
// values added to ss), then split into hi and lo planes as MFMA B fragments.
__device__ inline void make_planes(float4 a, float4 b, const float* gp, float& ss, u32x4& hi, u32x4& lo) {
    float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    if (gp) {
        const float4 ga = *reinterpret_cast<const float4*>(gp);
        const float4 gb = *reinterpret_cast<const float4*>(gp + 4);
        const float g[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            ss = fmaf(v[j], v[j], ss);
            v[j] *= g[j];
        }
    }
    unsigned h[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const unsigned h0 = bf16_bits(v[2 * j]), h1 = bf16_bits(v[2 * j + 1]);
        h[j] = h0 | (h1 << 16);
        l[j] = bf16_bits(v[2 * j] - __uint_as_float(h0 << 16)) |
               (bf16_bits(v[2 * j + 1] - __uint_as_float(h1 << 16)) << 16);
    }
    hi = u32x4{h[0], h[1], h[2], h[3]};
    lo = u32x4{l[0], l[1], l[2], l[3]};
}

// sum of squares of 8 inputs added to ss, in the order make_planes adds them
__device__ inline void sumsq8(float4 a, float4 b, float& ss) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; j++) ss = fmaf(v[j], v[j], ss);
}

__device__ inline float4 load4(const float* p, bool live) {
    return live ? *reinterpret_cast<const float4*>(p) : make_float4(0.f, 0.f, 0.f, 0.f);
}

__device__ inline floatx4 mac2(const u32x4& w, const u32x4& hi, const u32x4& lo, floatx4 acc) {
    const bf16x8 a = __builtin_bit_cast(bf16x8, w);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, hi), acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, lo), acc, 0, 0, 0);
}

// Sums the per-wavefront partial tiles and applies the epilogue to output (row0 + t/16, sequence
// t%16) for threads t < 256, after the partials are in LDS.  For the argmax epilogue the values go
// to `tot`, and after a barrier one thread per sequence scans the tile's 16 rows.
template <int NW, int NMAT, int EPI>
struct Finish {
    __device__ static inline void sum(float (*cpart)[NMAT][256], int tid, float (&v)[NMAT]) {
#pragma unroll
        for (int m = 0; m < NMAT; m++) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) t += cpart[w][m][tid];
            v[m] = t;
        }
    }
    __device__ static inline void outputs(const gemv::Params& p, float (*cpart)[NMAT][256], float (*ssw)[16],
                                          bool norm, int row0, int tid, float* tot) {
        if (tid >= 256) return;
        const int b = tid & 15;
        float v[NMAT];
        sum(cpart, tid, v);
        if (norm) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) s += ssw[w][b];
            const float rn = 1.0f / sqrtf(s / (float)p.cols + p.eps);
#pragma unroll
            for (int m = 0; m < NMAT; m++) v[m] *= rn;
        }
        emit(p, v, row0, tid, tot);
    }
    // epilogue of output (row0 + tid/16, sequence tid%16) given its finished dot products
    __device__ static inline void emit(const gemv::Params& p, float (&v)[NMAT], int row0, int tid, float* tot) {
        const int ri = tid >> 4, b = tid & 15, row = row0 + ri;
        const bool out = row < p.rows && b < p.batch;
        if (EPI == GEMV_EPI_ARGMAX) {
            if (p.y && out) p.y[(size_t)b * p.y_stride + row] = v[0];
            tot[tid] = v[0];
            return;
        }
        if (!out) return;
        float* yp = p.y + (size_t)b * p.y_stride + row;
        float val;
        if (EPI == GEMV_EPI_STORE) {
            val = p.bias ? v[0] + p.bias[row] : v[0];
        } else if (EPI == GEMV_EPI_RESIDUAL) {
            val = *yp + v[0];
        } else {  // SwiGLU: u * (g * 1/(exp(-g)+1))
            const float g = v[0], u = v[NMAT - 1];
            const float sg = 1.0f / (expf(-g) + 1.0f);
            val = u * (g * sg);
        }
        *yp = val;
        if (p.y_hi) {  // operand planes of the next GEMV's input
            const size_t o = (size_t)b * p.y_stride + row;
            bf16_planes(p.y_gain ? val * p.y_gain[row] : val, p.y_hi + o, p.y_lo + o);
        }
    }
    __device__ static inline void argmax(const gemv::Params& p, const float* tot, int row0, int tile, int tid) {
        if (tid >= p.batch) return;
        float bv = -INFINITY;
        int bi = 0x7FFFFFFF;
        for (int i = 0; i < 16; i++) {
            const int rr = row0 + i;
            if (rr < p.rows && gemv::better(tot[i * 16 + tid], rr, bv, bi)) {
                bv = tot[i * 16 + tid];
                bi = rr;
            }
        }
        if (bi != 0x7FFFFFFF)
            atomicMax(p.keys + (size_t)tid * kArgmaxSlots + (tile & (kArgmaxSlots - 1)), gemv::argmax_key(bv, bi));
    }
};

// One MFMA per k-step carries both planes, lanes 0-7 of each 16-lane row the hi plane of
// sequences 0-7 and lanes 8-15 the lo plane, so columns b and b + 8 of the result add up to sequence b's
// products (half the MFMAs and half the plane registers of one MFMA per plane).  A tile is 16 weight
// rows; for SwiGLU 8 gate rows and the same 8 up rows.
// One block of 8 wavefronts per CU walks tiles t, t + grid, ...; a wavefront's k-steps of the next SETS
// tiles are always in flight (register sets, two to four: some 100 KB per CU), across the tile's one barrier, which waits for LDS only
// (a barrier that waits for the loads too leaves the CU without any request once per tile).  Four
// wavefronts finish a tile while the others go on.
// In a decode step of the 4B shape, weights cold in HBM: QKV (6,144 x 2,560) 15.7 -> 13.7 us, 16,896-row
// head 31 -> 24, against one MFMA per plane, whole 16 + 16-row tiles and a full barrier.  Bound by HBM and, with
// few tiles per CU, by the first loads' latency and the last round.  Repeated calls on one matrix, which
// then stays in the last-level cache: 9,728 x 2,560 SwiGLU, 8 sequences, 34 -> 26 us (608 tiles on 256 CUs were
// 2.4 rounds).  Narrow inputs have instances of one and two k-steps: three loads a tile where one is needed
// cost more than the tile (8,192 x 256 SwiGLU, 8 sequences: 7.9 us with three, 5.5 with one; inputs of fewer than
// eight k-steps on the streaming form, a block per tile: 32,000 x 224 19.2 us, 6.1 here).  8-row tiles for the other epilogues too (QKV in one and a
// half rounds instead of two) measured slower: 14.7 us, twice the barriers for the same bytes.
template <int EPI, int KS>
__global__ __launch_bounds__(kPackWaves * 64, 2) void gemv_mfma_pack_kernel(gemv::Params p, int tiles) {
    constexpr int NW = kPackWaves, SETS = KS <= 6 ? 4 : KS <= 10 ? 3 : 2;  // tiles in flight
    constexpr bool SW = EPI == GEMV_EPI_SWIGLU;
    constexpr int TR = SW ? 8 : 16;  // output rows of a tile
    __shared__ float cpart[2][NW][256];
    __shared__ float ssw[NW][8];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15,
              q = lane >> 4, seq = r & 7;
    const int nsteps = p.cols / 32, s0 = nsteps * w / NW, ns = nsteps * (w + 1) / NW - s0;  // KS - 2 <= ns <= KS
    const int last = max(ns - 1, 0);  // (fewer k-steps than wavefronts: some have none, and read step s0)
    const bool live = seq < p.batch, norm = p.norm_w != nullptr;
    const int step = gridDim.x;

    // weight rows of this lane in tile t: row t * TR + lane's row of its matrix; tiles past the end read
    // one line over and over instead of branching, so the waits count loads exactly
    const uint16_t* const wm = reinterpret_cast<const uint16_t*>(SW && r >= 8 ? p.w2 : p.w);
    const int lrow = TR == 8 ? r & 7 : r;
    const size_t koff = (size_t)s0 * 32 + 8 * q;
    // (a line of its own for every wavefront: one line for all of them is one L2 channel's queue)
    const uint16_t* const idle = reinterpret_cast<const uint16_t*>(p.w) + (size_t)blockIdx.x * TR * p.cols + s0 * 32;
    u32x4 wv[SETS][KS];
    auto load = [&](int set, int t) __attribute__((always_inline)) {
        const bool in = t < tiles;
        const uint16_t* src = in ? wm + (size_t)min(t * TR + lrow, p.rows - 1) * p.cols + koff : idle;
        const int inc = in ? 32 : 0;
#pragma unroll
        for (int i = 0; i < KS; i++)  // (steps past ns repeat the last one; never multiplied)
            wv[set][i] = *reinterpret_cast<const u32x4*>(src + (i < KS - 2 ? i : min(i, last)) * inc);
    };
    int t = blockIdx.x;

    // this lane's plane of its sequence, once for all tiles: as written by the kernel that produced the
    // input, or converted here.  With planes the RMSNorm sum of squares still comes from the fp32 input:
    // lane l sums sequence l / 8, and its loads and the planes' go ahead of the weights of two tiles, so
    // nothing waits behind those and HBM has requests from the start
    u32x4 pv[KS];
    float ss = 0.f;
    const bool planes = p.x_hi != nullptr;
    const size_t xo = (size_t)min(seq, p.batch - 1) * p.x_stride + koff;
    if (planes) {
        float4 xs[KS];
        const int sseq = lane >> 3;
        const float* const xrow = p.x + (size_t)min(sseq, p.batch - 1) * p.x_stride + (size_t)s0 * 32 + 4 * (lane & 7);
        if (norm)
#pragma unroll
            for (int i = 0; i < KS; i++)
                xs[i] = *reinterpret_cast<const float4*>(xrow + (i < KS - 2 ? i : min(i, last)) * 32);
        const uint16_t* const pl = (r < 8 ? p.x_hi : p.x_lo) + xo;
#pragma unroll
        for (int i = 0; i < KS; i++)
            pv[i] = *reinterpret_cast<const u32x4*>(pl + (i < KS - 2 ? i : min(i, last)) * 32);
        if (KS <= 12) {  // (registers: above 12 steps after the sums)
            load(0, t);
            load(1, t + step);
        }
        if (norm) {
#pragma unroll
            for (int i = 0; i < KS; i++)
                if (i < KS - 2 || i < ns) {
                    ss = fmaf(xs[i].x, xs[i].x, ss);
                    ss = fmaf(xs[i].y, xs[i].y, ss);
                    ss = fmaf(xs[i].z, xs[i].z, ss);
                    ss = fmaf(xs[i].w, xs[i].w, ss);
                }
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) ss += __shfl_xor(ss, off, 64);
            if ((lane & 7) == 0) ssw[w][sseq] = ss;
        }
        if (KS > 12) {
            load(0, t);
            load(1, t + step);
        }
        if (!live)
#pragma unroll
            for (int i = 0; i < KS; i++) pv[i] = u32x4{0u, 0u, 0u, 0u};
    } else {
        load(0, t);
        if (KS <= 12) load(1, t + step);
#pragma unroll
        for (int i = 0; i < KS; i++) {
            const int k = (i < KS - 2 ? i : min(i, last)) * 32;
            const bool use = live && (i < KS - 2 || i < ns);
            u32x4 hi, lo;
            make_planes(load4(p.x + xo + k, use), load4(p.x + xo + k + 4, use), norm ? p.norm_w + koff + k : nullptr, ss,
                        hi, lo);
            pv[i] = r < 8 ? hi : lo;
        }
        if (norm) {
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            if (q == 0 && r < 8) ssw[w][r] = ss;
        }
        if (KS > 12) load(1, t + step);
    }
#pragma unroll
    for (int k = 2; k < SETS; k++) load(k, t + k * step);

    float rn = 1.f;          // finishing wavefronts: RMSNorm factor of sequence `seq`
    bool have_rn = false;
    int par = 0;             // partial-tile buffer of the next tile
    float best = -INFINITY;  // ARGMAX: this lane's best value and its row over every tile
    int besti = 0x7FFFFFFF;
    // rows of a finished tile by lane, gate row and up row of one output 32 lanes apart
    const int frow = (q & 1) + 2 * w + (q >> 1) * 8;
    auto tile = [&](int set) __attribute__((always_inline)) {
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < KS; i++)
            if (i < KS - 2 || i < ns)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[set][i]),
                                                              __builtin_bit_cast(bf16x8, pv[i]), acc, 0, 0, 0);
        load(set, t + SETS * step);
#pragma unroll
        for (int j = 0; j < 4; j++) cpart[par][w][(4 * q + j) * 16 + r] = acc[j];
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the weight loads stay in flight
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        par ^= 1;
        if (w >= 4) return;
        if (norm && !have_rn) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < NW; k++) s += ssw[k][seq];
            rn = 1.0f / sqrtf(s / (float)p.cols + p.eps);
            have_rn = true;
        }
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < NW; k++) v += cpart[par ^ 1][k][frow * 16 + r];
        v = (v + __shfl_xor(v, 8, 64)) * rn;  // hi + lo
        const float up = SW ? __shfl_xor(v, 32, 64) : 0.f;
        const int row = t * TR + frow;
        if (r >= 8 || !live || frow >= TR || row >= p.rows) return;
        if constexpr (EPI == GEMV_EPI_ARGMAX) {
            if (p.y) p.y[(size_t)seq * p.y_stride + row] = v;
            if (gemv::better(v, row, best, besti)) {
                best = v;
                besti = row;
            }
        } else {
            const size_t o = (size_t)seq * p.y_stride + row;
            float val;
            if constexpr (EPI == GEMV_EPI_STORE) {
                val = p.bias ? v + p.bias[row] : v;
            } else if constexpr (EPI == GEMV_EPI_RESIDUAL) {
                val = p.y[o] + v;
            } else {  // SwiGLU: u * (g * 1/(exp(-g)+1))
                const float sg = 1.0f / (expf(-v) + 1.0f);
                val = up * (v * sg);
            }
            p.y[o] = val;
            if (p.y_hi) bf16_planes(p.y_gain ? val * p.y_gain[row] : val, p.y_hi + o, p.y_lo + o);
        }
    };
    while (t < tiles) {
#pragma unroll
        for (int k = 0; k < SETS; k++) {
            tile(k);
            t += step;
            if (t >= tiles) break;
        }
    }
    if constexpr (EPI == GEMV_EPI_ARGMAX) {
        if (w >= 4) return;
        // the best of this wavefront's rows, then one key per sequence
#pragma unroll
        for (int off = 16; off < 64; off <<= 1) {
            const float ov = __shfl_xor(best, off, 64);
            const int oi = __shfl_xor(besti, off, 64);
            if (gemv::better(ov, oi, best, besti)) {
                best = ov;
                besti = oi;
            }
        }
        if (q == 0 && r < 8 && live && besti != 0x7FFFFFFF)
            atomicMax(p.keys + (size_t)seq * kArgmaxSlots + ((blockIdx.x * 4 + w) & (kArgmaxSlots - 1)),
                      gemv::argmax_key(best, besti));
    }
}

template <int EPI>
void launch_pack(const gemv::Params& p, int cus, hipStream_t st) {
    const int rows = EPI == GEMV_EPI_SWIGLU ? 8 : 16, tiles = (p.rows + rows - 1) / rows;
    const dim3 grid(std::min(tiles, cus)), block(64 * kPackWaves);
    const int ks = (p.cols / 32 + kPackWaves - 1) / kPackWaves;
#define AR_PACK(K) \
    if (ks <= K) return ar_launch((gemv_mfma_pack_kernel<EPI, K>), grid, block, 0, st, p, tiles)
    AR_PACK(1);
    AR_PACK(2);
    AR_PACK(3);
    AR_PACK(4);
    AR_PACK(5);
    AR_PACK(6);
    AR_PACK(8);
    AR_PACK(10);
    AR_PACK(12);
    AR_PACK(14);
    AR_PACK(16);
#undef AR_PACK
}

// NWS wavefronts per block; ks blocks per 16-row tile (block = tile * ks + k-slice), each taking
// a contiguous share of the k-steps.  With ks > 1 the blocks store their partial tiles in the
// workspace and the last one to arrive adds the ks partials in k-slice order and applies the
// epilogue (partials through agent-scope atomic accesses, as the attention merge would need; no
// device-wide fence).
template <int EPI, int NWS>
__global__ __launch_bounds__(NWS * 64, NWS == 8 ? 4 : 1) void gemv_mfma_stream_kernel(gemv::Params p, int kpw, int ks) {
    constexpr int NW = NWS, NMAT = (EPI == GEMV_EPI_SWIGLU) ? 2 : 1, KC = kStreamChunk;
    using F = Finish<NW, NMAT, EPI>;
    __shared__ float cpart[NW][NMAT][256];
    __shared__ float ssw[NW][16];
    __shared__ float tot[256];
    __shared__ int last_s;

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, q = lane >> 4;
    const int tile = blockIdx.x / ks, kh = blockIdx.x - tile * ks;
    const int row0 = tile * 16;
    const int nsteps = p.cols / 32;
    const int per = (nsteps + ks - 1) / ks;  // k-steps of this block: [kh*per, min((kh+1)*per, nsteps))
    const int kend = min((kh + 1) * per, nsteps);
    const int s0 = kh * per + w * kpw, s1 = min(s0 + kpw, kend);
    const bool live = r < p.batch;
    const bool norm = p.norm_w != nullptr;
    const size_t wrow = (size_t)min(row0 + r, p.rows - 1) * p.cols + 8 * q;
    const uint16_t* wa = reinterpret_cast<const uint16_t*>(p.w) + wrow;
    const uint16_t* wb = NMAT == 2 ? reinterpret_cast<const uint16_t*>(p.w2) + wrow : nullptr;
    const float* xp = p.x + (size_t)min(r, p.batch - 1) * p.x_stride + 8 * q;
    const float* gp = norm ? p.norm_w + 8 * q : nullptr;

    floatx4 acc[NMAT];
#pragma unroll
    for (int m = 0; m < NMAT; m++) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
    float ss = 0.f;
    // two chunk buffers: the next chunk's loads are in flight while the current one is multiplied
    u32x4 wv[2][NMAT][KC];
    float4 xa[2][KC], xb[2][KC];
    u32x4 ph[2][KC], pl[2][KC];  // operand planes read as written by the input's producer
    const bool planes = p.x_hi != nullptr;
    const uint16_t* phs = planes ? p.x_hi + (size_t)min(r, p.batch - 1) * p.x_stride + 8 * q : nullptr;
    const uint16_t* pls = planes ? p.x_lo + (size_t)min(r, p.batch - 1) * p.x_stride + 8 * q : nullptr;
    const u32x4 zero4 = {0u, 0u, 0u, 0u};
#define AR_MFMA_LOAD_CHUNK(buf_, sb_)                                                    \
    _Pragma("unroll") for (int i = 0; i < KC; i++) {                                     \
        const int k = min((sb_) + i, s1 - 1) * 32;                                       \
        wv[buf_][0][i] = *reinterpret_cast<const u32x4*>(wa + k);                        \
        if (NMAT == 2) wv[buf_][NMAT - 1][i] = *reinterpret_cast<const u32x4*>(wb + k);  \
        if (planes) {                                                                    \
            ph[buf_][i] = live ? *reinterpret_cast<const u32x4*>(phs + k) : zero4;       \
            pl[buf_][i] = live ? *reinterpret_cast<const u32x4*>(pls + k) : zero4;       \
        }                                                                                \
        if (!planes || norm) {                                                           \
            xa[buf_][i] = load4(xp + k, live);                                           \
            xb[buf_][i] = load4(xp + k + 4, live);                                       \
        }                                                                                \
    }
#define AR_MFMA_MUL_CHUNK(buf_, sb_)                                                                     \
    _Pragma("unroll") for (int i = 0; i < KC; i++) {                                                     \
        if ((sb_) + i < s1) { /* uniform over the wavefront */                                           \
            u32x4 hi, lo;                                                                                \
            if (planes) {                                                                                \
                hi = ph[buf_][i];                                                                        \
                lo = pl[buf_][i];                                                                        \
                if (norm) sumsq8(xa[buf_][i], xb[buf_][i], ss);                                         \
            } else {                                                                                     \
                make_planes(xa[buf_][i], xb[buf_][i], gp ? gp + ((sb_) + i) * 32 : nullptr, ss, hi, lo); \
            }                                                                                            \
            _Pragma("unroll") for (int m = 0; m < NMAT; m++) acc[m] = mac2(wv[buf_][m][i], hi, lo, acc[m]); \
        }                                                                                                \
    }
    if (s0 < s1) AR_MFMA_LOAD_CHUNK(0, s0)
    for (int sb = s0; sb < s1; sb += 2 * KC) {
        if (sb + KC < s1) AR_MFMA_LOAD_CHUNK(1, sb + KC)
        AR_MFMA_MUL_CHUNK(0, sb)
        if (sb + 2 * KC < s1) AR_MFMA_LOAD_CHUNK(0, sb + 2 * KC)
        if (sb + KC < s1) AR_MFMA_MUL_CHUNK(1, sb + KC)
    }
#undef AR_MFMA_LOAD_CHUNK
#undef AR_MFMA_MUL_CHUNK
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) cpart[w][m][(4 * q + j) * 16 + r] = acc[m][j];
    if (norm) {
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        if (q == 0) ssw[w][r] = ss;
    }
    __syncthreads();
    if (ks == 1) {
        F::outputs(p, cpart, ssw, norm, row0, tid, tot);
        if (EPI == GEMV_EPI_ARGMAX) {
            __syncthreads();
            F::argmax(p, tot, row0, tile, tid);
        }
        return;
    }
    // k-split (no RMSNorm, no argmax): partial tile -> workspace; the last block of the tile folds
    float v[NMAT];
    if (tid < 256) {
        F::sum(cpart, tid, v);
#pragma unroll
        for (int m = 0; m < NMAT; m++)
            __hip_atomic_store(p.kpart + ((size_t)blockIdx.x * NMAT + m) * 256 + tid, v[m], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0);  // this thread's partial stores have completed
    __syncthreads();
    if (tid == 0) {
        unsigned* c = p.kcount + tile;
        const unsigned prev = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = prev == (unsigned)(ks - 1);
        if (last) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_s = last;
    }
    __syncthreads();
    if (!last_s || tid >= 256) return;
#pragma unroll
    for (int m = 0; m < NMAT; m++) {
        float t = 0.f;
        for (int j = 0; j < ks; j++)
            t += __hip_atomic_load(p.kpart + ((size_t)(tile * ks + j) * NMAT + m) * 256 + tid, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        v[m] = t;
    }
    F::emit(p, v, row0, tid, tot);
}


template <int EPI>
int launch_epi(const gemv::Params& p, hipStream_t st) {
    constexpr int NMAT = (EPI == GEMV_EPI_SWIGLU) ? 2 : 1;
    const int nsteps = p.cols / 32, tiles = (p.rows + 15) / 16;
    const int persist = ar_device_cus(st);  // one packed block per CU of the stream's device
    // fewer tiles than CUs (the 2560-row projections at C5): one tile per 16-wavefront block spreads
    // the loads over more wavefronts (measured: O 4096 -> 2560 15.5 us streaming vs 23.7 with one block per
    // tile of 8 wavefronts).  The packed form takes up to 16 k-steps per wavefront.
    if (nsteps <= kPackWaves * kPackSteps && (NMAT == 2 ? (p.rows + 7) / 8 : tiles) >= persist) {
        launch_pack<EPI>(p, persist, st);
    } else {
        // fewer tiles than CUs and nothing that needs the whole row in one block: split k over
        // ks = 2*CUs / tiles blocks of 8 wavefronts (two per CU), partials folded in order
        int ks = 1;
        if (p.kpart && p.kcount && tiles <= p.kcount_n && !p.norm_w && EPI != GEMV_EPI_ARGMAX &&
            tiles < persist) {
            ks = std::min(kMaxKSplit, std::max(1, 2 * persist / tiles));
            while (ks > 1 && ((long long)tiles * ks * NMAT * 256 > p.kpart_floats || nsteps < ks * 8)) ks--;
        }
        if (ks > 1) {
            const int per = (nsteps + ks - 1) / ks, kpw = (per + 7) / 8;
            ar_launch((gemv_mfma_stream_kernel<EPI, 8>), dim3(tiles * ks), dim3(64 * 8), 0, st, p, kpw, ks);
        } else {
            const int kpw = (nsteps + kStreamWaves - 1) / kStreamWaves;
            ar_launch((gemv_mfma_stream_kernel<EPI, kStreamWaves>), dim3(tiles), dim3(64 * kStreamWaves), 0, st,
                               p, kpw, 1);
        }
    }
    AR_LAUNCH_CHECK();
    return AR_HIP_OK;
}

}  // namespace

int gemv_launch_mfma(const gemv::Params& p, int epi, hipStream_t st) {
    AR_CHECK_ARG(p.batch >= 1 && p.batch <= 8 && p.cols % 32 == 0, "MFMA GEMV: batch %d / cols %d unsupported",
                 p.batch, p.cols);
    switch (epi) {
        case GEMV_EPI_STORE: return launch_epi<GEMV_EPI_STORE>(p, st);
        case GEMV_EPI_RESIDUAL: return launch_epi<GEMV_EPI_RESIDUAL>(p, st);
        case GEMV_EPI_SWIGLU: return launch_epi<GEMV_EPI_SWIGLU>(p, st);
        case GEMV_EPI_ARGMAX: return launch_epi<GEMV_EPI_ARGMAX>(p, st);
        default: ar_set_error("GEMV: unknown epilogue %d", epi); return AR_HIP_ERR_INVALID;
    }
}
