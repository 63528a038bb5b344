// fp32 multi-token projection on the MFMA units (v_mfma_f32_32x32x2_f32): the prompt rows of an
// fp32-weight model in one product per projection instead of one decode step per token.
//
// C[M x N] = A[M x K] . W[N x K]^T, fp32 operands and accumulation -- the stacked-row form of
// LayerFeatures.dense (domain/graph/.../LayerFeatures.java:785-830) for prompt rows, which the
// reference feeds one per step (engine/ml/.../AutoregressiveModel.java:295-308).
//
// Bound by the fp32 matrix rate (157 TFLOP/s at 2.4 GHz; 137-150 over launches of 0.1-0.4 ms, whose
// clock is lower).  One block per CU, in whole rounds of blocks, or several small ones, at the tile that
// takes least time by the launch rule.
// Epilogues: STORE (+ bias), RESIDUAL (C += product), SWIGLU (C = (A.W2^T) * silu(A.W^T)), and
// k-slices stored separately for the consumer to add in a fixed order.
#include <atomic>

#include "ar_hip_internal.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));  // (a native vector: stays in registers)

constexpr int BK = 32;  // k values of one tile, and the granularity every launch accepts

struct Params {
    const float* A;   // [M][lda]
    const float* W;   // [N][ldw]
    const float* W2;  // SwiGLU up projection, or null
    const float* bias;
    float* C;         // [M][ldc] (ksplit > 1: slice s at C + s*M*ldc)
    int M, N, K, lda, ldw, ldc, ksplit;
};

// Output tile of block `bid`: consecutive blocks (one XCD takes every 8th) walk m fastest within
// groups of 8 n-tiles, so blocks running together on an XCD share W column tiles in its L2.
__device__ inline void tile_of(int bid, int mt, int nt, int* mi, int* ni) {
    const int nblk = mt * nt, q = nblk >> 3, r = nblk & 7, xcd = bid & 7;
    const int t = xcd * q + min(xcd, r) + (bid >> 3);
    *mi = t % mt;
    *ni = t / mt;
}

// Block barrier over LDS only: the weight loads of the next iteration stay in flight across it.
__device__ inline void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt left at their maxima
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// s_waitcnt immediates (vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] at [15:14]): vmcnt v, lgkmcnt l
constexpr int vm_imm(int v, int l = 15) { return (v & 15) | ((v >> 4) << 14) | (7 << 4) | (l << 8); }
typedef __attribute__((address_space(3))) void lds_void;

// A block of four wavefronts takes 32*MB rows x 32*WN output columns (WN column wavefronts x KG = 4/WN
// k-groups; SwiGLU blocks hold the gate and the up rows of their columns), one k-tile of 32 per
// iteration out of ST LDS stages.  Operands of one MFMA step: lanes 0-31 supply k = 8q + c, lanes 32-63
// k = 8q + 4 + c, for component c of the float4 each lane holds of chunk q, so the 32x32x2 MFMA pairs
// equal k values of A and W.  Both operands go from global memory straight into LDS
// (`global_load_lds_dwordx4`: 64 lanes x 16 contiguous bytes, coalesced, no staging registers), rows of
// 8 chunks of 16 bytes, chunk c of row r in slot c ^ (r & 7), so the lanes of one 16-byte read phase hit
// different bank groups.  The iteration's one barrier comes before its last MFMAs, once every fragment
// of the tile is read: behind it the next tile is whole and this tile's stage is free for tile
// ST ahead, and the last MFMAs cover the reads of the next tile's first fragments.  Each output is CH sums
// (k-groups times k-tiles modulo CH / KG) added at the end: shorter chains of roundings.
// The small tiles take eight or four stages: their products stream the weights, cold from HBM, and two
// stages ran the 128-row products of a 0.6B layer in 28 (gate/up) and 20 us (the others) against 24 and
// 13; the large tiles are as fast with two.
// A second large block on the CU makes the last round uneven (both blocks of a pair end together, the
// leftover blocks pair up again on the CUs that end first: 1,531 x 3,072 x 1,024 SwiGLU 164 us at one block
// per CU, 267 us at two), so their launches ask for more than half of a CU's LDS.  The 32-row tiles of many
// rows (CH 2) are the other way round: 32 x 64 has 512 cycles of MFMAs a k-tile, less than a load takes,
// so two stages and one block per CU leave the matrix units waiting, and its start and stores are a fifth
// of a short product.  With four stages, three (32 x 64) or two (32 x 128) blocks share a CU: 1,672 x
// 4,032 x 320 79 -> 51 us, 1,900 x 1,728 x 960 104 -> 70.
template <int MB, int WN, int CH, int EPI>
struct F32Shape {
    static constexpr int KG = 4 / WN, NB = EPI == GEMV_EPI_SWIGLU ? 2 : 1;
    static constexpr int BM = 32 * MB, NOUT = 32 * WN, BN = NOUT * NB;  // output tile BM x NOUT, BN weight rows
    static constexpr int STAGE = (BM + BN) * BK;               // floats of one stage
    static constexpr bool SHARE = CH <= 2 && MB == 1 && NB == 1;  // several blocks per CU
    // stages: two, four for blocks that share a CU, or for the small tiles (CH 4) eight or four, up to 152 KB
    static constexpr int ST = SHARE ? 4 : CH <= 2 ? 2 : 8 * STAGE <= 38 * 1024 ? 8 : 4;
    static constexpr int RED = KG > 1 ? WN * MB * NB * 1024 : 0;  // the second k-group's sums
    static constexpr int USED = (ST * STAGE > RED ? ST * STAGE : RED) * 4;
    // more than half of a CU's 160 KB (one block per CU), or 48 and 80 KB: three and two blocks
    static constexpr int LDS_BYTES = SHARE || USED > 82 * 1024 ? USED : 82 * 1024;
};

template <int MB, int WN, int CH, int EPI>
__global__ __launch_bounds__(256, 1) void gemm_f32_kernel(Params p, int mt, int nt) {
    using Sh = F32Shape<MB, WN, CH, EPI>;
    constexpr int ST = Sh::ST;
    constexpr int NB = Sh::NB, KG = Sh::KG, NA = CH / KG;  // NA sums per output and wavefront
    constexpr int NQ = BK / 8 / KG;                       // float4 chunks per lane of a k-tile
    constexpr int CP = (Sh::BM + Sh::BN) / 32;            // copies (8 rows each) per wavefront and stage
    extern __shared__ __attribute__((aligned(1024))) float dsm[];
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / WN, wn = wave % WN;
    const int tiles = mt * nt, ks = blockIdx.x / tiles;
    int mi, ni;
    tile_of(blockIdx.x - ks * tiles, mt, nt, &mi, &ni);
    const int m0 = mi * Sh::BM, n0 = ni * Sh::NOUT;
    const int kper = p.K / p.ksplit, kbase = ks * kper, nit = kper / BK;

    // a stage holds the A rows, then the W rows (gate, then up); copy i of this wavefront fills rows
    // 8*(4i + wave) .. +7, lane l slot l % 8 of row l / 8 (rows past M re-read the last row)
    const int drow = lane >> 3, dslot = lane & 7;
    const float* src[CP];
#pragma unroll
    for (int i = 0; i < CP; i++) {
        const int r = 8 * (4 * i + wave) + drow, w = r - Sh::BM;
        const float* row = r < Sh::BM ? p.A + (size_t)min(m0 + r, p.M - 1) * p.lda
                           : w < Sh::NOUT ? p.W + (size_t)(n0 + w) * p.ldw
                                          : p.W2 + (size_t)(n0 + w - Sh::NOUT) * p.ldw;
        src[i] = row + kbase + 4 * (dslot ^ (r & 7));
    }
    auto copy = [&](int it, int st) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < CP; i++)
            __builtin_amdgcn_global_load_lds((const void*)(src[i] + it * BK),
                                             (lds_void*)(dsm + st * Sh::STAGE + (4 * i + wave) * 256), 16, 0, 0);
    };

    floatx16 acc[NA][MB][NB];
#pragma unroll
    for (int k = 0; k < NA; k++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[k][i][j][r] = 0.f;
    f4 a[2][MB], w[2][NB];
    auto read = [&](int st, int q) __attribute__((always_inline)) {
        const float* const row = dsm + st * Sh::STAGE + l32 * BK + 4 * ((2 * (kg * NQ + q) + h) ^ (l32 & 7));
#pragma unroll
        for (int i = 0; i < MB; i++) a[q & 1][i] = *reinterpret_cast<const f4*>(row + 32 * i * BK);
#pragma unroll
        for (int j = 0; j < NB; j++) w[q & 1][j] = *reinterpret_cast<const f4*>(row + (Sh::BM + j * Sh::NOUT + 32 * wn) * BK);
    };
    auto step = [&](int it, int u) __attribute__((always_inline)) {  // u: it modulo U
        const int st = u % ST;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            if (q + 1 < NQ) {
                read(st, q + 1);
            } else {
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(vm_imm((ST - 2) * CP, 0));  // tile it + 1 copied, tile `it` read
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                read((st + 1) % ST, 0);
                copy(min(it + ST, nit - 1), st);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        acc[u % NA][i][j] =
                            __builtin_amdgcn_mfma_f32_32x32x2f32(a[q & 1][i][e], w[q & 1][j][e], acc[u % NA][i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // (past the last tile the copies re-read it into a stage nobody reads: a branch round them and waits counted
    // for the tail measured slower, 75.3 -> 76.4 us at 1,021 x 4,096 x 1,024 and 21.3 -> 24.3 at 253 x 704 x 2,080)
#pragma unroll
    for (int i = 0; i < ST; i++) copy(min(i, nit - 1), i);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(vm_imm((ST - 1) * CP));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    constexpr int U = ST > NA ? ST : NA;  // tiles per turn: the stage and the sum are compile-time indexes
    int it = 0;
    for (; it + U <= nit; it += U)
#pragma unroll
        for (int u = 0; u < U; u++) step(it + u, u);
#pragma unroll
    for (int u = 0; u < U - 1; u++)
        if (it + u < nit) step(it + u, u);
    __builtin_amdgcn_s_waitcnt(vm_imm(0, 0));
    __builtin_amdgcn_s_barrier();  // no copy and no read in flight
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 1; k < NA; k++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[0][i][j][r] += acc[k][i][j][r];
    if constexpr (KG > 1) {  // the second k-group hands its sums over
        float* const red = dsm + wn * (MB * NB * 1024) + lane;
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) red[((i * NB + j) * 16 + r) * 64] = acc[0][i][j][r];
        }
        lds_barrier();
        if (kg > 0) return;
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[0][i][j][r] += red[((i * NB + j) * 16 + r) * 64];
    }

    // output block: lane holds column (lane & 31), rows (r>>2)*8 + (lane>>5)*4 + (r&3)
    const int col = n0 + 32 * wn + l32;
    const float bias = EPI == GEMV_EPI_STORE && p.bias ? p.bias[col] : 0.f;
    float* const Cs = p.C + (size_t)ks * p.M * p.ldc + col;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = m0 + 32 * i + (r >> 2) * 8 + h * 4 + (r & 3);
            if (row >= p.M) continue;
            float* c = Cs + (size_t)row * p.ldc;
            if (EPI == GEMV_EPI_STORE) {
                *c = p.bias ? acc[0][i][0][r] + bias : acc[0][i][0][r];
            } else if (EPI == GEMV_EPI_RESIDUAL) {
                *c = *c + acc[0][i][0][r];
            } else {
                const float g = acc[0][i][0][r], u = acc[0][i][NB - 1][r];
                const float sg = 1.0f / (expf(-g) + 1.0f);
                *c = u * (g * sg);
            }
        }
}

template <int MB, int WN, int CH, int EPI>
int launch_t(const Params& p, hipStream_t st) {
    using Sh = F32Shape<MB, WN, CH, EPI>;
    static_assert(Sh::LDS_BYTES <= 160 * 1024, "LDS");
    const int mt = (p.M + Sh::BM - 1) / Sh::BM, nt = p.N / Sh::NOUT;
    const long long blocks = (long long)mt * nt * p.ksplit;
    AR_CHECK_ARG(blocks <= 0x7fffffffLL, "GEMM f32: too many blocks");
    auto kern = gemm_f32_kernel<MB, WN, CH, EPI>;
    // more than 64 KB of dynamic LDS needs the per-kernel opt-in, once per device
    static std::atomic<bool> attr_set[kMaxDevices];
    const int slot = ar_device_slot(st);
    if (slot < 0 || !attr_set[slot].load(std::memory_order_relaxed)) {
        AR_HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Sh::LDS_BYTES));
        if (slot >= 0) attr_set[slot].store(true, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), Sh::LDS_BYTES, st, p, mt, nt);
    AR_LAUNCH_CHECK();
    return AR_HIP_OK;
}

// The tile with the least time over whole rounds of blocks.  Time of a round in us: the MFMA cycles of a
// 32*MB x 32*WN tile at what they measured (0.48 ns a cycle; 0.58 and 0.495 for the 32 x 64 and 32 x 128
// blocks that share a CU), and the start, k-group fold and stores (1 + 2*MB; shared blocks 0.75 and 2.25, for
// the rest of it once a launch).  Fitted over 90 shapes of 512..2,048 rows, N 512..4,096, K 256..3,072 with every
// tile timed on each: 1% spread, and the tile chosen is 0.2% off the best of its shape on average, 5% at
// most.  Two terms in MFMA cycles and one block per CU throughout (the rule before) chose 32 x 64 in eleven rounds
// for 1,549 x 3,520 x 2,912: 432 us, 298 with shared blocks; the 64 x 64 form of two blocks per CU that ran
// there earlier took 364.  That form is still up to 8% faster where its blocks fill two rounds almost
// exactly (726 x 3,776 x 960: 56 and 61 us; 1,190 x 1,600 x 1,216: 47 and 50), and 1.4 times slower over the
// 90 shapes.  Below 512 rows the sums stay in four chains
// (as many roundings as the 32-row form with four k-groups that ran there), which leaves registers for
// at most 64 rows: 256 x 3,072 x 1,024 SwiGLU 48 -> 40, 128 x 4,096 x 1,024 15.6 -> 14.6 (us, repeated
// calls on the same operands); a round's start counts the same for all of them.
template <int EPI>
int launch_epi(const Params& p, hipStream_t st, int cus) {
    constexpr bool SW = EPI == GEMV_EPI_SWIGLU;
    const int kper = p.K / p.ksplit, max_mb = p.M >= 512 ? 4 : 2;
    int mb = 1, wn = 2;
    double best = 0;
    for (int w = 2; w <= (SW ? 2 : 4); w += 2)
        for (int b = 1; b <= max_mb; b++) {
            if (p.N % (32 * w)) continue;
            const long long blocks = (long long)((p.M + 32 * b - 1) / (32 * b)) * (p.N / (32 * w)) * p.ksplit;
            const double rounds = (double)((blocks + cus - 1) / cus), mfma = 8.0 * b * w * (SW ? 2 : 1) * kper;
            double cost = rounds * (0.48e-3 * mfma + 1.0 + (p.M >= 512 ? 2.0 * b : 0.0));
            if (p.M >= 512 && b == 1 && !SW)
                cost = w == 2 ? rounds * (0.58e-3 * mfma + 0.75) + 1.75 : rounds * (0.495e-3 * mfma + 2.25) + 1.0;
            if (best == 0 || cost < best) {
                best = cost;
                mb = b;
                wn = w;
            }
        }
#define AR_F32_TILE(MBV, WNV, CHV) \
    if (mb == MBV && wn == WNV) return launch_t<MBV, WNV, CHV, EPI>(p, st)
    if (p.M < 512) {
        AR_F32_TILE(1, 2, 4);
        AR_F32_TILE(2, 2, 4);
        if constexpr (!SW) {
            AR_F32_TILE(1, 4, 4);
            AR_F32_TILE(2, 4, 4);
        }
    } else {
        AR_F32_TILE(1, 2, 2);
        AR_F32_TILE(2, 2, 2);
        AR_F32_TILE(3, 2, 2);
        AR_F32_TILE(4, 2, 2);
        if constexpr (!SW) {
            AR_F32_TILE(1, 4, 2);
            AR_F32_TILE(2, 4, 2);
            AR_F32_TILE(3, 4, 2);
            AR_F32_TILE(4, 4, 2);
        }
    }
#undef AR_F32_TILE
    ar_set_error("GEMM f32: no tile for %d x %d", p.M, p.N);
    return AR_HIP_ERR_INVALID;
}

}  // namespace

// k-slices of a residual product whose partials the next RMSNorm folds: as many as fill the CUs with 32-row
// (from 512 rows 64-row) x 64 tiles.  The launch then takes the tile for the slices.
int gemm_f32_ksplit(int M, int N, int K, int cus) {
    const int bm = M >= 512 ? 64 : 32;
    const long long tiles = (long long)((M + bm - 1) / bm) * (N / 64);
    int s = 1;
    while (s < 8 && tiles * s * 2 <= cus && K % (256 * s * 2) == 0) s *= 2;
    return s;
}

int launch_gemm_f32(const GemmF32Launch& a, hipStream_t stream) {
    AR_CHECK_ARG(a.A && a.W && a.C, "GEMM f32: null operand");
    AR_CHECK_ARG(a.M > 0 && a.N > 0 && a.K > 0, "GEMM f32: empty shape");
    AR_CHECK_ARG(a.N % 64 == 0, "GEMM f32: N=%d must be a multiple of 64", a.N);
    AR_CHECK_ARG(a.ksplit >= 1 && a.K % (BK * a.ksplit) == 0, "GEMM f32: K=%d must be a multiple of %d", a.K,
                 BK * a.ksplit);
    AR_CHECK_ARG(a.ksplit == 1 || a.epilogue == GEMV_EPI_STORE, "GEMM f32: k-slices need the store epilogue");
    AR_CHECK_ARG(a.lda >= a.K && a.ldw >= a.K && a.ldc >= a.N && a.lda % 4 == 0 && a.ldw % 4 == 0,
                 "GEMM f32: bad leading dims");
    AR_CHECK_ARG((reinterpret_cast<uintptr_t>(a.A) & 15) == 0 && (reinterpret_cast<uintptr_t>(a.W) & 15) == 0 &&
                     (!a.W2 || (reinterpret_cast<uintptr_t>(a.W2) & 15) == 0),
                 "GEMM f32: operands must be 16-byte aligned");
    Params p;
    p.A = a.A; p.W = a.W; p.W2 = a.W2; p.bias = a.bias; p.C = a.C;
    p.M = a.M; p.N = a.N; p.K = a.K; p.lda = a.lda; p.ldw = a.ldw; p.ldc = a.ldc; p.ksplit = a.ksplit;
    const int cus = ar_device_cus(stream);
    switch (a.epilogue) {
        case GEMV_EPI_STORE: return launch_epi<GEMV_EPI_STORE>(p, stream, cus);
        case GEMV_EPI_RESIDUAL: return launch_epi<GEMV_EPI_RESIDUAL>(p, stream, cus);
        case GEMV_EPI_SWIGLU:
            AR_CHECK_ARG(a.W2, "GEMM f32: SwiGLU needs W2");
            return launch_epi<GEMV_EPI_SWIGLU>(p, stream, cus);
    }
    ar_set_error("GEMM f32: unsupported epilogue %d", a.epilogue);
    return AR_HIP_ERR_INVALID;
}
