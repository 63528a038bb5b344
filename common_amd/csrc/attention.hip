// Decode-step grouped-query attention with the QK-norm / RoPE / KV-cache-write prologue fused in.
//
// One launch covers what the reference builds as a chain of graph ops per layer
// (engine/ml/.../AttentionFeatures.java:785-929):
//   QK-norm        rmsnorm over the whole q / k vector (:840-845, :886-891) or per head
//   split-half RoPE reshapeToSplitHalfRope + ropeRotation + reshapeFromSplitHalfRope
//                  (:195-237; RotationFeatures.java:124-208), angles pos * exp(f * -2 ln(theta)/hd)
//                  evaluated in double
//   cache write    k, v at row pos (:858-864, :871-877; CollectionReceptor.java:95-105)
//   scores         q . K[t] / sqrt(hd) (attentionKeysStandard :531-559)
//   causal mask    rows t > pos are never visited; the reference adds -10000 there (:906-917),
//                  whose exp underflows to exactly 0, so skipping them is identical
//   softmax        max-subtracted (ActivationFeatures.java:135-143), computed online per split
//   values         sum_t a[t] V[t] (attentionValuesStandard :572-616)
//
// Layout: caches are compact and head-major, (batch, kv_heads, max_seq, hd) fp32; query head h
// reads KV head h / (heads / kv_heads), which holds exactly what the reference's GQA-expanded
// cache copy (:823-826) holds.
//
// Grid (max_splits, kv_heads, batch), 256 threads.  The live context [0, pos] is cut into
// nsplit contiguous splits of >= 16 rows (at most max_splits); block (s, g, b) handles split s
// for the heads/kv_heads query heads sharing KV head g:
// Each 16-lane group streams its own rows of the split (K and V row read once, for all heads of
// the group) in chunks of 4 rows with an online softmax, the next chunk's loads in flight while the
// current one is used; the groups' (max, sum, accumulator) states are merged by shuffles within a
// wavefront and through LDS across wavefronts.
// With one split the block writes the normalised output; otherwise it writes unnormalised
// partials (o, max, sum) that attn_combine_kernel merges in the next launch (the kernel boundary
// makes them visible, so no block needs a device-wide fence).
#include <type_traits>

#include "ar_hip_internal.h"

namespace {

constexpr int kThreads = 256;   // threads of the split (multi-block) form
constexpr int kMaxTile = 348;   // rows per split in that form (fp32 cache; C5, 8 x 8 KV heads x 8256
                                // rows: 24 splits of 344 rows 106.8 us/layer vs 33 of 251 rows 110.6,
                                // 20 of 413 rows 109.7, 16 of 516 rows 118.3)
constexpr int kMaxTile16 = 1040; // fp16 cache: the per-row work (fp16 -> fp32 conversions) makes
                                 // longer splits pay (C5, 8 x 8 KV heads x 8256 rows: 8 splits of
                                 // 1032 rows 5.55 ms/step vs 33 of 251 rows 6.32)
constexpr int kShortMax = 256;  // caches up to this many rows: one block per (sequence, KV head)
constexpr int kMaxSplits = 1024;

struct AttnParams {
    const float* q;        // [batch][stride]: this step's raw q, k, v (k and v may live elsewhere)
    const float* k;
    const float* v;
    int qkv_stride;
    const float* q_norm;
    const float* k_norm;
    float qk_eps;
    int per_head_norm;
    void* kcache;          // fp32, or fp16 for the KV16 instantiation
    void* vcache;
    int max_seq;
    const int* pos;        // device position, or null: pos_value
    int pos_value;
    int heads, kv_heads;
    double rope_c;  // -2 ln(theta) / hd
    const float2* rope_tab;  // [max_seq][hd/2] (cos, sin) or null
    int max_splits;
    float* part_o;
    float* part_ml;
    float* out;
    int out_stride;
    uint16_t* out_hi;  // bf16 operand planes of out for the next GEMV, or null
    uint16_t* out_lo;
};


// (cos, sin) of pos * exp(f * -2 ln(theta) / hd): from the table the model precomputes in
// double on the host, or evaluated here in double when no table is given.
__device__ inline void rope_cs(const float2* row, int pos, int f, double c, float* cs, float* sn) {
    if (row) {
        const float2 t = row[f];
        *cs = t.x;
        *sn = t.y;
        return;
    }
    const double invf = exp((double)f * c);
    const double ang = (double)pos * invf;
    *cs = (float)cos(ang);
    *sn = (float)sin(ang);
}

// NT threads: 256 when the context is cut into splits across blocks, 512 for a context of at most
// kShortMax rows handled by one block per (sequence, KV head) with no combine launch.  KV16: the
// cache holds fp16 rows (the new row is rounded before it is used, so every step sees exactly the
// values the cache holds).  TAB: the rotation angles come from the (cos, sin) table, else they
// are evaluated in double.  RU0: K/V rows per 16-lane group per chunk.
template <int HD, int G, int NT, bool KV16, bool TAB, int RU0>
__global__ __launch_bounds__(NT) void attn_decode_kernel(AttnParams p) {
    using KVT = typename std::conditional<KV16, _Float16, float>::type;
    constexpr int FD = HD / 2;
    constexpr int EPL = HD / 16;     // dims per lane: a 16-lane group holds one row; fp32 rows: lane gl
                                     // holds dims 64*(e/4) + 4*gl + e%4 (each 16-byte load of the group
                                     // covers 256 contiguous bytes); fp16 rows: dims EPL*gl + e (one
                                     // load per row)
    constexpr int NGR = NT / 16;     // 16-lane row groups
    constexpr int NWV = NT / 64;     // wavefronts
    // rows per group per chunk: RU0, chosen from the longest split (a chunk of NGR * RU rows covers
    // it; 16-row splits take one row per group, no clamped duplicate loads); at most 2 for G >= 8,
    // and for G >= 4 with fp32 rows (registers: G query fragments; the G = 4 fp32 instance holds 192
    // VGPRs at RU 4, two wavefronts per SIMD, and 136 at RU 2, three)
    constexpr int RU = ((G >= 8 || (G >= 4 && !KV16)) && RU0 > 2) ? 2 : RU0;
    __shared__ __attribute__((aligned(16))) float q_s[G][HD];
    __shared__ __attribute__((aligned(16))) float k_new[HD];
    __shared__ __attribute__((aligned(16))) float v_new[HD];
    __shared__ __attribute__((aligned(16))) float red_acc[NWV][G][HD];
    __shared__ float red_m[NWV][G], red_l[NWV][G];
    __shared__ float2 sq_s[NWV];
    __shared__ float rq_s[G], rk_s;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = tid >> 4, gl = tid & 15;
    const int b = blockIdx.z, kvh = blockIdx.y, split = blockIdx.x;
    const int heads = p.heads, kvH = p.kv_heads;
    const int q_dim = heads * HD, kv_dim = kvH * HD;
    const float* q_raw = p.q + (size_t)b * p.qkv_stride;
    const float* k_raw = p.k + (size_t)b * p.qkv_stride;
    const float* v_raw = p.v + (size_t)b * p.qkv_stride;
    const bool whole_norm = (p.q_norm || p.k_norm) && !p.per_head_norm;

    // ---- every load that does not depend on the position, issued together with it ----------
    const int pos = p.pos ? *p.pos : p.pos_value;
    constexpr int QPT = (G * FD + NT - 1) / NT;  // query (f, f+hd/2) pairs per thread
    float qx1[QPT], qx2[QPT], qg1[QPT], qg2[QPT];
#pragma unroll
    for (int j = 0; j < QPT; j++) {
        const int idx = min(tid + j * NT, G * FD - 1);
        const int g = idx / FD, f = idx - g * FD;
        const size_t off = (size_t)(kvh * G + g) * HD + f;
        qx1[j] = q_raw[off];
        qx2[j] = q_raw[off + FD];
        qg1[j] = p.q_norm ? p.q_norm[off] : 1.f;
        qg2[j] = p.q_norm ? p.q_norm[off + FD] : 1.f;
    }
    const int kf = min(tid, FD - 1);
    const float kx1 = k_raw[(size_t)kvh * HD + kf], kx2 = k_raw[(size_t)kvh * HD + kf + FD];
    const float kg1 = p.k_norm ? p.k_norm[(size_t)kvh * HD + kf] : 1.f;
    const float kg2 = p.k_norm ? p.k_norm[(size_t)kvh * HD + kf + FD] : 1.f;
    const float vnew = v_raw[(size_t)kvh * HD + min(tid, HD - 1)];
    // whole-vector QK-norm: this thread's float4 slices of q and k, held in registers (straight-line
    // loads, so no wait is needed before the position-dependent loads below are issued); vectors
    // longer than the register slices are finished by a loop after those loads
    constexpr int SQQ = (8192 / (NT * 4)) > 0 ? 8192 / (NT * 4) : 1;
    constexpr int SQK = (2048 / (NT * 4)) > 0 ? 2048 / (NT * 4) : 1;
    float4 wq[SQQ], wk[SQK];
    if (whole_norm) {
#pragma unroll
        for (int j = 0; j < SQQ; j++) {
            const int i = (tid + j * NT) * 4;
            wq[j] = i < q_dim ? *reinterpret_cast<const float4*>(q_raw + i) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int j = 0; j < SQK; j++) {
            const int i = (tid + j * NT) * 4;
            wk[j] = i < kv_dim ? *reinterpret_cast<const float4*>(k_raw + i) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }

    if (pos < 0 || pos >= p.max_seq) return;
    const int n = pos + 1;
    int nsplit, tile;
    attn_split_plan(n, p.max_splits, &nsplit, &tile);
    if (split >= nsplit) return;
    const int t0 = split * tile;
    const int t1 = min(t0 + tile, n);
    const size_t head_base = ((size_t)b * kvH + kvh) * (size_t)p.max_seq * HD;
    KVT* kc = reinterpret_cast<KVT*>(p.kcache) + head_base;
    KVT* vc = reinterpret_cast<KVT*>(p.vcache) + head_base;
    auto dim_of = [&](int e) { return KV16 ? EPL * gl + e : 16 * (e & ~3) + gl * 4 + (e & 3); };

    // ---- rows of the split: group `grp` takes rows t0 + grp + NGR*i (neighbouring groups read
    // neighbouring rows), chunk c = rows i in [c*RU, c*RU + RU).  The rotation row and the first
    // chunk's K and V rows are issued as soon as the position is known, before anything waits for
    // the loads above (loads complete in issue order: the rotation is needed first).  Rows are clamped to the split (their scores are masked below); row `pos` is
    // stale in the cache until this block writes it, so that row is taken from LDS instead.
    float kr[RU][EPL], vr[RU][EPL];
    auto load_rows = [&](float (&dst)[RU][EPL], const KVT* src, int c) {
#pragma unroll
        for (int j = 0; j < RU; j++) {
            const int t = min(t0 + grp + NGR * (c * RU + j), t1 - 1);
            if constexpr (KV16) {
                typedef _Float16 halfv __attribute__((ext_vector_type(EPL)));
                const halfv v = *reinterpret_cast<const halfv*>(src + (size_t)t * HD + EPL * gl);
#pragma unroll
                for (int e = 0; e < EPL; e++) dst[j][e] = (float)v[e];
            } else {
#pragma unroll
                for (int e = 0; e < EPL; e += 4) {
                    const float4 v = *reinterpret_cast<const float4*>(src + (size_t)t * HD + 16 * e + gl * 4);
                    dst[j][e] = v.x; dst[j][e + 1] = v.y; dst[j][e + 2] = v.z; dst[j][e + 3] = v.w;
                }
            }
        }
    };
    float2 qcs[QPT], kcs;
    if constexpr (TAB) {  // (cos, sin) row of the position from the table, ahead of the K/V rows
        const float2* rope_row = p.rope_tab + (size_t)pos * FD;
#pragma unroll
        for (int j = 0; j < QPT; j++) qcs[j] = rope_row[min(tid + j * NT, G * FD - 1) % FD];
        kcs = rope_row[kf];
    }
    load_rows(kr, kc, 0);
    load_rows(vr, vc, 0);
    if constexpr (!TAB) {
#pragma unroll
        for (int j = 0; j < QPT; j++) {
            const int idx = min(tid + j * NT, G * FD - 1);
            rope_cs(nullptr, pos, idx % FD, p.rope_c, &qcs[j].x, &qcs[j].y);
        }
        rope_cs(nullptr, pos, kf, p.rope_c, &kcs.x, &kcs.y);
    }

    // ---- QK-norm factors ----------------------------------------------------------
    float rq_w = 1.f, rk_w = 1.f;  // whole-vector factors (per-head factors go through LDS)
    if (p.q_norm || p.k_norm) {
        if (whole_norm) {
            float sq = 0.f, sk = 0.f;  // this thread's share of sum(q^2), sum(k^2), in index order
#pragma unroll
            for (int j = 0; j < SQQ; j++) sq += wq[j].x * wq[j].x + wq[j].y * wq[j].y + wq[j].z * wq[j].z + wq[j].w * wq[j].w;
            for (int i = (tid + SQQ * NT) * 4; i < q_dim; i += NT * 4) {
                const float4 v = *reinterpret_cast<const float4*>(q_raw + i);
                sq += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
            }
#pragma unroll
            for (int j = 0; j < SQK; j++) sk += wk[j].x * wk[j].x + wk[j].y * wk[j].y + wk[j].z * wk[j].z + wk[j].w * wk[j].w;
            for (int i = (tid + SQK * NT) * 4; i < kv_dim; i += NT * 4) {
                const float4 v = *reinterpret_cast<const float4*>(k_raw + i);
                sk += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
            }
            sq = wave_sum_lane63(sq);
            sk = wave_sum_lane63(sk);
            if (lane == 63) sq_s[wave] = make_float2(sq, sk);
            __syncthreads();
            float tq = 0.f, tk = 0.f;
#pragma unroll
            for (int w = 0; w < NWV; w++) {
                tq += sq_s[w].x;
                tk += sq_s[w].y;
            }
            rq_w = 1.0f / sqrtf(tq / (float)q_dim + p.qk_eps);
            rk_w = 1.0f / sqrtf(tk / (float)kv_dim + p.qk_eps);
        } else {
            // wave w reduces heads w, w+4, ...; the k head goes to the last slot
            for (int j = wave; j < G + 1; j += NWV) {
                const float* src = (j < G) ? q_raw + (size_t)(kvh * G + j) * HD : k_raw + (size_t)kvh * HD;
                float s = 0.f;
                for (int i = lane; i < HD; i += 64) s += src[i] * src[i];
                s = wave_sum_lane63(s);
                if (lane == 63) {
                    const float r = 1.0f / sqrtf(s / (float)HD + p.qk_eps);
                    if (j < G) rq_s[j] = r; else rk_s = r;
                }
            }
            __syncthreads();
        }
    }

    // ---- normalised, rotated queries of this group -> LDS ---------------------------
#pragma unroll
    for (int j = 0; j < QPT; j++) {
        const int idx = tid + j * NT;
        if (idx < G * FD) {
            const int g = idx / FD, f = idx - g * FD;
            float x1 = qx1[j], x2 = qx2[j];
            if (p.q_norm) {
                const float r = whole_norm ? rq_w : rq_s[g];
                x1 = (qg1[j] * x1) * r;
                x2 = (qg2[j] * x2) * r;
            }
            q_s[g][f] = x1 * qcs[j].x - x2 * qcs[j].y;
            q_s[g][f + FD] = x2 * qcs[j].x + x1 * qcs[j].y;
        }
    }
    // ---- the split holding `pos` writes this step's k and v rows (cache + LDS) ---------
    const bool has_pos = pos >= t0 && pos < t1;
    if (has_pos) {
        if (tid < FD) {
            float x1 = kx1, x2 = kx2;
            if (p.k_norm) {
                const float r = whole_norm ? rk_w : rk_s;
                x1 = (kg1 * x1) * r;
                x2 = (kg2 * x2) * r;
            }
            const KVT o1 = (KVT)(x1 * kcs.x - x2 * kcs.y), o2 = (KVT)(x2 * kcs.x + x1 * kcs.y);
            k_new[tid] = (float)o1;
            k_new[tid + FD] = (float)o2;
            kc[(size_t)pos * HD + tid] = o1;
            kc[(size_t)pos * HD + tid + FD] = o2;
        }
        if (tid < HD) {
            const KVT vv = (KVT)vnew;
            v_new[tid] = (float)vv;
            vc[(size_t)pos * HD + tid] = vv;
        }
    }
    __syncthreads();

    // ---- one pass over K and V: online softmax per group, chunk by chunk ---------------
    // Scores are kept in base 2: the query fragment is pre-multiplied by log2(e)/sqrt(hd), so
    // exp(s - m) = exp2(s2 - m2) and the hardware exp2 serves every weight; m2 converts back to
    // natural-log units for the split partials.
    const float c2 = 1.4426950408889634f / sqrtf((float)HD);
    float qf[G][EPL];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int e = 0; e < EPL; e += 4) {
            const float4 t = *reinterpret_cast<const float4*>(&q_s[g][dim_of(e)]);
            qf[g][e] = t.x * c2; qf[g][e + 1] = t.y * c2; qf[g][e + 2] = t.z * c2; qf[g][e + 3] = t.w * c2;
        }
    float m[G], l[G], acc[G][EPL];
#pragma unroll
    for (int g = 0; g < G; g++) {
        m[g] = -INFINITY;
        l[g] = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; e++) acc[g][e] = 0.f;
    }
    const int nch = (t1 - t0 + NGR * RU - 1) / (NGR * RU);
    for (int c = 0; c < nch; c++) {
        if (has_pos) {
            // row pos (and every clamped duplicate of it: pos is the split's last row) was loaded
            // stale from the cache; it takes this step's k and v, so a masked duplicate adds 0 * v
            // of a finite row even when the stale row holds an infinity or NaN
#pragma unroll
            for (int j = 0; j < RU; j++)
                if (min(t0 + grp + NGR * (c * RU + j), t1 - 1) == pos)
#pragma unroll
                    for (int e = 0; e < EPL; e++) {
                        kr[j][e] = k_new[dim_of(e)];
                        vr[j][e] = v_new[dim_of(e)];
                    }
        }
        // scores q . K[t] / sqrt(hd) of the chunk's rows (rows past the split: -inf)
        float sc[G][RU];
#pragma unroll
        for (int j = 0; j < RU; j++) {
            const bool valid = t0 + grp + NGR * (c * RU + j) < t1;
#pragma unroll
            for (int g = 0; g < G; g++) {
                float d = 0.f;
#pragma unroll
                for (int e = 0; e < EPL; e++) d = fmaf(qf[g][e], kr[j][e], d);
                d = row16_sum(d);
                sc[g][j] = valid ? d : -INFINITY;
            }
        }
        if (c + 1 < nch) load_rows(kr, kc, c + 1);  // K of the next chunk, in flight from here
#pragma unroll
        for (int g = 0; g < G; g++) {
            float mc = sc[g][0];
#pragma unroll
            for (int j = 1; j < RU; j++) mc = fmaxf(mc, sc[g][j]);
            const float mn = fmaxf(m[g], mc);
            if (mn == -INFINITY) continue;  // nothing valid yet for this group
            const float alpha = (m[g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[g] - mn);
            l[g] *= alpha;
#pragma unroll
            for (int e = 0; e < EPL; e++) acc[g][e] *= alpha;
#pragma unroll
            for (int j = 0; j < RU; j++) {
                const float pj = __builtin_amdgcn_exp2f(sc[g][j] - mn);  // masked: exp2(-inf) = 0
                l[g] += pj;
#pragma unroll
                for (int e = 0; e < EPL; e++) acc[g][e] = fmaf(pj, vr[j][e], acc[g][e]);
            }
            m[g] = mn;
        }
        if (c + 1 < nch) load_rows(vr, vc, c + 1);  // V of the next chunk
    }

    // ---- merge the groups: the four of a wavefront by lane swaps, the wavefronts through LDS ---
    auto merge_with = [&](auto partner) {
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float mo = partner(m[g]), lo = partner(l[g]);
            const float mn = fmaxf(m[g], mo);
            const float a = (m[g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[g] - mn);
            const float bo = (mo == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mo - mn);
            l[g] = l[g] * a + lo * bo;
#pragma unroll
            for (int e = 0; e < EPL; e++) {
                const float ao = partner(acc[g][e]);
                acc[g][e] = acc[g][e] * a + ao * bo;
            }
            m[g] = mn;
        }
    };
    merge_with([&](float v) { return xor16(v, lane); });
    merge_with([&](float v) { return xor32(v, lane); });
    if (lane < 16) {
#pragma unroll
        for (int g = 0; g < G; g++) {
#pragma unroll
            for (int e = 0; e < EPL; e++) red_acc[wave][g][dim_of(e)] = acc[g][e];
            if (lane == 0) {
                red_m[wave][g] = m[g];
                red_l[wave][g] = l[g];
            }
        }
    }
    __syncthreads();

    const int hbase = kvh * G;
    for (int idx = tid; idx < G * HD; idx += NT) {
        const int g = idx / HD, i = idx - g * HD;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NWV; w++) M = fmaxf(M, red_m[w][g]);
        float L = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < NWV; w++) {
            const float wt = (red_m[w][g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(red_m[w][g] - M);
            L = fmaf(red_l[w][g], wt, L);
            o = fmaf(red_acc[w][g][i], wt, o);
        }
        if (nsplit == 1) {
            const size_t oi = (size_t)b * p.out_stride + (size_t)(hbase + g) * HD + i;
            p.out[oi] = o / L;
            if (p.out_hi) bf16_planes(o / L, p.out_hi + oi, p.out_lo + oi);
        } else {
            const size_t slot = ((size_t)b * heads + hbase + g) * p.max_splits + split;
            p.part_o[slot * HD + i] = o;
            if (i == 0) {
                p.part_ml[slot * 2] = M * 0.6931471805599453f;  // back to natural-log units
                p.part_ml[slot * 2 + 1] = L;
            }
        }
    }
}

// Merges the split partials of every query head: o = sum_s e^(m_s - M) o_s / sum_s e^(m_s - M) l_s.
// NG groups of HD threads take every NGth split.  Every load that does not depend on the position (a
// thread's first kMergeRegs partial outputs and its (m, l) pair) is issued together with the position
// load, so the merge costs one memory round trip; splits past NG * kMergeRegs are read afterwards.
// One group covers 32 splits; above that four do (96 splits x 32 heads: 4.8 us, 7.3 with one group, whose
// loads past the 32nd wait one after another).
template <int HD, int NG>
__global__ __launch_bounds__(HD * NG) void attn_combine_kernel(AttnParams p) {
    constexpr int kMergeRegs = 32, NT = HD * NG;
    __shared__ float w_s[kMaxSplits];
    __shared__ float red[NT / 64];
    __shared__ float og[NG > 1 ? (NG - 1) * HD : 1];
    const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x, i = NG == 1 ? t : t % HD,
              grp = NG == 1 ? 0 : __builtin_amdgcn_readfirstlane(t / HD);
    const int lane = t & 63, wave = t >> 6;
    const size_t slot0 = ((size_t)b * p.heads + h) * p.max_splits;
    float ov[kMergeRegs];
#pragma unroll
    for (int s = 0; s < kMergeRegs; s++)
        ov[s] = grp + NG * s < p.max_splits ? p.part_o[(slot0 + grp + NG * s) * HD + i] : 0.f;
    const float2 ml = t < p.max_splits ? reinterpret_cast<const float2*>(p.part_ml)[slot0 + t]
                                       : make_float2(-INFINITY, 0.f);
    const int pos = p.pos ? *p.pos : p.pos_value;
    if (pos < 0 || pos >= p.max_seq) return;
    int nsplit, tile;
    attn_split_plan(pos + 1, p.max_splits, &nsplit, &tile);
    if (nsplit == 1) return;  // the attention kernel wrote the output itself
    float m_loc = t < nsplit ? ml.x : -INFINITY;
    for (int s = t + NT; s < nsplit; s += NT) m_loc = fmaxf(m_loc, p.part_ml[(slot0 + s) * 2]);
    m_loc = wave_max_lane63(m_loc);
    if (lane == 63) red[wave] = m_loc;
    __syncthreads();
    float M = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) M = fmaxf(M, red[w]);
    float l_loc = 0.f;
    if (t < nsplit) {
        const float w = expf(ml.x - M);
        w_s[t] = w;
        l_loc = fmaf(ml.y, w, l_loc);
    }
    for (int s = t + NT; s < nsplit; s += NT) {
        const float w = expf(p.part_ml[(slot0 + s) * 2] - M);
        w_s[s] = w;
        l_loc = fmaf(p.part_ml[(slot0 + s) * 2 + 1], w, l_loc);
    }
    l_loc = wave_sum_lane63(l_loc);
    __syncthreads();
    if (lane == 63) red[wave] = l_loc;
    __syncthreads();
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < NT / 64; w++) L += red[w];
    float O = 0.f;
#pragma unroll
    for (int s = 0; s < kMergeRegs; s++)
        if (grp + NG * s < nsplit) O = fmaf(ov[s], w_s[grp + NG * s], O);
    for (int s = grp + NG * kMergeRegs; s < nsplit; s += NG) O = fmaf(p.part_o[(slot0 + s) * HD + i], w_s[s], O);
    if constexpr (NG > 1) {
        if (grp > 0) og[(grp - 1) * HD + i] = O;
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 0; g < NG - 1; g++) O += og[g * HD + i];
    }
    const size_t oi = (size_t)b * p.out_stride + (size_t)h * HD + i;
    p.out[oi] = O / L;
    if (p.out_hi) bf16_planes(O / L, p.out_hi + oi, p.out_lo + oi);
}

template <int HD, int G, bool KV16>
int launch_t(const AttnLaunch& a, hipStream_t stream) {
    AttnParams p;
    p.q = a.qkv ? a.qkv : a.q;
    p.k = a.qkv ? a.qkv + (size_t)a.heads * a.head_dim : a.k;
    p.v = a.qkv ? a.qkv + (size_t)(a.heads + a.kv_heads) * a.head_dim : a.v;
    p.qkv_stride = a.qkv_stride; p.q_norm = a.q_norm; p.k_norm = a.k_norm;
    p.qk_eps = a.qk_eps; p.per_head_norm = a.per_head_norm; p.kcache = a.kcache; p.vcache = a.vcache;
    p.max_seq = a.max_seq; p.pos = a.pos; p.pos_value = a.pos_value; p.heads = a.heads; p.kv_heads = a.kv_heads;
    p.rope_c = -2.0 * log(a.rope_theta) / (double)HD;
    p.rope_tab = a.rope_tab;
    p.max_splits = a.max_splits; p.part_o = a.part_o; p.part_ml = a.part_ml;
    p.out = a.out; p.out_stride = a.out_stride; p.out_hi = a.out_hi; p.out_lo = a.out_lo;
    if (a.max_splits == 1 && a.max_seq <= kShortMax) {
        // whole context in one block
        constexpr int NT = 512;
        const dim3 grid(1, a.kv_heads, a.batch);
        if (p.rope_tab) ar_launch((attn_decode_kernel<HD, G, NT, KV16, true, 4>), grid, dim3(NT), 0, stream, p);
        else ar_launch((attn_decode_kernel<HD, G, NT, KV16, false, 4>), grid, dim3(NT), 0, stream, p);
        AR_LAUNCH_CHECK();
        return AR_HIP_OK;
    }
    const dim3 grid(a.max_splits, a.kv_heads, a.batch);
    // longest split of this launch: of the live context when the position is given, else of any
    // position the cache holds (attn_split_plan: splits of <= 16 rows until max_splits are in use)
    int longest;
    if (a.pos) {
        longest = (a.max_seq + a.max_splits - 1) / a.max_splits;
        if (longest < kAttnMinTile) longest = kAttnMinTile;
    } else {
        int ns;
        attn_split_plan(a.pos_value + 1, a.max_splits, &ns, &longest);
    }
    constexpr int NGR = kThreads / 16;
    if (p.rope_tab && longest <= NGR)
        ar_launch((attn_decode_kernel<HD, G, kThreads, KV16, true, 1>), grid, dim3(kThreads), 0, stream, p);
    else if (p.rope_tab && longest <= 2 * NGR)
        ar_launch((attn_decode_kernel<HD, G, kThreads, KV16, true, 2>), grid, dim3(kThreads), 0, stream, p);
    else if (p.rope_tab)
        ar_launch((attn_decode_kernel<HD, G, kThreads, KV16, true, 4>), grid, dim3(kThreads), 0, stream, p);
    else
        ar_launch((attn_decode_kernel<HD, G, kThreads, KV16, false, 4>), grid, dim3(kThreads), 0, stream, p);
    AR_LAUNCH_CHECK();
    if (a.max_splits > 1) {
        if (a.max_splits > 32)
            ar_launch((attn_combine_kernel<HD, 4>), dim3(a.heads, a.batch), dim3(4 * HD), 0, stream, p);
        else
            ar_launch((attn_combine_kernel<HD, 1>), dim3(a.heads, a.batch), dim3(HD), 0, stream, p);
        AR_LAUNCH_CHECK();
    }
    return AR_HIP_OK;
}

template <int HD, bool KV16>
int pick_g(const AttnLaunch& a, hipStream_t s) {
    switch (a.heads / a.kv_heads) {
        case 1: return launch_t<HD, 1, KV16>(a, s);
        case 2: return launch_t<HD, 2, KV16>(a, s);
        case 4: return launch_t<HD, 4, KV16>(a, s);
        case 8: return launch_t<HD, 8, KV16>(a, s);
    }
    ar_set_error("attention: heads/kv_heads = %d not in {1,2,4,8}", a.heads / a.kv_heads);
    return AR_HIP_ERR_INVALID;
}

// Causal attention of prompt rows in fp32, the attention of the fp32-weight prefill: row t of
// sequence b attends cache rows 0..p0+t of its KV head, fp32 products and sums throughout
// (v_mfma_f32_32x32x2_f32), online softmax in base 2 with the queries pre-scaled by
// log2(e)/sqrt(hd).  The cache rows of the prompt are written beforehand (qk_prep).
// q32: [B*T][heads*hd] normalised, rotated queries; caches fp32 [B][KV][S][hd]; out: [B*T][heads*hd].
//
// Bound by the fp32 matrix rate: a 32-key x 32-query tile is hd MFMA instructions of 64 cycles
// (hd 128: 8,192 cycles) against 32 KB of K and V, so the rows go straight from the caches into
// registers and nothing but the queries needs LDS.  One block of four wavefronts takes 32 query rows
// of one head; wavefront s takes key tiles s, s+4, ... (a causal block's work grows with its last
// row: quarter-length chains in blocks taken heaviest first fill the CUs evenly, two blocks per CU),
// and the four partial softmax states meet in LDS at the end, each wavefront folding a quarter of
// the outputs.  Both products are computed transposed, so a lane owns one query (lanes l and l^32
// hold the two halves of its scores) and the weights P feed the second product from the registers
// the first one left them in:
//   S^T (32 keys x 32 queries) = K . Q^T   contraction step (q, c): d = 8q + 4(l/32) + c, so a lane
//                                          reads its key row and its query row 16 bytes at a time
//   O^T (hd x 32 queries)     += V^T . P^T contraction step r: key (r/4)*8 + (l/32)*4 + r%4 (the
//                                          result layout of S^T); output row i of tile j is dim
//                                          NT*i + j, so one load per key row feeds every tile
// K and V of the wavefront's next tile are loaded half a tile at a time, as the registers of the one in use
// come free.  A score is added up in chains of 16 dims and an output in chains of 8 keys, each chain in one
// of two accumulators of its own and added to the sum by the vector units while the next one runs: one
// accumulator for a whole sum (128 dims, a quarter of the keys) was 1.5 to 1.9 times as far from 64 bits as
// this and as the vector form (3.1e-7, 1.9e-7 and 1.8e-7 at 100 rows), for 98 instead of 109 us.
// 0.6B shape (16 heads, 8 KV heads, hd 128), 1,531 rows: 109 us (88 TFLOP/s of the causal half; MFMA busy
// 53%, the rest is the uneven end of the causal blocks and each block's start and merge) against
// 382 us for one block per (row, KV head) on the vector units, where each row reads its whole context; 128
// rows 11.1 against 11.4 us.
struct PrefillAttnF32 {
    const float *q32, *kcache, *vcache;
    float* out;
    int T, p0, S, heads, kv_heads, pairs, nq;  // pairs: B * kv_heads; nq: query tiles of 32 rows
};

template <int HD>
__global__ __launch_bounds__(256, 2) void attn_prefill_f32_kernel(PrefillAttnF32 p) {
    typedef float floatx16 __attribute__((ext_vector_type(16)));
    constexpr int KS = 4, NT = HD / 32;
    constexpr int QC = 2, PC = 4;  // chains: 8 * QC dims of a score, 2 * PC keys of an output
    typedef float vrow __attribute__((ext_vector_type(NT)));
    constexpr int QROW = HD + 4;        // query row stride: conflict-free 16-byte reads
    constexpr int STATE = NT * 16 + 2;  // O^T, max and sum of a lane
    constexpr int LDS_FLOATS = KS * STATE * 64 > 32 * QROW ? KS * STATE * 64 : 32 * QROW;
    __shared__ __attribute__((aligned(16))) float lds[LDS_FLOATS];

    const int tid = threadIdx.x, lane = tid & 63, h2 = lane >> 5, lq = lane & 31;
    const int slice = __builtin_amdgcn_readfirstlane(tid >> 6);
    // block -> (head, query tile), heaviest tiles first; the heads of one (sequence, KV head) on one
    // XCD where the pair count allows, so its K and V stay in that XCD's L2
    const int G = p.heads / p.kv_heads, units = p.pairs * G;
    int pair, sub, qrank;
    if (p.pairs % 8 == 0) {
        const int slot = blockIdx.x >> 3, per = units >> 3, u = slot % per;
        pair = (blockIdx.x & 7) + 8 * (u / G);
        sub = u % G;
        qrank = slot / per;
    } else {
        const int u = blockIdx.x % units;
        pair = u / G;
        sub = u % G;
        qrank = blockIdx.x / units;
    }
    const int b = pair / p.kv_heads, head = (pair - b * p.kv_heads) * G + sub;
    const int row0 = (p.nq - 1 - qrank) * 32, myq = row0 + lq;
    const float* kc = p.kcache + (size_t)pair * p.S * HD;
    const float* vc = p.vcache + (size_t)pair * p.S * HD;
    const int kend = p.p0 + min(row0 + 32, p.T);  // keys the block needs: 0 .. kend-1
    const int ntiles = (kend + 31) / 32;

    float4 kf[HD / 8];
    vrow vf[16];
    // half a tile at a time (a half's registers come free in the middle of the product that uses the tile)
    auto load_k = [&](int t, int half) __attribute__((always_inline)) {
        const unsigned at = (unsigned)min(32 * t + lq, kend - 1) * HD + 4 * h2;  // (32-bit: scalar base + offset)
#pragma unroll
        for (int q = HD / 16 * half; q < HD / 16 * (half + 1); q++)
            kf[q] = *reinterpret_cast<const float4*>(kc + at + 8 * q);
    };
    auto load_v = [&](int t, int half) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 8 * half; r < 8 * half + 8; r++) {
            const unsigned key = min(32 * t + (r >> 2) * 8 + h2 * 4 + (r & 3), kend - 1);
            vf[r] = *reinterpret_cast<const vrow*>(vc + key * HD + NT * lq);
        }
    };
    // (past the wavefront's last tile the loads re-read the last key row: no branch around them, so the
    // waits count exactly the loads they need)
    const float c2 = 1.4426950408889634f / sqrtf((float)HD);
    constexpr int QL = 32 * HD / 4 / 256;  // 16-byte query loads per thread, issued ahead of K and V
    float4 qr[QL];
#pragma unroll
    for (int i = 0; i < QL; i++) {
        const int r = (tid + 256 * i) / (HD / 4), c = tid % (HD / 4), t = min(row0 + r, p.T - 1);
        qr[i] = *reinterpret_cast<const float4*>(p.q32 + ((size_t)b * p.T + t) * p.heads * HD + (size_t)head * HD + 4 * c);
    }
    load_k(slice, 0);
    load_k(slice, 1);
    load_v(slice, 0);
#pragma unroll
    for (int i = 0; i < QL; i++) {
        const int r = (tid + 256 * i) / (HD / 4), c = tid % (HD / 4);
        *reinterpret_cast<float4*>(&lds[r * QROW + 4 * c]) =
            make_float4(qr[i].x * c2, qr[i].y * c2, qr[i].z * c2, qr[i].w * c2);
    }
    // a barrier over LDS only: K and V stay in flight across it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    floatx16 o[NT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[j][r] = 0.f;
    float m = -INFINITY, l = 0.f;
    for (int t = slice; t < ntiles; t += KS) {
        floatx16 s, c[2];
        // (the query values of a step are read one step ahead and no further: registers)
        const float* const qrow = &lds[lq * QROW + 4 * h2];
        float4 qv = *reinterpret_cast<const float4*>(qrow);
#pragma unroll
        for (int q = 0; q < HD / 8; q++) {
            float4 qn = qv;
            if (q + 1 < HD / 8) qn = *reinterpret_cast<const float4*>(qrow + 8 * (q + 1));
            floatx16& x = c[q / QC & 1];
            if (q % QC == 0)
#pragma unroll
                for (int r = 0; r < 16; r++) x[r] = 0.f;
            __builtin_amdgcn_sched_barrier(0);
            x = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[q].x, qv.x, x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[q].y, qv.y, x, 0, 0, 0);
            if (q == QC) s = c[0];
            if (q > QC && q % QC == 0) s += c[(q / QC & 1) ^ 1];
            x = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[q].z, qv.z, x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[q].w, qv.w, x, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (q == HD / 16) load_v(t, 1);
            qv = qn;
        }
        s += c[(HD / 8 / QC - 1) & 1];
        load_k(t + KS, 0);
        const int k0 = 32 * t;
        if (k0 + 31 > p.p0 + row0) {  // tiles past the first row's own key (row0 + 31 >= T lies there too)
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (k0 + (r >> 2) * 8 + h2 * 4 + (r & 3) > min(p.p0 + myq, kend - 1)) s[r] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = max_xor32(mx);
        if (__ballot(mx > m)) {
            const float mn = fmaxf(m, mx);
            const float alpha = (m == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m - mn);
            l *= alpha;
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[j][r] *= alpha;
            m = mn;
        }
        // a query whose keys in this wavefront's tiles are all masked so far keeps m = -inf: weights 0
        const float mu = (m == -INFINITY) ? 0.f : m;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = __builtin_amdgcn_exp2f(s[r] - mu);
        float sum[8];
#pragma unroll
        for (int r = 0; r < 8; r++) sum[r] = s[r] + s[r + 8];
#pragma unroll
        for (int n = 4; n > 0; n /= 2)
#pragma unroll
            for (int r = 0; r < n; r++) sum[r] += sum[r + n];
        l += sum_xor32(sum[0]);
        constexpr int CHAINS = 16 / PC * NT;
#pragma unroll
        for (int n = 0; n < CHAINS; n++) {  // chain n: the keys of steps r0 .. r0 + PC - 1 into O^T tile j
            const int j = n % NT, r0 = n / NT * PC;
            floatx16& x = c[n & 1];
#pragma unroll
            for (int r = 0; r < 16; r++) x[r] = 0.f;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < PC; r++) {
                x = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[r0 + r][j], s[r0 + r], x, 0, 0, 0);
                if (r == PC / 2 - 1 && n > 0) o[(n - 1) % NT] += c[(n & 1) ^ 1];
            }
            __builtin_amdgcn_sched_barrier(0);
            if (n == CHAINS / 2) load_k(t + KS, 1);
        }
        o[NT - 1] += c[(CHAINS - 1) & 1];
        load_v(t + KS, 0);
    }

    __syncthreads();  // the queries are read: their LDS takes the states
    float* const st = lds + lane;  // [slice][value][lane]
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) st[(slice * STATE + j * 16 + r) * 64] = o[j][r];
    st[(slice * STATE + NT * 16) * 64] = m;
    st[(slice * STATE + NT * 16 + 1) * 64] = l;
    __syncthreads();
    if (myq >= p.T) return;
    // m is finite for slice 0 (key 0 is in its first tile); a slice without live keys keeps -inf
    float ms[KS], wgt[KS], M = -INFINITY, L = 0.f;
#pragma unroll
    for (int k = 0; k < KS; k++) {
        ms[k] = st[(k * STATE + NT * 16) * 64];
        M = fmaxf(M, ms[k]);
    }
#pragma unroll
    for (int k = 0; k < KS; k++) {
        wgt[k] = (ms[k] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(ms[k] - M);
        L = fmaf(st[(k * STATE + NT * 16 + 1) * 64], wgt[k], L);
    }
    float* orow = p.out + ((size_t)b * p.T + myq) * p.heads * HD + (size_t)head * HD;
#pragma unroll
    for (int i = 0; i < 4; i++) {  // result registers 4*slice + i: dims NT*(8*slice + 4*h2 + i) + j
        vrow v;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            float a = 0.f;
#pragma unroll
            for (int k = 0; k < KS; k++) a = fmaf(st[(k * STATE + j * 16 + 4 * slice + i) * 64], wgt[k], a);
            v[j] = a / L;
        }
        *reinterpret_cast<vrow*>(orow + NT * (8 * slice + 4 * h2 + i)) = v;
    }
}

}  // namespace

int launch_attention_prefill_f32(const float* q32, const float* kcache, const float* vcache, float* out, int B, int T,
                                 int p0, int S, int heads, int kv_heads, int hd, hipStream_t stream) {
    AR_CHECK_ARG(q32 && kcache && vcache && out && B > 0 && T > 0, "prefill attention: bad arguments");
    AR_CHECK_ARG(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "prefill attention: bad head counts");
    AR_CHECK_ARG(p0 >= 0 && p0 + T <= S, "prefill attention: rows %d..%d outside the %d-row cache", p0, p0 + T, S);
    AR_CHECK_ARG((long long)B * T <= 0x7fffffffLL && kv_heads <= 65535, "prefill attention: grid too large");
    const int G = heads / kv_heads;
    AR_CHECK_ARG(G == 1 || G == 2 || G == 4 || G == 8, "prefill attention: heads/kv_heads = %d not in {1,2,4,8}", G);
    PrefillAttnF32 p;
    p.q32 = q32; p.kcache = kcache; p.vcache = vcache; p.out = out; p.T = T; p.p0 = p0; p.S = S; p.heads = heads;
    p.kv_heads = kv_heads; p.pairs = B * kv_heads; p.nq = (T + 31) / 32;
    const long long blocks = (long long)p.pairs * G * p.nq;
    AR_CHECK_ARG(blocks <= 0x7fffffffLL, "prefill attention: grid too large");
    const dim3 grid((unsigned)blocks);
    if (hd == 128) {
        hipLaunchKernelGGL(attn_prefill_f32_kernel<128>, grid, dim3(256), 0, stream, p);
    } else if (hd == 64) {
        hipLaunchKernelGGL(attn_prefill_f32_kernel<64>, grid, dim3(256), 0, stream, p);
    } else {
        ar_set_error("prefill attention: head_dim %d not supported (64, 128)", hd);
        return AR_HIP_ERR_INVALID;
    }
    AR_LAUNCH_CHECK();
    return AR_HIP_OK;
}

size_t attention_partial_floats(int batch, int heads, int max_splits, int hd) {
    return (size_t)batch * heads * max_splits * (size_t)hd;
}

int attention_max_splits(int max_seq, int kv_heads, int batch, bool kv16) {
    if (max_seq <= kShortMax) return 1;  // one block per (sequence, KV head), no combine launch
    const int tmax = kv16 ? kMaxTile16 : kMaxTile;
    const int need = (max_seq + tmax - 1) / tmax;                // rows per split <= tmax
    // about one block per CU: each block then streams a tile long enough to amortise its prologue
    // (C2, 4097 rows: 32 splits of 129 rows; 128 splits of 33 rows measured 2.4x slower)
    const int want = (256 + kv_heads * batch - 1) / (kv_heads * batch);
    const int cap = (max_seq + kAttnMinTile - 1) / kAttnMinTile;  // splits of >= kAttnMinTile rows
    int s = want < cap ? want : cap;
    if (s < need) s = need;
    return s < 1 ? 1 : s;
}

// The splits of the stand-alone operator for a cache that needs more than one block per CU: whole blocks
// per CU (32 heads, 8 KV heads, 32,768 rows: 96 splits, three blocks per CU, 55.9 us against 58.5 with the
// 95 that cover the rows; 16,384 rows: 64, 33.8 against 36.0 with 48; the longest ways up, 12,000 and 23,000
// rows from 35 and 67 splits: 27.0 -> 23.2 and 39.6 -> 36.9).  A model keeps
// attention_max_splits, measured over its batches (kMaxTile).
int attention_whole_splits(int max_seq, int kv_heads, int cus) {
    const int s = attention_max_splits(max_seq, kv_heads, 1, false);
    const int cu = cus % kv_heads == 0 ? cus / kv_heads : 1;  // splits of one block per CU
    const int w = (s + cu - 1) / cu * cu;
    return s > cu && w <= kMaxSplits ? w : s;
}

int launch_attention_decode(const AttnLaunch& a, hipStream_t stream) {
    AR_CHECK_ARG((a.qkv || (a.q && a.k && a.v)) && a.kcache && a.vcache && a.out, "attention: null pointer");
    AR_CHECK_ARG(a.pos || (a.pos_value >= 0 && a.pos_value < a.max_seq), "attention: position %d outside %d rows",
                 a.pos_value, a.max_seq);
    AR_CHECK_ARG(a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0, "attention: bad head counts %d/%d",
                 a.heads, a.kv_heads);
    AR_CHECK_ARG(a.max_splits <= kMaxSplits, "attention: %d splits exceed %d", a.max_splits, kMaxSplits);
    const int tmax = a.kv16 ? kMaxTile16 : kMaxTile;
    AR_CHECK_ARG(a.max_splits >= 1 && ((long long)a.max_splits * tmax >= a.max_seq ||
                                       (a.max_splits == 1 && a.max_seq <= kShortMax)),
                 "attention: %d splits of at most %d rows do not cover %d rows", a.max_splits, tmax, a.max_seq);
    AR_CHECK_ARG(a.max_splits == 1 || (a.part_o && a.part_ml), "attention: missing split buffers");
    AR_CHECK_ARG(a.batch >= 1 && a.batch <= 65535, "attention: bad batch %d", a.batch);
    AR_CHECK_ARG((reinterpret_cast<uintptr_t>(a.kcache) & 15) == 0 && (reinterpret_cast<uintptr_t>(a.vcache) & 15) == 0,
                 "attention: caches must be 16-byte aligned");
    if (ar_check_ptrs_enabled()) {  // extents of the attention and combine kernels
        const char* k = "attention";
        const size_t hd = a.head_dim, qd = (size_t)a.heads * hd, kvd = (size_t)a.kv_heads * hd, B1 = a.batch - 1;
        const size_t elem = a.kv16 ? 2 : 4, cache = (size_t)a.batch * kvd * a.max_seq * elem;
        if (a.qkv) {
            AR_TRY(ar_check_range(a.qkv, (B1 * a.qkv_stride + qd + 2 * kvd) * 4, k, "q/k/v rows"));
        } else {
            AR_TRY(ar_check_range(a.q, (B1 * a.qkv_stride + qd) * 4, k, "q rows"));
            AR_TRY(ar_check_range(a.k, (B1 * a.qkv_stride + kvd) * 4, k, "k rows"));
            AR_TRY(ar_check_range(a.v, (B1 * a.qkv_stride + kvd) * 4, k, "v rows"));
        }
        AR_TRY(ar_check_range(a.q_norm, qd * 4, k, "q norm gain"));
        AR_TRY(ar_check_range(a.k_norm, kvd * 4, k, "k norm gain"));
        AR_TRY(ar_check_range(a.kcache, cache, k, "key cache"));
        AR_TRY(ar_check_range(a.vcache, cache, k, "value cache"));
        AR_TRY(ar_check_range(a.pos, 4, k, "position"));
        AR_TRY(ar_check_range(a.rope_tab, (size_t)a.max_seq * (hd / 2) * sizeof(float2), k, "RoPE table"));
        if (a.max_splits > 1) {
            AR_TRY(ar_check_range(a.part_o, attention_partial_floats(a.batch, a.heads, a.max_splits, a.head_dim) * 4,
                                  k, "split partials"));
            AR_TRY(ar_check_range(a.part_ml, (size_t)a.batch * a.heads * a.max_splits * 2 * 4, k, "split maxima / sums"));
        }
        AR_TRY(ar_check_range(a.out, (B1 * a.out_stride + qd) * 4, k, "output"));
        AR_TRY(ar_check_range(a.out_hi, (B1 * a.out_stride + qd) * 2, k, "output hi plane"));
        AR_TRY(ar_check_range(a.out_lo, (B1 * a.out_stride + qd) * 2, k, "output lo plane"));
    }
    if (a.head_dim == 128) return a.kv16 ? pick_g<128, true>(a, stream) : pick_g<128, false>(a, stream);
    if (a.head_dim == 64) return a.kv16 ? pick_g<64, true>(a, stream) : pick_g<64, false>(a, stream);
    ar_set_error("attention: head_dim %d not supported (64, 128)", a.head_dim);
    return AR_HIP_ERR_INVALID;
}
