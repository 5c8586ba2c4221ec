// attention.hip -- attention with a KV cache in HBM: decode steps (m H / KVH <= 16 new
// query rows a kv head) and prompt-length calls (any m; the tiled kernels further down).
//
// The cache's filled length is device state (the handle's `state`): the first kernel
// of a call reads it and publishes it for the second, which advances it by m.  So the
// kernels never take the length from the host, and a call captured into a HIP graph
// appends at a new position every replay.
//
// What it computes: LlamaAttention::forward_with_cache after the projections
// (crates/runtime/src/models_v2/llama.rs:1044-1150): RoPE on q and k at the
// positions len .. len + m - 1 (apply_rope_with_offset, llama.rs:827-883: the
// half-split rotation, inv_freq and angles in f32), k and v appended to the
// layer's cache (LayerKVCache::append, crates/runtime/src/kv_cache.rs:91-130),
// then softmax(q k^T / sqrt(hd) + causal mask) v for every head, head h reading
// kv head h / (H / KVH) (the reference expands k, v to all heads before
// caching; the cache here keeps the KVH heads, which is the same arithmetic).
// Bound: HBM -- the cached K and V are read once per step (2 KVH len hd 4 bytes,
// f32 like the reference's cache).
//
// Two kernels on the caller's stream.  attn_decode_kernel: a workgroup per (kv
// head g, chunk c of C positions), 256 threads:
//   1. the Q = m G queries of kv head g (the m tokens times the G = H / KVH heads
//      of the group): RoPE at position len + t, times 1 / sqrt(hd), into LDS;
//   2. the new positions len .. len + m - 1 inside this chunk: k rotated and v
//      into LDS, and appended to the cache (each position lies in exactly one
//      chunk, so exactly one workgroup writes it; the scores read these
//      positions from LDS, never back from the cache);
//   3. scores: LP = hd / 8 lanes per position, each with 8 dimensions of k and of
//      every query in registers (256 / LP positions at a time), the dot reduced
//      over the LP lanes by DPP; causal mask; into LDS;
//   4. per query (a wave each), the chunk's max and the exponentials and their sum;
//   5. p v: a float4 of dimensions per thread, positions split over 256 / (hd / 4)
//      thread groups, whose sums meet by lane shuffles within a wave and one LDS
//      pass across the four waves;
//   6. the chunk's (max, sum) pair and o[hd] per query to the workspace.
// attn_merge_kernel: a workgroup per (token, head) merges the chunks by
// log-sum-exp into the output rows [m, H hd].  The kernel boundary makes the
// chunk results of every XCD visible to it.  (Merging in the last workgroup of
// each kv head instead needs an agent-scope release -- an L2 write-back -- in
// every workgroup and serialises the merge on one CU a head: measured 3-9 us
// slower.)
// Everything a step reads from HBM beyond the cache is the m qkv rows and the
// per-chunk results (chunks (hd + 2) floats per query, written and read once).
#include <hip/hip_runtime.h>

#include <limits.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "internal.hpp"
#include "split.hpp"

namespace unillm {
namespace {

constexpr int kAttnMaxQ = 16;  // queries per kv head in one call: m * H / KVH
constexpr int kThreads = 256;
constexpr int kMaxChunk = 256;   // positions per workgroup
constexpr int kMaxChunks = 512;  // workgroups per kv head (L <= 131072)

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Sum over aligned groups of LP lanes (8, 16 or 32); every lane of a group gets it.
template <int LP>
__device__ __forceinline__ float group_sum(float v) {
    v += dpp<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp<0x4E>(v);   // quad_perm [2,3,0,1]: quad sums
    v += dpp<0x141>(v);  // row_half_mirror: lane i + lane 7 - i of each 8 -> 8-lane sums
    if constexpr (LP >= 16) v += dpp<0x140>(v);  // row_mirror: lane i + lane 15 - i
    if constexpr (LP >= 32) v += __shfl_xor(v, 16, 64);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ float wave_add(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Dynamic LDS (floats): qs[QB][D] | nk[m][D] | nv[m][D] | sp[QB][C] (scores, then
// exponentials) | red[4][QB][D] | stat[QB][2]
// state: the cache's device state ([0] filled length, [1] overflow flag, [2] this
// call's length, published by workgroup (0, 0) for the merge kernel).
template <int D, int QB>
__global__ __launch_bounds__(kThreads) void attn_decode_kernel(
    const float* __restrict__ qkv, int m, int H, int KVH, int* __restrict__ state, int C,
    int chunks, float scale, const float* __restrict__ inv_freq, float* __restrict__ kc,
    float* __restrict__ vc, int max_seq, float* __restrict__ part) {
    constexpr int LP = D / 8;             // lanes per position in the score pass
    constexpr int SG = kThreads / LP;     // positions at a time (32, 16, 8)
    constexpr int D4 = D / 4;             // float4 columns in the p v pass
    constexpr int NG = kThreads / D4;     // position groups in the p v pass (16, 8, 4)
    constexpr int HALF = D / 2;
    const int g = blockIdx.x, c = blockIdx.y;
    const int G = H / KVH, Q = m * G;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const float* kg = kc + (int64_t)g * max_seq * D;
    const float* vg = vc + (int64_t)g * max_seq * D;

    // score pass: group sg = tid / LP takes positions j0 + sg + SG u (+ UK SG per
    // iteration), lane l8 = tid % LP dimensions 8 l8 .. 8 l8 + 7; p v pass: group
    // pg = tid / D4 takes positions j0 + pg + NG u (+ UV NG per iteration), column
    // c4 = tid % D4.  Cached positions (< len) come from HBM, requested one iteration
    // ahead.  The first iteration's k and v are requested before anything else, the
    // length included: rows clamped into the cache, and a row at or past the filled
    // length is never used (new positions are read from LDS, positions past the
    // chunk's end are masked), so the length's latency and theirs overlap.
    // positions a thread per iteration, 2 of k and 4 of v: the registers leave room for
    // more waves (one query a kv head: 100 VGPRs, five waves a SIMD), and a 32-position
    // chunk is one iteration with no clamped repeats.  Against 4 / 8: the whole
    // Llama-2-7B decode step 1 % faster at L 1024 and L 4096 (KV from HBM), GQA 32/8
    // calls 7-10 % faster; deeper loops (8 / 16) were 8-20 % slower at L 1024
    constexpr int UK = 2, UV = 4;
    const int sg = tid / LP, l8 = tid % LP;
    const int pg = tid / D4, c4 = tid % D4;
    const int j0 = c * C;
    float kA[UK][8], kB[UK][8];
    float4 vA[UV], vB[UV];
#pragma unroll
    for (int u = 0; u < UK; ++u) {
        const float* src = kg + (int64_t)min(j0 + sg + u * SG, max_seq - 1) * D + 8 * l8;
        const float4 a = *reinterpret_cast<const float4*>(src);
        const float4 b = *reinterpret_cast<const float4*>(src + 4);
        kA[u][0] = a.x; kA[u][1] = a.y; kA[u][2] = a.z; kA[u][3] = a.w;
        kA[u][4] = b.x; kA[u][5] = b.y; kA[u][6] = b.z; kA[u][7] = b.w;
    }
#pragma unroll
    for (int u = 0; u < UV; ++u)
        vA[u] = *reinterpret_cast<const float4*>(vg + (int64_t)min(j0 + pg + u * NG, max_seq - 1) * D +
                                                 4 * c4);
    const int len = state[0];
    if (g == 0 && c == 0 && tid == 0) state[2] = len;
    if (len + m > max_seq) return;  // overflow: nothing appended; the merge reports it
    const int j1 = min(j0 + C, len + m);
    const int n = j1 - j0;
    if (n <= 0) {  // a chunk past the filled positions (a grid sized for max_seq): empty
        float* ms = part;
        float* po = part + (int64_t)m * H * chunks * 2;
        for (int i = tid; i < Q * D; i += kThreads) {
            const int qi = i / D, d = i - qi * D;
            const int t = qi / G, e = qi - t * G;
            const int64_t qc = ((int64_t)t * H + g * G + e) * chunks + c;
            if (d == 0) *reinterpret_cast<float2*>(ms + 2 * qc) = make_float2(-INFINITY, 0.0f);
            po[qc * D + d] = 0.0f;
        }
        return;
    }
    const int64_t W = (int64_t)(H + 2 * KVH) * D;  // floats per qkv row
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* qs = sm;
    float* nk = qs + QB * D;
    float* nv = nk + m * D;
    float* sp = nv + m * D;
    float* red = sp + QB * C;
    float* stat = red + 4 * QB * D;
    const int nit_k = (n + UK * SG - 1) / (UK * SG), nit_v = (n + UV * NG - 1) / (UV * NG);
    auto load_k = [&](float (&kr)[UK][8], int it) {
#pragma unroll
        for (int u = 0; u < UK; ++u) {
            const int j = j0 + min(it * UK * SG + sg + u * SG, n - 1);
            const float* src = kg + (int64_t)(j < len ? j : 0) * D + 8 * l8;  // branch-free
            const float4 a = *reinterpret_cast<const float4*>(src);
            const float4 b = *reinterpret_cast<const float4*>(src + 4);
            kr[u][0] = a.x; kr[u][1] = a.y; kr[u][2] = a.z; kr[u][3] = a.w;
            kr[u][4] = b.x; kr[u][5] = b.y; kr[u][6] = b.z; kr[u][7] = b.w;
        }
    };
    auto load_v = [&](float4 (&vr)[UV], int it) {
#pragma unroll
        for (int u = 0; u < UV; ++u) {
            const int j = j0 + min(it * UV * NG + pg + u * NG, n - 1);
            vr[u] = *reinterpret_cast<const float4*>(vg + (int64_t)(j < len ? j : 0) * D + 4 * c4);
        }
    };

    // 1. rotated, scaled queries
    for (int i = tid; i < Q * HALF; i += kThreads) {
        const int qi = i / HALF, p = i - qi * HALF;
        const int t = qi / G, e = qi - t * G;
        const float* x = qkv + t * W + (int64_t)(g * G + e) * D;
        float sn, cs;
        sincosf((float)(len + t) * inv_freq[p], &sn, &cs);
        const float a = x[p], b = x[p + HALF];
        qs[qi * D + p] = (a * cs - b * sn) * scale;
        qs[qi * D + p + HALF] = (a * sn + b * cs) * scale;
    }
    // 2. new positions [nb, j1) of this chunk: k rotated, v copied; into LDS and the cache
    const int nb = max(j0, len);
    for (int i = tid; i < (j1 - nb) * D; i += kThreads) {
        const int j = nb + i / D, d = i % D, t = j - len;
        const float* xk = qkv + t * W + (int64_t)(H + g) * D;
        const float* xv = qkv + t * W + (int64_t)(H + KVH + g) * D;
        const int p = d < HALF ? d : d - HALF;
        float sn, cs;
        sincosf((float)j * inv_freq[p], &sn, &cs);
        const float a = xk[p], b = xk[p + HALF];
        const float kv = d < HALF ? a * cs - b * sn : a * sn + b * cs;
        const float vv = xv[d];
        nk[t * D + d] = kv;
        nv[t * D + d] = vv;
        kc[((int64_t)g * max_seq + j) * D + d] = kv;
        vc[((int64_t)g * max_seq + j) * D + d] = vv;
    }
    __syncthreads();

    // 3. scores (causal mask applied), into sp
    {
        float qr[QB][8];
#pragma unroll
        for (int qi = 0; qi < QB; ++qi) {
            const float4 a = *reinterpret_cast<const float4*>(qs + min(qi, Q - 1) * D + 8 * l8);
            const float4 b = *reinterpret_cast<const float4*>(qs + min(qi, Q - 1) * D + 8 * l8 + 4);
            qr[qi][0] = a.x; qr[qi][1] = a.y; qr[qi][2] = a.z; qr[qi][3] = a.w;
            qr[qi][4] = b.x; qr[qi][5] = b.y; qr[qi][6] = b.z; qr[qi][7] = b.w;
        }
        auto score = [&](float (&kr)[UK][8], int it) {
#pragma unroll
            for (int u = 0; u < UK; ++u) {
                const int jl = it * UK * SG + sg + u * SG;
                const int j = j0 + min(jl, n - 1);
                if (j >= len) {  // a new position: its rotated k is in LDS
                    const float4 a = *reinterpret_cast<const float4*>(nk + (j - len) * D + 8 * l8);
                    const float4 b = *reinterpret_cast<const float4*>(nk + (j - len) * D + 8 * l8 + 4);
                    kr[u][0] = a.x; kr[u][1] = a.y; kr[u][2] = a.z; kr[u][3] = a.w;
                    kr[u][4] = b.x; kr[u][5] = b.y; kr[u][6] = b.z; kr[u][7] = b.w;
                }
#pragma unroll
                for (int qi = 0; qi < QB; ++qi) {
                    float s = 0.0f;
#pragma unroll
                    for (int d = 0; d < 8; ++d) s = fmaf(qr[qi][d], kr[u][d], s);
                    s = group_sum<LP>(s);
                    // lane qi % LP of the group stores query qi's score
                    if (jl < n && qi < Q && qi % LP == l8) {
                        const bool visible = j <= len + qi / G;  // causal
                        sp[qi * C + jl] = visible ? s : -INFINITY;
                    }
                }
            }
        };
        for (int it = 0; it < nit_k; it += 2) {  // wave-uniform trip count
            if (it + 1 < nit_k) load_k(kB, it + 1);
            score(kA, it);
            if (it + 1 < nit_k) {
                if (it + 2 < nit_k) load_k(kA, it + 2);
                score(kB, it + 1);
            }
        }
    }
    // the p v pass's second iteration, requested now (the k registers are free) so
    // its latency passes during the softmax
    if (nit_v > 1) load_v(vB, 1);
    __syncthreads();

    // 4. per query: the chunk's max, exponentials and their sum (a wave per query)
    for (int qi = wv; qi < Q; qi += kThreads / 64) {
        float mx = -INFINITY;
        for (int jl = lane; jl < n; jl += 64) mx = fmaxf(mx, sp[qi * C + jl]);
        mx = wave_max(mx);
        float sum = 0.0f;
        for (int jl = lane; jl < n; jl += 64) {
            const float pv = mx == -INFINITY ? 0.0f : expf(sp[qi * C + jl] - mx);
            sp[qi * C + jl] = pv;
            sum += pv;
        }
        sum = wave_add(sum);
        if (lane == 0) {
            stat[2 * qi] = mx;
            stat[2 * qi + 1] = sum;
        }
    }
    __syncthreads();

    // 5. o = p v
    {
        float4 o[QB];
#pragma unroll
        for (int qi = 0; qi < QB; ++qi) o[qi] = make_float4(0.f, 0.f, 0.f, 0.f);
        auto accumulate = [&](float4 (&vr)[UV], int it) {
#pragma unroll
            for (int u = 0; u < UV; ++u) {
                const int jl = it * UV * NG + pg + u * NG;
                if (jl >= n) break;
                const int j = j0 + jl;
                if (j >= len) vr[u] = *reinterpret_cast<const float4*>(nv + (j - len) * D + 4 * c4);
#pragma unroll
                for (int qi = 0; qi < QB; ++qi) {
                    if (qi >= Q) break;
                    const float p = sp[qi * C + jl];
                    o[qi].x = fmaf(p, vr[u].x, o[qi].x);
                    o[qi].y = fmaf(p, vr[u].y, o[qi].y);
                    o[qi].z = fmaf(p, vr[u].z, o[qi].z);
                    o[qi].w = fmaf(p, vr[u].w, o[qi].w);
                }
            }
        };
        for (int it = 0; it < nit_v; it += 2) {
            if (it > 0 && it + 1 < nit_v) load_v(vB, it + 1);
            accumulate(vA, it);
            if (it + 1 < nit_v) {
                if (it + 2 < nit_v) load_v(vA, it + 2);
                accumulate(vB, it + 1);
            }
        }
        // the NG groups' sums: the groups of one wave by lane shuffles, then the
        // four waves through red[w][qi][D], added up when the triples are written
        constexpr int GPW = 64 / D4;  // groups per wave (4, 2, 1)
#pragma unroll
        for (int qi = 0; qi < QB; ++qi) {
            if (qi >= Q) continue;  // wave-uniform
            float4 v = o[qi];
            if constexpr (GPW >= 4) {
                v.x += __shfl_xor(v.x, 16, 64); v.y += __shfl_xor(v.y, 16, 64);
                v.z += __shfl_xor(v.z, 16, 64); v.w += __shfl_xor(v.w, 16, 64);
            }
            if constexpr (GPW >= 2) {
                v.x += __shfl_xor(v.x, 32, 64); v.y += __shfl_xor(v.y, 32, 64);
                v.z += __shfl_xor(v.z, 32, 64); v.w += __shfl_xor(v.w, 32, 64);
            }
            if (lane < D4) *reinterpret_cast<float4*>(red + (wv * QB + qi) * D + 4 * c4) = v;
        }
    }
    __syncthreads();

    // 6. the chunk's (max, sum) pair and o of every query (ms [q][chunk][2], po
    //    [q][chunk][D], q = t H + h)
    float* ms = part;
    float* po = part + (int64_t)m * H * chunks * 2;
    for (int i = tid; i < Q * D; i += kThreads) {
        const int qi = i / D, d = i - qi * D;
        const int t = qi / G, e = qi - t * G;
        const int64_t qc = ((int64_t)t * H + g * G + e) * chunks + c;
        if (d == 0) *reinterpret_cast<float2*>(ms + 2 * qc) = make_float2(stat[2 * qi], stat[2 * qi + 1]);
        po[qc * D + d] = (red[qi * D + d] + red[(QB + qi) * D + d]) +
                         (red[(2 * QB + qi) * D + d] + red[(3 * QB + qi) * D + d]);
    }
}

// The merge, per (token t, head h) = blockIdx.x: wave 0 reads every chunk's (max, sum)
// pair (one pass of loads), forms the overall max M and sum S and each chunk's weight
// e^(M_c - M) / S in LDS; thread d sums o_c[d] times the weights, 32 chunks' loads in
// flight (the first 32 requested at entry).  A chunk whose queries were all masked has M_c = -inf and weight 0.
// The cache length advances here (workgroup 0, after every chunk has read it), or,
// when the call found len + m > max_seq, the output is NaN and the overflow flag set.
template <int D>
__global__ __launch_bounds__(D) void attn_merge_kernel(const float* __restrict__ part, int m,
                                                       int H, int chunks, float* __restrict__ out,
                                                       int* __restrict__ state, int max_seq) {
    extern __shared__ float wts[];  // [chunks] weights, then [chunks] the chunks' sums
    const int th = blockIdx.x;      // t H + h
    const int tid = threadIdx.x, lane = tid & 63;
    const float2* pq = reinterpret_cast<const float2*>(part) + (int64_t)th * chunks;
    const float* po = part + (int64_t)m * H * chunks * 2 + (int64_t)th * chunks * D + tid;
    // every load that needs no other is requested at once, before the length is
    // checked: the length, the first 64 chunks' (max, sum) and the first 32 chunks'
    // o[d] (the o loads do not depend on the weights, so they overlap the (max, sum)
    // pass)
    const int len = state[2];
    float2 v0 = make_float2(-INFINITY, 0.0f);
    if (tid < 64 && lane < chunks) v0 = pq[lane];
    float ov[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) ov[u] = po[(int64_t)min(u, chunks - 1) * D];
    if (len + m > max_seq) {
        out[(int64_t)th * D + tid] = __builtin_nanf("");
        if (th == 0 && tid == 0) state[1] = 1;
        return;
    }
    if (th == 0 && tid == 0) state[0] = len + m;
    if (tid < 64) {
        float* sy = wts + chunks;
        float M = v0.x;
        if (lane < chunks) {
            wts[lane] = v0.x;
            sy[lane] = v0.y;
        }
        for (int cc = lane + 64; cc < chunks; cc += 64) {
            const float2 v = pq[cc];
            wts[cc] = v.x;
            sy[cc] = v.y;
            M = fmaxf(M, v.x);
        }
        M = wave_max(M);
        float S = 0.0f;
        for (int cc = lane; cc < chunks; cc += 64) {
            const float mc = wts[cc];
            const float f = M == -INFINITY || mc == -INFINITY ? 0.0f : expf(mc - M);
            wts[cc] = f;
            S = fmaf(sy[cc], f, S);
        }
        S = wave_add(S);
        for (int cc = lane; cc < chunks; cc += 64) wts[cc] /= S;
    }
    __syncthreads();
    float O = 0.0f;
    for (int cc = 0; cc < chunks; cc += 32) {  // the last batch clamps its loads
        if (cc > 0)
#pragma unroll
            for (int u = 0; u < 32; ++u) ov[u] = po[(int64_t)min(cc + u, chunks - 1) * D];
#pragma unroll
        for (int u = 0; u < 32; ++u)
            if (cc + u < chunks) O = fmaf(ov[u], wts[cc + u], O);
    }
    out[(int64_t)th * D + tid] = O;
}

template <int D, int QB>
hipError_t launch_d_q(const KvCache& kv, const float* qkv, int m, int H, int C, int chunks,
                      float* part, float* out, hipStream_t s) {
    const size_t lds = sizeof(float) * ((size_t)QB * D * 5 + (size_t)m * D * 2 +
                                        (size_t)QB * C + 2 * QB);
    if (lds > 159 * 1024) return hipErrorInvalidValue;
    static const bool attr = hipFuncSetAttribute((const void*)attn_decode_kernel<D, QB>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 160 * 1024 - 1024) == hipSuccess;
    if (!attr) return hipErrorInvalidValue;
    attn_decode_kernel<D, QB><<<dim3((unsigned)kv.n_kv_heads, (unsigned)chunks), kThreads, lds, s>>>(
        qkv, m, H, (int)kv.n_kv_heads, kv.state, C, chunks, 1.0f / sqrtf((float)D), kv.inv_freq,
        kv.k, kv.v, (int)kv.max_seq, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    attn_merge_kernel<D><<<(unsigned)(m * H), D, sizeof(float) * 2 * (size_t)chunks, s>>>(
        part, m, H, chunks, out, kv.state, (int)kv.max_seq);
    return hipGetLastError();
}

template <int D>
hipError_t launch_d(const KvCache& kv, const float* qkv, int m, int H, int C, int chunks,
                    float* part, float* out, hipStream_t s) {
    const int Q = m * (H / (int)kv.n_kv_heads);
    if (Q <= 1) return launch_d_q<D, 1>(kv, qkv, m, H, C, chunks, part, out, s);
    if (Q <= 2) return launch_d_q<D, 2>(kv, qkv, m, H, C, chunks, part, out, s);
    if (Q <= 4) return launch_d_q<D, 4>(kv, qkv, m, H, C, chunks, part, out, s);
    if (Q <= 8) return launch_d_q<D, 8>(kv, qkv, m, H, C, chunks, part, out, s);
    return launch_d_q<D, 16>(kv, qkv, m, H, C, chunks, part, out, s);
}

// Chunk length for L positions: (kv head, chunk) workgroups to cover the CUs
// twice; chunks of 32 .. kMaxChunk positions (a multiple of 32), at most
// kMaxChunks of them.  0 when L is beyond kMaxChunk * kMaxChunks.
int64_t chunk_len(int64_t L, int64_t KVH) {
    // chunks for 4x the CUs up to 2048 positions, 2x beyond (MHA L1024: 12.7 -> 12.2 us
    // a call with 4x; L4096 measured slower with 4x, 31.2 against 27.1 us)
    const int64_t want = (L <= 2048 ? 4 : 2) * (int64_t)device_info().cu_count;
    // enough chunks for the CUs, but none longer than kMaxChunk: with many kv heads
    // the CUs fill with fewer, longer chunks, and the cap takes over from there
    int64_t C = std::min<int64_t>((L * KVH + want - 1) / want, kMaxChunk);
    C = std::max(C, (L + kMaxChunks - 1) / kMaxChunks);
    C = std::max<int64_t>(32, (C + 31) / 32 * 32);
    return C > kMaxChunk ? 0 : C;
}

// ---- prompt-length calls (m H / KVH beyond a decode step) ---------------------------------
//
// rope_append_kernel, a workgroup per (token t, head h0 + blockIdx.y): k heads rotated at
// position len + t and, with v, appended to the cache (the decode kernel's formulas, so
// either path writes the same cache); for hd 256 also q heads, rotated and scaled by
// 1 / sqrt(hd), into the workspace qw[H][m][hd].  Then, for hd 64 and 128,
// attn_prompt_kernel on the matrix cores (further down; it rotates its own queries; with
// its key range split, attn_merge_split_kernel after it); for hd 256,
// attn_prefill_kernel, a workgroup per (block of BQ queries, head h): flash-style causal
// attention over the cache in f32 --
//   - the block's queries Q^T [hd][BQ] stay in LDS; the key positions run in tiles of BK
//     (K^T [hd][BK] and V [BK][hd] in LDS), only up to the block's last query position;
//   - thread (tr, tc) of 16 x 16 computes scores for rows tr RT .. and columns tc CT ..
//     (RT = BQ / 16, CT = BK / 16), masks positions past each query (and past the
//     filled length), and keeps each row's running max and sum (online softmax: the
//     earlier partial output rescaled by e^(m_old - m_new)); the row reductions run over
//     the 16 lanes of one tc group by lane shuffles;
//   - the exponentials go to LDS as P^T [BK][BQ]; the same thread then accumulates
//     rows tr RT .. of O for output dimensions tc hd / 16 .., read P and V from LDS.
// f32 throughout, like the reference's cache and matmuls (llama.rs:1108-1146).  LDS
// rows are padded by 4 floats so the transposing stores spread over the banks.

template <int D>
__global__ __launch_bounds__(D / 2) void rope_append_kernel(
    const float* __restrict__ qkv, int m, int H, int KVH, int* __restrict__ state, float scale,
    const float* __restrict__ inv_freq, float* __restrict__ kc, float* __restrict__ vc,
    int max_seq, float* __restrict__ qw, int h0) {
    constexpr int HALF = D / 2;
    const int len = state[0];
    const int t = blockIdx.x, hh = h0 + blockIdx.y, p = threadIdx.x;
    if (t == 0 && blockIdx.y == 0 && p == 0) state[2] = len;  // this call's length, for the next kernel
    if (len + m > max_seq) return;  // overflow: nothing appended; the attention kernel reports it
    const float* row = qkv + (int64_t)t * (H + 2 * KVH) * D;
    float sn, cs;
    sincosf((float)(len + t) * inv_freq[p], &sn, &cs);
    if (hh < H) {
        const float* x = row + (int64_t)hh * D;
        const float a = x[p], b = x[p + HALF];
        float* q = qw + ((int64_t)hh * m + t) * D;
        q[p] = (a * cs - b * sn) * scale;
        q[p + HALF] = (a * sn + b * cs) * scale;
    } else {
        const int g = hh - H;
        const float* xk = row + (int64_t)(H + g) * D;
        const float* xv = row + (int64_t)(H + KVH + g) * D;
        const float a = xk[p], b = xk[p + HALF];
        const int64_t dst = ((int64_t)g * max_seq + len + t) * D;
        kc[dst + p] = a * cs - b * sn;
        kc[dst + p + HALF] = a * sn + b * cs;
        vc[dst + p] = xv[p];
        vc[dst + p + HALF] = xv[p + HALF];
    }
}

template <int D, int BQ, int BK>
struct PrefillLds {
    static constexpr int QP = BQ + 4, KP = BK + 4, VP = D + 4, PP = BQ + 4;  // padded rows
    static constexpr int FLOATS = D * QP + D * KP + BK * VP + BK * PP;
    static constexpr size_t BYTES = (size_t)FLOATS * sizeof(float);
};

template <int D, int BQ, int BK>
__global__ __launch_bounds__(256) void attn_prefill_kernel(const float* __restrict__ qw, int m,
                                                           int H, int KVH,
                                                           int* __restrict__ state,
                                                           const float* __restrict__ kc,
                                                           const float* __restrict__ vc,
                                                           int max_seq, float* __restrict__ out) {
    using L = PrefillLds<D, BQ, BK>;
    constexpr int RT = BQ / 16, CT = BK / 16, DC = D / 16;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* qT = sm;                 // [D][QP]
    float* kT = qT + D * L::QP;     // [D][KP]
    float* vs = kT + D * L::KP;     // [BK][VP]
    float* pT = vs + BK * L::VP;    // [BK][PP]
    const int h = blockIdx.y, g = h / (H / KVH);
    const int q0 = blockIdx.x * BQ;
    const int tid = threadIdx.x, tr = tid / 16, tc = tid % 16;
    const int len = state[2];
    const int nq = min(BQ, m - q0);  // real queries of the block
    if (len + m > max_seq) {
        for (int i = tid; i < nq * D; i += 256)
            out[(int64_t)(q0 + i / D) * H * D + (int64_t)h * D + i % D] = __builtin_nanf("");
        if (blockIdx.x == 0 && h == 0 && tid == 0) state[1] = 1;
        return;
    }
    // the length advances here: no workgroup of this kernel reads state[0], and the next
    // call's kernels run after this one
    if (blockIdx.x == 0 && h == 0 && tid == 0) state[0] = len + m;
    const int total = len + m;  // filled positions once this call's keys are in
    // the block's queries, transposed (rows past m repeat the last query)
    for (int i = tid; i < BQ * D; i += 256) {
        const int r = i / D, d = i - r * D;
        qT[d * L::QP + r] = qw[((int64_t)h * m + min(q0 + r, m - 1)) * D + d];
    }
    float mrow[RT], lrow[RT], o[RT][DC];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        mrow[r] = -INFINITY;
        lrow[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < DC; ++c) o[r][c] = 0.0f;
    }
    const int last_pos = len + q0 + nq - 1;  // the block's last query position
    const int nkb = last_pos / BK + 1;
    const float* kg = kc + (int64_t)g * max_seq * D;
    const float* vg = vc + (int64_t)g * max_seq * D;
    for (int kb = 0; kb < nkb; ++kb) {
        __syncthreads();  // the previous tile's readers are done (and Q is staged)
        for (int i = tid; i < BK * D; i += 256) {
            const int j = i / D, d = i - j * D;
            const int64_t src = (int64_t)min(kb * BK + j, total - 1) * D + d;
            kT[d * L::KP + j] = kg[src];
            vs[j * L::VP + d] = vg[src];
        }
        __syncthreads();
        float s[RT][CT];
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c) s[r][c] = 0.0f;
        for (int d = 0; d < D; ++d) {
            float qv[RT], kv[CT];
#pragma unroll
            for (int r = 0; r < RT; ++r) qv[r] = qT[d * L::QP + tr * RT + r];
#pragma unroll
            for (int c = 0; c < CT; ++c) kv[c] = kT[d * L::KP + tc * CT + c];
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int c = 0; c < CT; ++c) s[r][c] = fmaf(qv[r], kv[c], s[r][c]);
        }
        // causal mask (position j visible to query i when j <= len + i), running max
        // and sum per row over the 16 lanes of the row group
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int qpos = len + q0 + tr * RT + r;
            float mx = -INFINITY;
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const int kpos = kb * BK + tc * CT + c;
                if (kpos > qpos || kpos >= total) s[r][c] = -INFINITY;
                mx = fmaxf(mx, s[r][c]);
            }
#pragma unroll
            for (int o2 = 8; o2 > 0; o2 >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o2, 16));
            const float mnew = fmaxf(mrow[r], mx);
            const float alpha = mnew == -INFINITY ? 1.0f : expf(mrow[r] - mnew);
            float sum = 0.0f;
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const float p = s[r][c] == -INFINITY ? 0.0f : expf(s[r][c] - mnew);
                s[r][c] = p;
                sum += p;
            }
#pragma unroll
            for (int o2 = 8; o2 > 0; o2 >>= 1) sum += __shfl_xor(sum, o2, 16);
            lrow[r] = lrow[r] * alpha + sum;
            mrow[r] = mnew;
#pragma unroll
            for (int c = 0; c < DC; ++c) o[r][c] *= alpha;
#pragma unroll
            for (int c = 0; c < CT; ++c) pT[(tc * CT + c) * L::PP + tr * RT + r] = s[r][c];
        }
        __syncthreads();
        for (int j = 0; j < BK; ++j) {
            float pv[RT], vv[DC];
#pragma unroll
            for (int r = 0; r < RT; ++r) pv[r] = pT[j * L::PP + tr * RT + r];
#pragma unroll
            for (int c = 0; c < DC; ++c) vv[c] = vs[j * L::VP + tc * DC + c];
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int c = 0; c < DC; ++c) o[r][c] = fmaf(pv[r], vv[c], o[r][c]);
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int qi = q0 + tr * RT + r;
        if (qi >= m) continue;
        const float inv = 1.0f / lrow[r];
#pragma unroll
        for (int c = 0; c < DC; ++c)
            out[(int64_t)qi * H * D + (int64_t)h * D + tc * DC + c] = o[r][c] * inv;
    }
}

// ---- prompt-length attention on the matrix cores (hd 64 and 128) ---------------------------
//
// attn_prompt_kernel<D, QT>: a workgroup per (block of QT 32-query tiles, or two such
// blocks one after the other; head h), 2 QT waves: wave w takes query tile w % QT and every
// second key tile (kh = w / QT), and the two waves of a tile merge their sums at the block's
// end.  Both products keep f32's precision on the bf16 matrix cores: q, k, v and the
// exponentials p are split exactly into three bf16 parts (split.hpp), and the six products
// of parts above 2^-24 of theirs are summed in f32, the five small ones of q k in a sum of
// their own.  The products are formed transposed so that no row reduction crosses more than two
// lanes and P never leaves the registers:
//   S^T [32 keys][32 queries] = K . Q^T (v_mfma_f32_32x32x16_bf16: A lane l holds key
//     l % 32, dimensions 8 (l / 32) .. + 7 of each 16; B the same of query l % 32, rotated
//     (RoPE), scaled and split once a block by the tile's two waves: part 0 in registers,
//     parts 1 and 2 in LDS, which leaves registers for two waves a SIMD: all 256 of them at
//     hd 128, with 10 spilled, a few of those read back in each key step);
//   a lane's 16 accumulators are 16 keys of ONE query (rows 8 (r / 4) + 4 (l / 32) +
//     r % 4, column l % 32): the query's max and sum over the tile are a 16-value
//     register reduction and one exchange with lane l ^ 32;
//   O^T [D][32 queries] += V^T . P^T: MFMA kb contracts, in lane half hf, the 8 keys whose
//     exponentials that lane holds in accumulators 8 kb .. 8 kb + 7, so B is the lane's
//     own p and V^T is staged in that key order (chunk 2 kb + hf of a row).
// A step stages two key tiles of 32 positions in LDS as parts: K [2][3][32 keys][2 D bytes]
// and V^T [2][3][D][64 bytes], 16-byte chunks XOR-swizzled so that the 16 lanes a read
// serves together touch all banks once.  A thread's staging task is 8 dimensions of a key or
// 8 keys of a dimension.  V is split and stored after the wave's q k products, the next
// step's K after its p v products, each meeting the others at one barrier: every split
// runs beside another wave's MFMAs, without a second buffer.
// Bound by the matrix cores (12 D / 16 MFMAs of 32 cycles a tile and wave) with the softmax
// and the splits' VALU work beside them.  With the causal mask a block's work grows with
// its position: taking blocks i and last - i one after the other gives every workgroup the
// same (a form that paired a low and a high tile in two waves of one workgroup left one
// wave a SIMD half the time).  Measured, kernel alone: m2048, 32 heads of 128: 222-250 us
// (138-155 TFLOP/s of f32 product; 391 on the f32 matrix cores, 270 in the paired form), m500
// behind 777, 32 heads of 64 over 4: 42 us and the merge's 4.5 (65.6 and 4.8).  At m2048 the matrix
// cores are busy 41 % and the VALU 30 % of the cycles, and hardly at once.
// A non-finite k or v makes 0 * inf terms in the split products: a query whose sum or
// output comes out non-finite is recomputed in plain f32.
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 8 f32 (vector v, from element o) -> three parts
template <class V>
__device__ __forceinline__ void split8(const V& v, int o, u32x4 (&p)[3]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t a, b, c;
        split2(__float_as_uint(v[o + 2 * j]), __float_as_uint(v[o + 2 * j + 1]), a, b, c);
        p[0][j] = a;
        p[1][j] = b;
        p[2][j] = c;
    }
}

template <int D, int QT>
struct PromptLds {
    static constexpr int NW = 2 * QT;         // waves
    static constexpr int KROW = 2 * D;        // bytes of a key's part
    static constexpr int KP = 32 * KROW;      // a plane of K
    static constexpr int VP = 64 * D;         // a plane of V^T (the same size)
    static constexpr int TILE = 3 * KP;       // a staged K or V tile
    static constexpr int V0 = 2 * TILE;       // K tiles | V tiles | query parts 1 and 2
    static constexpr int Q1 = 4 * TILE;       // [QT][D / 16][2][64 lanes][16 B]
    static constexpr int BYTES = Q1 + QT * (D / 16) * 2048;
    static constexpr int TASKS = 8 * D / (64 * NW);  // staging tasks a thread for two K (or V) tiles
    // a block's first query parts, and its odd waves' sums, pass through the staging tiles
    static_assert(QT * (D / 16) * 1024 <= 4 * TILE && QT * (2 * D + 8) * 64 <= 4 * TILE, "");  // (and its redone queries)
    // the slot of chunk c in key row r: 8 or 16 chunks a row
    __device__ static uint32_t kslot(uint32_t r, uint32_t c) {
        return D == 128 ? c ^ (r & 15) : c ^ ((r >> 1) & 7);
    }
    __device__ static uint32_t vslot(uint32_t d, uint32_t c) { return c ^ ((d >> 2) & 3); }
};

template <int D, int QT>
__global__ __launch_bounds__(128 * QT, QT == 4 ? 2 : 1) void attn_prompt_kernel(
    const float* __restrict__ qrows, int64_t qstride, int m, int H, int KVH,
    int* __restrict__ state, float scale, const float* __restrict__ inv_freq,
    const float* __restrict__ kc, const float* __restrict__ vc, int max_seq, int blocks, int paired,
    float* __restrict__ out, float* __restrict__ part) {
    using L = PromptLds<D, QT>;
    constexpr int OT = D / 32, NB = D / 16, NT = 128 * QT;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int h = blockIdx.y, g = h / (H / KVH);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hf = lane >> 5;
    const int qt = wv % QT, kh = wv / QT;
    // gridDim.z > 1: this workgroup takes split blockIdx.z of each block's key tiles and
    // writes partials (max, sum, unnormalized o) for attn_merge_split_kernel, which then
    // also advances the length or reports the overflow
    const int S = gridDim.z, z = blockIdx.z;
    const int len = state[2];
    const int other = paired ? blocks - 1 - (int)blockIdx.x : (int)blockIdx.x;  // the second block
    const int nblk = other != (int)blockIdx.x ? 2 : 1;
    if (len + m > max_seq) {
        if (S == 1) {
            for (int bi = 0; bi < nblk; ++bi) {
                const int q0 = (bi ? other : (int)blockIdx.x) * 32 * QT;
                for (int i = tid; i < 32 * QT * D; i += NT) {
                    const int qq = q0 + i / D;
                    if (qq < m) out[(int64_t)qq * H * D + (int64_t)h * D + i % D] = __builtin_nanf("");
                }
            }
            if (blockIdx.x == 0 && h == 0 && tid == 0) state[1] = 1;
        }
        return;
    }
    if (S == 1 && blockIdx.x == 0 && h == 0 && tid == 0) state[0] = len + m;
    const int total = len + m;
    const float* kg = kc + (int64_t)g * max_seq * D;
    const float* vg = vc + (int64_t)g * max_seq * D;

    // staging task i of this thread, f = i NT + tid < 8 D: tile f / (4 D) of the step's two;
    // K: 8 dimensions 8 c .. of key row r; V: dimension d, the 8 keys of chunk ch
    typedef float stage_t __attribute__((ext_vector_type(8 * L::TASKS)));
    stage_t st;
    // (a tile past the filled length repeats the last row, always masked; whole tiles take
    // addresses of a uniform base and a lane's fixed offset)
    auto request = [&](const float* cache, int n, auto IsV) {
        int ti = tid;  // opaque: offsets are recomputed, not kept in registers
        asm volatile("" : "+v"(ti));
        auto each = [&](auto Whole) {
#pragma unroll
            for (int i = 0; i < L::TASKS; ++i) {
                const int tile = (i * NT + 64 * wv) / (4 * D);  // (wave-uniform)
                const int kt = Whole.value ? 2 * n + tile : min(2 * n + tile, (total - 1) / 32);
                const int lim = total - 1 - 32 * kt;
                const float* src = cache + (int64_t)kt * (32 * D);
                const int f = (i * NT + ti) % (4 * D);
                if constexpr (IsV.value) {
                    const int d = f % D, ch = f / D;
                    const int k0 = 16 * (ch / 2) + 4 * (ch % 2);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int r = k0 + 8 * (j / 4) + j % 4;
                        st[8 * i + j] = src[(Whole.value ? r : min(r, lim)) * D + d];
                    }
                } else {
                    const int r = f / (D / 8), c = f % (D / 8);
                    const float* row = src + (Whole.value ? r : min(r, lim)) * D + 8 * c;
                    const float4 a = *reinterpret_cast<const float4*>(row);
                    const float4 b = *reinterpret_cast<const float4*>(row + 4);
                    st[8 * i] = a.x, st[8 * i + 1] = a.y, st[8 * i + 2] = a.z, st[8 * i + 3] = a.w;
                    st[8 * i + 4] = b.x, st[8 * i + 5] = b.y, st[8 * i + 6] = b.z, st[8 * i + 7] = b.w;
                }
            }
        };
        if (64 * (n + 1) <= total) each(std::true_type{});
        else each(std::false_type{});
    };
    auto request_k = [&](int n) { request(kg, n, std::false_type{}); };
    auto request_v = [&](int n) { request(vg, n, std::true_type{}); };
    auto store = [&](auto IsV) {
#pragma unroll
        for (int i = 0; i < L::TASKS; ++i) {
            const int f = i * NT + tid;
            uint32_t off;
            if constexpr (IsV.value) {
                const uint32_t d = f % D, ch = f / D % 4;
                off = L::V0 + f / (4 * D) * L::TILE + d * 64 + L::vslot(d, ch) * 16;
            } else {
                const uint32_t r = f / (D / 8) % 32, c = f % (D / 8);
                off = f / (4 * D) * L::TILE + r * L::KROW + L::kslot(r, c) * 16;
            }
            u32x4 p[3];
            split8(st, 8 * i, p);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<u32x4*>(lds + off + q * L::KP) = p[q];
        }
    };
    constexpr std::false_type kK;
    constexpr std::true_type kV;

    const uint8_t* Ks = lds + kh * L::TILE;
    const uint8_t* Vs = lds + L::V0 + kh * L::TILE;
    const uint32_t voff = col * 64, vsw = L::vslot(col, 0);

    for (int bi = 0; bi < nblk; ++bi) {
        const int t0 = (bi ? other : (int)blockIdx.x) * QT;  // the block's first query tile
        const int mytile = t0 + qt;
        // the wave's last query position (below 0: no queries, every key tile skipped)
        const int wave_last = 32 * mytile < m ? len + min(32 * mytile + 31, m - 1) : -1;
        const int last_pos = len + min(32 * (t0 + QT) - 1, m - 1);
        const int steps = (last_pos / 32 + 2) / 2;  // pairs of key tiles
        const int n0 = z * steps / S, n1 = (z + 1) * steps / S;  // this workgroup's
        if (n0 < n1) request_k(n0);

        // this lane's query (rows past m repeat the last one): dimensions 16 b + 8 hf .. + 7
        // rotated at its position, scaled and split; the tile's two waves do half the
        // dimension pairs each and exchange them through LDS
        const int qi = 32 * mytile + col;
        const int qpos = len + qi;
        u32x4 q[NB];
        uint8_t* q1 = lds + L::Q1 + (qt * NB * 128 + lane) * 16;  // parts 1, 2 at (2 b + i - 1) 1024
        {
            uint8_t* qx = lds + (qt * NB * 64 + lane) * 16;  // part 0 of block b at b * 1024
            __syncthreads();  // the staging tiles are free (the block before is done)
            const int qr = min(qi, m - 1);
            const float* row = qrows + (int64_t)qr * qstride + (int64_t)h * D;
            typedef float f32x8 __attribute__((ext_vector_type(8)));
#pragma unroll
            for (int bb = 0; bb < NB / 4; ++bb) {
                const int b = kh * (NB / 4) + bb;
                f32x8 lo, hi;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int p = 16 * b + 8 * hf + j;
                    float sn, cs;
                    sincosf((float)(len + qr) * inv_freq[p], &sn, &cs);
                    const float a = row[p], c = row[p + D / 2];
                    lo[j] = (a * cs - c * sn) * scale;
                    hi[j] = (a * sn + c * cs) * scale;
                }
                u32x4 pl[3], ph[3];
                split8(lo, 0, pl);
                split8(hi, 0, ph);
                *reinterpret_cast<u32x4*>(qx + b * 1024) = pl[0];
                *reinterpret_cast<u32x4*>(qx + (b + NB / 2) * 1024) = ph[0];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    *reinterpret_cast<u32x4*>(q1 + (2 * b + i) * 1024) = pl[1 + i];
                    *reinterpret_cast<u32x4*>(q1 + (2 * (b + NB / 2) + i) * 1024) = ph[1 + i];
                }
            }
            __syncthreads();
#pragma unroll
            for (int b = 0; b < NB; ++b) q[b] = *reinterpret_cast<const u32x4*>(qx + b * 1024);
            __syncthreads();
        }
        if (n0 < n1) {
            store(kK);
            request_v(n0);
        }

        // the exponentials' reference, in units of log2 e (p = exp2(s log2 e - mrun))
        float mrun = -INFINITY, lrun = 0.0f;
        f32x16 o[OT];
#pragma unroll
        for (int t = 0; t < OT; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[t][e] = 0.0f;
        for (int n = n0; n < n1; ++n) {
            __syncthreads();  // K of step n is staged, V of step n - 1 read
            const int kt = 2 * n + kh;
            // wave-uniform: tiles past the wave's last query skipped
            const bool live = kt * 32 <= wave_last;
            f32x16 s, sl;
            // (the odd waves split V before their products, the even ones after: one's VALU
            // work runs beside the other's MFMAs)
            auto stage_v = [&] {
                store(kV);
                if (n + 1 < n1) request_k(n + 1);
            };
            if (kh == 1) stage_v();
            if (live) {
#pragma unroll
                for (int e = 0; e < 16; ++e) s[e] = 0.0f, sl[e] = 0.0f;
                // the next block's parts are read ahead of a block's MFMAs.  The large product
                // alone goes to s, one rounding a block: with the small ones dealt over both
                // sums the two chains alternate without a wait (m2048 265 against 272 us a
                // call), but short prompts' error rose above the f32 matrix cores' (m439, 32
                // heads of 128: 2.43e-7 against 2.25e-7, with parts cut off; 1.62e-7 in a sum of
                // their own with parts rounded)
                u32x4 k[2][5];
                auto read = [&](int b) {
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        k[b % 2][p] = *reinterpret_cast<const u32x4*>(
                            Ks + p * L::KP + col * L::KROW + L::kslot(col, 2 * b + hf) * 16);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        k[b % 2][3 + i] = *reinterpret_cast<const u32x4*>(q1 + (2 * b + i) * 1024);
                };
                read(0);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    if (b + 1 < NB) read(b + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    const u32x4(&kb)[5] = k[b % 2];
                    sl = mfma_bf16(kb[2], q[b], sl);
                    sl = mfma_bf16(kb[0], kb[4], sl);
                    s = mfma_bf16(kb[0], q[b], s);
                    sl = mfma_bf16(kb[1], kb[3], sl);
                    sl = mfma_bf16(kb[1], q[b], sl);
                    sl = mfma_bf16(kb[0], kb[3], sl);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (kh == 0) stage_v();
            u32x4 p[2][3];
            if (live) {
                s += sl;
                // causal mask (tiles that reach past the wave's first query) and the
                // query's running max / sum
                if (kt * 32 + 31 > len + 32 * mytile) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int kpos = kt * 32 + 8 * (r / 4) + 4 * hf + r % 4;
                        if (kpos > qpos || kpos >= total) s[r] = -INFINITY;
                    }
                }
                float tmax = s[0];
#pragma unroll
                for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, s[r]);
                tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
                tmax *= kLog2e;
                // O^T = alpha O^T + V^T . P^T.  The rescale moves the accumulators through
                // the VALU, so the reference the exponentials are taken against follows
                // the running max only when some query's rises past it by 8 (2^8 a sum's
                // terms at most): with random keys the max itself rises in most tiles.
                if (__any(tmax > mrun + 8.0f)) {
                    const float mnew = fmaxf(mrun, tmax);
                    // (no live key yet: mrun and mnew are -inf, o and l zero)
                    const float alpha = mnew == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(mrun - mnew);
                    lrun *= alpha;
#pragma unroll
                    for (int t = 0; t < OT; ++t)
#pragma unroll
                        for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
                    mrun = mnew;
                }
                const float ref = mrun == -INFINITY ? 0.0f : mrun;  // (all p are 0 then)
                float tsum = 0.0f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], kLog2e, -ref));
                    tsum += s[r];
                }
                lrun += tsum + __shfl_xor(tsum, 32, 64);
                split8(s, 0, p[0]);
                split8(s, 8, p[1]);
            }
            __syncthreads();  // V of step n is staged, K of step n read
            auto stage_k = [&] {
                if (n + 1 < n1) {
                    store(kK);
                    request_v(n + 1);
                }
            };
            if (kh == 1) stage_k();
            if (live) {
                // unit u: output tiles 2 (u / 2) and + 1, keys of MFMA u % 2; the next unit's
                // parts are read ahead
                u32x4 v[2][2][3];
                auto read = [&](int u) {
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int i = 0; i < 3; ++i)
                            v[u % 2][a][i] = *reinterpret_cast<const u32x4*>(
                                Vs + i * L::VP + (u / 2 * 2 + a) * 32 * 64 + voff +
                                (((2 * (u % 2) + hf) ^ vsw) * 16));
                };
                read(0);
#pragma unroll
                for (int u = 0; u < OT; ++u) {
                    if (u + 1 < OT) read(u + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    constexpr int kVi[6] = {2, 0, 1, 1, 0, 0}, kPi[6] = {0, 2, 1, 0, 1, 0};
                    const int t = u / 2 * 2;
#pragma unroll
                    for (int i = 0; i < 6; ++i)
#pragma unroll
                        for (int a = 0; a < 2; ++a)
                            o[t + a] = mfma_bf16(v[u % 2][a][kVi[i]], p[u % 2][kPi[i]], o[t + a]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (kh == 0) stage_k();
        }

        // the tile's two waves: the odd key tiles' sums through LDS to the even ones'
        int el = lane, eh = h;  // opaque: nothing below is computed ahead of the loops above
        asm volatile("" : "+v"(el), "+s"(eh));
        float* ox = reinterpret_cast<float*>(lds) + (qt * (D / 2 + 2)) * 64 + el;
        uint32_t* redo = reinterpret_cast<uint32_t*>(lds + L::Q1);  // [QT] non-finite queries
        __syncthreads();
        if (kh == 1) {
            ox[0] = mrun;
            ox[64] = lrun;
#pragma unroll
            for (int t = 0; t < OT; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) ox[(2 + 16 * t + e) * 64] = o[t][e];
        }
        __syncthreads();
        if (kh == 0) {
            const float m1 = ox[0], l1 = ox[64];
            const float mm = fmaxf(mrun, m1);
            // (a wave without live keys left -inf: weight 0)
            const float f0 = mrun == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mrun - mm);
            const float f1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mm);
            lrun = lrun * f0 + l1 * f1;
            mrun = mm;
            // O[q][32 t + 8 u + 4 hf + 0..3] = o[t][4 u + 0..3] / l, a float4 each; or, split,
            // partials as attn_merge_split_kernel reads them: (max, sum) at [q H + h][S], o at
            // [q H + h][S][hd] after all the pairs (a query with no live tile in this split
            // leaves (-inf, 0) and zeros, weight 0 in the merge)
            const float inv = S > 1 ? 1.0f : 1.0f / lrun;
            // o / l: the rounded product, corrected by its remainder
            auto ratio = [&](float a) {
                const float r = a * inv;
                return S > 1 ? a : fmaf(fmaf(-r, lrun, a), inv, r);
            };
            float chk = lrun * 0.0f;
#pragma unroll
            for (int t = 0; t < OT; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    o[t][e] = ratio(fmaf(ox[(2 + 16 * t + e) * 64], f1, o[t][e] * f0));
                    chk = fmaf(o[t][e], 0.0f, chk);
                }
            const int qi = 32 * mytile + el % 32;
            bool bad = qi < m && chk != 0.0f;  // (inf and NaN leave NaN)
            bad |= (bool)__shfl_xor((int)bad, 32, 64);
            if (qi < m && !bad) {
                const int64_t qc = ((int64_t)qi * H + eh) * S + z;
                float* orow = (S > 1 ? part + (int64_t)m * H * S * 2 + qc * D
                                     : out + (int64_t)qi * H * D + (int64_t)eh * D) + el / 32 * 4;
                if (S > 1 && el < 32)
                    *reinterpret_cast<float2*>(part + 2 * qc) = make_float2(mrun, lrun);
#pragma unroll
                for (int t = 0; t < OT; ++t)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        *reinterpret_cast<float4*>(orow + 32 * t + 8 * u) = make_float4(
                            o[t][4 * u], o[t][4 * u + 1], o[t][4 * u + 2], o[t][4 * u + 3]);
            }
            const uint32_t mask = (uint32_t)__ballot(bad);  // (both halves of a query agree)
            if (el == 0) redo[qt] = mask;
        }
        __syncthreads();
        // A non-finite query again in plain f32 over this split's keys: the block's dealt over
        // its waves, a whole wave each, 64 keys at a time: 8 lanes a key form its score, a lane
        // a key its weight against the running max, then a lane D / 64 dimensions adds the
        // weighted rows.  A row is NaN, and done, as soon as its query, its sum or all its
        // outputs are, and without a look at the keys if it sees the NaN key that ended an
        // earlier one.  m2048, 32 heads of 128, us a call (264 all finite): every row NaN 280,
        // one NaN row in the middle of the prompt 770, an infinite v row at the start (every
        // query redone in full) 5700.
        int nan_key = INT_MAX;  // the first key known to hold a NaN
        int tile = 0, turn = 0;
        uint32_t left = __builtin_amdgcn_readfirstlane(redo[0]);
        while (tile < QT) {
            if (left == 0) {
                if (++tile < QT) left = __builtin_amdgcn_readfirstlane(redo[tile]);
                continue;
            }
            const int query = 32 * (t0 + tile) + __builtin_ctz(left);
            left &= left - 1;
            if (turn++ % L::NW != wv) continue;
            float* qf = reinterpret_cast<float*>(lds) + wv * (D + 64);  // [D]
            float* sc = qf + D;                                         // [64]
            auto settle = [] {  // the wave's LDS stores before its reads after them
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            };
            constexpr int DL = D / 64;  // dimensions a lane: DL el ..
            typedef float dl_t __attribute__((ext_vector_type(DL)));
            dl_t acc = 0.0f;
            bool nan;
            {
                const float* row = qrows + (int64_t)query * qstride + (int64_t)eh * D;
                const int p = el % (D / 2);
                float sn, cs;
                sincosf((float)(len + query) * inv_freq[p], &sn, &cs);
                const float a = row[p], c = row[p + D / 2];
                const float lo = (a * cs - c * sn) * scale, hi = (a * sn + c * cs) * scale;
                nan = __any(lo != lo || hi != hi) || len + query >= nan_key;
                settle();
                qf[p] = lo;
                qf[p + D / 2] = hi;
                settle();
            }
            float mx = -INFINITY, l = 0.0f;
            const int k0 = 64 * n0, k1 = min(64 * n1, len + query + 1);
#pragma unroll 1
            for (int kc0 = k0; kc0 < k1 && !nan; kc0 += 64) {
                const float* qr = qf + el % 8 * (D / 8);
#pragma unroll 1
                for (int i0 = 0; i0 < 8; i0 += 4) {  // 32 keys, 4 a lane group
                    float4 kr[4][D / 32];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int kk = min(kc0 + 8 * (i0 + i) + el / 8, k1 - 1);
#pragma unroll
                        for (int e = 0; e < D / 32; ++e)
                            kr[i][e] = *reinterpret_cast<const float4*>(
                                kg + (int64_t)kk * D + el % 8 * (D / 8) + 4 * e);
                    }
                    __builtin_amdgcn_sched_barrier(0);  // (every load in flight before a use)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float dot = 0.0f;
#pragma unroll
                        for (int e = 0; e < D / 32; ++e) {
                            const float4 b = *reinterpret_cast<const float4*>(qr + 4 * e);
                            dot = fmaf(kr[i][e].x, b.x, dot);
                            dot = fmaf(kr[i][e].y, b.y, dot);
                            dot = fmaf(kr[i][e].z, b.z, dot);
                            dot = fmaf(kr[i][e].w, b.w, dot);
                        }
                        dot = group_sum<8>(dot);
                        if (el % 8 == 0) sc[8 * (i0 + i) + el / 8] = dot;
                    }
                }
                settle();
                const float sv = kc0 + el < k1 ? sc[el] : -INFINITY;
                const float mnew = fmaxf(mx, wave_max(sv));
                const float alpha = mx == -INFINITY ? 0.0f : expf(mx - mnew);
                // (a score of -inf has weight 0 also where no other is above it)
                const float p = sv == -INFINITY ? 0.0f : expf(sv - mnew);
                l = l * alpha + wave_add(p);
                mx = mnew;
                settle();
                sc[el] = p;
                settle();
                const uint64_t pn = __ballot(p != p);
                if (pn) {  // (the sum is NaN; a key with a NaN makes every later row's so)
                    const int kk = kc0 + __builtin_ctzll(pn);
                    const dl_t kv = *reinterpret_cast<const dl_t*>(kg + (int64_t)kk * D + DL * el);
                    bool kn = false;
#pragma unroll
                    for (int i = 0; i < DL; ++i) kn |= kv[i] != kv[i];
                    if (__any(kn)) nan_key = min(nan_key, kk);
                    nan = true;
                    break;
                }
                acc *= alpha;
                const int nk = min(64, k1 - kc0);
#pragma unroll 1
                for (int j0 = 0; j0 < nk; j0 += 16) {
                    dl_t vr[16];
#pragma unroll
                    for (int j = 0; j < 16; ++j)
                        vr[j] = *reinterpret_cast<const dl_t*>(
                            vg + (int64_t)(kc0 + min(j0 + j, nk - 1)) * D + DL * el);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < 16; ++j)
                        if (j0 + j < nk) {  // (a row past the last adds nothing, not 0 * inf)
                            const float pj = sc[j0 + j];
#pragma unroll
                            for (int i = 0; i < DL; ++i) acc[i] = fmaf(pj, vr[j][i], acc[i]);
                        }
                }
                settle();
                bool all = true;
#pragma unroll
                for (int i = 0; i < DL; ++i) all &= acc[i] != acc[i];
                nan = __any(l != l) || __all(all);
            }
            // split: the merge takes the max in units of log2 e, rounded as the matrix-core
            // loop's are; the weights above are against the natural one
            const float m2 = mx * kLog2e;
            const float f = nan               ? __builtin_nanf("")
                            : S == 1          ? 1.0f / l
                            : mx == -INFINITY ? 1.0f
                                              : __builtin_amdgcn_exp2f(fmaf(mx, kLog2e, -m2));
            const int64_t qc = ((int64_t)query * H + eh) * S + z;
            if (S > 1 && el == 0)
                *reinterpret_cast<float2*>(part + 2 * qc) =
                    nan ? make_float2(0.0f, f) : make_float2(m2, l * f);
            float* orow = (S > 1 ? part + (int64_t)m * H * S * 2 + qc * D
                                 : out + (int64_t)query * H * D + (int64_t)eh * D) +
                          DL * el;
            dl_t r = acc * f;
            if (nan) r = f;
            *reinterpret_cast<dl_t*>(orow) = r;
        }
    }
}

// The merge of a split prompt call (S splits of each workgroup's key tiles, a handful):
// a thread per (query q, head h, 4 dimensions); out = sum_z 2^(M_z - M) o_z /
// sum_z 2^(M_z - M) l_z over the splits' (M_z, l_z, o_z) partials (a split in which the
// query had no live key leaves M_z = -inf: weight 0).  The length advance and the
// overflow report are attn_merge_kernel's.
template <int D>
__global__ __launch_bounds__(256) void attn_merge_split_kernel(const float* __restrict__ part,
                                                               int m, int H, int S,
                                                               float* __restrict__ out,
                                                               int* __restrict__ state,
                                                               int max_seq) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (q H + h) (D / 4) + d4
    const int64_t total = (int64_t)m * H * (D / 4);
    const int len = state[2];
    if (len + m > max_seq) {
        if (i < total)
            reinterpret_cast<float4*>(out)[i] =
                make_float4(__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""),
                            __builtin_nanf(""));
        if (i == 0) state[1] = 1;
        return;
    }
    if (i == 0) state[0] = len + m;
    if (i >= total) return;
    const int64_t qh = i / (D / 4), d4 = i % (D / 4);
    const float2* ms = reinterpret_cast<const float2*>(part) + qh * S;
    const float4* po = reinterpret_cast<const float4*>(part + (int64_t)m * H * S * 2) + qh * S * (D / 4) + d4;
    float M = -INFINITY;
    for (int z = 0; z < S; ++z) M = fmaxf(M, ms[z].x);
    float l = 0.0f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int z = 0; z < S; ++z) {
        const float2 p = ms[z];
        const float f = p.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(p.x - M);
        const float4 v = po[(int64_t)z * (D / 4)];
        l = fmaf(p.y, f, l);
        o = make_float4(fmaf(v.x, f, o.x), fmaf(v.y, f, o.y), fmaf(v.z, f, o.z), fmaf(v.w, f, o.w));
    }
    reinterpret_cast<float4*>(out)[i] = make_float4(o.x / l, o.y / l, o.z / l, o.w / l);
}

// How a prompt call is dealt out: QT query tiles a block, blocks paired or not, S splits
// of the key tiles.
struct PromptPlan {
    int qt, paired, S;
};

// Whether an unsplit prompt call takes its queries from a copy: out shares memory with qkv.
bool prompt_copies_q(const float* qkv, int64_t m, int64_t H, int64_t KVH, int64_t D, int S,
                     const float* out) {
    const uintptr_t q0 = reinterpret_cast<uintptr_t>(qkv), o0 = reinterpret_cast<uintptr_t>(out);
    const uintptr_t q1 = q0 + (uintptr_t)(m * (H + 2 * KVH) * D) * sizeof(float),
                    o1 = o0 + (uintptr_t)(m * H * D) * sizeof(float);
    return S == 1 && q0 < o1 && o0 < q1;
}

template <int D, int QT>
hipError_t launch_prompt_qt(const KvCache& kv, const float* qkv, int m, int H, float* ws,
                            const PromptPlan& plan, float* out, hipStream_t s) {
    using L = PromptLds<D, QT>;
    static const bool attr = hipFuncSetAttribute((const void*)attn_prompt_kernel<D, QT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 L::BYTES) == hipSuccess;
    if (!attr) return hipErrorInvalidValue;
    const int KVH = (int)kv.n_kv_heads;
    const float scale = 1.0f / sqrtf((float)D);
    rope_append_kernel<D><<<dim3((unsigned)m, (unsigned)KVH), D / 2, 0, s>>>(
        qkv, m, H, KVH, kv.state, scale, kv.inv_freq, kv.k, kv.v, (int)kv.max_seq, nullptr, H);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // the attention kernel reads the queries while other workgroups store outputs: where out
    // lies over qkv, from a copy (a split call stores no output before its merge)
    const float* qrows = qkv;
    int64_t qstride = (int64_t)(H + 2 * KVH) * D;
    if (prompt_copies_q(qkv, m, H, KVH, D, plan.S, out)) {
        const size_t width = (size_t)H * D * sizeof(float);
        if ((e = hipMemcpy2DAsync(ws, width, qkv, (size_t)qstride * sizeof(float), width, (size_t)m,
                                  hipMemcpyDeviceToDevice, s)) != hipSuccess)
            return e;
        qrows = ws;
        qstride = (int64_t)H * D;
    }
    const int blocks = (m + 32 * QT - 1) / (32 * QT);
    const int grid = plan.paired ? (blocks + 1) / 2 : blocks;
    attn_prompt_kernel<D, QT><<<dim3((unsigned)grid, (unsigned)H, (unsigned)plan.S), 128 * QT,
                                L::BYTES, s>>>(qrows, qstride, m, H, KVH, kv.state, scale,
                                               kv.inv_freq, kv.k, kv.v, (int)kv.max_seq, blocks,
                                               plan.paired, out, ws);
    e = hipGetLastError();
    if (plan.S == 1 || e != hipSuccess) return e;
    const int64_t merge_threads = (int64_t)m * H * (D / 4);
    attn_merge_split_kernel<D><<<(unsigned)((merge_threads + 255) / 256), 256, 0, s>>>(
        ws, m, H, plan.S, out, kv.state, (int)kv.max_seq);
    return hipGetLastError();
}

template <int D>
hipError_t launch_prompt(const KvCache& kv, const float* qkv, int m, int H, float* ws,
                         const PromptPlan& plan, float* out, hipStream_t s) {
    return plan.qt == 4 ? launch_prompt_qt<D, 4>(kv, qkv, m, H, ws, plan, out, s)
                        : launch_prompt_qt<D, 2>(kv, qkv, m, H, ws, plan, out, s);
}

template <int D, int BQ, int BK>
hipError_t launch_prefill_attn(const KvCache& kv, const float* qkv, int m, int H, float* qw,
                               float* out, hipStream_t s) {
    using L = PrefillLds<D, BQ, BK>;
    static const bool attr = hipFuncSetAttribute((const void*)attn_prefill_kernel<D, BQ, BK>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)L::BYTES) == hipSuccess;
    if (!attr) return hipErrorInvalidValue;
    const int KVH = (int)kv.n_kv_heads;
    rope_append_kernel<D><<<dim3((unsigned)m, (unsigned)(H + KVH)), D / 2, 0, s>>>(
        qkv, m, H, KVH, kv.state, 1.0f / sqrtf((float)D), kv.inv_freq, kv.k, kv.v,
        (int)kv.max_seq, qw, 0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    attn_prefill_kernel<D, BQ, BK><<<dim3((unsigned)((m + BQ - 1) / BQ), (unsigned)H), 256,
                                     L::BYTES, s>>>(qw, m, H, KVH, kv.state, kv.k, kv.v,
                                                    (int)kv.max_seq, out);
    return hipGetLastError();
}

}  // namespace

namespace {
// A prompt call's plan: the cheapest of 4- and 2-tile blocks, paired or not, with the key
// tiles in 1, 2, 4 or 8 splits (at most two workgroups a CU), by the longest workgroup's
// steps times the rounds over the CUs, plus the partials written, read and merged.  A step
// of a 4-tile block was measured at 6.5 us (hd 128; 3.6 at hd 64), of a 2-tile one at 3/4 of
// it; a block's queries and its merge cost about two steps.  Measured against every choice
// (us a call, with the 21 of the rewind before it): m2048 at 32 heads of 128 paired 267,
// unpaired 411, split in two 314; m500 behind 777 at 32 heads of 64 unpaired in two splits
// 75, paired in four 82, whole 97; m250 at 32 heads of 64 2-tile blocks in two splits 49.
constexpr int kMaxPromptSplit = 8;
constexpr int64_t kPromptRounds = 2;  // workgroups a CU when the keys are split
// A captured call serves any length its cache reaches, and plans for this many positions in
// all and at most four splits.  Planned for an empty cache, up to 256 tokens keep their keys
// whole or in two, and a replay behind thousands of positions runs on a few workgroups (m32,
// 32 heads of 128, us at 0 / 2032 / 4064 positions: 26 / 149 / 267, now 30 / 64 / 97; m256, 32
// heads of 64 over 4, at 0 / 1920 / 3840: 30 / 104 / 174, now 29 / 69 / 110).  Eight splits take 33 / 51
// / 65 at m32, but 46 at 0 for m128 against 36.
constexpr int64_t kCapturedPositions = 512;
constexpr int kCapturedSplit = 4;

PromptPlan prompt_plan(int64_t m, int64_t H, int64_t D, int64_t len, int most_splits) {
    if (D != 64 && D != 128) return {4, 0, 1};
    const int64_t cus = device_info().cu_count;
    PromptPlan best{4, 1, 1};
    int64_t least = INT64_MAX;
    for (int qt : {4, 2})
        for (int paired = 1; paired >= 0; --paired) {
            const int64_t blocks = (m + 32 * qt - 1) / (32 * qt);
            const int64_t wgs = (paired ? (blocks + 1) / 2 : blocks) * H;
            // the key steps (64 positions) of the first, last and so of a pair of blocks
            const int64_t last = (len + m + 63) / 64, first = (len + std::min<int64_t>(m, 32 * qt) + 63) / 64;
            const int64_t steps = paired && blocks > 1 ? first + last : last;
            const int64_t nblk = paired && blocks > 1 ? 2 : 1;
            const int64_t step_ns = (D == 128 ? 6500 : 3600) * (qt == 4 ? 4 : 3) / 4;
            for (int S = 1; S <= most_splits; S *= 2) {
                if (S > 1 && (wgs * S > kPromptRounds * cus || S > last)) break;
                const int64_t rounds = (wgs * S + cus - 1) / cus;
                int64_t ns = rounds * ((steps + S - 1) / S + 2 * nblk) * step_ns;
                if (S > 1) ns += 3000 + S * m * H * D * 8 / 3000;
                if (ns < least) {
                    least = ns;
                    best = {qt, paired, S};
                }
            }
        }
    return best;
}

// Workspace (slot 2) of one call of m tokens: the decode path's per-chunk partials at
// any length (at most kMaxChunks chunks of (max, sum) and o[hd] per query); at hd 256 the
// prompt path's rotated queries [H][m][hd]; else a split prompt's S partials per query, or
// the copied queries [m][H hd] of an unsplit one whose out lies over its qkv.
size_t attention_call_bytes(const KvCache& kv, int64_t m, int64_t H, int S, bool copies_q) {
    const int64_t G = H / std::max<int64_t>(kv.n_kv_heads, 1), D = kv.head_dim;
    if (m * G <= kAttnMaxQ) return (size_t)m * H * kMaxChunks * (2 + D) * sizeof(float);
    if (S > 1) return (size_t)m * H * S * (2 + D) * sizeof(float);
    return D == 256 || copies_q ? (size_t)m * H * D * sizeof(float) : 0;
}
}  // namespace

// Enough for every call of up to m tokens (what unillm_hip_attention_reserve grows to): the
// longest decode step's partials, and a prompt's.  A split prompt's partial rows (S m H) are
// at most kMaxPromptSplit m H, and, as its workgroups are at most kPromptRounds a CU and
// hold at most two blocks of 128 queries each, at most 256 kPromptRounds CUs; an unsplit
// one's queries (rotated, or copied) are m H rows.
size_t attention_workspace_bytes(const KvCache& kv, int64_t m, int64_t H) {
    const int64_t G = H / std::max<int64_t>(kv.n_kv_heads, 1), D = kv.head_dim;
    size_t need = 0;
    const int64_t md = std::min(m, kAttnMaxQ / G);
    if (md >= 1) need = attention_call_bytes(kv, md, H, 1, false);
    if (m * G > kAttnMaxQ) {
        const int64_t rows = std::min<int64_t>(kMaxPromptSplit * m * H,
                                               256 * kPromptRounds * (int64_t)device_info().cu_count);
        need = std::max({need, (size_t)rows * (2 + D) * sizeof(float),
                         attention_call_bytes(kv, m, H, 1, true)});
    }
    return need;
}

hipError_t launch_attention(const KvCache& kv, const float* qkv, int64_t m, int64_t H,
                            float* out, int64_t len_hint, hipStream_t s) {
    const int D = (int)kv.head_dim;
    void* ws = nullptr;
    hipError_t e;
    if (m * (H / kv.n_kv_heads) > kAttnMaxQ) {
        // captured, the length at a replay is not known: planned for kCapturedPositions
        const int64_t len =
            len_hint >= 0 ? len_hint
                          : std::max<int64_t>(0, std::min<int64_t>(kCapturedPositions, kv.max_seq) - m);
        const PromptPlan plan =
            prompt_plan(m, H, D, len, len_hint >= 0 ? kMaxPromptSplit : kCapturedSplit);
        const size_t need = attention_call_bytes(
            kv, m, H, plan.S, prompt_copies_q(qkv, m, H, kv.n_kv_heads, D, plan.S, out));
        if ((e = stream_workspace(s, std::max<size_t>(need, 16), &ws, 2)) != hipSuccess) return e;
        float* f = static_cast<float*>(ws);
        if (D == 64) return launch_prompt<64>(kv, qkv, (int)m, (int)H, f, plan, out, s);
        if (D == 128) return launch_prompt<128>(kv, qkv, (int)m, (int)H, f, plan, out, s);
        return launch_prefill_attn<256, 32, 32>(kv, qkv, (int)m, (int)H, f, out, s);
    }
    // decode: chunks sized for the known length, or for the longest the cache holds
    const int64_t L = len_hint >= 0 ? len_hint + m
                                    : std::min<int64_t>(kv.max_seq, attention_max_positions());
    const int64_t C = chunk_len(L, kv.n_kv_heads);
    if (C == 0) return hipErrorInvalidValue;  // longer than kMaxChunk * kMaxChunks
    const int chunks = (int)((L + C - 1) / C);
    const size_t pbytes = (size_t)m * H * chunks * (2 + D) * sizeof(float);
    if ((e = stream_workspace(s, pbytes, &ws, 2)) != hipSuccess) return e;
    float* part = static_cast<float*>(ws);
    if (D == 64) return launch_d<64>(kv, qkv, (int)m, (int)H, (int)C, chunks, part, out, s);
    if (D == 128) return launch_d<128>(kv, qkv, (int)m, (int)H, (int)C, chunks, part, out, s);
    return launch_d<256>(kv, qkv, (int)m, (int)H, (int)C, chunks, part, out, s);
}

int attention_max_queries() { return kAttnMaxQ; }
int64_t attention_max_positions() { return (int64_t)kMaxChunk * kMaxChunks; }

}  // namespace unillm
