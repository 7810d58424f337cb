// Kernels of a batched forward pass over T tokens (the prompt pass of the
// packed decoder, gfx950), everything but the packed matmuls (those are the
// prefill GEMMs):
//
//   nb_rmsnorm_rows     per row: x = embedding[token] or x += add; then
//                       h = rmsnorm(x) * w   (generate_torch.py:29-38, 128-132, 150)
//   nb_silu_pairs_rows  act = silu(gate) * up from (gate, up) column pairs
//                       (generate_torch.py:116-117)
//   nb_silu_mul_rows    the same from separate gate and up arrays
//   nb_rope_kv_rows     RoPE of q and k at positions pos0 .. pos0 + T - 1, k and v
//                       appended to the caches, q * D^-0.5 kept for attention
//                       (generate_torch.py:48-60, 80-88)
//   nb_attention_rows   causal attention of T queries over cache positions
//                       0 .. pos0 + t (generate_torch.py:89-98)
//   nb_rope_kv_batch, nb_attention_batch   the last two for several sequences
//
// Arithmetic is fp32; outputs that feed a packed matmul may be rounded to
// bf16 (nearest even).  The cache layout is the decode step's: keys
// transposed [n_head][D][ctx], values [n_head][ctx][D].
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "nb_device.h"
#include "nb_internal.h"

namespace nb {
namespace {

__device__ __forceinline__ void store_out(void* p, int dtype, int64_t i, float v) {
    if (dtype == NB_BF16) {
        static_cast<bf16_bits*>(p)[i] = f32_to_bf16_rne(v);
    } else {
        static_cast<float*>(p)[i] = v;
    }
}

__device__ __forceinline__ float wsum(float v) { return wave64_sum(v); }

// ---------------------------------------------------------------------------
// rmsnorm of T rows, one workgroup per row
// ---------------------------------------------------------------------------
constexpr int kNormThreads = 256;
constexpr int kNormRegs = 16;      // elements per thread kept in registers (C <= 4096)

__global__ __launch_bounds__(kNormThreads) void rmsnorm_rows_kernel(
    float* __restrict__ x, const float* __restrict__ add, const float* __restrict__ emb,
    const int32_t* __restrict__ tokens, int vocab, const float* __restrict__ w,
    void* __restrict__ h, int h_dtype, int C, float eps) {
    __shared__ float red[kNormThreads / 64];
    const int t = blockIdx.x;
    float* xr = x + (int64_t)t * C;
    const int tok = tokens ? tokens[t] : 0;
    if (tokens && (tok < 0 || tok >= vocab)) {
        // a token outside the table reads nothing: its row of x and h is NaN
        // (the whole workgroup leaves here, before any barrier)
        for (int i = threadIdx.x; i < C; i += kNormThreads) {
            xr[i] = __builtin_nanf("");
            store_out(h, h_dtype, (int64_t)t * C + i, __builtin_nanf(""));
        }
        return;
    }
    const float* src = tokens ? emb + (int64_t)tok * C : nullptr;
    const float* ar = add ? add + (int64_t)t * C : nullptr;
    // rows of up to kNormRegs * 256 elements stay in registers between the
    // sum of squares and the scaling, with every load issued up front; 16
    // bytes a lane where the rows allow it
    float ss = 0.f;
    auto in_registers = [&](auto vec_c) {
        constexpr int V = decltype(vec_c)::value;   // elements a load
        typedef __attribute__((ext_vector_type(V))) float fv;
        constexpr int kLoads = kNormRegs / V;
        fv v[kLoads], wv[kLoads];
        const float* from = src ? src : xr;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int i = V * (threadIdx.x + j * kNormThreads);
            const int ic = i < C ? i : 0;
            v[j] = *reinterpret_cast<const fv*>(from + ic);
            if (ar) v[j] += *reinterpret_cast<const fv*>(ar + ic);
            wv[j] = *reinterpret_cast<const fv*>(w + ic);
        }
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int i = V * (threadIdx.x + j * kNormThreads);
            if (i < C) {
                if (src || ar) *reinterpret_cast<fv*>(xr + i) = v[j];
#pragma unroll
                for (int e = 0; e < V; ++e) ss += v[j][e] * v[j][e];
            }
        }
        ss = wsum(ss);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
        __syncthreads();
        float tot = 0.f;
        for (int k = 0; k < kNormThreads / 64; ++k) tot += red[k];  // same order everywhere
        const float norm = sqrtf(tot / (float)C + eps);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int i = V * (threadIdx.x + j * kNormThreads);
            if (i >= C) continue;
            // (x / norm) * w, as generate_torch.py:37
            fv r;
#pragma unroll
            for (int e = 0; e < V; ++e) r[e] = (v[j][e] / norm) * wv[j][e];
            const int64_t o = (int64_t)t * C + i;
            if (h_dtype == NB_F32) {
                *reinterpret_cast<fv*>(static_cast<float*>(h) + o) = r;
            } else {
                typedef __attribute__((ext_vector_type(V))) uint16_t hv;
                hv p;
#pragma unroll
                for (int e = 0; e < V; ++e) p[e] = f32_to_bf16_rne(r[e]);
                *reinterpret_cast<hv*>(static_cast<bf16_bits*>(h) + o) = p;
            }
        }
    };
    if (C <= kNormRegs * kNormThreads) {
        const uintptr_t all = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(add) |
                              reinterpret_cast<uintptr_t>(emb) | reinterpret_cast<uintptr_t>(w) |
                              reinterpret_cast<uintptr_t>(h);
        if (C % 4 == 0 && all % 16 == 0) {
            in_registers(std::integral_constant<int, 4>{});
        } else {
            in_registers(std::integral_constant<int, 1>{});
        }
        return;
    }
    for (int i = threadIdx.x; i < C; i += kNormThreads) {
        float v = src ? src[i] : xr[i];
        if (ar) v = v + ar[i];
        if (src || ar) xr[i] = v;
        ss += v * v;
    }
    ss = wsum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float tot = 0.f;
    for (int k = 0; k < kNormThreads / 64; ++k) tot += red[k];  // same order everywhere
    const float norm = sqrtf(tot / (float)C + eps);
    for (int i = threadIdx.x; i < C; i += kNormThreads) {
        // (x / norm) * w, as generate_torch.py:37
        store_out(h, h_dtype, (int64_t)t * C + i, (xr[i] / norm) * w[i]);
    }
}

// ---------------------------------------------------------------------------
// silu(gate) * up from interleaved columns
// ---------------------------------------------------------------------------
__global__ void silu_pairs_rows_kernel(const float* __restrict__ gu, void* __restrict__ act,
                                       int act_dtype, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float g = gu[2 * i], u = gu[2 * i + 1];
        store_out(act, act_dtype, i, (g / (1.0f + __expf(-g))) * u);
    }
}

// act = silu(gate) * up from two arrays, four elements a thread.
template <bool kVec>
__global__ __launch_bounds__(256) void silu_mul_rows_kernel(const float* __restrict__ gate,
                                                            const float* __restrict__ up,
                                                            void* __restrict__ act, int act_dtype,
                                                            int64_t n) {
    for (int64_t i = 4 * (blockIdx.x * 256LL + threadIdx.x); i < n; i += 4 * 256LL * gridDim.x) {
        float g[4], u[4];
        if (kVec && i + 3 < n) {
            const float4 a = *reinterpret_cast<const float4*>(gate + i);
            const float4 b = *reinterpret_cast<const float4*>(up + i);
            g[0] = a.x, g[1] = a.y, g[2] = a.z, g[3] = a.w;
            u[0] = b.x, u[1] = b.y, u[2] = b.z, u[3] = b.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                g[e] = i + e < n ? gate[i + e] : 0.f;
                u[e] = i + e < n ? up[i + e] : 0.f;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] = (g[e] / (1.0f + __expf(-g[e]))) * u[e];
        if (kVec && act_dtype == NB_F32 && i + 3 < n) {
            *reinterpret_cast<float4*>(static_cast<float*>(act) + i) = make_float4(g[0], g[1], g[2], g[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (i + e < n) store_out(act, act_dtype, i + e, g[e]);
        }
    }
}

// ---------------------------------------------------------------------------
// RoPE + cache append, two forms with the same arithmetic (launch_rope_kv_rows
// chooses).
//
// Few elements: a wave per token and head, lanes along the head's pairs; the
// rotated keys are written by the lanes that form them, each 4-byte store to
// a cache line of its own in the transposed cache.  Latency bound: 2.2-2.5 us
// for one token (any head count up to 160), 2.7 for 33 of 6 heads of 128,
// where the form below takes 2.8-3.3 and 4.9.
//
// Many: a workgroup takes kRT tokens of one head of one sequence.  The rows
// are read and q and v written a wave per token; the rotated keys pass
// through LDS so that they are written along positions, the transposed
// cache's fast index: 512 tokens of 20 heads of 128 (31 MB) in 8.1 us against
// 15.5 in the form above.
// ---------------------------------------------------------------------------
constexpr int kRT = 32;
constexpr int kRopeThreads = 256;
constexpr int kRopeMaxD = 128;

// x * cos2 + rotate(x) * sin2 of one pair (generate_torch.py:54-59)
__device__ __forceinline__ float2 rope_pair(float a, float b, float c, float s) {
    return make_float2(__fadd_rn(__fmul_rn(a, c), __fmul_rn(-b, s)),
                       __fadd_rn(__fmul_rn(b, c), __fmul_rn(a, s)));
}

__global__ __launch_bounds__(64) void rope_kv_token_kernel(
    const float* __restrict__ qkv, float* __restrict__ k_cache, float* __restrict__ v_cache,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, int pos0,
    float* __restrict__ q_out, int D, int ctx) {
    const int t = blockIdx.x, hd = blockIdx.y, b = blockIdx.z, n_head = gridDim.y;
    const int C = n_head * D, half = D / 2, pos = pos0 + t;
    const float scale = 1.0f / sqrtf((float)D);
    const int64_t tok = (int64_t)b * gridDim.x + t, bh = (int64_t)b * n_head + hd;
    const float* row = qkv + tok * 3 * C + hd * D;
    float* qo = q_out + tok * C + hd * D;
    float* ko = k_cache + bh * D * ctx + pos;
    float* vo = v_cache + (bh * ctx + pos) * D;
    for (int i = threadIdx.x; i < half; i += 64) {
        const float c = cos_t[(int64_t)pos * half + i], s = sin_t[(int64_t)pos * half + i];
        const float2 q = rope_pair(row[2 * i], row[2 * i + 1], c, s);
        const float2 k = rope_pair(row[C + 2 * i], row[C + 2 * i + 1], c, s);
        qo[2 * i] = __fmul_rn(q.x, scale);
        qo[2 * i + 1] = __fmul_rn(q.y, scale);
        ko[(int64_t)(2 * i) * ctx] = k.x;
        ko[(int64_t)(2 * i + 1) * ctx] = k.y;
    }
    for (int d = threadIdx.x; d < D; d += 64) vo[d] = row[2 * C + d];
}

__global__ __launch_bounds__(kRopeThreads) void rope_kv_rows_kernel(
    const float* __restrict__ qkv, float* __restrict__ k_cache, float* __restrict__ v_cache,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, int pos0, int T,
    float* __restrict__ q_out, int n_head, int D, int ctx, int tiles, int head0) {
    __shared__ float ks[kRopeMaxD][kRT + 1];
    const int h0 = blockIdx.x / tiles, t0 = (blockIdx.x - h0 * tiles) * kRT;
    const int bh = head0 + h0;
    const int b = bh / n_head, hd = bh - b * n_head;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int C = n_head * D, half = D / 2;
    const int nt = min(kRT, T - t0);
    const float scale = 1.0f / sqrtf((float)D);
#pragma unroll 4
    for (int t = wave; t < nt; t += kRopeThreads / 64) {
        const int64_t tok = (int64_t)b * T + t0 + t;
        const int pos = pos0 + t0 + t;
        const float* row = qkv + tok * 3 * C + hd * D;
        float* qo = q_out + tok * C + hd * D;
        float* vo = v_cache + ((int64_t)bh * ctx + pos) * D;
        for (int i = lane; i < half; i += 64) {
            const float c = cos_t[(int64_t)pos * half + i], s = sin_t[(int64_t)pos * half + i];
            const float2 q = rope_pair(row[2 * i], row[2 * i + 1], c, s);
            const float2 k = rope_pair(row[C + 2 * i], row[C + 2 * i + 1], c, s);
            const float v0 = row[2 * C + 2 * i], v1 = row[2 * C + 2 * i + 1];
            qo[2 * i] = __fmul_rn(q.x, scale);
            qo[2 * i + 1] = __fmul_rn(q.y, scale);
            ks[2 * i][t] = k.x;
            ks[2 * i + 1][t] = k.y;
            vo[2 * i] = v0;
            vo[2 * i + 1] = v1;
        }
    }
    __syncthreads();
    const int t = threadIdx.x % kRT;
    if (t < nt) {
        float* ko = k_cache + (int64_t)bh * D * ctx + pos0 + t0 + t;
        for (int d = threadIdx.x / kRT; d < D; d += kRopeThreads / kRT) ko[(int64_t)d * ctx] = ks[d][t];
    }
}

// ---------------------------------------------------------------------------
// causal attention of T queries: grid (batch * n_head, ceil(T / kQB)), 256
// threads.  The workgroup holds kQB queries of one head and walks the keys in tiles
// of kKT positions through LDS with an online softmax (running max and sum
// per query); query t sees positions 0 .. pos0 + t.  Head dims past D (up
// to a multiple of 4) are zero in LDS, so the dot products run over float4
// pieces and add exact zeros.
// ---------------------------------------------------------------------------
constexpr int kQB = 8;        // queries per workgroup (32 threads each)
constexpr int kKT = 64;       // keys per tile
constexpr int kAttThreads = 256;
constexpr int kRowsMaxD = 128;
constexpr int kQPitch = kRowsMaxD + 4;   // floats per LDS row of q and v (16-byte rows)
constexpr int kKPitch = kKT + 4;         // floats per LDS row of k (one head dim)

__global__ __launch_bounds__(kAttThreads) void attention_rows_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, int pos0, int T, void* __restrict__ out, int out_dtype,
    int n_head, int D, int ctx, int head0) {
    typedef __attribute__((ext_vector_type(4))) float f4;
    __shared__ __align__(16) float qs[kQB][kQPitch];
    __shared__ __align__(16) float ks[kRowsMaxD][kKPitch];   // keys transposed: [dim][position]
    __shared__ __align__(16) float vs[kKT][kQPitch];
    __shared__ __align__(16) float ps[kQB][kKPitch];
    const int bh = head0 + blockIdx.x, t0 = blockIdx.y * kQB;
    const int b = bh / n_head, hd = bh - b * n_head;
    const int tid = threadIdx.x;
    const int C = n_head * D;
    const int64_t row0 = (int64_t)b * T;   // of q and out
    const int D4 = (D + 3) & ~3;
    const int nq = min(kQB, T - t0);
    for (int e = tid; e < kQB * kQPitch; e += kAttThreads) {
        const int i = e / kQPitch, d = e - i * kQPitch;
        qs[i][d] = i < nq && d < D ? q[(row0 + t0 + i) * C + hd * D + d] : 0.f;
    }
    typedef __attribute__((ext_vector_type(2))) float f2;
    // scores: thread (sq, sp) takes query sq and keys 2 sp, 2 sp + 1
    const int sq = tid >> 5, sp = tid & 31;
    // weighted values: thread (oq, og) takes query oq and dims 4 og .. 4 og + 3
    const int oq = tid >> 5, og = tid & 31;
    f4 o0 = {0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;  // per query, kept by its 32 threads alike
    const int last = pos0 + t0 + nq - 1;  // the last position any query sees
    const float* kt = k_cache + (int64_t)bh * D * ctx;
    const float* vc = v_cache + (int64_t)bh * ctx * D;
    for (int p0 = 0; p0 <= last; p0 += kKT) {
        const int np = min(kKT, last + 1 - p0);
        __syncthreads();  // the previous tile is no longer read
        // the tile's keys and values, all loads of a thread issued together
        float kv[kRowsMaxD * kKT / kAttThreads], vv[kRowsMaxD * kKT / kAttThreads];
#pragma unroll
        for (int j = 0; j < kRowsMaxD * kKT / kAttThreads; ++j) {
            const int e = tid + j * kAttThreads;
            const int d = e / kKT, p = e % kKT;            // keys: position fastest
            kv[j] = d < D && p < np ? kt[(int64_t)d * ctx + p0 + p] : 0.f;
            const int pv = e / kRowsMaxD, dv = e % kRowsMaxD;  // values: dim fastest
            vv[j] = dv < D && pv < np ? vc[(int64_t)(p0 + pv) * D + dv] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < kRowsMaxD * kKT / kAttThreads; ++j) {
            const int e = tid + j * kAttThreads;
            ks[e / kKT][e % kKT] = kv[j];
            vs[e / kRowsMaxD][e % kRowsMaxD] = vv[j];
        }
        __syncthreads();
        // scores of this tile, masked past each query's own position
        f2 acc = {0.f, 0.f};
        for (int d = 0; d < D4; d += 4) {
            const f4 qv = *reinterpret_cast<const f4*>(&qs[sq][d]);
            const f2 k0 = *reinterpret_cast<const f2*>(&ks[d][2 * sp]);
            const f2 k1 = *reinterpret_cast<const f2*>(&ks[d + 1][2 * sp]);
            const f2 k2 = *reinterpret_cast<const f2*>(&ks[d + 2][2 * sp]);
            const f2 k3 = *reinterpret_cast<const f2*>(&ks[d + 3][2 * sp]);
            acc += qv.x * k0;   // head dims in order for every score
            acc += qv.y * k1;
            acc += qv.z * k2;
            acc += qv.w * k3;
        }
        float s[2] = {acc.x, acc.y};
        float tmax = -INFINITY;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int p = 2 * sp + j;
            const bool ok = sq < nq && p < np && p0 + p <= pos0 + t0 + sq;
            s[j] = ok ? s[j] : -INFINITY;
            tmax = fmaxf(tmax, s[j]);
        }
        // the 32 threads of a query (consecutive lanes, two rows of 16)
        // agree on its tile max
        tmax = row16_max(tmax);
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = m_new == -INFINITY ? 1.f : __expf(m_run - m_new);
        float lsum = 0.f;
        f2 e2;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float e = s[j] == -INFINITY ? 0.f : __expf(s[j] - m_new);
            e2[j] = e;
            lsum += e;
        }
        *reinterpret_cast<f2*>(&ps[sq][2 * sp]) = e2;
        lsum = row16_sum(lsum);
        lsum += __shfl_xor(lsum, 16);
        l_run = l_run * alpha + lsum;
        m_run = m_new;
        __syncthreads();
        o0 *= alpha;
        for (int p = 0; p < np; ++p) {
            o0 += ps[oq][p] * *reinterpret_cast<const f4*>(&vs[p][4 * og]);
        }
    }
    if (oq < nq) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int d = 4 * og + j;
            if (d < D) store_out(out, out_dtype, (row0 + t0 + oq) * C + hd * D + d, o0[j] / l_run);
        }
    }
}

}  // namespace

int launch_rmsnorm_rows(float* x, const float* add, const float* emb, const int32_t* tokens,
                        int vocab, const float* w, void* h, int h_dtype, int T, int C, float eps,
                        hipStream_t stream) {
    hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3(T), dim3(kNormThreads), 0, stream, x, add, emb,
                       tokens, vocab, w, h, h_dtype, C, eps);
    return check_launch("nb_rmsnorm_rows");
}

int launch_silu_pairs_rows(const float* gu, void* act, int act_dtype, int T, int F,
                           hipStream_t stream) {
    const int64_t n = (int64_t)T * F;
    const int blocks = (int)std::min<int64_t>(4096, (n + 255) / 256);
    hipLaunchKernelGGL(silu_pairs_rows_kernel, dim3(blocks), dim3(256), 0, stream, gu, act,
                       act_dtype, n);
    return check_launch("nb_silu_pairs_rows");
}

int launch_silu_mul_rows(const float* gate, const float* up, void* act, int act_dtype, int64_t n,
                         hipStream_t stream) {
    const int blocks = (int)std::min<int64_t>(4096, (n / 4 + 256) / 256);
    const bool vec = (reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) |
                      reinterpret_cast<uintptr_t>(act)) % 16 == 0;
    hipLaunchKernelGGL(vec ? silu_mul_rows_kernel<true> : silu_mul_rows_kernel<false>, dim3(blocks),
                       dim3(256), 0, stream, gate, up, act, act_dtype, n);
    return check_launch("nb_silu_mul_rows");
}

int launch_rope_kv_rows(const float* qkv, float* k_cache, float* v_cache, const float* cos_t,
                        const float* sin_t, int pos0, int T, float* q_out, int batch, int n_head,
                        int D, int ctx, hipStream_t stream) {
    static_assert(kRopeMaxD >= kRowsMaxD, "the callers' largest head dim");
    // One token, or up to 200 000 elements: with more the scattered stores
    // cost more than the pass through LDS.  Both are as fast at 1900 tokens
    // times heads of D = 128, 3900 of 64, 5900 of 32 and 9500 of 16 (4 to 60
    // heads); with 160 heads of 128 already between 4 tokens (3.3 us against
    // 3.5) and 8 (4.8 against 3.8).
    constexpr int kMaxYZ = 65535;   // of a grid
    const int64_t heads = (int64_t)batch * n_head;
    if (batch <= kMaxYZ && n_head <= kMaxYZ &&
        (T == 1 || (heads * T * D <= 200000 && (T <= 4 || heads < 128)))) {
        hipLaunchKernelGGL(rope_kv_token_kernel, dim3(T, n_head, batch), dim3(64), 0, stream, qkv,
                           k_cache, v_cache, cos_t, sin_t, pos0, q_out, D, ctx);
        return check_launch("nb_rope_kv_rows");
    }
    const int tiles = (T + kRT - 1) / kRT;
    for_head_ranges(heads, tiles, kRopeThreads, [&](int head0, int count) {
        hipLaunchKernelGGL(rope_kv_rows_kernel, dim3((unsigned)count * tiles), dim3(kRopeThreads), 0,
                           stream, qkv, k_cache, v_cache, cos_t, sin_t, pos0, T, q_out, n_head, D,
                           ctx, tiles, head0);
    });
    return check_launch("nb_rope_kv_rows");
}

int launch_attention_rows(const float* q, const float* k_cache, const float* v_cache, int pos0,
                          int T, void* out, int out_dtype, int batch, int n_head, int D, int ctx,
                          hipStream_t stream) {
    // fp32 MFMAs where the layout allows 16-byte loads; up to 32 positions at
    // head dim 128 the vector kernel below is as fast or faster while its
    // workgroups leave CUs idle (16 queries from position 0, 20 heads 8.1 us
    // against 8.8, 60 heads 8.3 against 8.9), from 128 heads over the batch on
    // it is not (160 heads 10.1 against 9.2, 320 heads 16.7 against 10.3; one
    // query 7.8 against 7.9 and 9.2 against 8.4).  Over 32 positions, 20
    // heads: 16 queries up to position 48 8.8 against 8.8, 64 9.2 against 8.9.
    if (attention_mfma_eligible(q, k_cache, v_cache, D, ctx) &&
        (D < 128 || pos0 + T > 32 || (int64_t)batch * n_head >= 128)) {
        return launch_attention_mfma(q, k_cache, v_cache, pos0, T, out, out_dtype, batch, n_head, D,
                                     ctx, stream);
    }
    for_head_ranges((int64_t)batch * n_head, 1, kAttThreads, [&](int head0, int count) {
        hipLaunchKernelGGL(attention_rows_kernel, dim3(count, (T + kQB - 1) / kQB),
                           dim3(kAttThreads), 0, stream, q, k_cache, v_cache, pos0, T, out,
                           out_dtype, n_head, D, ctx, head0);
    });
    return check_launch("nb_attention_rows");
}

int attention_rows_max_head_dim() { return kRowsMaxD; }

}  // namespace nb
