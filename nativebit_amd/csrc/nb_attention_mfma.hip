// Causal attention of T queries of each head over cached keys and values, in
// fp32 on the matrix cores (gfx950): nb_attention_rows / nb_attention_batch
// for head dims 64 and 128 (generate_torch.py:89-98).
//
// What bounds it: 4 T^2 / 2 D FLOP a head in fp32.  The FMAs of a vector
// kernel need an LDS read per one or two of them; v_mfma_f32_16x16x4_f32
// runs them at the card's full fp32 rate (256 FLOP a CU and clock) from
// registers, with the same fp32 products and sums.
//
// Layout: everything is computed transposed, so that a lane keeps one query
// from the scores to the output and nothing passes through LDS.  Lane (c, g)
// = (lane % 16, lane / 16) holds query c of the tile.
//   S^T = K Q^T: A = 16 keys x 4 dims, B = 4 dims x 16 queries.  A lane's
//     16-byte load of the transposed cache, keys p0 + 4c .. + 3 of dim
//     d = g D/4 + s, is the A operand of four 16-key MFMAs; key 4c + i in
//     row c of the i-th.  The lane then holds the scores of keys
//     p0 + 16g + 4j + i (accumulator j of MFMA i) for its query.
//   O^T = V^T P^T: the probabilities are the B operands as they are (keys
//     16g + 4j + i from lane group g); A = 16 dims x 4 keys, and a 16-byte
//     load of V's row, dims 64h + 4c .. + 3, feeds four 16-dim MFMAs.  The
//     lane ends with dims 64h + 16g + 4j + t of its query.
// Every load is 16 bytes a lane, 256 contiguous bytes per 16 lanes; chunks
// of eight (32 registers) are double buffered, 32 MFMAs (1024 cycles) ahead
// of their use.
//
// Split: a workgroup takes 16 queries of one head; its four waves take the
// 64-key tiles in turn, each with its own running maximum and sums, and the
// waves' results are combined through LDS once.  The grid goes through the
// heads in groups (whose keys and values the L2s hold) and in a group from
// the longest query tiles to the shortest, so that the CUs finish together:
// orders that put two long tiles on a CU and two short ones on the next
// measured up to 1.8 times as long.
//
// Measured (20 heads of 128, T queries from position 0): T = 128 / 500 / 700
// / 1000 in 9.3 / 32 / 49 / 80 us; the vector kernel (attention_rows_kernel)
// takes 16.4 / 99.5 / 171 / 319. One query at position 700: 17 us against 65.
// What is left, from a copy without the loads and with cached ones: MFMAs
// and the softmax's VALU work do not overlap between the waves of a SIMD (80 %
// of the fp32 MFMA rate without loads); a CU's loads from L2 come at about
// 17 bytes a clock, which is what two waves a SIMD need. Two query tiles a
// wave (half the loads, 256 registers) were no faster, nor were three waves a
// SIMD (168 registers, spills), nor 8 or 12 waves a workgroup.
#include <math.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "nb_device.h"
#include "nb_internal.h"

namespace nb {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kTile = 64;   // keys of a tile
constexpr int kWaves = 4;   // waves of a workgroup
constexpr int kHeads = 24;  // heads whose workgroups run together (three an XCD)

struct AttArgs {
    const float* q;         // [batch][T][n_head * D], scaled
    const float* k;         // [batch * n_head][D][ctx]
    const float* v;         // [batch * n_head][ctx][D]
    void* out;              // [batch][T][n_head * D]
    int out_dtype;
    int pos0, T, n_head, ctx;
    int head0, heads;       // heads of this launch, of the batch * n_head
    int qtiles;             // query tiles of a head
};

__device__ __forceinline__ float group_max(float v) {   // over lanes c, c + 16, c + 32, c + 48
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float group_sum(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

template <int D>
__global__ __launch_bounds__(64 * kWaves, 2) void attention_mfma_kernel(AttArgs a) {
    constexpr int kSteps = D / 4;    // K = 4 MFMAs of a score
    constexpr int kChunks = D / 32;  // chunks of eight 16-byte loads, of a tile's K and of its V
    constexpr int kH = D / 64;       // 64-dim halves
    constexpr int kKeysPerChunk = 8 / kH;
    constexpr int kPitch = D + 4;
    extern __shared__ __align__(16) float smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;

    // this workgroup's head and query tile: heads in groups of kHeads, the
    // longest query tiles of a group first
    const int per_group = kHeads * a.qtiles;
    const int group = blockIdx.x / per_group, i0 = blockIdx.x - group * per_group;
    const int in_group = min(kHeads, a.heads - group * kHeads);
    const int bh = a.head0 + group * kHeads + i0 % in_group;
    const int qt0 = a.qtiles - 1 - i0 / in_group;
    const int t0 = qt0 * 16;
    const int C = a.n_head * D;
    const int64_t row_base = (int64_t)(bh / a.n_head) * a.T * C + (bh % a.n_head) * D;
    const float* kh = a.k + (int64_t)bh * D * a.ctx;
    const float* vh = a.v + (int64_t)bh * a.ctx * D;
    const int last = a.pos0 + min(t0 + 16, a.T) - 1;  // last position any query sees
    const int ntiles = last / kTile + 1;

    // dims g D/4 .. + D/4 - 1 of each of the lane's queries (rows past T
    // repeat the last one and are not stored)
    float qv[kSteps];
    const int qt = min(t0 + c, a.T - 1), qpos = a.pos0 + qt;
    {
        const f32x4_t* qp = reinterpret_cast<const f32x4_t*>(a.q + row_base + (int64_t)qt * C + g * kSteps);
#pragma unroll
        for (int s = 0; s < kSteps / 4; ++s) {
            const f32x4_t w = qp[s];
#pragma unroll
            for (int e = 0; e < 4; ++e) qv[4 * s + e] = w[e];
        }
    }

    // chunk ch of a tile's keys: dims g D/4 + 8 ch + e (positions past the
    // cache read its end; they are masked)
    auto load_k = [&](int tile, int ch, f32x4_t (&b)[8]) {
        const int p = min(tile * kTile + 4 * c, a.ctx - 4);
        const uint32_t off = (uint32_t)(g * kSteps * a.ctx + p);   // (one head: under 2^32 bytes)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float* row = kh + (int64_t)(8 * ch + e) * a.ctx;
            b[e] = *reinterpret_cast<const f32x4_t*>(row + off);
        }
    };
    // chunk ch of a tile's values: keys 16 g + kKeysPerChunk ch + ..., each
    // kH pieces (positions past the last one seen read that one; their
    // probabilities are zero)
    auto load_v = [&](int tile, int ch, f32x4_t (&b)[8]) {
#pragma unroll
        for (int kk = 0; kk < kKeysPerChunk; ++kk) {
            const int p = min(tile * kTile + 16 * g + kKeysPerChunk * ch + kk, last);
            const uint32_t off = (uint32_t)(p * D + 4 * c);
#pragma unroll
            for (int h = 0; h < kH; ++h) b[kk * kH + h] = *reinterpret_cast<const f32x4_t*>(vh + off + 64 * h);
        }
    };

    f32x4_t out[4 * kH];
#pragma unroll
    for (int i = 0; i < 4 * kH; ++i) out[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    // the first tile with a masked key (at most one more follows it), and
    // the chunks of masked tiles whose values are not all finite
    const int tdiag = (a.pos0 + t0 + 1) / kTile;
    unsigned bad = 0;
    f32x4_t buf[2][8];
    if (wave < ntiles) load_k(wave, 0, buf[0]);
    for (int tile = wave; tile < ntiles; tile += kWaves) {
        f32x4_t s[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ch = 0; ch < kChunks; ++ch) {
            if (ch + 1 < kChunks) {
                load_k(tile, ch + 1, buf[(ch + 1) & 1]);
            } else {
                load_v(tile, 0, buf[0]);
            }
            __builtin_amdgcn_sched_barrier(0);   // (the loads stay ahead of the MFMAs)
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            buf[ch & 1][e][i], qv[8 * ch + e], s[i], 0, 0, 0);
        }
        // probabilities of the tile (s becomes p); a tile that ends past the
        // first query's position masks each query's own
        const bool diag = tile * kTile + kTile - 1 > a.pos0 + t0;
        {
            if (diag) {
                const int k0 = tile * kTile + 16 * g;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        s[i][j] = k0 + 4 * j + i <= qpos ? s[i][j] : -INFINITY;
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) tmax = fmaxf(tmax, s[i][j]);
            const float m_new = fmaxf(m_run, group_max(tmax));
            const float alpha = m_new == -INFINITY ? 1.f : __expf(m_run - m_new);
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float sv = s[i][j];
                    const float e = sv == -INFINITY ? 0.f : __expf(sv - m_new);
                    s[i][j] = e;
                    sum += e;
                }
            l_run = l_run * alpha + sum;   // this lane group's keys
            m_run = m_new;
#pragma unroll
            for (int i = 0; i < 4 * kH; ++i) out[i] *= alpha;
        }
#pragma unroll
        for (int ch = 0; ch < kChunks; ++ch) {
            f32x4_t(&b)[8] = buf[ch & 1];
            if (ch + 1 < kChunks) {
                load_v(tile, ch + 1, buf[(ch + 1) & 1]);
            } else if (tile + kWaves < ntiles) {
                load_k(tile + kWaves, 0, buf[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
            // A masked key's zero probability times an infinity or NaN in
            // its value would be a NaN in queries that do not see it: such
            // chunks of a masked tile are left to the loop below
            bool plain = true;
            if (diag) {
                float z = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int i = 0; i < 4; ++i) z = fmaf(b[e][i], 0.f, z);
                plain = __all(z == 0.f);
            }
            if (plain) {
#pragma unroll
                for (int kk = 0; kk < kKeysPerChunk; ++kk) {
                    constexpr int kpc = kKeysPerChunk;
                    const int key = kpc * ch + kk;   // of the lane group's 16
#pragma unroll
                        for (int h = 0; h < kH; ++h)
#pragma unroll
                            for (int t = 0; t < 4; ++t)
                                out[4 * h + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                    b[kk * kH + h][t], s[key & 3][key >> 2], out[4 * h + t],
                                    0, 0, 0);
                }
            } else {
                bad |= 1u << ((tile - tdiag) * kChunks + ch);
            }
        }
    }

    // chunks left out above: key by key to the queries that see the key, the
    // probability formed again from its dot product
    for (int bit = 0; bad >> bit; ++bit) {
        if (!(bad >> bit & 1)) continue;
        const int k0 = (tdiag + bit / kChunks) * kTile + kKeysPerChunk * (bit % kChunks);
#pragma nounroll
        for (int e = 0; e < 4 * kKeysPerChunk; ++e) {
            const int pos = k0 + 16 * (e / kKeysPerChunk) + e % kKeysPerChunk;
            if (pos > qpos) continue;
            const float* qp = a.q + row_base + (int64_t)qt * C;
            float dot = 0.f;
#pragma nounroll
            for (int d = 0; d < D; ++d) dot = fmaf(qp[d], kh[(int64_t)d * a.ctx + pos], dot);
            const float pr = dot == -INFINITY ? 0.f : __expf(dot - m_run);
#pragma unroll
            for (int h = 0; h < kH; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        out[4 * h + t][j] += pr * vh[(int64_t)pos * D + 64 * h + 16 * g + 4 * j + t];
        }
    }

    // combine the waves: maxima and sums per query, then the weighted outputs
    float* om = smem;                           // [kWaves][16]
    float* ol = om + kWaves * 16;              // [kWaves][16]
    float* oo = ol + kWaves * 16;              // [kWaves][16][kPitch]
    {
        const float l = group_sum(l_run);
        const int qi = wave * 16 + c;
        if (g == 0) {
            om[qi] = m_run;
            ol[qi] = l;
        }
#pragma unroll
        for (int h = 0; h < kH; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<f32x4_t*>(oo + qi * kPitch + 64 * h + 16 * g + 4 * j) =
                    f32x4_t{out[4 * h][j], out[4 * h + 1][j], out[4 * h + 2][j],
                            out[4 * h + 3][j]};
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * (D / 4); e += 64 * kWaves) {
        const int qi = e / (D / 4), d = 4 * (e % (D / 4));
        if (t0 + qi >= a.T) continue;
        float m = -INFINITY;
        for (int w = 0; w < kWaves; ++w) m = fmaxf(m, om[w * 16 + qi]);
        float l = 0.f;
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
        for (int w = 0; w < kWaves; ++w) {
            // (a wave that saw no key, or only scores of -inf, has f = 0; its
            // sums are zero, or NaN where such a key's value is not finite)
            const float f = __expf(om[w * 16 + qi] - m);
            l += f * ol[w * 16 + qi];
            v += f * *reinterpret_cast<const f32x4_t*>(oo + (w * 16 + qi) * kPitch + d);
        }
        const f32x4_t r = v / l;
        const int64_t at = row_base + (int64_t)(t0 + qi) * C + d;
        if (a.out_dtype == NB_BF16) {
            bf16_bits* op = static_cast<bf16_bits*>(a.out) + at;
#pragma unroll
            for (int i = 0; i < 4; ++i) op[i] = f32_to_bf16_rne(r[i]);
        } else {
            float* op = static_cast<float*>(a.out) + at;
#pragma unroll
            for (int i = 0; i < 4; ++i) op[i] = r[i];
        }
    }
}

template <int D>
void launch_att(AttArgs a, int64_t heads, hipStream_t stream) {
    a.qtiles = (a.T + 15) / 16;
    const size_t lds = (size_t)kWaves * 16 * (D + 4 + 2) * 4;
    for_head_ranges(heads, a.qtiles, 64 * kWaves, [&](int head0, int count) {
        a.head0 = head0;
        a.heads = count;
        hipLaunchKernelGGL((attention_mfma_kernel<D>), dim3((unsigned)count * a.qtiles),
                           dim3(64 * kWaves), lds, stream, a);
    });
}

}  // namespace

bool attention_mfma_eligible(const float* q, const float* k, const float* v, int D, int ctx) {
    if (D != 64 && D != 128) return false;
    if (ctx < 4 || ctx % 4 || (int64_t)D * ctx >= (1 << 29)) return false;   // (32-bit offsets in a head)
    return (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
            reinterpret_cast<uintptr_t>(v)) % 16 == 0;
}

int launch_attention_mfma(const float* q, const float* k, const float* v, int pos0, int T,
                          void* out, int out_dtype, int batch, int n_head, int D, int ctx,
                          hipStream_t stream) {
    const AttArgs a = {q, k, v, out, out_dtype, pos0, T, n_head, ctx, 0, 0, 0};
    if (D == 128) {
        launch_att<128>(a, (int64_t)batch * n_head, stream);
    } else {
        launch_att<64>(a, (int64_t)batch * n_head, stream);
    }
    return check_launch("nb_attention_rows");
}

}  // namespace nb
