// Bit-exact format kernels: unpack, pack and dequantize NativeBit index
// streams on gfx950 (their outputs must equal the reference's byte for
// byte).  The bulk of a stream goes through chunk kernels: a chunk is 32
// indices = 4 groups of 8 = BITS whole dwords of the LSB-first stream, so a
// thread moves BITS dwords one way and 32 index bytes (or 32 weights) the
// other with wide loads and stores, its field offsets fixed at compile time.
// The last count % 32 indices, and pointers without the chunk kernels'
// alignment, go through per-element grid-stride kernels.
//
// Reference semantics: nativebit/pack.py:21-169 (pack_3bit, unpack_3bit,
// pack_4bit, unpack_4bit, pack_nbits, unpack_nbits, reconstruct_weight),
// inference/triton_kernel.py:199-220 (pack_indices_to_3bit),
// inference/pack.py:21-35 (quantize_weight, fused here with the pack).
#include <math.h>

#include <type_traits>

#include "nb_device.h"
#include "nb_internal.h"
#include "nb_lookup.h"

namespace nb {
namespace {

constexpr int kThreads = 256;

// Grid for a grid-stride loop over `n` items: enough workgroups to cover
// every CU several times, never more than needed.
inline int grid_for(int64_t n) {
    int64_t want = (n + kThreads - 1) / kThreads;
    int64_t cap = (int64_t)device_cu_count() * 16;
    if (want < 1) want = 1;
    return (int)(want < cap ? want : cap);
}

__global__ __launch_bounds__(kThreads) void unpack_kernel(
    const uint8_t* __restrict__ packed, int64_t nbytes,
    uint8_t* __restrict__ out, int64_t first, int64_t count, int bits) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    for (int64_t i = first + (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count;
         i += stride) {
        out[i] = (uint8_t)read_field(packed, nbytes, i, bits);
    }
}

// One output byte per iteration: byte b holds stream bits [8b, 8b+8), i.e.
// the fields of indices floor(8b/bits) .. floor((8b+7)/bits).
__global__ __launch_bounds__(kThreads) void pack_kernel(
    const uint8_t* __restrict__ idx, int64_t count, int bits,
    uint8_t* __restrict__ out, int64_t first_byte, int64_t nbytes) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    const uint32_t mask = (1u << bits) - 1u;
    for (int64_t b = first_byte + (int64_t)blockIdx.x * kThreads + threadIdx.x; b < nbytes;
         b += stride) {
        const int64_t first_bit = b * 8;
        const int64_t i0 = first_bit / bits;
        const int64_t i1 = (first_bit + 7) / bits;
        uint32_t v = 0;
        for (int64_t i = i0; i <= i1 && i < count; ++i) {
            const int64_t shift = i * bits - first_bit;  // in (-bits, 8)
            const uint32_t f = idx[i] & mask;
            v |= shift >= 0 ? (f << shift) : (f >> (-shift));
        }
        out[b] = (uint8_t)(v & 0xFFu);
    }
}

// Nearest codebook entry of flat weight i: squared distance (w - c)^2 to
// each entry of its block's codebook in fp32, the first index on ties
// (strict <, as numpy's and torch's argmin); weights at or past `total`
// (the padded tail of the last block) are 0.0.  Inputs are finite.
__device__ __forceinline__ uint32_t nearest_entry(const float* __restrict__ w, int64_t total,
                                                  const float* __restrict__ cb, int n_entries,
                                                  int64_t blk, int64_t i) {
    const float v = i < total ? w[i] : 0.f;
    const float* c = cb + blk * n_entries;
    float d = v - c[0];
    float best_d = d * d;
    uint32_t best = 0;
    for (int e = 1; e < n_entries; ++e) {
        d = v - c[e];
        const float dd = d * d;
        if (dd < best_d) {
            best_d = dd;
            best = (uint32_t)e;
        }
    }
    return best;
}

// Quantize-at-pack: one thread per group of 8 indices, i.e. `bits` whole
// bytes of the LSB-first stream (8 fields of `bits` bits), each field the
// weight's nearest entry, so the (blocks x block_size x entries) distance
// tensor of the reference's quantize_weight never exists
// (inference/pack.py:21-35).  Up to 16 entries the block's codebook stays in
// registers while consecutive indices share a block; NE (4, 8 or 16, else
// 0 = any count up to 16) fixes the compare loop's length.
template <bool kSmallNE, int NE>
__global__ __launch_bounds__(kThreads) void quantize_pack_kernel(
    const float* __restrict__ w, int64_t total, const float* __restrict__ cb, int n_entries,
    int block_size, int64_t count, int bits, uint8_t* __restrict__ out, int64_t nbytes,
    int64_t first_group) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    const int64_t groups = (count + 7) / 8;
    for (int64_t t = first_group + (int64_t)blockIdx.x * kThreads + threadIdx.x; t < groups;
         t += stride) {
        float c[16];
        int64_t cur_block = -1;
        uint64_t acc = 0;  // 8 fields, LSB first (8 * bits <= 64)
        // block of index 8t + j, advanced one index at a time (one division
        // per group, not per weight)
        int64_t blk = (8 * t) / block_size;
        int in_blk = (int)(8 * t - blk * block_size);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t i = 8 * t + j;
            if (j > 0 && ++in_blk == block_size) {
                in_blk = 0;
                ++blk;
            }
            uint32_t f = 0;
            if (i < count) {
                if (kSmallNE) {
                    const float v = i < total ? w[i] : 0.f;
                    constexpr int kE = NE ? NE : 16;
                    if (blk != cur_block) {
                        cur_block = blk;
#pragma unroll
                        for (int e = 0; e < kE; ++e) c[e] = e < n_entries ? cb[blk * n_entries + e] : 0.f;
                    }
                    float d = v - c[0];
                    float best_d = d * d;
#pragma unroll
                    for (int e = 1; e < kE; ++e) {
                        d = v - c[e];
                        const float dd = d * d;
                        if ((NE || e < n_entries) && dd < best_d) {
                            best_d = dd;
                            f = (uint32_t)e;
                        }
                    }
                } else {
                    f = nearest_entry(w, total, cb, n_entries, blk, i);
                }
            }
            acc |= (uint64_t)f << (j * bits);
        }
        // bytes bits * t .. bits * t + bits - 1 of the stream
        for (int k = 0; k < bits; ++k) {
            const int64_t ob = (int64_t)bits * t + k;
            if (ob < nbytes) out[ob] = (uint8_t)(acc >> (8 * k));
        }
    }
}

// Quantize-at-pack for the standard formats (NE = 2^BITS entries, blocks a
// multiple of 32 weights): one thread per chunk of 32 real weights, which
// lies in one block -- the block's NE entries and the 32 weights come in
// with vector loads, the nearest-entry search is the same squared-distance
// compare (first index on ties), and the 32 fields leave as BITS dwords.
template <int BITS>
__global__ __launch_bounds__(kThreads) void quantize_chunks_kernel(
    const float4* __restrict__ w, const float4* __restrict__ cb, int block_size,
    uint32_t* __restrict__ out, int64_t chunks) {
    constexpr int NE = 1 << BITS;
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    for (int64_t c = (int64_t)blockIdx.x * kThreads + threadIdx.x; c < chunks; c += stride) {
        const float4* tp = cb + (c * 32 / block_size) * (NE / 4);
        float t[NE];
#pragma unroll
        for (int q = 0; q < NE / 4; ++q) {
            const float4 u = tp[q];
            t[4 * q] = u.x;
            t[4 * q + 1] = u.y;
            t[4 * q + 2] = u.z;
            t[4 * q + 3] = u.w;
        }
        float v[32];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 u = w[8 * c + q];
            v[4 * q] = u.x;
            v[4 * q + 1] = u.y;
            v[4 * q + 2] = u.z;
            v[4 * q + 3] = u.w;
        }
        uint32_t o[BITS];
#pragma unroll
        for (int k = 0; k < BITS; ++k) o[k] = 0;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            float d = v[j] - t[0];
            float best_d = d * d;
            uint32_t f = 0;
#pragma unroll
            for (int e = 1; e < NE; ++e) {
                d = v[j] - t[e];
                const float dd = d * d;
                if (dd < best_d) {
                    best_d = dd;
                    f = (uint32_t)e;
                }
            }
            const int bit = j * BITS;
            o[bit >> 5] |= f << (bit & 31);
            if ((bit & 31) + BITS > 32) o[(bit >> 5) + 1] |= f >> (32 - (bit & 31));
        }
#pragma unroll
        for (int k = 0; k < BITS; ++k) out[c * BITS + k] = o[k];
    }
}

// Per-block quantile codebooks: cb[b][e] = quantile(w_block, q_e) with
// linear interpolation, as torch.quantile(w_block, linspace(0, 1, NE))
// (nativebit/codebook_utils.py:6-22, called per block by
// nativebit/layers.py:76): sort the block, rank = q_e * (n - 1) in fp32,
// lower = (int) rank, upper = ceil(rank), weight = rank - lower, and
// torch's lerp, which rounds once: fma(weight, hi - lo, lo) for weight < 0.5,
// else fma(weight - 1, hi - lo, hi).  The last block takes only the weights
// that exist (n = total - first).  One 64-lane workgroup per block: the
// block is sorted in LDS by a bitonic network over the next power of two
// (+inf padding), every compare-exchange of a pass on its own lane, a
// barrier between passes.  Inputs are finite.
constexpr int kCbMaxBlock = 1024;
constexpr int kCbMaxEntries = 256;
struct QuantileFractions {
    float q[kCbMaxEntries];
};

__global__ __launch_bounds__(64) void block_codebooks_kernel(
    const float* __restrict__ w, int64_t total, int64_t num_blocks, int block_size, int n_entries,
    QuantileFractions qf, float* __restrict__ cb) {
    __shared__ float v[kCbMaxBlock];
    const int lane = threadIdx.x;
    for (int64_t b = blockIdx.x; b < num_blocks; b += gridDim.x) {
        const int64_t first = b * block_size;
        const int n = (int)min((int64_t)block_size, total - first);
        int P = 1;
        while (P < n) P <<= 1;
        for (int i = lane; i < P; i += 64) v[i] = i < n ? w[first + i] : INFINITY;
        __syncthreads();
        for (int k = 2; k <= P; k <<= 1) {
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int t = lane; t < P / 2; t += 64) {
                    // pair (i, i + j) of pass (k, j)
                    const int i = ((t / j) * 2 * j) + (t % j);
                    const float a = v[i], c = v[i + j];
                    const bool up = (i & k) == 0;
                    if ((a > c) == up) {
                        v[i] = c;
                        v[i + j] = a;
                    }
                }
                __syncthreads();
            }
        }
        const float last_index = (float)(n - 1);
        for (int e = lane; e < n_entries; e += 64) {
            // each product and difference rounded on its own, as torch's
            // CPU quantile computes them: no contraction into fma here
#pragma clang fp contract(off)
            const float rank = qf.q[e] * last_index;
            const int lo = (int)rank;
            const int hi = (int)ceilf(rank);
            const float wt = rank - (float)lo;
            const float a = v[lo], c = v[hi];
            const float r = fabsf(wt) < 0.5f ? __builtin_fmaf(wt, c - a, a)
                                             : __builtin_fmaf(wt - 1.0f, c - a, c);
            cb[b * n_entries + e] = r;
        }
        __syncthreads();
    }
}

// The same codebooks for blocks of at most 16 * R weights, four blocks a
// wave: sorted value i of a block is slot i % R of lane i / R of a 16-lane
// row, so every pass of the sorting network stays within a lane or a DPP row
// (no LDS, no barrier, no ds_bpermute).  Each lane sorts its R values (odd-
// even merge sort); then lane groups of 2, 4, 8 and 16 are merged: a group's
// first pass pairs lane l with its mirror image and slot r with R - 1 - r, the
// next ones lanes 4, 2, 1 apart, the last ones slots of a lane, the smaller
// value always to the smaller index.  A pass across lanes is a DPP move and a
// three-way median with the smallest or largest key (the smaller or larger
// of the two); values are compared as integers of the same order (-0 below
// +0).  What bounds it: 302 sorting instructions per four 128-weight blocks,
// 17 us over 138 240 blocks at full issue, beside 12 us of reads.  Measured
// (6912 x 2560): see launch_block_codebooks.
__device__ __forceinline__ int sort_key(float f) {
    const int i = __float_as_int(f);
    return i ^ ((i >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float sort_value(int k) {
    return __int_as_float(k ^ ((k >> 31) & 0x7fffffff));
}

__device__ __forceinline__ int med3(int a, int b, int c) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// The value of lane l ^ X of the row (X = 1, 2, 3, 4, 7 or 15).
template <int X>
__device__ __forceinline__ int row_xor(int v) {
    if constexpr (X == 4) {   // lanes 0-3 and 8-11 take lane + 4, the others lane - 4
        const int up = __builtin_amdgcn_update_dpp(v, v, 0x104, 0xf, 0x5, false);
        return __builtin_amdgcn_update_dpp(up, v, 0x114, 0xf, 0xa, false);
    } else {
        constexpr int ctrl = X == 1 ? 0xB1 : X == 2 ? 0x4E : X == 3 ? 0x1B : X == 7 ? 0x141 : 0x140;
        return __builtin_amdgcn_mov_dpp(v, ctrl, 0xf, 0xf, false);
    }
}

__device__ __forceinline__ void order2(int& a, int& b) {
    const int lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}

// Merges sorted runs of G / 2 lanes into runs of G lanes.
template <int R, int G>
__device__ __forceinline__ void merge_lanes(int (&v)[R], int lane) {
    int o[R];
#pragma unroll
    for (int r = 0; r < R; ++r) o[r] = row_xor<G - 1>(v[R - 1 - r]);
    int c = lane & (G / 2) ? INT32_MAX : INT32_MIN;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = med3(v[r], o[r], c);
    auto apart = [&](auto dc) {
        constexpr int d = decltype(dc)::value;
        c = lane & d ? INT32_MAX : INT32_MIN;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = med3(v[r], row_xor<d>(v[r]), c);
    };
    if constexpr (G >= 16) apart(std::integral_constant<int, 4>{});
    if constexpr (G >= 8) apart(std::integral_constant<int, 2>{});
    if constexpr (G >= 4) apart(std::integral_constant<int, 1>{});
#pragma unroll
    for (int d = R / 2; d > 0; d >>= 1) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (!(r & d)) order2(v[r], v[r + d]);
    }
}

template <int R>
__global__ __launch_bounds__(kThreads) void block_codebooks_row_kernel(
    const float* __restrict__ w, int64_t total, int64_t num_blocks, int block_size, int n_entries,
    bool vec, QuantileFractions qf, float* __restrict__ cb) {
    constexpr int P = 16 * R;
    __shared__ __align__(16) int sorted[kThreads / 16][P];
    // The fractions of over 16 entries, requested once and kept here: read
    // from the arguments where they are used they are a chain of up to 16
    // loads.  With four entries a lane at once, 256 entries of 64 weights: 20953
    // weights 6.7 -> 4.8 us (a block a wave 4.2), 17.7 M 123 -> 95 us (159).
    __shared__ float fractions[kCbMaxEntries];
    static_assert(kThreads >= kCbMaxEntries, "one fraction a thread");
    const int lane = threadIdx.x & 15, row = threadIdx.x >> 4;
    const bool many = n_entries > 16;
    const float fraction = qf.q[many ? threadIdx.x : lane];   // (zeros past n_entries)
    const int64_t nrows = ((int64_t)gridDim.x * kThreads) >> 4;
    // (rows past the last block repeat it and store nothing: every lane of a
    // wave takes part in the DPP moves)
    const int64_t rounds = (num_blocks + nrows - 1) / nrows;
    for (int64_t it = 0; it < rounds; ++it) {
        const int64_t b0 = it * nrows + (((int64_t)blockIdx.x * kThreads + threadIdx.x) >> 4);
        const int64_t b = b0 < num_blocks ? b0 : num_blocks - 1;
        const int64_t first = b * block_size;
        const int n = (int)min((int64_t)block_size, total - first);
        int v[R];
        if (vec && n == P) {
#pragma unroll
            for (int q = 0; q < R / 4; ++q) {
                const float4 f = reinterpret_cast<const float4*>(w + first)[q * 16 + lane];
                v[4 * q] = sort_key(f.x);
                v[4 * q + 1] = sort_key(f.y);
                v[4 * q + 2] = sort_key(f.z);
                v[4 * q + 3] = sort_key(f.w);
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int i = r * 16 + lane;
                v[r] = sort_key(i < n ? w[first + i] : INFINITY);
            }
        }
        // the lane's own values: odd-even merge sort
#pragma unroll
        for (int p = 1; p < R; p <<= 1) {
#pragma unroll
            for (int k = p; k >= 1; k >>= 1) {
#pragma unroll
                for (int j = k % p; j + k < R; j += 2 * k) {
#pragma unroll
                    for (int i = 0; i < k; ++i) {
                        if (i + j + k < R && (i + j) / (2 * p) == (i + j + k) / (2 * p)) {
                            order2(v[i + j], v[i + j + k]);
                        }
                    }
                }
            }
        }
        merge_lanes<R, 2>(v, lane);
        merge_lanes<R, 4>(v, lane);
        merge_lanes<R, 8>(v, lane);
        merge_lanes<R, 16>(v, lane);
        // entries: a lane fetches its two order statistics through LDS (a
        // wave's LDS operations complete in issue order)
#pragma unroll
        for (int q = 0; q < R / 4; ++q) {
            *reinterpret_cast<int4*>(&sorted[row][lane * R + 4 * q]) =
                make_int4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (many && it == 0) {   // (the same in every thread of the grid)
            fractions[threadIdx.x] = fraction;
            __syncthreads();
        }
        const float last_index = (float)(n - 1);
        auto entry = [&](float q) {
            float rank, wt;
            int lo, hi;
            {
                // each product and difference rounded on its own, as torch's
                // CPU quantile computes them: no contraction into fma here
#pragma clang fp contract(off)
                rank = q * last_index;
                lo = (int)rank;
                hi = (int)ceilf(rank);
                wt = rank - (float)lo;
            }
            const float a = sort_value(sorted[row][lo]), c = sort_value(sorted[row][hi]);
            return fabsf(wt) < 0.5f ? __builtin_fmaf(wt, c - a, a)
                                    : __builtin_fmaf(wt - 1.0f, c - a, c);
        };
        if (b0 < num_blocks && !many) {
            if (lane < n_entries) cb[b * n_entries + lane] = entry(fraction);
        } else if (b0 < num_blocks) {
            int e = lane;
            for (; e + 48 < n_entries; e += 64) {   // four chains of LDS reads at once
                float r[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) r[u] = entry(fractions[e + 16 * u]);
#pragma unroll
                for (int u = 0; u < 4; ++u) cb[b * n_entries + e + 16 * u] = r[u];
            }
            for (; e < n_entries; e += 16) cb[b * n_entries + e] = entry(fractions[e]);
        }
        __builtin_amdgcn_wave_barrier();   // (the next blocks' writes stay behind these reads)
    }
}

template <bool kBF16>
__global__ __launch_bounds__(kThreads) void dequant_kernel(
    const uint8_t* __restrict__ packed, int64_t nbytes,
    const float* __restrict__ cb, void* __restrict__ w, int64_t first, int64_t total,
    int bits, int n_entries, int block_size) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    const uint32_t last = (uint32_t)(n_entries - 1);
    for (int64_t i = first + (int64_t)blockIdx.x * kThreads + threadIdx.x; i < total;
         i += stride) {
        uint32_t e = read_field(packed, nbytes, i, bits);
        e = e < last ? e : last;
        const float v = cb[(i / block_size) * n_entries + e];
        if (kBF16) {
            static_cast<bf16_bits*>(w)[i] = f32_to_bf16_rne(v);
        } else {
            static_cast<float*>(w)[i] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// chunk kernels (32 indices <-> BITS dwords)
// ---------------------------------------------------------------------------
// Field j (0..31) of a chunk: bits [j*BITS, (j+1)*BITS) of the little-endian
// dwords d; j is a constant once the callers' loops are unrolled.
template <int BITS>
__device__ __forceinline__ uint32_t chunk_field(const uint32_t (&d)[BITS], int j) {
    const int bit = j * BITS;
    const int w = bit >> 5;
    const int off = bit & 31;
    const uint32_t mask = (1u << BITS) - 1u;
    if (off + BITS > 32) return __builtin_amdgcn_alignbit(d[w + 1], d[w], off) & mask;
    return (d[w] >> off) & mask;
}

template <int BITS>
__device__ __forceinline__ void load_chunk(const uint32_t* __restrict__ packed, int64_t c,
                                           uint32_t (&d)[BITS]) {
    const uint32_t* p = packed + c * BITS;
#pragma unroll
    for (int w = 0; w < BITS; ++w) d[w] = __builtin_nontemporal_load(p + w);
}

// Stores the Q 16-byte pieces of each lane's chunk so that every store
// instruction of the wave writes 64 consecutive pieces (1 KiB): the pieces go
// through the wave's LDS area (lane pitch Q + 1 pieces) and come back in
// output order.  Lane l holds chunk c0 + l; pieces at or past `limit` (the
// end of the output, counted from dst) are not stored.  Every lane of the
// wave calls this.  A wave's LDS operations complete in issue order, so the
// fences only keep the compiler from moving the accesses.
template <int Q>
__device__ __forceinline__ void wave_store_pieces(uint4* __restrict__ lds, const uint4 (&v)[Q],
                                                  uint4* __restrict__ dst, int64_t c0,
                                                  int64_t limit, int lane) {
#pragma unroll
    for (int q = 0; q < Q; ++q) lds[lane * (Q + 1) + q] = v[q];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const int i = k * 64 + lane;  // piece of the wave's output
        const uint4 u = lds[(i / Q) * (Q + 1) + (i % Q)];
        const int64_t o = c0 * Q + i;
        if (o < limit) dst[o] = u;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Grid-stride over chunks in whole waves: the loop condition is the wave's
// first chunk, so every lane of a wave runs the same iterations (the wave
// store needs all of them); lanes past the last chunk compute on chunk 0
// and store nothing.
#define NB_CHUNK_LOOP(chunks)                                                        \
    const int lane = threadIdx.x & 63;                                               \
    const int64_t stride = (int64_t)gridDim.x * kThreads;                            \
    for (int64_t c0 = (int64_t)blockIdx.x * kThreads + (threadIdx.x & ~63); c0 < (chunks); \
         c0 += stride)

template <int BITS>
__global__ __launch_bounds__(kThreads) void unpack_chunks_kernel(
    const uint32_t* __restrict__ packed, uint4* __restrict__ out, int64_t chunks) {
    __shared__ uint4 lds[kThreads / 64][64 * 3];
    NB_CHUNK_LOOP(chunks) {
        const int64_t c = c0 + lane < chunks ? c0 + lane : 0;
        uint32_t d[BITS];
        load_chunk<BITS>(packed, c, d);
        uint32_t o[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            o[k] = chunk_field<BITS>(d, 4 * k) | (chunk_field<BITS>(d, 4 * k + 1) << 8) |
                   (chunk_field<BITS>(d, 4 * k + 2) << 16) | (chunk_field<BITS>(d, 4 * k + 3) << 24);
        }
        const uint4 v[2] = {make_uint4(o[0], o[1], o[2], o[3]), make_uint4(o[4], o[5], o[6], o[7])};
        wave_store_pieces<2>(lds[threadIdx.x >> 6], v, out, c0, 2 * chunks, lane);
    }
}

template <int BITS>
__global__ __launch_bounds__(kThreads) void pack_chunks_kernel(
    const uint4* __restrict__ idx, uint32_t* __restrict__ out, int64_t chunks) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    const uint32_t mask = (1u << BITS) - 1u;
    for (int64_t c = (int64_t)blockIdx.x * kThreads + threadIdx.x; c < chunks; c += stride) {
        const uint4 a = idx[2 * c], b = idx[2 * c + 1];
        const uint32_t in[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t o[BITS];
#pragma unroll
        for (int w = 0; w < BITS; ++w) o[w] = 0;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint32_t f = (in[j >> 2] >> (8 * (j & 3))) & mask;
            const int bit = j * BITS;
            const int w = bit >> 5;
            const int off = bit & 31;
            o[w] |= f << off;
            if (off + BITS > 32) o[w + 1] |= f >> (32 - off);
        }
        uint32_t* p = out + c * BITS;
#pragma unroll
        for (int w = 0; w < BITS; ++w) p[w] = o[w];
    }
}

// Two finite fp32 values rounded to bf16 (nearest, ties to even), packed low
// | high: gfx950 converts a pair in one instruction (v_cvt_pk_bf16_f32).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2_rne(float lo, float hi) {
    const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

// block_size % 32 == 0, so a chunk lies inside one block.
template <int BITS, bool kBF16>
__global__ __launch_bounds__(kThreads) void dequant_chunks_kernel(
    const uint32_t* __restrict__ packed, const float* __restrict__ cb, void* __restrict__ w,
    int64_t chunks, int n_entries, int block_size) {
    constexpr int Q = kBF16 ? 4 : 8;  // 16-byte pieces per chunk
    __shared__ uint4 lds[kThreads / 64][64 * (Q + 1)];
    const uint32_t last = (uint32_t)(n_entries - 1);
    NB_CHUNK_LOOP(chunks) {
        const int64_t c = c0 + lane < chunks ? c0 + lane : 0;
        uint32_t d[BITS];
        load_chunk<BITS>(packed, c, d);
        const float* tab = cb + (c * 32 / block_size) * n_entries;
        float v[32];
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint32_t e = chunk_field<BITS>(d, j);
            v[j] = tab[e < last ? e : last];
        }
        uint4 pc[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if (kBF16) {
                uint32_t h[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) h[k] = pack_bf16x2_rne(v[8 * q + 2 * k], v[8 * q + 2 * k + 1]);
                pc[q] = make_uint4(h[0], h[1], h[2], h[3]);
            } else {
                pc[q] = make_uint4(__float_as_uint(v[4 * q]), __float_as_uint(v[4 * q + 1]),
                                   __float_as_uint(v[4 * q + 2]), __float_as_uint(v[4 * q + 3]));
            }
        }
        wave_store_pieces<Q>(lds[threadIdx.x >> 6], pc, static_cast<uint4*>(w), c0, Q * chunks,
                             lane);
    }
}

// The same for the formats with 2^BITS entries (4, 8 or 16): each lane copies
// its block's entries into a column of its own of the wave's LDS table (entry
// e of lane l at byte 256 e + 4 l, bf16 entries rounded once there), so a
// lookup is two VALU instructions and a conflict-free LDS read.  The
// lookups of the kernel above are loads whose 64 lanes read up to 64 tables:
// the address unit, not memory, was its limit (2560 x 6912, 16 entries, BS 64,
// to bf16: 20.9 us for 62 MB, now 13.3; 6912 x 2560, 8 entries, to fp32: 23.2 us
// for 82 MB, now 17.7).
template <int BITS, bool kBF16>
__global__ __launch_bounds__(kThreads) void dequant_tables_kernel(
    const uint32_t* __restrict__ packed, const float4* __restrict__ cb, void* __restrict__ w,
    int64_t chunks, int block_size) {
    constexpr int Q = kBF16 ? 4 : 8;  // 16-byte pieces per chunk
    constexpr int NE = 1 << BITS;
    __shared__ __align__(NE * 256) float tables[kThreads / 64][NE * 64];   // (read as float)
    __shared__ uint4 lds[kThreads / 64][64 * (Q + 1)];
    float* tab = tables[threadIdx.x >> 6];
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)tab +
                          4 * (threadIdx.x & 63);
    NB_CHUNK_LOOP(chunks) {
        const int64_t c = c0 + lane < chunks ? c0 + lane : 0;
        uint32_t d[BITS];
        load_chunk<BITS>(packed, c, d);
        const float4* tp = cb + (c * 32 / block_size) * (NE / 4);
        float4 t[NE / 4];
#pragma unroll
        for (int i = 0; i < NE / 4; ++i) t[i] = tp[i];
#pragma unroll
        for (int i = 0; i < NE / 4; ++i) {
            const float e[4] = {t[i].x, t[i].y, t[i].z, t[i].w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                tab[(4 * i + k) * 64 + lane] =
                    kBF16 ? __uint_as_float((uint32_t)f32_to_bf16_rne(e[k])) : e[k];
            }
        }
        float v[4][8];
        lookup8<BITS, 8, 0>(d, base, v[0], std::make_integer_sequence<int, 8>{});
        lookup8<BITS, 8, 8>(d, base, v[1], std::make_integer_sequence<int, 8>{});
        lookup8<BITS, 8, 16>(d, base, v[2], std::make_integer_sequence<int, 8>{});
        lookup8<BITS, 8, 24>(d, base, v[3], std::make_integer_sequence<int, 8>{});
        uint4 pc[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            uint32_t h[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (kBF16) {
                    h[k] = __float_as_uint(v[q][2 * k]) | (__float_as_uint(v[q][2 * k + 1]) << 16);
                } else {
                    h[k] = __float_as_uint(v[q >> 1][4 * (q & 1) + k]);
                }
            }
            pc[q] = make_uint4(h[0], h[1], h[2], h[3]);
        }
        wave_store_pieces<Q>(lds[threadIdx.x >> 6], pc, static_cast<uint4*>(w), c0, Q * chunks,
                             lane);
    }
}

// f(std::integral_constant<int, bits>) for bits 1..8.
template <typename F>
void with_bits(int bits, F&& f) {
    switch (bits) {
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
    }
}

inline bool is_aligned(const void* p, uintptr_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; }

}  // namespace

int launch_unpack(const uint8_t* packed, uint8_t* out, int64_t count, int bits,
                  hipStream_t stream) {
    if (count == 0) return NB_OK;
    const int64_t nbytes = packed_nbytes(count, bits);
    int64_t first = 0;
    if (is_aligned(packed, 4) && is_aligned(out, 16)) {
        const int64_t chunks = count / 32;
        if (chunks > 0) {
            with_bits(bits, [&](auto B) {
                hipLaunchKernelGGL(unpack_chunks_kernel<decltype(B)::value>, dim3(grid_for(chunks)),
                                   dim3(kThreads), 0, stream,
                                   reinterpret_cast<const uint32_t*>(packed),
                                   reinterpret_cast<uint4*>(out), chunks);
            });
            first = chunks * 32;
        }
    }
    if (first < count) {
        hipLaunchKernelGGL(unpack_kernel, dim3(grid_for(count - first)), dim3(kThreads), 0,
                           stream, packed, nbytes, out, first, count, bits);
    }
    return check_launch("nb_unpack");
}

int launch_pack(const uint8_t* idx, uint8_t* out, int64_t count, int bits,
                hipStream_t stream) {
    const int64_t nbytes = packed_nbytes(count, bits);
    if (nbytes == 0) return NB_OK;
    // chunk c writes stream bytes [4 * bits * c, 4 * bits * (c + 1)) from
    // indices [32c, 32c + 32); the per-byte kernel writes the rest, padding
    // included
    int64_t first_byte = 0;
    if (is_aligned(idx, 16) && is_aligned(out, 4)) {
        const int64_t chunks = count / 32;
        if (chunks > 0) {
            with_bits(bits, [&](auto B) {
                hipLaunchKernelGGL(pack_chunks_kernel<decltype(B)::value>, dim3(grid_for(chunks)),
                                   dim3(kThreads), 0, stream,
                                   reinterpret_cast<const uint4*>(idx),
                                   reinterpret_cast<uint32_t*>(out), chunks);
            });
            first_byte = chunks * 4 * bits;
        }
    }
    if (first_byte < nbytes) {
        hipLaunchKernelGGL(pack_kernel, dim3(grid_for(nbytes - first_byte)), dim3(kThreads), 0,
                           stream, idx, count, bits, out, first_byte, nbytes);
    }
    return check_launch("nb_pack");
}

int launch_quantize_pack(const float* w, int64_t total, const float* codebook,
                         int64_t num_blocks, int n_entries, int block_size, int bits,
                         uint8_t* out, hipStream_t stream) {
    const int64_t count = num_blocks * block_size;
    const int64_t nbytes = packed_nbytes(count, bits);
    if (nbytes == 0) return NB_OK;
    // chunks of 32 real weights in the standard formats; the general kernel
    // takes the remaining groups (the tail and the zero-padded weights)
    int64_t first_group = 0;
    if ((n_entries == 4 || n_entries == 8 || n_entries == 16) && n_entries == (1 << bits) &&
        block_size % 32 == 0 && is_aligned(w, 16) && is_aligned(codebook, 16) &&
        is_aligned(out, 4)) {
        const int64_t chunks = total / 32;
        if (chunks > 0) {
            auto chunk = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(grid_for(chunks)), dim3(kThreads), 0, stream,
                                   reinterpret_cast<const float4*>(w),
                                   reinterpret_cast<const float4*>(codebook), block_size,
                                   reinterpret_cast<uint32_t*>(out), chunks);
            };
            if (bits == 2) chunk(quantize_chunks_kernel<2>);
            if (bits == 3) chunk(quantize_chunks_kernel<3>);
            if (bits == 4) chunk(quantize_chunks_kernel<4>);
            first_group = chunks * 4;
        }
    }
    const int64_t groups = (count + 7) / 8;
    if (first_group >= groups) return check_launch("nb_quantize_pack");
    const int grid = grid_for(groups - first_group);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, stream, w, total, codebook,
                           n_entries, block_size, count, bits, out, nbytes, first_group);
    };
    switch (n_entries) {
        case 4: go(quantize_pack_kernel<true, 4>); break;
        case 8: go(quantize_pack_kernel<true, 8>); break;
        case 16: go(quantize_pack_kernel<true, 16>); break;
        default:
            if (n_entries < 16) {
                go(quantize_pack_kernel<true, 0>);
            } else {
                go(quantize_pack_kernel<false, 0>);
            }
    }
    return check_launch("nb_quantize_pack");
}

int launch_block_codebooks(const float* w, int64_t total, int64_t num_blocks, int block_size,
                           int n_entries, const float* q, float* cb, hipStream_t stream) {
    if (num_blocks == 0) return NB_OK;
    QuantileFractions qf;
    for (int e = 0; e < kCbMaxEntries; ++e) qf.q[e] = e < n_entries ? q[e] : 0.f;
    if (block_size <= 256) {
        // 6912 x 2560, 8 entries, cold weights: 90 us with one block a wave
        // sorted by ds_bpermute shuffles, 28 us with four (70.8 MB read: 2.5
        // TB/s)
        const int64_t want = (num_blocks + kThreads / 16 - 1) / (kThreads / 16);
        const int64_t cap = (int64_t)device_cu_count() * 8;
        const int grid = (int)(want < cap ? want : cap);
        const bool vec = is_aligned(w, 16) && block_size % 4 == 0;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, stream, w, total,
                               num_blocks, block_size, n_entries, vec, qf, cb);
        };
        if (block_size <= 64) {
            go(block_codebooks_row_kernel<4>);
        } else if (block_size <= 128) {
            go(block_codebooks_row_kernel<8>);
        } else {
            go(block_codebooks_row_kernel<16>);
        }
        return check_launch("nb_block_codebooks");
    }
    int64_t grid = num_blocks;
    const int64_t cap = (int64_t)device_cu_count() * 32;
    if (grid > cap) grid = cap;
    hipLaunchKernelGGL(block_codebooks_kernel, dim3((int)grid), dim3(64), 0, stream, w, total,
                       num_blocks, block_size, n_entries, qf, cb);
    return check_launch("nb_block_codebooks");
}

int launch_dequant(const uint8_t* packed, const float* codebook, void* w,
                   int w_dtype, int64_t total, int64_t num_blocks, int bits,
                   int n_entries, int block_size, hipStream_t stream) {
    if (total == 0) return NB_OK;
    (void)num_blocks;  // validated by the caller: num_blocks * block_size >= total
    // Fields of indices < total lie inside the first packed_nbytes(total)
    // bytes, so that is all the kernels may touch.
    const int64_t nbytes = packed_nbytes(total, bits);
    const bool bf16 = w_dtype == NB_BF16;
    int64_t first = 0;
    if (block_size % 32 == 0 && is_aligned(packed, 4) && is_aligned(w, 16)) {
        const int64_t chunks = total / 32;
        if (chunks > 0) {
            with_bits(bits, [&](auto B) {
                constexpr int kB = decltype(B)::value;
                if constexpr (kB >= 2 && kB <= 4) {
                    // (one wave's worth to bf16 waits longer for its table than for
                    // its lookups: 1024 weights of 16 entries 2.6 us against 2.3;
                    // 4096 are even, 8192 2.9-3.0 against 3.1-3.8)
                    if (n_entries == (1 << kB) && is_aligned(codebook, 16) &&
                        !(bf16 && chunks <= 64)) {
                        auto tables = bf16 ? dequant_tables_kernel<kB, true>
                                           : dequant_tables_kernel<kB, false>;
                        hipLaunchKernelGGL(tables, dim3(grid_for(chunks)), dim3(kThreads), 0, stream,
                                           reinterpret_cast<const uint32_t*>(packed),
                                           reinterpret_cast<const float4*>(codebook), w, chunks,
                                           block_size);
                        return;
                    }
                }
                auto kernel = bf16 ? dequant_chunks_kernel<kB, true> : dequant_chunks_kernel<kB, false>;
                hipLaunchKernelGGL(kernel, dim3(grid_for(chunks)), dim3(kThreads), 0, stream,
                                   reinterpret_cast<const uint32_t*>(packed), codebook, w, chunks,
                                   n_entries, block_size);
            });
            first = chunks * 32;
        }
    }
    if (first < total) {
        auto kernel = bf16 ? dequant_kernel<true> : dequant_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3(grid_for(total - first)), dim3(kThreads), 0, stream,
                           packed, nbytes, codebook, w, first, total, bits, n_entries,
                           block_size);
    }
    return check_launch("nb_dequant");
}

}  // namespace nb
