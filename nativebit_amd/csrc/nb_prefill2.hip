// Prefill contraction with a packed weight, large tiles (gfx950).
//
//   Y[m][n] = sum_k X[m][k] * bf16(W[n][k]),   W 3-bit / 8-entry / block-128
//
// The reference computes this as unpack + gather + a dense matmul that
// materialises W on every call (inference/triton_kernel.py:258-275; in bf16,
// inference/eval_ppl.py:149-174).  Here a 512-thread workgroup owns a BN x
// BM tile of Y^T (BN = 256 or 128 outputs x BM = 256, 128 or 64 tokens,
// chosen per launch by estimated time) and walks K in steps of 64:
//
//   * the X slice (BM tokens x 64 bf16) arrives by global_load_lds_dwordx4
//     (eight rows per instruction), 16-byte chunk c of row r in LDS slot
//     c ^ (r & 7), so that eight consecutive rows read one chunk from eight
//     different bank groups;
//   * the W slice (BN rows x 64 weights: 24 index bytes per row, the codebook
//     of the row's block) is loaded into registers two steps ahead; each
//     thread turns half a row (32 indices) into bf16 with v_perm_b32 lookups
//     into the block's codebook byte planes and stores it with the same
//     swizzle;
//   * eight waves (2 x 4) each own a (BN/4) x (BM/2) sub-tile of 16 x 16
//     v_mfma_f32_16x16x32_bf16 tiles with W as the A operand and X as B, so
//     a lane's accumulator holds four consecutive outputs n of one token m
//     and the epilogue stores them as one vector;
//   * two LDS stages and one barrier per step: while a step's MFMAs run, the
//     next step's X slice is in flight and its W slice is dequantized, and
//     the two waves of each SIMD overlap one's MFMAs with the other's
//     dequantization and LDS reads;
//   * a one-dimensional grid whose workgroups (dealt to the 8 XCDs in turn)
//     take tiles XCD by XCD in contiguous runs, so an XCD's L2 holds the X
//     tiles of one or two token blocks rather than of all of them.
// Weights are the codebook entries rounded to bf16 (RNE), as the bf16 path;
// accumulation is fp32.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "nb_device.h"
#include "nb_internal.h"

namespace nb {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

// waves per workgroup: 8 (two per SIMD) or 4 (one per SIMD, 128 x 128 per wave)
#ifndef NB_PREFILL_WAVES
#define NB_PREFILL_WAVES 8
#endif
constexpr int kBK = 64;            // K per step: half a codebook block
constexpr int kRowBytes = kBK * 2; // bf16 bytes of one row of a slice

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
    bf16x2_t v;
    v.x = (__bf16)lo;
    v.y = (__bf16)hi;
    return __builtin_bit_cast(uint32_t, v);
}

// 8 bf16 weights (natural order) of one 24-bit index group from the byte
// planes of the block's codebook: two selectors of four 3-bit indices, four
// v_perm_b32 lookups, two interleaves per bf16 pair.
__device__ __forceinline__ u32x4_t lookup8(uint32_t g, uint32_t lo0, uint32_t lo1, uint32_t hi0,
                                           uint32_t hi1) {
    const uint32_t h = (g & 0xfffu) | ((g << 4) & 0x0fff0000u);  // i0-3 low half, i4-7 high
    const uint32_t sa = (h & 0x00070007u) | ((h << 5) & 0x07000700u);          // i0 i1 i4 i5
    const uint32_t sb = ((h >> 6) & 0x00070007u) | ((h >> 1) & 0x07000700u);   // i2 i3 i6 i7
    const uint32_t la = __builtin_amdgcn_perm(lo1, lo0, sa);
    const uint32_t ha = __builtin_amdgcn_perm(hi1, hi0, sa);
    const uint32_t lb = __builtin_amdgcn_perm(lo1, lo0, sb);
    const uint32_t hb = __builtin_amdgcn_perm(hi1, hi0, sb);
    u32x4_t w;
    w.x = __builtin_amdgcn_perm(ha, la, 0x05010400u);  // i0 i1
    w.y = __builtin_amdgcn_perm(hb, lb, 0x05010400u);  // i2 i3
    w.z = __builtin_amdgcn_perm(ha, la, 0x07030602u);  // i4 i5
    w.w = __builtin_amdgcn_perm(hb, lb, 0x07030602u);  // i6 i7
    return w;
}

// LDS byte offset of 16-byte chunk c (0..7) of slice row r.
__device__ __forceinline__ uint32_t swz(int r, int c) {
    return (uint32_t)(r * kRowBytes + ((c ^ (r & 7)) << 4));
}

__device__ __forceinline__ void dma16(uint32_t lds, const void* src) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds), "v"(src)
                 : "memory", "m0");
}

template <typename T>
__device__ __forceinline__ uint32_t lds_addr(T* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) T*)p;
}

struct Prefill2Args {
    const uint16_t* x;
    int64_t ldx;
    const uint8_t* packed;
    const float* codebook;
    void* y;
    int64_t ldy;
    int y_dtype;
    int M, N, K;
    int ksplit;   // K ranges per output tile (1: the whole of K)
    float* part;  // ksplit > 1: fp32 partial products [ksplit][M][N], else null
};

// Tile of the calling workgroup.  Workgroups are dealt to the 8 XCDs in
// turn (workgroup g to XCD g % 8), each XCD with its own L2: XCD x takes a
// contiguous run of the tiles in (token tile, output tile) order, so its
// workgroups share one or two token tiles of X in its L2 rather than all of
// them.  With a K split, virtual tile v is K range v / ntiles of output
// tile v % ntiles, so an XCD's run holds neighbouring tiles of one K range
// (which share their X slices).
struct TileOf {
    int n0, m0;       // first output and first token of the tile
    int ks;           // K range of this workgroup
    int s0, nsteps;   // its K steps: [s0, s0 + nsteps) of the K / STEPK
};

template <int BM, int BN, int STEPK>
__device__ __forceinline__ TileOf tile_of(const Prefill2Args& a) {
    const int nn = (a.N + BN - 1) / BN;
    const int ntiles = nn * ((a.M + BM - 1) / BM);
    const int T = gridDim.x, g = blockIdx.x, full = T / 8, rem = T % 8, x = g % 8;
    const int v = x * full + min(x, rem) + g / 8;
    TileOf t;
    t.ks = v / ntiles;
    const int tile = v - t.ks * ntiles;
    t.n0 = (tile % nn) * BN;
    t.m0 = (tile / nn) * BM;
    t.s0 = (int)((int64_t)t.ks * (a.K / STEPK) / a.ksplit);
    t.nsteps = (int)((int64_t)(t.ks + 1) * (a.K / STEPK) / a.ksplit) - t.s0;
    return t;
}

// Epilogue: D fragment (i, j) of a wave whose A sub-tiles start at output
// nb and B sub-tiles at token mb -- the lane holds outputs
// nb + 16 i + 4 fq .. + 3 for token mb + 16 j + fr.  With a K split, the
// fp32 partial products go to plane ks of `part` (row stride N), summed by
// prefill_reduce_kernel.
template <int TI, int TJ>
__device__ __forceinline__ void store_tile(const Prefill2Args& a, const f32x4_t (&acc)[TI][TJ],
                                           int nb, int mb, int fq, int fr, int ks) {
    const bool partial = a.part != nullptr;
    const int y_dtype = partial ? NB_F32 : a.y_dtype;
    void* const yb = partial ? static_cast<void*>(a.part + (int64_t)ks * a.M * a.N) : a.y;
    const int64_t ldy = partial ? a.N : a.ldy;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int n = nb + i * 16 + fq * 4;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int m = mb + j * 16 + fr;
            if (m >= a.M) continue;
            const f32x4_t v = acc[i][j];
            if (y_dtype == NB_BF16) {
                bf16_bits* yp = static_cast<bf16_bits*>(yb) + (int64_t)m * ldy + n;
                // one 8-byte store where the four outputs exist and the
                // address allows it (y may be any 2-byte-aligned view)
                if (n + 3 < a.N && (reinterpret_cast<uintptr_t>(yp) & 7) == 0) {
                    u32x2_t p;
                    p.x = (uint32_t)f32_to_bf16_rne(v.x) | ((uint32_t)f32_to_bf16_rne(v.y) << 16);
                    p.y = (uint32_t)f32_to_bf16_rne(v.z) | ((uint32_t)f32_to_bf16_rne(v.w) << 16);
                    *reinterpret_cast<u32x2_t*>(yp) = p;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < a.N) yp[e] = f32_to_bf16_rne(v[e]);
                }
            } else {
                float* yp = static_cast<float*>(yb) + (int64_t)m * ldy + n;
                if (n + 3 < a.N && (reinterpret_cast<uintptr_t>(yp) & 15) == 0) {
                    *reinterpret_cast<f32x4_t*>(yp) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < a.N) yp[e] = v[e];
                }
            }
        }
    }
}

// One thread's share of a W slice: 12 index bytes (32 weights) per half
// row it takes (H = 1 or 2) and the codebook of the row's block.  Each
// 12-byte piece is one register tuple, so its loads land in place without
// copies.
template <int H>
struct WRegs {
    u32x4_t d[H];  // x, y, z of d[h]: the index bytes of half h
    u32x4_t c0, c1;
};

// kSplit: fp32 activations against the exact fp32 weights as three bf16
// products, x = hi + lo and W = hi + lo: hi.hi + hi.lo + lo.hi.  A step is 32
// of K instead of 64, an LDS row its 32 hi parts (chunks 0-3) and its 32 lo
// parts (chunks 4-7); x arrives already split, in that order (split_bf16_
// kernel).  Of the two threads of a W row one dequantizes the hi parts
// (entries rounded to bf16), the other the lo parts (what that rounding left,
// rounded to bf16).  The fragments of a step then feed three MFMAs instead of
// two, so this form reads less LDS per MFMA than the bf16 one.  Measured
// against three passes of the bf16 kernel that added to y (and a residual
// codebook made per call), with the fastest plans: 7680 x 2560 at M = 128 / 500
// / 2048 36 / 74 / 232 us (73 / 127 / 298), 2560 x 6912 34 / 70 / 234 us (74 /
// 144 / 308); 4.301e-6 from fp64 (4.295e-6: the three products share a sum).
template <int BM, int BN, int WAVES, bool kSplit>
__global__ __launch_bounds__(64 * WAVES) void prefill2_kernel(Prefill2Args a) {
    constexpr int kThreads = 64 * WAVES;
    constexpr int WGM = WAVES >= 16 ? 4 : 2;  // waves along the tokens
    constexpr int WGN = WAVES / WGM;     // waves along the outputs
    constexpr int WN = BN / WGN;         // outputs per wave (A operand rows)
    constexpr int WM = BM / WGM;         // tokens per wave (B operand rows)
    constexpr int TI = WN / 16, TJ = WM / 16;
    constexpr int kXBytes = BM * kRowBytes, kWBytes = BN * kRowBytes;
    constexpr int kStage = kXBytes + kWBytes;
    constexpr int kXLoads = BM / (8 * WAVES);  // dma16 per wave per step (8 rows each)
    // threads per W row: 2 (half a row each) or 1; with more threads than
    // two per row, the first 2 BN threads dequantize
    constexpr int TPR = kThreads >= 2 * BN ? 2 : kThreads / BN;
    constexpr int H = 2 / TPR;           // 32-weight halves per thread
    constexpr bool kAllDeq = kThreads <= 2 * BN;
    static_assert(TPR == 1 || TPR == 2, "one or two threads per W row");
    static_assert(!kSplit || TPR == 2, "one thread for the hi parts, one for the lo parts");
    constexpr int kStepK = kSplit ? kBK / 2 : kBK;
    using WR = WRegs<H>;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const TileOf t = tile_of<BM, BN, kStepK>(a);
    const int n0 = t.n0, m0 = t.m0, ks = t.ks, s0 = t.s0, nsteps = t.nsteps;
    const int bpr = a.K / 128;
    const uint32_t base = lds_addr(smem);

    // X slice: instruction i of wave w covers slice rows 8 (kXLoads w + i)
    // .. +7; lane l fills slot l & 7 of row 8 (...) + (l >> 3)
    auto load_x = [&](int step, int stage) {
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) {
            const int r0 = (wave * kXLoads + i) * 8;
            const int r = r0 + (lane >> 3);
            const int c = (lane & 7) ^ (r & 7);
            const int gm = min(m0 + r, a.M - 1);
            const uint16_t* src = a.x + (int64_t)gm * a.ldx + (int64_t)(s0 + step) * kBK + c * 8;
            dma16(__builtin_amdgcn_readfirstlane(base + stage * kStage + r0 * kRowBytes), src);
        }
    };
    // W slice: thread t takes halves h0 .. h0 + H - 1 of row t / TPR
    const int wr = (tid / TPR) % BN, h0 = (tid % TPR) * H;
    const int gn = min(n0 + wr, a.N - 1);
    const bool deq = kAllDeq || tid < 2 * BN;
    auto load_w = [&](int step, WR& w) {
        if (!deq) return;
        constexpr int kStepsLog = kSplit ? 2 : 1;   // steps a block
        const int64_t blk = (int64_t)gn * bpr + ((s0 + step) >> kStepsLog);
        const int in_blk = (s0 + step) & ((1 << kStepsLog) - 1);
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const uint32_t* ip = reinterpret_cast<const uint32_t*>(
                a.packed + blk * 48 + (kSplit ? in_blk * 12 : in_blk * 24 + (h0 + h) * 12));
            w.d[h].x = ip[0];
            w.d[h].y = ip[1];
            w.d[h].z = ip[2];
        }
        const u32x4_t* cp = reinterpret_cast<const u32x4_t*>(a.codebook + blk * 8);
        w.c0 = cp[0];
        w.c1 = cp[1];
    };
    auto store_w = [&](int stage, const WR& w) {
        if (!deq) return;
        uint32_t q0 = pack_bf16x2(__uint_as_float(w.c0.x), __uint_as_float(w.c0.y));
        uint32_t q1 = pack_bf16x2(__uint_as_float(w.c0.z), __uint_as_float(w.c0.w));
        uint32_t q2 = pack_bf16x2(__uint_as_float(w.c1.x), __uint_as_float(w.c1.y));
        uint32_t q3 = pack_bf16x2(__uint_as_float(w.c1.z), __uint_as_float(w.c1.w));
        if constexpr (kSplit) {
            // entry - bf16(entry), exact in fp32
            auto rest = [](uint32_t q, uint32_t a0, uint32_t a1) {
                return pack_bf16x2(__uint_as_float(a0) - __uint_as_float(q << 16),
                                   __uint_as_float(a1) - __uint_as_float(q & 0xffff0000u));
            };
            const bool lo = h0 != 0;
            q0 = lo ? rest(q0, w.c0.x, w.c0.y) : q0;
            q1 = lo ? rest(q1, w.c0.z, w.c0.w) : q1;
            q2 = lo ? rest(q2, w.c1.x, w.c1.y) : q2;
            q3 = lo ? rest(q3, w.c1.z, w.c1.w) : q3;
        }
        const uint32_t lo0 = __builtin_amdgcn_perm(q1, q0, 0x06040200u);
        const uint32_t hi0 = __builtin_amdgcn_perm(q1, q0, 0x07050301u);
        const uint32_t lo1 = __builtin_amdgcn_perm(q3, q2, 0x06040200u);
        const uint32_t hi1 = __builtin_amdgcn_perm(q3, q2, 0x07050301u);
        unsigned char* wt = smem + stage * kStage + kXBytes;
#pragma unroll
        for (int h = 0; h < H; ++h) {
            // the four 24-bit groups of the half's 96 index bits
            const u32x4_t d = w.d[h];
            const uint32_t g[4] = {d.x & 0xffffffu, __builtin_amdgcn_alignbit(d.y, d.x, 24),
                                   __builtin_amdgcn_alignbit(d.z, d.y, 16), d.z >> 8};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                *reinterpret_cast<u32x4_t*>(wt + swz(wr, (h0 + h) * 4 + j)) =
                    lookup8(g[j], lo0, lo1, hi0, hi1);
            }
        }
    };

    const int wm = wave / WGN, wn = wave % WGN;
    const int fr = lane & 15, fq = lane >> 4;
    f32x4_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    WR wq0, wq1;  // W slices of even / odd steps (named, so they stay in registers)
    load_x(0, 0);
    load_w(0, wq0);
    if (nsteps > 1) load_w(1, wq1);
    store_w(0, wq0);
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    __syncthreads();

    // One step on LDS stage CUR (= step & 1): the W slice of step + 2 goes
    // into the registers this step's came from (already in LDS) and the next
    // X slice is requested, the MFMAs run, then the next step's W slice
    // (loaded one step ago) is dequantized into the other stage.
    auto run_step = [&](int step, auto cur_c, WR& mine, WR& next) {
        constexpr int cur = decltype(cur_c)::value;
        // The next step's W slice was loaded a step ago and the previous
        // step ended with vmcnt(0): passing its registers through an empty
        // asm statement here puts the compiler's wait for them at this point
        // (where it costs nothing), so the dequantization below may sit
        // among the MFMAs without a wait that would also drain the X slice
        // requested next (the compiler cannot see that load).
#pragma unroll
        for (int h = 0; h < H; ++h) asm volatile("" : "+v"(next.d[h]));
        asm volatile("" : "+v"(next.c0), "+v"(next.c1));
        if (step + 2 < nsteps) load_w(step + 2, mine);
        if (step + 1 < nsteps) load_x(step + 1, cur ^ 1);
        const unsigned char* xt = smem + cur * kStage;
        const unsigned char* wt = xt + kXBytes;
        // The fragment reads and MFMAs are written out where they are used:
        // through helpers that take the fragment arrays by reference the
        // compiler puts all twelve reads before the first MFMA of a half step
        // (13824 x 2560 at M = 2048 173 us against 171).
        auto w_frag = [&](int i, int c) {   // 16-byte chunk c of the wave's W rows
            return *reinterpret_cast<const u32x4_t*>(wt + swz(wn * WN + i * 16 + fr, c));
        };
        auto x_frag = [&](int j, int c) {
            return *reinterpret_cast<const u32x4_t*>(xt + swz(wm * WM + j * 16 + fr, c));
        };
        auto mfma = [&](u32x4_t w, u32x4_t x, f32x4_t& sum) {
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                          __builtin_bit_cast(bf16x8_t, x), sum, 0,
                                                          0, 0);
        };
        if constexpr (kSplit) {
            const int ch = fq, cl = 4 + fq;
            u32x4_t wv[TI], xv[TJ], wlo[TI], xlo[TJ];
#pragma unroll
            for (int i = 0; i < TI; ++i) wv[i] = w_frag(i, ch);
#pragma unroll
            for (int j = 0; j < TJ; ++j) xv[j] = x_frag(j, ch);
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) mfma(wv[i], xv[j], acc[i][j]);
#pragma unroll
            for (int i = 0; i < TI; ++i) wlo[i] = w_frag(i, cl);
            if (step + 1 < nsteps) store_w(cur ^ 1, next);
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) mfma(wlo[i], xv[j], acc[i][j]);
#pragma unroll
            for (int j = 0; j < TJ; ++j) xlo[j] = x_frag(j, cl);
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) mfma(wv[i], xlo[j], acc[i][j]);
        } else {
            auto half_step = [&](int half) {   // 32 of the step's 64 K
                const int c = half * 4 + fq;
                u32x4_t av[TI], bv[TJ];
#pragma unroll
                for (int i = 0; i < TI; ++i) av[i] = w_frag(i, c);
#pragma unroll
                for (int j = 0; j < TJ; ++j) bv[j] = x_frag(j, c);
#pragma unroll
                for (int i = 0; i < TI; ++i)
#pragma unroll
                    for (int j = 0; j < TJ; ++j) mfma(av[i], bv[j], acc[i][j]);
            };
            half_step(0);
            if (step + 1 < nsteps) store_w(cur ^ 1, next);
            half_step(1);
        }
        // the next X slice (direct-to-LDS, not tracked by the compiler) must
        // be in LDS before the barrier; the W loads of step + 2, issued
        // before it, have had the whole step to arrive
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        __syncthreads();
    };
    for (int step = 0; step < nsteps; step += 2) {
        run_step(step, std::integral_constant<int, 0>{}, wq0, wq1);
        if (step + 1 < nsteps) run_step(step + 1, std::integral_constant<int, 1>{}, wq1, wq0);
    }

    store_tile<TI, TJ>(a, acc, n0 + wn * WN, m0 + wm * WM, fq, fr, ks);
}

// y[m][n] = sum over k ranges s = 0, 1, ... of part[s][m][n] (in that
// order, so the result does not depend on which workgroup finished first),
// converted to y's dtype.  Four consecutive outputs per thread where the
// rows allow it.
__global__ __launch_bounds__(256) void prefill_reduce_kernel(const float* __restrict__ part,
                                                             int S, int M, int N, void* y,
                                                             int y_dtype, int64_t ldy) {
    const int64_t plane = (int64_t)M * N;
    // four outputs a thread where every row starts on a 4-output boundary
    // of both part and y (rows of 4k outputs, bases aligned for the vector
    // width: 16 bytes for part and fp32 y, 8 for bf16 y)
    const uintptr_t y_align = y_dtype == NB_BF16 ? 7 : 15;
    const bool vec = ((N | ldy) & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & y_align) == 0 &&
                     (reinterpret_cast<uintptr_t>(part) & 15) == 0;
    const int64_t total = vec ? plane / 4 : plane;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * 256) {
        if (vec) {
            const int64_t e = 4 * i, m = e / N, n = e - m * N;
            f32x4_t v = *reinterpret_cast<const f32x4_t*>(part + e);
            for (int k = 1; k < S; ++k) v += *reinterpret_cast<const f32x4_t*>(part + k * plane + e);
            if (y_dtype == NB_BF16) {
                u32x2_t p;
                p.x = (uint32_t)f32_to_bf16_rne(v.x) | ((uint32_t)f32_to_bf16_rne(v.y) << 16);
                p.y = (uint32_t)f32_to_bf16_rne(v.z) | ((uint32_t)f32_to_bf16_rne(v.w) << 16);
                *reinterpret_cast<u32x2_t*>(static_cast<bf16_bits*>(y) + m * ldy + n) = p;
            } else {
                *reinterpret_cast<f32x4_t*>(static_cast<float*>(y) + m * ldy + n) = v;
            }
        } else {
            const int64_t m = i / N, n = i - m * N;
            float v = part[i];
            for (int k = 1; k < S; ++k) v += part[k * plane + i];
            if (y_dtype == NB_BF16) {
                static_cast<bf16_bits*>(y)[m * ldy + n] = f32_to_bf16_rne(v);
            } else {
                static_cast<float*>(y)[m * ldy + n] = v;
            }
        }
    }
}

struct PrefillPlan {
    int BM, BN, S;
};

// What a tile costs, in microseconds: `step[c - 1]` a K step of 64 with c of
// its workgroups resident on a CU (as many as its LDS allows), `start` from a
// workgroup's launch to its first step and from its last to its end.  Fitted
// to about 1900 measured plans on MI355X (six layer shapes from 1024 x 4096 to
// 13824 x 2560, M = 32 .. 2048, every tile, S = 1 .. 16; mean error 6 %).
struct TileCost {
    int BM, BN, resident;
    float start, step[3];
};
constexpr TileCost kBf16Tiles[] = {{256, 256, 1, 5.9f, {1.71f}},
                                   {256, 128, 1, 3.4f, {1.09f}},
                                   {128, 128, 2, 3.3f, {0.74f, 1.15f}},
                                   {64, 128, 3, 2.7f, {0.57f, 0.91f, 1.42f}}};
// three products (two steps of 32 per 64 of K; they spill at 256 x 256);
// fitted to 283 plans (four layer shapes, M = 17 .. 2048, mean error 3.4 %)
constexpr TileCost kF32Tiles[] = {{256, 128, 1, 0.0f, {2.63f}},
                                  {128, 128, 2, 0.9f, {1.73f, 2.65f}},
                                  {64, 128, 2, 2.2f, {1.25f, 1.88f}}};
constexpr int kMinSplitSteps = 4;

inline int64_t grid_of(int M, int N, int bm, int bn) {
    return (int64_t)((N + bn - 1) / bn) * ((M + bm - 1) / bm);
}

// Estimated time of S K ranges per tile: the busiest CU takes
// ceil(workgroups / CUs) of them, `resident` at a time (kTail: what is left
// over for the last round at the cost of that many, as the fp32 costs were
// fitted); S > 1 adds the reduction launch (r0) and the partial products'
// write and read (rb a MB).
template <bool kTail>
float plan_time(const TileCost& c, int S, int M, int N, int K, int64_t cus, float r0, float rb) {
    const int64_t per = (grid_of(M, N, c.BM, c.BN) * S + cus - 1) / cus;
    const float steps = (float)((K / kBK + S - 1) / S);
    float t;
    if (kTail) {
        t = (float)(per / c.resident) * (c.start + steps * c.step[c.resident - 1]);
        const int64_t rest = per % c.resident;
        if (rest) t += c.start + steps * c.step[rest - 1];
    } else {
        const int64_t conc = std::min<int64_t>(per, c.resident);
        t = (float)((per + conc - 1) / conc) * (c.start + steps * c.step[conc - 1]);
    }
    return S > 1 ? t + r0 + rb * 4e-6f * (float)S * (float)M * (float)N : t;
}

// The plan of least estimated time.  bf16: K ranges only where the unsplit
// grid of 128 x 128 tiles leaves more than 0.4 of the CUs without a
// workgroup -- few tokens or a narrow layer --, at most 8 of them with
// partial products of at most four times the packed weight's bytes; and,
// where a tile reaches that grid but leaves a tenth of the CUs idle over a
// long K, 256 x 256 over K ranges of at least 32 steps (down at M = 2048: 160
// tiles of 256 x 128 126-135 us, 3 x 80 of 256 x 256 92-98 us).
// Against fixed thresholds for the tile too: 2560 x 2560 at M = 32 / 64 23.5 /
// 24.0 -> 11.7 / 13.3 us, 1024 x 4096 35 -> 12 us, 5000 x 1024 at M = 300 22 ->
// 14.6 us, 2560 x 6912 at M = 700 55 -> 47 us; the sizes that the thresholds
// were tuned on keep their plans or ones as fast.
// A grid that reaches 0.6 of the CUs is split too where the caller gave the
// workspace of the fastest plan (kBest) and the estimate is a tenth less: 2560
// x 6912 at M = 1024 88 -> 56 us (three ranges of 256 x 128).  The plan follows
// from the shape and `space` alone, never from the size of the workspace.
PrefillPlan prefill_plan(int M, int N, int K, PlanSpace space) {
    const int64_t cus = device_cu_count();
    const int nsteps = K / kBK;
    const int64_t limit = 4 * ((int64_t)N * K / 128 * 80);
    PrefillPlan best = {64, 128, 1};
    float best_t = INFINITY;
    auto offer = [&](const TileCost& c, int S) {
        const float t = plan_time<false>(c, S, M, N, K, cus, 5.5f, 0.30f);
        if (t < best_t) {
            best_t = t;
            best = {c.BM, c.BN, S};
        }
    };
    for (const TileCost& c : kBf16Tiles) offer(c, 1);
    if (space == PlanSpace::kNone) return best;
    int64_t full = 0;   // the grid of the largest tile that fills 0.6 of the CUs
    for (int i = 0; i < 3 && !full; ++i) {
        const int64_t g = grid_of(M, N, kBf16Tiles[i].BM, kBf16Tiles[i].BN);
        if (g >= cus * 3 / 5) full = g;
    }
    if (full) {
        if (M >= 256 && full * 10 < cus * 9) {
            const int64_t g = grid_of(M, N, 256, 256);
            const int S = (int)std::min<int64_t>(cus / g, nsteps / 32);
            if (S >= 2 && g * S > full) offer(kBf16Tiles[0], S);
        }
        if (best.S > 1) return best;
        best_t *= 0.9f;
    } else {
        best_t *= 1.1f;   // (the estimates' error: split where it costs about the same)
    }
    const int64_t most = full && space != PlanSpace::kBest ? 0 : limit;
    for (const TileCost& c : kBf16Tiles) {
        for (int S = 2; S <= 8 && nsteps / S >= kMinSplitSteps; ++S) {
            if ((int64_t)S * M * N * 4 <= most) offer(c, S);
        }
    }
    return best;
}

// fp32 activations: any number of K ranges up to 16 whose partial products
// fit `limit` bytes (2560 x 2560 at M = 64 56 -> 22 us; 7680 x 2560 at M = 500
// in two ranges of 256 x 128 79 -> 71 us).  Unsplit plans take 1-9 % longer
// than estimated.
PrefillPlan prefill_f32_plan(int M, int N, int K, int64_t limit) {
    const int64_t cus = device_cu_count();
    PrefillPlan best = {64, 128, 1};
    float best_t = INFINITY;
    for (const TileCost& c : kF32Tiles) {
        for (int S = 1; S <= 16; ++S) {
            if (S > 1 && (K / kBK / S < kMinSplitSteps || (int64_t)S * M * N * 4 > limit)) break;
            const float t = plan_time<true>(c, S, M, N, K, cus, 8.75f, 0.312f) * (S > 1 ? 1.f : 1.06f);
            if (t < best_t) {
                best_t = t;
                best = {c.BM, c.BN, S};
            }
        }
    }
    return best;
}

// x (M rows, stride ldx, fp32) -> for every 32 columns of a row their hi =
// bf16(x), then their lo = bf16(x - hi): rows of 2K.  x - hi is exact in
// fp32, so hi + lo is x to 2^-18.  A thread takes eight columns (16-byte
// loads where kVec says that the rows allow them, 16-byte stores).
template <bool kVec>
__global__ __launch_bounds__(256) void split_bf16_kernel(const float* __restrict__ x, int64_t ldx,
                                                         bf16_bits* __restrict__ out, int M, int K) {
    const int k8 = K / 8;
    const int64_t total = (int64_t)M * k8;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * 256) {
        const int64_t m = i / k8;
        const int k = 8 * (int)(i - m * k8);
        const float* p = x + m * ldx + k;
        float v[8];
        if (kVec) {
            const f32x4_t a = reinterpret_cast<const f32x4_t*>(p)[0];
            const f32x4_t b = reinterpret_cast<const f32x4_t*>(p)[1];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = p[e];
        }
        u32x4_t hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bf16_bits h0 = f32_to_bf16_rne(v[2 * e]), h1 = f32_to_bf16_rne(v[2 * e + 1]);
            hi[e] = h0 | ((uint32_t)h1 << 16);
            lo[e] = f32_to_bf16_rne(v[2 * e] - bf16_to_f32(h0)) |
                    ((uint32_t)f32_to_bf16_rne(v[2 * e + 1] - bf16_to_f32(h1)) << 16);
        }
        bf16_bits* o = out + m * 2 * K + (k / 32) * 64 + k % 32;
        *reinterpret_cast<u32x4_t*>(o) = hi;
        *reinterpret_cast<u32x4_t*>(o + 32) = lo;
    }
}

inline int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }

inline int64_t partial_bytes(const PrefillPlan& p, int M, int N) {
    return p.S > 1 ? (int64_t)p.S * M * N * 4 : 0;
}

}  // namespace

int64_t prefill_split_bytes(int M, int N, int K, PlanSpace space) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128) return 0;
    return partial_bytes(prefill_plan(M, N, K, space), M, N);
}

namespace {

// The tiles of a plan, then the sum of their K ranges.
template <bool kSplit>
int launch_tiles(Prefill2Args a, const PrefillPlan& p, void* workspace, hipStream_t stream) {
    a.ksplit = p.S;
    a.part = p.S > 1 ? static_cast<float*>(workspace) : nullptr;
    constexpr int W = NB_PREFILL_WAVES;
    const int M = a.M, N = a.N;
    const unsigned grid = (unsigned)(((N + p.BN - 1) / p.BN) * ((M + p.BM - 1) / p.BM) * p.S);
#define NB_PREFILL2_LAUNCH(BMv, BNv)                                                          \
    hipLaunchKernelGGL((prefill2_kernel<BMv, BNv, W, kSplit>), dim3(grid), dim3(64 * W),     \
                       (size_t)2 * (BMv + BNv) * kRowBytes, stream, a)
    if (p.BN == 256) {
        if constexpr (!kSplit) NB_PREFILL2_LAUNCH(256, 256);   // (not in kF32Tiles)
    } else if (p.BM == 256) {
        NB_PREFILL2_LAUNCH(256, 128);
    } else if (p.BM == 128) {
        NB_PREFILL2_LAUNCH(128, 128);
    } else {
        NB_PREFILL2_LAUNCH(64, 128);
    }
#undef NB_PREFILL2_LAUNCH
    if (p.S > 1) {
        const int st = check_launch("nb_gemm_prefill");
        if (st) return st;
        const int64_t items = ((N | a.ldy) & 3) == 0 ? (int64_t)M * N / 4 : (int64_t)M * N;
        const unsigned rg = (unsigned)std::min<int64_t>((items + 255) / 256, 4096);
        hipLaunchKernelGGL(prefill_reduce_kernel, dim3(rg), dim3(256), 0, stream, a.part, p.S,
                           M, N, a.y, a.y_dtype, a.ldy);
    }
    return check_launch("nb_gemm_prefill");
}

}  // namespace

int launch_prefill2(const void* x, int64_t ldx, const uint8_t* packed, const float* codebook,
                    void* y, int y_dtype, int64_t ldy, int M, int N, int K, void* workspace,
                    PlanSpace space, hipStream_t stream) {
    return launch_tiles<false>({static_cast<const uint16_t*>(x), ldx, packed, codebook, y, ldy,
                                y_dtype, M, N, K, 1, nullptr},
                               prefill_plan(M, N, K, space), workspace, stream);
}

namespace {

// The least workspace: two bf16 parts of x, a codebook's size and the bf16
// kernel's partial products (the size that callers may have stored; what the
// parts of x leave goes to partial products).
int64_t prefill_f32_least(int M, int N, int K) {
    const int64_t xb = align256((int64_t)M * K * 2);
    const int64_t cb = align256((int64_t)N * (K / 128) * 8 * 4);
    return 2 * xb + cb + prefill_split_bytes(M, N, K, PlanSpace::kLeast);
}

// Partial products fit what the least workspace leaves beside the parts of x
// (kLeast), or 128 MiB where that is more (kBest).
PrefillPlan prefill_f32_plan(int M, int N, int K, PlanSpace space) {
    const int64_t left = prefill_f32_least(M, N, K) - align256((int64_t)M * K * 4);
    return prefill_f32_plan(M, N, K,
                            space == PlanSpace::kBest ? std::max<int64_t>(left, 128LL << 20) : left);
}

}  // namespace

int64_t prefill_f32_bytes(int M, int N, int K, PlanSpace space) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128) return 0;
    const int64_t least = prefill_f32_least(M, N, K);
    if (space != PlanSpace::kBest) return least;
    return std::max(least, align256((int64_t)M * K * 4) +
                               partial_bytes(prefill_f32_plan(M, N, K, space), M, N));
}

int launch_prefill_f32(const float* x, int64_t ldx, const uint8_t* packed, const float* codebook,
                       float* y, int64_t ldy, int M, int N, int K, void* workspace,
                       PlanSpace space, hipStream_t stream) {
    GemvArgs rows;
    rows.x = x;
    rows.x_dtype = NB_F32;
    rows.ldx = ldx;
    rows.packed = packed;
    rows.packed_bytes = packed_nbytes((int64_t)N * K, 3);
    rows.codebook = codebook;
    rows.y = y;
    rows.y_dtype = NB_F32;
    rows.ldy = ldy;
    rows.M = M;
    rows.N = N;
    rows.K = K;
    rows.bits = 3;
    rows.n_entries = 8;
    rows.block_size = 128;
    // Few rows of a small layer: the exact products on fp32 MFMAs, one launch
    // (2560 x 2560 at M = 17 / 48: 12 / 21 us; 7680 x 2560 at M = 17 / 32: 22
    // / 30 us against 26 / 26 below)
    if ((int64_t)M * N * K <= 400000000 && gemm_rows_f32_eligible(rows)) {
        return launch_gemm_rows_f32(rows, stream);
    }
    unsigned char* w = static_cast<unsigned char*>(workspace);
    bf16_bits* xs = reinterpret_cast<bf16_bits*>(w);
    const int64_t xbytes = align256((int64_t)M * K * 4);
    const unsigned g = (unsigned)std::min<int64_t>(((int64_t)M * (K / 8) + 255) / 256, 8192);
    const bool vec = reinterpret_cast<uintptr_t>(x) % 16 == 0 && ldx % 4 == 0;
    hipLaunchKernelGGL(vec ? split_bf16_kernel<true> : split_bf16_kernel<false>, dim3(g), dim3(256),
                       0, stream, x, ldx, xs, M, K);
    const int st = check_launch("nb_gemm_prefill_f32");
    if (st) return st;
    return launch_tiles<true>({xs, 2 * (int64_t)K, packed, codebook, y, ldy, NB_F32, M, N, K, 1,
                               nullptr},
                              prefill_f32_plan(M, N, K, space), w + xbytes, stream);
}

}  // namespace nb
