// Packed GEMM over a few fp32 activation rows (M <= 64) on gfx950, in exact
// fp32 arithmetic:
//
//   y[m][n] = sum_k x[m][k] * W[n][k],  W.flat[i] = cb[i / BS][field i]
//
// -- the reference's fused kernels' products (inference/cuda_kernel.py:53-81,
// inference/triton_kernel.py:174-183) for the batched branch of its
// PackedLinear (triton_kernel.py:258-275), W never materialised.
//
// What bounds it: at M <= 16 the packed bytes are read in 2-4 us, the fp32
// products are 2 M N K FLOP -- too many for one FMA per weight and row out of
// LDS, so they go to the matrix cores in fp32: v_mfma_f32_16x16x4_f32 (256
// FLOP per CU and clock, the card's full fp32 rate; 16 weight rows x 16
// activation rows x 4 columns).  A 16-row x 128-column unit of W is 32 of
// them: lane (r, g) holds row r, 32-column slice g, so the 32 weights of a
// lane's slice are the A operands of 32 MFMAs whose B operands are the same
// columns of activation row r -- any assignment of columns to the four lane
// groups is right as long as A and B agree.  A weight costs two VALU
// instructions and one LDS lookup (the lane's block entries in an
// entry-major column of its own: every lookup of a wave hits its own bank),
// 64 + 80 LDS clocks a unit beside 256 clocks of MFMAs.
//
// Split: a workgroup owns 16 output rows; its waves split K in whole
// 128-column units and add their accumulators through LDS once at the end,
// in wave order and fp64 (deterministic).  Activations are read from global memory
// (the L2 holds them: at most 64 rows) straight into registers, a group of 8
// columns at a time, the next groups requested as the current one is used;
// the next unit's index bytes and block entries are requested before the
// current unit is computed.
//
// Measured (graph replays over cold copies, 3-bit / BS 128, M = 8): 6912 x
// 2560 12.8 us, 2560 x 6912 15.8, 2560 x 2560 8.6 -- the one-row-per-workgroup
// gemv_generic_kernel took 157 / 160 / 60.  What is left at M = 8, from copies
// with parts taken out: 10 us the weights' loads and MFMAs, 1.2 the lookups,
// 2 the activations (5.4 at M = 16: a lane's 32 columns are a cache line of
// their own).  fp64 errors at M <= 16 8.0-9.3e-8 from 512 x 512 to 16384 x
// 2560 (gemv_generic_kernel 8.5e-8-1.3e-7): accumulators of 8 products, added
// pairwise; with ones of 32 products 1.2-1.4e-7 at up to 1 % less time, with
// one chain a wave 2-3e-7.
//
// Formats: 2/3/4-bit with 2^bits entries, BS 64/128/256, K % 128 == 0 and
// K % BS == 0, up to 16 rows; up to 64 for 3-bit / BS 128.
#include "nb_device.h"
#include "nb_internal.h"
#include "nb_lookup.h"
#include "nb_stream_common.h"

#include <algorithm>
#include <cstdint>

namespace nb {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// waves a workgroup at most: 16 (128 registers a lane) for up to two
// activation tiles, 8 beyond
constexpr int max_waves(int tm) { return tm <= 2 ? 16 : 8; }
constexpr int kUnitK = 128;   // columns of a unit: four 32-weight slices
constexpr int kMaxTiles = 4;  // 16-row activation tiles (M <= 64)

struct RowsArgs {
    const float* x;
    int64_t ldx;
    const uint8_t* packed;
    const float* codebook;
    void* y;
    int y_dtype;
    int64_t ldy;
    int M, N, K;
};

// One lane's part of a unit of W: the index dwords of its 32-weight slice
// and the entries of the slice's block.
template <int BITS>
struct UnitRegs {
    uint32_t d[BITS];
    f32x4_t c[(1 << BITS) / 4];
};

template <int BITS, int BS, int TM>
__global__ __launch_bounds__(64 * max_waves(TM)) void gemm_rows_f32_kernel(RowsArgs a) {
    constexpr int NE = 1 << BITS;
    constexpr uint32_t kTab = NE * 256;          // a wave's entry-major table
    // 8-column groups of x in registers (four beside 16 entries spill: 2000 x
    // 8192 at M = 5 27.0 us against 22.6)
    constexpr int D = TM == 1 && BITS < 4 ? 4 : 2;
    extern __shared__ __align__(16) unsigned char smem[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nwaves = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16;
    const int row = min(row0 + r, a.N - 1);      // rows past N repeat the last one
    const int nunits = a.K / kUnitK;
    const int u0 = (int)((int64_t)wave * nunits / nwaves);
    const int u1 = (int)((int64_t)(wave + 1) * nunits / nwaves);

    // tables from the first multiple of kTab (a lookup address is the
    // table's address OR'ed with field << 8)
    const uint32_t smem_lds = stream::lds_addr(smem);
    const uint32_t tab0 = ((smem_lds + kTab - 1) & ~(kTab - 1)) - smem_lds;
    float* tabw = reinterpret_cast<float*>(smem + tab0 + wave * kTab);
    const uint32_t pbase = stream::lds_addr(tabw) + (uint32_t)(lane * 4);

    auto load_unit = [&](int u, UnitRegs<BITS>& w) {
        const int64_t flat = (int64_t)row * a.K + (int64_t)u * kUnitK + 32 * g;
        const uint32_t* ip = reinterpret_cast<const uint32_t*>(a.packed + flat / 8 * BITS);
#pragma unroll
        for (int i = 0; i < BITS; ++i) w.d[i] = ip[i];
        const f32x4_t* cp = reinterpret_cast<const f32x4_t*>(a.codebook + flat / BS * NE);
#pragma unroll
        for (int i = 0; i < NE / 4; ++i) w.c[i] = cp[i];
    };
    const float* xrow[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        xrow[i] = a.x + (int64_t)min(16 * i + r, a.M - 1) * a.ldx + 32 * g;
    }
    // columns 8 q .. 8 q + 7 of the lane's slice of unit u, every tile
    auto load_x = [&](int u, int q, f32x4_t (&v)[TM][2]) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const f32x4_t* p = reinterpret_cast<const f32x4_t*>(xrow[i] + (int64_t)u * kUnitK + 8 * q);
            v[i][0] = p[0];
            v[i][1] = p[1];
        }
    };

    f32x4_t sum[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) sum[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (u0 < u1) {
        UnitRegs<BITS> w;
        f32x4_t xv[D][TM][2];
        load_unit(u0, w);
#pragma unroll
        for (int q = 0; q < D; ++q) load_x(u0, q, xv[q]);
        for (int u = u0; u < u1; ++u) {
            // the block's entries into the lane's column (a lane reads back
            // only what it wrote; a wave's LDS operations stay in order)
#pragma unroll
            for (int i = 0; i < NE; ++i) tabw[i * 64 + lane] = w.c[i >> 2][i & 3];
            uint32_t d[BITS];
#pragma unroll
            for (int i = 0; i < BITS; ++i) d[i] = w.d[i];
            if (u + 1 < u1) load_unit(u + 1, w);
            // four accumulators, of a group of 8 columns for up to 16 rows (8
            // products each), of the unit beyond (32), added pairwise and
            // then to the wave's sum
            constexpr bool kShort = TM == 1;
            const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
            f32x4_t acc[TM][4], half[2];
            auto group = [&](auto qc) {
                constexpr int q = decltype(qc)::value;
                float wv[8];
                lookup8<BITS, 8, 8 * q>(d, pbase, wv, std::make_integer_sequence<int, 8>{});
                f32x4_t(&x)[TM][2] = xv[q % D];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        acc[i][j & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            wv[j], x[i][j >> 2][j & 3],
                            j < 4 && (kShort || q == 0) ? zero : acc[i][j & 3], 0, 0, 0);
                    }
                }
                if constexpr (kShort) {
                    const f32x4_t p = (acc[0][0] + acc[0][1]) + (acc[0][2] + acc[0][3]);
                    half[q / 2] = q % 2 ? half[q / 2] + p : p;
                }
                // the group D ahead, into the registers just used
                if constexpr (q + D < 4) {
                    load_x(u, q + D, x);
                } else {
                    if (u + 1 < u1) load_x(u + 1, q + D - 4, x);
                }
            };
            group(std::integral_constant<int, 0>{});
            group(std::integral_constant<int, 1>{});
            group(std::integral_constant<int, 2>{});
            group(std::integral_constant<int, 3>{});
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                sum[i] += kShort ? half[0] + half[1]
                                 : (acc[i][0] + acc[i][1]) + (acc[i][2] + acc[i][3]);
            }
        }
    }

    // lane (r, g) of tile i holds W rows 4 g + v of activation row 16 i + r:
    // the waves' sums in wave order, in fp64 (rounded once)
    float* red = reinterpret_cast<float*>(smem);
    __syncthreads();   // the tables are no longer read
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        // [activation row][W row], pitch 20: 16-byte pieces, spread banks
        *reinterpret_cast<f32x4_t*>(red + ((wave * TM + i) * 16 + r) * 20 + 4 * g) = sum[i];
    }
    __syncthreads();
    for (int e = t; e < TM * 256; e += blockDim.x) {
        const int m = e >> 4, n = e & 15;
        if (m >= a.M || row0 + n >= a.N) continue;
        double sd = 0.0;
        for (int w = 0; w < nwaves; ++w) sd += red[(w * TM * 16 + m) * 20 + n];
        const float s = (float)sd;
        const int64_t o = (int64_t)m * a.ldy + row0 + n;
        if (a.y_dtype == NB_BF16) {
            static_cast<bf16_bits*>(a.y)[o] = f32_to_bf16_rne(s);
        } else {
            static_cast<float*>(a.y)[o] = s;
        }
    }
}

// Waves a workgroup: about six a CU over the grid, with equal numbers of units
// to within one, at most five a wave unless the workgroup's wave limit forces
// more (2560 x 16384: eight).  (More waves add their start and the final sum,
// fewer leave SIMDs idle: 2560 x 2560 at M = 8 in 8.6 us at six a CU, 10.0
// at 12, 8.2 at four; 6912 x 2560 in 12.8 / 13.1 / 14.3 us; 2560 x 6912 with
// six units a wave 16.6 us, with four 15.8.)
int rows_waves(int N, int K, int tm) {
    const int64_t cus = device_cu_count();
    const int64_t groups = (N + 15) / 16, units = K / kUnitK;
    const int64_t want = (6 * cus + groups - 1) / groups;
    const int64_t most = max_waves(tm);
    const int64_t per = std::max(std::min<int64_t>((units + want - 1) / want, 5),
                                 (units + most - 1) / most);
    return (int)((units + per - 1) / per);
}

template <int BITS, int BS, int TM>
void launch_rows(const RowsArgs& a, hipStream_t stream) {
    const int waves = rows_waves(a.N, a.K, TM);
    const size_t tables = (size_t)(waves + 1) * (1 << BITS) * 256;
    const size_t red = (size_t)waves * TM * 16 * 20 * 4;
    hipLaunchKernelGGL((gemm_rows_f32_kernel<BITS, BS, TM>), dim3((a.N + 15) / 16),
                       dim3(64 * waves), std::max(tables, red), stream, a);
}

// More than one activation tile only for the format that nb_gemm_prefill_f32
// takes (nb_gemv stops at 16 rows).
constexpr bool many_rows(int bits, int block_size) { return bits == 3 && block_size == 128; }

template <int BITS, int BS>
void launch_rows_m(const RowsArgs& a, hipStream_t stream) {
    if constexpr (many_rows(BITS, BS)) {
        switch ((a.M + 15) / 16) {
            case 1: break;
            case 2: return launch_rows<BITS, BS, 2>(a, stream);
            case 3: return launch_rows<BITS, BS, 3>(a, stream);
            default: return launch_rows<BITS, BS, 4>(a, stream);
        }
    }
    launch_rows<BITS, BS, 1>(a, stream);
}

template <int BITS>
void launch_rows_bs(const RowsArgs& a, int block_size, hipStream_t stream) {
    switch (block_size) {
        case 64: launch_rows_m<BITS, 64>(a, stream); break;
        case 128: launch_rows_m<BITS, 128>(a, stream); break;
        default: launch_rows_m<BITS, 256>(a, stream); break;
    }
}

}  // namespace

bool gemm_rows_f32_eligible(const GemvArgs& a) {
    if (a.x_dtype != NB_F32 || a.M < 1) return false;
    if (a.bits < 2 || a.bits > 4 || a.n_entries != (1 << a.bits)) return false;
    if (a.block_size != 64 && a.block_size != 128 && a.block_size != 256) return false;
    if (a.M > (many_rows(a.bits, a.block_size) ? 16 * kMaxTiles : 16)) return false;
    if (a.K <= 0 || a.K % kUnitK != 0 || a.K % a.block_size != 0) return false;
    // dword loads of the stream, 16-byte loads of the codebook and x
    if (reinterpret_cast<uintptr_t>(a.packed) % 4 != 0) return false;
    if (reinterpret_cast<uintptr_t>(a.codebook) % 16 != 0) return false;
    if (reinterpret_cast<uintptr_t>(a.x) % 16 != 0) return false;
    if (a.M > 1 && a.ldx % 4 != 0) return false;
    return true;
}

int launch_gemm_rows_f32(const GemvArgs& g, hipStream_t stream) {
    RowsArgs a;
    a.x = static_cast<const float*>(g.x);
    a.ldx = g.ldx;
    a.packed = g.packed;
    a.codebook = g.codebook;
    a.y = g.y;
    a.y_dtype = g.y_dtype;
    a.ldy = g.ldy;
    a.M = g.M;
    a.N = g.N;
    a.K = g.K;
    switch (g.bits) {
        case 2: launch_rows_bs<2>(a, g.block_size, stream); break;
        case 3: launch_rows_bs<3>(a, g.block_size, stream); break;
        default: launch_rows_bs<4>(a, g.block_size, stream); break;
    }
    return check_launch("nb_gemv (rows)");
}

}  // namespace nb
