// Codebook lookups through LDS tables, shared by the fp32 GEMV kernels
// (nb_gemv.hip, nb_gemm_rows.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

namespace nb {

// (a & mask) | b in one VALU op, the mask in a scalar register (the disjoint
// `or` would otherwise become an add after a separate and).
__device__ __forceinline__ uint32_t and_or_s(uint32_t a, uint32_t mask, uint32_t b) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(b));
    return r;
}

// LDS byte address of codebook entry (field j) in the lane's table:
// `base` | field << POS.  POS = 8 for a lane's entry-major copy (the wave's
// table holds entry e of lane l at byte 256 e + 4 l, so every lookup of a
// wave hits a bank of its own); POS = 2 for the block's own NE entries where
// they landed in LDS.  `base` has zeros in the field's bits.  The field is
// shifted straight to bit POS and merged with the base: two VALU ops a
// weight (the fields of a 3-bit slice that straddle a dword take a funnel
// shift).
template <int BITS, int J, int POS>
__device__ __forceinline__ uint32_t entry_offset(const uint32_t (&d)[BITS], uint32_t base) {
    constexpr int bit = J * BITS;
    constexpr int w = bit >> 5;
    constexpr int off = bit & 31;
    constexpr uint32_t kMask = ((1u << BITS) - 1u) << POS;
    uint32_t v;
    if constexpr (off + BITS > 32) {
        v = __builtin_amdgcn_alignbit(d[w + 1], d[w], off - POS);
    } else if constexpr (off >= POS) {
        v = d[w] >> (off - POS);
    } else {
        v = d[w] << (POS - off);
    }
    return and_or_s(v, kMask, base);
}

typedef __attribute__((address_space(3))) const float lds_f32;

template <int BITS, int POS, int J0, int... Js>
__device__ __forceinline__ void lookup8(const uint32_t (&d)[BITS], uint32_t base, float (&w)[8],
                                        std::integer_sequence<int, Js...>) {
    ((w[Js] = *(lds_f32*)(uintptr_t)entry_offset<BITS, J0 + Js, POS>(d, base)), ...);
}

}  // namespace nb
