// cbq_mfma.h - matrix-core primitives shared by the W8A16 kernels: the 16-bit
// MFMA by activation dtype and the widening of int8 codes to that dtype.
#pragma once

#include "cbq_device.h"

namespace cbq {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16x __attribute__((ext_vector_type(16)));

// Operands and staging registers use native vector types: HIP's uint4 is a
// struct around a union, and arrays of it are kept on the stack (scratch or
// LDS) instead of in VGPRs.
template <int ACT>
__device__ __forceinline__ f4 mfma16x16x32(const u32x4& a, const u32x4& b, f4 c) {
  if constexpr (ACT == kF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a),
                                                   __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

// 4 int8 codes -> 4 exact values of the activation dtype (2 words).
template <int ACT>
__device__ __forceinline__ void i8x4_to_act(uint32_t w, uint32_t& lo, uint32_t& hi) {
  if constexpr (ACT == kF16) {
    // One v_cvt_f16_i16 per code: the SDWA source select takes byte b of w
    // sign-extended, the destination select writes one half of lo / hi and
    // keeps the other (exact: every int8 is an fp16). The compiler does not
    // form these selects from shifts and casts itself (it shifts each byte
    // first and packs the halves: 5 instructions per word instead of 4).
    // Wait states the hardware needs and the compiler cannot insert inside
    // the statement (it does not look into asm text):
    // - a sub-dword (dst_sel WORD_n) write needs one before the next VALU
    //   instruction that touches the register, and the preserving write of
    //   the high half reads it: lo's and hi's writes alternate so that each
    //   pair has one instruction between them;
    // - an MFMA that reads a VGPR needs two after a VALU write of it. The
    //   compiler counts the statement as a sub-dword write, not as a VALU: it
    //   keeps one wait state (an s_nop 0 of its own, or any instruction)
    //   between the statement and the next reader of lo / hi, whatever that
    //   reader is. The closing s_nop 0 is the second one for an MFMA.
    //   (Bit-identical outputs; 0.5% at M = 4096 against no wait.)
    asm("v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
        "v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3\n\t"
        "s_nop 0"
        : "=&v"(lo), "=&v"(hi)
        : "v"(w));
  } else {
    float f[4];
    int8x4_to_f32(w, f);
    lo = pack2_out<kBF16>(f[0], f[1]);
    hi = pack2_out<kBF16>(f[2], f[3]);
  }
}

template <int ACT>
__device__ __forceinline__ f16x mfma32x32x16(const u32x4& a, const u32x4& b, f16x c) {
  if constexpr (ACT == kF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a),
                                                   __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

}  // namespace cbq
