// Pieces shared by the noisy-device fp16 MFMA reads (noisy_mfma.hip, noisy_block.hip).
#pragma once

#include "mf_kernels.h"

namespace mf {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4fn __attribute__((ext_vector_type(4)));

// Buffer resource over [base, base + bytes): loads past the end return zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t noisy_buffer(const void *base, i64 bytes) {
    const int records = bytes > 0x7FFFFFFF ? 0x7FFFFFFF : int(bytes < 0 ? 0 : bytes);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), short(0), records,
                                             0x00020000);
}

// Eight input digits (bytes of `word`, slice (shift, mask)) as eight fp16.  Each digit d
// (at most 8 bits) becomes the low byte of fp16 0x64dd = 1024 + d: one v_perm places two
// digits beside two 0x64 bytes, and one packed fp16 subtraction of 1024 leaves d exactly
// (the same fp16 values as a conversion).  Six instructions per four digits.
__device__ __forceinline__ v8h digits_f16(uint2 word, int shift, u32 mask4) {
    typedef _Float16 v2f16 __attribute__((ext_vector_type(2)));
    const v2f16 base = {_Float16(1024.0f), _Float16(1024.0f)};
    const u32 lo = (word.x >> shift) & mask4, hi = (word.y >> shift) & mask4;
    // Byte pool of v_perm(src0, src1, sel): src1 bytes 0-3 (0x64), src0 bytes 4-7.
    const u32 k64 = 0x64646464u;
    const u32 w[4] = {__builtin_amdgcn_perm(lo, k64, 0x00050004u), __builtin_amdgcn_perm(lo, k64, 0x00070006u),
                      __builtin_amdgcn_perm(hi, k64, 0x00050004u), __builtin_amdgcn_perm(hi, k64, 0x00070006u)};
    u32 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __builtin_bit_cast(u32, __builtin_bit_cast(v2f16, w[i]) - base);
    return __builtin_bit_cast(v8h, make_uint4(o[0], o[1], o[2], o[3]));
}

}  // namespace mf
