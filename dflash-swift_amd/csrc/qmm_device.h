/*
 * qmm_device.h -- device helpers shared by the gfx950 kernel sources: vector types, lane
 * swaps, exact code operands and 16-bit float conversions.
 */
#ifndef DFQ_QMM_DEVICE_H
#define DFQ_QMM_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

/* v_permlane16_swap / v_permlane32_swap with explicit wait states on both sides.  The
 * compiler (ROCm 7.2) pads the VALU-write -> swap-read side but not the swap-write ->
 * VALU-read side; a VALU op issued right after the swap has been seen to read the swapped
 * register's old contents on gfx950.  Semantics as the builtins: a is VDST, b is VSRC;
 * the 16-lane (32-lane) rows are exchanged between the two registers. */
__device__ __forceinline__ void permlane16_swap(uint32_t& a, uint32_t& b) {
    __asm__ volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 4" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void permlane32_swap(uint32_t& a, uint32_t& b) {
    __asm__ volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 4" : "+v"(a), "+v"(b));
}

/* 8 nibbles of a word -> bf16/fp16 (MAGIC + q) pairs (q_i, q_{i+4}) in VGPR i: seven VALU
 * ops per word (three shifts, four v_and_or_b32).  gfx9 VOP3 takes no literal constant, so
 * with constant mask and magic the compiler would split each and-or into a v_and_b32 and a
 * v_or_b32 with literals; the caller passes both as opaque register values (mask in an SGPR,
 * magic in a VGPR, loop-invariant) and the compiler forms v_and_or_b32 itself.  It has to
 * be the compiler's instruction, not inline asm: the MFMA that reads the result needs wait
 * states after a VALU write, and the compiler only pads hazards it can see. */
template <bool F16>
__device__ __forceinline__ u32x4_t nibble_operand(uint32_t p, uint32_t mask, uint32_t magic) {
    u32x4_t v;
    v[0] = (p & mask) | magic;
    v[1] = ((p >> 4) & mask) | magic;
    v[2] = ((p >> 8) & mask) | magic;
    v[3] = ((p >> 12) & mask) | magic;
    return v;
}

template <bool F16>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (F16) {
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
    } else {
        /* exact: integers <= 255 have zero low mantissa bits, so truncation is exact */
        return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    }
}

/* Two words of 4 bytes -> 8 exact 16-bit float codes in k order. */
template <bool F16>
__device__ __forceinline__ u32x4_t byte_operand(uint32_t a, uint32_t b) {
    u32x4_t v;
    v[0] = pack2<F16>((float)(a & 0xffu), (float)((a >> 8) & 0xffu));
    v[1] = pack2<F16>((float)((a >> 16) & 0xffu), (float)(a >> 24));
    v[2] = pack2<F16>((float)(b & 0xffu), (float)((b >> 8) & 0xffu));
    v[3] = pack2<F16>((float)((b >> 16) & 0xffu), (float)(b >> 24));
    return v;
}

template <bool F16>
__device__ __forceinline__ float elem_to_f32(uint32_t bits16) {
    if constexpr (F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
    else return __uint_as_float(bits16 << 16);
}

template <bool F16>
__device__ __forceinline__ uint16_t f32_to_out(float f) {
    if constexpr (F16) {
        return __builtin_bit_cast(uint16_t, (_Float16)f);
    } else {
        uint32_t u = __float_as_uint(f);
        if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
        u += 0x7fffu + ((u >> 16) & 1u);
        return (uint16_t)(u >> 16);
    }
}

/* s + the 8 elements of a 16-byte chunk, added pairwise in k order with v_dot2c against
 * (1, 1): four VALU ops per chunk.  Each element goes through a plain 32-bit temporary: the
 * builtin applied directly to an element of a 128-bit vector has been compiled (ROCm 7.2)
 * to read the vector's first register for every element.  It stays the compiler's own
 * instruction (not inline asm) so that the wait states a following DPP or MFMA read needs
 * are inserted. */
template <bool F16>
__device__ __forceinline__ float chunk_dot(u32x4_t v, float s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t e = v[i];
        if constexpr (F16)
            s = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, e),
                                       __builtin_bit_cast(f16x2_t, 0x3c003c00u), s, false);
        else
            s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, e),
                                                __builtin_bit_cast(bf16x2_t, 0x3f803f80u), s,
                                                false);
    }
    return s;
}

/* v from another lane of the same 16-lane row (DPP control CTRL; lanes whose source is
 * outside the row read 0). */
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

/* (x0..x7) -> (x0,x4, x1,x5, x2,x6, x3,x7): the k order of a nibble operand. */
__device__ __forceinline__ u32x4_t nibble_permute(u32x4_t v) {
    u32x4_t o;
    o[0] = __builtin_amdgcn_perm(v[2], v[0], 0x05040100u);
    o[1] = __builtin_amdgcn_perm(v[2], v[0], 0x07060302u);
    o[2] = __builtin_amdgcn_perm(v[3], v[1], 0x05040100u);
    o[3] = __builtin_amdgcn_perm(v[3], v[1], 0x07060302u);
    return o;
}

/* Element i of an array of dtype dt (0 bf16, 1 fp16, 2 fp32) as fp32, and the store of one. */
__device__ __forceinline__ float load_any(const void* ptr, int dt, size_t i) {
    if (dt == 2) return ((const float*)ptr)[i];
    const uint16_t h = ((const uint16_t*)ptr)[i];
    if (dt == 1) return (float)__builtin_bit_cast(_Float16, h);
    return __uint_as_float((uint32_t)h << 16);
}

__device__ __forceinline__ void store_any(void* ptr, int dt, size_t i, float f) {
    if (dt == 2) ((float*)ptr)[i] = f;
    else if (dt == 1) ((uint16_t*)ptr)[i] = f32_to_out<true>(f);
    else ((uint16_t*)ptr)[i] = f32_to_out<false>(f);
}

}  // namespace

#endif
