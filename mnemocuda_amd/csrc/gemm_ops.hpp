// gemm_ops.hpp -- operand conversions, matrix instruction and LDS copies shared by the plain
// GEMM (gemm.hip) and the grouped expert GEMM (gemm_grouped.hip).
#pragma once
#include "mnemo_common.hpp"

namespace mnemo {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ operand conversions
// Byte selectors placing bytes (0, 1) / (2, 3) of a dword under the f16 exponent byte 0x64:
// the pair (1024 + b0, 1024 + b1) exactly.
constexpr uint32_t kSelLo = 0x04010400u, kSelHi = 0x04030402u;

__device__ __forceinline__ h2 magic_pair(uint32_t v, uint32_t sel) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, v, sel));
}
// q * sc for two 4-bit quants: (1024 + q) * sc - 1024 * sc in one fused f16 fma, whose
// result q * sc <= 945 is an integer f16 holds exactly
__device__ __forceinline__ uint32_t q4_scaled(uint32_t v, uint32_t sel, h2 sc, h2 nsc) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(magic_pair(v, sel), sc, nsc));
}
// q8 as f16 integers: q8 ^ 0x80 under 0x64 is 1152 + q8 exactly
__device__ __forceinline__ void q8x4_exact(uint32_t v, uint32_t &o0, uint32_t &o1) {
    const h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const uint32_t u = v ^ 0x80808080u;
    o0 = __builtin_bit_cast(uint32_t, magic_pair(u, kSelLo) + off);
    o1 = __builtin_bit_cast(uint32_t, magic_pair(u, kSelHi) + off);
}
// Q6_K: two 6-bit quant bytes as the f16 pair (q - 32), exactly
__device__ __forceinline__ h2 q6_centered(uint32_t v, uint32_t sel) {
    const h2 off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
    return magic_pair(v, sel) + off;
}
__device__ __forceinline__ uint32_t h2u(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// byte i of the 12 packed scale bytes held in three dwords
__device__ __forceinline__ uint32_t sbyte(uint32_t s0, uint32_t s1, uint32_t s2, int i) {
    const uint32_t w = i < 4 ? s0 : (i < 8 ? s1 : s2);
    return (w >> (8 * (i & 3))) & 0xFFu;
}
// (sc, m) of sub-block j (get_scale_min_k4, kernels.cu:45-53)
__device__ __forceinline__ void q4k_scale_min(uint32_t s0, uint32_t s1, uint32_t s2, int j, uint32_t &sc,
                                              uint32_t &m) {
    if (j < 4) {
        sc = sbyte(s0, s1, s2, j) & 63;
        m = sbyte(s0, s1, s2, j + 4) & 63;
    } else {
        sc = (sbyte(s0, s1, s2, j + 4) & 15) | ((sbyte(s0, s1, s2, j - 4) >> 6) << 4);
        m = (sbyte(s0, s1, s2, j + 4) >> 4) | ((sbyte(s0, s1, s2, j) >> 6) << 4);
    }
}

// The 8 six-bit mins of a Q4_K super-block as bytes, sub-blocks 0-3 / 4-7 (the packed form of
// get_scale_min_k4, kernels.cu:45-53: m_j = scales[j+4] & 63 for j < 4, else
// (scales[j+4] >> 4) | ((scales[j] >> 6) << 4)); hdr.z, hdr.w hold scale bytes 4-7, 8-11.
__device__ __forceinline__ uint2 q4k_mins(const uint4 &hdr) {
    return make_uint2(hdr.z & 0x3F3F3F3Fu, ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u));
}
// Q4_K min-term operand of one super-block: for its 8 sub-blocks, -dmin * m_s as an exact
// f16 hi + lo pair (dmin is an f16, m a 6-bit integer: 17 significant bits), in packed f16:
// hi = the product rounded, lo = fma(m, -dmin, -hi), the remainder (at most 6 significant
// bits, a multiple of dmin's last place: exact, also in the subnormal range)
__device__ __forceinline__ void q4k_min_operand_m(uint2 mins, uint32_t dmin_bits, h8 &hi, h8 &lo) {
    const _Float16 nd = -__builtin_bit_cast(_Float16, (uint16_t)dmin_bits);
    const h2 ndd = {nd, nd};
    const h2 off = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    uint32_t H[4], L[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const h2 m = magic_pair(i < 2 ? mins.x : mins.y, (i & 1) ? kSelHi : kSelLo) + off;  // exact
        const h2 h = m * ndd;
        H[i] = h2u(h);
        L[i] = h2u(__builtin_elementwise_fma(m, ndd, -h));
    }
    hi = __builtin_bit_cast(h8, make_uint4(H[0], H[1], H[2], H[3]));
    lo = __builtin_bit_cast(h8, make_uint4(L[0], L[1], L[2], L[3]));
}
__device__ __forceinline__ void q4k_min_operand(const uint4 &hdr, h8 &hi, h8 &lo) {
    q4k_min_operand_m(q4k_mins(hdr), hdr.x >> 16, hi, lo);
}
// the ds halves of the 8 sub-blocks of a super-block: two Q8_1 block headers
__device__ __forceinline__ h8 ds_operand(const uint4 &b0, const uint4 &b1) {
    const uint32_t sel = 0x07060302u;  // the high halves of two dwords
    const uint4 u = make_uint4(__builtin_amdgcn_perm(b0.y, b0.x, sel), __builtin_amdgcn_perm(b0.w, b0.z, sel),
                               __builtin_amdgcn_perm(b1.y, b1.x, sel), __builtin_amdgcn_perm(b1.w, b1.z, sel));
    return __builtin_bit_cast(h8, u);
}

// Copies 16 (4) bytes per lane from global memory straight into LDS: lane i's bytes land at
// LDS address dst + 16 i (4 i), dst wave-uniform; the source is a lane's pointer, or a uniform base and a
// lane's byte offset.  The instruction is written out because the compiler, which cannot tell
// the copies' LDS targets from other LDS buffers, otherwise puts a wait for all of them in
// front of the next LDS read, and the copies never overlap anything (MoE prefill 856 -> 772 us
// at 512 tokens, 376 -> 327 us at 37; 128 experts of 4096 -> 1536, top-8).  Nothing waits for
// these copies but wait_vm.  (M0 holds their LDS address; the compiler keeps nothing in it.)
__device__ __forceinline__ uint32_t lds_addr(const void *p) {  // of a __shared__ object itself
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}
__device__ __forceinline__ void lds_copy16(const void *src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "memory");
}
__device__ __forceinline__ void lds_copy16(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void lds_copy4(const void *src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src) : "memory");
}
__device__ __forceinline__ void lds_copy4(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(dst), "v"(off), "s"(base)
                 : "memory");
}
// Waits until at most N of the wave's vector memory operations are outstanding (they complete
// in the order of their issue).
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ f4 mfma(const h8 &a, const h8 &b, const f4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma0(const h8 &a, const h8 &b) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
}

}  // namespace mnemo
