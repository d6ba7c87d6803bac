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
// The operands' element order: of 8 consecutive values, 0 2 1 3 4 6 5 7 -- a dword's bytes (0, 2)
// and, after a shift, (1, 3) lie where two f16 mantissas want them, so that one v_bitop3_b32
// (2.7 cycles per wave and SIMD, measured; v_perm_b32 and v_and_or_b32 4.3) masks them and sets
// the exponent byte.  Weights and activations use the same order, which leaves their products
// alone.  kMagic: (1024 + b0, 1024 + b2).
constexpr uint32_t kMagic = 0x64006400u;
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t m, uint32_t x) {
    return __builtin_amdgcn_bitop3_b32(v, m, x, 0xEA);  // (v & m) | x
}
__device__ __forceinline__ uint32_t and_xor(uint32_t v, uint32_t m, uint32_t x) {
    return __builtin_amdgcn_bitop3_b32(v, m, x, 0x6A);  // (v & m) ^ x
}
// q * sc for two 4-bit quants: (1024 + q) * sc - 1024 * sc in one fused f16 fma, whose
// result q * sc <= 945 is an integer f16 holds exactly
__device__ __forceinline__ uint32_t q4_scaled(uint32_t v, uint32_t mask, h2 sc, h2 nsc) {
    const h2 m = __builtin_bit_cast(h2, and_or(v, mask, kMagic));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(m, sc, nsc));
}
// four q8 as f16 integers in element order: q8 ^ 0x80 under 0x64 is 1152 + q8 exactly
__device__ __forceinline__ void q8x4_exact(uint32_t v, uint32_t &o0, uint32_t &o1) {
    const h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    o0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, and_xor(v, 0x00FF00FFu, 0x64806480u)) + off);
    o1 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, and_xor(v >> 8, 0x00FF00FFu, 0x64806480u)) + off);
}
// Q6_K: the 6-bit quant bytes 0, 2 of v as the f16 pair (q - 32), exactly
__device__ __forceinline__ h2 q6_centered(uint32_t v) {
    const h2 off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
    return __builtin_bit_cast(h2, and_or(v, 0x00FF00FFu, kMagic)) + off;
}
__device__ __forceinline__ uint32_t h2u(h2 v) { return __builtin_bit_cast(uint32_t, v); }

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
// dmin and the mins of a block header in two registers: dmin's nibbles take the places of the
// scales' low nibbles in hdr.w
__device__ __forceinline__ uint2 q4k_min_pack(const uint4 &hdr) {
    const uint32_t e = ((hdr.x >> 16) & 0x0F0Fu) | ((hdr.x >> 4) & 0x0F0F0000u);
    return make_uint2(hdr.z, (hdr.w & 0xF0F0F0F0u) | e);
}
__device__ __forceinline__ void q4k_min_operand(uint2 p, h8 &hi, h8 &lo) {
    const uint32_t d = (p.y & 0x0F0Fu) | ((p.y >> 12) & 0xF0F0u);
    q4k_min_operand_m(q4k_mins(make_uint4(0u, 0u, p.x, p.y)), d, hi, lo);
}

// ------------------------------------------------------------------ a lane's A operands
// Lane c + 16 q of a wave holds row c of a 16-row tile and, of every sub-block, values 8q .. 8q+7.
// Q4_K lane view of a tile's block: the header (d, dmin, scales) and the lane's qs bytes
struct Raw4 {
    uint4 h;
    uint2 a[4];  // qs bytes 32g + 8q .. +7
};
// A sub-block pair (2p, 2p + 1) shares its qs bytes: the low and the high nibbles.
// The pair's scales, from the 8 six-bit scales of the block (get_scale_min_k4, kernels.cu:45-53):
// sub-blocks 0-3 are the low 6 bits of bytes 0-3, 4-7 the low nibbles of bytes 8-11 with bits
// 6-7 of bytes 0-3 above them (the packed form of gemm_q4k.cu:53-56).  s = (sc, sc' / 16), n =
// -1024 s: the high nibbles are taken in place as bytes 16 q, and (1024 + 16 q) * sc / 16 - 64 sc
// = q * sc in the same exact fma.
struct Scales4 {
    h2 s, n;
};
__device__ __forceinline__ Scales4 scale_pair4(const uint4 &h, int p) {
    const uint32_t sc4 = p < 2 ? h.y & 0x3F3F3F3Fu : (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
    const h2 m = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    const h2 f = {(_Float16)1.0f, (_Float16)0.0625f};
    Scales4 o;
    o.s = (magic_pair(sc4, (p & 1) ? kSelHi : kSelLo) + m) * f;
    o.n = o.s * m;
    return o;
}
// the A operand of the pair's sub-block hi: sc * q for the lane's 8 values
__device__ __forceinline__ h8 operand4(const Raw4 &r, const Scales4 &T, int p, int hi) {
    const h2 S = {T.s[hi], T.s[hi]}, N = {T.n[hi], T.n[hi]};
    const uint2 c = r.a[p];
    const uint32_t msk = hi ? 0x00F000F0u : 0x000F000Fu;
    return __builtin_bit_cast(h8, make_uint4(q4_scaled(c.x, msk, S, N), q4_scaled(c.x >> 8, msk, S, N),
                                             q4_scaled(c.y, msk, S, N), q4_scaled(c.y >> 8, msk, S, N)));
}

// Q6_K raw bytes of one row tile's lane values for one block
struct Raw6 {
    uint2 ql[4];     // ql bytes 64H + 32p + 8q .. +7 (index 2H + p)
    uint2 qh[2];     // qh bytes 32H + 8q .. +7
    uint32_t sc[2];  // the lane's scale bytes of halves 0 / 1 (byte grp: scale 8H + 2grp + q/2)
};
// the two factors of the lane's scales of the sub-block pair p (sc - b and b, b = sc & 1) as f16
// pairs; zero when d is zero
struct Scales6 {
    h2 e, b;
};
__device__ __forceinline__ Scales6 scale_pair6(uint32_t sc, int p) {  // sc: the half's four scale bytes
    const uint32_t sel = (p & 1) ? kSelHi : kSelLo;
    const h2 off = {(_Float16)-1024.0f, (_Float16)-1024.0f}, off8 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    Scales6 o;
    o.e = magic_pair((sc & 0xFEFEFEFEu) ^ 0x80808080u, sel) + off8;  // the even parts of the signed bytes
    o.b = magic_pair(sc & 0x01010101u, sel) + off;
    return o;
}
// the planes (sc - b)(q - 32) and b(q - 32) of sub-block j
__device__ __forceinline__ void operand6(const Raw6 &r, const Scales6 &S, int j, h8 &a1, h8 &a2) {
    const int H = j >> 2, grp = j & 3;
    const h2 E = {S.e[grp & 1], S.e[grp & 1]}, B = {S.b[grp & 1], S.b[grp & 1]};
    const uint2 l = r.ql[2 * H + (grp & 1)], hq = r.qh[H];
    const int shl = 4 * (grp >> 1), shh = 2 * grp;
    const uint32_t v0 = ((l.x >> shl) & 0x0F0F0F0Fu) | (((hq.x >> shh) & 0x03030303u) << 4);
    const uint32_t v1 = ((l.y >> shl) & 0x0F0F0F0Fu) | (((hq.y >> shh) & 0x03030303u) << 4);
    const h2 c0 = q6_centered(v0), c1 = q6_centered(v0 >> 8), c2 = q6_centered(v1), c3 = q6_centered(v1 >> 8);
    a1 = __builtin_bit_cast(h8, make_uint4(h2u(c0 * E), h2u(c1 * E), h2u(c2 * E), h2u(c3 * E)));
    a2 = __builtin_bit_cast(h8, make_uint4(h2u(c0 * B), h2u(c1 * B), h2u(c2 * B), h2u(c3 * B)));
}

// a / b to within an ulp of the quotient (the plain product with the reciprocal where that is
// not finite)
__device__ __forceinline__ float ratio(float a, float b) {
    const float r = __builtin_amdgcn_rcpf(b), q = a * r;
    const float e = __builtin_fmaf(__builtin_fmaf(-q, b, a), r, q);
    return e == e ? e : q;
}

// ------------------------------------------------------------------ LDS copies and the MFMA
// Copies 16 (4) bytes per lane from global memory straight into LDS: lane i's bytes land at
// LDS address dst + 16 i (4 i), dst wave-uniform; the source is a lane's pointer, or a uniform base and a
// lane's byte offset.  The instruction is written out because the compiler, which cannot tell
// the copies' LDS targets from other LDS buffers, otherwise puts a wait for all of them in
// front of the next LDS read, and the copies never overlap anything (MoE prefill 856 -> 772 us
// at 512 tokens, 376 -> 327 us at 37; 128 experts of 4096 -> 1536, top-8).  Nothing waits for
// these copies but wait_vm.  M0 holds their LDS address: a reserved register, which may not be named as a
// clobber (the compiler warns); nothing else in these kernels uses it, which a test checks.
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
// LDS accesses at a lane's byte address plus a constant (an offset of the instruction): the
// address is hidden from the compiler, which otherwise keeps one sum per row in registers
template <typename T>
__device__ __forceinline__ T lds_get(uint32_t addr, uint32_t off) {
    return *(__attribute__((address_space(3))) const T *)(uintptr_t)(addr + off);
}
template <typename T>
__device__ __forceinline__ void lds_put(uint32_t addr, uint32_t off, T v) {
    *(__attribute__((address_space(3))) T *)(uintptr_t)(addr + off) = v;
}
// Waits until at most N of the wave's vector memory operations are outstanding.  Of the copies above,
// those of 16 bytes are relied on to complete in the order of their issue; 4-byte copies and loads
// into registers are not (a load into a register has been seen to overtake the copies), and need N = 0.
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ f4 mfma(const h8 &a, const h8 &b, const f4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

}  // namespace mnemo
