// gemm.hip -- Q4_K / Q6_K x Q8_1 GEMM for prefill and batched experts (gfx950 MFMA).
//
// Semantics (MnemoCUDA gemm_q4k.cu:103-112, 164-166, 194), per 32-value sub-block s:
//   Q4_K: out[j*M + i] = sum_s (d*sc_s)_i * d8_js * (sum_{k in s} q_ik * q8_jk) - (dmin*m_s)_i * ds_js
//   Q6_K: out[j*M + i] = sum_s d_i * d8_js * (sum over the two 16-value groups g of s of
//                                            sc_g * sum_{k in g} (q_ik - 32) * q8_jk)
// with W GGUF blocks [M][K], the activations Q8_1 MMQ blocks [N][K/128] x 144 B
// (half2 (d8, ds) per 32 values, ds = d8 * sum of the unquantized values), and the output
// column-major [N][M].  The scales d*sc and dmin*m are exact in fp32 (the reference rounds
// them to f16 in registers, gemm_q4k.cu:106-111; this build keeps the GEMV's fp32
// dequantisation, kernels.cu:114-136).
//
// Exact integer sub-block sums on f16 matrix cores.
//   * Operands are integers that f16 holds exactly: A = sc * q (Q4_K, <= 63 * 15 = 945) and
//     B = q8 (|q8| <= 127).  A 16x16x32 f16 MFMA over one sub-block sums 32 exact products
//     below 2^22 in fp32, so its result t is the exact integer sub-block sum.  Q6_K's
//     sc * (q - 32) reaches 4096 in magnitude, where f16 holds only even integers: it is
//     split into two exact planes, (sc - b) * (q - 32) (even) and b * (q - 32) with
//     b = sc & 1, and the two MFMAs chain into t (|t| < 2^24, still exact).
//   * The fp32 rescale is a running scale: the accumulator holds the sum of a span of K in units of
//     the current (row scale d) x (token scale d8).  Each sub-block is one fma, acc = acc * rho + t
//     with rho = d8_prev / d8 of the token: one rounding per sub-block.  A span is a super-block
//     where a wave holds at most 8 output tiles (R NB <= 8): its sum, times d * d8 (exact, two f16
//     factors), joins an absolute total by one more fma, so that the roundings at the full sum's
//     magnitude are one per super-block.  Wider tiles have no registers for the totals: their span
//     is a window of 1024 values, acc is also multiplied by d_prev / d of the rows at super-block
//     boundaries, becomes absolute at the window's end, and the scales start again from 1.  Q4_K's
//     wide tiles form acc * rho and let the MFMA add the products to it (two roundings): forming t
//     first costs them 5 % (M = 4096, K = 4096, N = 1024: 69.0 against 73.2 us with the quantizer).  A zero scale
//     leaves the running scale unchanged and zeroes its block's operand (its products are zero).
//   * Q4_K's min term, sum_s -(dmin*m_s) * ds_js, is one more product over the sub-block
//     index: -dmin*m (an f16 times a 6-bit integer, 17 significant bits) is split into an
//     f16 hi + lo pair that is exact, ds is an f16 already, and two MFMAs per window (32
//     sub-blocks) form it.
//   Relative L2 against the fp64 value, N(0, 1) activations: K = 256 7.5e-8, K = 4096 9.5e-8 (wide tiles
//   2.5e-7 and 2.2e-7, Q4_K and Q6_K), K = 16384 1.0e-7 to 1.2e-7 (wide 5.0e-7 and 4.4e-7).  With
//   one running sum per slice of K and two (Q6_K: three) roundings per sub-block: 9.1e-8, 1.4e-7
//   (2.5e-7), 2.5e-7 (5.2e-7).
//
// An int8 MFMA does not fit this product on gfx950: v_mfma_i32_16x16x64_i8 sums 64 values,
// two sub-blocks with different token scales, and the 32-deep v_mfma_i32_16x16x32_i8 runs
// at the f16 MFMA's rate (16 cycles for 16x16x32, measured) while needing three VALU
// operations per output per sub-block (int -> float, the product of the row and token
// scales, the fma) where the exact f16 form needs one.
#include <algorithm>
#include <cstddef>

#include "gemm_ops.hpp"
#include "mnemo_common.hpp"
#include "mnemo_internal.hpp"

namespace mnemo {

// ------------------------------------------------------------------ tiled kernel
// A workgroup is RG x KS waves.  Wave (rg, ks) multiplies R 16-row weight tiles (their operands
// converted in its own registers) with the workgroup's 16 NB tokens over slice ks of K (whole
// super-blocks); the slices meet through LDS at the end.  So a weight is converted once per
// token tile, no wave waits for another's weights, and the only shared operand is the
// activation tile: the RG waves of a slice turn the Q8_1 rows of a 64-value stage into f16 in
// LDS, one stage ahead of the multiplication (double-buffered; the raw bytes one stage
// earlier still, in registers).
//
// What bounds it: the issue rate of a wave (one instruction per ~4.8 cycles, two waves per SIMD)
// and what a stage serialises: per stage of the 256 x 128 shape ~1900 of ~3300 cycles multiply
// (30 per MFMA with its four rescales), the rest is the conversion and the barrier.  Everything
// that a stage or window waited for was moved out of it: the Q4_K min term's operands come from
// LDS (read from memory at each window's end they cost 8 400 cycles per window), the conversion
// of the next stage sits in front of the multiplication in the same basic block (so the two
// interleave), addresses are scalars plus constants.  M = 8192, K = 4096, N = 512: 81.4 -> 62 us
// (550 TOPS); M = 4096, K = 8192, N = 1999: 319 -> 198 us (677 TOPS); N = 7: 25.5 -> 13 us, with
// the tiled kernel before (128 x 128 tiles, operands of both sides through LDS, K split over
// workgroups by atomics) on the left.
constexpr int kStageK = 64;  // K per stage
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

template <int TYPE, int R, int RG, int KS, int NB>
struct GemmLds {
    static constexpr int kPer = R * NB * 4 * 64;  // floats of a wave's accumulators
    static constexpr bool kTotals = R * NB <= 8;  // a total per output beside the super-block's sum
    union {
        _Float16 b[KS][2][NB * 16 * kStageK];  // q8 of a stage's tokens, chunks XOR-swizzled (b_off)
        float red[KS > 1 ? kPer * RG : 1];  // after the loop: a slice's sums, lane-minor
    };
    float rho[KS][2][2][NB * 16];  // token scale ratios of the stage's sub-blocks
    float unit[KS][2][NB * 16];    // the tokens' d8 units at the end of the span (two spans)
    // Q4_K: the f16 ds of the tokens' sub-blocks in the current window and the next
    uint16_t ds[TYPE == kTypeQ4K ? KS : 1][2][NB * 16][32];
    // .. and a lane's packed mins and dmin of the window's block 4 w + q, by row tile
    u4v mins[TYPE == kTypeQ4K ? RG * KS : 1][R][64];
};

// f16 rows of 64 K-columns = 8 chunks of 16 B (a row is 128 B, half of the 64 x 4 B LDS banks),
// stored without padding with the chunk index XOR-ed by (row / 2) % 8: the 16 rows of an MFMA
// fragment read (one chunk each) cover the 64 banks once
__device__ __forceinline__ int b_off(int row, int chunk) { return row * kStageK + ((chunk ^ ((row >> 1) & 7)) << 3); }

struct GemmArgs {
    const uint8_t *W;  // weights [M][K]
    const uint8_t *A;  // Q8_1 MMQ rows [N]
    float *out;
    int M, K, N;
    int ld;            // out[j * ld + i]
};

// Loads at a uniform base + a uniform offset + a lane's 32-bit offset (no 64-bit address per
// lane and load: those took 20 registers and as many VALU operations per stage).  The base is the
// workgroup's first row, so its rows span less than 4 GiB (gemm_plan)
struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ explicit Buf(const uint8_t *p)
        : r(__builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0xFFFFFFFF, 0x00020000)) {}
    __device__ __forceinline__ uint2 ld8(uint32_t lane, uint32_t uni) const {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, lane, uni, 0));
    }
    __device__ __forceinline__ uint4 ld16(uint32_t lane, uint32_t uni) const {
        return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, lane, uni, 0));
    }
    __device__ __forceinline__ uint32_t ld2(uint32_t lane, uint32_t uni) const {
        return __builtin_amdgcn_raw_buffer_load_b16(r, lane, uni, 0);
    }
};

// The lane's raw weights of one super-block of its row: the quants of the four sub-block pairs
// are replaced by the next block's as soon as a pair's operands are formed, the header is held
// for this block and the next
template <int TYPE>
struct RawW;
template <>
struct RawW<kTypeQ4K> {
    Raw4 r;
    // u: the block's offset, o: the lane's row
    __device__ __forceinline__ void load_pair(const Buf &w, uint32_t u, uint32_t o, int q, int p) {
        r.a[p] = w.ld8(o + 8 * q, u + 16 + 32 * p);
    }
    __device__ __forceinline__ void load_head(const Buf &w, uint32_t u, uint32_t o) { r.h = w.ld16(o, u); }
    // from here on (nothing is formed from the loads before this point: the compiler would wait
    // for them there)
    __device__ __forceinline__ void pin_pair(int p) { asm volatile("" : "+v"(r.a[p].x), "+v"(r.a[p].y)); }
    __device__ __forceinline__ void next_head() {
        asm volatile("" : "+v"(r.h.x), "+v"(r.h.y), "+v"(r.h.z), "+v"(r.h.w));
    }
    __device__ __forceinline__ uint32_t d_bits() const { return r.h.x & 0xFFFFu; }
};
template <>
struct RawW<kTypeQ6K> {
    Raw6 r;
    uint4 sc;
    uint32_t d;
    // pairs 2H, 2H + 1 share qh; pair p = 2H + u holds the nibbles u of both ql groups
    __device__ __forceinline__ void load_pair(const Buf &w, uint32_t u, uint32_t o, int q, int p) {
        if (p & 1) {  // both pairs of half H are formed
            const int H = p >> 1;
            r.ql[2 * H] = w.ld8(o + 8 * q, u + 64 * H);
            r.ql[2 * H + 1] = w.ld8(o + 8 * q, u + 64 * H + 32);
            r.qh[H] = w.ld8(o + 8 * q, u + 128 + 32 * H);
        }
    }
    __device__ __forceinline__ void load_head(const Buf &w, uint32_t u, uint32_t o) {
        sc = w.ld16(o, u + 192);
        d = w.ld2(o, u + 208);
    }
    __device__ __forceinline__ void pin_pair(int p) {
        const int H = p >> 1;
        if (!(p & 1))
            asm volatile("" : "+v"(r.ql[2 * H].x), "+v"(r.ql[2 * H].y), "+v"(r.ql[2 * H + 1].x), "+v"(r.ql[2 * H + 1].y),
                         "+v"(r.qh[H].x), "+v"(r.qh[H].y));
    }
    uint32_t dc;
    __device__ __forceinline__ void next_head(int q) {
        asm volatile("" : "+v"(sc.x), "+v"(sc.y), "+v"(sc.z), "+v"(sc.w), "+v"(d));
        // of the 16 scale bytes the lane needs 8H + 2grp + q/2
        const uint32_t sel = 0x06040200u + 0x01010101u * (uint32_t)(q >> 1);
        r.sc[0] = __builtin_amdgcn_perm(sc.y, sc.x, sel);
        r.sc[1] = __builtin_amdgcn_perm(sc.w, sc.z, sel);
        dc = d;
    }
    __device__ __forceinline__ uint32_t d_bits() const { return dc; }
};

template <int TYPE, int R, int RG, int KS, int NB, bool ONCE>
__global__ void __launch_bounds__(64 * RG * KS) __attribute__((amdgpu_waves_per_eu(R * NB <= 4 && KS * NB <= 8 ? 4 : 2)))
gemm_q8_1_kernel(GemmArgs g) {
    using Lds = GemmLds<TYPE, R, RG, KS, NB>;
    constexpr bool Q4 = TYPE == kTypeQ4K;
    constexpr int kTok = NB * 16;
    constexpr int kBlk = Q4 ? kQ4KBytes : kQ6KBytes;
    __shared__ __align__(16) Lds L;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, ks = wave / RG, q = lane >> 4, c = lane & 15;
    const int nsb = g.K / 256;
    const int sb0 = nsb * ks / KS, n = nsb * (ks + 1) / KS - sb0;  // the slice's super-blocks
    const int nmax = (nsb + KS - 1) / KS;                          // .. at most this many in any slice
    const int i0 = (blockIdx.x * RG + rg) * 16 * R, j0 = blockIdx.y * kTok;

    // the lane's weight rows (rows past the end re-read the last): byte offsets from the workgroup's
    // first row
    const uint32_t wrow = (uint32_t)nsb * kBlk;
    const int iw = blockIdx.x * RG * 16 * R;
    const Buf wb(g.W + (size_t)iw * wrow + (size_t)sb0 * kBlk);
    uint32_t wo[R];
#pragma unroll
    for (int a = 0; a < R; a++) wo[a] = (uint32_t)(min(i0 + 16 * a + c, g.M - 1) - iw) * wrow;
    // loader role in the slice: thread -> token lt, values VP lp .. of each stage
    constexpr int VP = kTok * kStageK / (64 * RG);
    constexpr int PT = kStageK / VP;  // threads per token
    static_assert(VP >= 8 && kTok * PT == 64 * RG, "every thread of a slice loads whole chunks of one token");
    const int ltid = rg * 64 + lane, lt = ltid / PT, lp = ltid % PT;
    const Buf ab(g.A + ((size_t)j0 * (g.K / 128) + 2 * sb0) * kQ81Bytes);  // the tile's first token
    const uint32_t ao = (uint32_t)(min(j0 + lt, g.N - 1) - j0) * (uint32_t)(g.K / 128) * kQ81Bytes;
    struct RawA {
        uint32_t v[VP / 4];
        uint2 hd;  // (d8, ds) of the stage's two sub-blocks
    };
    auto load_a = [&](int t, RawA &r) {  // stage t of the slice
        const uint32_t u = (uint32_t)(t >> 1) * kQ81Bytes;
        r.hd = ab.ld8(ao, u + 8 * (t & 1));
        const uint32_t p = u + 64 * (t & 1);
        if constexpr (VP == 8) {
            const uint2 v = ab.ld8(ao + VP * lp, p + 16);
            r.v[0] = v.x; r.v[1] = v.y;
        } else {
#pragma unroll
            for (int i = 0; i < VP / 16; i++) {
                const uint4 v = ab.ld16(ao + VP * lp, p + 16 + 16 * i);
                r.v[4 * i] = v.x; r.v[4 * i + 1] = v.y; r.v[4 * i + 2] = v.z; r.v[4 * i + 3] = v.w;
            }
        }
    };
    // LDS addresses: the lane's fragment chunks of both sub-blocks of a stage, its token column's
    // ratios, the chunks and ratios that it writes
    const uint32_t lds = lds_addr(&L);
    const uint32_t kRow = kStageK * 2, kBuf = kTok * kRow;  // bytes of a row, of a buffer
    const uint32_t lb = lds + offsetof(Lds, b) + (uint32_t)ks * 2 * kBuf;
    const uint32_t lr = lds + offsetof(Lds, rho) + (uint32_t)ks * 4 * kTok * 4;
    const uint32_t ld = lds + offsetof(Lds, ds) + (uint32_t)ks * 2 * kTok * 64;
    uint32_t wd = ld + 64 * lt, dq = ld + 64 * c + 16 * q;  // ds: written, and the lane's window operand
    uint32_t wu = lds + offsetof(Lds, unit) + ((uint32_t)ks * 2 * kTok + lt) * 4;
    uint32_t mn0 = lds + offsetof(Lds, mins) + (uint32_t)wave * R * 1024 + 16 * lane;
    uint32_t fr[2], rr0 = lr + 4 * c, wr = lr + 4 * lt, wc[VP / 8];
#pragma unroll
    for (int jj = 0; jj < 2; jj++) fr[jj] = lb + 2 * b_off(c, 4 * jj + q);
#pragma unroll
    for (int i = 0; i < VP / 8; i++) wc[i] = lb + 2 * b_off(lt, VP / 8 * lp + i);
    asm volatile("" : "+v"(fr[0]), "+v"(fr[1]), "+v"(rr0), "+v"(wr), "+v"(mn0), "+v"(wd), "+v"(dq), "+v"(wu));
#pragma unroll
    for (int i = 0; i < VP / 8; i++) asm volatile("" : "+v"(wc[i]));
    // the token's running d8: 1 at a span's start, unchanged by d8 = 0.  A span is a super-block
    // (kTotals) or a window of four
    constexpr bool kTotals = Lds::kTotals;
    constexpr int kSpan = kTotals ? 2 : 4;  // log2 of its stages
    float unit = 1.0f;
    auto convert_a = [&](int t, RawA &r, int buf) {
#pragma unroll
        for (int i = 0; i < VP / 4; i++) asm volatile("" : "+v"(r.v[i]));  // pins, as RawW's
        asm volatile("" : "+v"(r.hd.x), "+v"(r.hd.y));
        const float d0 = h2f(r.hd.x & 0xFFFFu), d1 = h2f(r.hd.y & 0xFFFFu);
        if ((t & ((1 << kSpan) - 1)) == 0) unit = 1.0f;
        const float c0 = d0 != 0.0f ? d0 : unit, c1 = d1 != 0.0f ? d1 : c0;
        // the PT threads of a token write the same values
        lds_put<float>(wr, buf * 2 * kTok * 4, ratio(unit, c0));
        lds_put<float>(wr, (buf * 2 + 1) * kTok * 4, ratio(c0, c1));
        lds_put<float>(wu, ((t >> kSpan) & 1) * kTok * 4, c1);
        if constexpr (Q4)
            lds_put<uint32_t>(wd, ((t >> 4) & 1) * kTok * 64 + (t & 15) * 4,
                              __builtin_amdgcn_perm(r.hd.y, r.hd.x, 0x07060302u));  // the high halves
#pragma unroll
        for (int i = 0; i < VP / 8; i++) {
            const int ch = VP / 8 * lp + i;
            // a block whose d rounds to f16 zero keeps quants up to +-127: its values are 0 * q8
            const bool zero = (ch < 4 ? d0 : d1) == 0.0f;
            uint4 o;
            q8x4_exact(zero ? 0u : r.v[2 * i], o.x, o.y);
            q8x4_exact(zero ? 0u : r.v[2 * i + 1], o.z, o.w);
            lds_put<u4v>(wc[i], buf * kBuf, u4v{o.x, o.y, o.z, o.w});
        }
        unit = c1;
    };

    constexpr f4 kZero = {0.f, 0.f, 0.f, 0.f};
    f4 acc[R][NB];                                // the span's sum
    f4 tot[kTotals ? R : 1][kTotals ? NB : 1];  // the absolute sum of the spans before
    float deff[R];  // d of the lane's row of each tile (a window's: its last nonzero d, 1 before)
#pragma unroll
    for (int a = 0; a < R; a++) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            acc[a][b] = kZero;
            if constexpr (kTotals) tot[a][b] = kZero;
        }
        deff[a] = 1.0f;
    }
    RawW<TYPE> w[R];
    RawA ra;
    if (n > 0) {
        load_a(0, ra);
#pragma unroll
        for (int a = 0; a < R; a++) {
            w[a].load_head(wb, 0, wo[a]);
#pragma unroll
            for (int p = 0; p < 4; p++) w[a].load_pair(wb, 0, wo[a], q, p);
        }
        convert_a(0, ra, 0);
        load_a(1, ra);
    }
    lds_barrier();

    for (int k = 0; k < nmax; k++) {
        if (k < n) {  // wave-uniform (slices differ by one super-block at most)
            const uint32_t next = (uint32_t)min(k + 1, n - 1) * kBlk;
#pragma unroll
            for (int a = 0; a < R; a++) {
                if constexpr (Q4) w[a].next_head();
                else w[a].next_head(q);
                if constexpr (!Q4) w[a].load_head(wb, next, wo[a]);
                const float d = h2f(w[a].d_bits());
                if constexpr (Q4) {
                    if ((k & 3) == q) {
                        const uint2 mn = q4k_mins(w[a].r.h);
                        lds_put<u4v>(mn0, a * 1024, u4v{mn.x, mn.y, w[a].r.h.x >> 16, 0u});
                    }
                    if (d == 0.0f) w[a].r.h.y = w[a].r.h.w = 0u;  // scales 0: the block's products are zero
                } else {
                    if (d == 0.0f) w[a].r.sc[0] = w[a].r.sc[1] = 0u;
                }
                if constexpr (kTotals) {
                    deff[a] = d;
                    continue;
                }
                // the running row scale: lane c owns row c; the lane's outputs are rows 4q + x
                const float nd = d == 0.0f ? deff[a] : d;
                const float sg = ratio(deff[a], nd);
                deff[a] = nd;
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const float se = __shfl(sg, 4 * q + x);
#pragma unroll
                    for (int b = 0; b < NB; b++) acc[a][b][x] *= se;
                }
            }
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int t = 4 * k + s, buf = s & 1;
                convert_a(t + 1, ra, buf ^ 1);
                load_a(min(t + 2, 4 * n - 1), ra);
                Scales4 s4[R];
                Scales6 s6[R];
#pragma unroll
                for (int jj = 0; jj < 2; jj++) {
                    h8 bf[NB];
                    float rr[NB];
#pragma unroll
                    for (int b = 0; b < NB; b++) {
                        rr[b] = lds_get<float>(rr0, ((buf * 2 + jj) * kTok + 16 * b) * 4);
                        bf[b] = lds_get<h8>(fr[jj], buf * kBuf + 16 * b * kRow);
                    }
                    h8 a1[R], a2[R];
#pragma unroll
                    for (int a = 0; a < R; a++) {
                        if (jj == 0) w[a].pin_pair(s);
                        if constexpr (Q4) {
                            if (jj == 0) s4[a] = scale_pair4(w[a].r.h, s);
                            if (jj == 1 && s == 3) w[a].load_head(wb, next, wo[a]);  // the block's last scales are formed
                            a1[a] = operand4(w[a].r, s4[a], s, jj);
                        } else {
                            if (jj == 0) s6[a] = scale_pair6(w[a].r.sc[s >> 1], s);
                            operand6(w[a].r, s6[a], 2 * s + jj, a1[a], a2[a]);
                        }
                        if (jj == 1) w[a].load_pair(wb, next, wo[a], q, s);
                    }
#pragma unroll
                    for (int b = 0; b < NB; b++)
#pragma unroll
                        for (int a = 0; a < R; a++) {
                            f4 &ac = acc[a][b];
                            if constexpr (!ONCE) {
                                ac *= rr[b];
                                ac = mfma(a1[a], bf[b], ac);
                            } else {
                                f4 t = mfma(a1[a], bf[b], kZero);
                                if constexpr (!Q4) t = mfma(a2[a], bf[b], t);
                                if (kTotals && s == 0 && jj == 0) ac = t;
                                else ac = __builtin_elementwise_fma(ac, f4{rr[b], rr[b], rr[b], rr[b]}, t);
                            }
                        }
                }
                const bool wend = (k & 3) == 3 || k == n - 1;  // the window's last super-block
                if (s == 3 && (kTotals || wend)) {             // the span's end
                    // The sum becomes absolute, and the Q4_K min term of the window's 32 sub-blocks,
                    // sum_s -(dmin*m_s)_i * ds_js, joins: lane group q holds super-block 4w + q of its row
                    // and token (K index 8q + s of the MFMA = sub-block s); groups past the end add
                    // nothing.  With totals the term goes to the total first, so that the span's sum is
                    // the only addition at the new magnitude.
                    const int kw = (k & ~3) + q;
                    const bool valid = kw < n;
                    constexpr int NC = NB > 4 ? NB / 2 : NB;  // columns at a time
                    const int wp = (k >> 2) & 1, up = kTotals ? k & 1 : wp;
                    // the term of column b, on top of c
                    auto min_term = [&](const h8 &hi, const h8 &lo, int b, const f4 &c) {
                        h8 bd = lds_get<h8>(dq, wp * kTok * 64 + 16 * b * 64);
                        if (!valid) bd = h8{};
                        return mfma(lo, bd, mfma(hi, bd, c));
                    };
                    auto min_rows = [&](int a, h8 &hi, h8 &lo) {
                        const u4v mn = lds_get<u4v>(mn0, a * 1024);
                        q4k_min_operand_m(make_uint2(mn.x, mn.y), valid ? mn.z : 0u, hi, lo);
                    };
                    if constexpr (kTotals) {
                        // the sums are formed here: the compiler would sink them past the branch, since
                        // only the total uses them, and keep every product until then
#pragma unroll
                        for (int a = 0; a < R; a++)
#pragma unroll
                            for (int b = 0; b < NB; b++) asm volatile("" : "+v"(acc[a][b]));
                    }
                    if constexpr (Q4 && kTotals) {
                        if (wend) {
#pragma unroll
                            for (int a = 0; a < R; a++) {
                                h8 hi, lo;
                                min_rows(a, hi, lo);
#pragma unroll
                                for (int b = 0; b < NB; b++) tot[a][b] = min_term(hi, lo, b, tot[a][b]);
                                __builtin_amdgcn_sched_barrier(0);
                            }
                        }
                    }
#pragma unroll
                    for (int b0 = 0; b0 < NB; b0 += NC) {
                        float dt[NC];
#pragma unroll
                        for (int b = 0; b < NC; b++) dt[b] = L.unit[ks][up][16 * (b0 + b) + c];
#pragma unroll
                        for (int a = 0; a < R; a++) {
                            float dr[4];
#pragma unroll
                            for (int x = 0; x < 4; x++) dr[x] = __shfl(deff[a], 4 * q + x);
                            h8 hi, lo;
                            if constexpr (Q4 && !kTotals) min_rows(a, hi, lo);
#pragma unroll
                            for (int b = 0; b < NC; b++) {
                                f4 &ac = acc[a][b0 + b];
                                f4 to = kZero;
                                if constexpr (kTotals) to = tot[a][b0 + b];
                                else if constexpr (Q4) to = min_term(hi, lo, b0 + b, kZero);
#pragma unroll
                                for (int x = 0; x < 4; x++) to[x] = __builtin_fmaf(ac[x], dr[x] * dt[b], to[x]);
                                if constexpr (kTotals) tot[a][b0 + b] = to;
                                else ac = to;
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int a = 0; a < R; a++) deff[a] = 1.0f;
                }
                lds_barrier();
            }
        } else {
            for (int s = 0; s < 4; s++) lds_barrier();
        }
    }

    if constexpr (kTotals) {
#pragma unroll
        for (int a = 0; a < R; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = tot[a][b];
    }
    // the slices' sums meet in slice 0's waves, through the (now idle) stages, lane-minor so that
    // the accesses are conflict-free
    if constexpr (KS > 1) {
        float *red = L.red;
        constexpr int kPer = Lds::kPer;
        constexpr int kUnion = sizeof L.b > sizeof L.red ? sizeof L.b : sizeof L.red;
        constexpr int kFit = kUnion / (int)(sizeof(float) * kPer * RG);  // slices at a time
#pragma unroll
        for (int z0 = 1; z0 < KS; z0 += kFit) {
            if (z0 > 1) lds_barrier();
            if (ks >= z0 && ks < z0 + kFit) {
#pragma unroll
                for (int a = 0; a < R; a++)
#pragma unroll
                    for (int b = 0; b < NB; b++)
#pragma unroll
                        for (int x = 0; x < 4; x++)
                            red[((ks - z0) * RG + rg) * kPer + ((a * NB + b) * 4 + x) * 64 + lane] = acc[a][b][x];
            }
            lds_barrier();
            if (ks == 0) {
#pragma unroll
                for (int a = 0; a < R; a++)
#pragma unroll
                    for (int b = 0; b < NB; b++)
#pragma unroll
                        for (int x = 0; x < 4; x++) {
                            // summed as a tree: fewer roundings at the full sum's magnitude
                            float v[kFit];
                            const int n = KS - z0 < kFit ? KS - z0 : kFit;
#pragma unroll
                            for (int z = 0; z < n; z++)
                                v[z] = red[(z * RG + rg) * kPer + ((a * NB + b) * 4 + x) * 64 + lane];
#pragma unroll
                            for (int st = 1; st < n; st <<= 1)
#pragma unroll
                                for (int z = 0; z + st < n; z += 2 * st) v[z] += v[z + st];
                            acc[a][b][x] += v[0];
                        }
            }
        }
        if (ks) return;
    }
    // D layout (16x16 f32): lane l holds rows 4*(l/16)+x, column l%16.  Rows index weights (A
    // operand), columns tokens (B operand).
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int j = j0 + 16 * b + c;
        if (j >= g.N) continue;
        float *o = g.out + (size_t)j * g.ld + i0 + 4 * q;
#pragma unroll
        for (int a = 0; a < R; a++) {
            const int i = i0 + 16 * a + 4 * q;
            if (i + 3 < g.M && (g.ld & 3) == 0) {
                *(f4 *)(o + 16 * a) = acc[a][b];
            } else {
#pragma unroll
                for (int x = 0; x < 4; x++)
                    if (i + x < g.M) o[16 * a + x] = acc[a][b][x];
            }
        }
    }
}

// ------------------------------------------------------------------ activation staging
// fp32 rows [N][K] -> the grouped kernel's operand form of cuda_quantize_mmq_q8_1's output
// (per 32 values d = amax/127, q = rint(x*127/amax) clamped to +-127, ds = f16(d * sum x);
// gemm_q4k.cu:327-358): q8 as f16 integers [N][K] in the operands' element order
// (gemm_ops.hpp), the f16 ds [N][K/32], the running-scale
// ratio rho_s = d8eff_{s-1} / d8eff_s [N][K/32] and d8eff at the end of every 256 values
// [N][K/256].  d8eff is the last nonzero f16 d8 at or before s in s's window of 32 sub-blocks
// (1024 values), 1 before the window's first.  K a multiple of 256.  One wave per row.
constexpr int kStageThreads = 256;

__global__ void __launch_bounds__(kStageThreads) stage_f32_kernel(const float *__restrict__ x, int K, int N,
                                                                  _Float16 *__restrict__ q8, float *__restrict__ rho,
                                                                  uint16_t *__restrict__ dsv,
                                                                  float *__restrict__ dlast) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * (kStageThreads / 64) + (threadIdx.x >> 6);
    if (row >= N) return;
    const int nsub = K / 32;
    const float4 *xr = (const float4 *)(x + (size_t)row * K);
    _Float16 *qrow = q8 + (size_t)row * K;
    const uint64_t below = (1ull << lane) - 1;                       // the lanes before this one ..
    const uint64_t window = lane < 32 ? 0xFFFFFFFFull : ~0xFFFFFFFFull;  // .. and those of its window
    for (int b0 = 0; b0 < nsub; b0 += 64) {
        const int b = b0 + lane;
        float d8 = 0.0f;
        if (b < nsub) {
            // the arithmetic of quantize_q8_1_kernel (router.hip), so the values agree bit
            // for bit with cuda_quantize_mmq_q8_1
            float xv[32];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4 v = xr[8 * b + i];
                xv[4 * i] = v.x; xv[4 * i + 1] = v.y; xv[4 * i + 2] = v.z; xv[4 * i + 3] = v.w;
            }
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(xv[i]));
            const float d = amax / 127.0f;
            const float id = (amax > 0.0f) ? 127.0f / amax : 0.0f;
            float sum = 0.0f;
            uint32_t o[16];
#pragma unroll
            for (int i = 0; i < 32; i++) sum += xv[i];
#pragma unroll
            for (int i = 0; i < 16; i++) {  // the operands' element order: values 0 2 | 1 3 of each four
                const int v = 4 * (i / 2) + (i & 1);
                float r0 = rintf(xv[v] * id), r1 = rintf(xv[v + 2] * id);
                r0 = fminf(fmaxf(r0, -127.0f), 127.0f);
                r1 = fminf(fmaxf(r1, -127.0f), 127.0f);
                o[i] = h2u(h2{(_Float16)r0, (_Float16)r1});
            }
            float dsum = d * sum;
            asm volatile("" : "+v"(dsum));  // fp32 product, then the f16 rounding
            const uint16_t dh = f2h_bits(d);
            d8 = h2f(dh);
            dsv[(size_t)row * nsub + b] = f2h_bits(dsum);
            // a block whose d rounds to f16 zero (amax < 2^-25 * 127) still has quants up to
            // +-127; its values d8 * q8 are zero, and so are the staged operands (the running
            // scale skips the block)
            const uint32_t keep = d8 != 0.0f ? ~0u : 0u;
            uint4 *dst = (uint4 *)(qrow + 32 * b);
#pragma unroll
            for (int i = 0; i < 4; i++)
                dst[i] = make_uint4(o[4 * i] & keep, o[4 * i + 1] & keep, o[4 * i + 2] & keep, o[4 * i + 3] & keep);
        }
        // running scale: the last nonzero d8 before each block in its window
        const uint64_t m = __ballot(d8 != 0.0f) & below & window;
        const float prev_in = __shfl(d8, m ? 63 - __builtin_clzll(m) : 0);
        const float prev = m ? prev_in : 1.0f;
        const float cur = d8 != 0.0f ? d8 : prev;
        if (b < nsub) {
            rho[(size_t)row * nsub + b] = prev / cur;
            if ((b & 7) == 7) dlast[(size_t)row * (nsub / 8) + b / 8] = cur;
        }
    }
}

int launch_stage_f32(const float *x, int K, int N, StagedAct sa, hipStream_t s) {
    hipLaunchKernelGGL(stage_f32_kernel, dim3((N + 3) / 4), dim3(kStageThreads), 0, s, x, K, N, sa.q8, sa.rho, sa.ds,
                       sa.dlast);
    return check_launch("stage_f32");
}

static int device_cus_gemm() {
    static int cus = 0;
    if (!cus) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            cus = n;
        else
            cus = 256;
    }
    return cus;
}

// The workgroup shapes and what each costs: t tiles on C CUs, nsb super-blocks in ks slices, take
//   c0 + ceil(t / C) (c1 ceil(nsb / ks) + c2) + t / C (c3 nsb / ks + c4)  us:
// the launch; the rounds, each as long as its longest slice; and what the tiles cost each other (a
// wave's issue rate and the memory).  Where a shape's LDS and registers let two workgroups share a CU, a
// second one is not free: two rounds of the 64 x 64 tile of two slices take 1.7 times one.  Constants
// fitted to 891 sizes (M 64-10^4, K 256-12,288, N 1-2,350, both types; rms of the shapes near the
// best 8 % Q4_K, 15 % Q6_K): the choice is 2 % slower than the fastest shape on average and 23 % at worst.
// Large products take the wide tiles (fewest conversions and LDS reads per MFMA), small ones
// narrow tiles with K in up to 16 slices, so that the launch still covers the chip.  Shapes 8 to 11 are
// for few tiles of long rows, above all of Q6_K, whose super-blocks take a wave longest:
// M = 1836, K = 8960, N = 39 38.3 us without them, 26 with; 1359 x 4352, N = 776 74 and 59.
struct GemmShape {
    int r, rg, ks, nb;
    double q4[5], q6[5];
};
#define MNEMO_GEMM_SHAPES(X) \
    X(0, 2, 8, 1, 8, {0, 5.92, 5.13, 0.28, 20.42}, {5.99, 9.02, 0.81, 0.26, 21.96})     /* 256 x 128 */  \
    X(1, 2, 4, 2, 8, {3.88, 6.19, 2.18, 0.43, 10.28}, {1.98, 10.28, 0.08, 0.24, 13.92}) /* 128 x 128 */  \
    X(2, 2, 4, 2, 4, {4.18, 3.86, 0.91, 0.82, 4.56}, {3.09, 6.91, 0, 0.76, 6.43})       /* 128 x 64 */   \
    X(3, 1, 4, 2, 4, {5.73, 2.5, 0, 0.14, 1.08}, {4.58, 4.06, 0, 0, 1.12})              /* 64 x 64 */    \
    X(4, 1, 4, 4, 4, {2.87, 3.98, 1.95, 1.86, 0.5}, {1.13, 6.19, 2.13, 3.57, 0})        /* 64 x 64 */    \
    X(5, 1, 4, 4, 2, {4.82, 2.6, 0.94, 1.44, 0}, {3.94, 4.85, 0, 3.38, 0})              /* 64 x 32 */    \
    X(6, 1, 2, 8, 2, {4.97, 3.24, 0.26, 2.02, 0}, {2.34, 6.45, 0, 2.45, 0})             /* 32 x 32 */    \
    X(7, 2, 1, 8, 1, {6.16, 2.17, 0, 1.07, 0}, {2.96, 5.78, 0, 1.34, 0})                /* 32 x 16 */    \
    X(8, 1, 1, 16, 1, {5.98, 2.23, 0, 2.87, 0}, {6.27, 2.01, 0, 8.09, 0})               /* 16 x 16 */    \
    X(9, 1, 4, 2, 8, {1.92, 4.37, 2.82, 0.84, 3.36}, {1.51, 5.22, 2.56, 0.83, 3.23})    /* 64 x 128 */   \
    X(10, 1, 2, 4, 4, {3.57, 3.16, 1.69, 1.11, 0}, {4.74, 4.17, 0, 1.01, 0})            /* 32 x 64 */    \
    X(11, 1, 1, 8, 2, {5.81, 2.33, 0, 1.9, 0}, {5.05, 3.3, 0, 1.52, 0})                 /* 16 x 32 */
#define MNEMO_GEMM_SHAPE(I_, R_, RG_, KS_, NB_, ...) {R_, RG_, KS_, NB_, __VA_ARGS__},
static const GemmShape kShapes[] = {MNEMO_GEMM_SHAPES(MNEMO_GEMM_SHAPE)};

template <int TYPE, int I, int R, int RG, int KS, int NB>
static void gemm_shape_launch(const GemmArgs &g, dim3 grid, hipStream_t stream) {
    constexpr bool kOnce = TYPE == kTypeQ6K || GemmLds<TYPE, R, RG, KS, NB>::kTotals;
    if constexpr (TYPE == kTypeQ4K && I == 0) {
        if (g.K == 256) {
            hipLaunchKernelGGL((gemm_q8_1_kernel<TYPE, R, RG, KS, NB, true>), grid, dim3(64 * RG * KS), 0, stream, g);
            return;
        }
    }
    hipLaunchKernelGGL((gemm_q8_1_kernel<TYPE, R, RG, KS, NB, kOnce>), grid, dim3(64 * RG * KS), 0, stream, g);
}

static int gemm_tiles(int n, int tile) { return (int)(((long)n + tile - 1) / tile); }

// The workgroup shape for a product, and the rows and tokens of one launch: all of them, unless even
// the smallest tile's rows would span 4 GiB (K above 10^8), where launches of fewer rows take turns.
struct GemmPlan {
    int shape, rows, toks;
};

static GemmPlan gemm_plan(int type, int M, int K, int N, int cus) {
    constexpr size_t kSpan = 0xFFFFFFFFu;
    const int nsb = K / 256;
    const size_t wrow = (size_t)nsb * (type == kTypeQ4K ? kQ4KBytes : kQ6KBytes), arow = (size_t)(K / 128) * kQ81Bytes;
    // the first pass takes the shapes whose tiles fit, the second, if there was none, any shape
    // over fewer rows (a multiple of 4 of them where it can be, for the stores' alignment)
    for (;;) {
        GemmPlan p{-1, M, N};
        double least = 0;
        for (int i = 0; i < (int)(sizeof kShapes / sizeof kShapes[0]); i++) {
            const GemmShape &h = kShapes[i];
            const double *c = type == kTypeQ4K ? h.q4 : h.q6;
            if ((size_t)std::min(M, 16 * h.r * h.rg) * wrow > kSpan || (size_t)std::min(N, 16 * h.nb) * arow > kSpan)
                continue;
            if (i && gemm_tiles(N, 16 * h.nb) > 65535) continue;  // the grid's second dimension
            // (Q4_K's wide tiles round twice per sub-block, which shows in a sum of one super-block: of them
            // only shape 0 has a form that rounds once)
            if (type == kTypeQ4K && nsb == 1 && h.r * h.nb > 8 && i) continue;
            const long tiles = (long)gemm_tiles(M, 16 * h.r * h.rg) * gemm_tiles(N, 16 * h.nb);
            const double t = c[0] + (double)((tiles + cus - 1) / cus) * (c[1] * ((nsb + h.ks - 1) / h.ks) + c[2]) +
                             (double)tiles / cus * (c[3] * nsb / h.ks + c[4]);
            if (p.shape < 0 || t < least) {
                p.shape = i;
                least = t;
            }
        }
        if (p.shape >= 0) return p;
        const int rows = (int)std::min<size_t>(M, kSpan / wrow);
        M = rows > 4 ? rows & ~3 : rows;
        N = (int)std::min<size_t>(N, kSpan / arow);
    }
}

// For the tests: the plan of a product on a device of cus CUs.  Returns the shape's index and writes
// its tile (rows, tokens, slices of K) and the rows and tokens of one launch.
extern "C" int mnemo_internal_gemm_plan(int type, int M, int K, int N, int cus, int out[5]) {
    const GemmPlan p = gemm_plan(type, M, K, N, cus);
    const GemmShape &h = kShapes[p.shape];
    const int v[5] = {16 * h.r * h.rg, 16 * h.nb, h.ks, p.rows, p.toks};
    for (int i = 0; i < 5; i++) out[i] = v[i];
    return p.shape;
}

int launch_gemm_q8_1(int type, const void *w, const void *act, float *out, int M, int K, int N,
                     hipStream_t stream) {
    if (!w || !act || !out || M <= 0 || N <= 0 || K <= 0 || K % 256 != 0)
        return set_error(kErrBadArg, "gemm: need non-null pointers, M, N > 0 and K %% 256 == 0");
    if (type != kTypeQ4K && type != kTypeQ6K) return set_error(kErrUnsupportedType, "gemm: unsupported type %d", type);
    if (((uintptr_t)out & 15) != 0) return set_error(kErrBadArg, "gemm: output must be 16-byte aligned");
    if (((uintptr_t)act & 3) != 0) return set_error(kErrBadArg, "gemm: activation blocks must be 4-byte aligned");
    // activations are read as Q8_1 blocks and converted per tile: nothing is allocated, so
    // the call may sit inside a graph capture
    const GemmPlan plan = gemm_plan(type, M, K, N, device_cus_gemm());
    const GemmShape &h = kShapes[plan.shape];
    const size_t wrow = (size_t)(K / 256) * (type == kTypeQ4K ? kQ4KBytes : kQ6KBytes);
    const size_t arow = (size_t)(K / 128) * kQ81Bytes;
    for (int r0 = 0; r0 < M; r0 += plan.rows)
        for (int t0 = 0; t0 < N; t0 += plan.toks) {
            const GemmArgs g{(const uint8_t *)w + r0 * wrow, (const uint8_t *)act + t0 * arow, out + (size_t)t0 * M + r0,
                             std::min(M - r0, plan.rows), K, std::min(N - t0, plan.toks), M};
            const dim3 grid(gemm_tiles(g.M, 16 * h.r * h.rg), gemm_tiles(g.N, 16 * h.nb));
#define MNEMO_GEMM(I_, R_, RG_, KS_, NB_, ...)                                                              \
            case I_:                                                                                            \
                if (type == kTypeQ4K) gemm_shape_launch<kTypeQ4K, I_, R_, RG_, KS_, NB_>(g, grid, stream);      \
                else gemm_shape_launch<kTypeQ6K, I_, R_, RG_, KS_, NB_>(g, grid, stream);                       \
                break;
            switch (plan.shape) { MNEMO_GEMM_SHAPES(MNEMO_GEMM) }
#undef MNEMO_GEMM
        }
    return check_launch("gemm_q8_1");
}

}  // namespace mnemo
