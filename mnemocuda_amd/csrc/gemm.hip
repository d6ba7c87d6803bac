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
//   * The fp32 rescale is a running scale: the accumulator holds the sum in units of the
//     current (row scale d) x (token scale d8).  Every sub-block multiplies acc by
//     rho = d8_prev / d8 of the token (one multiply per output per sub-block) and the MFMA
//     then adds the sub-block's products straight into that rescaled accumulator, so t is
//     never formed on its own: each step rounds like an fp32 sum of the exact products onto
//     acc * rho.  At a super-block boundary the rows' acc is multiplied by d_prev / d once.  The epilogue
//     multiplies by the last d8 * d.  A zero scale leaves the running scale unchanged and
//     zeroes its block's operand (its products are zero).
//   * Q4_K's min term, sum_s -(dmin*m_s) * ds_js, is one more product over the sub-block
//     index: -dmin*m (an f16 times a 6-bit integer, 17 significant bits) is split into an
//     f16 hi + lo pair that is exact, ds is an f16 already, and two MFMAs per 32 sub-blocks
//     add it to the finished absolute accumulator.
//   Against the fp64 value the roundings are the rescale multiply and the MFMA's fp32
//   accumulation per output per sub-block, and the rho quotients (measured ~1e-7 relative
//   L2).
//
// An int8 MFMA does not fit this product on gfx950: v_mfma_i32_16x16x64_i8 sums 64 values,
// two sub-blocks with different token scales, and the 32-deep v_mfma_i32_16x16x32_i8 runs
// at the f16 MFMA's rate (16 cycles for 16x16x32, measured) while needing three VALU
// operations per output per sub-block (int -> float, the product of the row and token
// scales, the fma) where the exact f16 form needs one.
#include <algorithm>

#include "gemm_ops.hpp"
#include "mnemo_common.hpp"
#include "mnemo_internal.hpp"

namespace mnemo {

// ------------------------------------------------------------------ tiled kernel
// A workgroup computes a 128 x 128 tile (weight rows x tokens) over one K slice (blockIdx.z
// of `splits`, whole super-blocks).  Its waves form a 2 (rows: 64 each) x kWC (tokens) x 2
// (sub-block parity) grid: wave (wi, wj, kh) multiplies rows wi .. wi+63 with tokens
// wj .. wj+kWTok-1 over sub-block kh of every 64-wide K step (the step's sub-blocks 2ks and
// 2ks + 1); the two parities are summed through LDS at the end.  All threads load and
// convert the step's weights and activations once into LDS: thread t owns weight row /
// token t / kParts and part t % kParts (kVP values) of the step.
#ifndef MNEMO_GEMM_THREADS
#define MNEMO_GEMM_THREADS 512
#endif
constexpr int kThreads = MNEMO_GEMM_THREADS;  // 512 or 1024
constexpr int kWaves = kThreads / 64;
constexpr int kBM = 128, kBN = 128;
constexpr int kKS = 64;                // K per step
constexpr int kWC = kWaves / 4;        // token groups
constexpr int kWTok = kBN / kWC;       // tokens per wave
constexpr int kNB = kWTok / 16;        // 16-token MFMA columns per wave
constexpr int kParts = kThreads / 128; // loader parts per row and step
constexpr int kVP = kKS / kParts;      // values per part (16 or 8)
static_assert(kVP == 8 || kVP == 16, "loader parts of 8 or 16 values");
// raw ring slots: loads run kPF-2 steps ahead of their conversion
#ifndef MNEMO_GEMM_PF
#define MNEMO_GEMM_PF 3
#endif
constexpr int kPF = MNEMO_GEMM_PF;
// lcm(kPF, 3 LDS stages, 4 steps per super-block): every ring slot, stage and super-block
// boundary of the unrolled loop is a compile-time constant
constexpr int kUnroll = 12;
static_assert(kUnroll % kPF == 0, "ring size must divide the unroll");

// kVP raw bytes as dwords
struct PartBytes {
    uint32_t w[kVP / 4];
};
__device__ __forceinline__ PartBytes ld_part(const uint8_t *p) {
    PartBytes r;
    if constexpr (kVP == 16) {
        const uint4 v = ld16(p);
        r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
    } else {
        const uint2 v = ld8(p);
        r.w[0] = v.x; r.w[1] = v.y;
    }
    return r;
}
__device__ __forceinline__ PartBytes ld_part_a2(const uint8_t *p) {
    PartBytes r;
    if constexpr (kVP == 16) {
        const uint4 v = ld16_a2(p);
        r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
    } else {
        const uint2 v = ld8_a2(p);
        r.w[0] = v.x; r.w[1] = v.y;
    }
    return r;
}

struct RawW {
    uint4 h;         // Q4_K: the super-block header (d, dmin, 12 scale bytes)
    PartBytes a, b;  // Q4_K: a = qs bytes;  Q6_K: a = ql bytes, b = qh bytes
    uint32_t s, dd;  // Q6_K: the int8 scale of the values, f16 d
};
struct RawA {
    PartBytes q;  // int8 quants
    uint32_t ds;  // half2 (d8, ds) of their 32-value sub-block
};

// Part p of step ks covers K columns kVP*p .. +kVP-1 of the step: sub-block 2(ks%4) + c/32 of
// super-block ks/4, positions c%32 .. (c = kVP*p).
// Q4_K: qs bytes 32(ks%4) + c%32 .., the low (c < 32) or high nibbles.
__device__ __forceinline__ void load_w_q4k(const uint8_t *__restrict__ wrow, int ks, int p, RawW &r) {
    const uint8_t *blk = wrow + (size_t)(ks >> 2) * kQ4KBytes;
    r.h = ld16(blk);
    r.a = ld_part(blk + 16 + 32 * (ks & 3) + ((kVP * p) & 31));
}
// Q6_K: values v0 = 64(ks%4) + c of the super-block: half hh = (ks%4)/2, group
// grp = 2(ks%2) + c/32, positions l0 = c%32: ql bytes 64hh + 32(grp%2) + l0 (high nibbles if
// grp >= 2), qh bytes 32hh + l0 at bit 2grp, scale byte 8hh + 2grp + l0/16.
__device__ __forceinline__ void load_w_q6k(const uint8_t *__restrict__ wrow, int ks, int p, RawW &r) {
    const uint8_t *blk = wrow + (size_t)(ks >> 2) * kQ6KBytes;
    const int c = kVP * p, hh = (ks & 3) >> 1, grp = 2 * (ks & 1) + (c >> 5), l0 = c & 31;
    r.a = ld_part_a2(blk + 64 * hh + 32 * (grp & 1) + l0);
    r.b = ld_part_a2(blk + 128 + 32 * hh + l0);
    uint8_t sc;
    uint16_t dd;
    __builtin_memcpy(&sc, blk + 192 + 8 * hh + 2 * grp + (l0 >> 4), 1);
    __builtin_memcpy(&dd, blk + 208, 2);
    r.s = sc;
    r.dd = dd;
}
// Activations of step ks, part p: values 64ks + kVP*p .. of the token's Q8_1 MMQ row
// (block v/128, sub-block (v/32)%4).
__device__ __forceinline__ void load_a(const uint8_t *__restrict__ arow, int ks, int p, RawA &r) {
    const int v0 = ks * kKS + kVP * p;
    const uint8_t *blk = arow + (size_t)(v0 >> 7) * kQ81Bytes;
    __builtin_memcpy(&r.ds, blk + 4 * ((v0 >> 5) & 3), 4);
    r.q = ld_part(blk + 16 + (v0 & 127));
}

// f16 tiles of 64 K-columns per row = 8 chunks of 16 B (a row is 128 B, half of the 64 x 4 B
// LDS banks), stored without padding with the chunk index XOR-ed by (row / 2) % 8: the 16
// rows of an MFMA fragment read (one chunk each) cover the 64 banks once, and so do the
// lanes of a conversion store.
__device__ __forceinline__ int tile_off(int row, int chunk) { return row * kKS + ((chunk ^ ((row >> 1) & 7)) << 3); }
// the part's converted values (kVP / 2 dwords of f16 pairs) into its chunks
__device__ __forceinline__ void put_part(_Float16 *tile, int row, int p, const uint32_t (&o)[kVP / 2]) {
#pragma unroll
    for (int c = 0; c < kVP / 8; c++)
        *(uint4 *)(tile + tile_off(row, (kVP / 8) * p + c)) = make_uint4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
}

// One LDS stage: the step's operand tiles and the running-scale factors.
template <int TYPE>
struct Stage {
    static constexpr int kPlanes = TYPE == kTypeQ4K ? 1 : 2;
    _Float16 a[kPlanes][kBM * kKS];  // weights: sc*q (Q4_K) or the two Q6_K planes
    _Float16 b[kBN * kKS];           // q8
    float rho[2][kBN];               // token scale ratio of sub-block 2ks + p
    float sig[kBM];                  // row scale ratio (written at super-block starts)
};

// Running scales of a loader thread: the last nonzero d of its weight row (part 0 threads)
// and the last nonzero d8 of its token for the sub-block parity of its part (the first part
// of each sub-block).  Both start at 1.
struct LoaderState {
    float deff, d8eff;
};

__device__ __forceinline__ void row_scale_step(float d, int ks, int p, float *sig, int row, LoaderState &ls, bool live) {
    if (p == 0 && (ks & 3) == 0 && live) {  // super-block start: the row scale changes
        const float dn = d != 0.0f ? d : ls.deff;
        sig[row] = ls.deff * __builtin_amdgcn_rcpf(dn);
        ls.deff = dn;
    }
}

__device__ __forceinline__ void store_w_q4k(const RawW &r, int ks, int p, Stage<kTypeQ4K> &st, int row,
                                            LoaderState &ls, bool live) {
    const int c = kVP * p;
    const int j = 2 * (ks & 3) + (c >> 5);
    uint32_t sc, m;
    q4k_scale_min(r.h.y, r.h.z, r.h.w, j, sc, m);
    const float d = h2f(r.h.x & 0xFFFFu);
    if (d == 0.0f) sc = 0;  // the block's products are zero
    // the pair (sc, -1024 sc) from sc under the 0x64 exponent; high nibbles are taken in
    // place as the bytes 16 q with (sc / 16, -64 sc): (1024 + 16 q) sc / 16 - 64 sc = q sc
    const bool hi = (c >> 5) != 0;
    const h2 F = hi ? h2{(_Float16)0.0625f, (_Float16)0.0625f} : h2{(_Float16)1.0f, (_Float16)1.0f};
    const h2 mk = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    const h2 S = __builtin_elementwise_fma(magic_pair(sc, 0x04000400u), F, F * mk);
    const h2 N = S * mk;
    const uint32_t msk = hi ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
    uint32_t o[kVP / 2];
#pragma unroll
    for (int k = 0; k < kVP / 4; k++) {
        const uint32_t w = r.a.w[k] & msk;
        o[2 * k] = q4_scaled(w, kSelLo, S, N);
        o[2 * k + 1] = q4_scaled(w, kSelHi, S, N);
    }
    put_part(st.a[0], row, p, o);
    row_scale_step(d, ks, p, st.sig, row, ls, live);
}

// Q6_K planes (sc - b)(q - 32) and b(q - 32), b = sc & 1
__device__ __forceinline__ void store_w_q6k(const RawW &r, int ks, int p, Stage<kTypeQ6K> &st, int row,
                                            LoaderState &ls, bool live) {
    const int c = kVP * p, grp = 2 * (ks & 1) + (c >> 5);
    const float d = h2f(r.dd);
    int sc = (int)(int8_t)(r.s & 0xFF);
    if (d == 0.0f) sc = 0;
    const int b1 = sc & 1;
    const _Float16 e = (_Float16)(float)(sc - b1), bb = (_Float16)(float)b1;
    const h2 E = {e, e}, B = {bb, bb};
    const int shl = grp >= 2 ? 4 : 0;
    uint32_t o1[kVP / 2], o2[kVP / 2];
#pragma unroll
    for (int k = 0; k < kVP / 4; k++) {
        const uint32_t lo = (r.a.w[k] >> shl) & 0x0F0F0F0Fu;
        const uint32_t qh = r.b.w[k];
        const uint32_t hi = (2 * grp <= 4 ? (qh << (4 - 2 * grp)) : (qh >> (2 * grp - 4))) & 0x30303030u;
        const uint32_t v = lo | hi;
        const h2 c0 = q6_centered(v, kSelLo), c1 = q6_centered(v, kSelHi);
        o1[2 * k] = h2u(c0 * E);
        o1[2 * k + 1] = h2u(c1 * E);
        o2[2 * k] = h2u(c0 * B);
        o2[2 * k + 1] = h2u(c1 * B);
    }
    put_part(st.a[0], row, p, o1);
    put_part(st.a[1], row, p, o2);
    row_scale_step(d, ks, p, st.sig, row, ls, live);
}

template <int TYPE>
__device__ __forceinline__ void store_a(const RawA &r, int p, Stage<TYPE> &st, int row, LoaderState &ls, bool live) {
    const float d8 = h2f(r.ds & 0xFFFFu);
    const bool zero = d8 == 0.0f;  // x = 0 * q8 = 0 whatever the quants hold (a block whose d
                                   // rounds to f16 zero keeps quants up to +-127)
    uint32_t o[kVP / 2];
#pragma unroll
    for (int k = 0; k < kVP / 4; k++) q8x4_exact(zero ? 0u : r.q.w[k], o[2 * k], o[2 * k + 1]);
    put_part(st.b, row, p, o);
    const int c = kVP * p;
    if ((c & 31) == 0 && live) {  // first part of a sub-block: its token scale ratio
        const float dn = zero ? ls.d8eff : d8;
        st.rho[c >> 5][row] = ls.d8eff * __builtin_amdgcn_rcpf(dn);
        ls.d8eff = dn;
    }
}

template <int TYPE>
__device__ __forceinline__ void load_step(const uint8_t *wrow, const uint8_t *arow, int ks, int p, RawW &rw,
                                          RawA &ra) {
    if (TYPE == kTypeQ4K) load_w_q4k(wrow, ks, p, rw);
    else load_w_q6k(wrow, ks, p, rw);
    load_a(arow, ks, p, ra);
}
template <int TYPE>
__device__ __forceinline__ void store_step(const RawW &rw, const RawA &ra, int ks, int p, Stage<TYPE> &st, int row,
                                           LoaderState &ls, bool live) {
    if constexpr (TYPE == kTypeQ4K) store_w_q4k(rw, ks, p, st, row, ls, live);
    else store_w_q6k(rw, ks, p, st, row, ls, live);
    store_a<TYPE>(ra, p, st, row, ls, live);
}

// A wave's operands of one step: fragments of its sub-block (kh) for 4 x kNB MFMA tiles, the
// token scale ratios of its 16-token columns, and (at super-block starts) the row ratios of
// the rows its accumulators hold.
template <int TYPE>
struct Frags {
    h8 a[Stage<TYPE>::kPlanes][4];
    h8 b[kNB];
    float rho[kNB];
};
template <int TYPE>
__device__ __forceinline__ void read_frags(const Stage<TYPE> &st, int wi, int wj, int kh, int lane, Frags<TYPE> &f) {
    const int chunk = 4 * kh + (lane >> 4);
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int ra = wi + 16 * t + (lane & 15);
#pragma unroll
        for (int p = 0; p < Stage<TYPE>::kPlanes; p++) f.a[p][t] = *(const h8 *)(st.a[p] + tile_off(ra, chunk));
    }
#pragma unroll
    for (int t = 0; t < kNB; t++) {
        const int rb = wj + 16 * t + (lane & 15);
        f.b[t] = *(const h8 *)(st.b + tile_off(rb, chunk));
        f.rho[t] = st.rho[kh][rb];
    }
}

// acc = acc * rho, then the MFMA adds the step's exact products to the rescaled accumulator
// (rounded as fp32 sums onto it)
// (at a super-block start the row ratios come first, read from the step's own stage, which
// no thread writes during the step)
template <int TYPE>
__device__ __forceinline__ void mfma_step(const Frags<TYPE> &f, const Stage<TYPE> &st, int wi, int lane,
                                          f4 (&acc)[4][kNB], bool sb_start) {
    if (sb_start) {
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const f4 sg = *(const f4 *)(st.sig + wi + 16 * a + 4 * (lane >> 4));
#pragma unroll
            for (int b = 0; b < kNB; b++) acc[a][b] *= sg;
        }
    }
#pragma unroll
    for (int b = 0; b < kNB; b++) {
#pragma unroll
        for (int a = 0; a < 4; a++) {
            acc[a][b] *= f.rho[b];
            acc[a][b] = mfma(f.a[0][a], f.b[b], acc[a][b]);
            if constexpr (TYPE == kTypeQ6K) acc[a][b] = mfma(f.a[1][a], f.b[b], acc[a][b]);
        }
    }
}

struct GemmArgs {
    const uint8_t *W;  // weights [M][K]
    const uint8_t *A;  // Q8_1 MMQ rows [N]
    float *out;
    int M, K, N, splits;
    int out_ld;
};

template <int TYPE, bool ATOMIC>
__global__ void __launch_bounds__(kThreads) gemm_q8_1_kernel(GemmArgs g) {
    __shared__ __align__(16) Stage<TYPE> lds[3];
    __shared__ float dlast[kBM], d8last[2][kBN];
    // Q4_K min term: the operands of the split's super-blocks (up to kMhSb), kept as the
    // loaders pass them -- per weight row and super-block the 8 six-bit mins (one byte each)
    // and dmin, per token and sub-block the f16 ds of its Q8_1 block
    constexpr int kMhSb = 16;
    constexpr int kQ4 = TYPE == kTypeQ4K;
    __shared__ uint2 mhm[kQ4 ? kBM * kMhSb : 1];
    __shared__ uint16_t mhd[kQ4 ? kBM * kMhSb : 1];
    __shared__ __align__(16) uint16_t dsk[kQ4 ? kBN * kMhSb * 8 : 8];
    const int tid = threadIdx.x;
    // the wave index as a scalar, so that every per-wave decision below is a scalar branch
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = g.K;
    const int wi = (wave & 1) * 64, wj = ((wave >> 1) % kWC) * kWTok, kh = wave / (2 * kWC);
    const int bbytes = TYPE == kTypeQ4K ? kQ4KBytes : kQ6KBytes;
    const size_t wrow_bytes = (size_t)(K / 256) * bbytes;
    // this split's super-blocks [sb0, sb1) = steps [ks0, ks1)
    const int nsb = K / 256;
    const int sb0 = (int)((long)nsb * blockIdx.z / g.splits), sb1 = (int)((long)nsb * (blockIdx.z + 1) / g.splits);
    const int ks0 = 4 * sb0, ks1 = 4 * sb1, last = ks1 - 1;
    const int i0 = blockIdx.x * kBM, j0 = blockIdx.y * kBN;

    // loader role: thread -> (row / token lr, part lp); rows past the end re-read the last
    const int lr = tid / kParts, lp = tid % kParts;
    const uint8_t *wrow = g.W + (size_t)min(i0 + lr, g.M - 1) * wrow_bytes;
    const uint8_t *arow = g.A + (size_t)min(j0 + lr, g.N - 1) * (K / 128) * kQ81Bytes;
    LoaderState ls{1.0f, 1.0f};

    f4 acc[4][kNB];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < kNB; b++) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};

    // Pipeline: three LDS stages.  In step ks a wave multiplies the fragments of step ks
    // (read during step ks-1), reads the fragments of step ks+1 (its stage was completed
    // before the previous barrier), converts step ks+2 into the third stage, then meets
    // the barrier.  Raw blocks sit in a ring of kPF register slots, loaded kPF-2 steps
    // before their conversion.  Conversions past the last step fill idle stages and leave
    // the running scales alone.
    RawW rw[kPF];
    RawA ra[kPF];
#pragma unroll
    for (int p = 0; p < kPF; p++) load_step<TYPE>(wrow, arow, min(ks0 + p, last), lp, rw[p], ra[p]);
    const bool keep_min = TYPE == kTypeQ4K && sb1 - sb0 <= kMhSb;  // uniform
    // step q (relative to ks0) of the split: the loader of a row's first part keeps its mins
    // and dmin at the super-block's first step, the loader of a sub-block's first values its ds
    auto keep = [&](const RawW &w, const RawA &a, int q, bool first_step, bool live) {
        if (!keep_min || !live) return;
        if (lp == 0 && first_step) {
            mhm[lr * kMhSb + (q >> 2)] = q4k_mins(w.h);
            mhd[lr * kMhSb + (q >> 2)] = (uint16_t)(w.h.x >> 16);
        }
        if (((kVP * lp) & 31) == 0)
            dsk[lr * kMhSb * 8 + (q >> 2) * 8 + 2 * (q & 3) + ((kVP * lp) >> 5)] = (uint16_t)(a.ds >> 16);
    };
    store_step<TYPE>(rw[0], ra[0], ks0, lp, lds[0], lr, ls, true);
    keep(rw[0], ra[0], 0, true, true);
    store_step<TYPE>(rw[1], ra[1], ks0 + 1, lp, lds[1], lr, ls, ks0 + 1 < ks1);
    keep(rw[1], ra[1], 1, false, ks0 + 1 < ks1);
    lds_barrier();
    Frags<TYPE> fr;
    read_frags<TYPE>(lds[0], wi, wj, kh, lane, fr);

    for (int kb = ks0; kb < ks1; kb += kUnroll) {
#pragma unroll
        for (int p = 0; p < kUnroll; p++) {
            const int ks = kb + p;
            if (ks < ks1) {  // uniform
                // kb - ks0 is a multiple of kUnroll and ks0 of 4, so these are compile-time
                // constants
                const int r = p % kPF, b = p % 3;
                load_step<TYPE>(wrow, arow, min(ks + kPF, last), lp, rw[r], ra[r]);
                mfma_step<TYPE>(fr, lds[b], wi, lane, acc, p % 4 == 0);
                read_frags<TYPE>(lds[(b + 1) % 3], wi, wj, kh, lane, fr);
                store_step<TYPE>(rw[(r + 2) % kPF], ra[(r + 2) % kPF], ks + 2, lp, lds[(b + 2) % 3], lr, ls,
                                 ks + 2 < ks1);
                // (ks + 2 - ks0) % 4 == (p + 2) % 4: a compile-time test
                keep(rw[(r + 2) % kPF], ra[(r + 2) % kPF], ks + 2 - ks0, ((p + 2) & 3) == 0, ks + 2 < ks1);
                lds_barrier();
            }
        }
    }
    // absolute values: the last nonzero scales of each row and each token (per parity)
    if (lp == 0) dlast[lr] = ls.deff;
    if (((kVP * lp) & 31) == 0) d8last[(kVP * lp) >> 5][lr] = ls.d8eff;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; a++) {
        const f4 dr = *(const f4 *)(dlast + wi + 16 * a + 4 * (lane >> 4));
#pragma unroll
        for (int b = 0; b < kNB; b++) {
            const float dt = d8last[kh][wj + 16 * b + (lane & 15)];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[a][b][e] *= dr[e] * dt;
        }
    }

    // Q4_K min term, sum_s -(dmin*m_s)_i * ds_js, added to the absolute accumulator after
    // the loop, from the operands the loaders kept in LDS (up to 16 super-blocks per split;
    // reading the headers and the Q8_1 block heads again from memory touched every weight
    // line a second time and 4096 activation lines per workgroup).  Windows of 32 sub-blocks
    // (4 super-blocks), wave parity kh taking windows kh, kh+2, ...; lane group q = lane/16
    // holds super-block 4w + q of its row / token (K index 8q + s of the MFMA = sub-block s of
    // that super-block).
    if constexpr (TYPE == kTypeQ4K) {
        const int q = lane >> 4;
        const int nwin = (sb1 - sb0 + 3) / 4;
        for (int w = kh; w < nwin; w += 2) {
            const int sb = sb0 + 4 * w + q;
            const bool valid = sb < sb1;
            uint4 hdr[4], blk[kNB][2];
            if (keep_min) {  // the operands the loaders kept: no second pass over weights or activations
                const int rs = valid ? sb - sb0 : 0;
                h8 bd[kNB];
#pragma unroll
                for (int b = 0; b < kNB; b++) {
                    bd[b] = *(const h8 *)&dsk[(wj + 16 * b + (lane & 15)) * kMhSb * 8 + rs * 8];
                    if (!valid) bd[b] = h8{};
                }
#pragma unroll
                for (int a = 0; a < 4; a++) {
                    const int row = wi + 16 * a + (lane & 15);
                    h8 hi, lo;
                    q4k_min_operand_m(mhm[row * kMhSb + rs], valid ? mhd[row * kMhSb + rs] : 0u, hi, lo);
#pragma unroll
                    for (int b = 0; b < kNB; b++) acc[a][b] = mfma(lo, bd[b], mfma(hi, bd[b], acc[a][b]));
                }
                continue;
            }
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const uint8_t *rp = g.W + (size_t)min(i0 + wi + 16 * a + (lane & 15), g.M - 1) * wrow_bytes;
                hdr[a] = valid ? ld16(rp + (size_t)sb * kQ4KBytes) : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int b = 0; b < kNB; b++) {
                const uint8_t *ap = g.A +
                                    (size_t)min(j0 + wj + 16 * b + (lane & 15), g.N - 1) * (K / 128) * kQ81Bytes;
                blk[b][0] = valid ? ld16(ap + (size_t)(2 * sb) * kQ81Bytes) : make_uint4(0, 0, 0, 0);
                blk[b][1] = valid ? ld16(ap + (size_t)(2 * sb + 1) * kQ81Bytes) : make_uint4(0, 0, 0, 0);
            }
            h8 bd[kNB];
#pragma unroll
            for (int b = 0; b < kNB; b++) bd[b] = ds_operand(blk[b][0], blk[b][1]);
#pragma unroll
            for (int a = 0; a < 4; a++) {
                h8 hi, lo;
                q4k_min_operand(hdr[a], hi, lo);
#pragma unroll
                for (int b = 0; b < kNB; b++) acc[a][b] = mfma(lo, bd[b], mfma(hi, bd[b], acc[a][b]));
            }
        }
    }

    // sum the two parities: the kh = 1 waves hand their tiles to their kh = 0 counterparts
    // through the (now idle) stages, laid out lane-minor so the accesses are conflict-free
    __syncthreads();
    float *red = (float *)&lds[0] + (size_t)(wave % (kWaves / 2)) * (64 * kWTok);
    if (kh) {
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < kNB; b++)
#pragma unroll
                for (int e = 0; e < 4; e++) red[((a * kNB + b) * 4 + e) * 64 + lane] = acc[a][b][e];
    }
    __syncthreads();
    if (kh) return;
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < kNB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[a][b][e] += red[((a * kNB + b) * 4 + e) * 64 + lane];
    // D layout (16x16 f32): lane l holds rows 4*(l/16)+e, column l%16.  Rows index
    // weights (A operand), columns tokens (B operand).
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < kNB; b++) {
            const int j = j0 + wj + 16 * b + (lane & 15);
            const int ib = i0 + wi + 16 * a + 4 * (lane >> 4);
            if (j >= g.N) continue;
            float *o = g.out + (size_t)j * g.out_ld + ib;
            if (ATOMIC) {
                // to the wave's own (idle) reduction buffer, token-major, 16-byte groups
                // XOR-swizzled by token so that the row-wise reads below are conflict-free
                *(f4 *)(red + (16 * b + (lane & 15)) * 64 + (((4 * a + (lane >> 4)) ^ (lane & 15)) << 2)) = acc[a][b];
            } else if (ib + 3 < g.M && ((g.out_ld & 3) == 0)) {
                *(f4 *)o = acc[a][b];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (ib + e < g.M) o[e] = acc[a][b][e];
            }
        }
    if (ATOMIC) {
        // one atomic instruction per token covers 64 consecutive outputs (two cache lines);
        // the MFMA layout would spread each instruction over 16 token rows, which measured
        // twice as slow in the L2 atomic units
        const int ib = i0 + wi + lane;
        for (int t = 0; t < kWTok; t++) {
            const int j = j0 + wj + t;
            if (j >= g.N) break;
            if (ib < g.M)
                __hip_atomic_fetch_add(g.out + (size_t)j * g.out_ld + ib,
                                       red[t * 64 + ((((lane >> 2) ^ (t & 15)) << 2) | (lane & 3))], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ------------------------------------------------------------------ activation staging
// fp32 rows [N][K] -> the grouped kernel's operand form of cuda_quantize_mmq_q8_1's output
// (per 32 values d = amax/127, q = rint(x*127/amax) clamped to +-127, ds = f16(d * sum x);
// gemm_q4k.cu:327-358): q8 as f16 integers [N][K], the f16 ds [N][K/32], the running-scale
// ratio rho_s = d8eff_{s-1} / d8eff_s [N][K/32] and d8eff at the end of every window of 32
// sub-blocks (1024 values) [N][ceil(K/1024)].  d8eff is the last nonzero f16 d8 at or before s
// in s's window, 1 before the window's first.  One wave per row.
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
            for (int i = 0; i < 16; i++) {
                float r0 = rintf(xv[2 * i] * id), r1 = rintf(xv[2 * i + 1] * id);
                r0 = fminf(fmaxf(r0, -127.0f), 127.0f);
                r1 = fminf(fmaxf(r1, -127.0f), 127.0f);
                sum += xv[2 * i];
                sum += xv[2 * i + 1];
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
            if ((b & 31) == 31 || b == nsub - 1) dlast[(size_t)row * ((nsub + 31) / 32) + b / 32] = cur;
        }
    }
}

int launch_stage_f32(const float *x, int K, int N, StagedAct sa, hipStream_t s) {
    hipLaunchKernelGGL(stage_f32_kernel, dim3((N + 3) / 4), dim3(kStageThreads), 0, s, x, K, N, sa.q8, sa.rho, sa.ds,
                       sa.dlast);
    return check_launch("stage_f32");
}

__global__ void zero_kernel(float4 *__restrict__ p, long n4) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n4; i += (long)gridDim.x * blockDim.x)
        p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
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

int launch_gemm_q8_1(int type, const void *w, const void *act, float *out, int M, int K, int N,
                     hipStream_t stream) {
    if (!w || !act || !out || M <= 0 || N <= 0 || K <= 0 || K % 256 != 0)
        return set_error(kErrBadArg, "gemm: need non-null pointers, M, N > 0 and K %% 256 == 0");
    if (type != kTypeQ4K && type != kTypeQ6K) return set_error(kErrUnsupportedType, "gemm: unsupported type %d", type);
    if (((uintptr_t)out & 15) != 0) return set_error(kErrBadArg, "gemm: output must be 16-byte aligned");
    if (((uintptr_t)act & 3) != 0) return set_error(kErrBadArg, "gemm: activation blocks must be 4-byte aligned");
    const int tm = (M + kBM - 1) / kBM, tn = (N + kBN - 1) / kBN;
    // split K (whole super-blocks) while the split grid still fits the CUs once, keeping
    // at least 2 super-blocks per split
    const int nsb = K / 256;
    int splits = 1;
    while (2 * tm * tn * splits <= device_cus_gemm() && nsb / (splits * 2) >= 2) splits *= 2;
    if (((long)M * N) % 4 != 0) splits = 1;  // the fill kernel clears float4s
    // activations are read as Q8_1 blocks and converted per tile: nothing is allocated, so
    // the call may sit inside a graph capture
    GemmArgs g{};
    g.W = (const uint8_t *)w;
    g.A = (const uint8_t *)act;
    g.out = out;
    g.M = M;
    g.K = K;
    g.N = N;
    g.splits = splits;
    g.out_ld = M;
    if (splits > 1) {
        const long n = (long)M * N;
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)std::min<long>((n / 4 + 255) / 256, 4096)), dim3(256), 0,
                           stream, (float4 *)out, n / 4);
    }
    const dim3 grid(tm, tn, splits);
#define MNEMO_GEMM_LAUNCH(T_, A_) hipLaunchKernelGGL((gemm_q8_1_kernel<T_, A_>), grid, dim3(kThreads), 0, stream, g)
    if (type == kTypeQ4K) {
        if (splits > 1) MNEMO_GEMM_LAUNCH(kTypeQ4K, true);
        else MNEMO_GEMM_LAUNCH(kTypeQ4K, false);
    } else {
        if (splits > 1) MNEMO_GEMM_LAUNCH(kTypeQ6K, true);
        else MNEMO_GEMM_LAUNCH(kTypeQ6K, false);
    }
#undef MNEMO_GEMM_LAUNCH
    return check_launch("gemm_q8_1");
}

}  // namespace mnemo
