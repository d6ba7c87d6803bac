// gemm_grouped.hip -- grouped expert GEMMs of the MoE prefill (Q4_K / Q6_K x staged Q8_1 rows).
//
// An expert receives from one to a few hundred tokens, so its tokens are cut into tiles of at
// most kGroupTile (128) rows and a workgroup multiplies one token tile with a strip of weight
// rows.  Every wave owns R row tiles of 16 and converts its own A operands in registers; the
// tile's staged activation rows are shared through LDS.  Each MFMA covers one sub-block (the
// running scale needs the exact per-sub-block sums, gemm.hip): lane group q = lane/16 holds
// values 8q .. 8q+7 of the sub-block, i.e.
//   Q4_K sub-block j = 2g + h: qs bytes 32g + 8q .. +7, nibble h;
//   Q6_K sub-block j = 4H + grp: ql bytes 64H + 32(grp%2) + 8q .. +7 (nibble grp/2), qh bytes
//        32H + 8q .. +7 (bits 2grp), scale 8H + 2grp + q/2;
// and the activation fragment is the staged row's values 32j + 8q .. +7, in the
// same order of elements as the weights' (gemm_ops.hpp).
//
// What bounds it: up to ~32 tokens per expert the weights' bytes; above, the VALU (per 16 x 32
// weights ~12 operations to form the operand, and 4 per 16 x 16 outputs for the running
// scale, against one 16-cycle MFMA).  Both need work in flight from phases that do not
// coincide, so the kernel runs as several small workgroups per CU (Q4_K: three of 4 waves,
// 52 KB of LDS and at most 168 registers each; Q6_K: two of 8 waves, 128 registers): one workgroup's
// copies, barriers, first loads and final stores pass while the others multiply.  No
// instantiation spills: a reload in the loop waits for every copy issued before it (14 spilled
// registers in the 128-token tiles: 423 against 398 us, below).
// MoE prefill of 512 tokens (128 experts of 4096 -> 1536, top-8, Q6_K down): 830 -> 609 us; of 37
// tokens 363 -> 277; of 2048 (2048 -> 768, Q4_K down) 654 -> 388; before: one
// workgroup of 8 or 16 waves per CU, 64-token tiles.
#include <cstddef>

#include "gemm_ops.hpp"
#include "mnemo_common.hpp"
#include "mnemo_internal.hpp"

namespace mnemo {

struct GroupedArgs {
    const uint8_t *W;        // expert table base
    const _Float16 *A;       // staged q8 rows, f16 integers [rows][K]
    const float *a_rho;      // [rows][K/32] token scale ratios
    const uint16_t *a_ds;    // [rows][K/32] f16 ds
    const float *a_dlast;    // [rows][K/256] d8 unit at the end of each block
    float *out;
    int K, out_ld;           // K a multiple of 256
    int row_blocks;          // workgroups per token tile
    size_t expert_stride, w_off, w_off2;  // expert e's matrix at W + e*stride + w_off (up: w_off2)
    const int *counts;       // [n_experts] rows per expert
    const int *offsets;      // [n_experts] first expert-sorted row
    const int *perm;         // [rows] expert-sorted row -> token (SwiGLU gather)
    const int *tiles;        // [max_tiles] (expert << 16) | n_tile; tiles[-1] = count
};

// Shape of a launch by weight type: waves per workgroup, 16-row tiles per wave, bytes of a
// wave's weight area, and kLast, the 16-byte copies that end a block's weight copies.  The first
// stage of a block waits until at most kLast operations are outstanding.  All that relies on is
// that 16-byte LDS copies complete in order among themselves: everything the next stage reads was
// either copied in 16-byte units before the last kLast of them or stored by the waves before the
// barrier (gw_tile's copy_r).  4-byte copies and loads into registers may complete
// in any order (a wait that counted Q6_K's d among the younger operations let a stage read stale ratios
// about once in 10^5 workgroups); they are needed only after a wait for all.  SwiGLU (MODE 1): the
// wave's tiles are the gate and up rows of the same 16 features.
template <int TYPE>
struct Gw;
template <>
struct Gw<kTypeQ4K> {
    static constexpr int kWaves = 4, kR = 2, kArea = 2 * 16 * kQ4KBytes, kLast = 4, kPerEu = 3;
};
// Q6_K blocks (210 B, every other one at 2 mod 4) are copied from the dword that holds their
// first byte (sh = block offset & 2 bytes before it), 15 chunk slots of 16 B per row (240 B:
// the 16 rows' reads fall in distinct banks).  Chunks 0-12 are window bytes 16 ch ..; chunk 13
// is window bytes 196-211 when sh = 2 (block bytes 194-209) and a repeat of chunk 12 when
// sh = 0; chunk 14 repeats chunk 12.  So no copy reads past its block, and the block's bytes
// 0-207 are in the area; d (bytes 208-209) is loaded by the lanes themselves.  Slot
// t = 64 i + lane is written by copy i; slots past 239 repeat row 15's chunk 12.
constexpr int kSlots6 = 15;
template <>
struct Gw<kTypeQ6K> {
    static constexpr int kWaves = 8, kR = 1, kArea = 4096, kLast = 4, kPerEu = 4;
};

// Activations of one stage in LDS: 64 token rows x 128 K values, or 128 rows x 64 values
// (tiles of more than 64 tokens), double-buffered.
template <int NB>
constexpr int gw_stage_k() { return NB <= 4 ? 128 : 64; }

template <int TYPE>
struct GwLds {
    _Float16 b[2][64 * 128];
    float rho[2][256];  // the rows' scale ratios of the stage's 4 (2) sub-blocks
    uint32_t row[kGroupTile];  // the tile's token rows
    uint8_t w[Gw<TYPE>::kWaves][Gw<TYPE>::kArea];  // each wave's row tiles of one block
};

// element offset of staged chunk u (8 values) of row r; the chunk index is XOR-ed by the row
// so that the 16 rows of a fragment read cover the banks once
template <int SK>
__device__ __forceinline__ int gw_slot(int r, int u) {
    return SK == 128 ? r * 128 + ((u ^ (r & 15)) << 3) : r * 64 + ((u ^ ((r >> 1) & 7)) << 3);
}
template <int SK>
__device__ __forceinline__ int gw_unslot(int r, int pc) {  // the chunk stored at position pc
    return SK == 128 ? pc ^ (r & 15) : pc ^ ((r >> 1) & 7);
}

// the lane's values of row c of a Q4_K tile in the wave's LDS area
__device__ __forceinline__ Raw4 read4(const uint8_t *tile, int c, int q) {
    Raw4 r;
    const uint8_t *row = tile + c * kQ4KBytes;
    r.h = *(const uint4 *)row;
#pragma unroll
    for (int g = 0; g < 4; g++) r.a[g] = *(const uint2 *)(row + 16 + 32 * g + 8 * q);
    return r;
}
// the lane's raw values of row c's block from the wave's LDS area (sh: the block's
// misalignment, 0 or 2 bytes)
__device__ __forceinline__ Raw6 read6(const uint8_t *area, int c, int q, uint32_t sh) {
    Raw6 r;
    const uint32_t *a = (const uint32_t *)area + 4 * kSlots6 * c;
    auto rd8 = [&](int o) {  // block bytes o .. o + 7, o a multiple of 8
        const uint32_t w0 = a[o >> 2], w1 = a[(o >> 2) + 1], w2 = a[(o >> 2) + 2];
        return make_uint2(__builtin_amdgcn_alignbyte(w1, w0, sh), __builtin_amdgcn_alignbyte(w2, w1, sh));
    };
#pragma unroll
    for (int i = 0; i < 4; i++) r.ql[i] = rd8(64 * (i >> 1) + 32 * (i & 1) + 8 * q);
#pragma unroll
    for (int H = 0; H < 2; H++) r.qh[H] = rd8(128 + 32 * H + 8 * q);
    // of the 16 scale bytes the lane needs 8H + 2grp + q/2: bytes q/2, 2 + q/2, .. of each
    // dword, packed per half; window dword 52 (sh = 2 only) is the last of chunk 13
    uint32_t w[5];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = a[48 + i];
    w[4] = a[sh ? 55 : 52];
    uint4 sc;
    sc.x = __builtin_amdgcn_alignbyte(w[1], w[0], sh);
    sc.y = __builtin_amdgcn_alignbyte(w[2], w[1], sh);
    sc.z = __builtin_amdgcn_alignbyte(w[3], w[2], sh);
    sc.w = __builtin_amdgcn_alignbyte(w[4], w[3], sh);
    const uint32_t sel = 0x06040200u + 0x01010101u * (uint32_t)(q >> 1);
    r.sc[0] = __builtin_amdgcn_perm(sc.y, sc.x, sel);
    r.sc[1] = __builtin_amdgcn_perm(sc.w, sc.z, sel);
    return r;
}
// the lane's index, formed where it is used and not held in a register through the main loop
__device__ __forceinline__ uint32_t lane_here() {
    uint32_t l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}
// One token tile of NB 16-row columns against the workgroup's weight rows.
template <int TYPE, int MODE, int NB>
__device__ __forceinline__ void gw_tile(const GroupedArgs &g, const GwLds<TYPE> &L, uint32_t lds, int rb, int wave,
                                        int e, int j0, int n_rows, int row_base) {
    using T = Gw<TYPE>;
    constexpr int W = T::kWaves, R = T::kR;
    constexpr bool Q4 = TYPE == kTypeQ4K;
    constexpr int SK = gw_stage_k<NB>(), NS = 256 / SK, SJ = SK / 32;  // stages per block, sub-blocks per stage
    constexpr int CH = SK / 8;                                         // 16-byte chunks per staged row
    constexpr int P = (NB * 16 * CH + 64 * W - 1) / (64 * W);          // copies per wave and stage
    // formed per instantiation: what the switch's arms share is held, and spilled, through their loops
    const int lane = lane_here(), tid = 64 * wave + lane, q = lane >> 4, c = lane & 15;
    const int K = g.K, nkb = K / 256;
    const uint32_t wrow_bytes = (uint32_t)nkb * (Q4 ? kQ4KBytes : kQ6KBytes);
    const uint8_t *Wm = g.W + (size_t)e * g.expert_stride + g.w_off;
    // first weight row of the wave's tiles (SwiGLU: first feature)
    const int base = (rb * W + wave) * (MODE == 1 ? 16 : 16 * R);
    // the wave's tiles: 16 consecutive rows each
    const uint8_t *tp[R];
    tp[0] = Wm + (size_t)base * wrow_bytes;
    if constexpr (R == 2)
        tp[1] = MODE == 1 ? g.W + (size_t)e * g.expert_stride + g.w_off2 + (size_t)base * wrow_bytes
                          : tp[0] + (size_t)16 * wrow_bytes;

    // weight copies.  Q4_K: a tile's block is 144 chunks of 16 B, row ch/9, bytes 16(ch%9);
    // chunks 0-127 in two copies, 128-143 as 64 dwords in a third.
    uint32_t wo[Q4 ? 3 : 4];
    uint32_t roff = 0;
    if constexpr (Q4) {
#pragma unroll
        for (int i = 0; i < 2; i++) wo[i] = ((64 * i + lane) / 9) * wrow_bytes + 16 * ((64 * i + lane) % 9);
        wo[2] = ((128 + lane / 4) / 9) * wrow_bytes + 16 * ((128 + lane / 4) % 9) + 4 * (lane & 3);
#pragma unroll
        for (int i = 0; i < 3; i++) asm volatile("" : "+v"(wo[i]));
    } else {
        // offsets from the tile's first byte, which is 4-byte aligned (16 rows are a multiple of 4
        // bytes, the table's matrices are checked); bit 0 set for chunk 13, which moves 4 bytes on
        // when sh = 2
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = 64 * i + lane, row = t < 16 * kSlots6 ? t / kSlots6 : 15;
            const int ch = t < 16 * kSlots6 ? t % kSlots6 : 12;
            wo[i] = row * wrow_bytes + (ch <= 12 ? 16u * (uint32_t)ch : ch == 13 ? 192u + 1u : 192u);
        }
        roff = c * wrow_bytes;
    }
    const uint8_t *area = L.w[wave];
    // LDS addresses of the copies' targets (scalars)
    const uint32_t lds_w = lds + (uint32_t)offsetof(GwLds<TYPE>, w) + wave * T::kArea;
    const uint32_t lds_b = lds + wave * 1024, lds_r = lds + (uint32_t)offsetof(GwLds<TYPE>, rho);
    auto copy_w = [&](int k) {
        if constexpr (Q4) {
#pragma unroll
            for (int a = 0; a < R; a++) {
                lds_copy4(tp[a] + (size_t)k * kQ4KBytes, wo[2], lds_w + 2304 * a + 2048);
            }
#pragma unroll
            for (int a = 0; a < R; a++) {
                const uint8_t *s = tp[a] + (size_t)k * kQ4KBytes;
                lds_copy16(s, wo[0], lds_w + 2304 * a);
                lds_copy16(s, wo[1], lds_w + 2304 * a + 1024);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t a = wo[i] + (uint32_t)(kQ6KBytes * k);
                lds_copy16(tp[0], (a & ~3u) + ((a & 1u) ? (a & 2u) << 1 : 0u), lds_w + 1024 * i);
            }
        }
    };
    // activation copies: LDS chunk slot s = 64 W i + tid holds chunk gw_unslot(s % CH) of row
    // s / CH; rows past the tile's last repeat it
    auto stage_row = [&](int r) {
        const int j = min(j0 + r, n_rows - 1);
        return MODE == 1 ? g.perm[row_base + j] : row_base + j;
    };
    // offsets from the tile's first row (gathered rows: from the first of all; 32 bits of 16-byte units
    // reach 2^35 values of x, whose fp32 source, staged rows, down rows and output take 480 GB)
    const int row0 = MODE == 1 ? 0 : row_base + j0;
    const _Float16 *A0 = g.A + (size_t)row0 * K;
    const float *rho0 = g.a_rho + (size_t)row0 * (K / 32);
    uint32_t ao[P];  // in 16-byte units
#pragma unroll
    for (int i = 0; i < P; i++) {
        const int s = 64 * W * i + tid, r = s / CH;
        ao[i] = (uint32_t)(stage_row(r) - row0) * (uint32_t)(K / 8) + gw_unslot<SK>(r, s % CH);
        asm volatile("" : "+v"(ao[i]));
    }
    // The stage's ratios, [row][sub-block].  128-value stages: a row's four are 16 bytes, one copy of
    // wave 0 (lane = row).  64-value stages: float tid of the array, a 4-byte copy, which a
    // block's second stage may not use (the first stage's counted wait does not cover it): its ratios
    // come through a register, loaded during the last stage before the block, which ends in a wait
    // for all.  (16-byte copies of two stages' ratios would need 2 KB more LDS, one workgroup per CU
    // less; the register in 128-value stages too costs 1 % at 37 tokens.)
    constexpr bool kReg = SK == 64;
    uint32_t ro = kReg ? (uint32_t)(stage_row((tid & 255) / SJ) - row0) * (uint32_t)(K / 32) + tid % SJ
                       : (uint32_t)(stage_row(lane) - row0) * (uint32_t)(K / 32);
    asm volatile("" : "+v"(ro));
    auto copy_r = [&](int t, int buf) {
        const uint32_t dst = buf * (uint32_t)sizeof L.rho[0];
        if constexpr (!kReg) {
            if (wave == 0) lds_copy16(rho0 + (size_t)t * SJ, 4 * ro, lds_r + dst);
        } else if (W == 4 || wave < 4) {
            lds_copy4(rho0 + (size_t)t * SJ + ro, lds_r + dst + wave * 256);
        }
    };
    float rn = 0.0f;
    auto load_r = [&](int k) {
        if constexpr (kReg) rn = rho0[((size_t)k * NS + 1) * SJ + ro];
    };
    auto pin_r = [&] {
        if constexpr (kReg) asm volatile("" : "+v"(rn));
    };
    auto copy_b = [&](int t, int buf) {  // stage t (t * SK values into the rows)
#pragma unroll
        for (int i = 0; i < P; i++)
            if (64 * W * (i + 1) <= NB * 16 * CH || 64 * W * i + 64 * wave < NB * 16 * CH)  // wave-uniform
                lds_copy16(A0 + (size_t)t * SK + 8 * (size_t)ao[i], lds_b + buf * (uint32_t)sizeof L.b[0] + 1024 * W * i);
    };

    // the lane's LDS addresses: its fragment chunk of each sub-block of a stage, its column's ratios
    uint32_t fra[SJ], rra = lds + (uint32_t)offsetof(GwLds<TYPE>, rho) + 4 * SJ * c;
#pragma unroll
    for (int jj = 0; jj < SJ; jj++) {
        fra[jj] = lds + 2 * gw_slot<SK>(c, 4 * jj + q);
        asm volatile("" : "+v"(fra[jj]));
    }
    asm volatile("" : "+v"(rra));

    constexpr f4 kZero = {0.f, 0.f, 0.f, 0.f};
    constexpr bool kTot = Q4 && MODE == 2 && NB <= 4;
    f4 acc[R][NB];
    f4 tot[kTot ? R : 1][kTot ? NB : 1];  // the sums of the blocks before
    float deff[R];  // running d of the lane's A row c of each tile (kTot: the block's d)
#pragma unroll
    for (int a = 0; a < R; a++) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            acc[a][b] = kZero;
            if constexpr (kTot) tot[a][b] = kZero;
        }
        deff[a] = 1.0f;
    }
    if (tid < 16 * NB) lds_put<uint32_t>(lds + (uint32_t)offsetof(GwLds<TYPE>, row), 4 * tid, (uint32_t)stage_row(tid));
    copy_r(0, 0);
    copy_b(0, 0);
    load_r(0);
    copy_w(0);
    uint32_t dn = 0;  // Q6_K: f16 d of row c's next block
    auto load_d6 = [&](int k) {
        uint16_t dd;
        __builtin_memcpy(&dd, tp[0] + roff + (size_t)k * kQ6KBytes + 208, 2);
        dn = dd;
    };
    if constexpr (!Q4) load_d6(0);

    // Q4_K's min term, sum_s -(dmin*m_s)_i * ds_js, is one product over the sub-block index: two
    // MFMAs (hi + lo operand) per window of 32 sub-blocks (4 blocks), lane group q holding the window's
    // block 4 w + q (K index 8 q + s of the MFMA = sub-block s of that block).
    // Gate/up: the lanes keep the packed mins and dmin as they read the headers; at the window's
    // end the term is formed on zero and the accumulators join it by one fma, which makes them absolute
    // (4.9e-7 relative L2 against 64 bits, 5.1e-7 with the term added to the absolute accumulators;
    // SwiGLU rows of K = 4096).
    // Down: the products are larger than their sum with the term where activations are large, and the
    // roundings scale with the sum so far.  Up to 64 tokens the registers hold a total beside the
    // block's sum, so that only one rounding per block is at the total's magnitude (K = 1024 7.5e-8;
    // 1.6e-7 in one sum.  Gate/up would gain as much and take 1.4 % longer at 37 and 512 tokens).  Wider tiles
    // start their accumulators as the whole term, which keeps the sum near the result all the way:
    // K = 768 1.07e-7, 1.39e-7 with the term at the windows' ends; K = 512 9.0e-8 and 9.9e-8.
    // (Activations several times larger, near where ds leaves the f16 range, favour the other order.)
    // It reads the headers' lines once more: at K = 768, M = 2048 130 us instead of 123 for
    // 16,384 rows; narrow tiles, which the weights' bytes bound, would take 10 % longer.
    constexpr bool kMins = Q4 && (MODE == 1 || kTot);
    uint2 mins[kMins ? R : 1];
    if constexpr (Q4 && !kMins) {
        for (int w = 0; 4 * w < nkb; w++) {
            const bool valid = 4 * w + q < nkb;  // lane groups past the row's end add nothing
            const int sb = min(4 * w + q, nkb - 1);
            uint4 hd[R], bd[NB];
#pragma unroll
            for (int a = 0; a < R; a++) hd[a] = ld16(tp[a] + c * wrow_bytes + (size_t)sb * kQ4KBytes);
#pragma unroll
            for (int b = 0; b < NB; b++)
                bd[b] = ld16((const uint8_t *)(g.a_ds + (size_t)stage_row(16 * b + c) * (K / 32) + 8 * sb));
#pragma unroll
            for (int a = 0; a < R; a++) {
                h8 hi, lo;
                q4k_min_operand_m(q4k_mins(hd[a]), valid ? hd[a].x >> 16 : 0u, hi, lo);
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const h8 bv = valid ? __builtin_bit_cast(h8, bd[b]) : h8{};
                    acc[a][b] = mfma(lo, bv, mfma(hi, bv, acc[a][b]));
                }
            }
        }
    }
    // every wave's copies of the first stage and block have landed before any wave passes
    wait_vm<0>();
    pin_r();
    lds_barrier();

    // LDS address of the token row of the lane's column
    auto row_addr = [&] { return lds + (uint32_t)offsetof(GwLds<TYPE>, row) + 4 * (lane_here() & 15); };
    for (int k = 0; k < nkb; k++) {
        const int kn = min(k + 1, nkb - 1);  // past the end the last block is copied again
        // block k's weights into registers; the area is refilled once they are there
        Raw4 w4[Q4 ? R : 1];
        Raw6 w6;
        float d[R];
        if constexpr (Q4) {
#pragma unroll
            for (int a = 0; a < R; a++) w4[a] = read4(area + 2304 * a, c, q);
        } else {
            d[0] = h2f(dn);
            w6 = read6(area, c, q, (roff + (uint32_t)(kQ6KBytes * k)) & 2u);
            asm volatile("" : "+v"(d[0]));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int buf = s & 1;
            // the next stage's activations go first, then (first stage) the next block's
            // weights: the first stage's barrier leaves the weights in flight
            const int tn = s + 1 < NS ? k * NS + s + 1 : kn * NS;
            if (!kReg || s) copy_r(tn, buf ^ 1);
            else if (W == 4 || wave < 4) lds_put<float>(lds_r + 4 * (uint32_t)tid, sizeof L.rho[0], rn);
            copy_b(tn, buf ^ 1);
            if (s == NS - 1) load_r(kn);
            float dtk[kTot ? NB : 1];  // the tokens' units at the block's end
            if constexpr (kTot) {
                if (s == NS - 1) {
                    const uint32_t rowa = row_addr();
#pragma unroll
                    for (int b = 0; b < NB; b++) dtk[b] = g.a_dlast[(size_t)lds_get<uint32_t>(rowa, 64 * b) * nkb + k];
                }
            }
            if (s == 0) {
                copy_w(kn);
                if constexpr (!Q4) load_d6(kn);
                if constexpr (Q4) {
#pragma unroll
                    for (int a = 0; a < R; a++) {
                        d[a] = h2f(w4[a].h.x & 0xFFFFu);
                        if constexpr (kMins) {
                            const bool cap = (k & 3) == q;
                            const uint2 mn = q4k_min_pack(w4[a].h);
                            mins[a].x = cap ? mn.x : mins[a].x;
                            mins[a].y = cap ? mn.y : mins[a].y;
                        }
                        if (d[a] == 0.0f) w4[a].h.y = w4[a].h.w = 0u;  // scales 0: the block's products are zero
                    }
                } else if (d[0] == 0.0f) {
                    w6.sc[0] = w6.sc[1] = 0u;
                }
                // the running row scales: lane c owns A row c of each tile; the lane's outputs are
                // rows 4q + x, whose ratios come from lanes 4q + x
#pragma unroll
                for (int a = 0; a < R; a++) {
                    if constexpr (kTot) {
                        deff[a] = d[a];
                        continue;
                    }
                    const float nd = d[a] == 0.0f ? deff[a] : d[a];
                    const float sg = ratio(deff[a], nd);
                    deff[a] = nd;
#pragma unroll
                    for (int x = 0; x < 4; x++) {
                        const float se = __shfl(sg, 4 * q + x);
#pragma unroll
                        for (int b = 0; b < NB; b++) acc[a][b][x] *= se;
                    }
                }
            }
            Scales4 s4[Q4 ? R : 1];
            Scales6 s6;
#pragma unroll
            for (int jj = 0; jj < SJ; jj++) {
                const int j = SJ * s + jj;  // sub-block of the block
                h8 a1[R], a2[Q4 ? 1 : R];
#pragma unroll
                for (int a = 0; a < R; a++) {
                    if constexpr (Q4) {
                        if ((jj & 1) == 0) s4[a] = scale_pair4(w4[a].h, j >> 1);
                        a1[a] = operand4(w4[a], s4[a], j >> 1, jj & 1);
                    } else {
                        if ((jj & 1) == 0) s6 = scale_pair6(w6.sc[j >> 2], j >> 1);
                        operand6(w6, s6, j, a1[a], a2[a]);
                    }
                }
                constexpr int NG = NB > 4 ? NB / 2 : 1, NC = NB / NG;  // columns in groups of at most 4
#pragma unroll
                for (int gr = 0; gr < NG; gr++) {
                    h8 bf[NC];
                    float rr[NC];  // the token columns' ratios
#pragma unroll
                    for (int b = 0; b < NC; b++)
                        rr[b] = lds_get<float>(rra, (buf * 256 + 16 * (NC * gr + b) * SJ + jj) * 4);
#pragma unroll
                    for (int b = 0; b < NC; b++)
                        bf[b] = lds_get<h8>(fra[jj], buf * (uint32_t)sizeof L.b[0] + 16 * (NC * gr + b) * SK * 2);
#pragma unroll
                    for (int a = 0; a < R; a++)
#pragma unroll
                        for (int b = 0; b < NC; b++) {
                            f4 &ac = acc[a][NC * gr + b];
                            if (kTot && j == 0) ac = kZero;
                            else ac *= rr[b];
                            ac = mfma(a1[a], bf[b], ac);
                            if constexpr (!Q4) ac = mfma(a2[a], bf[b], ac);
                        }
                    if constexpr (NB >= 6) __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (s == NS - 1 && ((k & 3) == 3 || k == nkb - 1)) {  // uniform: the window's end
                // the window's last blocks: lane groups past the row's end add nothing
                const bool valid = (k & ~3) + q < nkb;
                const int sb = min((k & ~3) + q, nkb - 1);
                const uint32_t rowa = row_addr();
                // a group's operands are loaded before the first is used: the lane's fragments are dead
                // here, and their registers take them
                constexpr int NC = NB > 4 && kMins ? NB / 2 : NB;  // columns at a time
#pragma unroll
                for (int b0 = 0; b0 < NB; b0 += NC) {
                    float dt[NC];
                    h8 bd[kMins ? NC : 1];
#pragma unroll
                    for (int b = 0; b < NC; b++) {
                        const size_t tok = lds_get<uint32_t>(rowa, 64 * (b0 + b));
                        if constexpr (!kTot) dt[b] = (g.a_dlast + k)[(uint32_t)tok * (uint32_t)nkb];
                        if constexpr (kMins)
                            bd[b] = __builtin_bit_cast(h8, ld16((const uint8_t *)(g.a_ds + tok * (K / 32) + 8 * sb)));
                    }
#pragma unroll
                    for (int a = 0; a < R; a++) {
                        float dr[4];
                        if constexpr (!kTot) {
#pragma unroll
                            for (int x = 0; x < 4; x++) dr[x] = __shfl(deff[a], 4 * q + x);
                        }
                        h8 hi, lo;
                        if constexpr (kMins) q4k_min_operand(valid ? mins[a] : make_uint2(0u, 0u), hi, lo);
#pragma unroll
                        for (int b = 0; b < NC; b++) {
                            f4 &ac = acc[a][b0 + b];
                            f4 to = kZero;
                            if constexpr (kTot) to = tot[a][b0 + b];
                            if constexpr (kMins) {
                                const h8 bv = valid ? bd[b] : h8{};
                                to = mfma(lo, bv, mfma(hi, bv, to));
                            }
                            if constexpr (kTot) {
                                tot[a][b0 + b] = to;
                            } else {
#pragma unroll
                                for (int x = 0; x < 4; x++) ac[x] = __builtin_fmaf(ac[x], dr[x] * dt[b], to[x]);
                            }
                        }
                    }
                    if constexpr (NC < NB) __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int a = 0; a < R; a++)
                    if constexpr (!kTot) deff[a] = 1.0f;
            }
            if constexpr (kTot) {
                if (s == NS - 1)  // the block's sum, absolute, joins the total
#pragma unroll
                    for (int a = 0; a < R; a++) {
                        float dr[4];
#pragma unroll
                        for (int x = 0; x < 4; x++) dr[x] = __shfl(deff[a], 4 * q + x);
#pragma unroll
                        for (int b = 0; b < NB; b++)
#pragma unroll
                            for (int x = 0; x < 4; x++)
                                tot[a][b][x] = __builtin_fmaf(acc[a][b][x], dr[x] * dtk[b], tot[a][b][x]);
                    }
            }
            // the next stage's activations have landed for every wave (and, from the second
            // stage on, the next block's weights)
            if (s == 0) wait_vm<T::kLast>();
            else wait_vm<0>();
            if (s == NS - 1) pin_r();
            lds_barrier();
        }
    }

    if constexpr (kTot) {
#pragma unroll
        for (int a = 0; a < R; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = tot[a][b];
    }
    // D layout: lane holds weight rows 4q + x of each 16-row tile, token column c
    const int le = lane_here();
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int j = j0 + 16 * b + (le & 15);
        if (j >= n_rows) continue;
        float *orow = g.out + (size_t)(row_base + j) * g.out_ld + base + 4 * (le >> 4);
        if constexpr (MODE == 1) {
            f4 v;
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const float gt = acc[0][b][x], up = acc[R - 1][b][x];
                v[x] = gt / (1.0f + expf(-gt)) * up;
            }
            *(f4 *)orow = v;
        } else {
#pragma unroll
            for (int a = 0; a < R; a++) *(f4 *)(orow + 16 * a) = acc[a][b];
        }
    }
}

// MODE 1: SwiGLU (gate and up rows of the same features, activation rows gathered through
// perm[], out[q*ld + f] = silu(gate) * up); MODE 2: the expert-sorted rows themselves.
template <int TYPE, int MODE>
__global__ void __launch_bounds__(64 * Gw<TYPE>::kWaves)
    __attribute__((amdgpu_waves_per_eu(Gw<TYPE>::kPerEu, Gw<TYPE>::kPerEu))) gemm_grouped_kernel(GroupedArgs g) {
    __shared__ __align__(16) GwLds<TYPE> L;
    const uint32_t lds = lds_addr(&L);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroups go to the 8 XCDs in turn.  The row blocks of one tile share its activation rows, so
    // they run on one XCD (tiles are dealt to the XCDs in turn, heaviest first) and read them from
    // its L2; the last n % 8 tiles are spread over all XCDs.  With every tile spread, the rows came
    // from beyond the L2 for each XCD (512 tokens, gate/up: 1.44 GB fetched for 0.91 GB of weights).
    const int n = g.tiles[-1], nb = g.row_blocks;
    int id = blockIdx.x, tile, rb;
    const int even = (n & ~7) * nb;
    if (id < even) {
        const int l = id >> 3;
        tile = (l / nb) * 8 + (id & 7);
        rb = l % nb;
    } else {
        id -= even;
        tile = (n & ~7) + id / nb;
        rb = id % nb;
    }
    if (tile >= n) return;
    const int tl = g.tiles[tile];
    const int e = tl >> 16, nt = tl & 0xFFFF;
    const int n_rows = g.counts[e], row_base = g.offsets[e], j0 = nt * kGroupTile;
    const int nvalid = min(kGroupTile, n_rows - j0);
#define MNEMO_GW(NB_) gw_tile<TYPE, MODE, NB_>(g, L, lds, rb, wave, e, j0, n_rows, row_base)
    // one instantiation per count of 16-row column tiles, so every MFMA is unconditional (5
    // and 7 run padded to 6 and 8)
    switch ((nvalid + 15) >> 4) {
    case 1: MNEMO_GW(1); break;
    case 2: MNEMO_GW(2); break;
    case 3: MNEMO_GW(3); break;
    case 4: MNEMO_GW(4); break;
    case 5:
    case 6: MNEMO_GW(6); break;
    default: MNEMO_GW(8); break;
    }
#undef MNEMO_GW
}

// Grouped launches used by the MoE prefill path (moe.hip): tiles[] and the routing arrays
// live in device memory, the grid covers max_tiles tile-list entries.  M and K are multiples of
// 256, so every wave's rows exist.
int launch_gemm_grouped(int type, int swiglu, const void *experts, size_t expert_stride, size_t w_off,
                        size_t w_off2, StagedAct act, const int *counts, const int *offsets, const int *perm,
                        const int *tiles, int max_tiles, float *out, int out_ld, int M, int K, hipStream_t stream) {
    GroupedArgs g{};
    g.W = (const uint8_t *)experts;
    g.A = act.q8;
    g.a_rho = act.rho;
    g.a_ds = act.ds;
    g.a_dlast = act.dlast;
    g.out = out;
    g.K = K;
    g.out_ld = out_ld;
    g.expert_stride = expert_stride;
    g.w_off = w_off;
    g.w_off2 = w_off2;
    g.counts = counts;
    g.offsets = offsets;
    g.perm = perm;
    g.tiles = tiles;
    if (swiglu && type != kTypeQ4K)
        return set_error(kErrUnsupportedType, "grouped gate/up GEMM: Q4_K only (type %d)", type);
#define MNEMO_GROUPED(T_, M_)                                                                              \
    do {                                                                                                   \
        const int rows = (M_ == 1 ? 16 : 16 * Gw<T_>::kR) * Gw<T_>::kWaves;                                \
        g.row_blocks = M / rows;                                                                           \
        hipLaunchKernelGGL((gemm_grouped_kernel<T_, M_>), dim3(g.row_blocks * max_tiles),                  \
                           dim3(64 * Gw<T_>::kWaves), 0, stream, g);                                       \
    } while (0)
    if (swiglu) MNEMO_GROUPED(kTypeQ4K, 1);
    else if (type == kTypeQ4K) MNEMO_GROUPED(kTypeQ4K, 2);
    else MNEMO_GROUPED(kTypeQ6K, 2);
#undef MNEMO_GROUPED
    return check_launch("gemm_grouped");
}

}  // namespace mnemo
