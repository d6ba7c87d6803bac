// sample.hip -- next-token selection from the lm_head logits (MnemoCUDA kernels.cu:2020-2174,
// wrapper kernels.cu:2208-2215), one workgroup of 1024 threads.
//
// Semantics kept from the reference (they decide which token is drawn for a given seed):
//  * temperature <= 0: argmax (this build breaks exact ties toward the lower index).
//  * temperature > 0: p_i = exp((z_i - max z) / T); the nucleus is drawn from 2048
//    candidates: for each residue class c = i mod 256, the 8 largest p of the class (equal
//    p: the lower index first, which is what the reference's in-order scan that only
//    replaces its minimum by a strictly larger value keeps).  Candidates are taken in
//    decreasing p until their running sum reaches top_p * total (total = sum of all p),
//    the kept ones are renormalised and one is drawn with u from xoroshiro128+ (s0 =
//    rng_state, s1 = rng_state ^ 0xDEADBEEFCAFEBABE, three warm-up steps, u = (s0 + s1) >> 11
//    as a float times 2^-53).
// What differs: the reference sums in one order on 256 threads and runs a selection sort and
// the running sums on one thread (up to 2048 x nucleus comparisons, then three sequential
// passes).  Here four threads share a class, the candidates are sorted by a bitonic network
// and the running sums are a parallel scan: fp32 sums in another order, which can change
// the drawn token only when the draw or top_p * total lies within rounding (~1e-6 of the
// mass) of a cumulative boundary; equal p are ordered by token id.
#include "mnemo_common.hpp"
#include "mnemo_internal.hpp"

namespace mnemo {

constexpr int kSampleThreads = 1024;
constexpr int kClasses = 256, kPerClass = 8, kSub = kSampleThreads / kClasses;  // 4 threads per class
constexpr int kCands = kClasses * kPerClass;                                    // 2048

__device__ __forceinline__ uint64_t xoro_next(uint64_t &s0, uint64_t &s1) {
    const uint64_t t = s0 ^ (s0 << 23);
    s0 = s1;
    s1 = t ^ s1 ^ (t >> 17) ^ (s1 >> 26);
    return s0 + s1;
}

__device__ __forceinline__ bool before(float pa, int ia, float pb, int ib) {
    return pa > pb || (pa == pb && ia < ib);
}

// ------------------------------------------------------------------ top-p selection
// The 2048 candidates are sorted by (p desc, id asc) on 1024 threads, 2 per thread.  A
// candidate's order is that of one 64-bit key, {p bits, ~id} (p >= 0 orders like its bits); an
// empty slot (p < 0, NaN) is key 0 and sorts last.  Bitonic network: stride 1 inside a thread,
// 2 .. 64 between the lanes of a wave (DPP, lane swaps at 32 and 64), 128 .. 1024 through LDS.
// Then, on 256 threads of 8 sorted positions, the running sums (inclusive, in sorted order:
// sequential within a thread, a scan over the threads), the nucleus and the draw.
constexpr int kSelThreads = kCands / 8;  // 256
constexpr int kSelWaves = kSelThreads / 64;

__device__ __forceinline__ uint64_t cand_key(float p, int id) {
    if (!(p >= 0.0f)) return 0ull;
    return ((uint64_t)__float_as_uint(fabsf(p)) << 32) | (uint32_t)~(uint32_t)id;
}

// keep the better (larger key) of a and b in a when `better_here`, the other one otherwise
__device__ __forceinline__ uint64_t keep(uint64_t a, uint64_t b, bool better_here) {
    return (a > b) == better_here ? a : b;  // one compare, one select (keys are distinct or equal)
}

// v of lane ^ M: DPP within rows of 16 lanes (quad permutes; row rotations, where lane i
// reads lane (i - n) mod 16), row and half swaps of the vector unit beyond
template <int M>
__device__ __forceinline__ uint32_t xor_lane(uint32_t v) {
    if constexpr (M == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kDppXor1, 0xF, 0xF, false);
    else if constexpr (M == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kDppXor2, 0xF, 0xF, false);
    else if constexpr (M == 4) {
        const uint32_t dn = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, false);  // i - 4
        const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x12C, 0xF, 0xF, false);  // i + 4
        return (lane_id() & 4) ? dn : up;
    } else if constexpr (M == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, false);
    else if constexpr (M == 16) {  // rows 1, 3 of the first operand trade places with rows 0, 2 of the second
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (lane_id() & 16) ? r[0] : r[1];
    } else {
        static_assert(M == 32, "strides within a wave");
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (lane_id() & 32) ? r[0] : r[1];
    }
}

// a bitonic pass between lanes t and t ^ M (strides 2M)
template <int M>
__device__ __forceinline__ void lane_pass(uint64_t (&k)[2], bool better_here) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const uint64_t o = ((uint64_t)xor_lane<M>((uint32_t)(k[r] >> 32)) << 32) | xor_lane<M>((uint32_t)k[r]);
        k[r] = keep(k[r], o, better_here);
    }
}

struct SelLds {
    alignas(16) uint64_t xch[2][kCands];
    float wsum[kSelWaves];
    int wmin[2][kSelWaves];
    float cs_last;
};

// Every thread of the workgroup calls this (it holds barriers) with two candidates in any
// order.  total = the sum of all p.
// One workgroup, so the sort's instructions bound it: 66 passes of the network over 2048 keys.
// On 1024 threads a SIMD has four waves to issue from (with 8 keys on each of 256 threads it
// had one, which issues at half the rate and waits out every exchange): the workspace form's
// second launch 23.4 us, from 26.5 (vocabulary 151,936); both launches 35.3 -> 32.1, the
// one-launch form 136.8 -> 126.7.
__device__ void select_sorted(uint64_t (&kk2)[2], float total, float top_p, unsigned long long seed, SelLds &L,
                              int *__restrict__ out) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    // bitonic sort, best first: at level kk the pair (e, e ^ j), e < e ^ j, puts the better
    // key at e when (e & kk) == 0; thread t holds positions 2t, 2t + 1
    int buf = 0;
    for (int kk = 2; kk <= kCands; kk <<= 1) {
        const bool up = ((2 * t) & kk) == 0;
        for (int m = kk >> 2; m >= 1; m >>= 1) {  // partner thread t ^ m (uniform)
            const bool b = up == ((t & m) == 0);
            switch (m) {
            case 1: lane_pass<1>(kk2, b); break;
            case 2: lane_pass<2>(kk2, b); break;
            case 4: lane_pass<4>(kk2, b); break;
            case 8: lane_pass<8>(kk2, b); break;
            case 16: lane_pass<16>(kk2, b); break;
            case 32: lane_pass<32>(kk2, b); break;
            default:  // between waves; the buffers alternate, so one barrier orders both their uses
                *(ulonglong2 *)&L.xch[buf][2 * t] = make_ulonglong2(kk2[0], kk2[1]);
                __syncthreads();
                const ulonglong2 o = *(const ulonglong2 *)&L.xch[buf][2 * (t ^ m)];
                kk2[0] = keep(kk2[0], o.x, b);
                kk2[1] = keep(kk2[1], o.y, b);
                buf ^= 1;
            }
        }
        const uint64_t x = kk2[0], y = kk2[1];
        kk2[0] = keep(x, y, up);
        kk2[1] = keep(x, y, !up);
    }
    *(ulonglong2 *)&L.xch[buf][2 * t] = make_ulonglong2(kk2[0], kk2[1]);
    __syncthreads();
    // from here on 256 threads hold 8 sorted positions each, 8t .. 8t + 7
    const bool act = t < kSelThreads;
    uint64_t k[8];
#pragma unroll
    for (int r = 0; r < 8; r += 2) {
        const ulonglong2 v = act ? *(const ulonglong2 *)&L.xch[buf][8 * t + r] : make_ulonglong2(0, 0);
        k[r] = v.x;
        k[r + 1] = v.y;
    }
    // inclusive running sums of the positive p in sorted order
    float p[8], c[8];
#pragma unroll
    for (int r = 0; r < 8; r++) p[r] = act ? __uint_as_float((uint32_t)(k[r] >> 32)) : 0.0f;
    c[0] = p[0];
#pragma unroll
    for (int r = 1; r < 8; r++) c[r] = c[r - 1] + p[r];
    float s = c[7];  // inclusive scan of the thread totals over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float v = __shfl_up(s, o);
        if (lane >= o) s += v;
    }
    float excl = __shfl_up(s, 1);
    if (lane == 0) excl = 0.0f;
    if (act && lane == 63) L.wsum[w] = s;
    __syncthreads();
    float off = 0.0f;
    for (int i = 0; i < w && i < kSelWaves; i++) off += L.wsum[i];
    const float pre = off + excl;
#pragma unroll
    for (int r = 0; r < 8; r++) c[r] = pre + c[r];
    // nucleus size n: 1 + the first position whose running sum reaches top_p * total, the
    // position of the first candidate with p <= 0, or all of them
    const float mass = top_p * total;
    int nc = kCands;
#pragma unroll
    for (int r = 7; r >= 0; r--)
        if (act && (p[r] <= 0.0f || c[r] >= mass)) nc = p[r] <= 0.0f ? 8 * t + r : 8 * t + r + 1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) nc = min(nc, __shfl_xor(nc, o));
    if (act && lane == 0) L.wmin[0][w] = nc;
    __syncthreads();
    int n = kCands;
    for (int i = 0; i < kSelWaves; i++) n = min(n, L.wmin[0][i]);
    if (act && n > 0 && t == (n - 1) >> 3) {
        float v = c[0];
#pragma unroll
        for (int r = 1; r < 8; r++) v = r == ((n - 1) & 7) ? c[r] : v;
        L.cs_last = v;
    }
    __syncthreads();
    uint64_t s0 = seed, s1 = seed ^ 0xDEADBEEFCAFEBABEull;
    for (int i = 0; i < 3; i++) xoro_next(s0, s1);
    const float u = (float)(xoro_next(s0, s1) >> 11) * (1.0f / 9007199254740992.0f);
    const float target = u * (n > 0 ? L.cs_last : 0.0f);
    // the draw: the first position below n whose running sum reaches the target
    int pk = 0x7FFFFFFF;
#pragma unroll
    for (int r = 7; r >= 0; r--)
        if (act && 8 * t + r < n && c[r] >= target) pk = 8 * t + r;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pk = min(pk, __shfl_xor(pk, o));
    if (act && lane == 0) L.wmin[1][w] = pk;
    __syncthreads();
    int pick = 0x7FFFFFFF;
    for (int i = 0; i < kSelWaves; i++) pick = min(pick, L.wmin[1][i]);
    if (pick == 0x7FFFFFFF) pick = 0;
    if (act && t == pick >> 3) {
        uint64_t kv = k[0];
#pragma unroll
        for (int r = 1; r < 8; r++) kv = r == (pick & 7) ? k[r] : kv;
        const int id = kv ? (int)~(uint32_t)kv : -1;
        *out = (id < 0 || id == 0x7FFFFFFF) ? 0 : id;
    }
}

__global__ void __launch_bounds__(kSampleThreads) sample_token_kernel(const float *__restrict__ logits, int V,
                                                                      float temperature, float top_p,
                                                                      unsigned long long seed, int *__restrict__ out) {
    __shared__ float red_f[kSampleThreads];
    __shared__ int red_i[kSampleThreads];
    __shared__ float cp[kCands];
    __shared__ int ci[kCands];
    __shared__ float mp[kSampleThreads * kPerClass];  // every thread's list before the class merge
    __shared__ int mi[kSampleThreads * kPerClass];
    const int tid = threadIdx.x;

    float m = -1e30f;
    for (int i0 = tid; i0 < V; i0 += kSampleThreads * 8) {
        float zb[8];
#pragma unroll
        for (int u = 0; u < 8; u++) zb[u] = logits[min(i0 + u * kSampleThreads, V - 1)];  // clamped: a repeat
#pragma unroll
        for (int u = 0; u < 8; u++) m = fmaxf(m, zb[u]);
    }
    red_f[tid] = m;
    __syncthreads();
    for (int s = kSampleThreads / 2; s > 0; s >>= 1) {
        if (tid < s) red_f[tid] = fmaxf(red_f[tid], red_f[tid + s]);
        __syncthreads();
    }
    const float gmax = red_f[0];
    __syncthreads();

    if (temperature <= 0.0f) {  // argmax, ties to the lower index
        float bv = -1e30f;
        int bi = 0x7FFFFFFF;
        for (int i = tid; i < V; i += kSampleThreads) {
            const float v = logits[i];
            if (v > bv) { bv = v; bi = i; }
        }
        red_f[tid] = bv;
        red_i[tid] = bi;
        __syncthreads();
        for (int s = kSampleThreads / 2; s > 0; s >>= 1) {
            if (tid < s && before(red_f[tid + s], red_i[tid + s], red_f[tid], red_i[tid])) {
                red_f[tid] = red_f[tid + s];
                red_i[tid] = red_i[tid + s];
            }
            __syncthreads();
        }
        if (tid == 0) *out = red_i[0] == 0x7FFFFFFF ? 0 : red_i[0];
        return;
    }

    // thread (sub = tid / 256, class c = tid % 256) scans indices c + 256 * (sub + 4 t) in
    // increasing order (adjacent lanes read adjacent logits), keeping its 8 largest p (ties:
    // the earliest) and its sum
    const int c = tid % kClasses, sub = tid / kClasses;
    float sum = 0.0f;
    float hv[kPerClass];
    int hi[kPerClass];
#pragma unroll
    for (int k = 0; k < kPerClass; k++) {
        hv[k] = -1.0f;
        hi[k] = -1;
    }
    float hmin = -1.0f;  // the current minimum of hv
    // logits are loaded kBatch at a time (independent loads in flight), then scanned in order
    constexpr int kStride = kClasses * kSub, kBatch = 16;
    for (int i0 = c + kClasses * sub; i0 < V; i0 += kStride * kBatch) {
        float zb[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) zb[u] = logits[min(i0 + u * kStride, V - 1)];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
        const int i = i0 + u * kStride;
        if (i >= V) break;
        const float p = expf((zb[u] - gmax) / temperature);
        sum += p;
        if (p > hmin) {
            int at = 0;  // first position holding the minimum
#pragma unroll
            for (int k = kPerClass - 1; k >= 0; k--) at = hv[k] == hmin ? k : at;
#pragma unroll
            for (int k = 0; k < kPerClass; k++)
                if (k == at) {
                    hv[k] = p;
                    hi[k] = i;
                }
            hmin = hv[0];
#pragma unroll
            for (int k = 1; k < kPerClass; k++) hmin = fminf(hmin, hv[k]);
        }
        }
    }
#pragma unroll
    for (int k = 0; k < kPerClass; k++) {
        mp[tid * kPerClass + k] = hv[k];
        mi[tid * kPerClass + k] = hi[k];
    }
    red_f[tid] = sum;
    __syncthreads();
    // merge the class's 4 lists (threads c, c + 256, c + 512, c + 768): the first 8 of 32 by
    // (p desc, index asc)
    if (sub == 0) {
        for (int k = 0; k < kPerClass; k++) {
            int best = -1;
            float bp = -2.0f;
            int bi = 0x7FFFFFFF;
            for (int j = 0; j < kSub * kPerClass; j++) {
                const int at = ((j / kPerClass) * kClasses + c) * kPerClass + j % kPerClass;
                const float pj = mp[at];
                const int ij = mi[at];
                if (ij >= 0 && before(pj, ij, bp, bi)) {
                    bp = pj;
                    bi = ij;
                    best = at;
                }
            }
            cp[c * kPerClass + k] = best >= 0 ? bp : -1.0f;
            ci[c * kPerClass + k] = best >= 0 ? bi : 0x7FFFFFFF;
            if (best >= 0) mi[best] = -1;
        }
    }
    for (int s = kSampleThreads / 2; s > 0; s >>= 1) {
        if (tid < s) red_f[tid] += red_f[tid + s];
        __syncthreads();
    }
    const float total = red_f[0];

    __shared__ SelLds sel;
    uint64_t key[2];
#pragma unroll
    for (int r = 0; r < 2; r++) key[r] = cand_key(cp[2 * tid + r], ci[2 * tid + r]);
    select_sorted(key, total, top_p, seed, sel, out);
}

// ------------------------------------------------------------------ workspace form
// The same selection over two launches that spread the scan of the vocabulary:
//  1. sample_classes_kernel, 64 workgroups: workgroup w takes the residue classes 4w .. 4w+3
//     (i mod 256) over the whole vocabulary, each class on 64 threads; it writes its 32
//     class winners -- the 8 largest logits of each class, equal logits by the lower index
//     (the order of p = exp((z - max) / T), which is increasing in z) -- with their ids, its
//     largest logit m_w and S_w = sum exp((z - m_w) / T) over its classes;
//  2. sample_finish_kernel, one workgroup: M = max m_w, total = sum_w S_w exp((m_w - M) / T),
//     p of the 2048 winners from their logits as the one-launch form computes them, then the
//     same sort, nucleus and draw; temperature <= 0: sample_argmax_kernel, the first winner in
//     (z desc, id asc) order.
// Differences to the one-launch form: the total is summed per class group first (fp32 sums
// in another order); a class's 8th and 9th largest p can only be exchanged when their
// logits differ but round to the same p.
constexpr int kClsGroups = 64;                 // workgroups of the first launch
constexpr int kClsPerGroup = kClasses / kClsGroups;  // 4
constexpr int kClsThreads = 256;               // 64 threads per class
constexpr int kClsPerThread = 16;              // logits per thread: vocab <= 16 * 64 * 256 = 262144
struct SampleWs {
    float m[kClsGroups], s[kClsGroups];
    float z[kCands];
    int id[kCands];
};

size_t sample_workspace_bytes() { return sizeof(SampleWs); }

__global__ void __launch_bounds__(kClsThreads) sample_classes_kernel(const float *__restrict__ logits, int V,
                                                                     float temperature, SampleWs *__restrict__ ws) {
    __shared__ float lz[kClsThreads * kPerClass];
    __shared__ int li[kClsThreads * kPerClass];
    __shared__ float red[kClsThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int cl = tid & (kClsPerGroup - 1);                   // class within the group
    const int c = (int)blockIdx.x * kClsPerGroup + cl, j0 = tid / kClsPerGroup;  // 64 threads per class
    float z[kClsPerThread];
    float m = -INFINITY;
#pragma unroll
    for (int u = 0; u < kClsPerThread; u++) {
        const int i = c + kClasses * (j0 + 64 * u);
        z[u] = i < V ? logits[i] : -INFINITY;
        m = fmaxf(m, z[u]);
    }
    // the group's largest logit
    m = wave_max_all(m);
    if (lane == 0) red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // this thread's 8 largest (z desc, index asc: its indices increase with u) and its sum
    float hv[kPerClass];
    int hi[kPerClass];
#pragma unroll
    for (int k = 0; k < kPerClass; k++) {
        hv[k] = -INFINITY;
        hi[k] = 0x7FFFFFFF;
    }
    float sum = 0.0f;
#pragma unroll
    for (int u = 0; u < kClsPerThread; u++) {
        const int i = c + kClasses * (j0 + 64 * u);
        if (i < V) {
            sum += expf((z[u] - m) / temperature);
            // insert (z[u], i) keeping hv sorted descending; a later equal z goes after
            float v = z[u];
            int id = i;
#pragma unroll
            for (int k = 0; k < kPerClass; k++) {
                const bool take = v > hv[k];
                const float tv = hv[k];
                const int ti = hi[k];
                hv[k] = take ? v : hv[k];
                hi[k] = take ? id : hi[k];
                v = take ? tv : v;
                id = take ? ti : id;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kPerClass; k++) {
        lz[tid * kPerClass + k] = hv[k];
        li[tid * kPerClass + k] = hi[k];
    }
    sum = sum64_lane63(sum);
    __syncthreads();
    if (lane == 63) red[tid >> 6] = sum;
    __syncthreads();
    if (tid == 0) {
        ws->m[blockIdx.x] = m;
        ws->s[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
    }
    // wave w merges class w's 64 lists (512 entries, 8 per lane) by 8 rounds of wave argmax
    const int w = tid >> 6;
    const int cw = (int)blockIdx.x * kClsPerGroup + w;
    float bz[kPerClass];
    int bi[kPerClass];
#pragma unroll
    for (int k = 0; k < kPerClass; k++) {
        const int t = kClsPerGroup * lane + w;  // thread of class w in slot `lane`
        bz[k] = lz[t * kPerClass + k];
        bi[k] = li[t * kPerClass + k];
    }
    int head = 0;  // the lane's list is sorted: its best remaining entry is bz[head]
    for (int r = 0; r < kPerClass; r++) {
        float v = -INFINITY;
        int id = 0x7FFFFFFF;
#pragma unroll
        for (int k = 0; k < kPerClass; k++)
            if (k == head) {
                v = bz[k];
                id = bi[k];
            }
        float bv = v;
        int bid = id;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o);
            const int oi = __shfl_xor(bid, o);
            if (ov > bv || (ov == bv && oi < bid)) {
                bv = ov;
                bid = oi;
            }
        }
        if (id == bid && v == bv && bid != 0x7FFFFFFF) head++;  // the owner drops its head
        if (lane == 0) {
            ws->z[cw * kPerClass + r] = bv;
            ws->id[cw * kPerClass + r] = bid;
        }
    }
}

// temperature <= 0: the best class winner (ties to the lower id).  Thread c holds class c's first
// winner; the groups' sums are not needed (both launches 12.6 -> 11.7 us; 13.5 with this as a
// branch of the sampling kernel's 1024 threads).
__global__ void __launch_bounds__(kClasses) sample_argmax_kernel(const SampleWs *__restrict__ ws, int *__restrict__ out) {
    __shared__ float wv[kClasses / 64];
    __shared__ int wi[kClasses / 64];
    const int tid = threadIdx.x;
    float bv = ws->z[tid * kPerClass];
    int bi = ws->id[tid * kPerClass];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o);
        const int oi = __shfl_xor(bi, o);
        if (ov > bv || (ov == bv && oi < bi)) {
            bv = ov;
            bi = oi;
        }
    }
    if ((tid & 63) == 0) {
        wv[tid >> 6] = bv;
        wi[tid >> 6] = bi;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kClasses / 64; w++)
            if (wv[w] > bv || (wv[w] == bv && wi[w] < bi)) {
                bv = wv[w];
                bi = wi[w];
            }
        *out = bi == 0x7FFFFFFF ? 0 : bi;
    }
}

__global__ void __launch_bounds__(kSampleThreads) sample_finish_kernel(const SampleWs *__restrict__ ws,
                                                                    float temperature, float top_p,
                                                                    unsigned long long seed, int *__restrict__ out) {
    __shared__ SelLds sel;
    __shared__ float tot;
    __shared__ float Ms;
    const int tid = threadIdx.x;
    // winners 2 tid, 2 tid + 1 of the 2048 (8 per class), loaded with the groups' values
    static_assert(kCands == 2 * kSampleThreads, "two candidates per thread");
    const float2 cz = *(const float2 *)(ws->z + 2 * tid);
    const int2 ci = *(const int2 *)(ws->id + 2 * tid);
    if (tid < 64) {
        // one group per lane: the common max and the rescaled total as wave reductions
        // (one round trip to the workspace, a fixed summation order)
        static_assert(kClsGroups == 64, "one class group per lane");
        const float mg = ws->m[tid], sg = ws->s[tid];
        const float M = wave_max_all(mg);
        const float t = wave_sum_all(mg > -INFINITY ? sg * expf((mg - M) / temperature) : 0.0f);
        if (tid == 0) {
            Ms = M;
            tot = t;
        }
    }
    __syncthreads();
    const float M = Ms;
    // p as the one-launch form computes it
    uint64_t key[2];
    key[0] = cand_key(ci.x == 0x7FFFFFFF ? -1.0f : expf((cz.x - M) / temperature), ci.x);
    key[1] = cand_key(ci.y == 0x7FFFFFFF ? -1.0f : expf((cz.y - M) / temperature), ci.y);
    select_sorted(key, tot, top_p, seed, sel, out);
}

int launch_sample_token_ws(const float *logits, int V, float temperature, float top_p, unsigned long long seed,
                           void *ws, size_t ws_bytes, int *out, hipStream_t stream) {
    if (!logits || !out || !ws || V <= 0) return set_error(kErrBadArg, "sample_token_ws: bad arguments");
    if (V > kClasses * 64 * kClsPerThread)
        return set_error(kErrBadArg, "sample_token_ws: vocabulary above %d", kClasses * 64 * kClsPerThread);
    if (ws_bytes < sizeof(SampleWs) || ((uintptr_t)ws & 15))
        return set_error(kErrBadArg, "sample_token_ws: workspace of %zu bytes (need %zu, 16-byte aligned)", ws_bytes,
                         sizeof(SampleWs));
    SampleWs *w = (SampleWs *)ws;
    hipLaunchKernelGGL(sample_classes_kernel, dim3(kClsGroups), dim3(kClsThreads), 0, stream, logits, V,
                       temperature > 0.0f ? temperature : 1.0f, w);
    if (temperature <= 0.0f) hipLaunchKernelGGL(sample_argmax_kernel, dim3(1), dim3(kClasses), 0, stream, w, out);
    else
        hipLaunchKernelGGL(sample_finish_kernel, dim3(1), dim3(kSampleThreads), 0, stream, w, temperature, top_p, seed,
                           out);
    return check_launch("sample_token_ws");
}

int launch_sample_token(const float *logits, int V, float temperature, float top_p, unsigned long long seed,
                        int *out, hipStream_t stream) {
    if (!logits || !out || V <= 0) return set_error(kErrBadArg, "sample_token: bad arguments");
    hipLaunchKernelGGL(sample_token_kernel, dim3(1), dim3(kSampleThreads), 0, stream, logits, V, temperature, top_p,
                       seed, out);
    return check_launch("sample_token");
}

}  // namespace mnemo
