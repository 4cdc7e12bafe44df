// attn_prompt.hip - ggml_flash_attn_ext over an f16 KV cache for several query rows (a prompt chunk,
// a few speculative rows) on the matrix cores (runtime/src/ops.cpp:217-243 ->
// runtime/include/ggml_compiler_ops.h:133-136, GGML_PREC_F32). Semantics as in attn.hip.
//
// A wavefront takes 32 rows, a row being a (query, head) pair of one KV head: row q * G + g, so the G
// heads that share K / V are rows of one tile, whatever G is. Key blocks of 64 go through LDS,
// double-buffered, K as rows, V transposed (4 keys x 4 dims per lane, turned in registers):
//   - scores S^T[key][row] = K Q^T with v_mfma_f32_32x32x16_f16 (Q rounded to f16): lane (row, half lk)
//     is left with keys 8 i + 4 lk + r of its row, so a row's softmax needs one exchange with lane ^ 32;
//   - O^T[dim][row] += V^T P^T: P is used where the scores lie (the MFMA's k slots are those keys, V^T
//     read in the same order), scaled by 2^15, as NP f16 parts: its rounding, the remainder's rounding, ..
//     Two parts hold 22 bits of a weight down to 2^-17 of 2^R below, three all 24 bits down to 2^-16; smaller
//     weights to an absolute 2^-40 of 2^R (f16's finest step), the f32 sum's own rounding being 2^-24 of more.
// The softmax runs in powers of two against an integer reference R >= the running maximum: raising
// R rescales by an exact power of two and is rare, and splits with the same R merge without rounding.
// Blocks that no row of the workgroup sees (mask all -inf: k_attn_mask_bits looks the mask over first; or
// past the causal edge) are left out, and a block without a mask value takes no mask work. A finite mask value
// is added to the scaled score before the exponent, as in attn.hip: divided by the scale and added to the dot it was
// rounded at its own size times 1 / scale (1.2 to 1.6 times the error, masks of N(0, 2), 1000 and -65504).
//
// Wavefronts: RW row groups x KW key halves of each block (KW = 2 where the rows are few; the halves
// meet in LDS at the end). Grid (row tile, KV head, key split); the splits' partials have k_attn_split's
// layout and go through the same merges.
//
// What bounds it: per 32 rows x 32 keys at D = 128, 24 MFMAs (8 for the scores, 16 for the two parts of
// P V) of 32 clocks, about 300 other VALU operations, and the latency of the LDS operands, which two
// wavefronts per SIMD (256 registers) do not hide: the matrix cores are busy 28 % of the cycles. 32 / 8
// heads x 128, 512 rows over 4096 keys, causal mask: 817 us with the per-row kernel (K / V read again for
// every query row, dots on the VALU), 92 us so with the look at the mask and the merge (the kernel
// 86); 2048 rows over 2048 keys: 1661 -> 131 us. Off 64 bits at 4096 keys: 1.9e-7, the per-row
// kernel 2.3e-7.
#include "gcq_common.h"

#include <algorithm>

namespace gcq {

namespace {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int KB = 64;          // keys per block
constexpr int VP = KB + 4;      // pitch of a V^T row (halves): 16 lanes' 8-byte reads in distinct banks
// Up to these keys, or 64 rows of a KV head, every block takes the mask: looking it over first costs a launch (129 rows x 256
// keys, 14 / 2 heads of 64: 22.2 us with it, 18.9 without; 2 rows x 32768 keys, 8 heads of 64: 27.9 us and 23.5 in k_attn_split).
constexpr int kBitsKeys = 512;
constexpr float kPScale = 32768.0f;  // P's scale

struct PromptArgs {
    const float * q;
    int64_t q_h, q_s;
    const uint16_t * k, * v;
    int64_t k_h, k_j, v_h, v_j;
    const uint16_t * mask;
    int64_t m_s;
    const uint2 * bits;  // k_attn_mask_bits
    float scale2;   // |scale| * log2(e); negate: the scale is negative (Q's sign turns)
    float mag;      // |scale|
    bool negate;
    int Sq, H, G, n_kv, pos0, blocks, nsplit;  // blocks: key blocks per split
    float * out, * part_o;
    float2 * part_ml;
};

__device__ __forceinline__ float xhalf_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

enum { kAllKeys = 0, kMask = 1, kCausal = 2 };

// What of a mask a row tile (queries q0 .. of `tile` rows) sees of each key block: bits[tile][word].x bit i, some
// value of block 32 word + i is not -inf; .y, some value is not 0. A wavefront takes two blocks.
__global__ __launch_bounds__(1024) void k_attn_mask_bits(const uint16_t * __restrict__ mask, int64_t m_s, int Sq, int G,
                                                         int n_kv, int tile, uint2 * __restrict__ bits) {
    __shared__ uint32_t sh[2];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t r0 = (int64_t) blockIdx.y * tile, r1 = min(r0 + tile, (int64_t) Sq * G) - 1;
    const int q0 = (int) (r0 / G), q1 = (int) (r1 / G);
    if (tid < 2) sh[tid] = 0;
    __syncthreads();
    for (int k = 0; k < 2; k++) {
        const int i = 2 * wave + k, j = ((int) blockIdx.x * 32 + i) * KB + 8 * (lane & 7);
        uint32_t seen = 0, val = 0;
#pragma unroll 4
        for (int q = q0 + (lane >> 3); q <= q1; q += 8) {
            const uint16_t * p = mask + (int64_t) q * m_s + j;
            if (j + 8 <= n_kv) {
                u4_t m;
                __builtin_memcpy(&m, p, 16);
                constexpr uint32_t inf2 = 0xfc00fc00u;
                seen |= (m.x ^ inf2) | (m.y ^ inf2) | (m.z ^ inf2) | (m.w ^ inf2);
                val |= m.x | m.y | m.z | m.w;
            } else {
                for (int e = 0; e < 8; e++)
                    if (j + e < n_kv) {
                        seen |= p[e] ^ 0xfc00u;
                        val |= p[e];
                    }
            }
        }
        const bool s = __any(seen != 0), v = __any(val != 0);
        if (lane == 0 && s) atomicOr(&sh[0], 1u << i);
        if (lane == 0 && v) atomicOr(&sh[1], 1u << i);
    }
    __syncthreads();
    if (tid == 0) bits[(int64_t) blockIdx.y * gridDim.x + blockIdx.x] = make_uint2(sh[0], sh[1]);
}

template <int D, int RW, int KW, int NP, int MODE>
__global__ __launch_bounds__(64 * RW * KW, RW == 1 ? 1 : 2) void k_attn_prompt(const PromptArgs a) {
    constexpr int NW = RW * KW, NT = 64 * NW, KT = 2 / KW;
    constexpr int KP = D + 8;                       // pitch of a K row (halves)
    constexpr int KL = KB * (D / 8) / NT;           // 16-byte K pieces per thread
    constexpr int VL = (D / 32) * (KB / 32) / NW;   // 4-key x 4-dim V tiles per lane
    struct Lds {
        _Float16 k[KB * KP];
        _Float16 v[D * VP];
    };
    __shared__ __align__(16) Lds L[2];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int rw = wave % RW, kw = wave / RW, lr = lane & 31, lk = lane >> 5;
    const int rows = a.Sq * a.G, tiles = (rows + 32 * RW - 1) / (32 * RW);
    // An XCD takes a contiguous run of (KV head, split, row tile), row tiles fastest: the workgroups that
    // read the same K / V rows share its L2.
    int id = blockIdx.x;
    if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
    const int tile = id % tiles, split = id / tiles % a.nsplit, hk = id / tiles / a.nsplit;
    const int r0 = tile * 32 * RW + rw * 32;  // this wavefront's first row
    const int row = min(r0 + lr, rows - 1), s = row / a.G, h = hk * a.G + row % a.G;
    const int s_first = min(r0, rows - 1) / a.G;

    // This lane's row of Q, f16: dims 16 c + 8 lk + 0..7.
    h8_t qf[D / 16];
    {
        const float * qp = a.q + (int64_t) h * a.q_h + (int64_t) s * a.q_s + 8 * lk;
#pragma unroll
        for (int c = 0; c < D / 16; c++) {
            f4_t f[2];
            __builtin_memcpy(&f[0], qp + 16 * c, 16);
            __builtin_memcpy(&f[1], qp + 16 * c + 4, 16);
#pragma unroll
            for (int j = 0; j < 8; j++) qf[c][j] = (_Float16) (a.negate ? -f[j >> 2][j & 3] : f[j >> 2][j & 3]);
        }
    }

    const int nblk = (a.n_kv + KB - 1) / KB;
    const int b0 = split * a.blocks;
    int b1 = min(nblk, b0 + a.blocks);
    if (MODE == kCausal) {  // no row of the workgroup sees a key past its last row's position
        const int sl = min((tile + 1) * 32 * RW - 1, rows - 1) / a.G;
        b1 = min(b1, (min(a.n_kv, a.pos0 + sl + 1) + KB - 1) / KB);
    }

    // The next block to compute from b on, b1 if none: every block, or those whose mask bits say seen.
    const uint2 * bits = MODE == kMask && a.bits ? a.bits + (int64_t) tile * ((nblk + 31) / 32) : nullptr;
    const auto next = [&](int b) {
        if (MODE == kMask && bits) {
            while (b < b1) {
                const uint32_t w = (uint32_t) __builtin_amdgcn_readfirstlane((int) bits[b >> 5].x) >> (b & 31);
                if (w) return min(b + __builtin_ctz(w), b1);
                b = (b | 31) + 1;
            }
        }
        return min(b, b1);
    };

    const uint16_t * kb = a.k + (int64_t) hk * a.k_h;
    const uint16_t * vb = a.v + (int64_t) hk * a.v_h;
    // (native vector types: HIP's uint4 structs put the staged loads in scratch memory)
    u4_t kr[KL];
    u2_t vr[VL][4];
    // Blocks through buffers that begin at the block's first row and end with row n_kv - 1: rows past it
    // read zeros (their scores are dropped), and one offset register serves all of a thread's loads.
    const uint32_t kj2 = 2 * (uint32_t) a.k_j, vj2 = 2 * (uint32_t) a.v_j;
    const uint32_t ok = tid / (D / 8) * kj2 + 16 * (tid % (D / 8)), ov = 4 * (lane >> 3) * vj2 + 8 * (lane & 7);
    const auto load = [&](int b) {
        const uint32_t last = (uint32_t) min(KB, a.n_kv - b * KB) - 1;
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t *>(kb + (int64_t) b * KB * a.k_j), 0, (int) (last * kj2 + 2 * D), 0x00020000);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t *>(vb + (int64_t) b * KB * a.v_j), 0, (int) (last * vj2 + 2 * D), 0x00020000);
#pragma unroll
        for (int i = 0; i < KL; i++)
            kr[i] = __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, ok + i * (NT / (D / 8)) * kj2, 0, 0));
#pragma unroll
        for (int i = 0; i < VL; i++) {
            const int u = wave + NW * i;  // dims 32 (u % (D / 32)) .., keys 32 (u / (D / 32)) ..
#pragma unroll
            for (int e = 0; e < 4; e++)
                vr[i][e] = __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(
                                                        rv, ov + (32 * (u / (D / 32)) + e) * vj2 + 64 * (u % (D / 32)), 0, 0));
        }
    };
    const auto store = [&](Lds & l) {
#pragma unroll
        for (int i = 0; i < KL; i++) {
            const int p = tid + NT * i;
            *reinterpret_cast<u4_t *>(l.k + (p / (D / 8)) * KP + 8 * (p % (D / 8))) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < VL; i++) {
            const int u = wave + NW * i, dg = (u % (D / 32)) * 8 + (lane & 7), kg = (u / (D / 32)) * 8 + (lane >> 3);
#pragma unroll
            for (int d = 0; d < 4; d++) {  // dim 4 dg + d of the four keys
                const auto w = [&](int e) { return d < 2 ? vr[i][e].x : vr[i][e].y; };
                const uint32_t sel = d & 1 ? 0x07060302u : 0x05040100u;
                *reinterpret_cast<u2_t *>(l.v + (4 * dg + d) * VP + 4 * kg) =
                    u2_t{__builtin_amdgcn_perm(w(1), w(0), sel), __builtin_amdgcn_perm(w(3), w(2), sel)};
            }
        }
    };
    float O[D / 32][16];  // (not vectors: they are updated one by one, and 16-register groups do not pack)
#pragma unroll
    for (int t = 0; t < D / 32; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) O[t][e] = 0.0f;
    float R = -INFINITY, l = 0.0f;  // reference exponent (an integer) and this lane's half of the weights' sum

    // A block's mask values of this lane's keys k0 .. k0 + 3 (past the row's end: the last four, shifted where they are
    // used). KW == 1 loads them at the block's start, before the next block's K and V (a load waits for all before it); KW == 2,
    // whose rows are few and whose registers are not, a block ahead.
    const auto k0 = [&](int t, int i) { return 32 * (KW == 2 ? kw : t) + 8 * i + 4 * lk; };
    uint64_t mw[MODE == kMask ? KT : 1][4];
    const auto load_mask = [&](int b) {
        const uint16_t * mr = a.mask + (int64_t) s * a.m_s + b * KB;
#pragma unroll
        for (int t = 0; t < (MODE == kMask ? KT : 1); t++)
#pragma unroll
            for (int i = 0; i < 4; i++) __builtin_memcpy(&mw[t][i], mr + min(k0(t, i), a.n_kv - b * KB - 4), 8);
        asm volatile("");
    };

    int b = next(b0), slot = 0;
    if (MODE == kMask && KW == 2 && b < b1) load_mask(b);
    if (b < b1) {
        load(b);
        store(L[0]);
    }
    __syncthreads();
    while (b < b1) {
        const Lds & lds = L[slot];
        const int bn = next(b + 1);
        // some row of this wavefront does not see every key of the block, or with a mask value
        bool some = b * KB + KB > a.n_kv;
        if constexpr (MODE == kCausal) some = some || b * KB + KB - 1 > a.pos0 + s_first;
        if constexpr (MODE == kMask) some = some || !bits || ((uint32_t) __builtin_amdgcn_readfirstlane((int) bits[b >> 5].y) >> (b & 31) & 1);
        const int left = a.n_kv - b * KB;
        if (MODE == kMask && KW == 1 && some) load_mask(b);
        load(min(bn, b1 - 1));
        // Dots of D values: chains of two MFMAs, added in f32. A sum inside the MFMA is cut off, not rounded, against a
        // growing accumulator (one chain of eight: 1.10 times the error of f32 dots, chains of two 0.95).
        v16f S[KT];
        const _Float16 * kp = lds.k + (32 * (KW == 2 ? kw : 0) + lr) * KP + 8 * lk;
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const auto dot = [&](int c) {  // dims 16 c .. 16 c + 31
                v16f A{};
#pragma unroll
                for (int e = 0; e < 2; e++)
                    A = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8_t *>(kp + 32 * t * KP + 16 * (c + e)), qf[c + e], A, 0, 0, 0);
                return A;
            };
            S[t] = dot(0) + dot(2);
            if constexpr (D == 128) {
                __builtin_amdgcn_sched_barrier(0);  // (all four chains at once: their registers spill others)
                S[t] += dot(4) + dot(6);
            }
        }
        float c2 = a.scale2;  // a key's exponent is c2 S
        float mx = -INFINITY;
        if (some) {
            asm volatile("");  // a branch: as selects this runs for every block
            const int seen = MODE == kCausal ? min(left, a.pos0 + s + 1 - b * KB) : left;
            const auto value = [&](int t, int i, int r) {
                return h2f((uint16_t) (mw[t][i] >> (16 * min(k0(t, i) - min(k0(t, i), left - 4), 3)) >> (16 * r)));
            };
            bool add = false;  // a mask value that is neither 0 nor -inf
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    bool drop = k0(t, e >> 2) + (e & 3) >= seen;
                    if constexpr (MODE == kMask) {
                        const float mv = value(t, e >> 2, e & 3);
                        drop = drop || mv == -INFINITY;
                        add = add || (!drop && mv != 0.0f);
                    }
                    S[t][e] = drop ? -INFINITY : S[t][e];
                }
            if constexpr (MODE == kMask)
                if (__any(add)) {  // scores and values summed at the values' own size
                    asm volatile("");
#pragma unroll
                    for (int t = 0; t < KT; t++)
#pragma unroll
                        for (int e = 0; e < 16; e++)
                            S[t][e] = S[t][e] == -INFINITY ? S[t][e] : fmaf(S[t][e], a.mag, value(t, e >> 2, e & 3));
                    c2 = 1.44269504088896341f;
                }
        }
        if (MODE == kMask && KW == 2) load_mask(min(bn, b1 - 1));
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) mx = fmaxf(mx, S[t][e]);
        mx = ceilf(xhalf_max(mx) * c2);
        // a power of two, nearly always 1
        const float Rn = fmaxf(R, mx), al = R == Rn ? 1.0f : R == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(R - Rn);
        R = Rn;
        // 2^(c2 S - R) with one rounding of the small difference, then the exact scale
        const float base = R == -INFINITY ? 0.0f : R;
        // From 2^22 on R is c2 S rounded by up to a quarter and more: the largest S must be rounded alike.
        if (__builtin_expect(__any(fabsf(base) >= 0x1p22f), 0)) {
            asm volatile("");
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) S[t][e] *= c2;
            c2 = 1.0f;
        }
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) S[t][e] = __builtin_amdgcn_exp2f(fmaf(S[t][e], c2, -base)) * kPScale;
        // The weights as NP f16 parts, each rounded to nearest. Two: the sum of weights is of what the parts hold, so that
        // numerator and denominator see the same weights; three: all 24 bits.
        float ls[2] = {0.0f, 0.0f};
        h8_t ph[NP][2 * KT];  // 16 keys each: k slot (lk, j) is key 16 c + 4 lk + j, or + 8 + 4 lk + j - 4
        constexpr h2_t one = {(_Float16) 1.0f, (_Float16) 1.0f};
#pragma unroll
        for (int c = 0; c < 2 * KT; c++)
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                float p0 = S[c >> 1][8 * (c & 1) + j], p1 = S[c >> 1][8 * (c & 1) + j + 1];
                if constexpr (NP == 3) ls[0] += p0, ls[1] += p1;
#pragma unroll
                for (int n = 0; n < NP; n++) {
                    const h2_t w = {(_Float16) p0, (_Float16) p1};
                    if constexpr (NP == 2) ls[n] = __builtin_amdgcn_fdot2(w, one, ls[n], false);
                    p0 = fmaf((float) w.x, -1.0f, p0);
                    p1 = fmaf((float) w.y, -1.0f, p1);
                    ph[n][c][j] = w.x, ph[n][c][j + 1] = w.y;
                }
            }
        l = fmaf(l, al, ls[0] + ls[1]);
        // The block's P V from zero, its first part and the others in chains of their own, then one multiply-add into
        // the sums (with their rescaling): few additions inside the MFMAs (as above), and one f32 rounding per block.
        const _Float16 * vp = lds.v + lr * VP + 32 * (KW == 2 ? kw : 0) + 4 * lk;
#pragma unroll
        for (int d = 0; d < D / 32; d++) {  // one at a time (more leave no registers for the staged loads)
            __builtin_amdgcn_sched_barrier(0);
            v16f T{}, Tl{};
#pragma unroll
            for (int c = 0; c < 2 * KT; c++) {
                const u2_t v0 = *reinterpret_cast<const u2_t *>(vp + 32 * d * VP + 16 * c);
                const u2_t v1 = *reinterpret_cast<const u2_t *>(vp + 32 * d * VP + 16 * c + 8);
                const h8_t vf = __builtin_bit_cast(h8_t, u4_t{v0.x, v0.y, v1.x, v1.y});
#pragma unroll
                for (int n = NP - 1; n > 0; n--) Tl = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, ph[n][c], Tl, 0, 0, 0);
                T = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, ph[0][c], T, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 16; e++) O[d][e] = fmaf(O[d][e], al, T[e] + Tl[e]);
        }
        slot ^= 1;
        store(L[slot]);
        __syncthreads();
        b = bn;
    }
    l = xhalf_sum(l);
    if (R == -INFINITY) {  // no key seen, or only NaN scores: the row's sums are zero
        l = 0.0f;
#pragma unroll
        for (int t = 0; t < D / 32; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) O[t][e] = 0.0f;
    }

    // An infinite V value: its product with P's remainder (0 or negative for most weights) has made a NaN of the sums.
    // A wavefront whose sums are not all finite forms them again key by key, with the weights in f32.
    float fin = 0.0f;
#pragma unroll
    for (int t = 0; t < D / 32; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) fin = fmaf(O[t][e], 0.0f, fin);  // NaN if any is not finite
    if (__builtin_expect(__any(fin != fin), 0)) {
        asm volatile("");
#pragma unroll
        for (int t = 0; t < D / 32; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) O[t][e] = 0.0f;
        for (int bs = next(b0); bs < b1; bs = next(bs + 1)) {
            const int j0 = bs * KB + (KW == 2 ? 32 * kw : 0);
            int j1 = min(j0 + KB / KW, a.n_kv);
            if (MODE == kCausal) j1 = min(j1, a.pos0 + s + 1);
#pragma unroll 1
            for (int j = j0; j < min(j0 + KB / KW, a.n_kv); j++) {
                float x = 0.0f;  // lanes lr and lr + 32 hold the dims in halves
#pragma unroll
                for (int c = 0; c < D / 16; c++) {
                    u4_t kf;
                    __builtin_memcpy(&kf, kb + (int64_t) j * a.k_j + 16 * c + 8 * lk, 16);
                    const u4_t qc = __builtin_bit_cast(u4_t, qf[c]);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t kw2 = kf[i], qw2 = qc[i];  // (a bit_cast of kf[i] itself takes element 0)
                        x = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, kw2), __builtin_bit_cast(h2_t, qw2), x, false);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                x = xhalf_sum(x);
                bool drop = j >= j1;
                if constexpr (MODE == kMask) {
                    const float mv = h2f(a.mask[(int64_t) s * a.m_s + j]);
                    drop = drop || mv == -INFINITY;
                    x = fmaf(x, a.mag, mv) * 1.44269504088896341f;
                } else {
                    x *= a.scale2;
                }
                const float p = __builtin_amdgcn_exp2f(x - R) * kPScale;
                if (drop || R == -INFINITY) continue;
                const uint16_t * vj = vb + (int64_t) j * a.v_j + 4 * lk;
#pragma unroll
                for (int t = 0; t < D / 32; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        u2_t w;
                        __builtin_memcpy(&w, vj + 32 * t + 8 * i, 8);
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            O[t][4 * i + r] = fmaf(p, h2f((uint16_t) ((r < 2 ? w.x : w.y) >> (16 * (r & 1)))), O[t][4 * i + r]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }
    }

    if constexpr (KW == 2) {  // the two key halves: the second hands its sums to the first
        float * ex = reinterpret_cast<float *>(&L[0]) + (size_t) rw * 64 * (D / 2 + 2) + lane;
        static_assert(sizeof(L) >= (size_t) RW * 64 * (D / 2 + 2) * 4, "exchange fits");
        if (kw == 1) {
            ex[0] = R;
            ex[64] = l;
#pragma unroll
            for (int t = 0; t < D / 32; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) ex[64 * (2 + 16 * t + e)] = O[t][e];
        }
        __syncthreads();
        if (kw == 1) return;
        const float R1 = ex[0], Rn = fmaxf(R, R1);
        const float a0 = R == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(R - Rn);
        const float a1 = R1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(R1 - Rn);
        R = Rn;
        l = a0 * l + a1 * ex[64];
#pragma unroll
        for (int t = 0; t < D / 32; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) O[t][e] = a0 * O[t][e] + a1 * ex[64 * (2 + 16 * t + e)];
    }
    if (r0 + lr >= rows) return;
    const int64_t sh = (int64_t) s * a.H + h;
    if (a.out) {
        float * o = a.out + sh * D + 4 * lk;
#pragma unroll
        for (int t = 0; t < D / 32; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                f4_t y;
#pragma unroll
                for (int r = 0; r < 4; r++) y[r] = l == 0.0f ? 0.0f : O[t][4 * i + r] / l;
                __builtin_memcpy(o + 32 * t + 8 * i, &y, sizeof y);
            }
        return;
    }
    // The merge's maximum m is R ln 2 rounded to f32; the sums take what the rounding leaves (16 and more: 1e-6 of a
    // split's weight, at a mask value of -65504 2e-3).
    const float m = R * 0.693147180559945309f;
    if (fabsf(R) < 0x1p22f) {
        const float f = __expf(fmaf(R, -1.904654323148236017e-09f, fmaf(R, 0.693147180559945309f, -m)));  // ln 2 in two parts
        l *= f;
#pragma unroll
        for (int t = 0; t < D / 32; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) O[t][e] *= f;
    }
    float * o = a.part_o + (sh * a.nsplit + split) * D + 4 * lk;
#pragma unroll
    for (int t = 0; t < D / 32; t++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<f4_t *>(o + 32 * t + 8 * i) = f4_t{O[t][4 * i], O[t][4 * i + 1], O[t][4 * i + 2], O[t][4 * i + 3]};
    if (lk == 0) a.part_ml[sh * a.nsplit + split] = make_float2(m, l);
}

// Row groups of a workgroup for `rows` rows of a KV head: 4 (128 rows), 2, or 1 with the key blocks halved.
int row_groups(int64_t rows) { return rows <= 32 ? 1 : rows <= 64 ? 2 : 4; }

template <int D, int RW, int KW, int NP>
void run(const PromptArgs & a, int Hkv, int mode, hipStream_t s) {
    const unsigned grid = (unsigned) (((int64_t) a.Sq * a.G + 32 * RW - 1) / (32 * RW) * Hkv * a.nsplit);
    if (mode == kMask) k_attn_prompt<D, RW, KW, NP, kMask><<<grid, 64 * RW * KW, 0, s>>>(a);
    else if (mode == kCausal) k_attn_prompt<D, RW, KW, NP, kCausal><<<grid, 64 * RW * KW, 0, s>>>(a);
    else k_attn_prompt<D, RW, KW, NP, kAllKeys><<<grid, 64 * RW * KW, 0, s>>>(a);
}

// Weights in three parts where the keys are few enough for single weights to show (up to 64 rows and 512 keys: 3 rows over 4
// keys 1.0 of the per-row kernel's error, 1.07 in two parts); two beyond (6 rows over 32768 keys, 32 heads of 64: 81 us in
// three, 68 in two) and for more rows, where the third costs most (512 rows over 4096 keys: 136 us and 92).
constexpr int kFewKeys = 512;
template <int D>
void run_rows(const PromptArgs & a, int Hkv, int mode, int rg, hipStream_t s) {
    const bool few = a.n_kv <= kFewKeys;
    if (rg == 4) run<D, 4, 1, 2>(a, Hkv, mode, s);
    else if (rg == 2 && few) run<D, 2, 2, 3>(a, Hkv, mode, s);
    else if (rg == 2) run<D, 2, 2, 2>(a, Hkv, mode, s);
    else if (few) run<D, 1, 2, 3>(a, Hkv, mode, s);
    else run<D, 1, 2, 2>(a, Hkv, mode, s);
}

}  // namespace

// (A mask needs rows of at least four values: launch_attn_prompt.) The scale's range: a dropped key's weight is
// 2^(scale -inf), no 0 where the scale is 0, and near the ends of f32 scale2 or its products leave it; k_attn_split takes the
// rest.
bool attn_prompt_fits(int D, int Sq, int H, int Hkv, float scale) {
    return (D == 64 || D == 128) && Sq > 1 && H % Hkv == 0 && H / Hkv <= 8 && (int64_t) Sq * (H / Hkv) < INT32_MAX &&
           fabsf(scale) >= 0x1p-60f && fabsf(scale) <= 0x1p60f;
}

// Key splits: about 512 workgroups in all (two per CU), each split of at least two key blocks, or one where the merge
// stays small (16 splits for up to 256 output rows, 8 for up to 2048): 33 rows of 32 heads over 300 keys 23.0 us in two splits
// of three blocks, 16.1 in five of one; 129 rows over 512 keys 18.5 in four of two, 24.4 in eight of one. No more for a smaller
// n_kv, so a bound for every KV length up to n_kv.
int attn_prompt_max_split(int Sq, int H, int Hkv, int n_kv) {
    const int64_t rows = (int64_t) Sq * (H / Hkv), tile = 32 * row_groups(rows);
    const int64_t wgs = (rows + tile - 1) / tile * Hkv;
    const int nblk = (n_kv + KB - 1) / KB;
    const int64_t out = (int64_t) Sq * H;
    const int singles = std::min(nblk, out <= 256 ? 16 : out <= 2048 ? 8 : 1);
    return (int) std::max<int64_t>(1, std::min<int64_t>({512 / wgs, std::max(singles, nblk / 2), 64}));
}
AttnPlan attn_plan_prompt(int Sq, int H, int Hkv, int n_kv) {
    const int nblk = (n_kv + KB - 1) / KB, most = attn_prompt_max_split(Sq, H, Hkv, n_kv);
    const int blocks = (nblk + most - 1) / most;
    return {(nblk + blocks - 1) / blocks, blocks * KB};
}

// Bytes of the mask's block bits.
size_t attn_prompt_bits(int Sq, int H, int Hkv, int n_kv) {
    const int64_t rows = (int64_t) Sq * (H / Hkv), tile = 32 * row_groups(rows);
    return align256((size_t) ((rows + tile - 1) / tile) * ((n_kv + 32 * KB - 1) / (32 * KB)) * sizeof(uint2));
}

// Sq query rows over n_kv keys. mask: [Sq][m_s] f16 (added to the scaled scores; -inf drops a key), or null;
// pos0 >= 0 (mask null): row s sees keys 0 .. pos0 + s. out [s][h][D] (one split), or null: partials
// (part_o, part_ml) for a merge. bits: attn_prompt_bits bytes for a mask, else null.
void launch_attn_prompt(const float * q, int64_t q_h, int64_t q_s, const void * k, int64_t k_h, int64_t k_j,
                        const void * v, int64_t v_h, int64_t v_j, const void * mask, int64_t m_s, int pos0, int D, int Sq,
                        int H, int Hkv, int n_kv, float scale, float * out, float * part_o, float2 * part_ml,
                        const AttnPlan & p, void * bits, hipStream_t s) {
    require(attn_prompt_fits(D, Sq, H, Hkv, scale), "attn prompt: D 64 or 128, several query rows, at most 8 heads per KV head, a scale within 2^-60 .. 2^60");
    require(p.chunk % KB == 0 && (int64_t) p.nsplit * p.chunk >= n_kv, "attn prompt: the splits must cover the keys");
    require(((int64_t) Sq * (H / Hkv) / 32 + 1) * Hkv * p.nsplit < INT32_MAX, "attn prompt: too many row tiles");
    require(!out || p.nsplit == 1, "attn prompt: several splits go to the merge");
    require(!mask || n_kv >= 4, "attn prompt: a mask of at least four keys");
    require(k_j < (1 << 24) && v_j < (1 << 24), "attn prompt: K / V row strides below 2^24");
    require(k_j % 8 == 0 && v_j % 8 == 0 && k_h % 8 == 0 && v_h % 8 == 0 && ((uintptr_t) k & 15) == 0 &&
                ((uintptr_t) v & 15) == 0,
            "attn prompt: 16-byte aligned K / V rows");
    PromptArgs a{};
    a.q = q, a.q_h = q_h, a.q_s = q_s;
    a.k = (const uint16_t *) k, a.k_h = k_h, a.k_j = k_j;
    a.v = (const uint16_t *) v, a.v_h = v_h, a.v_j = v_j;
    a.mask = (const uint16_t *) mask, a.m_s = m_s;
    a.scale2 = (float) (fabs((double) scale) * 1.4426950408889634074);
    a.negate = scale < 0.0f;
    a.mag = fabsf(scale);
    a.Sq = Sq, a.H = H, a.G = H / Hkv, a.n_kv = n_kv, a.pos0 = pos0, a.blocks = p.chunk / KB, a.nsplit = p.nsplit;
    a.out = out, a.part_o = part_o, a.part_ml = part_ml;
    const int mode = mask ? kMask : pos0 >= 0 ? kCausal : kAllKeys;
    const int rg = row_groups((int64_t) Sq * a.G);
    if (mask && n_kv > kBitsKeys && rg == 4) {
        const int tile = 32 * rg;
        const int64_t tiles = ((int64_t) Sq * a.G + tile - 1) / tile;
        require(bits && tiles <= 65535, "attn prompt: a mask needs its bits' workspace and at most 65535 row tiles");
        a.bits = (const uint2 *) bits;
        k_attn_mask_bits<<<dim3((unsigned) ((n_kv + 32 * KB - 1) / (32 * KB)), (unsigned) tiles), 1024, 0, s>>>(
            a.mask, m_s, Sq, a.G, n_kv, tile, (uint2 *) bits);
    }
    if (D == 64) run_rows<64>(a, Hkv, mode, rg, s);
    else run_rows<128>(a, Hkv, mode, rg, s);
    check_launch("attn prompt");
}

}  // namespace gcq
