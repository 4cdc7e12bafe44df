// gemm_kq.hip - quantized mat-mul for prefill (M > 8 activation rows) with K-quant weights (Q4_K,
// Q5_K, Q6_K) on int8 MFMA.
//
// Replaces ggml_mul_mat of a K-quant weight with an f32 src1 of many rows
// (runtime/src/ops.cpp:107-119). As ggml (vec_dot_type Q8_K), src1 is quantized to Q8_K per 256
// values (quant.hip); per super-block i and output (m, n) the integer parts of ggml's
// vec_dot_q{4,5,6}_K_q8_K are exact and the float part scales them:
//   Q4_K / Q5_K: I1 = sum_j sc_j(n) isum_j(m, n), I2 = sum_j m_j(n) (bsum_2j + bsum_2j+1)(m) over the
//                8 sub-blocks of 32; y += d_x(m) (d_w(n) I1 - dmin_w(n) I2)
//   Q6_K:        I1 = sum_j sc_j(n) isum_j(m, n) over the 16 sub-blocks of 16 (codes q - 32);
//                y += d_x(m) d_w(n) I1
//
// The sub-block scales go into the weight operand, so I1 is formed by the matrix cores alone: a
// weight enters as two int8 codes, hi and lo, with I1 = S sum(hi x) + sum(lo x) over the whole
// super-block in two int32 accumulators (v_mfma_i32_32x32x32_i8, twice the MFMAs of the bare codes).
//   Q4_K: sc = 8 sh + sl (sh, sl < 8): hi = sh q, lo = sl q (<= 105), S = 8
//   Q5_K: the same with q <= 31 (products <= 217 fit a byte but not an int8): taken minus 128, and both
//         accumulators start from 128 times the row's code sum of the super-block
//   Q6_K: v = sc (q - 32) in [-4096, 4096]: hi = v >> 6, lo = v & 63, S = 64
// I2 is one f16 MFMA of K 16 per tile and super-block: the activation's block sums in two f16 parts
// (a multiple of 64 and the rest) against the 6-bit mins, exact in f32.
//
// A workgroup is KG K groups of WN wavefronts; a wavefront takes 32 XT rows (m) x 32 columns (n), its tile
// 32 XT x 32 WN. Group g takes the super-blocks g, g + KG, ...; the groups' sums meet in LDS at the end
// (more wavefronts where the tiles are few). The activation codes go through LDS, double-buffered
// in steps of half a super-block (rows of 128 B at a pitch of 144 B: 8 lanes' 16-byte reads fall in
// distinct banks). So do the weights, as they are in memory (loaded in whole rows, 5 KB a step):
// lane (column, k half) reads its column's 16-byte pieces and expands them to hi and lo codes right
// where the MFMA takes them, its column's header (scales, mins, d) in its own registers.
//
// What bounds it: the VALU's issue (about 200 operations per wavefront and half super-block beside 17
// MFMAs: the expansion, then 5 operations per output and super-block; the matrix cores are busy 38 % of the
// cycles at two wavefronts per SIMD). Measured, the GEMM alone
// at Q4_K 1999 x 14336 x 4096: 435 us with the sub-block scales applied on the VALU (an integer
// multiply-add per output and 32 values), 340 us as here; 33 x 4096 x 14336 (KG = 8): 133 -> 21 us.
#include "gcq_common.h"

namespace gcq {

int cu_count();

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));

// LDS row pitches (bytes) of half a super-block's codes, low bits and high bits: 8 lanes' 16-byte reads
// of consecutive rows fall in distinct banks.
constexpr int KP = 128 + 16, WP = 64 + 16, QP = 32 + 16;

template <int TYPE>
struct Kq {
    static constexpr bool MIN = TYPE != T_Q6_K;   // a min term (Q4_K / Q5_K)
    static constexpr bool BIAS = TYPE == T_Q5_K;  // operand bytes taken minus 128
    static constexpr int QH = TYPE == T_Q6_K ? 64 : 32;  // high-bit bytes per super-block
};

struct KqArgs {
    const uint8_t * w;      // packed weight's low bits: [N][nsb][128] (nibbles / Q6_K's ql)
    const uint16_t * wd;    // Q6_K: fp16 d [N][nsb]
    const uint8_t * wqh;    // Q5_K: the fifth bits [N][nsb][32]; Q6_K: qh [N][nsb][64]
    const uint8_t * whdr;   // Q4_K / Q5_K: the headers (d, dmin, scales[12]) [N][nsb][16]; Q6_K: scales[16]
    const int8_t * xc;      // Q8_K codes [M][K]
    const int16_t * xbs;    // block sums [M][K / 16]
    const float * xd;       // d [M][K / 256]
    float * y;
    const float * res;
    int32_t * raw;          // RAW: the integer parts of super-block raw_sb, [M][N][2] (Q6_K: [M][N][1])
    int M, N, nsb, ldy, raw_sb;
};

// A step's share of a thread between its global loads and its LDS store (thread t of the K group's NT).
template <int AP>
struct KqStage {
    v4i a[AP];         // activation codes, 16-byte pieces t + NT i: row / 8, part % 8
    v4i e;             // first half: row t / PR, 8 of its 16 block sums (int16)
    float dx;          // and its d
    v4i b[2], q;       // weight columns: 16-byte pieces of low bits (t + NT i: column / 4, part % 4), of high bits (t: column / 2, part % 2)
};
// The header of a lane's column (Q6_K: its scales and d).
struct KqHead {
    v4i h;
    uint32_t d;
};

__device__ __forceinline__ uint32_t u32(int x) { return (uint32_t) x; }

// One K group's codes and weight bytes of a step; activation scales of a super-block.
template <int TYPE, int XT, int WN>
struct KqCodes {
    int8_t a[32 * XT * KP];
    uint8_t b[32 * WN * WP];
    uint8_t q[TYPE == T_Q4_K ? 16 : 32 * WN * QP];
};
template <int TYPE, int XT>
struct KqScales {
    float dx[32 * XT];
    int t128[Kq<TYPE>::BIAS ? 32 * XT : 4];  // 128 times the row's code sum
    // the block sum of sub-block j as two f16 values: [row][j] its multiple of 64, [row][8 + j] the rest
    __align__(16) _Float16 bs[Kq<TYPE>::MIN ? 32 * XT : 1][16];
};

template <int TYPE, int XT, int WN, int AP>
__device__ __forceinline__ void kq_store(const KqStage<AP> & st, KqCodes<TYPE, XT, WN> & L, KqScales<TYPE, XT> & S, int t,
                                         int h) {
    constexpr int NT = 64 * WN, PR = NT / (32 * XT);
#pragma unroll
    for (int i = 0; i < AP; i++) {
        const int p = t + NT * i;
        *reinterpret_cast<v4i *>(L.a + (p >> 3) * KP + 16 * (p & 7)) = st.a[i];
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int p = t + NT * i;
        *reinterpret_cast<v4i *>(L.b + (p >> 2) * WP + 16 * (p & 3)) = st.b[i];
    }
    if constexpr (TYPE != T_Q4_K) *reinterpret_cast<v4i *>(L.q + (t >> 1) * QP + 16 * (t & 1)) = st.q;
    if (h != 0) return;
    const int row = t / PR, part = t % PR;
    if constexpr (Kq<TYPE>::MIN) {
        int total = 0;
        h4_t hi, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // bsums 2j and 2j + 1: the two int16 halves of word j
            const int bs = (int) (int16_t) (st.e[j] & 0xffff) + (st.e[j] >> 16);  // |bs| <= 32 * 128
            total += bs;
            hi[j] = (_Float16) (float) (bs & ~63);
            lo[j] = (_Float16) (float) (bs & 63);
        }
        if constexpr (Kq<TYPE>::BIAS) total += __shfl_xor(total, 1, 64);
        if (part < 2) {
            *reinterpret_cast<h4_t *>(&S.bs[row][4 * part]) = hi;
            *reinterpret_cast<h4_t *>(&S.bs[row][8 + 4 * part]) = lo;
        }
        if constexpr (Kq<TYPE>::BIAS)
            if (part == 0) S.t128[row] = 128 * total;
    }
    if (part == 0) S.dx[row] = st.dx;
}

// Four bytes times a scale below 8 (no carry between bytes: bytes <= 31).
__device__ __forceinline__ uint32_t bytes_times(uint32_t q, uint32_t s2) {
    return __builtin_bit_cast(uint32_t, (u16x2) (__builtin_bit_cast(u16x2, q) * __builtin_bit_cast(u16x2, s2)));
}

// Q6_K: hi and lo codes of four values q (bytes, 0..63) of scale sc.
__device__ __forceinline__ void q6_hi_lo(uint32_t q, int sc, uint32_t & hi, uint32_t & lo) {
    const i16x2 s = {(int16_t) sc, (int16_t) sc}, o = s * (int16_t) -32;
    const i16x2 e = __builtin_bit_cast(i16x2, q & 0x00FF00FFu) * s + o;
    const i16x2 d = __builtin_bit_cast(i16x2, (q >> 8) & 0x00FF00FFu) * s + o;
    lo = (__builtin_bit_cast(uint32_t, e) & 0x003F003Fu) | ((__builtin_bit_cast(uint32_t, d) & 0x003F003Fu) << 8);
    const uint32_t he = __builtin_bit_cast(uint32_t, (i16x2) (e >> 6)), ho = __builtin_bit_cast(uint32_t, (i16x2) (d >> 6));
    hi = __builtin_amdgcn_perm(ho, he, 0x06020400u);
}

// The hi and lo operands of piece i of half h for this lane (k half lk of its column): from the low
// nibbles (o[0], o[1]) and the high ones (o[2], o[3]).
template <int TYPE>
__device__ __forceinline__ void kq_expand(const v4i & b, const v4i & q, const KqHead & hd, int h, int i, int lk, v4i (&o)[4]) {
    if constexpr (TYPE == T_Q6_K) {
        // the low nibbles are values 32 i + 16 lk .. of the half, the high ones those 64 on; their
        // 16-value sub-blocks 8 h + 2 i + lk and 8 h + 4 + 2 i + lk
        const int sc0 = (int) (int8_t) (hd.h[2 * h] >> (16 * i + 8 * lk)), sc1 = (int) (int8_t) (hd.h[2 * h + 1] >> (16 * i + 8 * lk));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t x = u32(b[e]), hq = u32(q[e]) >> (2 * i);
            uint32_t hi, lo;
            q6_hi_lo((x & 0x0F0F0F0Fu) | ((hq & 0x03030303u) << 4), sc0, hi, lo);
            o[0][e] = (int) hi, o[1][e] = (int) lo;
            q6_hi_lo(((x >> 4) & 0x0F0F0F0Fu) | (hq & 0x30303030u), sc1, hi, lo);
            o[2][e] = (int) hi, o[3][e] = (int) lo;
        }
    } else {
        // the low nibbles are values 16 lk .. of sub-block 4 h + 2 i, the high ones of the next; 6-bit scales
        // (get_scale_min_k4): bytes 0..3 of the 12 for j < 4, else byte 4 + j's low nibble and byte j - 4's top bits
        uint32_t sc0, sc1;
        const uint32_t q0 = u32(hd.h[1]) >> (16 * i), q2 = u32(hd.h[3]) >> (16 * i);
        if (h == 0) {
            sc0 = q0 & 63;
            sc1 = (q0 >> 8) & 63;
        } else {
            sc0 = (q2 & 15) | ((q0 >> 2) & 0x30);
            sc1 = ((q2 >> 8) & 15) | ((q0 >> 10) & 0x30);
        }
        const uint32_t sh0 = (sc0 >> 3) * 0x10001u, sl0 = (sc0 & 7) * 0x10001u;
        const uint32_t sh1 = (sc1 >> 3) * 0x10001u, sl1 = (sc1 & 7) * 0x10001u;
        constexpr uint32_t bias = Kq<TYPE>::BIAS ? 0x80808080u : 0u;  // p ^ 0x80 as int8 is p - 128
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t x = u32(b[e]);
            uint32_t v0 = x & 0x0F0F0F0Fu, v1 = (x >> 4) & 0x0F0F0F0Fu;
            if constexpr (TYPE == T_Q5_K) {
                const uint32_t hq = u32(q[e]) >> (4 * h + 2 * i);
                v0 |= (hq & 0x01010101u) << 4;
                v1 |= (hq & 0x02020202u) << 3;
            }
            o[0][e] = (int) (bytes_times(v0, sh0) ^ bias);
            o[1][e] = (int) (bytes_times(v0, sl0) ^ bias);
            o[2][e] = (int) (bytes_times(v1, sh1) ^ bias);
            o[3][e] = (int) (bytes_times(v1, sl1) ^ bias);
        }
    }
}

// 8 unsigned bytes as f16: byte b under the exponent of 1024 is the f16 1024 + b.
__device__ __forceinline__ h8_t bytes_to_h8(uint32_t b0, uint32_t b1) {
    h8_t o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const h2_t h = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, i < 2 ? b0 : b1, i & 1 ? 0x04030402u : 0x04010400u));
        o[2 * i] = h.x - (_Float16) 1024.0f;
        o[2 * i + 1] = h.y - (_Float16) 1024.0f;
    }
    return o;
}

template <int TYPE, int XT, int WN, int KG, bool RAW, class Sum = float>
__global__ __launch_bounds__(64 * WN * KG, 2) void k_gemm_kq(const KqArgs a) {
    constexpr int TM = 32 * XT, TN = 32 * WN, NT = 64 * WN, AP = 4 * XT / WN;
    constexpr int SHIFT = TYPE == T_Q6_K ? 6 : 3;
    constexpr int GM = 8;  // row tiles per group of tiles
    struct Lds {
        KqCodes<TYPE, XT, WN> c[2];
        KqScales<TYPE, XT> s[2];
    };
    constexpr size_t kRed = KG > 1 ? (size_t) (KG - 1) * WN * XT * 1024 * sizeof(Sum) : 0;  // the groups' sums
    constexpr size_t kLds = sizeof(Lds) * KG > kRed ? sizeof(Lds) * KG : kRed;
    __shared__ __align__(16) uint8_t lds[kLds];
    const int mt = (a.M + TM - 1) / TM, nt = (a.N + TN - 1) / TN, total = mt * nt;
    // XCD x holds a contiguous run of tiles; in it, GM row tiles by as many columns as run together, so that
    // their rows and columns stay in its L2
    int id = blockIdx.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    const int g0 = id / (GM * nt) * GM, gm = min(GM, mt - g0), in = id - g0 * nt;
    const int m0 = (g0 + in % gm) * TM, n0 = in / gm * TN;
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int kg = wave / WN, t = threadIdx.x - kg * NT;
    const int lr = lane & 31, lk = lane >> 5;
    const int nw = (wave % WN) * 32, n = n0 + nw + lr;  // this wavefront's columns, this lane's
    Lds & L = reinterpret_cast<Lds *>(lds)[kg];

    // Where this thread reads. Rows past M or N read the last row (never stored).
    const int8_t * pa[AP];
#pragma unroll
    for (int i = 0; i < AP; i++) {
        const int p = t + NT * i;
        pa[i] = a.xc + (size_t) min(m0 + (p >> 3), a.M - 1) * a.nsb * 256 + 16 * (p & 7);
    }
    constexpr int PR = NT / TM;
    const size_t mi = (size_t) min(m0 + t / PR, a.M - 1) * a.nsb;
    const uint8_t * pb[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int p = t + NT * i;
        pb[i] = a.w + (size_t) min(n0 + (p >> 2), a.N - 1) * a.nsb * 128 + 16 * (p & 3);
    }
    const uint8_t * pq = TYPE == T_Q4_K ? nullptr : a.wqh + (size_t) min(n0 + (t >> 1), a.N - 1) * a.nsb * Kq<TYPE>::QH + 16 * (t & 1);
    const size_t bi = (size_t) min(n, a.N - 1) * a.nsb;
    const auto load = [&](KqStage<AP> & s, int sb, int h) {
#pragma unroll
        for (int i = 0; i < AP; i++) s.a[i] = *reinterpret_cast<const v4i *>(pa[i] + (size_t) sb * 256 + 128 * h);
#pragma unroll
        for (int i = 0; i < 2; i++) s.b[i] = *reinterpret_cast<const v4i *>(pb[i] + (size_t) sb * 128 + 64 * h);
        if constexpr (TYPE == T_Q5_K) s.q = *reinterpret_cast<const v4i *>(pq + (size_t) sb * 32);
        if constexpr (TYPE == T_Q6_K) s.q = *reinterpret_cast<const v4i *>(pq + (size_t) sb * 64 + 32 * h);
        if (h == 0) {
            s.dx = a.xd[mi + sb];
            if constexpr (Kq<TYPE>::MIN) s.e = *reinterpret_cast<const v4i *>(a.xbs + (mi + sb) * 16 + 8 * (t & 1));
        }
    };
    const auto load_head = [&](KqHead & hd, int sb) {
        hd.h = *reinterpret_cast<const v4i *>(a.whdr + (bi + sb) * 16);
        if constexpr (TYPE == T_Q6_K) hd.d = a.wd[bi + sb];
    };

    Sum acc[XT][16]{};
    v16i ih[XT], il[XT];

    // This group's super-blocks: the same number of rounds for every group (barriers), a round past the
    // end computing nothing. Loads past the end read the last super-block again: a load under a
    // condition makes the compiler wait for every load in flight where the paths meet.
    const int sb_begin = RAW ? a.raw_sb : min(kg, a.nsb - 1), sb_end = RAW ? a.raw_sb + 1 : a.nsb;
    const int rounds = RAW ? 1 : (a.nsb + KG - 1) / KG;
    KqStage<AP> st;
    KqHead hd, hn;
    load(st, sb_begin, 0);
    load_head(hd, sb_begin);
    kq_store<TYPE, XT, WN>(st, L.c[0], L.s[0], t, 0);
    load(st, sb_begin, 1);
    __syncthreads();

    for (int it = 0; it < rounds; it++) {
        const int sb = RAW ? a.raw_sb : min(kg + it * KG, sb_end - 1), next = min(sb + KG, sb_end - 1), sc = it & 1;
        const bool on = KG == 1 || kg + it * KG < sb_end;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // the next step into the other buffer, the loads of the step after
            kq_store<TYPE, XT, WN>(st, L.c[h ^ 1], L.s[sc ^ h], t, h ^ 1);
            load(st, next, h);
            if (h == 1) load_head(hn, next);
            if (on) {
                const KqScales<TYPE, XT> & s = L.s[sc];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    v4i o[4], q{};
                    if constexpr (TYPE == T_Q5_K || TYPE == T_Q6_K) q = *reinterpret_cast<const v4i *>(L.c[h].q + (nw + lr) * QP + 16 * lk);
                    kq_expand<TYPE>(*reinterpret_cast<const v4i *>(L.c[h].b + (nw + lr) * WP + 32 * i + 16 * lk), q, hd, h, i, lk, o);
#pragma unroll
                    for (int e = 0; e < 2; e++) {  // low nibbles, high nibbles: 32 values each
                        const int k0 = TYPE == T_Q6_K ? 32 * i + 64 * e : 64 * i + 32 * e;
#pragma unroll
                        for (int x = 0; x < XT; x++) {
                            const v4i af = *reinterpret_cast<const v4i *>(L.c[h].a + (x * 32 + lr) * KP + k0 + 16 * lk);
                            const bool first = h == 0 && i == 0 && e == 0;
                            v16i init{};
                            if constexpr (Kq<TYPE>::BIAS)
                                if (first) {
#pragma unroll
                                    for (int q = 0; q < 4; q++) {
                                        const v4i t4 = *reinterpret_cast<const v4i *>(&s.t128[x * 32 + 8 * q + 4 * lk]);
#pragma unroll
                                        for (int r = 0; r < 4; r++) init[4 * q + r] = t4[r];
                                    }
                                }
                            ih[x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, o[2 * e], first ? init : ih[x], 0, 0, 0);
                            il[x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, o[2 * e + 1], first ? init : il[x], 0, 0, 0);
                        }
                    }
                }
                if (h == 1) {  // the super-block is complete: its integer parts into the f32 sums
                    h8_t bm{};
                    float dw, dm = 0.0f;
                    if constexpr (Kq<TYPE>::MIN) {
                        dw = h2f((uint16_t) (u32(hd.h[0]) & 0xffffu));
                        dm = h2f((uint16_t) (u32(hd.h[0]) >> 16));
                        asm volatile("" : "+v"(dm));  // an f32 register: from f16 the multiply-adds take the mixed form, half the rate
                        // mins: bytes 4..7 (6 bits) of the 12; then byte 8 + j's high nibble with byte 4 + j's top two bits
                        const uint32_t q1 = u32(hd.h[2]), q2 = u32(hd.h[3]);
                        bm = bytes_to_h8(q1 & 0x3F3F3F3Fu, ((q2 >> 4) & 0x0F0F0F0Fu) | ((q1 >> 2) & 0x30303030u));
                    } else {
                        dw = h2f((uint16_t) hd.d);
                    }
#pragma unroll
                    for (int x = 0; x < XT; x++) {
                        // I2 = sum_j m_j(n) bs_j(m): lanes 0..31 the multiples of 64, lanes 32..63 the rest
                        v16f i2{};
                        if constexpr (Kq<TYPE>::MIN) {
                            const h8_t as = *reinterpret_cast<const h8_t *>(&s.bs[x * 32 + lr][8 * lk]);
                            i2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(as, bm, v16f{}, 0, 0, 0);
                        }
                        if constexpr (RAW) {  // the one super-block's integers, stored here
#pragma unroll
                            for (int r = 0; r < 16; r++) {
                                const int m = m0 + x * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
                                if (m >= a.M || n >= a.N) continue;
                                int32_t * out = a.raw + ((size_t) m * a.N + n) * (Kq<TYPE>::MIN ? 2 : 1);
                                out[0] = (ih[x][r] << SHIFT) + il[x][r];
                                if constexpr (Kq<TYPE>::MIN) out[1] = (int) i2[r];
                            }
                        } else {
#pragma unroll
                            for (int q = 0; q < 4; q++) {
                                // d_x of this lane's rows: element 4 q + r is row 8 q + 4 lk + r of the MFMA tile
                                const float4 d4 = *reinterpret_cast<const float4 *>(&s.dx[x * 32 + 8 * q + 4 * lk]);
                                const float dx[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                                for (int r = 0; r < 4; r++) {
                                    const int e = 4 * q + r;
                                    float v = dw * (float) ((ih[x][e] << SHIFT) + il[x][e]);
                                    if constexpr (Kq<TYPE>::MIN) v = fmaf(-dm, i2[e], v);
                                    acc[x][e] = __builtin_elementwise_fma((Sum) dx[r], (Sum) v, acc[x][e]);
                                }
                            }
                        }
                    }
                }
            }
            if (h == 1) hd = hn;
            __syncthreads();
        }
    }
    if constexpr (RAW) return;

    if constexpr (KG > 1) {  // groups 1.. hand their sums to group 0, which adds them in pairs
        static_assert((KG & (KG - 1)) == 0, "pairs of groups");
        constexpr int RS = WN * XT * 1024;
        Sum * red = reinterpret_cast<Sum *>(lds) + (size_t) (wave % WN) * XT * 1024 + lane;
        if (kg > 0) {
#pragma unroll
            for (int x = 0; x < XT; x++)
#pragma unroll
                for (int r = 0; r < 16; r++) red[(size_t) (kg - 1) * RS + x * 1024 + r * 64] = acc[x][r];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int x = 0; x < XT; x++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                Sum v[KG];
                v[0] = acc[x][r];
#pragma unroll
                for (int g = 1; g < KG; g++) v[g] = red[(size_t) (g - 1) * RS + x * 1024 + r * 64];
#pragma unroll
                for (int o = 1; o < KG; o <<= 1)
#pragma unroll
                    for (int g = 0; g < KG; g += 2 * o) v[g] += v[g + o];
                acc[x][r] = v[0];
            }
    }
    if (n >= a.N) return;
#pragma unroll
    for (int x = 0; x < XT; x++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = m0 + x * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
            if (m >= a.M) continue;
            const size_t o = (size_t) m * a.ldy + n;
            const float v = (float) acc[x][r];
            a.y[o] = a.res ? v + a.res[o] : v;
        }
}

template <int TYPE, bool RAW>
void run_kq(const void * wv, int64_t N, int64_t K, const void * act, int64_t M, float * y, int64_t ldy,
            const float * res, int32_t * raw, int raw_sb, hipStream_t s) {
    const WeightLayout WL = weight_layout(TYPE, N, K);
    const ActLayout AL = act_layout(TYPE, M, K);
    const uint8_t * w = (const uint8_t *) wv;
    const uint8_t * x = (const uint8_t *) act;
    KqArgs a{};
    a.w = w + WL.qs;
    a.wd = TYPE == T_Q6_K ? (const uint16_t *) (w + WL.d) : nullptr;
    a.wqh = TYPE == T_Q4_K ? nullptr : w + WL.qh;
    a.whdr = TYPE == T_Q6_K ? w + WL.sc : w + WL.d;
    a.xc = (const int8_t *) (x + AL.codes);
    a.xbs = (const int16_t *) (x + AL.meta);
    a.xd = (const float *) (x + AL.d);
    a.y = y;
    a.res = res;
    a.raw = raw;
    a.M = (int) M;
    a.N = (int) N;
    a.nsb = (int) (K / 256);
    a.ldy = (int) ldy;
    a.raw_sb = raw_sb;
    const auto tiles = [&](int64_t tm, int64_t tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
    // 64 x 128 tiles where they fill the chip; else 64 x 64 in two K groups; where 32 x 32 tiles are few, those in
    // eight. Each K group needs super-blocks: one or two, and most groups only wait; below eight, 64 x 128 tiles are worth
    // half as many of them and 32 x 32 tiles only one per CU. Kernel times, Q4_K, us for 64 x 128 / 64 x 64 / 32 x 32 tiles:
    // 512 x 4096 x 14336 115 / 92 / 164; 128 x 4096 x 4096 32 / 21 / 19; 128 x 4096 x 256 6.2 / 7.1 / 11.2; 256 x 2048 x 512
    // 8.2 / 7.3 / 11.7; 65 x 4096 x 1024 11.3 / 8.9 / 11.3; 33 x 4096 x 1024 10.9 / 8.3 / 6.9.
    // The groups' sums must be no further from 64 bits than one f32 chain over K. Eight sums of a super-block or two
    // added one by one were 1.12 times as far (Q6_K, K 2048); in pairs they are not from eight super-blocks on, below that the
    // 32 x 32 tiles sum in f64 (5-10 % of their time), and 64 x 64 tiles start at four.
    if constexpr (RAW) {
        k_gemm_kq<TYPE, 2, 4, 1, RAW><<<(unsigned) tiles(64, 128), 256, 0, s>>>(a);
    } else {
        const int64_t cus = cu_count();
        const bool few = a.nsb < 8;
        if (a.nsb > 2 && tiles(64, 128) <= (few ? cus / 2 : cus) && tiles(32, 32) <= (few ? cus : 2 * cus)) {
            if (few) k_gemm_kq<TYPE, 1, 1, 8, RAW, double><<<(unsigned) tiles(32, 32), 512, 0, s>>>(a);
            else k_gemm_kq<TYPE, 1, 1, 8, RAW><<<(unsigned) tiles(32, 32), 512, 0, s>>>(a);
        } else if (a.nsb > 3 && tiles(64, 128) <= (few ? cus / 2 : cus)) {
            k_gemm_kq<TYPE, 2, 2, 2, RAW><<<(unsigned) tiles(64, 64), 256, 0, s>>>(a);
        } else {
            k_gemm_kq<TYPE, 2, 4, 1, RAW><<<(unsigned) tiles(64, 128), 256, 0, s>>>(a);
        }
    }
}

}  // namespace

bool gemm_kq_fits(int type, int64_t K) { return is_kquant(type) && K > 0 && K % 256 == 0; }

// ggml_mul_mat of a packed K-quant weight [N][K] with M > 8 Q8_K activation rows (gcq_act_size's
// layout): y[m * ldy + n] (+ res).
void launch_gemm_kq(int type, const void * w, int64_t N, int64_t K, const void * act, int64_t M, float * y, int64_t ldy,
                    hipStream_t s, const float * res) {
    require(gemm_kq_fits(type, K), "gemm kq: K-quant weight and K a multiple of 256");
    require(N > 0 && M > 0 && N < INT32_MAX && M < INT32_MAX && ldy < INT32_MAX, "gemm kq: sizes");
    if (type == T_Q4_K) run_kq<T_Q4_K, false>(w, N, K, act, M, y, ldy, res, nullptr, 0, s);
    else if (type == T_Q5_K) run_kq<T_Q5_K, false>(w, N, K, act, M, y, ldy, res, nullptr, 0, s);
    else run_kq<T_Q6_K, false>(w, N, K, act, M, y, ldy, res, nullptr, 0, s);
    check_launch("gemm kq");
}

// The integer parts of super-block sb: out[(m N + n) 2 + {0, 1}] = {I1, I2} (Q4_K / Q5_K), or
// out[m N + n] = I1 (Q6_K).
void launch_gemm_kq_isums(int type, const void * w, int64_t N, int64_t K, const void * act, int64_t M, int sb,
                          int32_t * out, hipStream_t s) {
    require(gemm_kq_fits(type, K) && sb >= 0 && sb < K / 256, "gemm kq isums: K-quant weight, super-block in range");
    require(N > 0 && M > 0 && N < INT32_MAX && M < INT32_MAX, "gemm kq isums: sizes");
    if (type == T_Q4_K) run_kq<T_Q4_K, true>(w, N, K, act, M, nullptr, 0, nullptr, out, sb, s);
    else if (type == T_Q5_K) run_kq<T_Q5_K, true>(w, N, K, act, M, nullptr, 0, nullptr, out, sb, s);
    else run_kq<T_Q6_K, true>(w, N, K, act, M, nullptr, 0, nullptr, out, sb, s);
    check_launch("gemm kq isums");
}

}  // namespace gcq
