// gemm.hip - quantized mat-mul for prefill (M > 8 activation rows) on int8 MFMA.
//
// Replaces ggml_mul_mat of a Q8_0 / Q4_0 weight with an f32 src1 of many rows
// (runtime/src/ops.cpp:107-119). As ggml, src1 is quantized to Q8_0 per 32 values (quant.hip);
// then out[m, n] = sum_blk d_x[m, blk] * d_w[n, blk] * isum(m, n, blk) with isum the exact int32
// dot of one 32-value block.
//
// gfx950's v_mfma_i32_32x32x32_i8 has a depth of exactly one quant block, so every MFMA yields
// the 32x32 tile of block sums isum(., ., blk) exactly; the fp16-scale epilogue folds it into fp32
// accumulators (d_w and d_x from LDS). Workgroup tile 128 (m) x 128 (n), 4 wavefronts of 64x64
// (2x2 MFMA tiles); two LDS stages of 2 K-blocks each of A (activation codes) and B (weight codes,
// Q4_0 nibbles expanded to signed int8 q-8), with a 16-byte row pad against bank conflicts. Tiles
// are numbered so that the workgroups sharing one weight tile land on the same XCD (and L2).
//
// Where 128 x 128 tiles are too few for the chip, two K groups of 4 wavefronts share one, or (fewer still) the
// wavefronts of 32 x 32 tiles share K (k_gemm_kg, the rule in run_gemm).
//
// The per-block epilogue (2 VALU operations per output element per K-block of 32, against one
// 32-deep MFMA step) bounds this kernel: ggml's semantics put a scale on every block, so the block
// sums cannot stay in the int32 accumulator. With a conversion as a third operation Q8_0 512 x 14336
// x 4096 took 114.8 us with the activation's quantization; taken out by the start value below, 104.0 us.
#include "gcq_common.h"

namespace gcq {

int cu_count();

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int GBM = 128, GBN = 128;  // workgroup tile
constexpr int GKB = 2;               // K-blocks (of 32) per LDS stage
constexpr int GPITCH = GKB * 32 + 16;  // LDS row pitch in bytes (16 B pad against bank conflicts)

// The MFMAs start from the bits of 1.5 * 2^23 instead of 0, so an int32 block sum (|isum| < 2^22) comes
// out as the bits of the float 1.5 * 2^23 + isum: no conversion. d_w is an fp16 value, so
// fma(that, d_w, -1.5 * 2^23 d_w) has an exact product and an exact constant: one rounding, of
// isum * d_w, the same float that converting and multiplying gives.
constexpr int kMagicBits = 0x4B400000;
constexpr float kMagic = 12582912.0f;

__device__ __forceinline__ uint32_t q4_to_s8(uint32_t w) {  // 4 nibbles (0..15) -> 4 int8 (q - 8)
    return (((w & 0x0F0F0F0Fu) | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
}

// One LDS stage's worth of global data held in registers between its load and its LDS store.
// A stage is GKB K-blocks of the workgroup's 128 activation rows and 128 weight rows.
constexpr int GA = GBM * GKB * 2 / 256;  // 16-byte activation chunks per thread (two per row-block)
constexpr int GS = GBM * GKB / 256;      // row-blocks per thread for the scales and Q4_0 nibbles
static_assert(GA >= 1 && GS >= 1, "stage size");

// Native vector types, not HIP's int4 / uint4 structs: struct copies become memcpys through a
// stack object that is not promoted to registers, which puts the staged loads in scratch memory
// and makes every chunk wait for its global loads before computing.
template <int TYPE>
struct GemmStage {
    v4i a[GA];                                // activation codes
    v4i b[TYPE == T_Q8_0 ? GA : GS];          // weight codes: Q8_0 like a, Q4_0 one block's 16 B of nibbles
    float dx[GS];                             // activation scales
    uint32_t dw[GS];                          // weight scales (fp16 bits)
};

// Chunk c (K-blocks kb0 .. kb0 + GKB) of this workgroup's tile: thread t's share. Rows past M or
// N reload the last row; blocks past nb reload the last block (never used).
template <int TYPE>
__device__ __forceinline__ void gemm_load(GemmStage<TYPE> & st, const uint8_t * __restrict__ wqs,
                                          const uint16_t * __restrict__ wd, const int8_t * __restrict__ xc,
                                          const float2 * __restrict__ xm, int m0, int n0, int M, int N, int nb, int kb0) {
    const int t = threadIdx.x & 255;
    const int K = nb * 32;
#pragma unroll
    for (int i = 0; i < GA; i++) {  // A: 128 rows x GKB*32 B in chunks of 16 B
        const int c = t + 256 * i;
        const int row = c / (GKB * 2), part = c % (GKB * 2);
        const int gm = min(m0 + row, M - 1);
        const int kb = min(kb0 + part / 2, nb - 1);
        st.a[i] = *reinterpret_cast<const v4i *>(xc + (size_t) gm * K + (size_t) kb * 32 + (part & 1) * 16);
    }
    if constexpr (TYPE == T_Q8_0) {
#pragma unroll
        for (int i = 0; i < GA; i++) {
            const int c = t + 256 * i;
            const int row = c / (GKB * 2), part = c % (GKB * 2);
            const int gn = min(n0 + row, N - 1);
            const int kb = min(kb0 + part / 2, nb - 1);
            st.b[i] = *reinterpret_cast<const v4i *>(wqs + ((size_t) gn * nb + kb) * 32 + (part & 1) * 16);
        }
    } else {  // 128 rows x GKB blocks of 16 B
#pragma unroll
        for (int i = 0; i < GS; i++) {
            const int c = t + 256 * i;
            const int row = c / GKB, j = c % GKB;
            const int gn = min(n0 + row, N - 1);
            const int kb = min(kb0 + j, nb - 1);
            st.b[i] = *reinterpret_cast<const v4i *>(wqs + ((size_t) gn * nb + kb) * 16);
        }
    }
#pragma unroll
    for (int i = 0; i < GS; i++) {  // scales: 128 rows x GKB blocks each
        const int c = t + 256 * i;
        const int row = c / GKB, j = c % GKB;
        const int kb = min(kb0 + j, nb - 1);
        st.dx[i] = xm[(size_t) min(m0 + row, M - 1) * nb + kb].x;
        st.dw[i] = wd[(size_t) min(n0 + row, N - 1) * nb + kb];
    }
}

template <int TYPE>
__device__ __forceinline__ void gemm_store(const GemmStage<TYPE> & st, int8_t * sA, int8_t * sB, float * sdx,
                                           float * sdw) {
    const int t = threadIdx.x & 255;
#pragma unroll
    for (int i = 0; i < GA; i++) {
        const int c = t + 256 * i;
        const int row = c / (GKB * 2), part = c % (GKB * 2);
        *reinterpret_cast<v4i *>(sA + row * GPITCH + part * 16) = st.a[i];
    }
    if constexpr (TYPE == T_Q8_0) {
#pragma unroll
        for (int i = 0; i < GA; i++) {
            const int c = t + 256 * i;
            const int row = c / (GKB * 2), part = c % (GKB * 2);
            *reinterpret_cast<v4i *>(sB + row * GPITCH + part * 16) = st.b[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < GS; i++) {
            const int c = t + 256 * i;
            const int row = c / GKB, j = c % GKB;
            const v4i w = st.b[i];
            v4i lo, hi;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                lo[e] = (int) q4_to_s8((uint32_t) w[e]);
                hi[e] = (int) q4_to_s8((uint32_t) w[e] >> 4);
            }
            *reinterpret_cast<v4i *>(sB + row * GPITCH + j * 32) = lo;
            *reinterpret_cast<v4i *>(sB + row * GPITCH + j * 32 + 16) = hi;
        }
    }
#pragma unroll
    for (int i = 0; i < GS; i++) {
        const int c = t + 256 * i;
        const int row = c / GKB, j = c % GKB;
        sdx[j * GBM + row] = st.dx[i];
        sdw[j * GBN + row] = h2f((uint16_t) st.dw[i]);
    }
}

// RAW: write the int32 block sums of block `raw_blk` instead of the scaled result.
//
// Pipeline: chunk c + 1's global loads are issued into registers before chunk c is computed from
// LDS, then stored to the other LDS buffer; one barrier per chunk. Per K-block each wavefront
// issues its four 32x32x32 MFMAs, then folds each block sum into the fp32 accumulators as
// (isum * d_w) * d_x, the scales read from LDS once per block as vectors.
template <int TYPE, bool RAW, int KG>
__global__ __launch_bounds__(256 * KG) void k_gemm(const uint8_t * __restrict__ wqs, const uint16_t * __restrict__ wd,
                                              const int8_t * __restrict__ xc, const float2 * __restrict__ xm,
                                              float * y, const float * res, int32_t * __restrict__ yraw, int M, int N,
                                              int nb, int ldy, int raw_blk) {
    struct Lds {
        __align__(16) int8_t sA[2][GBM * GPITCH];
        __align__(16) int8_t sB[2][GBN * GPITCH];
        __align__(16) float sdx[2][GKB * GBM];
        __align__(16) float sdw[2][GKB * GBN];
    };
    __shared__ Lds lds[KG];
    static_assert(KG <= 2 && sizeof(Lds) * KG >= (KG - 1) * GBM * GBN * 4, "the second group's sums fit");
    const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 8) : 0;
    auto & [sA, sB, sdx, sdw] = lds[kg];

    // Tile numbering: ids id, id+8, ... run on one XCD; give each XCD a contiguous run of tiles,
    // m-tiles fastest, so the workgroups that read one weight tile share an L2.
    const int mt = (M + GBM - 1) / GBM, nt = (N + GBN - 1) / GBN;
    const int total = mt * nt;
    int id = blockIdx.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    const int m0 = (id % mt) * GBM, n0 = (id / mt) * GBN;

    const int tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
    const int wm = wave >> 1, wn = wave & 1;
    float acc[2][2][16];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;

    v16i magic;
#pragma unroll
    for (int r = 0; r < 16; r++) magic[r] = kMagicBits;
    asm volatile("" : "+v"(magic));  // kept in registers: known constants are written again before every block

    const int kb_begin = RAW ? raw_blk : 0;
    const int kb_end = RAW ? raw_blk + 1 : nb;
    const int nchunk = (kb_end - kb_begin + GKB - 1) / GKB;
    GemmStage<TYPE> st;
    const int rounds = (nchunk + KG - 1) / KG;  // the same for every group (barriers): a chunk past the end computes nothing
    gemm_load<TYPE>(st, wqs, wd, xc, xm, m0, n0, M, N, nb, kb_begin + kg * GKB);
    gemm_store<TYPE>(st, sA[0], sB[0], sdx[0], sdw[0]);
    __syncthreads();

    for (int c = 0; c < rounds; c++) {
        const int buf = c & 1;
        const int kb0 = kb_begin + (c * KG + kg) * GKB;
        if (c + 1 < rounds) gemm_load<TYPE>(st, wqs, wd, xc, xm, m0, n0, M, N, nb, kb0 + KG * GKB);
        const int nblk = min(GKB, kb_end - kb0);
#pragma unroll
        for (int j = 0; j < GKB; j++) {
            if (j >= nblk) break;
            v4i af[2], bf[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                af[t] = *reinterpret_cast<const v4i *>(sA[buf] + (wm * 64 + t * 32 + (lane & 31)) * GPITCH + j * 32 +
                                                       16 * (lane >> 5));
                bf[t] = *reinterpret_cast<const v4i *>(sB[buf] + (wn * 64 + t * 32 + (lane & 31)) * GPITCH + j * 32 +
                                                       16 * (lane >> 5));
            }
            v16i cc[2][2];
#pragma unroll
            for (int tm = 0; tm < 2; tm++)
#pragma unroll
                for (int tn = 0; tn < 2; tn++)
                    cc[tm][tn] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[tm], bf[tn], magic, 0, 0, 0);
            if constexpr (RAW) {
#pragma unroll
                for (int tm = 0; tm < 2; tm++)
#pragma unroll
                    for (int tn = 0; tn < 2; tn++)
#pragma unroll
                        for (int r = 0; r < 16; r++) acc[tm][tn][r] = __int_as_float(cc[tm][tn][r] - kMagicBits);
            } else {
                // d_x of this lane's rows: element r of tile tm is row wm*64 + tm*32 + 8*(r/4) + 4*(lane/32) + r%4
                float4 dx[2][4];
#pragma unroll
                for (int tm = 0; tm < 2; tm++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        dx[tm][q] = *reinterpret_cast<const float4 *>(sdx[buf] + j * GBM + wm * 64 + tm * 32 + q * 8 +
                                                                      (lane >> 5) * 4);
                float dwv[2], cw[2];
#pragma unroll
                for (int tn = 0; tn < 2; tn++) {
                    dwv[tn] = sdw[buf][j * GBN + wn * 64 + tn * 32 + (lane & 31)];
                    cw[tn] = -kMagic * dwv[tn];
                }
                if (__builtin_expect(__any(__builtin_isinf(dwv[0]) || __builtin_isinf(dwv[1])), 0)) {
                    // an infinite weight scale: isum * inf, which inf - inf would make a NaN
#pragma unroll
                    for (int tm = 0; tm < 2; tm++)
#pragma unroll
                        for (int tn = 0; tn < 2; tn++)
#pragma unroll
                            for (int r = 0; r < 16; r++)
                                cc[tm][tn][r] = __float_as_int(__int_as_float(cc[tm][tn][r]) - kMagic);
                    cw[0] = cw[1] = 0.0f;
                }
#pragma unroll
                for (int tm = 0; tm < 2; tm++)
#pragma unroll
                    for (int tn = 0; tn < 2; tn++)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            acc[tm][tn][4 * q + 0] = fmaf(fmaf(__int_as_float(cc[tm][tn][4 * q + 0]), dwv[tn], cw[tn]), dx[tm][q].x, acc[tm][tn][4 * q + 0]);
                            acc[tm][tn][4 * q + 1] = fmaf(fmaf(__int_as_float(cc[tm][tn][4 * q + 1]), dwv[tn], cw[tn]), dx[tm][q].y, acc[tm][tn][4 * q + 1]);
                            acc[tm][tn][4 * q + 2] = fmaf(fmaf(__int_as_float(cc[tm][tn][4 * q + 2]), dwv[tn], cw[tn]), dx[tm][q].z, acc[tm][tn][4 * q + 2]);
                            acc[tm][tn][4 * q + 3] = fmaf(fmaf(__int_as_float(cc[tm][tn][4 * q + 3]), dwv[tn], cw[tn]), dx[tm][q].w, acc[tm][tn][4 * q + 3]);
                        }
            }
        }
        if (c + 1 < rounds) gemm_store<TYPE>(st, sA[buf ^ 1], sB[buf ^ 1], sdx[buf ^ 1], sdw[buf ^ 1]);
        __syncthreads();
    }

    if constexpr (KG > 1) {  // the second group's sums to the first
        float * red = reinterpret_cast<float *>(lds) + tid;
        if (kg == 1) {
#pragma unroll
            for (int e = 0; e < 64; e++) red[e * 256] = acc[e >> 5][(e >> 4) & 1][e & 15];
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int e = 0; e < 64; e++) acc[e >> 5][(e >> 4) & 1][e & 15] += red[e * 256];
    }
#pragma unroll
    for (int tm = 0; tm < 2; tm++)
#pragma unroll
        for (int tn = 0; tn < 2; tn++) {
            const int n = n0 + wn * 64 + tn * 32 + (lane & 31);
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = m0 + wm * 64 + tm * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (m >= M) continue;
                if constexpr (RAW) yraw[(size_t) m * N + n] = __float_as_int(acc[tm][tn][r]);
                else {
                    const size_t o = (size_t) m * ldy + n;
                    y[o] = res ? acc[tm][tn][r] + res[o] : acc[tm][tn][r];
                }
            }
        }
}

// The first block that a step of n blocks from kb0 reads: no block past the last is read, the step starts
// earlier instead, and the blocks that are not its own (gemm_own) get zero scales.
__device__ __forceinline__ int gemm_base(int kb0, int n, int nb) { return max(min(kb0, nb - n), 0); }
__device__ __forceinline__ bool gemm_own(int j, int base, int kb0, int nb) { return base + j >= kb0 && base + j < nb; }

// Few tiles (short prompts, narrow outputs): a workgroup takes one tile of 32 x 32 and its KG wavefronts share
// K instead of the tile. Wavefront g takes the steps g, g + KG, .. of S K-blocks through LDS of its own (its
// DS operations are in order, so the loop has no barrier), the next step's global loads in flight; the sums meet
// in LDS at the end. Bound: the latency of a step (load, LDS, MFMA, epilogue) when the tiles are few, hidden by
// more wavefronts; with many tiles, LDS reads: a 32 x 32 tile reads d_x from LDS once per MFMA, a 64 x 64
// wavefront tile (k_gemm) once per two. 64 x 32 and 32 x 64 wavefront tiles measured the same or slower (fewer
// wavefronts); 64 x 64 spills. Q4_0, 33 x 4096 x 14336: 236 us in k_gemm, 24 here (KG = 8); 128 x 4096 x 4096:
// 72 -> 15 (KG = 4).
template <int TYPE, int S, int KG>
__global__ __launch_bounds__(64 * KG, 2) void k_gemm_kg(const uint8_t * __restrict__ wqs, const uint16_t * __restrict__ wd,
                                                        const int8_t * __restrict__ xc, const float2 * __restrict__ xm,
                                                        float * y, const float * res, int M, int N, int nb, int ldy) {
    constexpr int P = S * 32 + 16;
    constexpr int AP = S, BP = TYPE == T_Q8_0 ? S : S / 2;  // 16-byte pieces per lane
    constexpr int SP = S / 2;                               // scales per lane, of each operand
    constexpr int BS = TYPE == T_Q8_0 ? 32 : 16;            // code bytes per block
    constexpr int BR = S * BS / 16;                         // 16-byte weight pieces per row
    struct Lds {
        __align__(16) int8_t a[32 * P];
        __align__(16) int8_t b[32 * P];
        __align__(16) float dx[S * 32];
        __align__(16) float dw[S * 32];
    };
    constexpr int REGS = 16;
    constexpr size_t kRed = (size_t) KG * REGS * 64 * 4;
    __shared__ __align__(16) uint8_t lds[sizeof(Lds) * KG > kRed ? sizeof(Lds) * KG : kRed];

    const int mt = (M + 31) / 32, nt = (N + 31) / 32, total = mt * nt;
    const int xcd = blockIdx.x % 8;  // each XCD a contiguous run of tiles, m-tiles fastest (a weight tile's readers share an L2)
    const int id = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
    const int m0 = (id % mt) * 32, n0 = (id / mt) * 32;
    const int g = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lr = lane & 31, lk = lane >> 5;
    Lds & L = reinterpret_cast<Lds *>(lds)[g];

    // Offsets of this lane's pieces from the tile's first row (rows past M or N read the last row, never stored).
    uint32_t oa[AP], ob[BP], ox[SP], ow[SP];
    const uint32_t K = (uint32_t) nb * 32;
#pragma unroll
    for (int i = 0; i < AP; i++) {
        const int c = lane + 64 * i;
        oa[i] = (uint32_t) min(c / (2 * S), M - 1 - m0) * K + 32u * min(c / 2 % S, nb - 1) + 16u * (c & 1);
    }
#pragma unroll
    for (int i = 0; i < BP; i++) {
        const int c = lane + 64 * i;
        ob[i] = (uint32_t) min(c / BR, N - 1 - n0) * (uint32_t) (nb * BS) + (TYPE == T_Q8_0 ? 32u * min(c / 2 % S, nb - 1) + 16u * (c & 1) : 16u * min(c % S, nb - 1));
    }
#pragma unroll
    for (int i = 0; i < SP; i++) {
        const int c = lane + 64 * i;
        const uint32_t j = (uint32_t) min(c % S, nb - 1);
        ox[i] = (uint32_t) min(c / S, M - 1 - m0) * (uint32_t) nb + j;
        ow[i] = (uint32_t) min(c / S, N - 1 - n0) * (uint32_t) nb + j;
    }
    const int8_t * pa = xc + (size_t) m0 * K;
    const uint8_t * pb = wqs + (size_t) n0 * nb * BS;
    const float2 * px = xm + (size_t) m0 * nb;
    const uint16_t * pw = wd + (size_t) n0 * nb;

    v4i ra[AP], rb[BP];
    float rx[SP];
    uint32_t rw[SP];
    const auto load = [&](int step) {
        const int kb = gemm_base(step * S, S, nb);
#pragma unroll
        for (int i = 0; i < AP; i++) ra[i] = *reinterpret_cast<const v4i *>(pa + (size_t) kb * 32 + oa[i]);
#pragma unroll
        for (int i = 0; i < BP; i++) rb[i] = *reinterpret_cast<const v4i *>(pb + (size_t) kb * BS + ob[i]);
#pragma unroll
        for (int i = 0; i < SP; i++) {
            rx[i] = (px + kb)[ox[i]].x;
            rw[i] = (pw + kb)[ow[i]];
        }
    };
    const auto store = [&](int step) {
        const int base = gemm_base(step * S, S, nb);
#pragma unroll
        for (int i = 0; i < AP; i++) {
            const int c = lane + 64 * i;
            *reinterpret_cast<v4i *>(L.a + (c / (2 * S)) * P + 16 * (c % (2 * S))) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < BP; i++) {
            const int c = lane + 64 * i;
            int8_t * o = L.b + (c / BR) * P + (TYPE == T_Q8_0 ? 16 : 32) * (c % BR);
            if constexpr (TYPE == T_Q8_0) {
                *reinterpret_cast<v4i *>(o) = rb[i];
            } else {
                v4i lo, hi;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    lo[e] = (int) q4_to_s8((uint32_t) rb[i][e]);
                    hi[e] = (int) q4_to_s8((uint32_t) rb[i][e] >> 4);
                }
                *reinterpret_cast<v4i *>(o) = lo;
                *reinterpret_cast<v4i *>(o + 16) = hi;
            }
        }
#pragma unroll
        for (int i = 0; i < SP; i++) {
            const int c = lane + 64 * i;
            const bool own = gemm_own(c % S, base, step * S, nb);
            L.dx[(c % S) * 32 + c / S] = own ? rx[i] : 0.0f;
            L.dw[(c % S) * 32 + c / S] = own ? h2f((uint16_t) rw[i]) : 0.0f;
        }
    };
    // LDS writes of one lane are read by others of the wavefront: keep the compiler from moving either across.
    const auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    v16f acc{};
    v16i magic;
#pragma unroll
    for (int r = 0; r < 16; r++) magic[r] = kMagicBits;
    asm volatile("" : "+v"(magic));

    const int steps = (nb + S - 1) / S;
    if (g < steps) load(g);
    for (int step = g; step < steps; step += KG) {
        sync();
        store(step);
        sync();
        load(min(step + KG, steps - 1));
#pragma unroll
        for (int j = 0; j < S; j++) {
            const v4i af = *reinterpret_cast<const v4i *>(L.a + lr * P + j * 32 + 16 * lk);
            const v4i bf = *reinterpret_cast<const v4i *>(L.b + lr * P + j * 32 + 16 * lk);
            const float dwv = L.dw[j * 32 + lr];
            float cw = -kMagic * dwv;
            v16i cc = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, magic, 0, 0, 0);
            if (__builtin_expect(__any(__builtin_isinf(dwv)), 0)) {  // an infinite weight scale (as in k_gemm)
#pragma unroll
                for (int r = 0; r < 16; r++) cc[r] = __float_as_int(__int_as_float(cc[r]) - kMagic);
                cw = 0.0f;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 d4 = *reinterpret_cast<const float4 *>(&L.dx[j * 32 + q * 8 + lk * 4]);
                const float dx[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                for (int r = 0; r < 4; r++)
                    acc[4 * q + r] = fmaf(fmaf(__int_as_float(cc[4 * q + r]), dwv, cw), dx[r], acc[4 * q + r]);
            }
            // one block's sums in registers at a time (the MFMAs of all S blocks first: 230 registers for 130, and slower)
            asm volatile("" : "+v"(magic), "+v"(acc));
        }
    }

    // The groups' sums, added in the groups' order: each wavefront finishes its share of the accumulators.
    __syncthreads();
    float * red = reinterpret_cast<float *>(lds) + lane;
#pragma unroll
    for (int r = 0; r < REGS; r++) red[(g * REGS + r) * 64] = acc[r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < REGS / KG; i++) {
        const int r = g * (REGS / KG) + i;
        float v = red[r * 64];
#pragma unroll
        for (int k = 1; k < KG; k++) v += red[(k * REGS + r) * 64];
        const int m = m0 + (r >> 2) * 8 + lk * 4 + (r & 3), n = n0 + lr;
        if (m >= M || n >= N) continue;
        const size_t o = (size_t) m * ldy + n;
        y[o] = res ? v + res[o] : v;
    }
}

template <int TYPE>
static void run_gemm(const void * wv, int64_t N, int64_t K, const void * act, int64_t M, float * y, int64_t ldy, hipStream_t s,
                     const float * res) {
    const WeightLayout L = weight_layout(TYPE, N, K);
    const ActLayout A = act_layout(TYPE, M, K);
    const uint8_t * qs = (const uint8_t *) wv + L.qs;
    const uint16_t * d = (const uint16_t *) ((const uint8_t *) wv + L.d);
    const int8_t * xc = (const int8_t *) ((const uint8_t *) act + A.codes);
    const float2 * xm = (const float2 *) ((const uint8_t *) act + A.meta);
    const int nb = (int) (K / 32), m = (int) M, n = (int) N, ld = (int) ldy;
    const auto tiles = [&](int64_t tm, int64_t tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
    const int64_t cus = cu_count(), t32 = tiles(32, 32), t128 = tiles(128, 128);
    // Kernel times at K = 4096, us, for 32 x 32 tiles in eight and in four wavefronts and 128 x 128 tiles in two K groups
    // and without. 32 x 32 tiles: about 9 us plus 5 for every tile per CU; 128 x 128 tiles in two groups 50-70 up to a
    // tile per CU (each workgroup's serial chain over K). They meet at 11 32 x 32 tiles per CU. With more than one
    // 128 x 128 tile per CU two workgroups share it and groups only add the sums. Up to 32 rows fill a quarter of a 128-row tile
    // at most, whatever N is.
    //                      Q4_0                       Q8_0
    //   33 x 4096       9.5 / 12.8 / 50 / 69      11 /  13 /  53 /  67
    //   512 x 2048       27 /  26 /  59 / 72      33 /  28 /  59 /  70
    //   512 x 4096       49 /  45 /  60 / 74      63 /  48 /  63 /  72
    //   1024 x 4096     104 /  94 /  68 / 81     135 /  98 /  71 /  79
    //   129 x 32000     108 / 102 / 123 / 99     140 / 102 / 125 / 100
    //   16 x 128256     100 /  96 / 218 / 210    144 / 130 / 248 / 194
    //   32 x 128256     123 / 117 / 232 / 214    175 / 151 / 259 / 234
    // 765 shapes of 9 to 2048 rows, 96 to 128256 columns and K 256 to 14336: within 1 % of the best of the four on average for
    // both types; the farthest off it 39 % (Q8_0 129 x 2048 x 256) and 30 % (Q8_0 33 x 128256 x 4096).
    if (2 * t32 <= 3 * cus) k_gemm_kg<TYPE, 4, 8><<<(unsigned) t32, 512, 0, s>>>(qs, d, xc, xm, y, res, m, n, nb, ld);
    else if (t32 <= 11 * cus || m <= 32) k_gemm_kg<TYPE, 4, 4><<<(unsigned) t32, 256, 0, s>>>(qs, d, xc, xm, y, res, m, n, nb, ld);
    else if (t128 <= cus) k_gemm<TYPE, false, 2><<<(unsigned) t128, 512, 0, s>>>(qs, d, xc, xm, y, res, nullptr, m, n, nb, ld, 0);
    else k_gemm<TYPE, false, 1><<<(unsigned) t128, 256, 0, s>>>(qs, d, xc, xm, y, res, nullptr, m, n, nb, ld, 0);
}

void launch_gemm(int type, const void * wv, int64_t N, int64_t K, const void * act, int64_t M, float * y, int64_t ldy,
                 hipStream_t s, const float * res) {
    if (type == T_Q8_0) run_gemm<T_Q8_0>(wv, N, K, act, M, y, ldy, s, res);
    else if (type == T_Q4_0) run_gemm<T_Q4_0>(wv, N, K, act, M, y, ldy, s, res);
    else
        fail("gemm: unsupported weight type " + std::to_string(type));
    check_launch("gemm");
}

void launch_gemm_block_isums(int type, const void * wv, int64_t N, int64_t K, const void * act, int64_t M, int blk,
                             int32_t * out, hipStream_t s) {
    const WeightLayout L = weight_layout(type, N, K);
    const ActLayout A = act_layout(type, M, K);
    const uint8_t * w = (const uint8_t *) wv;
    const uint8_t * a = (const uint8_t *) act;
    const unsigned grid = (unsigned) (((M + GBM - 1) / GBM) * ((N + GBN - 1) / GBN));
    const int nb = (int) (K / 32);
    if (type == T_Q8_0)
        k_gemm<T_Q8_0, true, 1><<<grid, 256, 0, s>>>(w + L.qs, (const uint16_t *) (w + L.d), (const int8_t *) (a + A.codes),
                                                   (const float2 *) (a + A.meta), nullptr, nullptr, out, (int) M, (int) N, nb, 0,
                                                   blk);
    else if (type == T_Q4_0)
        k_gemm<T_Q4_0, true, 1><<<grid, 256, 0, s>>>(w + L.qs, (const uint16_t *) (w + L.d), (const int8_t *) (a + A.codes),
                                                   (const float2 *) (a + A.meta), nullptr, nullptr, out, (int) M, (int) N, nb, 0,
                                                   blk);
    else
        fail("gemm: unsupported weight type " + std::to_string(type));
    check_launch("gemm isums");
}

}  // namespace gcq
