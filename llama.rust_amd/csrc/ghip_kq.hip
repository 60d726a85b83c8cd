// ghip_kq.hip -- prefill MUL_MAT with Q2_K, Q3_K and Q6_K weights: the exact
// integer sum of a super-block on the int8 matrix cores.
//
// Reference (vec_dot.rs:758-834, :998-1028; tiled.rs): per super-block
//   is  = sum over 16-element groups g of sc[g] * sum (q * q8)     (exact integer)
//   im  = sum over g of m[g] * bsum16[g]                            (Q2_K)
//   out += (d * is - dmin * im) * d8
//
// The scale is multiplied into the codes, so is = sum (sc * q) * q8 needs no
// fold below the super-block:
//   Q3_K  -(sc * q), sc in -32..31, q in -4..3: -128..124, one int8 plane (the
//         sign goes to d; sc * q itself reaches 128);
//   Q2_K  sc * q <= 45, one int8 plane; im is one f16 MFMA (m <= 15, |bsum16| <=
//         2032: exact in f32);
//   Q6_K  p = sc * q, |p| <= 4096, as p = 128 * (p >> 7) + (p & 127): two int8
//         planes, made in registers from the codes and scales (18 vector
//         instructions per plane and 16 values; kept planes would be 2 bytes
//         a weight).
// Every partial sum fits int32 (|is| <= 2^27), so is is exact for any block, and
// the f32 work is one conversion, one product and one fma per output and
// super-block.  Eight super-blocks (Q3_K: four) add up apart from the total, whose own
// roundings are carried along: a plain chain is further from the 64-bit value
// than the decode kernels' trees (Q3_K, K = 14336: 8.6e-8 with groups of four and
// a plain total, 7.7e-8 the trees, 7.1e-8 with eights; 300 x 4096 -> 14336: trees
// 6.5e-8, eights 6.6e-8 in 54 us, fours 5.7e-8 in 55).
//
// Bound, at 64 tokens x 128 rows a workgroup, by the wavefronts' serial steps
// (LDS reads, MFMAs, the f32 work) with two wavefronts a SIMD.  300 x 4096 ->
// 14336 Q3_K, kept records: 940 us in 75 launches of the 4-column decode kernel,
// 55 us here; 512 x 14336 -> 4096 Q6_K, kept records: 157 us on f16 planes from
// 336-byte records with 152 KB of LDS a workgroup, 114 us.
#include "ghip_common.h"
#include "ghip_kplanes.h"

typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

namespace {

constexpr int KQ_BM = 64, KQ_BN = 128;  // tokens, weight rows per workgroup
// Weight records, one per (32-row tile, super-block), tiles major: eight 1 KB
// pieces (32 elements each) in which lane 32h + r of a wavefront finds row r's
// elements 16h .. 16h+15, then per type
//   Q6_K  per lane the eight pieces' scales (8 bytes) | d f32 [32]
//   Q3_K  -d f32 [32]
//   Q2_K  per lane (32h + r) the mins of groups 8h .. 8h+7 of row r, f16 | d f32 [32] | dmin f32 [32]
constexpr int kq_rec(int type) { return type == 6 ? 8192 + 512 + 128 : type == 3 ? 8192 + 128 : 8192 + 1024 + 256; }

// one wavefront per record: lane 32n + r writes row r's pieces 4n .. 4n+3 (the
// elements 128n .. 128n+127, which share their bytes of qs / ql and qh)
template <int TYPE>
__device__ __forceinline__ void kq_repack_impl(const uint8_t *__restrict__ W, int64_t w_row_bytes, int N, int nb,
                                               int64_t nrec, uint8_t *__restrict__ out) {
    constexpr int BB = TYPE == 6 ? 210 : TYPE == 3 ? 110 : 84;
    const int64_t ri = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (ri >= nrec) return;
    const int r = threadIdx.x & 31, n = (threadIdx.x >> 5) & 1;
    const int64_t tile = ri / nb, row = tile * 32 + r;
    const int b = (int)(ri - tile * nb);
    const bool live = row < N;  // rows past the matrix: zeros
    const uint32_t lm = live ? ~0u : 0u;
    const uint8_t *blk = W + (live ? row : 0) * w_row_bytes + (int64_t)b * BB;
    uint8_t *rec = out + ri * kq_rec(TYPE);
    auto dwords = [&](const uint8_t *p, uint32_t (&v)[8]) {
        const uint4 a = ld16(p), e = ld16(p + 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = e.x; v[5] = e.y; v[6] = e.z; v[7] = e.w;
    };
    uint32_t lo[2][8], hi[8], sc[4];  // sc: the 16 (Q3_K: 12) scale bytes
    if constexpr (TYPE == 6) {
        dwords(blk + 64 * n, lo[0]);
        dwords(blk + 64 * n + 32, lo[1]);
        dwords(blk + 128 + 32 * n, hi);
    } else {
        dwords(blk + (TYPE == 3 ? 32 : 16) + 32 * n, lo[0]);
        if constexpr (TYPE == 3) {
            dwords(blk, hi);
            const uint32_t a0 = ld4(blk + 96), a1 = ld4(blk + 100), a2 = ld4(blk + 104);
            // the de-packed 16 six-bit scales (quants.rs:475-484)
            sc[0] = (a0 & 0x0f0f0f0fu) | ((a2 & 0x03030303u) << 4);
            sc[1] = (a1 & 0x0f0f0f0fu) | (((a2 >> 2) & 0x03030303u) << 4);
            sc[2] = ((a0 >> 4) & 0x0f0f0f0fu) | (((a2 >> 4) & 0x03030303u) << 4);
            sc[3] = ((a1 >> 4) & 0x0f0f0f0fu) | (((a2 >> 6) & 0x03030303u) << 4);
        } else {
            const uint4 a = ld16(blk);
            sc[0] = a.x; sc[1] = a.y; sc[2] = a.z; sc[3] = a.w;
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t v[8];
        if constexpr (TYPE == 6) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                v[i] = ((lo[j & 1][i] >> (4 * (j >> 1))) & 0x0f0f0f0fu) | (((hi[i] >> (2 * j)) & 0x03030303u) << 4);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                // group 8n + 2j + i / 4: byte 2(j & 1) + i / 4 of scale dword 2n + j / 2
                const uint32_t sw = n ? sc[2 + (j >> 1)] : sc[j >> 1];
                const int s8 = (int)((sw >> (16 * (j & 1) + 8 * (i >> 2))) & 0xffu);
                const int m = TYPE == 3 ? 32 - s8 : s8 & 15;  // Q3_K: minus the scale
                uint32_t q = (lo[0][i] >> (2 * j)) & 0x03030303u;
                if constexpr (TYPE == 3) q |= ((hi[i] >> (4 * n + j)) & 0x01010101u) << 2;  // code + 4
                const v2s m2 = {(short)m, (short)m}, o2 = {(short)(TYPE == 3 ? -4 * m : 0), (short)(TYPE == 3 ? -4 * m : 0)};
                const v2s a = __builtin_bit_cast(v2s, __builtin_amdgcn_perm(0u, q, 0x0c010c00u)) * m2 + o2;
                const v2s e = __builtin_bit_cast(v2s, __builtin_amdgcn_perm(0u, q, 0x0c030c02u)) * m2 + o2;
                v[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, e), __builtin_bit_cast(uint32_t, a), 0x06040200u);
            }
        }
        uint8_t *o = rec + (4 * n + j) * 1024 + r * 16;
        *reinterpret_cast<uint4 *>(o) = make_uint4(v[0] & lm, v[1] & lm, v[2] & lm, v[3] & lm);
        *reinterpret_cast<uint4 *>(o + 512) = make_uint4(v[4] & lm, v[5] & lm, v[6] & lm, v[7] & lm);
    }
    // the lane's half n of the scales (Q6_K) or mins (Q2_K), the block scales
    if constexpr (TYPE == 6) {
        uint32_t s[2] = {0, 0};
#pragma unroll
        for (int k = 0; k < 8; k++) s[k >> 2] |= (uint32_t)blk[192 + 2 * k + n] << (8 * (k & 3));
        *reinterpret_cast<uint2 *>(rec + 8192 + (32 * n + r) * 8) = make_uint2(s[0] & lm, s[1] & lm);
        if (n == 0) *reinterpret_cast<float *>(rec + 8704 + 4 * r) = live ? h2f(ld2(blk + 208)) : 0.0f;
    } else if constexpr (TYPE == 3) {
        if (n == 0) *reinterpret_cast<float *>(rec + 8192 + 4 * r) = live ? -h2f(ld2(blk + 108)) : 0.0f;
    } else {
        v8h m;
#pragma unroll
        for (int k = 0; k < 8; k++)
            m[k] = (_Float16)(unsigned short)((((n ? sc[2 + (k >> 2)] : sc[k >> 2]) & lm) >> (8 * (k & 3) + 4)) & 15u);
        *reinterpret_cast<v8h *>(rec + 8192 + (32 * n + r) * 16) = m;
        *reinterpret_cast<float *>(rec + 9216 + 128 * n + 4 * r) = live ? h2f(ld2(blk + 80 + 2 * n)) : 0.0f;
    }
}

// 64 tokens x 128 rows per 256-thread workgroup, wavefront w rows 32w .. 32w+31
// and both 32-token tiles; C[token][row].  The activations, shared by the four
// wavefronts, go through registers into one of two LDS stages (16-byte pieces
// swizzled by token), one super-block ahead; each wavefront's weights go from
// memory straight to its registers, the next super-block's piece c loaded as
// soon as piece c is multiplied.  K may be split over blockIdx.y (nbs
// super-blocks each, partial results zstride apart).
template <int TYPE, bool SUBSUMS>
__device__ __forceinline__ void gemm_kq_impl(const uint8_t *__restrict__ R, int N, int nb,
                                             const int8_t *__restrict__ codes, const _Float16 *__restrict__ bsT,
                                             const float *__restrict__ dT, int M, int Mpad, float *__restrict__ dst,
                                             int64_t ldd, int32_t *__restrict__ sub, int nbs, int64_t zstride) {
    constexpr int REC = kq_rec(TYPE), NP = TYPE == 6 ? 2 : 1;
    __shared__ __attribute__((aligned(16))) uint4 act[2][KQ_BM * 16];
    __shared__ __attribute__((aligned(16))) float da[2][KQ_BM];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, h = lane >> 5;
    const int tm_n = (M + KQ_BM - 1) / KQ_BM;
    // tiles in order on every XCD (workgroup b runs on XCD b % 8), the token
    // tiles of one weight slice next to each other
    const int total = (int)gridDim.x, bx = (int)blockIdx.x, xcd = bx % 8;
    const int id = xcd * (total / 8) + min(xcd, total % 8) + bx / 8;
    const int m0 = id % tm_n * KQ_BM, n0 = id / tm_n * KQ_BN;
    const int b0 = (int)blockIdx.y * nbs, b1 = min(nb, b0 + nbs);
    dst += (int64_t)blockIdx.y * zstride;
    const int rt = min(n0 / 32 + w, (N - 1) / 32);  // past the matrix: the last tile, not stored
    const uint8_t *wr = R + (int64_t)rt * nb * REC;

    // this thread's share of a super-block's activations: 64 bytes of one token
    const int st = tid >> 2, sp = 4 * (tid & 3);
    const int8_t *ap = codes + (int64_t)(m0 + st) * nb * QK_K + 16 * sp;
    struct Next {  // loads of the next super-block
        uint4 a[4];
        float da;
        uint2 sc;      // Q6_K
        float dw, dm;  // dm: Q2_K
        uint4 mn, bs[2];
    } nx = {};
    uint4 bq[8];
    auto load = [&](int b) {
#pragma unroll
        for (int i = 0; i < 4; i++) nx.a[i] = *reinterpret_cast<const uint4 *>(ap + (int64_t)b * QK_K + 16 * i);
        nx.da = dT[(int64_t)b * Mpad + m0 + (tid & 63)];
        const uint8_t *rec = wr + (int64_t)b * REC;
        if constexpr (TYPE == 6) {
            nx.sc = *reinterpret_cast<const uint2 *>(rec + 8192 + 8 * lane);
            nx.dw = *reinterpret_cast<const float *>(rec + 8704 + 4 * li);
        } else if constexpr (TYPE == 3) {
            nx.dw = *reinterpret_cast<const float *>(rec + 8192 + 4 * li);
        } else {
            nx.mn = *reinterpret_cast<const uint4 *>(rec + 8192 + 16 * lane);
            nx.dw = *reinterpret_cast<const float *>(rec + 9216 + 4 * li);
            nx.dm = *reinterpret_cast<const float *>(rec + 9344 + 4 * li);
#pragma unroll
            for (int t = 0; t < 2; t++)
                nx.bs[t] = *reinterpret_cast<const uint4 *>(bsT + ((int64_t)b * Mpad + m0 + 32 * t + li) * 16 + 8 * h);
        }
    };
    auto stage = [&](int p) {
#pragma unroll
        for (int i = 0; i < 4; i++) act[p][st * 16 + ((sp + i) ^ (st & 15))] = nx.a[i];
        if (tid < KQ_BM) da[p][tid] = nx.da;
    };
    auto piece = [&](int b, int c) { return *reinterpret_cast<const uint4 *>(wr + (int64_t)b * REC + c * 1024 + 16 * lane); };

    constexpr int GROUP = TYPE == 3 ? 4 : 8;  // super-blocks that add up apart from the total
    v16f part[2] = {}, sum[2] = {}, comp[2] = {};
    auto total_up = [&]() {  // sum += part, comp what the sum's rounding lost
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const v16f y = part[t] + comp[t], s2 = sum[t] + y;
            comp[t] = y - (s2 - sum[t]);
#pragma unroll
            for (int v = 0; v < 16; v++) comp[t][v] = sum_lost(comp[t][v]);
            sum[t] = s2;
            part[t] = v16f{};
        }
    };
    load(b0);
#pragma unroll
    for (int c = 0; c < 8; c++) bq[c] = piece(b0, c);
    stage(0);
    __syncthreads();
    for (int b = b0; b < b1; b++) {
        const int p = (b - b0) & 1, bn = min(b + 1, b1 - 1);
        const uint2 sc = nx.sc;
        const float dw = nx.dw, dm = nx.dm;
        const uint4 mn = nx.mn, bs[2] = {nx.bs[0], nx.bs[1]};
        load(bn);
        v16i acc[NP][2];
        v16f im[2];
        if constexpr (TYPE == 2) {
#pragma unroll
            for (int t = 0; t < 2; t++)
                im[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, bs[t]), __builtin_bit_cast(v8h, mn),
                                                               v16f{}, 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
            v4i a[2], bw[NP];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int tk = 32 * t + li;
                a[t] = __builtin_bit_cast(v4i, act[p][tk * 16 + ((2 * c + h) ^ (tk & 15))]);
            }
            if constexpr (TYPE == 6)
                kq_planes(bq[c], (int)(int8_t)((c < 4 ? sc.x : sc.y) >> (8 * (c & 3))), bw[0], bw[1]);
            else
                bw[0] = __builtin_bit_cast(v4i, bq[c]);
            bq[c] = piece(bn, c);
#pragma unroll
            for (int k = 0; k < NP; k++)
#pragma unroll
                for (int t = 0; t < 2; t++)
                    acc[k][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[t], bw[k], c == 0 ? v16i{} : acc[k][t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 d4 = *reinterpret_cast<const float4 *>(&da[p][32 * t + 8 * q + 4 * h]);
                const float dd[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int v = 4 * q + e;
                    const int is = TYPE == 6 ? acc[NP - 1][t][v] * 128 + acc[0][t][v] : acc[0][t][v];
                    float res = dw * (float)is;
                    if constexpr (TYPE == 2) res = fmaf(-dm, im[t][v], res);
                    part[t][v] = fmaf(res, dd[e], part[t][v]);
                    if constexpr (SUBSUMS) {
                        const int m = m0 + 32 * t + 8 * q + 4 * h + e, n = n0 + 32 * w + li;
                        if (m < M && n < N) {
                            const int64_t o = ((int64_t)m * N + n) * nb + b;
                            if constexpr (TYPE == 2) {
                                sub[2 * o] = is;
                                sub[2 * o + 1] = (int)im[t][v];
                            } else {
                                sub[o] = TYPE == 3 ? -is : is;
                            }
                        }
                    }
                }
            }
        if ((b - b0) % GROUP == GROUP - 1) total_up();
        stage(p ^ 1);
        __syncthreads();
    }
    total_up();
    const int n = n0 + 32 * w + li;
    if (n >= N) return;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int m = m0 + 32 * t + 8 * (v >> 2) + 4 * h + (v & 3);
            if (m < M) dst[(int64_t)m * ldd + n] = sum[t][v];
        }
}

}  // namespace

#define KQ_ARGS                                                                                                     \
    const uint8_t *__restrict__ R, int N, int nb, const int8_t *__restrict__ codes, const _Float16 *__restrict__ bsT, \
        const float *__restrict__ dT, int M, int Mpad, float *__restrict__ dst, int64_t ldd,                        \
        int32_t *__restrict__ sub, int nbs, int64_t zstride
#define KQ_INST(TN, TYPE)                                                                                           \
    extern "C" __global__ void __launch_bounds__(256, 2) ghip_gemm_kq_##TN(KQ_ARGS) {                               \
        gemm_kq_impl<TYPE, false>(R, N, nb, codes, bsT, dT, M, Mpad, dst, ldd, sub, nbs, zstride);                  \
    }                                                                                                               \
    extern "C" __global__ void __launch_bounds__(256, 2) ghip_gemm_kq_##TN##_sub(KQ_ARGS) {                         \
        gemm_kq_impl<TYPE, true>(R, N, nb, codes, bsT, dT, M, Mpad, dst, ldd, sub, nbs, zstride);                   \
    }                                                                                                               \
    extern "C" __global__ void __launch_bounds__(256)                                                               \
        ghip_kq_repack_##TN(const uint8_t *__restrict__ W, int64_t w_row_bytes, int N, int nb,                      \
                            int64_t nrec, uint8_t *__restrict__ out) {                                              \
        kq_repack_impl<TYPE>(W, w_row_bytes, N, nb, nrec, out);                                                     \
    }
KQ_INST(q2_K, 2)
KQ_INST(q3_K, 3)
KQ_INST(q6_K, 6)
