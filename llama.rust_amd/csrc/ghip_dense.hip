// ghip_dense.hip -- MUL_MAT with F32, F16 and BF16 weights: the decode kernel
// (up to 8 activation rows a launch) and, for F16 / BF16 from 9 rows (a few rows
// of a long K aside: dense_decode_pays in ghip.cpp), the
// prefill GEMM on the matrix cores.
//
// Reference (compute.rs:1680-1745; vec_dot.rs:1700-1727): F16 / BF16 weights
// take the f32 activation row rounded to the weight type (round to nearest
// even), so every product of two f16 (two bf16) values is exact in f32; F32
// weights multiply the f32 activation as it is.  Products are accumulated in
// f32 here (lane chains, then the workgroup's tree), the reference in its own
// f32 / f64 order: the results agree to fp32 summation rounding.
//
// Workgroup: 256 threads, 8 weight rows.  Thread j walks the row in chunks of
// 8 elements (j, j + 256, ...), loads each chunk of the 8 rows once (16 bytes
// per row for F16 / BF16, 32 for F32) and the matching activation chunk of
// every column, and keeps 8 x NC f32 partial sums.
#include "ghip_common.h"

namespace {

constexpr int WT_F32 = 0, WT_F16 = 1, WT_BF16 = 30;
constexpr int DRB = 8;  // weight rows per workgroup

DEV float bf16_to_f32(uint32_t h) { return __uint_as_float(h << 16); }
// f32 -> bf16 -> f32, round to nearest even (NaN stays NaN)
DEV float round_bf16(float x) {
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return __uint_as_float((u | 0x00400000u) & 0xffff0000u);
    return __uint_as_float((u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u);
}
DEV float round_f16(float x) { return (float)(_Float16)x; }

template <int WT> DEV float round_act(float x) {
    if constexpr (WT == WT_F16) return round_f16(x);
    else if constexpr (WT == WT_BF16) return round_bf16(x);
    else return x;
}
// element e of a weight row
template <int WT> DEV float wval(const uint8_t *row, int e) {
    if constexpr (WT == WT_F32) return __uint_as_float(ld4(row + 4 * e));
    else if constexpr (WT == WT_F16) return h2f(ld2(row + 2 * e));
    else return bf16_to_f32(ld2(row + 2 * e));
}
// the 8 elements of chunk c of a row (VEC: the row's chunks are 16-byte aligned)
template <int WT, bool VEC> DEV void wchunk(const uint8_t *row, int c, float *w) {
    if constexpr (VEC && WT != WT_F32) {
        const uint4 v = ld16(row + 16 * c);
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if constexpr (WT == WT_F16) {
                w[2 * k] = h2f(x[k] & 0xffffu);
                w[2 * k + 1] = h2f(x[k] >> 16);
            } else {
                w[2 * k] = bf16_to_f32(x[k] & 0xffffu);
                w[2 * k + 1] = bf16_to_f32(x[k] >> 16);
            }
        }
    } else if constexpr (VEC) {
        const uint4 a = ld16(row + 32 * c), b = ld16(row + 32 * c + 16);
        const uint32_t x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int k = 0; k < 8; k++) w[k] = __uint_as_float(x[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) w[k] = wval<WT>(row, 8 * c + k);
    }
}

template <int WT, int NC, bool VEC>
__device__ __forceinline__ void gemv_dense_impl(const uint8_t *__restrict__ W, int64_t w_row_bytes, int rows, int K,
                                                const float *__restrict__ x, int64_t x_stride, int ncols,
                                                float *__restrict__ dst, int64_t ldd) {
    __shared__ float red[4][DRB * NC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r0 = (int)blockIdx.x * DRB;
    const int nrow = min(DRB, rows - r0);
    float acc[DRB][NC];
#pragma unroll
    for (int r = 0; r < DRB; r++)
#pragma unroll
        for (int c = 0; c < NC; c++) acc[r][c] = 0.0f;
    const int nch = K / 8;
    for (int ch = tid; ch < nch; ch += 256) {
        float xv[NC][8];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const float *xc = x + (int64_t)min(c, ncols - 1) * x_stride + 8 * ch;
            const uint4 a = ld16(reinterpret_cast<const uint8_t *>(xc)), b = ld16(reinterpret_cast<const uint8_t *>(xc + 4));
            const uint32_t u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int k = 0; k < 8; k++) xv[c][k] = round_act<WT>(__uint_as_float(u[k]));
        }
#pragma unroll
        for (int r = 0; r < DRB; r++) {
            float w[8];
            wchunk<WT, VEC>(W + (int64_t)(r0 + min(r, nrow - 1)) * w_row_bytes, ch, w);
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int k = 0; k < 8; k++) acc[r][c] = fmaf(w[k], xv[c][k], acc[r][c]);
        }
    }
    // the K % 8 tail, one element per thread
    for (int e = 8 * nch + tid; e < K; e += 256) {
#pragma unroll
        for (int r = 0; r < DRB; r++) {
            const float w = wval<WT>(W + (int64_t)(r0 + min(r, nrow - 1)) * w_row_bytes, e);
#pragma unroll
            for (int c = 0; c < NC; c++)
                acc[r][c] = fmaf(w, round_act<WT>(x[(int64_t)min(c, ncols - 1) * x_stride + e]), acc[r][c]);
        }
    }
#pragma unroll
    for (int r = 0; r < DRB; r++)
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const float s = wave_sum_dpp(acc[r][c]);
            if (lane == 0) red[wave][r * NC + c] = s;
        }
    __syncthreads();
    if (tid < DRB * NC) {
        const int r = tid / NC, c = tid - r * NC;
        if (r < nrow && c < ncols)
            dst[(int64_t)c * ldd + r0 + r] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
    }
}

// ------------------------------------------------------------ prefill GEMM
// F16 / BF16 weights from 9 activation rows.  C[token][weight row] on
// v_mfma_f32_32x32x16_{f16,bf16}: every product of two halves is exact, sums
// are f32.  A workgroup owns BM tokens x BN weight rows (WM x WN wavefronts of
// 32 x 32 tiles, times WK that share K) and walks K in steps of KB; f32
// activations are rounded to the weight type on their way into LDS (no
// converted copy in memory, so no workspace).  NS steps are in flight in
// registers, two in LDS, one barrier per step.  An LDS row's 16-byte pieces
// are XOR-swizzled by the row.
//
// Sums: the MFMAs of 64 elements start from zero, eight such groups add up in
// a second register set and those in a third.  With chains of 16 MFMAs and
// one level the results were further from the 64-bit value (1.3e-7 at
// K = 4096) than the decode kernel's 16-element chains and tree (1.0e-7);
// these three levels are 0.94e-7 from it.  BF16, whose decode kernel is 0.78e-7
// from it (its products have fewer bits to lose) where the three levels are 0.85e-7,
// adds the groups to one sum that carries its roundings along: 0.67e-7, for 1-4 % of
// the time (200 x 4096 -> 4096 38.8 -> 40.2 us, 300 x 2048 -> 12000 80 -> 83; 512 x 1024
// -> 16384 49 -> 55).
//
// Bound by a step's latency (LDS writes, barrier, LDS reads, MFMAs and the
// next loads one after another) on one or two workgroups per CU, then by the
// operands' way into the CU (64 bytes a clock): BM x 4 + BN x 2 bytes per k
// against BM x BN / 512 MFMA clocks.  So long steps, and the largest tile that
// gives the chip enough workgroups (dense_gemm_tile in ghip.cpp); with few
// tiles, 32 x 32 ones whose four wavefronts share K.  F16 4096 x 4096, 200
// tokens: 419 us in 25 launches of the decode kernel, 44 us with steps of 64
// and one in flight, 40 us with four in flight, 26-30 us with steps of 128 and K
// shared by two wavefronts.
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

template <int WT> DEV v16f mfma_dense(uint4 a, uint4 b, v16f c) {
    if constexpr (WT == WT_F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}
// two activations as halves of the weight type
template <int WT> DEV uint32_t pack_act(float a, float b) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    if constexpr (WT == WT_F16) return __builtin_bit_cast(uint32_t, v2h{(_Float16)a, (_Float16)b});
    else return (__float_as_uint(round_bf16(a)) >> 16) | (__float_as_uint(round_bf16(b)) & 0xffff0000u);
}

DEV uint4 pin(uint4 v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
    return v;
}

// VEC: K is a multiple of 8 (whole pieces); else the rows' last piece is put
// together element by element
template <int WT, int BM, int BN, int KB, int WM, int WN, int WK, int NS, bool VEC>
__device__ __forceinline__ void gemm_dense_impl(const uint8_t *__restrict__ W, int64_t w_row_bytes, int rows, int K,
                                                const float *__restrict__ x, int64_t x_stride, int ncols,
                                                float *__restrict__ dst, int64_t ldd) {
    constexpr int NT = 64 * WM * WN * WK, P = KB / 8;         // threads; 8-element pieces per row and step
    constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN);  // 32 x 32 tiles per wavefront
    constexpr int PX = BM * P / NT, PW = BN * P / NT;        // ... and per thread
    constexpr int KG = KB / (64 * WK);                       // 64-element groups per wavefront and step
    __shared__ __attribute__((aligned(16))) uint4 lds[2][(BM + BN) * P];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wk = w / (WM * WN), wm = w % (WM * WN) / WN, wn = w % WN;
    const int l32 = lane & 31, h = lane >> 5;
    // tiles in order on every XCD (workgroup b runs on XCD b % 8), the token
    // tiles of one weight slice next to each other
    const int total = (int)gridDim.x, b = (int)blockIdx.x, q = total / 8, rem = total % 8, xcd = b % 8;
    const int id = xcd * q + min(xcd, rem) + b / 8;
    const int tm = (ncols + BM - 1) / BM;
    const int m0 = id % tm * BM, n0 = id / tm * BN;

    const float *xp[PX];
    const uint8_t *wp[PW];
    const int k8 = tid % P;
#pragma unroll
    for (int i = 0; i < PX; i++) xp[i] = x + (int64_t)min(m0 + (i * NT + tid) / P, ncols - 1) * x_stride;
#pragma unroll
    for (int i = 0; i < PW; i++) wp[i] = W + (int64_t)min(n0 + (i * NT + tid) / P, rows - 1) * w_row_bytes;
    struct Regs {
        uint4 x[PX][2], w[PW];
    };
    auto load = [&](int st, Regs &r) {
        const int k = st * KB + 8 * k8;
        if constexpr (VEC) {
            const int kc = min(k, K - 8);  // past the end: any piece, zeroed by stage
#pragma unroll
            for (int i = 0; i < PX; i++) {
                r.x[i][0] = ld16(reinterpret_cast<const uint8_t *>(xp[i] + kc));
                r.x[i][1] = ld16(reinterpret_cast<const uint8_t *>(xp[i] + kc + 4));
            }
#pragma unroll
            for (int i = 0; i < PW; i++) r.w[i] = ld16(wp[i] + 2 * kc);
        } else {
#pragma unroll
            for (int i = 0; i < PX; i++) {
                uint32_t t[8];
#pragma unroll
                for (int e = 0; e < 8; e++) t[e] = k + e < K ? __float_as_uint(xp[i][k + e]) : 0u;
                r.x[i][0] = make_uint4(t[0], t[1], t[2], t[3]);
                r.x[i][1] = make_uint4(t[4], t[5], t[6], t[7]);
            }
#pragma unroll
            for (int i = 0; i < PW; i++) {
                uint32_t t[4];
#pragma unroll
                for (int e = 0; e < 4; e++)
                    t[e] = (k + 2 * e < K ? ld2(wp[i] + 2 * (k + 2 * e)) : 0u) |
                           (k + 2 * e + 1 < K ? (uint32_t)ld2(wp[i] + 2 * (k + 2 * e + 1)) << 16 : 0u);
                r.w[i] = make_uint4(t[0], t[1], t[2], t[3]);
            }
        }
    };
    auto stage = [&](int st, const Regs &r) {
        const uint32_t in = !VEC || st * KB + 8 * k8 < K ? ~0u : 0u;  // else zeros
        uint4 *l = lds[st & 1];
#pragma unroll
        for (int i = 0; i < PX; i++) {
            const int row = (i * NT + tid) / P;
            // (as loaded until here: rounding them as they land would wait for
            // each step's loads as soon as they are issued)
            const uint4 a = pin(r.x[i][0]), c = pin(r.x[i][1]);
            auto f = [](uint32_t u) { return __uint_as_float(u); };
            const uint4 p = make_uint4(pack_act<WT>(f(a.x), f(a.y)), pack_act<WT>(f(a.z), f(a.w)),
                                       pack_act<WT>(f(c.x), f(c.y)), pack_act<WT>(f(c.z), f(c.w)));
            l[row * P + (k8 ^ (row & 7))] = make_uint4(p.x & in, p.y & in, p.z & in, p.w & in);
        }
#pragma unroll
        for (int i = 0; i < PW; i++) {
            const int row = (i * NT + tid) / P;
            const uint4 p = pin(r.w[i]);
            l[(BM + row) * P + (k8 ^ (row & 7))] = make_uint4(p.x & in, p.y & in, p.z & in, p.w & in);
        }
    };
    // of a wavefront's last (up to) eight groups (BF16: what the sum's roundings dropped); of those before (all)
    v16f part[TM][TN] = {}, sum[TM][TN] = {};
    const int nstep = (K + KB - 1) / KB;
    constexpr int FOLD = 8 / (KG * NS) > 1 ? 8 / (KG * NS) : 1;  // loop rounds per eight 64-element groups
    auto mult = [&](int st) {
        const uint4 *l = lds[st & 1];
#pragma unroll
        for (int g = 0; g < KG; g++) {
            uint4 a[4][TM], bw[4][TN];
            v16f acc[TM][TN];
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                const int s = 4 * (wk * KG + g) + s4;  // the step's 16-element slice
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const int r = (wm * TM + i) * 32 + l32;
                    a[s4][i] = l[r * P + ((2 * s + h) ^ (r & 7))];
                }
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int r = (wn * TN + j) * 32 + l32;
                    bw[s4][j] = l[(BM + r) * P + ((2 * s + h) ^ (r & 7))];
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // all reads on their way before the first product waits
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = mfma_dense<WT>(a[s4][i], bw[s4][j], s4 == 0 ? v16f{} : acc[i][j]);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    if constexpr (WT == WT_BF16) {
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const float y = acc[i][j][v] + part[i][j][v], t = sum[i][j][v] + y;
                            part[i][j][v] = sum_lost(y - (t - sum[i][j][v]));
                            sum[i][j][v] = t;
                        }
                    } else {
                        part[i][j] += acc[i][j];
                    }
                }
        }
    };
    auto fold = [&]() {
        if constexpr (WT == WT_BF16) return;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                sum[i][j] += part[i][j];
                part[i][j] = v16f{};
            }
    };
    // step st in r[st % NS]; steps past the last one stage zeros and load the
    // rows' last pieces, so that no branch merges the waits
    Regs r[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
        load(i, r[i]);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int st = 0; st < nstep; st += NS) {
#pragma unroll
        for (int i = 0; i < NS; i++) {
            stage(st + i, r[i]);
            load(st + i + NS, r[i]);
            __syncthreads();
            mult(st + i);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (st / NS % FOLD == FOLD - 1) fold();
    }
    fold();
    if constexpr (WK > 1) {  // one 32 x 32 tile per wavefront: the parts over K meet in LDS, tile by tile
        static_assert(TM == 1 && TN == 1, "one tile per wavefront");
        float *red = reinterpret_cast<float *>(&lds[0][0]);  // [wk][tile][v][lane]
        constexpr int NTL = WM * WN;
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; v++) red[(w * 16 + v) * 64 + lane] = sum[0][0][v];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 16 / WK; u++) {
            const int v = 16 / WK * wk + u, tl = w % NTL;
            const int t = m0 + wm * 32 + 8 * (v >> 2) + 4 * h + (v & 3), row = n0 + wn * 32 + l32;
            float s4[WK];
#pragma unroll
            for (int k = 0; k < WK; k++) s4[k] = red[((k * NTL + tl) * 16 + v) * 64 + lane];
            float y;
            if constexpr (WK == 4) y = (s4[0] + s4[1]) + (s4[2] + s4[3]);
            else y = s4[0] + s4[1];
            if (t < ncols && row < rows) dst[(int64_t)t * ldd + row] = y;
        }
    } else {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int row = n0 + (wn * TN + j) * 32 + l32;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int t = m0 + (wm * TM + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
                    if (t < ncols && row < rows) dst[(int64_t)t * ldd + row] = sum[i][j][v];
                }
            }
    }
}

}  // namespace

#define DENSE_INST(TN, WT, NC)                                                                                      \
    extern "C" __global__ void __launch_bounds__(256)                                                               \
        ghip_gemv_dense_##TN##_c##NC(const uint8_t *__restrict__ W, int64_t w_row_bytes, int rows, int K,            \
                                     const float *__restrict__ x, int64_t x_stride, int ncols,                      \
                                     float *__restrict__ dst, int64_t ldd, int vec) {                               \
        if (vec) gemv_dense_impl<WT, NC, true>(W, w_row_bytes, rows, K, x, x_stride, ncols, dst, ldd);              \
        else gemv_dense_impl<WT, NC, false>(W, w_row_bytes, rows, K, x, x_stride, ncols, dst, ldd);                 \
    }
#define DENSE_TYPE(TN, WT) DENSE_INST(TN, WT, 1) DENSE_INST(TN, WT, 2) DENSE_INST(TN, WT, 4) DENSE_INST(TN, WT, 8)
DENSE_TYPE(f32, WT_F32)
DENSE_TYPE(f16, WT_F16)
DENSE_TYPE(bf16, WT_BF16)

#define DENSE_GEMM(TN, WT, T, WAVES, VEC, BM, BN, KB, WM, WN, WK, NS)                                               \
    extern "C" __global__ void __launch_bounds__(64 * WM * WN * WK)                                                 \
        __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))                                                          \
        ghip_gemm_dense_##TN##_##T(const uint8_t *__restrict__ W, int64_t w_row_bytes, int rows, int K,              \
                                   const float *__restrict__ x, int64_t x_stride, int ncols,                        \
                                   float *__restrict__ dst, int64_t ldd) {                                          \
        gemm_dense_impl<WT, BM, BN, KB, WM, WN, WK, NS, VEC>(W, w_row_bytes, rows, K, x, x_stride, ncols, dst, ldd); \
    }
#define DENSE_GEMMS(TN, WT)                                                                                         \
    DENSE_GEMM(TN, WT, t128, 2, true, 128, 128, 128, 4, 2, 1, 1)                                                    \
    DENSE_GEMM(TN, WT, t64, 2, true, 64, 64, 128, 2, 2, 2, 2)                                                       \
    DENSE_GEMM(TN, WT, t32, 2, true, 32, 32, 256, 1, 1, 4, 2)                                                       \
    DENSE_GEMM(TN, WT, odd, 2, false, 32, 32, 256, 1, 1, 4, 1)
DENSE_GEMMS(f16, WT_F16)
DENSE_GEMMS(bf16, WT_BF16)
