// k_band.hip -- two-stage reduction of the batched FP32 eigensolver (gfx950),
// replacing the one-stage Householder tridiagonalisation of magma_ssyevd_gpu
// (calcIR.cu:420-448) for Hamiltonians of up to sb_max_n().
//
//   Stage 1, dense -> band of half-width kBandNB (LAPACK sytrd_sy2sb form):
//     for each panel of kBandNB columns, sb_panel_kernel factors the panel
//     below the band, A(r0:n, j0:j0+NB) = Q R, by Householder reflectors in
//     registers (one workgroup per matrix); the trailing matrix then gets the
//     two-sided update A22 <- Q^T A22 Q on its lower triangle, batched over
//     every matrix: X = A22 Yh with Yh = Y T (sb_symm_kernel), W = X -
//     Y (Yh^T X)/2 (sb_w_kernel), A22 -= W Y^T + Y W^T
//     (sb_syr2k_kernel), on 32x32x2 FP32 MFMA.
//   Stage 2, band -> tridiagonal (sb2st_kernel): bulge chasing, one workgroup
//     per matrix, sweeps in groups of kSbG run by the group's waves with a
//     lag of two tasks (the tasks of one step touch disjoint elements), the
//     groups one after the other as a stream of steps (SbStream); the band rows
//     that the waves touch live in a circular LDS window over the stream.
//   Q2 back-transform (q2_*): the bulge-chasing reflectors of kQ2G
//     consecutive sweeps at one block position form a compact-WY block; the
//     rows of a column slab of the eigenvectors stream through a workgroup's
//     waves, each applying its groups' blocks; groups last to first, block
//     positions in ascending order.
//
// Storage (per matrix):
//   BND   band rows: element (r, c), 0 <= r - c < 2 NB, at BND[r * 2NB + r - c]
//         (the bulge region r - c > NB is zero outside the chase)
//   A     column j0 + l of panel j0 holds reflector l below row r0 = j0 + NB:
//         rows r0..r0+l-1 zero, row r0+l one, rows below the reflector, the
//         layout the compact-WY back-transform reads (offset NB)

#include <algorithm>
#include <cfloat>

#include "band.hpp"
#include "split_bf16.hpp"
#include "tuner.hpp"

namespace cir {

constexpr int kPanNT = 512;  // threads per matrix in the panel factorisation
constexpr int kPanNW = kPanNT / 64;

// DPP row rotation by CTRL (row_ror 8, 4, 2, 1) within 16-lane rows.
template <int CTRL>
__device__ __forceinline__ float bdpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float brow_sum16(float x) {
    x += bdpp<0x128>(x);
    x += bdpp<0x124>(x);
    x += bdpp<0x122>(x);
    x += bdpp<0x121>(x);
    return x;
}
__device__ __forceinline__ float bwave_sum(float x) {
    x = brow_sum16(x);
    // rows of 16 lanes: add the other row of the half, then the other half
    auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
    auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
}

// Wave sums of 32 per-lane values x[k], written to out[k] (LDS).  Two lane
// swaps halve the values per lane (after them lane l holds the partials of
// columns k + 8 (l >> 4), k < 8), 16-lane row sums finish them, and lane
// 16 R + i (i < 8) stores column 8 R + i.
__device__ __forceinline__ void wave_colsums32(const float (&x)[32], int lane, float* out) {
    float y[16], z[8];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[k]), __float_as_uint(x[k + 16]), false,
                                                         false);
        y[k] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[k]), __float_as_uint(y[k + 8]), false,
                                                         false);
        z[k] = brow_sum16(__uint_as_float(sw[0]) + __uint_as_float(sw[1]));
    }
    const int i = lane & 15;
    float v = z[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) v = (i == k) ? z[k] : v;
    if (i < 8) out[8 * (lane >> 4) + i] = v;
}

// Householder scalars for a vector with first element alpha and tail square sum
// sigma > 0: beta = -sign(alpha) |x|, tau = (beta - alpha) / beta, scale = 1 /
// (alpha - beta).  |x| from the hardware's reciprocal root y with one
// Newton step each way (the residual of |x|^2, of tau beta and of scale
// (alpha - beta), each by one FMA, so each result is within an ulp); the IEEE
// root and quotients are three chains of a dozen dependent instructions on a
// task's critical path.  Squares too large for the hardware root take those.
// False, and nothing done, for squares below kSbTiny: nearly equal columns leave
// vectors whose length falls by FP32's rounding from column to column, and below
// that the squares are lost to underflow, and with them the reflector its
// orthogonality (eigenvalues off by 1e-4 of the spectrum).  The caller then sums
// the squares of kSbUp x (sb_householder_up).
constexpr float kSbTiny = 1e-30f, kSbUp = 0x1p60f;
__device__ __forceinline__ bool sb_householder(float alpha, float sigma, float& beta, float& tau, float& scale) {
    const float a2 = alpha * alpha + sigma;
    if (!(a2 >= kSbTiny && a2 <= 1e30f)) {
        if (a2 < kSbTiny) return false;
        const float nrm = sqrtf(a2);
        beta = alpha >= 0.f ? -nrm : nrm;
        tau = (beta - alpha) / beta;
        scale = 1.f / (alpha - beta);
        return true;
    }
    const float y = __builtin_amdgcn_rsqf(a2);
    float nrm = a2 * y;
    nrm = fmaf(fmaf(-nrm, nrm, a2), 0.5f * y, nrm);
    beta = alpha >= 0.f ? -nrm : nrm;
    const float yb = alpha >= 0.f ? -y : y;  // about 1 / beta
    const float den = alpha - beta;
    tau = -den * yb;
    tau = fmaf(fmaf(-tau, beta, -den), yb, tau);
    const float r = __builtin_amdgcn_rcpf(den);
    scale = fmaf(fmaf(-den, r, 1.f), r, r);
    return true;
}
// The scalars from alpha and the square sum of kSbUp x.  What is still too short
// (1e-33) is taken as zero.
__device__ __forceinline__ void sb_householder_up(float alpha, float sigma, float& beta, float& tau, float& scale) {
    if (!(sigma > 0.f) || !sb_householder(alpha * kSbUp, sigma, beta, tau, scale)) return;
    beta *= 1.f / kSbUp;
    scale *= kSbUp;
}

// Householder QR of one panel below the band and everything the trailing
// update needs.  Panel rows r0..n-1 (m = n - r0 of them) are spread over the
// threads, rows tid + 512 i (i < RPT) per thread, all NB columns in
// registers.  One block sum per column c: the 32 products of its part below
// row c, x, with every column (x itself among them, so the norm); with row c,
// which its thread publishes, v^T P(:, c') = scale x^T P(:, c') + P(c, c') for
// v = (1, scale x): the trailing columns' w and, for c' < c, the Gram column
// Y^T v of the T factor.  One barrier per column: every wave adds up the
// waves' partial sums itself, lane q the total of column q, and takes the
// updates' factors from its lanes.  Columns are worked on in blocks of 8,
// rotated to the front of the registers, so that register indices are
// constants in a loop body of 8 columns.  Bound by the chain of a column
// (sums, scalars, update); a norm sum, the products and the totals as three
// sums with three barriers, and selects over all 32 columns, took 145 .. 190
// us per panel for up to a matrix per CU; this takes 47 .. 71 us (RPT 1 .. 4,
// one matrix; 256 matrices of RPT = 4 move 270 MB and take 155 us).  Outputs: the diagonal block and R
// into BND, tau, Y into A (back-transform layout) and into the Y half of the
// row-major panel P (absolute rows, pitch 2 NB), Yh = Y T row-major (panel
// rows, pitch NB).
template <int RPT>
__global__ void __launch_bounds__(kPanNT) sb_panel_kernel(int n, int ld, int j0, float* __restrict__ Aall,
                                                          float* __restrict__ BNDall, float* __restrict__ tauall,
                                                          float* __restrict__ Pall, float* __restrict__ Yhall) {
    constexpr int NB = kBandNB, CB = 8;
    static_assert(NB == 32, "the column sums and the rotation are written for 32 columns");
    __shared__ float redC[2][kPanNW][NB], redS[kPanNW], taus[NB];
    __shared__ __align__(16) float rowc[2][NB], gram[NB][NB + 4], Tc[NB][NB + 4];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* A = Aall + size_t(b) * n * ld;
    float* BND = BNDall + size_t(b) * n * kBandW;
    float* P = Pall + size_t(b) * n * 2 * NB;
    float* Yh = Yhall + size_t(b) * n * NB;
    const int r0 = j0 + NB, m = n - r0;

    // the panel's diagonal block is final: lower triangle into the band rows
    for (int q = tid; q < NB * NB; q += kPanNT) {
        const int i = q / NB, c = q % NB;
        if (c <= i && j0 + i < n) BND[size_t(j0 + i) * kBandW + (i - c)] = A[size_t(j0 + c) * ld + j0 + i];
    }
    float p[RPT][NB];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int row = tid + kPanNT * i;
#pragma unroll
        for (int c = 0; c < NB; ++c) p[i][c] = (row < m) ? A[size_t(j0 + c) * ld + r0 + row] : 0.f;
    }

    // register column q holds column (q + CB blk) mod NB
#pragma unroll 1
    for (int blk = 0; blk < NB / CB; ++blk) {
#pragma unroll
        for (int cc = 0; cc < CB; ++cc) {
            const int c = CB * blk + cc, buf = cc & 1;
            float dots[NB];
#pragma unroll
            for (int q = 0; q < NB; ++q) dots[q] = 0.f;
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                const float x = (tid + kPanNT * i > c) ? p[i][cc] : 0.f;
#pragma unroll
                for (int q = 0; q < NB; ++q) dots[q] += x * p[i][q];
            }
            wave_colsums32(dots, lane, redC[buf][wave]);
            if (tid == c) {
#pragma unroll
                for (int q = 0; q < NB; q += 4)
                    *reinterpret_cast<float4*>(&rowc[buf][q]) = float4{p[0][q], p[0][q + 1], p[0][q + 2], p[0][q + 3]};
            }
            __syncthreads();
            const int q = lane & 31;
            float tot = 0.f;
#pragma unroll
            for (int w = 0; w < kPanNW; ++w) tot += redC[buf][w][q];
            const float pcq = rowc[buf][q];
            const float sigma = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tot), cc));
            const float alpha = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pcq), cc));
            float tau = 0.f, beta = alpha, scale = 0.f;
            if (sigma > 0.f && !sb_householder(alpha, sigma, beta, tau, scale)) {
                // (alpha and sigma are the same in every thread)
                float x2 = 0.f;
#pragma unroll
                for (int i = 0; i < RPT; ++i) {
                    const float x = (tid + kPanNT * i > c) ? p[i][cc] * kSbUp : 0.f;
                    x2 += x * x;
                }
                x2 = bwave_sum(x2);
                if (lane == 0) redS[wave] = x2;
                __syncthreads();
                x2 = 0.f;
#pragma unroll
                for (int w = 0; w < kPanNW; ++w) x2 += redS[w];
                sb_householder_up(alpha, x2, beta, tau, scale);
            }
            tot = scale * tot + pcq;  // v^T P(:, column of register q)
            if (wave == 0) {
                const int qc = (q + CB * blk) & (NB - 1);
                if (lane < NB && qc < c) gram[c][qc] = tot;
                if (lane == 0) taus[c] = tau;
            }
            const float f = tau * tot;
            float v[RPT];
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                const int row = tid + kPanNT * i;
                const float y = p[i][cc] * scale;
                v[i] = (row > c) ? y : (row == c ? 1.f : 0.f);
                p[i][cc] = (row > c) ? y : (row == c ? beta : p[i][cc]);
            }
            // trailing panel columns: P(:, c') -= tau v (v^T P(:, c'))
            auto update = [&](int q0, int q1) {
#pragma unroll
                for (int u = q0; u < q1; ++u) {
                    const float fu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), u));
#pragma unroll
                    for (int i = 0; i < RPT; ++i) p[i][u] -= fu * v[i];
                }
            };
            update(cc + 1, CB);
            if (blk < 3) update(CB, 2 * CB);
            if (blk < 2) update(2 * CB, 3 * CB);
            if (blk < 1) update(3 * CB, 4 * CB);
        }
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            float t[CB];
#pragma unroll
            for (int q = 0; q < CB; ++q) t[q] = p[i][q];
#pragma unroll
            for (int q = 0; q < NB - CB; ++q) p[i][q] = p[i][q + CB];
#pragma unroll
            for (int q = 0; q < CB; ++q) p[i][NB - CB + q] = t[q];
        }
    }

    // T factor (forward, columnwise): T(c, c) = tau_c, T(0:c, c) = -tau_c
    // T(0:c, 0:c) Y^T v_c; wave 0, lane t the row t of T in registers
    if (wave == 0) {
        wave_lds_sync();
        const int t = lane;
        float Tr[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            float acc = 0.f;
#pragma unroll
            for (int q = 0; q < c; ++q) acc += Tr[q] * gram[c][q];
            const float tc = taus[c];
            Tr[c] = (t == c) ? tc : (t < c ? -tc * acc : 0.f);
            if (t < NB) Tc[c][t] = Tr[c];
        }
        if (t < NB) tauall[size_t(b) * n + j0 + t] = taus[t];
    }
    // R (upper triangle of rows r0..r0+NB-1) into the band rows
    if (tid < NB && tid < m) {
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (c >= tid) BND[size_t(r0 + tid) * kBandW + (NB + tid - c)] = p[0][c];
    }
    // column j0 + c above the reflector's unit is zero from row 0 (the
    // back-transform reads whole passes of columns from their first row, and
    // the band part of these columns is in BND now)
    for (int c = 0; c < NB; ++c)
        for (int r = tid; r < r0 + c && r < n; r += kPanNT) A[size_t(j0 + c) * ld + r] = 0.f;
    // Y into A and P
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int row = tid + kPanNT * i;
#pragma unroll
        for (int c = 0; c < NB; ++c) p[i][c] = (row < c) ? 0.f : (row == c ? 1.f : p[i][c]);
        if (row >= m) continue;
#pragma unroll
        for (int c = 0; c < NB; ++c) A[size_t(j0 + c) * ld + r0 + row] = p[i][c];
        float4* pr = reinterpret_cast<float4*>(P + size_t(r0 + row) * 2 * NB);
#pragma unroll
        for (int q = 0; q < NB / 4; ++q)
            pr[q] = float4{p[i][4 * q], p[i][4 * q + 1], p[i][4 * q + 2], p[i][4 * q + 3]};
    }
    __syncthreads();
    // Yh = Y T, four columns at a time
#pragma unroll
    for (int c0 = 0; c0 < NB; c0 += 4) {
        float acc[RPT][4];
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][e] = 0.f;
#pragma unroll
        for (int q = 0; q < c0 + 4; q += 4)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float4 t = *reinterpret_cast<const float4*>(&Tc[c0 + e][q]);  // T(q .. q + 3, c0 + e)
#pragma unroll
                for (int i = 0; i < RPT; ++i)
                    acc[i][e] += p[i][q] * t.x + p[i][q + 1] * t.y + p[i][q + 2] * t.z + p[i][q + 3] * t.w;
            }
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int row = tid + kPanNT * i;
            if (row < m)
                *reinterpret_cast<float4*>(Yh + size_t(row) * NB + c0) = float4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
        }
    }
}

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Workgroup x of matrix b in a grid of gx workgroups per matrix over batch
// matrices, launched one-dimensional (xcd_grid): workgroup i runs on XCD i
// mod 8 (round-robin dispatch) and XCD x takes the x-th eighth of the
// (matrix, workgroup) list, so a matrix's workgroups run together on one XCD
// and share its panel through that XCD's L2.  False for the padding past the
// list.
__device__ __forceinline__ bool xcd_slot(int gx, int batch, int& x, int& b) {
    const int64_t total = int64_t(gx) * batch, per = (total + kXcds - 1) / kXcds;
    const int64_t pos = int64_t(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (pos >= total) return false;
    b = int(pos / gx);
    x = int(pos % gx);
    return true;
}
inline dim3 xcd_grid(int gx, int batch) { return dim3(unsigned(ceil_div(int64_t(gx) * batch, int64_t(kXcds)) * kXcds)); }

constexpr int kSyWaves = 4;  // waves per block row of the trailing matrix

// X = A22 Yh on the lower triangle of A22 (m x m, column-major, pitch ld,
// first row and column r0), X row-major with pitch 2 NB in the W half of the
// row-major panel P (rows r0.., P[r * 2NB + NB + p]); Yh row-major, pitch NB
// (panel rows).  Workgroup x owns block row I = x, wave w its tiles J = w, w +
// WV, ..., summed in wave order at the end.  Every tile is read from its own
// side: the row tiles (I, J < I) go straight into the MFMA A operand (lanes
// along rows, coalesced), the column tiles (J >= I, I) are read along their
// rows too and transposed through the wave's LDS tile.  The next tile's loads
// are in flight while a tile's MFMA chain runs.  32x32x2 FP32 MFMA, K = 32 per
// tile.  Bound by latency where there are few matrices, by memory (4 TB/s) where
// there are many.  With a block row per wave, up to nbt tiles one after the
// other: 63 calls for one matrix of N = 2048 2.78 ms, 128 matrices 12.6, 48 of N
// = 768 0.52; with 4 waves to a row 0.90, 11.4, 0.37; with 8 0.77 for the one
// matrix, but 0.45 for the 48 (the sums cost more than the shorter chains give).
__global__ void __launch_bounds__(64 * kSyWaves) sb_symm_kernel(int n, int ld, int r0, const float* __restrict__ Aall,
                                                      const float* __restrict__ Yhall, float* __restrict__ Pall,
                                                      int batch) {
    constexpr int NB = kBandNB, WV = kSyWaves;
    __shared__ float tl[WV][32][33];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = n - r0, nbt = (m + 31) / 32;
    int x, b;
    if (!xcd_slot(nbt, batch, x, b)) return;
    const int I = x;
    const float* A = Aall + size_t(b) * n * ld + size_t(r0) * ld + r0;
    const float* Yh = Yhall + size_t(b) * n * NB;
    float* P = Pall + size_t(b) * n * 2 * NB + size_t(r0) * 2 * NB;
    const int l32 = lane & 31, h = lane >> 5;
    const int ri = I * 32 + l32;  // this lane's row of block row I (M index)
    float (*T)[33] = tl[wave];
    // raw loads of tile J: the B operand (Yh rows J*32 + 2q + h) and the A
    // tile, as the A operand itself (row tile) or along the tile's rows for
    // the LDS transpose (column tile, T[2q + h][l32] = A22(J*32 + l32, I*32 + 2q + h))
    // Every load is issued with its index clamped below m and nothing is
    // masked until the values are used (the loads of a tile go out back to
    // back, a tile ahead): rows and columns of the output past m are never
    // stored, and K indices past m are cancelled by zeroing the B operand.
    const int ric = min(ri, m - 1);
    auto load = [&](int J, float (&bv)[16], float (&raw)[16]) {
#pragma unroll
        for (int q = 0; q < 16; ++q) bv[q] = Yh[size_t(min(J * 32 + 2 * q + h, m - 1)) * NB + l32];
        // row tile (J < I): A(J*32 + 2q + h, ri); column tile: A(I*32 + 2q + h,
        // J*32 + l32) (columns of the column-major lower triangle)
        const bool rowt = J < I;
        const int c0 = (rowt ? J : I) * 32 + h;
        const float* base = A + (rowt ? ric : min(J * 32 + l32, m - 1));
#pragma unroll
        for (int q = 0; q < 16; ++q) raw[q] = base[size_t(min(c0 + 2 * q, m - 1)) * ld];
    };
    floatx16 acc;
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.f;
    // tile J from (bv, raw) while the next one is read into (bn, rn) (past the
    // last tile: clamped reads, never used); the two buffer pairs alternate,
    // so no copy waits for a read in flight
    auto tile = [&](int J, float (&bv)[16], float (&raw)[16], float (&bn)[16], float (&rn)[16]) {
        load(J + WV, bn, rn);
        __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the products
#pragma unroll
        for (int q = 0; q < 16; ++q) bv[q] = (J * 32 + 2 * q + h < m) ? bv[q] : 0.f;
        float av[16];
        if (J < I) {
#pragma unroll
            for (int q = 0; q < 16; ++q) av[q] = raw[q];
        } else {
#pragma unroll
            for (int q = 0; q < 16; ++q) T[2 * q + h][l32] = raw[q];
            wave_lds_sync();
            // A operand A22(ri, J*32 + k) = A(J*32 + k, ri): T[l32][k]; the
            // diagonal tile's upper part mirrored from its lower part
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int k = 2 * q + h;
                av[q] = (J > I || k >= l32) ? T[l32][k] : T[k][l32];
            }
            wave_lds_sync();
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[q], bv[q], acc, 0, 0, 0);
    };
    float b0[16], r0v[16], b1[16], r1v[16];
    load(wave, b0, r0v);
    for (int J = wave; J < nbt; J += 2 * WV) {
        tile(J, b0, r0v, b1, r1v);
        if (J + WV >= nbt) break;
        tile(J + WV, b1, r1v, b0, r0v);
    }
    // acc(i, p): lane l holds column p = l32, rows 8 a + 4 h + c
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < 16; ++q) T[8 * (q >> 2) + 4 * h + (q & 3)][l32] = acc[q];
    __syncthreads();
    for (int e = tid; e < 32 * 32; e += 64 * WV) {
        const int i = e / 32, p = e % 32, r = I * 32 + i;
        float t = tl[0][i][p];
#pragma unroll
        for (int w = 1; w < WV; ++w) t += tl[w][i][p];
        if (r < m) P[size_t(r) * 2 * NB + NB + p] = t;
    }
}

// W = X - Y (Yh^T X) / 2 in place of X, one workgroup per matrix: the 32 x 32
// product M = Yh^T X with the rows split over the waves in blocks of 32 (its
// partial sums added in wave order), then each wave's blocks of W, formed
// transposed (MFMA row = column of W) so that a lane holds 4 consecutive
// columns of its row.  32x32x2 FP32 MFMA; lane half h takes positions 16 h + q
// of a K = 32 sum.  As two launches of the general product, one workgroup of
// 64 x 64 tiles each for the first: 54 us for one matrix of N = 2048; this
// takes 22 us.
__global__ void __launch_bounds__(kPanNT) sb_w_kernel(int n, int r0, const float* __restrict__ Yhall,
                                                      float* __restrict__ Pall) {
    constexpr int NB = kBandNB;
    __shared__ float red[kPanNW][NB][NB + 1];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = n - r0, nblk = (m + 31) / 32;
    const float* Yh = Yhall + size_t(b) * n * NB;
    float* P = Pall + size_t(b) * n * 2 * NB + size_t(r0) * 2 * NB;
    floatx16 acc;
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.f;
    float a0[16], x0[16];
    auto load = [&](int blk) {  // rows past m: clamped, Yh zeroed below
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int r = min(blk * 32 + 2 * q + h, m - 1);
            a0[q] = Yh[size_t(r) * NB + l32];
            x0[q] = P[size_t(r) * 2 * NB + NB + l32];
        }
    };
    if (wave < nblk) load(wave);
    for (int blk = wave; blk < nblk; blk += kPanNW) {
        float a[16], x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            a[q] = (blk * 32 + 2 * q + h < m) ? a0[q] : 0.f;
            x[q] = x0[q];
        }
        if (blk + kPanNW < nblk) load(blk + kPanNW);
#pragma unroll
        for (int q = 0; q < 16; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q], x[q], acc, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) red[wave][8 * (q >> 2) + 4 * h + (q & 3)][l32] = acc[q];
    __syncthreads();
    for (int e = tid; e < NB * NB; e += kPanNT) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kPanNW; ++w) t += red[w][e / NB][e % NB];
        red[0][e / NB][e % NB] = -0.5f * t;  // (an element is read and written by one thread)
    }
    __syncthreads();
    float mk[16];  // -M(16 h + q, l32) / 2
#pragma unroll
    for (int q = 0; q < 16; ++q) mk[q] = red[0][16 * h + q][l32];
    for (int blk = wave; blk < nblk; blk += kPanNW) {
        const int r = blk * 32 + l32;
        float* row = P + size_t(min(r, m - 1)) * 2 * NB;
        float y[16];
        floatx16 d;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 t = *reinterpret_cast<const float4*>(row + 16 * h + 4 * q);
            y[4 * q] = t.x;
            y[4 * q + 1] = t.y;
            y[4 * q + 2] = t.z;
            y[4 * q + 3] = t.w;
            const float4 u = *reinterpret_cast<const float4*>(row + NB + 8 * q + 4 * h);
            d[4 * q] = u.x;
            d[4 * q + 1] = u.y;
            d[4 * q + 2] = u.z;
            d[4 * q + 3] = u.w;
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) d = __builtin_amdgcn_mfma_f32_32x32x2f32(mk[q], y[q], d, 0, 0, 0);
        if (r < m) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4*>(row + NB + 8 * q + 4 * h) =
                    float4{d[4 * q], d[4 * q + 1], d[4 * q + 2], d[4 * q + 3]};
        }
    }
}

// Word 3 of a raw buffer resource on gfx9-family GPUs (32-bit data format,
// no swizzle, range checking on offsets).
constexpr int kBufferWord3 = 0x00020000;

// A22 -= W Y^T + Y W^T on the lower triangle, from the row-major panel P
// (P[r * 2NB + k]: Y(r, k) for k < NB, W(r, k - NB) after).  Workgroup x owns
// block row br = x, wave w its block columns bc = w, w + 4, ... <= br.
// The tile is formed transposed (MFMA row = column of A, MFMA column = row
// of A) so that lanes run along rows of the column-major A; step s of the
// K = 2NB sum takes panel position 32 h + s from lane half h, the A operand
// from the panel row of the tile's column at that position, the B operand
// from the panel row of the tile's row at the swapped half (k ^ NB).  The
// next tile's A values and operand are in flight while a tile's MFMA chain
// runs.  Bound by memory (each element of A22 read and written, 3.3 TB/s) where
// there are many matrices.  With a block row per wave 63 calls for one matrix of N = 2048 took
// 3.48 ms, 24 matrices of N = 3072 12.6, 48 of N = 768 0.62; with 4 waves to a row
// 1.20, 10.0, 0.50.
__global__ void __launch_bounds__(64 * kSyWaves) sb_syr2k_kernel(int n, int ld, int r0, float* __restrict__ Aall,
                                                       const float* __restrict__ Pall, int batch) {
    constexpr int NB = kBandNB, PW = 2 * kBandNB, WV = kSyWaves;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = n - r0, nbt = (m + 31) / 32;
    int x, b;
    if (!xcd_slot(nbt, batch, x, b)) return;
    const int br = x;
    if (br >= nbt || wave > br) return;
    float* A = Aall + size_t(b) * n * ld + size_t(r0) * ld + r0;
    const float* P = Pall + size_t(b) * n * PW + size_t(r0) * PW;
    const int h = lane >> 5, l32 = lane & 31;
    const int r = br * 32 + l32;  // row of A22 this lane's column of the output holds
    // Loads are issued with row and column indices clamped below m and never
    // masked: an output element past m, or above the diagonal, is not stored,
    // and no K index runs past the panel.
    auto panel_row = [&](int row, int half, float (&v)[32]) {
        const float4* src = reinterpret_cast<const float4*>(P + size_t(min(row, m - 1)) * PW + half * NB);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 t = src[q];
            v[4 * q] = t.x;
            v[4 * q + 1] = t.y;
            v[4 * q + 2] = t.z;
            v[4 * q + 3] = t.w;
        }
    };
    // A22 of this matrix as a raw buffer (offsets in bytes, at most n * ld * 4)
    const __amdgpu_buffer_rsrc_t rsA = __builtin_amdgcn_make_buffer_rsrc(A, 0, 0x7fffffff, kBufferWord3);
    const int rc = min(r, m - 1);
    auto load_old = [&](int bc, float (&o)[16]) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int c = bc * 32 + 8 * (q >> 2) + 4 * h + (q & 3);
            o[q] = A[size_t(min(c, m - 1)) * ld + rc];
        }
    };
    float bv[32];
    panel_row(r, 1 - h, bv);
    // tile bc from (av, old) while the next tile's operand and old values are
    // read into (an, on) (past the last tile: clamped reads, never used); the
    // two buffer pairs alternate, so no copy waits for a read in flight
    auto tile = [&](int bc, float (&av)[32], float (&old)[16], float (&an)[32], float (&on)[16]) {
        panel_row((bc + WV) * 32 + l32, h, an);
        load_old(bc + WV, on);
        __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the products
        floatx16 acc;
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[q] = 0.f;
#pragma unroll
        for (int q = 0; q < 32; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[q], bv[q], acc, 0, 0, 0);
        // buffer stores, an element outside the lower triangle of A22 given
        // an offset past the buffer's range (the store is dropped): no branch,
        // so the count of memory operations in flight stays known and no wait
        // lands on the reads of the next tile
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int c = bc * 32 + 8 * (q >> 2) + 4 * h + (q & 3);
            const bool ok = c < m && r < m && r >= c;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(old[q] - acc[q]), rsA,
                                                  ok ? (c * ld + r) * 4 : int(0x80000000), 0, 0);
        }
    };
    float a0[32], o0[16], a1[32], o1[16];
    panel_row(wave * 32 + l32, h, a0);
    load_old(wave, o0);
    for (int bc = wave; bc <= br; bc += 2 * WV) {
        tile(bc, a0, o0, a1, o1);
        if (bc + WV > br) break;
        tile(bc + WV, a1, o1, a0, o0);
    }
}

// Zero the band rows, then the last (unfactored) diagonal block's lower
// triangle into them: columns jl..n-1, rows jl..n-1 (at most NB + 1 of them).
__global__ void __launch_bounds__(256) sb_band_zero_kernel(int n, float* __restrict__ BNDall) {
    const int b = blockIdx.y;
    const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (e >= int64_t(n) * kBandW) return;
    BNDall[size_t(b) * n * kBandW + e] = 0.f;
}
__global__ void __launch_bounds__(256) sb_band_tail_kernel(int n, int ld, int jl, const float* __restrict__ Aall,
                                                           float* __restrict__ BNDall) {
    const int b = blockIdx.x;
    const float* A = Aall + size_t(b) * n * ld;
    float* BND = BNDall + size_t(b) * n * kBandW;
    const int k = n - jl;
    for (int q = threadIdx.x; q < k * k; q += 256) {
        const int i = q / k, c = q % k;
        if (c <= i) BND[size_t(jl + i) * kBandW + (i - c)] = A[size_t(jl + c) * ld + jl + i];
    }
}

int sy2sb(int batch, int n, int ld, float* A, float* BND, float* tau, float* P, float* Yh, hipStream_t s) {
    constexpr int NB = kBandNB;
    if (n > sb_max_n()) return fail(CIR_ERR_ARG, "sy2sb: n too large for the register panel");
    {
        dim3 grid(unsigned(ceil_div(int64_t(n) * kBandW, 256)), unsigned(batch));
        hipLaunchKernelGGL(sb_band_zero_kernel, grid, dim3(256), 0, s, n, BND);
        CIR_CHECK_LAUNCH();
    }
    int j0 = 0;
    for (; j0 + NB < n - 1; j0 += NB) {
        const int r0 = j0 + NB, m = n - r0;
        const int rpt = int(ceil_div(m, kPanNT));
        auto panel = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(unsigned(batch)), dim3(kPanNT), 0, s, n, ld, j0, A, BND, tau, P, Yh);
        };
        switch (rpt) {
            case 1: panel(sb_panel_kernel<1>); break;
            case 2: panel(sb_panel_kernel<2>); break;
            case 3: panel(sb_panel_kernel<3>); break;
            case 4: panel(sb_panel_kernel<4>); break;
            case 5: panel(sb_panel_kernel<5>); break;
            default: panel(sb_panel_kernel<6>); break;
        }
        CIR_CHECK_LAUNCH();
        const int nbt = int(ceil_div(m, 32));
        const dim3 grid = xcd_grid(nbt, batch);
        // X = A22 Yh into the W half of P
        hipLaunchKernelGGL(sb_symm_kernel, grid, dim3(64 * kSyWaves), 0, s, n, ld, r0, A,
                           Yh, P, batch);
        CIR_CHECK_LAUNCH();
        // W = X - Y (Yh^T X) / 2 in place of X
        hipLaunchKernelGGL(sb_w_kernel, dim3(unsigned(batch)), dim3(kPanNT), 0, s, n, r0, Yh, P);
        CIR_CHECK_LAUNCH();
        // A22 -= W Y^T + Y W^T (lower triangle)
        hipLaunchKernelGGL(sb_syr2k_kernel, grid, dim3(64 * kSyWaves), 0, s, n, ld, r0, A, P,
                           batch);
        CIR_CHECK_LAUNCH();
    }
    // the last diagonal block (n - j0 <= NB + 1 rows) is already banded
    hipLaunchKernelGGL(sb_band_tail_kernel, dim3(unsigned(batch)), dim3(256), 0, s, n, ld, j0, A, BND);
    CIR_CHECK_LAUNCH();
    return CIR_OK;
}

}  // namespace cir

namespace cir {

// ---------------------------------------------------------------------------
// Stage 2: band -> tridiagonal by bulge chasing.
// ---------------------------------------------------------------------------
constexpr int kSbG = 8;                  // sweeps per group = waves per workgroup
constexpr int kSbNT = 64 * kSbG;
constexpr int kSbWR = 512;               // window rows (power of two)
constexpr int kSbWP = kBandW;            // window row pitch (floats)
// window, per-wave task scratch (v and a per-lane sink),
// and one 16-byte sink for the read-ahead pieces of threads with no row to add
constexpr int kSbScratch = kBandNB + 64;
constexpr size_t kSbSmemFloats = size_t(kSbWR) * kSbWP + size_t(kSbG) * kSbScratch + 4;
static_assert(kBandNB * (kBandW / 4) <= kSbNT, "one step's new band rows must fit one 16-byte piece per thread");
static_assert((2 * kSbG - 1) * kBandNB + kBandNB <= kSbWR, "window must hold a step's rows plus the read-ahead");


// Row r of a group's band is stream row v = r + off (SbStream), which sits in
// window row v mod kSbWR; its element (r, c), r - c < kBandW, is r - c floats
// into that row.
// The groups' band rows as one stream.  Group g (sweeps kSbG g ..) starts at
// step st(g) and its row r is stream row r - kSbG g + 32 st(g), so that task k
// of the group's wave j, at step t = st(g) + k + 2 j, works on the 32 stream
// rows from 32 (t - 2 j) + j + 1, whatever the group.  The next group starts
// once wave 0 is through this one's rows, and no sooner than kSbGap steps
// later: its tasks then follow the last wave's (a lag of 2 kSbG steps), and
// its reads of the band, two steps ahead, follow this group's write-backs.
constexpr int kSbGap = 2 * kSbG + 2;
static_assert(kBandNB == 32, "stream rows are counted in steps of 32");
struct SbStream {
    int g = 0, st = 0, next;  // group, its first step and the next group's
    __device__ __forceinline__ explicit SbStream(int n) { next = gap(n, 0); }
    static __host__ __device__ __forceinline__ int gap(int n, int g) { return max(kSbGap, (n - kSbG * g + 31) / 32); }
    __device__ __forceinline__ void advance(int n) {
        ++g;
        st = next;
        next += gap(n, g);
    }
    // band row of stream row v, which lies in this group or the next one
    __device__ __forceinline__ int row(int v) const {
        return v < 32 * next ? v - 32 * st + kSbG * g : v - 32 * next + kSbG * (g + 1);
    }
    // whether v is a row of a group with sweeps (between groups there may be none)
    __device__ __forceinline__ bool has(int n, int v) const {
        return kSbG * (g + (v >= 32 * next ? 1 : 0)) < n - 2 && row(v) < n;
    }
};

// Sum of a value over the two lanes i and i + 32 of a wave, in both.
__device__ __forceinline__ float half_pair_sum(float x) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}
// The value of lane i (i < 32) in lanes i and i + 32.
__device__ __forceinline__ float from_low_half(float x) {
    return __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false)[0]);
}

// Sum over the 32 lanes of each half wave, in every lane of the half.
__device__ __forceinline__ float half_sum(float x) {
    x = brow_sum16(x);
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

// Column of the block that register c of a lane of half h holds (the row that
// register c of a 32x32 MFMA accumulator holds there).
__device__ __forceinline__ constexpr int sb_col(int c, int h) { return 8 * (c >> 2) + 4 * h + (c & 3); }

// One wave's share of a bulge-chasing step: task (s, k) of its sweep.
// Lane l: row i = l & 31 of the task's blocks and 16 of their columns, sb_col(c,
// l >> 5).  pv / pvi / ptau: the sweep's previous reflector (at this lane's 16
// columns, at column i, its factor), replaced by this task's; q2val: this task's
// reflector as a Q2 block column.  The wave's scratch sc holds v and a per-lane
// sink for masked-off stores.
// FULL: a block of 32 rows, every task but a sweep's last.  The last one's
// lanes outside the block read a row inside it and discard the value.  All the
// window's reads are issued together at the start; read where they are used,
// the compiler put each of the masked ones into a branch of its own with a wait
// behind it (16 LDS latencies per task).  dofs: window offset of D(max(i, j),
// min(i, j)) for column j = sb_col(c, h), against the block's first row; rows
// are 64 floats, so an offset past the window's end wraps with a mask.
// Issue-bound (two waves per SIMD): the block below, B, is read a second time
// by columns (tb: rows sb_col(c, h) of column i), so that v^T B is a sum within
// the lane like the other products, with the right application's part (v . f)
// pv taken off afterwards, and the two rank-one updates of either block are one
// 32x32x2 MFMA.  With v^T B reduced across lanes after the right application,
// both reduced vectors handed round through LDS and the updates on the vector
// units: 23.4 ms for one matrix of N = 2048, 4.4 for 48 of N = 766; this takes
// 19.7 and 3.8.
template <bool FULL>
__device__ __forceinline__ void sb_task(int n, int s, int k, int off, float* w, float* sc, const int (&dofs)[16],
                                        float (&pv)[16], float& pvi, float& ptau, float& q2val, int lane) {
    constexpr int NB = kBandNB;
    constexpr int WMASK = kSbWR * kSbWP - 1;
    float* vs = sc;
    float* sink = sc + NB + lane;
    const int i = lane & 31, h = lane >> 5;
    const int r0 = s + 1 + k * NB;
    const int len = FULL ? NB : min(NB, n - r0);
    const bool rowok = FULL || i < len;
    const int R = ((r0 + off) & (kSbWR - 1)) * kSbWP;  // window offset of the block's first row
    // this lane's row (clamped into the block): element (row, c) at wr[row - c]
    const int ic = FULL ? i : min(i, len - 1);
    float* const wr = w + ((R + ic * kSbWP) & WMASK);
    floatx16 bk, dd;
    float tb[16];
    float x = 0.f;
    if (k == 0) {
        x = wr[ic + 1];  // column s
    } else {
        // the block below the previous one
        const float* bp = wr + (NB + ic - 4 * h - 27);
#pragma unroll
        for (int c = 0; c < 16; ++c) bk[c] = bp[27 - sb_col(c, 0)];
    }
    // the diagonal block D (rows/cols r0 .. r0+len-1), both triangles, from
    // its lower triangle, and B by columns
    if (FULL && R <= (kSbWR - NB) * kSbWP) {  // no row wraps
        const float* base = w + R;
        const float* tp = base + (NB - i + 4 * h * (kSbWP + 1));
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            dd[c] = base[dofs[c]];
            tb[c] = tp[sb_col(c, 0) * (kSbWP + 1)];
        }
    } else {
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int j = sb_col(c, h), jc = FULL ? j : min(j, len - 1);
            if constexpr (FULL) {
                dd[c] = w[(R + dofs[c]) & WMASK];
            } else {
                const int ra = min(max(i, j), len - 1), cb = min(min(i, j), ra);
                dd[c] = w[(R + ra * kSbWP + ra - cb) & WMASK];
            }
            tb[c] = w[((R + jc * kSbWP) & WMASK) + NB + jc - i];
        }
    }
    if constexpr (!FULL) {
#pragma unroll
        for (int c = 0; c < 16; ++c) {  // read above, masked here
            float t = dd[c];
            asm volatile("" : "+v"(t));
            dd[c] = (rowok && sb_col(c, h) < len) ? t : 0.f;
        }
        if (k == 0) {
            x = rowok ? x : 0.f;
        } else {
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                float t = bk[c];
                asm volatile("" : "+v"(t));
                bk[c] = rowok ? t : 0.f;
            }
        }
    }
    float f = 0.f;
    if (k > 0) {
        // the previous reflector from the right (this fills the bulge): B -= f
        // pv^T, applied with the new one's below; of it the first column here
        // (pv(0) = 1), from the h = 0 lanes
        float u0 = 0.f, u1 = 0.f;
#pragma unroll
        for (int c = 0; c < 16; c += 2) {
            u0 += bk[c] * pv[c];
            u1 += bk[c + 1] * pv[c + 1];
        }
        f = ptau * half_pair_sum(u0 + u1);
        x = from_low_half(bk[0]) - f;
    }
    // reflector annihilating x[1..len) (x is the same in both halves)
    const float sigma = half_sum((i >= 1 && rowok) ? x * x : 0.f);
    const float alpha = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 0));
    float tau = 0.f, beta = alpha, scale = 0.f;
    if (__builtin_amdgcn_readfirstlane(__float_as_int(sigma)) != 0 &&
        !sb_householder(alpha, sigma, beta, tau, scale)) {
        const float xu = x * kSbUp;
        sb_householder_up(alpha, half_sum((i >= 1 && rowok) ? xu * xu : 0.f), beta, tau, scale);
    }
    const float vi = (i == 0) ? 1.f : (rowok ? x * scale : 0.f);
    if (h == 0) vs[i] = vi;
    wave_lds_sync();
    float vj[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 t = *reinterpret_cast<const float4*>(vs + 8 * q + 4 * h);
        vj[4 * q] = t.x;
        vj[4 * q + 1] = t.y;
        vj[4 * q + 2] = t.z;
        vj[4 * q + 3] = t.w;
    }
    // D: p = tau D v, K = -tau/2 p.v, w = p + K v
    float p0a = 0.f, p1a = 0.f;
#pragma unroll
    for (int c = 0; c < 16; c += 2) {
        p0a += dd[c] * vj[c];
        p1a += dd[c + 1] * vj[c + 1];
    }
    const float pp = tau * half_pair_sum(p0a + p1a);
    if (k > 0) {
        // the new reflector from the left on the block's other columns: w =
        // B^T v - (v . f) pv in lane i for column i, B -= f pv^T + tau v w^T
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int c = 0; c < 16; c += 2) {
            s0 += tb[c] * vj[c];
            s1 += tb[c + 1] * vj[c + 1];
        }
        const float vf = half_sum(vi * f);
        const float tw = half_pair_sum(s0 + s1) - vf * pvi;
        bk = __builtin_amdgcn_mfma_f32_32x32x2f32(h == 0 ? pvi : tw, h == 0 ? -f : -tau * vi, bk, 0, 0, 0);
    }
    const float kk = half_sum(pp * vi);  // (pp is the same in both halves)
    const float wi = pp - 0.5f * tau * kk * vi;
    dd = __builtin_amdgcn_mfma_f32_32x32x2f32(h == 0 ? vi : wi, h == 0 ? -wi : -vi, dd, 0, 0, 0);
    if (k > 0) {
        if (h == 0) bk[0] = (i == 0) ? beta : 0.f;  // the annihilated column
        if (rowok) {
            float* bq = wr + (NB + ic - 4 * h - 27);
#pragma unroll
            for (int c = 0; c < 16; ++c) bq[27 - sb_col(c, 0)] = bk[c];
        }
    } else if (h == 0 && rowok) {
        wr[ic + 1] = (i == 0) ? beta : 0.f;
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        const int j = sb_col(c, h);
        float* dst = (rowok && j <= i) ? wr + (i - j) : sink;
        *dst = dd[c];
    }
    // the reflector as its Q2 block column (48 rows, zero outside [jq, jq +
    // len)): lane r < 48 holds row r
    const int jq = s % kQ2G;
    const int rr = lane - jq;
    const float vv = __shfl(vi, rr & 31, 64);  // every lane takes part in the shuffle
    q2val = (rr >= 0 && rr < NB) ? vv : 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c) pv[c] = vj[c];
    pvi = vi;
    ptau = tau;
    wave_lds_sync();
}

// Band -> tridiagonal for one matrix per workgroup.  Sweep s annihilates
// column s below the subdiagonal; its task k (rows s+1+k NB ..) applies the
// previous reflector from the right to the block below it, annihilates the
// block's first column with a new reflector, applies that from the left to
// the rest of the block and to the diagonal block from both sides.  The
// sweeps of a group run one per wave, task k of wave j at step k + 2 j: the
// tasks of one step touch disjoint elements, and a task runs after every
// task of the sweep before it that touches its rows.  A wave that is through
// its sweep goes on with the next group's (SbStream), so the pipeline of
// waves fills and drains once per matrix and not once per group (n = 2048:
// 8.3 instead of 11.9 thousand steps).  The rows the waves need at a step (at
// most (2 kSbG - 1) NB of them) live in a circular LDS window over the stream;
// 32 rows enter it per step, read from the band two steps ahead, and 32 leave.
// Bound by the latency and issue of a step's tasks, two waves per SIMD.
__global__ void __launch_bounds__(kSbNT) sb2st_kernel(int n, float* __restrict__ BNDall, float* __restrict__ dall,
                                                       float* __restrict__ eall, float* __restrict__ Q2all) {
    constexpr int NB = kBandNB;
    extern __shared__ __align__(16) float sb_smem[];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* BND = BNDall + size_t(b) * n * kBandW;
    float* Q2 = Q2all + size_t(b) * q2_block_offset(n, q2_groups(n)) * kQ2BlockFloats;
    float* const win = sb_smem;
    float* sc = sb_smem + size_t(kSbWR) * kSbWP + wave * kSbScratch;
    const int nsweep = n - 2;

    if (nsweep > 0) {
        // steps until the last task of the last group
        const int glast = (nsweep - 1) / kSbG;
        int nstep = 0;
        {
            int st = 0;
            for (int g = 0; g < glast; ++g) st += SbStream::gap(n, g);
            for (int s = kSbG * glast; s < nsweep; ++s) nstep = max(nstep, st + 2 * (s - kSbG * glast) + sb_tasks(n, s));
        }
        // this thread's 16-byte piece of the 32 rows entering or leaving
        const int pr = tid / (kBandW / 4), pc = (tid % (kBandW / 4)) * 4;
        float* sink = sb_smem + kSbSmemFloats - 4;
        // entering: stream rows 32 c + 1 .. 32 c + 32 before step c (row 0
        // before step 0); leaving: 32 (t - 14) + 8 .. + 39 after step t
        SbStream in(n), out(n);
        auto read = [&](int c, bool& ok) {  // (c never decreasing, by one)
            if (in.next <= c) in.advance(n);
            const int v = 32 * c + 1 + pr;
            ok = in.has(n, v);
            return *reinterpret_cast<const float4*>(BND + size_t(ok ? in.row(v) : n - 1) * kBandW + pc);
        };
        auto enter = [&](int c, bool ok, const float4& x) {
            *reinterpret_cast<float4*>(ok ? win + ((32 * c + 1 + pr) & (kSbWR - 1)) * kSbWP + pc : sink) = x;
        };
        auto leave = [&](int t) {
            const int v0 = 32 * (t - 2 * (kSbG - 1)) + kSbG;
            if (v0 + 31 < 0) return;
            if (32 * out.next <= v0) out.advance(n);
            const int v = v0 + pr;
            if (v >= 0 && out.has(n, v))
                *reinterpret_cast<float4*>(BND + size_t(out.row(v)) * kBandW + pc) =
                    *reinterpret_cast<const float4*>(win + (v & (kSbWR - 1)) * kSbWP + pc);
        };
        // (each piece is read and written by every thread, so that the wait
        // for it is on every path: a thread with no row reads the last row
        // and writes the sink)
        if (pr == 0)
            *reinterpret_cast<float4*>(win + pc) = *reinterpret_cast<const float4*>(BND + pc);  // row 0
        bool pre;
        {
            const float4 x = read(0, pre);
            enter(0, pre, x);
        }
        float4 pf = read(1, pre);
        float pv[16], pvi = 0.f, ptau = 0.f;
#pragma unroll
        for (int c = 0; c < 16; ++c) pv[c] = 0.f;
        int dofs[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int i = lane & 31, j = sb_col(c, lane >> 5);
            dofs[c] = max(i, j) * kSbWP + abs(i - j);
        }
        SbStream my(n);
        int64_t q2o = 0;  // first Q2 block of this wave's sweep
        for (int t = 0; t < nstep; ++t) {
            __syncthreads();
            int s = kSbG * my.g + wave, k = t - my.st - 2 * wave;
            if (k >= sb_tasks(n, s) && k >= 0 && my.g < glast && t >= my.next + 2 * wave) {
                // the blocks of kQ2G sweeps share their group's block positions
                if ((my.g + 1) % (kQ2G / kSbG) == 0) q2o += sb_tasks(n, (kSbG * my.g / kQ2G) * kQ2G);
                my.advance(n);
                s = kSbG * my.g + wave;
                k = t - my.st - 2 * wave;
            }
            const bool act = s < nsweep && k >= 0 && k < sb_tasks(n, s);
            float q2val = 0.f;
            if (act) {
                const int off = 32 * my.st - kSbG * my.g;
                if (s + 1 + (k + 1) * NB <= n)
                    sb_task<true>(n, s, k, off, win, sc, dofs, pv, pvi, ptau, q2val, lane);
                else
                    sb_task<false>(n, s, k, off, win, sc, dofs, pv, pvi, ptau, q2val, lane);
            }
            __syncthreads();
            // the rows read ahead are written before this step's stores are
            // issued, so waiting for the read waits only for memory operations
            // issued before the tasks
            enter(t + 1, pre, pf);
            leave(t);
            if (act) {
                float* blk = Q2 + (q2o + k) * kQ2BlockFloats;
                const int jq = s % kQ2G;
                if (lane < kQ2R) blk[jq * kQ2R + lane] = q2val;
                if (lane == 0) blk[kQ2R * kQ2G + jq] = ptau;
            }
            pf = read(t + 2, pre);
        }
        // the rows still in the window
        __syncthreads();
        for (int t = nstep; t < nstep + 2 * kSbG; ++t) leave(t);
    }
    __syncthreads();
    // d and e of T from the band
    float* d = dall + size_t(b) * n;
    float* e = eall + size_t(b) * n;
    for (int i = tid; i < n; i += kSbNT) {
        d[i] = BND[size_t(i) * kBandW];
        e[i] = (i + 1 < n) ? BND[size_t(i + 1) * kBandW + 1] : 0.f;
    }
}

// (the documented range of the deterministic key, short of sb_max_n())
int deterministic_eigh_max() { return 2080; }
bool deterministic_eigh_size(int n) { return n >= 2 * kBandNB + 2 && n <= deterministic_eigh_max(); }

int sb2st(int batch, int n, float* BND, float* d, float* e, float* Q2, hipStream_t s) {
    if (n < 1) return fail(CIR_ERR_ARG, "sb2st: bad size");
    const size_t sm = kSbSmemFloats * sizeof(float);
    CIR_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&sb2st_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(sm)));
    hipLaunchKernelGGL(sb2st_kernel, dim3(unsigned(batch)), dim3(kSbNT), sm, s, n, BND, d, e, Q2);
    CIR_CHECK_LAUNCH();
    return CIR_OK;
}

}  // namespace cir

namespace cir {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Q2: the bulge-chasing reflectors as compact-WY blocks.
// ---------------------------------------------------------------------------

// Group and position of block q of a matrix.
__device__ __forceinline__ void q2_block_gk(int n, int64_t q, int* g, int* k) {
    int lo = 0, hi = q2_groups(n);  // the last group that starts at or before q
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (q2_block_offset(n, mid) <= q)
            lo = mid;
        else
            hi = mid;
    }
    *g = lo;
    *k = int(q - q2_block_offset(n, lo));
}

// Four values as the 16 bytes of their BF16 parts: hi (8 bytes), then lo.
__device__ __forceinline__ float4 q2_split4(const float (&v)[4]) {
    unsigned h0, l0, h1, l1;
    split_bf16x2(v[0], v[1], h0, l0);
    split_bf16x2(v[2], v[3], h1, l1);
    return float4{__uint_as_float(h0), __uint_as_float(h1), __uint_as_float(l0), __uint_as_float(l1)};
}

// Per block (one wave): reflectors that do not exist (sweeps past n - 3, or
// past their last task) are zeroed; T is formed (forward, columnwise), and V
// and -V T are stored in the operand order of the MFMA products that apply the
// block (Z <- Z + (-V T) (V^T Z)), 16 bytes a lane and load: register 4 q + e of
// lane (lq, l16) holds V(16 q + 4 lq + e, l16), V^T as the A operand of the W
// product, and of -V T, as the A operand of the update, NV(16 q + l16, 4 e + lq)
// for FP32 16x16x4 steps and NV(16 q + l16, 4 lq + e) for split-BF16 products.
// The split-BF16 operands are split here, once per block instead of once per
// block and slab: each 16 bytes hold the hi and lo parts of 4 values.  V_op
// replaces V in place.
// V^T V and (-V T)^T are FP32 MFMA products, the second with T's columns in the
// order that leaves the result in that layout; T's rows are a recursion in one
// lane each.  With every product a sum over LDS, a thousand LDS instructions a
// block, 256 matrices of N = 2048 took 6.2 ms; this takes 2.4, half of it memory.
__global__ void __launch_bounds__(64) q2_prep_kernel(int n, int64_t nblk, float* __restrict__ Q2all, int bf16) {
    __shared__ float sv[kQ2R][kQ2G + 1], st[kQ2G][kQ2G + 1], stau[kQ2G];
    __shared__ __align__(16) float sgm[kQ2G][kQ2G + 4];
    const int64_t q = blockIdx.x;
    const int b = blockIdx.y, lane = threadIdx.x, l16 = lane & 15, lq = lane >> 4;
    if (q >= nblk) return;
    float* blk = Q2all + (size_t(b) * nblk + q) * kQ2BlockFloats;
    float* V = blk;
    float* tau = blk + kQ2R * kQ2G;
    float* NVT = tau + kQ2G;
    int g, k;
    q2_block_gk(n, q, &g, &k);
#pragma unroll
    for (int u = 0; u < kQ2R * kQ2G / 64; ++u) {
        const int e = lane + 64 * u, j = e / kQ2R, r = e % kQ2R;
        const float v = V[e];
        sv[r][j] = k < sb_tasks(n, g * kQ2G + j) ? v : 0.f;
    }
    if (lane < kQ2G) {
        const float t = tau[lane];
        stau[lane] = k < sb_tasks(n, g * kQ2G + lane) ? t : 0.f;
    }
    __syncthreads();
    float vs[12];
#pragma unroll
    for (int e = 0; e < 12; ++e) vs[e] = sv[16 * (e / 4) + 4 * lq + e % 4][l16];
    floatx4 gm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 12; ++e) gm = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[e], vs[e], gm, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) sgm[4 * lq + r][l16] = gm[r];
    __syncthreads();
    // T(0:l, l) = -tau_l T(0:l, 0:l) G(0:l, l), lane l16 the row l16 (G is
    // symmetric: its column l is row l)
    float Tr[kQ2G];
#pragma unroll
    for (int l = 0; l < kQ2G; ++l) {
        float acc = 0.f;
#pragma unroll
        for (int c = 0; c < l; ++c) acc += Tr[c] * sgm[l][c];
        const float tl = stau[l];
        Tr[l] = l16 == l ? tl : (l16 < l ? -tl * acc : 0.f);
    }
#pragma unroll
    for (int l = 0; l < kQ2G; ++l)
        if (lq == l / 4) st[l16][l] = Tr[l];
    __syncthreads();
    const int jt = bf16 ? l16 : 4 * (l16 & 3) + (l16 >> 2);
    float tt[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) tt[s] = -st[4 * s + lq][jt];
    float4 vp[3];
#pragma unroll
    for (int rt = 0; rt < 3; ++rt) {
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(tt[s], sv[16 * rt + l16][4 * s + lq], acc, 0, 0, 0);
        const float v[4] = {vs[4 * rt], vs[4 * rt + 1], vs[4 * rt + 2], vs[4 * rt + 3]};
        const float w[4] = {acc[0], acc[1], acc[2], acc[3]};
        float4* vo = reinterpret_cast<float4*>(V) + 64 * rt + lane;
        float4* wo = reinterpret_cast<float4*>(NVT) + 64 * rt + lane;
        if (bf16) {
            vp[rt] = q2_split4(v);
            *wo = q2_split4(w);
        } else {
            *vo = float4{v[0], v[1], v[2], v[3]};
            *wo = float4{w[0], w[1], w[2], w[3]};
        }
    }
    if (bf16) {
        // V: the hi parts of row tiles 0 and 1, their lo parts, both of tile 2
        float4* vo = reinterpret_cast<float4*>(V) + lane;
        vo[0] = float4{vp[0].x, vp[0].y, vp[1].x, vp[1].y};
        vo[64] = float4{vp[0].z, vp[0].w, vp[1].z, vp[1].w};
        vo[128] = vp[2];
    }
    if (lane < kQ2G) tau[lane] = stau[lane];
}

typedef short short8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned long long q2_parts __attribute__((ext_vector_type(2)));
// Four values split into their BF16 parts: lo's four and hi's four, 8 bytes each.
__device__ __forceinline__ q2_parts q2_split(floatx4 v) {
    unsigned h0, l0, h1, l1;
    split_bf16x2(v[0], v[1], h0, l0);
    split_bf16x2(v[2], v[3], h1, l1);
    return q2_parts{l0 | (unsigned long long)(l1) << 32, h0 | (unsigned long long)(h1) << 32};
}
__device__ __forceinline__ short8 q2_lo_hi(q2_parts p) { return __builtin_bit_cast(short8, p); }
__device__ __forceinline__ short8 q2_hi_lo(q2_parts p) { return __builtin_bit_cast(short8, q2_parts{p[1], p[0]}); }
__device__ __forceinline__ short8 q2_ops(float4 a) {
    return __builtin_bit_cast(short8, floatx4{a.x, a.y, a.z, a.w});
}
__device__ __forceinline__ floatx4 q2_mfma32(short8 a, short8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Z <- Q2 Z on one slab of 16 CT columns of one matrix.  Blocks apply group by
// group from the last group g = NG - 1 (gi = NG - 1 - g ascending), positions
// k in ascending order; block (g, k) covers the row tiles (16 rows each, tile
// i from row 16 i + 1) g + 2 k .. g + 2 k + 2.
//
// The rows stream through the workgroup's waves: wave w takes the groups gi =
// w, w + NW, ..., holds the three tiles of its block in registers, and after
// block k passes the first two, which its group does not touch again, on as
// slot k to the next wave, whose own block k needs just them behind the tile
// it carries (its group starts one tile earlier; that first tile no earlier
// group touches, so it comes from Z).  Slots go through short queues in LDS
// (kQ2Fifo deep); the last wave's go back to Z and the first wave reads them
// there for the following round of groups.  A group has as many slots as
// blocks, ceil of its tiles / 2, and its successor at most one more, for which
// the rows are past the end: zeros.
//
// Every wait is for a slot of an earlier group or for the room that a later
// group's reads leave, the waves take their blocks in the order of (round,
// k), and a group of the first wave waits for nothing of its own round, so
// every wait ends (and is bounded all the same: one that ran far past any
// block's time marks the slab, which is then written as NaN).
//
// Bound by the issue of the split's vector instructions (70% of the cycles)
// beside the MFMAs.  A block's operands, 6 KB, are read per wave straight into
// registers a block ahead, and serve all of the wave's columns: they pass the
// CU's vector cache and the L2 once per 16 CT columns.  The whole slab in LDS
// (16 columns, 128 KB at N = 2048, which also bounded N) moved them for every
// 16 columns, in three times the lines: 47.7 ms for 256 matrices of N = 2048 in
// split BF16, 34.7 with CT = 4.
constexpr int kQ2Fifo = 2;
constexpr int kQ2Cus = 256;

// One block on CT column tiles of three row tiles each, the column tiles'
// chains side by side.
template <int CT, bool BF>
__device__ __forceinline__ void q2_block(const float4 (&va)[3], const float4 (&na)[3], floatx4 (&z0)[CT],
                                         floatx4 (&z1)[CT], floatx4 (&z2)[CT]) {
    if constexpr (BF) {
        // split BF16 (x = hi + lo), the operands' parts stored by
        // q2_prep_kernel.  Lane (lq, l16) holds k = 4 lq .. 4 lq + 3 of its
        // row (A) or column (B), so W = V^T Zb comes out as the update's B
        // operand, W(4 lq + r, l16) in register r, with no transpose.  Two
        // 16-deep products share one 16x16x32 MFMA (the same 16 cycles as a
        // 16x16x16): for W the row tiles 0 and 1 side by side (hi*lo, lo*hi,
        // hi*hi), elsewhere the operand's (hi, lo) with the columns' (lo, hi)
        // and then with their (hi, lo), which adds the lo*lo part as well and
        // needs no zero halves.  (A 16x16x16 and a 16x16x32 one after the
        // other on the same accumulator gave wrong sums on this device.)
        const short8 vh = q2_ops(va[0]), vl = q2_ops(va[1]), v2 = q2_ops(va[2]);
        q2_parts p2[CT], pw[CT];
        short8 zh[CT], zl[CT];
        floatx4 w[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            const q2_parts p0 = q2_split(z0[j]), p1 = q2_split(z1[j]);
            zl[j] = __builtin_bit_cast(short8, q2_parts{p0[0], p1[0]});
            zh[j] = __builtin_bit_cast(short8, q2_parts{p0[1], p1[1]});
            w[j] = q2_mfma32(vh, zl[j], floatx4{0.f, 0.f, 0.f, 0.f});
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) w[j] = q2_mfma32(vl, zh[j], w[j]);
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            p2[j] = q2_split(z2[j]);
            w[j] = q2_mfma32(v2, q2_lo_hi(p2[j]), w[j]);
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) w[j] = q2_mfma32(v2, q2_hi_lo(p2[j]), w[j]);
#pragma unroll
        for (int j = 0; j < CT; ++j) w[j] = q2_mfma32(vh, zh[j], w[j]);
#pragma unroll
        for (int j = 0; j < CT; ++j) pw[j] = q2_split(w[j]);
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            z0[j] = q2_mfma32(q2_ops(na[0]), q2_lo_hi(pw[j]), z0[j]);
            z1[j] = q2_mfma32(q2_ops(na[1]), q2_lo_hi(pw[j]), z1[j]);
            z2[j] = q2_mfma32(q2_ops(na[2]), q2_lo_hi(pw[j]), z2[j]);
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            z0[j] = q2_mfma32(q2_ops(na[0]), q2_hi_lo(pw[j]), z0[j]);
            z1[j] = q2_mfma32(q2_ops(na[1]), q2_hi_lo(pw[j]), z1[j]);
            z2[j] = q2_mfma32(q2_ops(na[2]), q2_hi_lo(pw[j]), z2[j]);
        }
    } else {
        const float vs[12] = {va[0].x, va[0].y, va[0].z, va[0].w, va[1].x, va[1].y,
                              va[1].z, va[1].w, va[2].x, va[2].y, va[2].z, va[2].w};
        const float ns[12] = {na[0].x, na[0].y, na[0].z, na[0].w, na[1].x, na[1].y,
                              na[1].z, na[1].w, na[2].x, na[2].y, na[2].z, na[2].w};
        floatx4 w0[CT], w1[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) w0[j] = w1[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int e = 0; e < 4; e += 2)
#pragma unroll
                for (int j = 0; j < CT; ++j) {
                    const floatx4 z = q == 0 ? z0[j] : q == 1 ? z1[j] : z2[j];
                    w0[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[4 * q + e], z[e], w0[j], 0, 0, 0);
                    w1[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[4 * q + e + 1], z[e + 1], w1[j], 0, 0, 0);
                }
        // W as the next product's B operand: register s of lane (lq, l16)
        // must hold W(4 s + lq, l16), the accumulator holds W(4 lq + r, l16)
        // in register r, so the 4 x 4 (lq, r) blocks of each column are
        // transposed across lanes: the off-diagonal 2 x 2 blocks by
        // v_permlane32_swap, then each 2 x 2 block by v_permlane16_swap
        float wb[CT][4];
#pragma unroll
        for (int j = 0; j < CT; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) wb[j][r] = w0[j][r] + w1[j][r];
            auto p0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(wb[j][0]), __float_as_uint(wb[j][2]), false, false);
            auto p1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(wb[j][1]), __float_as_uint(wb[j][3]), false, false);
            auto q0 = __builtin_amdgcn_permlane16_swap(p0[0], p1[0], false, false);
            auto q1 = __builtin_amdgcn_permlane16_swap(p0[1], p1[1], false, false);
            wb[j][0] = __uint_as_float(q0[0]);
            wb[j][1] = __uint_as_float(q0[1]);
            wb[j][2] = __uint_as_float(q1[0]);
            wb[j][3] = __uint_as_float(q1[1]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                z0[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ns[s], wb[j][s], z0[j], 0, 0, 0);
                z1[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ns[4 + s], wb[j][s], z1[j], 0, 0, 0);
                z2[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ns[8 + s], wb[j][s], z2[j], 0, 0, 0);
            }
    }
}

template <int NW, int CT, bool BF>
__global__ void __launch_bounds__(64 * NW) q2_apply_kernel(int n, int ld, const float* __restrict__ Q2all,
                                                           float* __restrict__ Zall, int64_t nblk, int nmat) {
    constexpr int S = 16 * CT;  // columns
    extern __shared__ __align__(16) float q2_smem[];
    // slots passed on by each wave (the last wave: stored to Z), slots taken
    __shared__ int made[NW], taken[NW], stuck;
    // Workgroup i runs on XCD i mod 8 (round-robin dispatch); XCD x takes the
    // x-th eighth of the (matrix, slab) list in order, so the slabs that run
    // together on one XCD belong to one matrix, start together, and read the
    // same block operands through that XCD's L2.
    const int nslab = (n + S - 1) / S;
    const int64_t total = int64_t(nslab) * nmat, per = (total + kXcds - 1) / kXcds;
    const int64_t pos = int64_t(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (pos >= total) return;
    const int b = int(pos / nslab), slab = int(pos % nslab);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int c0 = slab * S;
    float* Z = Zall + size_t(b) * n * ld;
    const float* Q2 = Q2all + size_t(b) * nblk * kQ2BlockFloats;
    const int NG = q2_groups(n);
    if (tid < NW) made[tid] = taken[tid] = 0;
    if (tid == 0) stuck = 0;
    __syncthreads();
    // tasks of group gi, none before the first
    auto tasks_of = [&](int gi) { return gi < 0 ? 0 : sb_tasks(n, (NG - 1 - gi) * kQ2G); };
    auto wait_for = [&](int* count, int need) {
        for (int spin = 0; __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < need; ++spin) {
            if (spin > (1 << 22) || stuck) {
                stuck = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    };
    auto publish = [&](int* count, int v) {
        if (lane == 0) __hip_atomic_store(count, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // this matrix as a raw buffer, offsets in bytes: rows past n lie past its
    // end, where reads give zeros and stores are dropped (as are the stores of
    // columns past n, given an offset past any buffer's)
    const __amdgpu_buffer_rsrc_t rsZ = __builtin_amdgcn_make_buffer_rsrc(Z, 0, n * ld * 4, kBufferWord3);
    // row tile i of Z
    auto load_tile = [&](int i, floatx4 (&x)[CT]) {
        const int at = ((16 * i + 1 + 4 * lq) * ld + c0 + l16) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < CT; ++j)
                x[j][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsZ, at + r * ld * 4 + 64 * j, 0, 0));
    };
    auto store_tile = [&](int i, const floatx4 (&x)[CT]) {
        const int at = ((16 * i + 1 + 4 * lq) * ld + c0 + l16) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < CT; ++j)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[j][r]), rsZ,
                                                      c0 + 16 * j + l16 < n ? at + r * ld * 4 + 64 * j : int(0x80000000),
                                                      0, 0);
    };
    // the operands of block (gi, k) at first, then of each next block of this
    // wave in turn (past the last: of the last again)
    const float4* ops = reinterpret_cast<const float4*>(Q2) +
                        (wv < NG ? q2_block_offset(n, NG - 1 - wv) : 0) * (kQ2BlockFloats / 4);
    auto load_ops = [&](float4 (&va)[3], float4 (&na)[3]) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            va[i] = ops[64 * i + lane];
            na[i] = ops[(kQ2R * kQ2G + kQ2G) / 4 + 64 * i + lane];
        }
    };
    constexpr size_t kSlot = 2 * 16 * S;  // floats per slot
    int gi = wv, k = 0, K = tasks_of(gi < NG ? gi : -1), Kp = tasks_of(gi < NG ? gi - 1 : -1);
    int in = 0, out = 0;  // slots taken from the wave before, and passed on
    floatx4 x0[CT], xa[CT], xb[CT];  // the block's three row tiles
    floatx4 xn[CT];        // the next group's first tile
    // first wave: slot k of group gi from Z, once the wave of the group before
    // has stored it
    auto fetch = [&](int slot, floatx4 (&pa)[CT], floatx4 (&pb)[CT]) {
        if (slot >= K) return;
        if (slot < Kp) {
            wait_for(&made[NW - 1], in + 1);
            ++in;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const int i = NG - 1 - gi + 2 * slot + 1;
        load_tile(i, pa);
        load_tile(i + 1, pb);
    };
    // one block from operands (va, na) while the next block's are read into
    // (vn, nn); the two buffer pairs alternate, so no copy waits for a read
    // in flight
    auto block = [&](const float4 (&va)[3], const float4 (&na)[3], floatx4 (&pa)[CT], floatx4 (&pb)[CT],
                     float4 (&vn)[3], float4 (&nn)[3], floatx4 (&qa)[CT], floatx4 (&qb)[CT]) {
        const int g = NG - 1 - gi;
        const bool lastk = k + 1 == K;
        if (!lastk)
            ops += kQ2BlockFloats / 4;
        else if (gi + NW < NG)
            ops = reinterpret_cast<const float4*>(Q2) + q2_block_offset(n, g - NW) * (kQ2BlockFloats / 4);
        load_ops(vn, nn);
        if (k == 0) {
#pragma unroll
            for (int j = 0; j < CT; ++j) x0[j] = xn[j];
            if (gi + NW < NG) load_tile(g - NW, xn);
        }
        if (wv == 0) {
            // slot k, with slot k + 1 on its way
            if (k == 0) {
                fetch(0, pa, pb);
                fetch(1, qa, qb);
            }
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                xa[j] = pa[j];
                xb[j] = pb[j];
            }
            fetch(k + 2, pa, pb);
        } else if (k < Kp) {
            wait_for(&made[wv - 1], in + 1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            const floatx4* slot = reinterpret_cast<const floatx4*>(q2_smem + (size_t(wv - 1) * kQ2Fifo + in % kQ2Fifo) *
                                                                                 kSlot) + lane;
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                xa[j] = slot[64 * j];
                xb[j] = slot[64 * (CT + j)];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            publish(&taken[wv], ++in);
        } else {
#pragma unroll
            for (int j = 0; j < CT; ++j) xa[j] = xb[j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the block
        if constexpr (CT == 4) {
            q2_block<2, BF>(va, na, *reinterpret_cast<floatx4(*)[2]>(&x0[0]), *reinterpret_cast<floatx4(*)[2]>(&xa[0]),
                            *reinterpret_cast<floatx4(*)[2]>(&xb[0]));
            q2_block<2, BF>(va, na, *reinterpret_cast<floatx4(*)[2]>(&x0[2]), *reinterpret_cast<floatx4(*)[2]>(&xa[2]),
                            *reinterpret_cast<floatx4(*)[2]>(&xb[2]));
        } else {
            q2_block<CT, BF>(va, na, x0, xa, xb);
        }
        if (wv == NW - 1 || gi == NG - 1) {
            // stored slots are published a block later, when their stores
            // have long gone, or at the group's end
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            publish(&made[wv], out);
            store_tile(g + 2 * k, x0);
            store_tile(g + 2 * k + 1, xa);
            ++out;
            if (lastk) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                publish(&made[wv], out);
            }
        } else {
            wait_for(&taken[wv + 1], out - kQ2Fifo + 1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            floatx4* slot = reinterpret_cast<floatx4*>(q2_smem + (size_t(wv) * kQ2Fifo + out % kQ2Fifo) * kSlot) + lane;
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                slot[64 * j] = x0[j];
                slot[64 * (CT + j)] = xa[j];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            publish(&made[wv], ++out);
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) x0[j] = xb[j];
        ++k;
        if (lastk) {
            gi += NW;
            k = 0;
            K = tasks_of(gi < NG ? gi : -1);
            Kp = tasks_of(gi < NG ? gi - 1 : -1);
        }
    };
    if (gi < NG) {
        float4 va[3], na[3], vb[3], nb[3];
        floatx4 pa[CT], pb[CT], qa[CT], qb[CT];  // the first wave's slots, read from Z ahead
        load_tile(NG - 1 - gi, xn);
        load_ops(va, na);
        while (true) {
            block(va, na, pa, pb, vb, nb, qa, qb);
            if (gi >= NG) break;
            block(vb, nb, qa, qb, va, na, pa, pb);
            if (gi >= NG) break;
        }
    }
    __syncthreads();
    if (stuck)
        for (int e = tid; e < n * S; e += 64 * NW)
            if (c0 + e % S < n) Z[size_t(e / S) * ld + c0 + e % S] = __builtin_nanf("");
}

int q2_prep(int batch, int n, float* Q2, hipStream_t s, bool bf16) {
    const int64_t nblk = q2_blocks(n);
    if (nblk <= 0) return CIR_OK;
    dim3 grid(static_cast<unsigned>(nblk), static_cast<unsigned>(batch));
    hipLaunchKernelGGL(q2_prep_kernel, grid, dim3(64), 0, s, n, nblk, Q2, bf16 ? 1 : 0);
    CIR_CHECK_LAUNCH();
    return CIR_OK;
}

// Waves of q2_apply_kernel's workgroup: 12 (candidate 0) or 8, timed per size
// bucket on the first call (tuner.hpp) over a copy of the first few matrices'
// eigenvectors (the kernel works in place).
template <int NW, int CT, bool BF>
static int q2_launch(int batch, int n, int ld, const float* Q2, float* Z, int64_t nblk, hipStream_t s) {
    constexpr size_t sm = size_t(NW - 1) * kQ2Fifo * 2 * CT * 256 * sizeof(float);
    CIR_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q2_apply_kernel<NW, CT, BF>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(sm)));
    // the one-dimensional grid holds at most 2^32 - 1 threads: very large
    // batches go in several launches
    const int64_t nslab = ceil_div(n, 16 * CT);
    const int64_t most = std::max<int64_t>(1, ((int64_t(1) << 32) - 1) / (int64_t(64 * NW) * nslab) - kXcds);
    for (int64_t b0 = 0; b0 < batch; b0 += most) {
        const int nb = int(std::min<int64_t>(most, batch - b0));
        dim3 grid(unsigned(ceil_div(nslab * nb, int64_t(kXcds)) * kXcds));
        hipLaunchKernelGGL((q2_apply_kernel<NW, CT, BF>), grid, dim3(64 * NW), sm, s, n, ld,
                           Q2 + size_t(b0) * nblk * kQ2BlockFloats, Z + size_t(b0) * n * ld, nblk, nb);
        CIR_CHECK_LAUNCH();
    }
    return CIR_OK;
}

// 32 columns per workgroup, or 16 where that leaves CUs idle.
template <int NW, bool BF>
static int q2_launch(int batch, int n, int ld, const float* Q2, float* Z, int64_t nblk, hipStream_t s) {
    return ceil_div(n, 32) * batch >= 2 * kQ2Cus ? q2_launch<NW, 2, BF>(batch, n, ld, Q2, Z, nblk, s)
                                                 : q2_launch<NW, 1, BF>(batch, n, ld, Q2, Z, nblk, s);
}

int q2_apply(int batch, int n, int ld, const float* Q2, float* Z, hipStream_t s, bool bf16) {
    const int64_t nblk = q2_blocks(n);
    if (nblk <= 0) return CIR_OK;
    // split BF16, slabs of 64 columns for two rounds of the CUs or more: 8
    // waves of 64 columns, each block's operands and bookkeeping serving twice
    // the columns (256 matrices of N = 2048: 34.7 ms, 12 waves of 32 columns
    // 39.3; a workgroup takes 1.1 ms against 0.64, so fewer than two rounds
    // are better off with the narrower one).  FP32 is bound by its MFMAs.
    if (bf16 && ceil_div(n, 64) * batch >= 2 * kQ2Cus) return q2_launch<8, 4, true>(batch, n, ld, Q2, Z, nblk, s);
    auto launch = [&](int cand, int nb, float* Zp) {
        if (bf16)
            return cand == 0 ? q2_launch<12, true>(nb, n, ld, Q2, Zp, nblk, s)
                             : q2_launch<8, true>(nb, n, ld, Q2, Zp, nblk, s);
        return cand == 0 ? q2_launch<12, false>(nb, n, ld, Q2, Zp, nblk, s)
                         : q2_launch<8, false>(nb, n, ld, Q2, Zp, nblk, s);
    };
    const TuneKey key{"q2_apply_threads", {size_bucket(n), bf16 ? 1 : 0, 0, 0, 0}};
    int cand = tune_lookup(key);
    if (cand < 0 && tune_allowed(s)) {
        const int nb = std::min(batch, 8);
        const size_t bytes = size_t(nb) * n * ld * sizeof(float);
        float* scratch = nullptr;
        if (hipMalloc(&scratch, bytes) != hipSuccess) {
            (void)hipGetLastError();  // no room to time: the default width
            scratch = nullptr;
        } else {
            int err = CIR_OK;
            const hipError_t he = hipMemcpyAsync(scratch, Z, bytes, hipMemcpyDeviceToDevice, s);
            if (he != hipSuccess) err = hip_fail(he, "hipMemcpyAsync", __FILE__, __LINE__);
            if (err == CIR_OK) cand = tune_time(key, 2, s, [&](int c) { return launch(c, nb, scratch); }, &err);
            (void)hipStreamSynchronize(s);
            (void)hipFree(scratch);
            if (err != CIR_OK) return err;
        }
    }
    return launch(cand < 0 ? 0 : cand, batch, Z);
}

}  // namespace cir
