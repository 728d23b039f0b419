// gemm_f32.hip — F32 GEMM on the BF16 matrix cores (ta_gemm_f32, cublasSgemm
// semantics: src/backend/cuda/tensor.cu:168-182).
//
// Row-major problem: C[m, n] = alpha sum_k X(m,k) Y(k,n) + beta C[m, n] with
// F32 operands of either layout.  Each F32 value is split into three BF16
// parts, s0 = bf16(s), s1 = bf16(s - s0), s2 = bf16(s - s0 - s1), whose sum
// carries s to about 2^-24 relative (24 bits of significand), and a product
// is the six part products whose magnitude reaches 2^-24 of it: x2 y0, x1 y1,
// x0 y2, x1 y0, x0 y1 and x0 y0, each exact in the MFMA's F32 arithmetic.
// The five small ones accumulate apart from x0 y0, so the small sums are
// complete before they meet the large one.
//
// The split happens between the global load and the LDS store of a tile: the
// operands are read once, as F32, and nothing else is written.  (Splitting
// them in a pass of its own, six BF16 copies per operand in device memory,
// took 937 us for the 8192 x 1536 operand of a LoRA weight gradient, with
// 2-byte stores 98 KB apart where the operand is K-strided, and the product
// then read 12 bytes per element; this kernel takes 21 to 27 us by layout for
// the whole 1536 x 16 product over K = 8192, operands cached.)
//
// What bounds it: reading the operands for the LoRA weight gradients (one of
// the two outer sizes is the rank), six MFMAs per 16 k for square products.
#include <algorithm>

#include "ta_backend.h"
#include "ta_internal.hpp"

namespace ta {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int FK = 64;        // k per stage
constexpr int FLD = FK + 8;   // BF16 elements per LDS row (16-byte fragment reads
                              // of 8 consecutive rows hit disjoint banks)

struct GemmF32Args {
    int M, N, K;
    const float* X;
    int64_t ldx;
    const float* Y;
    int64_t ldy;
    float* C;   // or the splits' partials, [splits][M][N] (alpha 1, beta 0)
    int64_t ldc, split_stride;
    float alpha, beta;
    int tiles_m, tiles_n, k_per_split;
    bool vx, vy;  // 16-byte loads allowed
};

// One ROWS x FK tile of an operand: each thread holds UNITS units of eight k
// of one row (KMAJ: two float4 along k) or of four rows (else: eight float4
// along the rows), so that the split parts leave as whole 16-byte LDS chunks.
template <int ROWS, bool KMAJ>
struct F32Tile {
    static constexpr int RPU = KMAJ ? 1 : 4;            // rows per unit
    static constexpr int TOTAL = ROWS / RPU * (FK / 8);  // units per tile
    static constexpr int UNITS = (TOTAL + 255) / 256;
    float v[UNITS][RPU * 8];  // [row of the unit][k]

    __device__ __forceinline__ static void pos(int u, int& row, int& k) {
        if (KMAJ) {
            row = u / (FK / 8);
            k = 8 * (u % (FK / 8));
        } else {
            row = 4 * (u % (ROWS / 4));
            k = 8 * (u / (ROWS / 4));
        }
    }
    __device__ __forceinline__ void load(const float* __restrict__ P, int64_t ld, int row0, int k0,
                                         int rows, int kend, bool vec) {
#pragma unroll
        for (int i = 0; i < UNITS; i++) {
            const int u = threadIdx.x + 256 * i;
            if (TOTAL % 256 != 0 && u >= TOTAL) break;
            int r, k;
            pos(u, r, k);
            r += row0;
            k += k0;
            if (KMAJ) {
                if (vec && r < rows && k + 8 <= kend) {
                    const float4 a = *(const float4*)(P + (int64_t)r * ld + k);
                    const float4 b = *(const float4*)(P + (int64_t)r * ld + k + 4);
                    v[i][0] = a.x, v[i][1] = a.y, v[i][2] = a.z, v[i][3] = a.w;
                    v[i][4] = b.x, v[i][5] = b.y, v[i][6] = b.z, v[i][7] = b.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        v[i][e] = (r < rows && k + e < kend) ? P[(int64_t)r * ld + k + e] : 0.f;
                }
            } else if (vec && r + 4 <= rows && k + 8 <= kend) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float4 a = *(const float4*)(P + (int64_t)(k + e) * ld + r);
                    v[i][e] = a.x, v[i][8 + e] = a.y, v[i][16 + e] = a.z, v[i][24 + e] = a.w;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int q = 0; q < RPU; q++)
                        v[i][8 * q + e] =
                            (k + e < kend && r + q < rows) ? P[(int64_t)(k + e) * ld + r + q] : 0.f;
            }
        }
    }
    // the three parts into planes S, S + ROWS FLD, S + 2 ROWS FLD
    __device__ __forceinline__ void store(bf16* __restrict__ S) const {
#pragma unroll
        for (int i = 0; i < UNITS; i++) {
            const int u = threadIdx.x + 256 * i;
            if (TOTAL % 256 != 0 && u >= TOTAL) break;
            int r, k;
            pos(u, r, k);
#pragma unroll
            for (int q = 0; q < RPU; q++) {
                bf16x8v p[3];
#pragma unroll
                for (int h = 0; h < 4; h++) {
                    const float a = v[i][8 * q + 2 * h], b = v[i][8 * q + 2 * h + 1];
                    p[0].w[h] = pack2(a, b);
                    const float a1 = a - lo2f(p[0].w[h]), b1 = b - hi2f(p[0].w[h]);
                    p[1].w[h] = pack2(a1, b1);
                    p[2].w[h] = pack2(a1 - lo2f(p[1].w[h]), b1 - hi2f(p[1].w[h]));
                }
#pragma unroll
                for (int c = 0; c < 3; c++)
                    *(bf16x8v*)(S + (c * ROWS + r + q) * FLD + k) = p[c];
            }
        }
    }
};

// Block tile BM x BN, 4 waves as WM x WN; one LDS stage, the next stage's
// operands in registers while the current one computes.
template <int BM, int BN, int WM, int WN, bool XK, bool YK>
__global__ __launch_bounds__(256) void k_gemm_f32(GemmF32Args a) {
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    static_assert(WM * WN == 4 && TM >= 1 && TN >= 1, "4 waves of 32 x 32 fragments");
    __shared__ __attribute__((aligned(16))) bf16 sX[3 * BM * FLD];
    __shared__ __attribute__((aligned(16))) bf16 sY[3 * BN * FLD];
    const int bid = xcd_band(), nt = a.tiles_m * a.tiles_n, zs = bid / nt, tile = bid - zs * nt;
    const int m0 = tile / a.tiles_n * BM, n0 = tile % a.tiles_n * BN;
    const int kbeg = zs * a.k_per_split, kend = min(a.K, kbeg + a.k_per_split);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, wm = wv / WN, wn = wv % WN;

    floatx16 big[TM][TN], small[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) big[i][j][r] = small[i][j][r] = 0.f;

    F32Tile<BM, XK> lx;
    F32Tile<BN, YK> ly;
    lx.load(a.X, a.ldx, m0, kbeg, a.M, kend, a.vx);
    ly.load(a.Y, a.ldy, n0, kbeg, a.N, kend, a.vy);
    for (int k0 = kbeg; k0 < kend; k0 += FK) {
        lx.store(sX);
        ly.store(sY);
        __syncthreads();
        if (k0 + FK < kend) {
            lx.load(a.X, a.ldx, m0, k0 + FK, a.M, kend, a.vx);
            ly.load(a.Y, a.ldy, n0, k0 + FK, a.N, kend, a.vy);
        }
        const bf16* SX = sX + (wm * TM * 32 + (lane & 31)) * FLD + (lane >> 5) * 8;
        const bf16* SY = sY + (wn * TN * 32 + (lane & 31)) * FLD + (lane >> 5) * 8;
#pragma unroll
        for (int kk = 0; kk < FK / 16; kk++) {
            bf16x8_t fx[3][TM], fy[3][TN];
#pragma unroll
            for (int c = 0; c < 3; c++) {
#pragma unroll
                for (int i = 0; i < TM; i++)
                    fx[c][i] = *(const bf16x8_t*)(SX + (c * BM + i * 32) * FLD + kk * 16);
#pragma unroll
                for (int j = 0; j < TN; j++)
                    fy[c][j] = *(const bf16x8_t*)(SY + (c * BN + j * 32) * FLD + kk * 16);
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    floatx16 s = small[i][j];
                    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[2][i], fy[0][j], s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[1][i], fy[1][j], s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[0][i], fy[2][j], s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[1][i], fy[0][j], s, 0, 0, 0);
                    small[i][j] =
                        __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[0][i], fy[1][j], s, 0, 0, 0);
                    big[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[0][i], fy[0][j],
                                                                        big[i][j], 0, 0, 0);
                }
        }
        __syncthreads();
    }

    // lane holds column n = lane%32 of each fragment, rows 8(r/4) + 4(lane/32) + r%4
    float* const C = a.C + (int64_t)zs * a.split_stride;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn * TN + j) * 32 + (lane & 31);
            if (n >= a.N) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = m0 + (wm * TM + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m >= a.M) continue;
                float* c = C + (int64_t)m * a.ldc + n;
                float o = a.alpha * (big[i][j][r] + small[i][j][r]);
                if (a.beta != 0.f) o += a.beta * (*c);
                *c = o;
            }
        }
}

template <int BM, int BN, int WM, int WN>
static void launch_f32(bool xk, bool yk, const GemmF32Args& a, dim3 grid, hipStream_t s) {
    if (xk && yk)
        tlaunch(k_gemm_f32<BM, BN, WM, WN, true, true>, grid, dim3(256), s, a);
    else if (xk)
        tlaunch(k_gemm_f32<BM, BN, WM, WN, true, false>, grid, dim3(256), s, a);
    else if (yk)
        tlaunch(k_gemm_f32<BM, BN, WM, WN, false, true>, grid, dim3(256), s, a);
    else
        tlaunch(k_gemm_f32<BM, BN, WM, WN, false, false>, grid, dim3(256), s, a);
}

static int gemm_f32(bool xk, bool yk, int M, int N, int K, float alpha, const float* X, int64_t ldx,
                    const float* Y, int64_t ldy, float beta, float* C, int64_t ldc, hipStream_t s) {
    GemmF32Args a{};
    a.M = M;
    a.N = N;
    a.K = K;
    a.X = X;
    a.ldx = ldx;
    a.Y = Y;
    a.ldy = ldy;
    a.vx = ((uintptr_t)X & 15) == 0 && ldx % 4 == 0;
    a.vy = ((uintptr_t)Y & 15) == 0 && ldy % 4 == 0;
    // a 32-wide tile for an outer size of at most 32 (the ranks up to 32 of a
    // weight gradient), 64 for one of at most 64, on either side
    const int BN = N <= 32 ? 32 : N <= 64 ? 64 : 128;
    const int BM = BN < 128 ? 128 : M <= 32 ? 32 : M <= 64 ? 64 : 128;
    a.tiles_m = (M + BM - 1) / BM;
    a.tiles_n = (N + BN - 1) / BN;
    // split K while the tiles leave CUs idle: two blocks per CU, at least two
    // stages each (the LoRA weight gradients: 12 tiles over K = 8192 tokens)
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    const int ksteps = (K + FK - 1) / FK;
    int splits = tiles < 256 ? (int)std::min<int64_t>((512 + tiles - 1) / tiles, ksteps / 2) : 1;
    splits = std::max(splits, 1);
    const int per = (ksteps + splits - 1) / splits;
    splits = (ksteps + per - 1) / per;
    a.k_per_split = per * FK;
    const bool part = splits > 1;
    float* p = nullptr;
    if (part) {
        const size_t bytes = (size_t)splits * M * N * sizeof(float);
        p = (float*)scratch_get(bytes, s);
        if (!p) return set_error(-2, "gemm_f32: scratch allocation of %zu bytes failed", bytes);
    }
    a.C = part ? p : C;
    a.ldc = part ? N : ldc;
    a.split_stride = part ? (int64_t)M * N : 0;
    a.alpha = part ? 1.f : alpha;
    a.beta = part ? 0.f : beta;
    const dim3 grid((unsigned)tiles, 1, splits);
    if (BN == 32)
        launch_f32<128, 32, 4, 1>(xk, yk, a, grid, s);
    else if (BN == 64)
        launch_f32<128, 64, 2, 2>(xk, yk, a, grid, s);
    else if (BM == 32)
        launch_f32<32, 128, 1, 4>(xk, yk, a, grid, s);
    else if (BM == 64)
        launch_f32<64, 128, 2, 2>(xk, yk, a, grid, s);
    else
        launch_f32<128, 128, 2, 2>(xk, yk, a, grid, s);
    if (part) splitk_reduce(p, splits, M, N, C, ldc, alpha, beta, nullptr, true, s);
    return check_launch("gemm_f32");
}

}  // namespace ta

using namespace ta;

extern "C" {

int ta_gemm_f32(int transA, int transB, int M, int N, int K, float alpha, const float* A, int lda,
                const float* B, int ldb, float beta, float* C, int ldc, void* stream) {
    TA_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: M/N/K must be > 0");
    TA_REQUIRE(lda > 0 && ldb > 0 && ldc > 0, "gemm_f32: leading dims must be > 0");
    // row-major: C^T [N x M] with X = op(B) by output column (K contiguous
    // when !transB) and Y = op(A) by output row (K contiguous when transA)
    return gemm_f32(!transB, transA != 0, N, M, K, alpha, B, ldb, A, lda, beta, C, ldc,
                    (hipStream_t)stream);
}

}  // extern "C"
