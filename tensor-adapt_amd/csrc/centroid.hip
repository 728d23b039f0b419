// centroid.hip — the Centroid Accumulator's per-token gradient-norm weighted
// sum and the centroid-merge k-means, on the device.
//
// Accumulate (src/centroid/centroid_accumulator.cpp:54-69, intended math):
//   n_t = ||g_t||_2 ; C[d] += h[t,d] * n_t ; W += n_t.
// The reference synchronises, copies two [BT, D] F32 tensors to the host per
// layer and loops on one core.  Here one launch reads h and g once (BF16,
// straight from the step's activations, no cast kernels), each block folds
// 16 (BF16) or 64 (F32) tokens into an F32 partial row, and a second launch
// adds the partial rows in block order into an F64 accumulator [D+1] (entry
// D holds W).  The result is deterministic and within 1e-7 relative of an
// F64 evaluation.
//
// k-means (centroid_accumulator.cpp:114-157 and the stress mode): small
// merges run on one workgroup, others as one launch per Lloyd pass with one
// block per center.  Squared distances are summed sequentially over d in F32
// with no contraction (__fmul_rn/__fadd_rn), exactly like a scalar CPU loop,
// so assignments are bit-reproducible; center sums run over each center's
// members in snapshot index order.  Every loop is bounded by max_iters /
// iters, so the launches always drain.
#include <float.h>

#include <algorithm>
#include <mutex>

#include "kmeans_stop.hpp"
#include "ta_internal.hpp"

// Partial rows of ta_centroid_accumulate_bf16_noalloc, in a file-scope device
// array instead of allocated memory: every GPU the library runs on holds its
// own copy until the process ends.  In host code this name is a host-side
// stand-in, not a device address; host code uses only the per-device address
// from hipGetSymbolAddress (noalloc_scratch below).
constexpr size_t kNoAllocScratchBytes = (size_t)8 << 20;
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

namespace ta {

constexpr int kTok = 16;   // tokens per block, BF16 inputs (512 blocks at BT = 8192)
constexpr int kTokF = 64;  // tokens per block, F32 inputs (1024 blocks per 65536 tokens)

// Per-block partial row: part[blk][d] = sum_{t in block} h[t][d] * n_t,
// part[blk][D] = sum n_t.  Rows move as 16-byte vectors when D % 8 == 0.
// Every block of a 65536-token call is resident at once, so what precedes a
// block's first row load is idle memory time: given norms are copied without
// the per-token reduction and the first 16 rows load ahead of the barrier
// (65536 x 512 F32: 31.8 -> 25.9 us, 5.2 TB/s).
template <bool BF16IN, int KT = BF16IN ? kTok : kTokF>
__global__ __launch_bounds__(256) void k_centroid_part(const void* __restrict__ hv,
                                                       const void* __restrict__ gv,
                                                       const float* __restrict__ nv,
                                                       int64_t BT, int D,
                                                       float* __restrict__ part) {
    __shared__ float nrm[KT];
    int64_t t0 = (int64_t)blockIdx.x * KT;
    int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool v8 = BF16IN && (D & 7) == 0;
    const bool v4 = !BF16IN && (D & 3) == 0;
    // 1. per-token gradient norms (one wave per token; a wave's 16-byte
    // loads of its rows are issued together)
    if (nv)
        for (int j = threadIdx.x; j < KT; j += 256) nrm[j] = t0 + j < BT ? nv[t0 + j] : 0.f;
    for (int j = wv; j < KT && !nv; j += 4) {
        int64_t t = t0 + j;
        float ss = 0.f;
        if (t < BT) {
            if (v8) {
                const bf16x8v* g = (const bf16x8v*)((const bf16*)gv + t * D);
                constexpr int U = 4;
                for (int c0 = lane; c0 < (D >> 3); c0 += 64 * U) {
                    bf16x8v gg[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int c = c0 + 64 * u;
                        gg[u] = g[c < (D >> 3) ? c : c0];
                    }
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        if (c0 + 64 * u >= (D >> 3)) continue;
                        float f[8];
                        unpack8(gg[u], f);
#pragma unroll
                        for (int e = 0; e < 8; e++) ss += f[e] * f[e];
                    }
                }
            } else if (BF16IN) {
                const bf16* g = (const bf16*)gv + t * D;
                for (int d = lane; d < D; d += 64) {
                    float f = bf2f(g[d]);
                    ss += f * f;
                }
            } else if (v4) {
                const float4* g = (const float4*)((const float*)gv + t * D);
                for (int c = lane; c < (D >> 2); c += 64) {
                    const float4 f = g[c];
                    ss += f.x * f.x;
                    ss += f.y * f.y;
                    ss += f.z * f.z;
                    ss += f.w * f.w;
                }
            } else {
                const float* g = (const float*)gv + t * D;
                for (int d = lane; d < D; d += 64) ss += g[d] * g[d];
            }
        }
        ss = wave_sum(ss);
        if (lane == 0) nrm[j] = (t < BT) ? sqrtf(ss) : 0.f;
    }
    // (F32 rows with given norms load their first rows ahead of this barrier)
    const bool early = v4 && nv;
    if (!early) __syncthreads();
    // 2. weighted column sums over this block's tokens
    float* out = part + (int64_t)blockIdx.x * (D + 1);
    if (v8) {
        for (int c = threadIdx.x; c < (D >> 3); c += 256) {
            float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            // all KT row loads first (rows past BT re-read the last row;
            // their weight is 0), then the sums in token order
            bf16x8v hh[KT];
#pragma unroll
            for (int j = 0; j < KT; j++) {
                const int64_t t = min(t0 + j, BT - 1);
                hh[j] = ((const bf16x8v*)((const bf16*)hv + t * D))[c];
            }
#pragma unroll
            for (int j = 0; j < KT; j++) {
                float f[8];
                unpack8(hh[j], f);
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] += f[e] * nrm[j];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) out[c * 8 + e] = acc[e];
        }
    } else if (v4) {
        // F32 rows as 16-byte vectors.  When D/4 columns leave threads over
        // (D = 512: 128 columns), the block's G = 256 / (D/4) thread groups
        // take consecutive token ranges of KT/G tokens each; each group sums
        // its range in token order (16 row loads in flight per batch) and the
        // group sums are added in group order.
        __shared__ float4 gsum[256];
        const int nc4 = D >> 2;
        const int G = (nc4 <= 128 && 256 % nc4 == 0 && KT % (16 * (256 / nc4)) == 0)
                          ? 256 / nc4 : 1;
        const int TG = KT / G;
        float4 hh[16];
        auto rows16 = [&](int j0, int c) {
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const int64_t t = min(t0 + j0 + j, BT - 1);
                hh[j] = ((const float4*)((const float*)hv + t * D))[c];
            }
        };
        if (early) {
            if ((int)threadIdx.x < nc4 * G)
                rows16((int)threadIdx.x / nc4 * TG, (int)threadIdx.x % nc4);
            __syncthreads();
        }
        for (int base = 0; base < nc4 * G; base += 256) {
            const int q = base + threadIdx.x, c = q % nc4, g = q / nc4;
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
            if (q < nc4 * G) {
                for (int j0 = g * TG; j0 < (g + 1) * TG; j0 += 16) {
                    if (!(early && base == 0 && j0 == g * TG)) rows16(j0, c);
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        const float w = nrm[j0 + j];
                        acc.x += hh[j].x * w;
                        acc.y += hh[j].y * w;
                        acc.z += hh[j].z * w;
                        acc.w += hh[j].w * w;
                    }
                }
            }
            if (G > 1) {
                gsum[threadIdx.x] = acc;
                __syncthreads();
                if (threadIdx.x < nc4) {
                    acc = gsum[threadIdx.x];
                    for (int gg = 1; gg < G; gg++) {
                        const float4 o = gsum[gg * nc4 + threadIdx.x];
                        acc.x += o.x;
                        acc.y += o.y;
                        acc.z += o.z;
                        acc.w += o.w;
                    }
                }
            }
            if ((G > 1 ? threadIdx.x < nc4 : q < nc4)) {
                const int cc = G > 1 ? threadIdx.x : c;
                // (partial rows are D + 1 floats apart: 4-byte stores)
                out[4 * cc + 0] = acc.x;
                out[4 * cc + 1] = acc.y;
                out[4 * cc + 2] = acc.z;
                out[4 * cc + 3] = acc.w;
            }
        }
    } else {
        for (int d = threadIdx.x; d < D; d += 256) {
            float acc = 0.f;
            for (int j = 0; j < KT; j++) {
                int64_t t = t0 + j;
                if (t >= BT) break;
                float h = BF16IN ? bf2f(((const bf16*)hv)[t * D + d]) : ((const float*)hv)[t * D + d];
                acc += h * nrm[j];
            }
            out[d] = acc;
        }
    }
    if (threadIdx.x == 0) {
        float w = 0.f;
        for (int j = 0; j < KT; j++) w += nrm[j];
        out[D] = w;
    }
}

// acc[d] += sum over blocks of part[b][d], in F64: 16 columns per block, one
// thread per column and slice of the blocks; a slice is summed in block order
// and the slices are added in order, a fixed order, so the result is
// deterministic.  Narrow blocks spread the partial rows over more CUs, whose
// own load rate bounds this launch (64 columns per block read 2.1 MB through
// 9 CUs).
constexpr int kRW = 16, kRC = 16;  // slices, columns per block
__global__ __launch_bounds__(kRC* kRW) void k_centroid_reduce(const float* __restrict__ part,
                                                              int nblk, int D1,
                                                              double* __restrict__ acc,
                                                              const int32_t* __restrict__ skip) {
    if (skip && *skip) return;
    __shared__ double q[kRW][kRC];
    const int c = threadIdx.x % kRC, w = threadIdx.x / kRC;
    const int d = blockIdx.x * kRC + c;
    const int per = (nblk + kRW - 1) / kRW, b0 = w * per, b1 = min(nblk, b0 + per);
    double s = 0.0;
    if (d < D1) {
        int b = b0;
        for (; b + 16 <= b1; b += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = part[(int64_t)(b + u) * D1 + d];
#pragma unroll
            for (int u = 0; u < 16; u++) s += (double)v[u];
        }
#pragma unroll 8
        for (; b < b1; b++) s += (double)part[(int64_t)b * D1 + d];
    }
    q[w][c] = s;
    __syncthreads();
    if (w == 0 && d < D1) {
        double t = q[0][c];
        for (int i = 1; i < kRW; i++) t += q[i][c];
        acc[d] += t;
    }
}

// ── k-means ────────────────────────────────────────────────────────────
// Squared distances are sums over i = 0 .. D-1 in order, in F32, each term
// (a_i - b_i)^2 rounded before it is added (no contraction), like the
// reference's scalar loop.
//
// Snapshots staged in LDS keep row n's 16-byte chunks XOR-permuted by
// n & sw (sw + 1: the largest power of two up to 16 dividing D / 4):
// element (n, i) sits at n * D + snap_col(n, i, sw).  Rows read at one
// chunk by the lanes (the distance chains, one row per lane) then fall in
// distinct bank groups, and 64 consecutive columns of one row (the center
// sums, one column per lane) in distinct banks; every chain still visits i
// in order.  Snapshots read from global memory are not permuted (sw = 0).
__device__ __forceinline__ int snap_swizzle(int D) {
    return D % 4 == 0 ? min(16, (D >> 2) & -(D >> 2)) - 1 : 0;
}
__device__ __forceinline__ int snap_col(int n, int i, int sw) {
    return ((((i >> 2) ^ (n & sw))) << 2) | (i & 3);
}

// (a - b)^2 as the reference rounds it: hipcc would contract v * v + d into
// one FMA (one rounding where the sequential form rounds twice), so each
// product passes through an empty asm statement, which no instruction
// combiner can look through
__device__ __forceinline__ float sq_term(float a, float b) {
    const float v = __fsub_rn(a, b);
    float q = __fmul_rn(v, v);
    asm volatile("" : "+v"(q));
    return q;
}

// J distance chains: row n[r] of the snapshots X (permuted by sw) against
// the center at cb[r] (its chunks permuted by kb[r]).  With vec (D % 4 == 0,
// rows and centers 16-byte aligned) the operands move as 16-byte chunks, CH
// elements of every chain loaded before the dependent chains over them.
template <int J, int CH>
__device__ __forceinline__ void sqdist_chains(const float* __restrict__ X, int D, int sw, bool vec,
                                              const int (&n)[J], const float* const (&cb)[J],
                                              const int (&kb)[J], float (&out)[J]) {
    static_assert(CH % 4 == 0, "whole chunks");
    float d[J];
    int ka[J];
    const float* ar[J];
#pragma unroll
    for (int r = 0; r < J; r++) {
        d[r] = 0.f;
        ka[r] = n[r] & sw;
        ar[r] = X + (int64_t)n[r] * D;
    }
    int i = 0;
    if (vec) {
        for (; i + CH <= D; i += CH) {
            float4 av[J][CH / 4], bv[J][CH / 4];
#pragma unroll
            for (int r = 0; r < J; r++)
#pragma unroll
                for (int q = 0; q < CH / 4; q++) {
                    const int ch = (i >> 2) + q;
                    av[r][q] = *(const float4*)(ar[r] + ((ch ^ ka[r]) << 2));
                    bv[r][q] = *(const float4*)(cb[r] + ((ch ^ kb[r]) << 2));
                }
#pragma unroll
            for (int q = 0; q < CH / 4; q++)
#pragma unroll
                for (int r = 0; r < J; r++) {
                    d[r] = __fadd_rn(d[r], sq_term(av[r][q].x, bv[r][q].x));
                    d[r] = __fadd_rn(d[r], sq_term(av[r][q].y, bv[r][q].y));
                    d[r] = __fadd_rn(d[r], sq_term(av[r][q].z, bv[r][q].z));
                    d[r] = __fadd_rn(d[r], sq_term(av[r][q].w, bv[r][q].w));
                }
        }
    }
    for (; i < D; i++)
#pragma unroll
        for (int r = 0; r < J; r++)
            d[r] = __fadd_rn(d[r], sq_term(ar[r][snap_col(n[r], i, sw)], cb[r][snap_col(kb[r], i, sw)]));
#pragma unroll
    for (int r = 0; r < J; r++) out[r] = d[r];
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double u01(uint64_t& s) {
    return (double)(splitmix64(s) >> 11) * (1.0 / 9007199254740992.0);
}

// Assignment pass: every (center, snapshot) distance into dist [k][N], then
// each snapshot's argmin over the centers (strict <, so the first of equal
// distances).  A wave takes one center at a time (read at one address by all
// its lanes) against 64 snapshots (one per lane), two such units at once.
// C: the centers [k][D], not permuted.  Returns whether any assignment
// changed (block-wide).
__device__ __forceinline__ int kmeans_assign(const float* __restrict__ X, int sw, bool vec,
                                             const float* __restrict__ C, int N, int D, int k,
                                             float* __restrict__ dist, int32_t* __restrict__ asg) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    const int nb = (N + 63) / 64, units = k * nb;
    for (int u = w; u < units; u += 2 * nw) {
        const int u1 = u + nw < units ? u + nw : u;
        const int c0 = u / nb, c1 = u1 / nb;
        const int r0 = (u % nb) * 64 + lane, r1 = (u1 % nb) * 64 + lane;
        const int n[2] = {min(r0, N - 1), min(r1, N - 1)};
        const float* const cb[2] = {C + (int64_t)c0 * D, C + (int64_t)c1 * D};
        const int kb[2] = {0, 0};
        float d[2];
        sqdist_chains<2, 16>(X, D, sw, vec, n, cb, kb, d);
        if (r0 < N) dist[(int64_t)c0 * N + r0] = d[0];
        if (u1 != u && r1 < N) dist[(int64_t)c1 * N + r1] = d[1];
    }
    __syncthreads();
    int changed = 0;
    for (int n = threadIdx.x; n < N; n += blockDim.x) {
        float best = 1e38f;
        int bk = 0;
        for (int c = 0; c < k; c++) {
            const float d = dist[(int64_t)c * N + n];
            if (d < best) {
                best = d;
                bk = c;
            }
        }
        if (asg[n] != bk) {
            asg[n] = bk;
            changed = 1;
        }
    }
    return __syncthreads_or(changed);
}

// Update pass: center c = the mean of its members, summed in snapshot index
// order; an empty center becomes zero (reference mode) or stays (stress
// mode).  When every wave's 64 outputs belong to one center (D a multiple of
// 64), a ballot over 64 assignments at a time gives its members in index
// order and only their values are read; otherwise each output scans every
// snapshot.  Either way the same chain of additions.
__device__ __forceinline__ void kmeans_update(const float* __restrict__ X, int sw,
                                              float* __restrict__ C, int N, int D, int k,
                                              const int32_t* __restrict__ asg,
                                              bool empty_to_zero) {
    const bool ballot = D % 64 == 0 && blockDim.x % 64 == 0;
    const int lane = threadIdx.x & 63;
    // the first 256 assignments stay in registers for every output
    int a4[4];
#pragma unroll
    for (int q = 0; q < 4; q++) a4[q] = ballot && 64 * q + lane < N ? asg[64 * q + lane] : -1;
    for (int p = threadIdx.x; p < k * D; p += blockDim.x) {
        const int c = p / D, d = p % D;
        float s = 0.f;
        int cnt = 0;
        if (ballot) {
            for (int n0 = 0; n0 < N; n0 += 64) {
                const int a = n0 < 256 ? a4[n0 >> 6] : n0 + lane < N ? asg[n0 + lane] : -1;
                uint64_t mem = __ballot(a == c);
                // up to four members' values loaded together, then added in
                // index order
                while (mem) {
                    float xv[4];
                    int nm = 0;
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        if (!mem) break;
                        const int n = n0 + __builtin_ctzll(mem);
                        mem &= mem - 1;
                        xv[u] = X[(int64_t)n * D + snap_col(n, d, sw)];
                        nm++;
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (u < nm) s = __fadd_rn(s, xv[u]);
                    cnt += nm;
                }
            }
        } else {
            for (int n = 0; n < N; n++)
                if (asg[n] == c) {
                    s = __fadd_rn(s, X[(int64_t)n * D + snap_col(n, d, sw)]);
                    cnt++;
                }
        }
        if (cnt > 0)
            C[p] = s / (float)cnt;
        else if (empty_to_zero)
            C[p] = 0.f;
    }
    __syncthreads();
}

// Snapshots that fit kXs floats are copied into LDS once (XL, permuted as
// above): the distance chains and the center sums then read them from LDS.
constexpr int kXs = 32768;  // 128 KB

template <bool XL>
__device__ __forceinline__ const float* stage_snapshots(const float* __restrict__ Xg, float* xs,
                                                        int N, int D, int& sw) {
    if constexpr (!XL) {
        sw = 0;
        return Xg;
    }
    sw = snap_swizzle(D);
    for (int p = threadIdx.x; p < N * D; p += blockDim.x) {
        const int n = p / D, d = p % D;
        xs[(int64_t)n * D + snap_col(n, d, sw)] = Xg[p];
    }
    __syncthreads();
    return xs;
}

template <bool XL>
__global__ __launch_bounds__(1024) void k_kmeans_ref(const float* __restrict__ Xg, int N, int D,
                                                     int k, int max_iters,
                                                     float* __restrict__ C,
                                                     int32_t* __restrict__ asg,
                                                     float* __restrict__ dist,
                                                     int32_t* __restrict__ iters_out, bool vec) {
    __shared__ __attribute__((aligned(16))) float xs[XL ? kXs : 1];
    int sw = 0;
    const float* __restrict__ X = stage_snapshots<XL>(Xg, xs, N, D, sw);
    for (int p = threadIdx.x; p < k * D; p += blockDim.x) {
        const int c = p / D, d = p % D, n = (int)(((int64_t)c * N) / k);
        C[p] = X[(int64_t)n * D + snap_col(n, d, sw)];
    }
    for (int n = threadIdx.x; n < N; n += blockDim.x) asg[n] = 0;
    __syncthreads();
    int it = 0;
    for (; it < max_iters; it++) {
        int changed = kmeans_assign(X, sw, vec, C, N, D, k, dist, asg);
        if (!changed) break;
        kmeans_update(X, sw, C, N, D, k, asg, true);
    }
    if (threadIdx.x == 0 && iters_out) *iters_out = it;
}

// Stress-mode merge of a few short snapshots in one launch (the rule is at
// ta_kmeans_pp): everything sits in LDS, and a pass costs its barriers and two
// chains of D additions where a launch would cost more than that.  The same
// chains in the same order as the launches below, so the same bits.  Passes
// stop where one changes no assignment, as there.
constexpr int kSmallX = 8192;        // N D and k D floats
constexpr int kSmallN = 128;         // snapshots and centers
constexpr int kSmallDist = 64 * 64;  // distances
__global__ __launch_bounds__(1024) void k_kmeans_pp_small(const float* __restrict__ Xg,
                                                          const float* __restrict__ W, int N, int D,
                                                          int k, int iters, uint64_t seed,
                                                          float* __restrict__ C_out,
                                                          int32_t* __restrict__ asg_out,
                                                          double* __restrict__ mass_out,
                                                          int32_t* __restrict__ seeds_out) {
    __shared__ __attribute__((aligned(16))) float X[kSmallX], C[kSmallX];
    __shared__ float dist[kSmallDist], d2[kSmallN];
    __shared__ int asg[kSmallN], chosen[kSmallN], order[kSmallN], rank_of[kSmallN];
    __shared__ double mass[kSmallN];
    const bool vec = D % 4 == 0;
    for (int p = threadIdx.x; p < N * D; p += blockDim.x) X[p] = Xg[p];
    uint64_t rng = seed;  // thread 0's
    if (threadIdx.x == 0) {
        const int first = (int)(u01(rng) * N);
        chosen[0] = first >= N ? N - 1 : first;
    }
    if (threadIdx.x < N) {
        d2[threadIdx.x] = FLT_MAX;
        asg[threadIdx.x] = 0;
    }
    __syncthreads();
    for (int m = 1; m < k; m++) {
        const int n[1] = {(int)threadIdx.x}, cm = chosen[m - 1];
        if (n[0] < N) {
            const float* const cb[1] = {X + cm * D};
            const int kb[1] = {0};
            float d[1];
            sqdist_chains<1, 32>(X, D, 0, vec, n, cb, kb, d);
            if (d[0] < d2[n[0]]) d2[n[0]] = d[0];
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double total = 0.0, run = 0.0;
            for (int i = 0; i < N; i++) total += (double)d2[i];
            const double target = u01(rng) * total;
            int pick = -1, last_pos = -1;
            for (int i = 0; i < N; i++) {
                run += (double)d2[i];
                if (d2[i] > 0.f) last_pos = i;
                if (pick < 0 && run > target && d2[i] > 0.f) pick = i;
            }
            chosen[m] = pick >= 0 ? pick : last_pos >= 0 ? last_pos : m % N;
        }
        __syncthreads();
    }
    for (int p = threadIdx.x; p < k * D; p += blockDim.x) C[p] = X[chosen[p / D] * D + p % D];
    __syncthreads();
    for (int it = 0; it <= iters; it++) {
        const int changed = kmeans_assign(X, 0, vec, C, N, D, k, dist, asg);
        if (it == iters || (it > 0 && !changed)) break;
        kmeans_update(X, 0, C, N, D, k, asg, false);
    }
    // rank by member weight (F64, index order), stable descending
    if (threadIdx.x == 0) {
        for (int c = 0; c < k; c++) {
            mass[c] = 0.0;
            order[c] = c;
        }
        for (int n = 0; n < N; n++) mass[asg[n]] += (double)W[n];
        for (int i = 1; i < k; i++) {
            const int v = order[i];
            int j = i - 1;
            while (j >= 0 && mass[order[j]] < mass[v]) {
                order[j + 1] = order[j];
                j--;
            }
            order[j + 1] = v;
        }
        for (int r = 0; r < k; r++) rank_of[order[r]] = r;
    }
    __syncthreads();
    for (int p = threadIdx.x; p < k * D; p += blockDim.x) C_out[p] = C[order[p / D] * D + p % D];
    if (threadIdx.x < N) asg_out[threadIdx.x] = rank_of[asg[threadIdx.x]];
    if (threadIdx.x < k) {
        if (mass_out) mass_out[threadIdx.x] = mass[order[threadIdx.x]];
        if (seeds_out) seeds_out[threadIdx.x] = chosen[threadIdx.x];
    }
}

// ── k-means spread over the GPU ───────────────────────────────────────────
// Every value is a chain of F32 (or F64) additions that has to run in order,
// so what the work costs is latency: the chains of a pass run side by side,
// one per lane, and a Lloyd iteration is one launch of one block per center
// (k_kmeans_iter) with nothing to wait for inside a launch.  The snapshots
// are kept transposed as well, so that 64 chains read 64 neighbouring values.
// 64 snapshots of 512, k = 32, 25 passes: 126 us, against 849 us with the
// distances spread out and everything else on one workgroup, and 3.1 ms on
// one workgroup alone.

// values of a center or snapshot held in LDS; k_kmeans_cdist forms the
// distances of longer centers
constexpr int kIterC = 4096;

// XT[d][n] = X[n][d], 32 x 32 tiles in one grid dimension (N or D alone may
// need more tiles than the other dimensions take)
__global__ __launch_bounds__(256) void k_kmeans_transpose(const float* __restrict__ X,
                                                          float* __restrict__ XT, int N, int D) {
    __shared__ float t[32][33];
    const int64_t td = (D + 31) / 32, tiles = td * ((N + 31) / 32);
    const int c = threadIdx.x & 31;
    for (int64_t q = blockIdx.x; q < tiles; q += gridDim.x) {
        const int n0 = (int)(q / td) * 32, d0 = (int)(q % td) * 32;
        for (int r = threadIdx.x >> 5; r < 32; r += 8)
            if (n0 + r < N && d0 + c < D) t[r][c] = X[(int64_t)(n0 + r) * D + d0 + c];
        __syncthreads();
        for (int r = threadIdx.x >> 5; r < 32; r += 8)
            if (d0 + r < D && n0 + c < N) XT[(int64_t)(d0 + r) * N + n0 + c] = t[c][r];
        __syncthreads();
    }
}

// The chain of snapshot n (column n of XT) against the D values at b (read
// at one address by all lanes).  32 elements at a time: the next 32 are in
// flight, the squares form independently of one another, and only the
// additions wait for each other.
__device__ __forceinline__ void col32(const float* __restrict__ XT, int N, uint32_t n, int i,
                                      float (&v)[32]) {
#pragma unroll
    for (int u = 0; u < 32; u++) v[u] = (XT + (int64_t)(i + u) * N)[n];
}
__device__ __forceinline__ float chain32(float d, const float (&v)[32], const float* b) {
    float q[32];
#pragma unroll
    for (int u = 0; u < 32; u++) q[u] = b[u];
#pragma unroll
    for (int u = 0; u < 32; u++) q[u] = sq_term(v[u], q[u]);
#pragma unroll
    for (int u = 0; u < 32; u++) d = __fadd_rn(d, q[u]);
    return d;
}
__device__ __forceinline__ float sqdist_col(const float* __restrict__ XT, int N, int D, uint32_t n,
                                            const float* b) {
    float d = 0.f;
    int i = 0;
    if (D >= 32) {
        float v[32], w[32];
        col32(XT, N, n, 0, v);
        for (; i + 96 <= D; i += 64) {
            col32(XT, N, n, i + 32, w);
            d = chain32(d, v, b + i);
            col32(XT, N, n, i + 64, v);
            d = chain32(d, w, b + i + 32);
        }
        if (i + 64 <= D) {
            col32(XT, N, n, i + 32, w);
            d = chain32(d, v, b + i);
            d = chain32(d, w, b + i + 32);
            i += 64;
        } else {
            d = chain32(d, v, b + i);
            i += 32;
        }
    }
    for (; i < D; i++) d = __fadd_rn(d, sq_term((XT + (int64_t)i * N)[n], b[i]));
    return d;
}

// out[r][n]: distance of snapshot n to snapshot r (block y = r, 64 snapshots
// per block), or, with k > 0, to the r-th of the reference's k initial
// centers, snapshot (r N) / k, which is also copied to C[r]
__global__ __launch_bounds__(64) void k_kmeans_rows(const float* __restrict__ X,
                                                    const float* __restrict__ XT, int N, int D,
                                                    int k, float* __restrict__ C,
                                                    float* __restrict__ out,
                                                    int32_t* __restrict__ done) {
    __shared__ __attribute__((aligned(16))) float b[kIterC];
    const int r = blockIdx.y, n = blockIdx.x * 64 + threadIdx.x;
    const int row = k > 0 ? (int)(((int64_t)r * N) / k) : r;
    if (D <= kIterC) {
        for (int i = threadIdx.x; i < D; i += 64) b[i] = X[(int64_t)row * D + i];
        __syncthreads();
    }
    const float d = D <= kIterC ? sqdist_col(XT, N, D, min(n, N - 1), b)
                                : sqdist_col(XT, N, D, min(n, N - 1), X + (int64_t)row * D);
    if (n < N) out[(int64_t)r * N + n] = d;
    if (k > 0 && blockIdx.x == 0) {
        for (int i = threadIdx.x; i < D; i += 64) C[(int64_t)r * D + i] = X[(int64_t)row * D + i];
        if (r == 0 && threadIdx.x == 0) *done = kKmeansRunning;
    }
}

// k-means++ seeding (one block), then the initial centers C and their
// distances dist [k][N].  A draw's running sum is an F64 chain in index
// order, kept per snapshot (pre), so the pick is the first snapshot whose
// prefix passes the target.
//
// PD: the distances between all snapshots [N][N] (N <= 1024).  Wave 0 then
// draws alone, from rows of PD (in LDS for N <= 128), with nothing to wait
// for but its own chain: 31 draws over 64 snapshots took 128 us with the
// block's barriers and a row from global memory in each.  PD NULL: the block
// forms each draw's chains to the center drawn last.
constexpr int kPairMax = 1024, kPairLds = 128;
__global__ __launch_bounds__(1024) void k_kmeans_seed(const float* __restrict__ X,
                                                      const float* __restrict__ XT,
                                                      const float* __restrict__ PD, int N, int D,
                                                      int k, uint64_t seed, float* d2, double* pre,
                                                      float* __restrict__ C,
                                                      float* __restrict__ dist,
                                                      int32_t* __restrict__ chosen,
                                                      int32_t* __restrict__ done) {
    __shared__ int last;
    __shared__ float spd[kPairLds * kPairLds];
    __shared__ float sd2[kPairMax];
    __shared__ double spre[kPairMax];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const bool lds = PD && N <= kPairLds;
    if (PD) {
        d2 = sd2;
        pre = spre;
    }
    if (lds)
        for (int p = threadIdx.x; p < N * N; p += 1024) spd[p] = PD[p];
    uint64_t rng = seed;  // wave 0's, the same in every lane
    if (w == 0) {
        int first = (int)(u01(rng) * N);
        if (first >= N) first = N - 1;
        if (lane == 0) {
            chosen[0] = last = first;
            *done = kKmeansRunning;
        }
    }
    for (int n = threadIdx.x; n < N; n += 1024) d2[n] = FLT_MAX;
    __syncthreads();
    // draw m by wave 0, from d2
    auto draw = [&](int m) -> int {
        double run = 0.0;
        for (int n0 = 0; n0 < N; n0 += 64) {
            const float v = n0 + lane < N ? d2[n0 + lane] : 0.f;
            double mine = 0.0;
            if (n0 + 64 <= N) {
#pragma unroll
                for (int l = 0; l < 64; l++) {
                    run += (double)__uint_as_float(
                        __builtin_amdgcn_readlane(__float_as_uint(v), l));
                    mine = lane == l ? run : mine;
                }
            } else {
                for (int l = 0; n0 + l < N; l++) {
                    run += (double)__uint_as_float(
                        __builtin_amdgcn_readlane(__float_as_uint(v), l));
                    mine = lane == l ? run : mine;
                }
            }
            if (n0 + lane < N) pre[n0 + lane] = mine;
        }
        const double target = u01(rng) * run;
        int pick = -1, last_pos = -1;
        for (int n0 = 0; n0 < N; n0 += 64) {
            const int n = n0 + lane;
            const bool pos = n < N && d2[n] > 0.f;
            const uint64_t some = __ballot(pos);
            const uint64_t past = __ballot(pos && pre[n] > target);
            if (some) last_pos = n0 + 63 - __builtin_clzll(some);
            if (pick < 0 && past) pick = n0 + __builtin_ctzll(past);
        }
        return pick >= 0 ? pick : last_pos >= 0 ? last_pos : m % N;
    };
    if (PD) {
        if (w == 0) {
            int cm = __builtin_amdgcn_readfirstlane(last);
            for (int m = 1; m < k; m++) {
                // (one wave: each lane reads back only what it wrote itself)
                for (int n = lane; n < N; n += 64) {
                    const float d = lds ? spd[cm * N + n] : PD[(int64_t)cm * N + n];
                    if (d < d2[n]) d2[n] = d;
                }
                cm = draw(m);
                if (lane == 0) chosen[m] = cm;
            }
        }
    } else {
        for (int m = 1; m < k; m++) {
            const int cm = last;
            for (int n = threadIdx.x; n < N; n += 1024) {
                const float d = sqdist_col(XT, N, D, n, X + (int64_t)cm * D);
                if (d < d2[n]) d2[n] = d;
            }
            __syncthreads();
            if (w == 0) {
                const int pick = draw(m);
                if (lane == 0) chosen[m] = last = pick;
            }
            __syncthreads();
        }
    }
    __syncthreads();
    for (int c = w; c < k; c += 16) {
        const int row = chosen[c];
        for (int i = lane; i < D; i += 64) C[(int64_t)c * D + i] = X[(int64_t)row * D + i];
        for (int n = lane; n < N; n += 64)
            dist[(int64_t)c * N + n] = PD ? PD[(int64_t)row * N + n]
                                          : sqdist_col(XT, N, D, n, X + (int64_t)row * D);
    }
}

// The nearest center (strict <, so the first of equal distances; 0 when none
// is below 1e38) of snapshots n0 .. n0 + 63, one per lane, from dist [k][N]:
// the block's four waves take a quarter of the centers each and wave 0 joins
// them in center order.  The result is valid in wave 0; the caller puts a
// barrier between calls.
__device__ __forceinline__ int nearest64(const float* __restrict__ dist, int N, int k, int n0,
                                         float (&sb)[4][64], int (&si)[4][64]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, kq = (k + 3) / 4;
    const int n = min(n0 + lane, N - 1), c1 = min(k, (w + 1) * kq);
    float best = 1e38f;
    int bk = 0;
    for (int c0 = w * kq; c0 < c1; c0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = c0 + u < c1 ? dist[(int64_t)(c0 + u) * N + n] : 1e38f;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (c0 + u < c1 && v[u] < best) {
                best = v[u];
                bk = c0 + u;
            }
    }
    sb[w][lane] = best;
    si[w][lane] = bk;
    __syncthreads();
    best = 1e38f;
    bk = 0;
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (sb[q][lane] < best) {
            best = sb[q][lane];
            bk = si[q][lane];
        }
    return bk;
}

// Iteration `it` of Lloyd's loop, block c for center c: every snapshot's
// nearest center from the distances din [k][N], center c as the mean of its
// members summed in snapshot index order, and the new center's distances into
// dout.  Each block forms the assignments for itself, k^2 N cached loads a pass:
// 2.6 ms a pass at 4096 x 64 into 1024, against 38 ms on one workgroup.  An empty center becomes zero
// (REF, the reference's loop) or stays.  A pass that changes no assignment
// ends the loop: the centers and distances of every later pass would be the
// same values, so *done makes later launches return at once.
// asg_in / asg_out: the previous and this pass's assignments (REF's first
// pass compares against zeros); asg_fin always holds the latest.
template <bool REF>
__global__ __launch_bounds__(256) void k_kmeans_iter(
    const float* __restrict__ X, const float* __restrict__ XT, float* __restrict__ C, int N, int D,
    int k, int it, const float* __restrict__ din, float* __restrict__ dout,
    const int32_t* __restrict__ asg_in, int32_t* __restrict__ asg_out,
    int32_t* __restrict__ asg_fin, uint64_t* __restrict__ masks, int32_t* done,
    int32_t* __restrict__ iters_out, bool last) {
    __shared__ float sb[4][64];
    __shared__ int si[4][64];
    __shared__ __attribute__((aligned(16))) float cen[kIterC];
    __shared__ uint64_t smask[64];
    // (block 0 may store while others read: either value gives this launch the
    // same answer)
    if (kmeans_stopped(__hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), it))
        return;
    const int c = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nb = (N + 63) / 64;
    // members of c, a bit per snapshot (in LDS up to 4096 snapshots)
    uint64_t* const mask = nb <= 64 ? smask : masks + (int64_t)c * nb;
    int changed = !REF && it == 0;
    for (int j = 0; j < nb; j++) {
        const int n = 64 * j + lane;
        const int a = nearest64(din, N, k, 64 * j, sb, si);
        if (w == 0) {
            const uint64_t mem = __ballot(n < N && a == c);
            if (lane == 0) mask[j] = mem;
            if (n < N) {
                if (it > 0 || REF) changed |= (it == 0 ? 0 : asg_in[n]) != a;
                if (c == 0) asg_out[n] = asg_fin[n] = a;
            }
        }
        __syncthreads();
    }
    changed = __syncthreads_or(changed);
    if (!changed) {
        if (c == 0 && threadIdx.x == 0) {
            if (REF && iters_out) *iters_out = it;
            __hip_atomic_store(done, kmeans_stop_after(it), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    if (REF && c == 0 && threadIdx.x == 0 && iters_out) *iters_out = it + 1;
    float* const Cc = C + (int64_t)c * D;
    const bool with_dist = !last && D <= kIterC;
    for (int d = threadIdx.x; d < D; d += 256) {
        float s = 0.f;
        int cnt = 0;
        for (int j = 0; j < nb; j++) {
            uint64_t mem = mask[j];
            cnt += __popcll(mem);
            // up to eight members' values loaded together, added in order
            while (mem) {
                float xv[8];
                int nm = 0;
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    if (!mem) break;
                    xv[u] = X[(int64_t)(64 * j + __builtin_ctzll(mem)) * D + d];
                    mem &= mem - 1;
                    nm++;
                }
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (u < nm) s = __fadd_rn(s, xv[u]);
            }
        }
        const float v = cnt > 0 ? s / (float)cnt : REF ? 0.f : Cc[d];
        Cc[d] = v;
        if (with_dist) cen[d] = v;
    }
    if (!with_dist) return;
    __syncthreads();
    for (int j = w; j < nb; j += 4) {
        const int n = 64 * j + lane;
        const float d = sqdist_col(XT, N, D, min(n, N - 1), cen);
        if (n < N) dout[(int64_t)c * N + n] = d;
    }
}

// dist[c][n] of centers too long for k_kmeans_iter's LDS (blocks of 64
// snapshots), after its launch
__global__ __launch_bounds__(64) void k_kmeans_cdist(const float* __restrict__ XT,
                                                     const float* __restrict__ C, int N, int D,
                                                     float* __restrict__ dist,
                                                     const int32_t* __restrict__ done) {
    if (*done != kKmeansRunning) return;
    const int c = blockIdx.y, n = blockIdx.x * 64 + threadIdx.x;
    const float d = sqdist_col(XT, N, D, min(n, N - 1), C + (int64_t)c * D);
    if (n < N) dist[(int64_t)c * N + n] = d;
}

// Final assignments (from the last distances unless the loop ended on a
// fixed point), then the centers ranked by the weight of their members:
// masses summed in F64 in snapshot index order, one lane per center; stable
// descending order (a center's rank is the number of centers that precede
// it; with a NaN mass, which no count can order, the insertion sort that
// defines the order runs as it stands).
__global__ __launch_bounds__(1024) void k_kmeans_rank(const float* __restrict__ W, int N, int D,
                                                      int k, const float* __restrict__ dist,
                                                      const float* __restrict__ C,
                                                      int32_t* __restrict__ asg,
                                                      const int32_t* __restrict__ chosen,
                                                      const int32_t* __restrict__ done,
                                                      float* __restrict__ C_out,
                                                      int32_t* __restrict__ asg_out,
                                                      double* __restrict__ mass_out,
                                                      int32_t* __restrict__ seeds_out) {
    __shared__ double mass[1024];
    __shared__ int order[1024], rank_of[1024];
    __shared__ float sw[1024];
    __shared__ int sa[1024];
    const int t = threadIdx.x;
    const bool have = *done != kKmeansRunning;
    double m = 0.0;
    for (int n0 = 0; n0 < N; n0 += 1024) {
        const int n = n0 + t, cnt = min(1024, N - n0);
        if (n < N) {
            int bk = 0;
            if (have) {
                bk = asg[n];
            } else {
                float best = 1e38f;
                for (int c0 = 0; c0 < k; c0 += 16) {
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; u++)
                        v[u] = c0 + u < k ? dist[(int64_t)(c0 + u) * N + n] : 1e38f;
#pragma unroll
                    for (int u = 0; u < 16; u++)
                        if (c0 + u < k && v[u] < best) {
                            best = v[u];
                            bk = c0 + u;
                        }
                }
                asg[n] = bk;
            }
            sa[t] = bk;
            sw[t] = W[n];
        }
        __syncthreads();
        if (t < k)
            for (int i = 0; i < cnt; i++)
                if (sa[i] == t) m += (double)sw[i];
        __syncthreads();
    }
    if (t < k) mass[t] = m;
    if (__syncthreads_or(t < k && m != m)) {
        if (t == 0) {
            for (int c = 0; c < k; c++) order[c] = c;
            for (int i = 1; i < k; i++) {  // insertion sort: stable
                const int v = order[i];
                int j = i - 1;
                while (j >= 0 && mass[order[j]] < mass[v]) {
                    order[j + 1] = order[j];
                    j--;
                }
                order[j + 1] = v;
            }
            for (int r = 0; r < k; r++) rank_of[order[r]] = r;
        }
    } else if (t < k) {
        int r = 0;
        for (int j = 0; j < k; j++) r += mass[j] > m || (mass[j] == m && j < t);
        rank_of[t] = r;
        order[r] = t;
    }
    __syncthreads();
    for (int r = t >> 6; r < k; r += 16)
        for (int i = t & 63; i < D; i += 64)
            C_out[(int64_t)r * D + i] = C[(int64_t)order[r] * D + i];
    for (int n = t; n < N; n += 1024) asg_out[n] = rank_of[asg[n]];
    if (t < k) {
        if (mass_out) mass_out[t] = mass[order[t]];
        if (seeds_out) seeds_out[t] = chosen[t];
    }
}

}  // namespace ta

using namespace ta;

static int centroid_acc(const void* h, const void* g, const float* n, int64_t BT, int D,
                        double* acc, bool bf16in, void* stream, const int32_t* skip = nullptr) {
    TA_REQUIRE(BT >= 0 && D > 0, "centroid_accumulate: bad shape BT=%lld D=%d", (long long)BT, D);
    if (BT == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int kt = bf16in ? kTok : kTokF;
    int64_t nblk = (BT + kt - 1) / kt;
    TA_REQUIRE(nblk < (1ll << 31), "centroid_accumulate: BT too large");
    float* part = (float*)scratch_get((size_t)nblk * (D + 1) * sizeof(float), s);
    TA_REQUIRE(part, "centroid_accumulate: scratch allocation failed");
    if (bf16in)
        tlaunch(k_centroid_part<true>, dim3((int)nblk), dim3(256), s, h, g, nullptr, BT, D, part);
    else
        tlaunch(k_centroid_part<false>, dim3((int)nblk), dim3(256), s, h, g, n, BT, D, part);
    tlaunch(k_centroid_reduce, dim3((D + kRC) / kRC), dim3(kRC * kRW), s, part, (int)nblk, D + 1, acc, skip);
    return check_launch("centroid_accumulate");
}

namespace ta {
int centroid_acc_bf16(const bf16* h, const bf16* g, int64_t BT, int D, double* acc,
                      const int32_t* skip, hipStream_t s) {
    return centroid_acc(h, g, nullptr, BT, D, acc, true, s, skip);
}
}  // namespace ta

// Device address of `scratch` on device dev, looked up once per device with
// that device current and kept.
static std::mutex g_na_mu;
static float* g_na_ptr[64];

static int noalloc_scratch(int dev, float** out) {
    TA_REQUIRE(dev >= 0 && dev < 64, "centroid_accumulate_bf16_noalloc: device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[dev]) {
        void* p = nullptr;
        TA_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        TA_REQUIRE(p, "centroid_accumulate_bf16_noalloc: no device address for the scratch");
        g_na_ptr[dev] = (float*)p;
    }
    *out = g_na_ptr[dev];
    return 0;
}

// Makes `dev` the current device for the lifetime of the object and restores
// the caller's device afterwards.
struct DeviceScope {
    int prev = -1;
    hipError_t err = hipSuccess;
    explicit DeviceScope(int dev) {
        err = hipGetDevice(&prev);
        if (err == hipSuccess && prev != dev) err = hipSetDevice(dev);
    }
    ~DeviceScope() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

// Work arrays of the merge, carved from one scratch buffer.  pd_rows: rows of
// the snapshot-to-snapshot distances (0: the reference's loop, which seeds
// from fixed snapshots and keeps its centers and assignments in the caller's
// arrays).
struct KmeansScratch {
    float *xt, *pd, *d2, *c, *dist[2];
    double* pre;
    uint64_t* masks;
    int32_t *asg[3], *chosen, *done;
    bool get(int N, int D, int k, int pd_rows, hipStream_t s) {
        const bool pp = pd_rows > 0;
        const int64_t nb = (N + 63) / 64;
        const size_t n = (size_t)N, sz[] = {n * D * 4,
                                            pp ? (size_t)pd_rows * N * 4 : 0,
                                            pp ? n * 4 : 0,
                                            pp ? (size_t)k * D * 4 : 0,
                                            n * k * 4,
                                            n * k * 4,
                                            pp ? n * 8 : 0,
                                            nb > 64 ? (size_t)k * nb * 8 : 0,
                                            n * 4,
                                            n * 4,
                                            n * 4,
                                            (size_t)k * 4,
                                            4};
        size_t off[13], total = 0;
        for (int i = 0; i < 13; i++) {
            off[i] = total;
            total += (sz[i] + 255) & ~(size_t)255;
        }
        char* b = (char*)ta::scratch_get(total, s);
        if (!b) return false;
        xt = (float*)(b + off[0]);
        pd = (float*)(b + off[1]);
        d2 = (float*)(b + off[2]);
        c = (float*)(b + off[3]);
        dist[0] = (float*)(b + off[4]);
        dist[1] = (float*)(b + off[5]);
        pre = (double*)(b + off[6]);
        masks = (uint64_t*)(b + off[7]);
        for (int i = 0; i < 3; i++) asg[i] = (int32_t*)(b + off[8 + i]);
        chosen = (int32_t*)(b + off[11]);
        done = (int32_t*)(b + off[12]);
        return true;
    }
};
static dim3 transpose_grid(int N, int D) {
    return dim3((unsigned)std::min<int64_t>((int64_t)((N + 31) / 32) * ((D + 31) / 32), 1 << 20));
}
// Whether the reference's loop runs as one launch per pass.  Nothing tells the
// host that the data has settled, so every pass up to the cap is launched, at
// 3.7 us each when it has nothing left to do (twice that with
// k_kmeans_cdist); the loop on one workgroup stops by itself, at pass_us a
// pass (within a factor of 1.7 of 27 of 28 measured sizes).
// Launches where three passes of the loop cost as much: data that settles in
// the second pass, the first that can end it, then loses a little, and data
// that settles later gains.  64 x 512, k = 32: cap 25 87 or 168 us in the loop
// (settling in two passes or in five), 101 or 107 launched; cap 50, where the
// loop stays, 200 launched.  96 x 1536, k = 4, cap 50: 376 or 1160 against 195
// or 336.  Caps below 25 count as 25 and small work stays in the loop: k N D
// below 2^20 with the snapshots in its LDS (64 x 512, k = 16, cap 25: 78 or 150
// against 103 or 96), below 2^17 without (32 x 1536, k = 2: 127 or 193 against
// 107 or 139).
static bool ref_launched(int N, int D, int k, int max_iters) {
    const bool lds = (int64_t)N * D <= kXs;
    if (max_iters <= 0 || max_iters > 128 || k > 65535 ||
        (int64_t)k * N * D < (int64_t(1) << (lds ? 20 : 17)))
        return false;
    const double units = (double)k * (((int64_t)N + 63) / 64);  // waves' worth of chains
    double pass_us = D * (lds ? 0.01 + 0.0018 * units : 0.02 + 0.0075 * units);
    if (D % 64 != 0)  // every output of the center sums scans all snapshots
        pass_us += (lds ? 0.03 : 0.15) * N * (((int64_t)k * D + 1023) / 1024);
    return 3.0 * pass_us >= (D > kIterC ? 7.4 : 3.7) * std::max(max_iters, 25);
}

extern "C" {

int ta_centroid_accumulate_bf16(const uint16_t* h, const uint16_t* g, int64_t BT, int D,
                                double* acc, void* stream) {
    return centroid_acc(h, g, nullptr, BT, D, acc, true, stream);
}

int ta_centroid_accumulate_bf16_noalloc(const uint16_t* h, const uint16_t* g, int64_t BT, int D,
                                        double* acc, void* stream) {
    TA_REQUIRE(h && g && acc, "centroid_accumulate_bf16_noalloc: null argument");
    TA_REQUIRE(BT >= 0 && D > 0, "centroid_accumulate_bf16_noalloc: bad shape BT=%lld D=%d",
               (long long)BT, D);
    if (BT == 0) return 0;
    const int64_t nblk = (BT + kTok - 1) / kTok;
    const int64_t max_blk = (int64_t)(kNoAllocScratchBytes / sizeof(float)) / (D + 1);
    TA_REQUIRE(nblk <= max_blk,
               "centroid_accumulate_bf16_noalloc: BT=%lld at D=%d needs %lld partial rows of "
               "D+1 floats, over the %zu-byte static scratch (at most BT=%lld at this D)",
               (long long)BT, D, (long long)nblk, kNoAllocScratchBytes,
               (long long)(max_blk * kTok));
    hipStream_t s = (hipStream_t)stream;
    // the stream's device (the current one for the null stream) holds the
    // scratch copy and runs the kernels
    int dev = 0;
    if (s)
        TA_HIP(hipStreamGetDevice(s, &dev));
    else
        TA_HIP(hipGetDevice(&dev));
    DeviceScope scope(dev);
    TA_HIP(scope.err);
    float* part = nullptr;
    const int rc = noalloc_scratch(dev, &part);
    if (rc != 0) return rc;
    // the same kernels and order as ta_centroid_accumulate_bf16: every
    // partial row is written in full before the reduce reads it
    tlaunch(k_centroid_part<true>, dim3((int)nblk), dim3(256), s, h, g, nullptr, BT, D, part);
    tlaunch(k_centroid_reduce, dim3((D + kRC) / kRC), dim3(kRC * kRW), s, part, (int)nblk, D + 1, acc,
                                                             nullptr);
    return check_launch("centroid_accumulate_bf16_noalloc");
}

int ta_centroid_accumulate_f32(const float* h, const float* g, int64_t BT, int D, double* acc,
                               void* stream) {
    TA_REQUIRE(h && g && acc, "centroid_accumulate_f32: null argument");
    return centroid_acc(h, g, nullptr, BT, D, acc, false, stream);
}

int ta_centroid_accumulate_f32n(const float* h, const float* n, int64_t BT, int D, double* acc,
                                void* stream) {
    return centroid_acc(h, nullptr, n, BT, D, acc, false, stream);
}

int ta_kmeans_ref(const float* snaps, int N, int D, int k, int max_iters, float* centers,
                  int32_t* assign, int32_t* iters_out, void* stream) {
    TA_REQUIRE(N > 0 && D > 0 && k > 0 && max_iters >= 0, "kmeans_ref: bad N=%d D=%d k=%d", N, D,
               k);
    if (k > N) k = N;
    hipStream_t s = (hipStream_t)stream;
    if (ref_launched(N, D, k, max_iters)) {
        KmeansScratch m;
        TA_REQUIRE(m.get(N, D, k, 0, s), "kmeans_ref: scratch allocation failed");
        tlaunch(k_kmeans_transpose, transpose_grid(N, D), dim3(256), s, snaps, m.xt, N,
                D);
        tlaunch(k_kmeans_rows, dim3((N + 63) / 64, k), dim3(64), s, snaps, m.xt, N, D, k, centers,
                m.dist[0], m.done);
        for (int it = 0; it < max_iters; it++) {
            tlaunch(k_kmeans_iter<true>, dim3(k), dim3(256), s, snaps, m.xt, centers, N, D, k, it,
                    m.dist[it & 1], m.dist[(it + 1) & 1], m.asg[it & 1], m.asg[(it + 1) & 1],
                    assign, m.masks, m.done, iters_out, it + 1 == max_iters);
            if (D > kIterC && it + 1 < max_iters)
                tlaunch(k_kmeans_cdist, dim3((N + 63) / 64, k), dim3(64), s, m.xt, centers, N, D,
                        m.dist[(it + 1) & 1], m.done);
        }
        return check_launch("kmeans_ref");
    }
    float* dist = (float*)scratch_get((size_t)N * k * sizeof(float), s);
    TA_REQUIRE(dist, "kmeans_ref: scratch allocation failed");
    // 16-byte operand loads: whole chunks, and aligned snapshots (when read
    // from global memory) and centers
    const bool xl = (int64_t)N * D <= kXs;
    const bool vec = D % 4 == 0 && ((uintptr_t)centers & 15) == 0 &&
                     (xl || ((uintptr_t)snaps & 15) == 0);
    if (xl)
        tlaunch(k_kmeans_ref<true>, dim3(1), dim3(1024), s, snaps, N, D, k, max_iters, centers, assign, dist,
                                              iters_out, vec);
    else
        tlaunch(k_kmeans_ref<false>, dim3(1), dim3(1024), s, snaps, N, D, k, max_iters, centers, assign, dist,
                                               iters_out, vec);
    return check_launch("kmeans_ref");
}

int ta_kmeans_pp(const float* snaps, const float* weights, int N, int D, int k, int iters,
                 uint64_t seed, float* centers, int32_t* assign, double* mass, int32_t* seeds,
                 void* stream) {
    TA_REQUIRE(N > 0 && D > 0 && k > 0 && iters >= 0, "kmeans_pp: bad N=%d D=%d k=%d", N, D, k);
    if (k > N) k = N;
    TA_REQUIRE(k <= 1024, "kmeans_pp: k=%d exceeds 1024", k);
    hipStream_t s = (hipStream_t)stream;
    // one workgroup where its draws (one at a time: 0.06 us per snapshot and
    // 0.014 us per dimension, four times that where no 16-byte load fits, less
    // the 0.6 us of a draw among the launches) cost less than the launches' fixed
    // 13 us and what passes launched after the data has settled take, counted at
    // 2 of their 3.7 us (fit to 2068 timed sizes, of which the slower form takes
    // 1.41 times the other at worst; 4 x 16, k = 2: 7 us against 34 with 5 passes
    // launched; 16 x 256, k = 4: 32 against 28 with one; 64 x 64, k = 64: 446
    // against 115)
    if (N <= kSmallN && (int64_t)N * D <= kSmallX && N * k <= kSmallDist &&
        (int64_t)(k - 1) * (60 * N + 14 * (D % 4 ? 4 * D : D) - 600) <=
            13000 + 2000 * ((int64_t)iters - 1)) {
        tlaunch(k_kmeans_pp_small, dim3(1), dim3(1024), s, snaps, weights, N, D, k, iters, seed,
                centers, assign, mass, seeds);
        return check_launch("kmeans_pp");
    }
    KmeansScratch m;
    const bool pairs = N <= kPairMax && k > 1;  // (one center: nothing is drawn by distance)
    TA_REQUIRE(m.get(N, D, k, pairs ? N : 1, s), "kmeans_pp: scratch allocation failed");
    tlaunch(k_kmeans_transpose, transpose_grid(N, D), dim3(256), s, snaps, m.xt, N, D);
    if (pairs)
        tlaunch(k_kmeans_rows, dim3((N + 63) / 64, N), dim3(64), s, snaps, m.xt, N, D, 0, nullptr,
                m.pd, nullptr);
    tlaunch(k_kmeans_seed, dim3(1), dim3(1024), s, snaps, m.xt, pairs ? m.pd : nullptr, N, D, k,
            seed, m.d2, m.pre, m.c, m.dist[0], m.chosen, m.done);
    for (int it = 0; it < iters; it++) {
        tlaunch(k_kmeans_iter<false>, dim3(k), dim3(256), s, snaps, m.xt, m.c, N, D, k, it,
                m.dist[it & 1], m.dist[(it + 1) & 1], m.asg[it & 1], m.asg[(it + 1) & 1], m.asg[2],
                m.masks, m.done, nullptr, false);
        if (D > kIterC)
            tlaunch(k_kmeans_cdist, dim3((N + 63) / 64, k), dim3(64), s, m.xt, m.c, N, D,
                    m.dist[(it + 1) & 1], m.done);
    }
    tlaunch(k_kmeans_rank, dim3(1), dim3(1024), s, weights, N, D, k, m.dist[iters & 1], m.c,
            m.asg[2], m.chosen, m.done, centers, assign, mass, seeds);
    return check_launch("kmeans_pp");
}

}  // extern "C"
