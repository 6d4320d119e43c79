// aclblasStrsm: triangular solve with multiple right-hand sides, FP32,
// column-major: B := alpha op(A)^-1 B (left) or alpha B op(A)^-1 (right).
//
// Reference: blas/trsm/arch35/strsm_host.cpp:406-483 (entry, argument checks
// and their order, alpha == 0 writes zeros), :143-153 (zero path) and its
// blocked left path :216-404 (diagonal-panel solve, then a GEMM update of the
// rows still to be solved).
//
// MI355X design: one blocked algorithm for every side / uplo / trans case.
// op(A) is walked in 128 x 128 diagonal blocks in the order its triangle
// dictates (forward when the effective factor is lower, backward otherwise):
//   1. the diagonal block is solved against all right-hand sides in the
//      operation order of netlib strsm.f, so an order up to 128 (one block)
//      rounds exactly as the reference's golden: column sweeps on 16 x 16
//      tiles (TrsmSweepKernel), or, where strsm.f accumulates ascending inner
//      products, one lane per vector (TrsmInnerKernel).  With several blocks
//      the updates between them round in the GEMM's order anyway, and the
//      sweep, whose steps run in parallel over the rows, takes every block;
//   2. the rest of B is updated by the library's FP32 MFMA GEMM
//      (aclblasSgemm, alpha -1, beta 1; operands addressed in place in A and
//      B, transposition through the GEMM's op flags).
// alpha != 1 is applied by one elementwise pass, before the solve or, for
// B op(A)^-T, after it (where strsm.f applies it).  No workspace,
// no allocation, no host synchronisation: the call captures into a graph.
#include "cann_ops_blas.h"
#include "device_common.h"
#include "internal.h"
#include "tile16.h"

namespace aclblas {
namespace {

constexpr int kTb = 128;         // diagonal block order
constexpr int kVec = 16;         // tile order, and vectors per workgroup of the sweep kernel
constexpr int kDiagThreads = 64;  // vectors per workgroup of the inner-product kernel

// B[i + j ldb] *= alpha (or = 0 when zero), i < m, j < n.
__global__ __launch_bounds__(256) void TrsmScaleKernel(float* __restrict__ B, int m, int n, int ldb, float alpha,
                                                      int zero)
{
    const long long total = static_cast<long long>(m) * n;
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < total; idx += stride) {
        const int j = static_cast<int>(idx / m);
        const int i = static_cast<int>(idx - static_cast<long long>(j) * m);
        float& v = B[i + static_cast<size_t>(j) * ldb];
        v = zero != 0 ? 0.0f : alpha * v;
    }
}

// One diagonal block M y = b for `vectors` right-hand-side vectors.  M
// (kb x kb) is the block of op(A) for the left side and of op(A)^T for the
// right side: M(i, j) = A(k0 + i, k0 + j) when readDirect, else
// A(k0 + j, k0 + i); lower (forward) or upper.  Left side: vector = column c
// of B, b_i = B(k0 + i, c); right side: vector = row r, b_i = B(r, k0 + i).
// The substitution follows netlib strsm.f operation for operation: every
// multiply-subtract rounded separately (so no matrix instruction), the
// diagonal divides (left) or multiplies by its reciprocal (right), a unit
// diagonal is not read.
struct DiagArgs {
    const float* A;
    float* B;
    int lda, ldb;
    int k0, kb;
    int vectors;
    int readDirect, unit;
};

__device__ __forceinline__ float LoadM(const DiagArgs& p, int i, int j)
{
    return p.readDirect != 0 ? dev::G(p.A)[(p.k0 + i) + static_cast<size_t>(p.k0 + j) * p.lda]
                             : dev::G(p.A)[(p.k0 + j) + static_cast<size_t>(p.k0 + i) * p.lda];
}

template <bool LEFT>
__device__ __forceinline__ size_t BOffset(const DiagArgs& p, int i, int vec)
{
    return LEFT ? (p.k0 + i) + static_cast<size_t>(vec) * p.ldb : vec + static_cast<size_t>(p.k0 + i) * p.ldb;
}

// Column sweeps (forward: k ascending, else descending; each finished y_k is
// subtracted from the rows still open), 16 vectors per workgroup of NT waves
// (eight for a whole block).  Wave I holds rows 16 I .. 16 I + 15 as one tile (dev::F32x4 layout);
// in phase J wave J solves its 16 x 16 block and publishes y, then the waves
// behind it subtract the block's 16 columns in k order, wave J + 1 first of
// all finishing its tile.  The block lies in LDS as [column][row], so a wave
// reads the four rows of a lane at once.
//
// What bounds it: the chain of kb quotients, broadcasts and subtractions.  One
// lane per vector with its values in LDS (before) took 255 us for a block of
// 128 and 1000 vectors: 16 waves on the GPU, one dependent LDS round trip per
// multiply-subtract; this takes 19 us (504 waves).
template <bool LEFT, bool FORWARD, int NT>
__global__ __launch_bounds__(NT * dev::kWave) void TrsmSweepKernel(DiagArgs p)
{
    constexpr int kN = NT * kVec;
    constexpr int kThreads = NT * dev::kWave;
    constexpr int kBlockLoads = kN * kN / kThreads;
    __shared__ __attribute__((aligned(16))) float T[kN][kN + 4];    // [column][row]
    __shared__ float ys[2][kVec][kVec];                             // y of the solved block, [k][vector]
    const int tid = threadIdx.x;
    const int lane = dev::LaneId();
    const int wave = dev::Uniform(tid / dev::kWave);
    const int r16 = lane & 15;
    const int grp = lane >> 4;
    const int nt = (p.kb + kVec - 1) / kVec;
    const int vec = static_cast<int>(blockIdx.x) * kVec + r16;
    float x[4];
    dev::StaticFor<0, 4>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const int i = kVec * wave + 4 * grp + j;
        x[j] = dev::G(p.B)[BOffset<LEFT>(p, min(i, p.kb - 1), min(vec, p.vectors - 1))];
    });
    // the whole block in flight: unconditional loads at clamped indices (a load
    // under a lane's condition would be waited for on its own), selected after.
    // Rows and columns past kb are the identity's: their y is b = 0.
    float m[kBlockLoads];
    dev::StaticFor<0, kBlockLoads>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int fast = min(tid % kN, p.kb - 1);
        const int slow = min(tid / kN + q * (kThreads / kN), p.kb - 1);
        m[q] = p.readDirect != 0 ? LoadM(p, fast, slow) : LoadM(p, slow, fast);
    });
    dev::StaticFor<0, 4>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        x[j] = kVec * wave + 4 * grp + j < p.kb && vec < p.vectors ? x[j] : 0.0f;
    });
    dev::StaticFor<0, kBlockLoads>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int fast = tid % kN;
        const int slow = tid / kN + q * (kThreads / kN);
        const int i = p.readDirect != 0 ? fast : slow;
        const int j = p.readDirect != 0 ? slow : fast;
        const bool in = i < p.kb && j < p.kb && (i == j ? p.unit == 0 : (FORWARD ? i > j : i < j));
        T[j][i] = in ? m[q] : (i == j ? 1.0f : 0.0f);
    });
    __syncthreads();
    for (int ph = 0; ph < nt; ++ph) {
        const int J = FORWARD ? ph : nt - 1 - ph;
        float (*yb)[kVec] = ys[ph & 1];
        if (wave == J) {
            float u[4];
            dev::StaticFor<0, 4>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const int i = kVec * J + 4 * grp + j;
                u[j] = LEFT ? T[i][i] : 1.0f / T[i][i];
            });
            dev::StaticFor<0, kVec>([&](auto sc) {
                constexpr int k = FORWARD ? decltype(sc)::value : kVec - 1 - decltype(sc)::value;
                constexpr int g = k / 4;
                constexpr int e = k % 4;
                const dev::F32x4 d = *reinterpret_cast<const dev::F32x4*>(&T[kVec * J + k][kVec * J + 4 * grp]);
                const float q = LEFT ? x[e] / u[e] : u[e] * x[e];  // group g holds row k
                x[e] = grp == g ? q : x[e];
                const float yk = dev::GroupBroadcast<g>(q);
                dev::StaticFor<0, 4>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const bool open = FORWARD ? (j > e ? grp >= g : grp > g) : (j < e ? grp <= g : grp < g);
                    const float z = x[j] - d[j] * yk;
                    x[j] = open ? z : x[j];
                });
            });
            dev::StaticFor<0, 4>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                yb[4 * grp + j][r16] = x[j];
            });
        }
        __syncthreads();
        if (FORWARD ? wave > J && wave < nt : wave < J) {
            dev::StaticFor<0, kVec>([&](auto sc) {
                constexpr int k = FORWARD ? decltype(sc)::value : kVec - 1 - decltype(sc)::value;
                const dev::F32x4 d = *reinterpret_cast<const dev::F32x4*>(&T[kVec * J + k][kVec * wave + 4 * grp]);
                const float yk = yb[k][r16];
                dev::StaticFor<0, 4>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    x[j] = x[j] - d[j] * yk;
                });
            });
        }
    }
    dev::StaticFor<0, 4>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const int i = kVec * wave + 4 * grp + j;
        if (i < p.kb && vec < p.vectors) {
            dev::G(p.B)[BOffset<LEFT>(p, i, vec)] = x[j];
        }
    });
}

// Ascending inner products, the order strsm.f uses for the backward solves
// with A itself on the right or A^T on the left: y_i takes the products with
// y_{i+1}, y_{i+2}, ... in that order, so each y_i starts with the value
// solved last and the whole block is one chain of kb^2 / 2 subtractions: one
// lane per vector, the vectors' values in LDS columns.  128 x 1000: 210 us
// with an LDS round trip per product, 159 us.
template <bool LEFT, int NT>
__global__ __launch_bounds__(kDiagThreads) void TrsmInnerKernel(DiagArgs p)
{
    constexpr int kN = NT * kVec;
    constexpr int kRowLoads = (kN + kDiagThreads - 1) / kDiagThreads;
    __shared__ __attribute__((aligned(16))) float T[kN][kN];  // [row][column]
    __shared__ float ys[kN][kDiagThreads];
    const int tid = threadIdx.x;
#pragma unroll 8
    for (int i = 0; i < p.kb; ++i) {
        float m[kRowLoads];
#pragma unroll
        for (int q = 0; q < kRowLoads; ++q) {
            m[q] = LoadM(p, i, min(tid + q * kDiagThreads, p.kb - 1));
        }
#pragma unroll
        for (int q = 0; q < kRowLoads; ++q) {
            const int j = tid + q * kDiagThreads;
            if (j < kN) {
                T[i][j] = j < p.kb && (i == j ? p.unit == 0 : i < j) ? m[q] : (i == j ? 1.0f : 0.0f);
            }
        }
    }
    const int vec = static_cast<int>(blockIdx.x) * kDiagThreads + tid;
    const bool valid = vec < p.vectors;
#pragma unroll 8
    for (int i = 0; i < p.kb; ++i) {
        const float v = dev::G(p.B)[BOffset<LEFT>(p, i, min(vec, p.vectors - 1))];
        ys[i][tid] = valid ? v : 0.0f;
    }
    for (int i = p.kb; i < ((p.kb + 7) & ~7); ++i) {
        ys[i][tid] = 0.0f;  // columns past kb, to a whole group of eight: zero products
    }
    __syncthreads();
    // eight products at a time, the next eight operands loaded before the
    // subtractions that use these
    struct Group {
        dev::F32x4 m[2];
        float y[8];
    };
    const auto load = [&](int i, int k) {
        Group q;
        q.m[0] = *reinterpret_cast<const dev::F32x4*>(&T[i][k]);
        q.m[1] = *reinterpret_cast<const dev::F32x4*>(&T[i][k + 4]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            q.y[e] = ys[k + e][tid];
        }
        return q;
    };
    for (int i = p.kb - 1; i >= 0; --i) {
        float t = ys[i][tid];
        const int k0 = (i + 1) & ~7;
        if (k0 < p.kb) {
            Group cur = load(i, k0);
            float prod[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                // entries up to the diagonal: t - (+0) is t
                prod[e] = k0 + e > i ? cur.m[e / 4][e % 4] * cur.y[e] : 0.0f;
            }
            for (int k = k0 + 8; k < p.kb; k += 8) {
                cur = load(i, k);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    t = t - prod[e];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    prod[e] = cur.m[e / 4][e % 4] * cur.y[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                t = t - prod[e];
            }
        }
        ys[i][tid] = LEFT ? t / T[i][i] : (1.0f / T[i][i]) * t;
    }
    if (valid) {
        for (int i = 0; i < p.kb; ++i) {
            dev::G(p.B)[BOffset<LEFT>(p, i, vec)] = ys[i][tid];
        }
    }
}

// NT tiles: the block's order at most 16 NT.  inner: ascending inner products
// instead of the backward column sweep.
template <int NT>
void LaunchTiles(hipStream_t st, bool left, const DiagArgs& p, bool forward, bool inner)
{
    const int per = inner ? kDiagThreads : kVec;
    const dim3 grid(static_cast<unsigned>((p.vectors + per - 1) / per));
    const dim3 block(inner ? kDiagThreads : NT * dev::kWave);
    if (inner) {
        if (left) {
            hipLaunchKernelGGL((TrsmInnerKernel<true, NT>), grid, block, 0, st, p);
        } else {
            hipLaunchKernelGGL((TrsmInnerKernel<false, NT>), grid, block, 0, st, p);
        }
    } else if (left) {
        if (forward) {
            hipLaunchKernelGGL((TrsmSweepKernel<true, true, NT>), grid, block, 0, st, p);
        } else {
            hipLaunchKernelGGL((TrsmSweepKernel<true, false, NT>), grid, block, 0, st, p);
        }
    } else {
        if (forward) {
            hipLaunchKernelGGL((TrsmSweepKernel<false, true, NT>), grid, block, 0, st, p);
        } else {
            hipLaunchKernelGGL((TrsmSweepKernel<false, false, NT>), grid, block, 0, st, p);
        }
    }
}

// A small block on an instance of its size: with the LDS and the waves of a
// block of 128 the sweep takes 611 us for order 4 and 10^6 vectors (45 us on
// one wave a workgroup) and 132 us for order 16 and 200000 (13 us), the inner
// products 279 and 120 us (13 and 13 us).
void LaunchSlice(hipStream_t st, bool left, const DiagArgs& p, bool forward, bool inner)
{
    if (p.kb <= kVec) {
        LaunchTiles<1>(st, left, p, forward, inner);
    } else if (p.kb <= 2 * kVec) {
        LaunchTiles<2>(st, left, p, forward, inner);
    } else {
        LaunchTiles<kTb / kVec>(st, left, p, forward, inner);
    }
}

// A launch has fewer than 2^32 threads, and the sweep takes up to 32 a vector:
// at most kSlice vectors (2^31 threads) each.
void LaunchDiag(hipStream_t st, bool left, const DiagArgs& p, bool forward, bool inner)
{
    constexpr long long kSlice = 1ll << 26;
    for (long long v0 = 0; v0 < p.vectors; v0 += kSlice) {
        DiagArgs q = p;
        q.B = p.B + (left ? v0 * p.ldb : v0);
        q.vectors = static_cast<int>(p.vectors - v0 < kSlice ? p.vectors - v0 : kSlice);
        LaunchSlice(st, left, q, forward, inner);
    }
}

void LaunchScale(hipStream_t st, float* B, int m, int n, int ldb, float alpha, bool zero)
{
    const long long total = static_cast<long long>(m) * n;
    long long blocks = (total + 255) / 256;
    blocks = blocks > 4096 ? 4096 : (blocks < 1 ? 1 : blocks);
    hipLaunchKernelGGL(TrsmScaleKernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, B, m, n, ldb, alpha,
                       zero ? 1 : 0);
}

}  // namespace
}  // namespace aclblas

extern "C" aclblasStatus_t aclblasStrsm(aclblasHandle_t handle, aclblasSideMode_t side, aclblasFillMode_t uplo,
                                        aclblasOperation_t trans, aclblasDiagType_t diag, int m, int n,
                                        const float* alpha, const float* A, int lda, float* B, int ldb)
{
    using namespace aclblas;
    // argument checks in the reference's order (strsm_host.cpp:406-452)
    if (handle == nullptr) {
        return ACLBLAS_STATUS_HANDLE_IS_NULLPTR;
    }
    if (EnumBits(side) != ACLBLAS_SIDE_LEFT && EnumBits(side) != ACLBLAS_SIDE_RIGHT) {
        return ACLBLAS_STATUS_INVALID_VALUE;
    }
    if (m < 0 || n < 0) {
        return ACLBLAS_STATUS_INVALID_VALUE;
    }
    if ((EnumBits(uplo) != ACLBLAS_UPPER && EnumBits(uplo) != ACLBLAS_LOWER) || !IsValidOp(trans) ||
        (EnumBits(diag) != ACLBLAS_NON_UNIT && EnumBits(diag) != ACLBLAS_UNIT) || alpha == nullptr) {
        return ACLBLAS_STATUS_INVALID_VALUE;
    }
    if (m == 0 || n == 0) {
        return ACLBLAS_STATUS_SUCCESS;
    }
    if (B == nullptr) {
        return ACLBLAS_STATUS_INVALID_VALUE;
    }
    const float a = *alpha;
    if (a != 0.0f && A == nullptr) {
        return ACLBLAS_STATUS_INVALID_VALUE;
    }
    const int k = side == ACLBLAS_SIDE_LEFT ? m : n;
    if (lda < MaxInt(1, k) || ldb < MaxInt(1, m)) {
        return ACLBLAS_STATUS_INVALID_VALUE;
    }
    if (!HandleHasDevice(handle)) {
        return ACLBLAS_STATUS_EXECUTION_FAILED;
    }
    hipStream_t st = handle->stream;
    if (a == 0.0f) {
        LaunchScale(st, B, m, n, ldb, 0.0f, true);
        return LaunchStatus("aclblasStrsm");
    }
    const bool upper = uplo == ACLBLAS_UPPER;
    const bool tr = trans != ACLBLAS_OP_N;
    const bool left = side == ACLBLAS_SIDE_LEFT;
    // strsm.f scales B by alpha before the solve, except for B op(A)^-T where
    // each finished column is scaled after it has been used
    const bool scaleAfter = !left && tr;
    if (a != 1.0f && !scaleAfter) {
        LaunchScale(st, B, m, n, ldb, a, false);
    }
    const int unit = diag == ACLBLAS_UNIT ? 1 : 0;
    // Left: op(A) lower <=> forward.  Right: op(A)^T lower <=> forward.
    const bool opLower = upper == tr;
    const bool forward = left ? opLower : !opLower;
    // M(i, j) read directly from A when M is A itself: left N, right T.
    const int readDirect = (left != tr) ? 1 : 0;
    const int vectors = left ? n : m;
    const int blocks = (k + kTb - 1) / kTb;
    // backward solves whose strsm.f loop accumulates inner products upward
    const bool inner = !forward && left == tr && blocks == 1;
    const float minus1 = -1.0f;
    const float one = 1.0f;
    for (int s = 0; s < blocks; ++s) {
        const int bi = forward ? s : blocks - 1 - s;
        const int k0 = bi * kTb;
        const int kb = k - k0 < kTb ? k - k0 : kTb;
        LaunchDiag(st, left, DiagArgs{A, B, lda, ldb, k0, kb, vectors, readDirect, unit}, forward, inner);
        aclblasStatus_t rs = LaunchStatus("aclblasStrsm");
        if (rs != ACLBLAS_STATUS_SUCCESS) {
            return rs;
        }
        const size_t k0s = static_cast<size_t>(k0);
        const size_t ldas = static_cast<size_t>(lda);
        const size_t ldbs = static_cast<size_t>(ldb);
        if (forward) {
            const int r1 = k0 + kb;
            const int rest = k - r1;
            if (rest <= 0) {
                continue;
            }
            const size_t r1s = static_cast<size_t>(r1);
            if (left) {
                // B[r1:, :] -= op(A)[r1:, k0:r1] Y
                rs = tr ? aclblasSgemm(handle, ACLBLAS_OP_T, ACLBLAS_OP_N, rest, n, kb, &minus1, A + k0s + r1s * ldas,
                                       lda, B + k0s, ldb, &one, B + r1s, ldb)
                        : aclblasSgemm(handle, ACLBLAS_OP_N, ACLBLAS_OP_N, rest, n, kb, &minus1, A + r1s + k0s * ldas,
                                       lda, B + k0s, ldb, &one, B + r1s, ldb);
            } else {
                // B[:, r1:] -= Y op(A)[k0:r1, r1:]
                rs = tr ? aclblasSgemm(handle, ACLBLAS_OP_N, ACLBLAS_OP_T, m, rest, kb, &minus1, B + k0s * ldbs, ldb,
                                       A + r1s + k0s * ldas, lda, &one, B + r1s * ldbs, ldb)
                        : aclblasSgemm(handle, ACLBLAS_OP_N, ACLBLAS_OP_N, m, rest, kb, &minus1, B + k0s * ldbs, ldb,
                                       A + k0s + r1s * ldas, lda, &one, B + r1s * ldbs, ldb);
            }
        } else {
            if (k0 == 0) {
                continue;
            }
            if (left) {
                // B[0:k0, :] -= op(A)[0:k0, k0:k0+kb] Y
                rs = tr ? aclblasSgemm(handle, ACLBLAS_OP_T, ACLBLAS_OP_N, k0, n, kb, &minus1, A + k0s, lda, B + k0s,
                                       ldb, &one, B, ldb)
                        : aclblasSgemm(handle, ACLBLAS_OP_N, ACLBLAS_OP_N, k0, n, kb, &minus1, A + k0s * ldas, lda,
                                       B + k0s, ldb, &one, B, ldb);
            } else {
                // B[:, 0:k0] -= Y op(A)[k0:k0+kb, 0:k0]
                rs = tr ? aclblasSgemm(handle, ACLBLAS_OP_N, ACLBLAS_OP_T, m, k0, kb, &minus1, B + k0s * ldbs, ldb,
                                       A + k0s * ldas, lda, &one, B, ldb)
                        : aclblasSgemm(handle, ACLBLAS_OP_N, ACLBLAS_OP_N, m, k0, kb, &minus1, B + k0s * ldbs, ldb,
                                       A + k0s, lda, &one, B, ldb);
            }
        }
        if (rs != ACLBLAS_STATUS_SUCCESS) {
            return rs;
        }
    }
    if (a != 1.0f && scaleAfter) {
        LaunchScale(st, B, m, n, ldb, a, false);
        return LaunchStatus("aclblasStrsm");
    }
    return ACLBLAS_STATUS_SUCCESS;
}
