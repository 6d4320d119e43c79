// Batched LU for n > 256: blocked right-looking LU over many workgroups per
// matrix, one launch per 32-column panel, in place in the caller's matrices.
//
// Reference: blas/getrf_batched/arch35/sgetrf_batched_kernel.cpp:38-221 (pivot
// rule, division multipliers, rank-1 updates, stop at the first exact zero
// pivot).
//
// Look-ahead inside a launch.  Launch p finds panel p factored.  For every
// matrix one "lead" workgroup applies panel p to the columns of panel p + 1
// only and factors them at once, while the other workgroups apply panel p to
// the remaining trailing columns (32 each) and its row interchanges to the
// columns left of it.  Workgroups of a launch touch disjoint columns and read
// only panel p, so nothing inside a launch waits for another workgroup.
//
// What bounds it: the lead's chain of n columns, each one reduction, one
// barrier and one pivot-row exchange.  The unblocked kernel before it kept a
// matrix on one CU and moved the whole trailing matrix through L2 for every
// column: eight matrices of order 1000 took 75.3 ms on eight CUs, 1.47 ms here
// (33 launches of 45 us).
//
// Same bits as the unblocked order.  Every entry sees l = a / p and a =
// fma(-l, u, a) for ascending k, whichever kernel runs: v_mfma_f32_16x16x4_f32
// is exactly that chain of four fused multiply-adds (measured bit for bit over
// random, subnormal, infinite and NaN operands), so the update runs on matrix
// cores.  Columns of a panel past an exact zero pivot enter it as (-0) * (+0),
// which leaves every accumulator as it is, signed zeros included.
#include "device_common.h"
#include "internal.h"
#include "lapack_kernels.h"

namespace aclblas {
namespace {

using dev::kWave;

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int kStrip = 32;     // columns per update workgroup
constexpr int kLeftCols = 64;  // columns per interchange workgroup

typedef float f32x4 __attribute__((ext_vector_type(4)));

// No workspace: the state between launches is the matrix, ipiv and info.
struct LargeArgs {
    float* const* A;
    int n, lda;
    int* ipiv;  // null: no pivoting
    int* info;  // may be null without pivoting
    int batch;
    int k0;     // first column of the factored panel (-NB: none yet, only factor panel 0)
};

template <int NB>
struct LargeShared {
    alignas(16) float cand[2][kWaves][NB];  // each wave's best row, by column parity
    uint2 key[2][kWaves];                   // its |a| key and position (0xFFFF: no candidate)
    int pw[NB];                             // position the pivot of each column came from
    int swapTo[2 * NB];                     // interchanges as target <- source rows
    int swapFrom[2 * NB];
    alignas(16) float l11[NB][NB + 4];      // unit lower block, multipliers past a zero pivot 0
    alignas(16) float u[kStrip][NB + 4];    // U12 of the strip, [column][k]
};

// Columns of the panel at k0 that were eliminated: NB, fewer when it stopped
// at an exact zero pivot, -1 when an earlier panel did.  info says so (a value
// the lead of this same launch may be writing lies past the panel and reads as
// "not stopped"); without info the diagonal of U does.
template <int NB>
__device__ __forceinline__ int PanelSteps(const LargeArgs& p, const float* A, int b)
{
    int z = -1;
    if (p.info != nullptr) {
        z = __hip_atomic_load(p.info + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - 1;
    } else {
        __shared__ int first;
        if (threadIdx.x == 0) {
            first = p.n;
        }
        __syncthreads();
        for (int j = threadIdx.x; j < min(p.n, p.k0 + NB); j += kThreads) {
            if (dev::G(A)[j + static_cast<size_t>(j) * p.lda] == 0.0f) {
                atomicMin(&first, j);
            }
        }
        __syncthreads();
        z = first < p.n ? first : -1;
    }
    z = dev::Uniform(z);
    if (z >= 0 && z < p.k0) {
        return -1;
    }
    return z >= 0 && z < p.k0 + NB ? z - p.k0 : min(NB, p.n - p.k0);
}

// The panel's interchanges as at most 2 NB moves target <- source (wave 0,
// one target per lane): its NB rows and the rows their pivots came from, each
// target traced back through the swap list.  Duplicate targets are equal moves.
template <int NB>
__device__ __forceinline__ void SwapMoves(const LargeArgs& p, int b, int count, LargeShared<NB>& sh)
{
    const int t = threadIdx.x;
    if (t < kWave) {
        const int mine = t < count ? p.ipiv[static_cast<size_t>(b) * p.n + p.k0 + t] - 1 : -1;
        const int other = __shfl(mine, t - NB, kWave);
        int q = t < NB ? p.k0 + t : other;
        if (t >= 2 * NB || (t < NB ? t >= count : t - NB >= count)) {
            q = -1;
        }
        int src = q;
        for (int j = count - 1; j >= 0; --j) {
            const int pj = __builtin_amdgcn_readlane(mine, j);
            const int r = p.k0 + j;
            src = src == r ? pj : (src == pj ? r : src);
        }
        if (t < 2 * NB) {
            sh.swapTo[t] = q;
            sh.swapFrom[t] = src;
        }
    }
}

// Columns [c0, c1): a wave takes a column at a time, lane i move i; all of a
// column's loads come back before its stores go out.
template <int NB>
__device__ __forceinline__ void SwapColumns(float* A, int lda, int c0, int c1, const LargeShared<NB>& sh)
{
    const int lane = dev::LaneId();
    const int to = lane < 2 * NB ? sh.swapTo[lane] : -1;
    const int from = lane < 2 * NB ? sh.swapFrom[lane] : -1;
    const bool move = to >= 0 && to != from;
    for (int c = c0 + static_cast<int>(threadIdx.x) / kWave; c < c1; c += 4 * kWaves) {
        float v[4];
        dev::StaticFor<0, 4>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int cc = c + i * kWaves;
            v[i] = move && cc < c1 ? dev::G(A)[from + static_cast<size_t>(cc) * lda] : 0.0f;
        });
        dev::StaticFor<0, 4>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int cc = c + i * kWaves;
            if (move && cc < c1) {
                dev::G(A)[to + static_cast<size_t>(cc) * lda] = v[i];
            }
        });
    }
}

// Applies the panel at k0 (steps columns of it) to columns [c0, c0 + kStrip):
// interchanges, U12 by substitution in LDS, then A22 -= L21 U12, accumulated
// transposed (16 lanes hold 16 consecutive rows of a column).
template <int NB>
__device__ __forceinline__ void ApplyPanel(const LargeArgs& p, float* Aptr, int c0, int steps, LargeShared<NB>& sh)
{
    const auto A = dev::G(Aptr);
    const size_t lda = static_cast<size_t>(p.lda);
    const int t = threadIdx.x;
    const int lane = dev::LaneId();
    const int wave = dev::Uniform(t / kWave);
    const int n = p.n;
    const int k0 = p.k0;
    const int cols = min(kStrip, n - c0);
    if (p.ipiv != nullptr) {
        SwapColumns<NB>(Aptr, p.lda, c0, c0 + cols, sh);
    }
    __syncthreads();
    for (int e = t; e < NB * NB; e += kThreads) {
        const int i = e % NB;
        const int k = e / NB;
        sh.l11[i][k] = k < steps && i > k ? A[(k0 + i) + (k0 + k) * lda] : 0.0f;
    }
    for (int e = t; e < NB * kStrip; e += kThreads) {
        const int i = e % NB;
        const int c = e / NB;
        sh.u[c][i] = c < cols ? A[(k0 + i) + (c0 + c) * lda] : 0.0f;
    }
    __syncthreads();
    // one column per lane; the multipliers are read four at a time by all lanes alike
    if (t < kStrip) {
        float x[NB];
        dev::StaticFor<0, NB / 4>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            const float4 v = *reinterpret_cast<const float4*>(&sh.u[t][4 * c]);
            x[4 * c] = v.x;
            x[4 * c + 1] = v.y;
            x[4 * c + 2] = v.z;
            x[4 * c + 3] = v.w;
        });
        const auto substitute = [&](auto full) {
            dev::StaticFor<1, NB>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                dev::StaticFor<0, (i + 3) / 4>([&](auto cc) {
                    constexpr int c = decltype(cc)::value;
                    const float4 lv = *reinterpret_cast<const float4*>(&sh.l11[i][4 * c]);
                    const float l4[4] = {lv.x, lv.y, lv.z, lv.w};
                    dev::StaticFor<0, 4>([&](auto ec) {
                        constexpr int k = 4 * c + decltype(ec)::value;
                        if constexpr (k < i) {
                            if (decltype(full)::value || k < steps) {
                                x[i] = fmaf(-l4[k - 4 * c], x[k], x[i]);
                            }
                        }
                    });
                });
            });
        };
        if (steps == NB) {
            substitute(std::true_type{});
        } else {
            substitute(std::false_type{});
        }
        // the update reads U12 rows past a zero pivot as +0
        dev::StaticFor<0, NB / 4>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            float v[4];
            dev::StaticFor<0, 4>([&](auto ec) {
                constexpr int i = 4 * c + decltype(ec)::value;
                if (t < cols) {
                    A[(k0 + i) + (c0 + t) * lda] = x[i];
                }
                v[i - 4 * c] = i < steps ? x[i] : 0.0f;
            });
            *reinterpret_cast<float4*>(&sh.u[t][4 * c]) = make_float4(v[0], v[1], v[2], v[3]);
        });
    }
    __syncthreads();
    const int r16 = lane & 15;
    const int grp = lane >> 4;
    constexpr int kSteps = NB / 4;
    float ua[2][kSteps];
    dev::StaticFor<0, 2>([&](auto hc) {
        constexpr int h = decltype(hc)::value;
        dev::StaticFor<0, kSteps>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            ua[h][s] = sh.u[16 * h + r16][4 * s + grp];
        });
    });
    // a wave takes 32 rows at a time; clamped rows and columns are loaded and not stored
    const int r0 = k0 + NB;
    for (int rb = r0 + wave * 32; rb < n; rb += 32 * kWaves) {
        float l[2][kSteps];
        f32x4 acc[2][2];
        dev::StaticFor<0, 2>([&](auto tc) {
            constexpr int q = decltype(tc)::value;
            const int row = min(rb + 16 * q + r16, n - 1);
            dev::StaticFor<0, kSteps>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                l[q][s] = A[row + (k0 + 4 * s + grp) * lda];
            });
            dev::StaticFor<0, 2>([&](auto hc) {
                constexpr int h = decltype(hc)::value;
                dev::StaticFor<0, 4>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    acc[q][h][j] = A[row + min(c0 + 16 * h + 4 * grp + j, n - 1) * lda];
                });
            });
        });
        dev::StaticFor<0, kSteps>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            dev::StaticFor<0, 2>([&](auto tc) {
                constexpr int q = decltype(tc)::value;
                const float neg = 4 * s + grp < steps ? -l[q][s] : -0.0f;
                dev::StaticFor<0, 2>([&](auto hc) {
                    constexpr int h = decltype(hc)::value;
                    acc[q][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(ua[h][s], neg, acc[q][h], 0, 0, 0);
                });
            });
        });
        dev::StaticFor<0, 2>([&](auto tc) {
            constexpr int q = decltype(tc)::value;
            const int row = rb + 16 * q + r16;
            dev::StaticFor<0, 2>([&](auto hc) {
                constexpr int h = decltype(hc)::value;
                dev::StaticFor<0, 4>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const int col = 16 * h + 4 * grp + j;
                    if (row < n && col < cols) {
                        A[row + (c0 + col) * lda] = acc[q][h][j];
                    }
                });
            });
        });
    }
}

// Factors the panel at column k1: R rows per thread in registers (row t +
// 1024 q of the panel), NB columns.  Per column every wave reduces its |a|
// keys, its best lane publishes the row, one barrier, and every wave picks the
// same winner from the 16 published keys.  Rows keep a position instead of
// moving and are written back in pivoted order.
template <int NB, int R, bool PIVOT>
__device__ __forceinline__ void FactorLead(const LargeArgs& p, float* Aptr, int b, int k1, LargeShared<NB>& sh)
{
    const auto A = dev::G(Aptr);
    const size_t lda = static_cast<size_t>(p.lda);
    const int t = threadIdx.x;
    const int lane = dev::LaneId();
    const int wave = dev::Uniform(t / kWave);
    const int rows = p.n - k1;
    const int w = min(NB, rows);
    const bool active = wave * kWave < rows;
    float a[R][NB];
    int pos[R];
    dev::StaticFor<0, R>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int r = t + kThreads * q;
        pos[q] = r < rows ? r : -1;
        dev::StaticFor<0, NB>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            a[q][j] = A[k1 + min(r, rows - 1) + (k1 + min(j, w - 1)) * lda];
        });
    });
    if (!active && lane == 0) {
        sh.key[0][wave] = make_uint2(0u, 0xFFFFu);
        sh.key[1][wave] = make_uint2(0u, 0xFFFFu);
    }
    int zero = -1;
    dev::StaticFor<0, NB>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        constexpr int buf = j & 1;
        const bool live = j < w && zero < 0;  // uniform over the workgroup
        if (live && active) {
            uint32_t key = 0;
            uint32_t at = 0xFFFFu;
            int mine = 0;
            dev::StaticFor<0, R>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                const bool cand = PIVOT ? pos[q] >= j : pos[q] == j;
                const uint32_t k = cand ? dev::MagKey(a[q][j]) : 0u;
                const uint32_t pq = cand ? static_cast<uint32_t>(pos[q]) : 0xFFFFu;
                const bool better = k > key || (k == key && pq < at);
                key = better ? k : key;
                at = better ? pq : at;
                mine = better ? q : mine;
            });
            const uint32_t best = dev::SegReduce<kWave, true>(key);
            const bool tied = key == best && at != 0xFFFFu;
            uint64_t tmask = __builtin_amdgcn_ballot_w64(tied);
            if (tmask & (tmask - 1)) {
                const uint32_t lowest = dev::SegReduce<kWave, false>(tied ? at : 0xFFFFu);
                tmask = __builtin_amdgcn_ballot_w64(tied && at == lowest);
            }
            if (tmask == 0) {
                if (lane == 0) {
                    sh.key[buf][wave] = make_uint2(0u, 0xFFFFu);
                }
            } else if (lane == static_cast<int>(__builtin_ctzll(tmask))) {
                dev::StaticFor<0, R>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    if (R == 1 || mine == q) {
                        dev::StaticFor<j / 4, NB / 4>([&](auto cc) {
                            constexpr int c = decltype(cc)::value;
                            *reinterpret_cast<float4*>(&sh.cand[buf][wave][4 * c]) =
                                make_float4(a[q][4 * c], a[q][4 * c + 1], a[q][4 * c + 2], a[q][4 * c + 3]);
                        });
                    }
                });
                sh.key[buf][wave] = make_uint2(key, at);
            }
        }
        if (live) {
            __syncthreads();
            const uint2 kp = sh.key[buf][lane & (kWaves - 1)];
            const uint32_t best = dev::SegReduce<kWaves, true>(kp.x);
            uint32_t m = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(kp.x == best && kp.y != 0xFFFFu)) & 0xFFFFu;
            if (m & (m - 1)) {
                const uint32_t lowest = dev::SegReduce<kWaves, false>(kp.x == best ? kp.y : 0xFFFFu);
                m = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(kp.x == best && kp.y == lowest)) & 0xFFFFu;
            }
            const int wb = __builtin_ctz(m | 0x10000u) & (kWaves - 1);
            const int pw = __builtin_amdgcn_readlane(static_cast<int>(kp.y), wb);
            if (t == 0) {
                sh.pw[j] = pw;
            }
            const float pivot = sh.cand[buf][wb][j];
            if (pivot == 0.0f) {
                zero = j;
            } else if (active) {
                float u[NB];
                dev::StaticFor<j / 4, NB / 4>([&](auto cc) {
                    constexpr int c = decltype(cc)::value;
                    const float4 v = *reinterpret_cast<const float4*>(&sh.cand[buf][wb][4 * c]);
                    u[4 * c] = v.x;
                    u[4 * c + 1] = v.y;
                    u[4 * c + 2] = v.z;
                    u[4 * c + 3] = v.w;
                });
                dev::StaticFor<0, R>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    // the row at position j and the pivot's trade places
                    pos[q] = pos[q] == pw ? j : (pos[q] == j ? pw : pos[q]);
                    const bool upd = pos[q] > j;
                    const float l = a[q][j] / pivot;
                    a[q][j] = upd ? l : a[q][j];
                    dev::StaticFor<j + 1, NB>([&](auto cc) {
                        constexpr int c = decltype(cc)::value;
                        a[q][c] = upd ? fmaf(-l, u[c], a[q][c]) : a[q][c];
                    });
                });
            }
        }
    });
    dev::StaticFor<0, R>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if (pos[q] >= 0) {
            dev::StaticFor<0, NB>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                if (j < w) {
                    A[(k1 + pos[q]) + (k1 + j) * lda] = a[q][j];
                }
            });
        }
    });
    __syncthreads();
    if (PIVOT && t < (zero < 0 ? w : zero + 1)) {
        p.ipiv[static_cast<size_t>(b) * p.n + k1 + t] = k1 + sh.pw[t] + 1;
    }
    if (p.info != nullptr && t == 0 && (zero >= 0 || k1 == 0)) {
        __hip_atomic_store(p.info + b, zero < 0 ? 0 : k1 + zero + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Blocks: one lead per matrix first (their chain is the launch's length), then
// the trailing strips, then the columns left of the panel.
template <int NB, int R, bool PIVOT>
__global__ __launch_bounds__(kThreads) void GetrfLargeKernel(LargeArgs p)
{
    __shared__ LargeShared<NB> sh;
    const int b = static_cast<int>(blockIdx.x) % p.batch;
    const int part = static_cast<int>(blockIdx.x) / p.batch;
    float* const A = p.A[b];
    const int k1 = p.k0 + NB;
    const int tail = p.n - k1;  // columns right of the panel
    if (p.k0 >= 0) {
        const int steps = PanelSteps<NB>(p, A, b);
        if (steps < 0) {
            return;
        }
        const int w = min(NB, p.n - p.k0);
        if (PIVOT) {
            SwapMoves<NB>(p, b, min(steps + 1, w), sh);
            __syncthreads();
        }
        // the lead's strip is the next panel's NB columns, the others follow in kStrip steps
        const int strips = tail > 0 ? 1 + (max(0, tail - NB) + kStrip - 1) / kStrip : 0;
        if (part >= strips) {
            const int c0 = (part - strips) * kLeftCols;
            SwapColumns<NB>(A, p.lda, c0, min(p.k0, c0 + kLeftCols), sh);
            return;
        }
        ApplyPanel<NB>(p, A, part == 0 ? k1 : k1 + NB + (part - 1) * kStrip, steps, sh);
        if (part != 0 || steps < NB) {
            return;
        }
        __syncthreads();
    }
    FactorLead<NB, R, PIVOT>(p, A, b, k1, sh);
}

template <int NB, int R, bool PIVOT>
void LaunchStep(hipStream_t st, const LargeArgs& p)
{
    const int tail = p.n - p.k0 - NB;
    long long parts = 1;
    if (p.k0 >= 0) {
        parts = tail > 0 ? 1 + ((tail > NB ? tail - NB : 0) + kStrip - 1) / kStrip : 0;
        parts += PIVOT ? (p.k0 + kLeftCols - 1) / kLeftCols : 0;
    }
    if (parts > 0) {
        hipLaunchKernelGGL((GetrfLargeKernel<NB, R, PIVOT>), dim3(static_cast<unsigned>(parts * p.batch)),
                           dim3(kThreads), 0, st, p);
    }
}

}  // namespace

template <bool PIVOT>
void LaunchGetrfLarge(hipStream_t st, float* const* A, int n, int lda, int* ipiv, int* info, int batch)
{
    constexpr int NB = kStrip;
    // slices keep a launch's threads below 2^32 (at most 96 workgroups per matrix)
    constexpr int kSlice = 16384;
    for (int b0 = 0; b0 < batch; b0 += kSlice) {
        const int count = batch - b0 < kSlice ? batch - b0 : kSlice;
        LargeArgs p{A + b0, n, lda, PIVOT ? ipiv + static_cast<size_t>(b0) * n : nullptr,
                    info != nullptr ? info + b0 : nullptr, count, -NB};
        for (; p.k0 < n; p.k0 += NB) {
            // rows of the panel this step factors: one or two per thread
            if (n - p.k0 - NB <= kThreads) {
                LaunchStep<NB, 1, PIVOT>(st, p);
            } else {
                LaunchStep<NB, 2, PIVOT>(st, p);
            }
        }
    }
}

template void LaunchGetrfLarge<true>(hipStream_t, float* const*, int, int, int*, int*, int);
template void LaunchGetrfLarge<false>(hipStream_t, float* const*, int, int, int*, int*, int);

}  // namespace aclblas
