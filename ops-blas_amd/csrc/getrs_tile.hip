// Triangular solves and inverses with the LU factors of orders 65..2048:
// one workgroup per unit of a system and 16 (or, of many, 4) right-hand sides, the
// unknowns as 16 x 16 tiles in LDS, everything off the diagonal blocks on the FP32 matrix
// instruction.
//
// Reference: blas/getrs_batched/arch35/sgetrs_batched_kernel.cpp:83-410 (N: P,
// L^-1, U^-1; T: U^-T, L^-T, P^T; out-of-range pivots skipped) and
// blas/getri_batched/arch35/getri_batched_kernel.cpp:39-308 (C = I, P, L^-1,
// U^-1; info = j + 1 for the zero u_jj with the largest j).
//
// The operations are those of column-oriented substitution, element by element
// (x_j = b_j / u_jj, b_i = fma(-t_ij, x_j, b_i) for j in solve order): four
// k of v_mfma_f32_16x16x4_f32 are exactly that chain of fused multiply-adds, so
// the blocking and the matrix cores change no bit.  Entries past the order
// enter the chain as (-0) * (+0), which leaves every sum as it is.
//
// What bounds it: the chain over the diagonal blocks (16 steps of a quotient, a
// broadcast and a multiply-add each, then the LDS exchange).  Many units run as
// one wave each (SolveAlone: no barriers, the operands of a tile loaded while
// the block before it is solved); few units as one workgroup each
// (SolveShared: the wave that owns tile J updates and solves it first while
// the others apply X(J-1) to the tiles behind it, operands a phase ahead).
// The kernel before it solved 64-row blocks with one row per lane (a division
// and a broadcast per right-hand side and step) and built the row permutation
// with one thread.  Measured before and now:
//   2048 systems of order 128, 8 right-hand sides: N 277 -> 65 us, T 283 -> 74 us
//   inverse of 500 matrices of order 100: 717 -> 103 us
//   8 systems of order 1000, 4 right-hand sides, T: 1095 -> 378 us
#include "device_common.h"
#include "internal.h"
#include "lapack_kernels.h"
#include "lds_dma.h"
#include "tile16.h"

namespace aclblas {
namespace {

using dev::kWave;

constexpr int kT = 16;        // tile order, and most right-hand sides of a unit
constexpr int kFew = 4;       // right-hand sides of a narrow unit
constexpr int kSwaps = 64;    // interchanges composed per step of the permutation
constexpr int kAheadTiles = 4;  // tiles of a wave whose operands are loaded a phase ahead

using f32x4 = dev::F32x4;

// Unknown (row, rhs) in LDS.  COLS 16: rows of 16, each quad of rows rotated by
// its own number, so that both a quarter-wave's four consecutive rows (matrix
// operand) and rows four apart (accumulators) fall into distinct banks.  COLS
// 4: rows of 4, conflict-free in order; lanes past the fourth column repeat the
// first four.
template <int COLS>
__device__ __forceinline__ int XOff(int row, int rhs)
{
    if constexpr (COLS == kT) {
        return ((row & ~3) + ((row + (row >> 2)) & 3)) * kT + rhs;
    } else {
        return row * COLS + (rhs & (COLS - 1));
    }
}

// Makes LDS writes of the WAVES waves that work together visible to them.
template <int WAVES>
__device__ __forceinline__ void Sync()
{
    if constexpr (WAVES == 1) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

// perm with (P b)[i] = b[perm[i]] for the LAPACK swap list piv (entries outside
// [1, n] skipped).  The waves trace the targets of 64 swaps each (the 64 rows
// and the rows they trade with), then one wave composes the groups in order.
template <int WAVES>
__device__ __forceinline__ void BuildPerm(uint16_t* perm, uint16_t* from, const int* piv, int n, int wave)
{
    const int lane = dev::LaneId();
    const int groups = (n + kSwaps - 1) / kSwaps;
    for (int i = wave * kWave + lane; i < n; i += WAVES * kWave) {
        perm[i] = static_cast<uint16_t>(i);
    }
    const auto partner = [&](int row) {
        const int p = row < n ? dev::G(piv)[row] - 1 : row;
        return (p < 0 || p >= n) ? row : p;
    };
    for (int c = wave; c < groups; c += WAVES) {
        const int k0 = c * kSwaps;
        const int row = k0 + lane;
        const int mine = partner(row);
        int s0 = row;
        int s1 = mine;
        for (int j = min(kSwaps, n - k0) - 1; j >= 0; --j) {
            const int pj = __builtin_amdgcn_readlane(mine, j);
            const int r = k0 + j;
            s0 = s0 == r ? pj : (s0 == pj ? r : s0);
            s1 = s1 == r ? pj : (s1 == pj ? r : s1);
        }
        from[2 * kSwaps * c + lane] = static_cast<uint16_t>(s0);
        from[2 * kSwaps * c + kSwaps + lane] = static_cast<uint16_t>(s1);
    }
    Sync<WAVES>();
    if (wave == 0) {
        for (int c = 0; c < groups; ++c) {
            const int row = c * kSwaps + lane;
            const bool ok = row < n;
            const int to = partner(row);
            const uint16_t v0 = ok ? perm[from[2 * kSwaps * c + lane]] : 0;
            const uint16_t v1 = ok ? perm[from[2 * kSwaps * c + kSwaps + lane]] : 0;
            Sync<1>();
            if (ok) {
                perm[to] = v1;
                perm[row] = v0;
            }
            Sync<1>();
        }
    }
    Sync<WAVES>();
}

// The steps of a 16 x 16 diagonal block d ([column][row], in LDS) on the tile
// y (accumulator layout: lane l holds rows 4 (l / 16) + j of right-hand side
// l % 16), straight-line.  LOWER: k ascending, else descending.  The columns
// are read from LDS kAhead steps early: kept whole they would take 64
// registers and halve the waves in flight.  FAST: quotients by DivideBy;
// returns whether a lane divided something outside its range.
template <bool LOWER, bool UNIT, bool FAST>
__device__ __forceinline__ bool DiagSteps(float (&y)[4], const float (*d)[kT + 4], const float (&u)[4],
                                          const float (&r)[4], int rows, int grp)
{
    constexpr int kAhead = 3;
    const auto col = [&](int step) {
        const int k = LOWER ? step : kT - 1 - step;
        return *reinterpret_cast<const f32x4*>(&d[k][4 * grp]);
    };
    f32x4 ring[kAhead + 1];
    dev::StaticFor<0, kAhead>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        ring[i] = col(i);
    });
    bool off = false;
    dev::StaticFor<0, kT>([&](auto ic) {
        constexpr int step = decltype(ic)::value;
        constexpr int k = LOWER ? step : kT - 1 - step;
        constexpr int g = k / 4;
        constexpr int e = k % 4;
        if constexpr (step + kAhead < kT) {
            ring[(step + kAhead) % (kAhead + 1)] = col(step + kAhead);
        }
        const f32x4 dk = ring[step % (kAhead + 1)];
        float v = y[e];
        if constexpr (!UNIT) {
            // meaningful in group g, which holds row k
            if constexpr (FAST) {
                off = off || (grp == g && !dev::Dividable<true>(v));
                v = dev::DivideBy(v, u[e], r[e]);
            } else {
                v = v / u[e];
            }
            y[e] = grp == g ? v : y[e];
        }
        const float xk = dev::GroupBroadcast<g>(v);
        // rows past the order come last in a forward solve; in a backward one their steps change nothing
        const bool live = LOWER || k < rows;
        dev::StaticFor<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const bool open = live && (LOWER ? (j > e ? grp >= g : grp > g) : (j < e ? grp <= g : grp < g));
            const float z = fmaf(-dk[j], xk, y[j]);
            y[j] = open ? z : y[j];
        });
        __builtin_amdgcn_sched_barrier(0);
    });
    return off;
}

// Solves the diagonal block against the tile x.  The reciprocals of the
// diagonal are formed once for all right-hand sides and steps; a tile with an
// operand outside DivideBy's range is solved again with plain divisions.
template <bool LOWER, bool UNIT>
__device__ __forceinline__ void SolveDiag(f32x4& x, const float (*d)[kT + 4], int rows, int grp)
{
    float y[4] = {x[0], x[1], x[2], x[3]};
    float u[4];
    float r[4];
    if constexpr (UNIT) {
        DiagSteps<LOWER, true, true>(y, d, u, r, rows, grp);
    } else {
        bool off = false;
        dev::StaticFor<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            u[j] = d[4 * grp + j][4 * grp + j];
            r[j] = 1.0f / u[j];
            off = off || (4 * grp + j < rows && !dev::Dividable<false>(u[j]));
        });
        off = DiagSteps<LOWER, false, true>(y, d, u, r, rows, grp) || off;
        if (__builtin_amdgcn_ballot_w64(off) != 0) {
            dev::StaticFor<0, 4>([&](auto jc) { y[decltype(jc)::value] = x[decltype(jc)::value]; });
            DiagSteps<LOWER, false, false>(y, d, u, r, rows, grp);
        }
    }
    x = f32x4{y[0], y[1], y[2], y[3]};
}

struct SolveTileArgs {
    const float* const* A;
    int n, lda;
    const int* ipiv;  // null: no interchanges
    float* const* B;
    int ldb, nrhs, chunks;
    int* info;
    long long units;  // batch * chunks
};

// 4 x 4 transpose between the four lane groups and the four registers.
__device__ __forceinline__ void TransposeGroups(f32x4& v)
{
    const auto swap16 = [](float& a, float& b) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(p[0]);
        b = __uint_as_float(p[1]);
    };
    const auto swap32 = [](float& a, float& b) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(p[0]);
        b = __uint_as_float(p[1]);
    };
    float r0 = v[0], r1 = v[1], r2 = v[2], r3 = v[3];
    swap16(r0, r1);
    swap16(r2, r3);
    swap32(r0, r2);
    swap32(r1, r3);
    v = f32x4{r0, r1, r2, r3};
}

// Tiles of one triangular solve, in solve order (phase 0 first), for one wave.
// TR: the factor is read transposed; then vec says that its columns are
// 16-byte aligned and whole tiles are read with one 16-byte load per lane
// (four consecutive columns of op, put into chain order by a 4 x 4 transpose
// between lane groups).
template <bool LOWER, bool TR, int COLS>
struct Tiles {
    const float* Aptr;
    size_t ld;
    int n, nt;
    bool vec;
    float* xs;
    int r16, grp;

    __device__ __forceinline__ Tiles(const float* a, int lda, int order, bool v, float* x)
        : Aptr(a), ld(static_cast<size_t>(lda)), n(order), nt((order + kT - 1) / kT), vec(v), xs(x),
          r16(dev::LaneId() & 15), grp(dev::LaneId() >> 4)
    {
    }
    __device__ __forceinline__ int Tile(int ph) const { return LOWER ? ph : nt - 1 - ph; }
    __device__ __forceinline__ float At(int i, int j) const
    {
        i = min(i, n - 1);
        j = min(j, n - 1);
        return TR ? dev::G(Aptr)[j + i * ld] : dev::G(Aptr)[i + j * ld];
    }
    // column 16 J + 4 s + grp of tile J in chain order (ascending or descending)
    __device__ __forceinline__ int Column(int J, int s) const
    {
        return LOWER ? kT * J + 4 * s + grp : kT * J + kT - 1 - (4 * s + grp);
    }
    __device__ __forceinline__ bool Wide(int J) const { return TR && vec && kT * J + kT <= n; }
    // matrix operand of tile (I, J): row 16 I + r16, four columns per lane
    __device__ __forceinline__ f32x4 LoadOp(int I, int J) const
    {
        if (Wide(J)) {
            const int j = LOWER ? kT * J + 4 * grp : kT * J + kT - 4 - 4 * grp;
            const f32x4 v = dev::LoadG<f32x4>(Aptr + j + min(kT * I + r16, n - 1) * ld);
            return LOWER ? v : f32x4{v[3], v[2], v[1], v[0]};
        }
        f32x4 v;
        dev::StaticFor<0, 4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            v[s] = At(kT * I + r16, Column(J, s));
        });
        return v;
    }
    // the diagonal block of tile J: loaded coalesced, stored as [column][row]
    __device__ __forceinline__ f32x4 LoadDiag(int J) const
    {
        f32x4 v;
        dev::StaticFor<0, 4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            v[s] = TR ? At(kT * J + 4 * s + grp, kT * J + r16) : At(kT * J + r16, kT * J + 4 * s + grp);
        });
        return v;
    }
    __device__ __forceinline__ void StoreDiag(float (*db)[kT + 4], const f32x4& v) const
    {
        dev::StaticFor<0, 4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if (TR) {
                db[r16][4 * s + grp] = v[s];
            } else {
                db[4 * s + grp][r16] = v[s];
            }
        });
    }
    __device__ __forceinline__ f32x4 LoadX(int I) const
    {
        f32x4 x;
        dev::StaticFor<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            x[j] = xs[XOff<COLS>(kT * I + 4 * grp + j, r16)];
        });
        return x;
    }
    __device__ __forceinline__ void StoreX(int I, const f32x4& x) const
    {
        dev::StaticFor<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const int row = kT * I + 4 * grp + j;
            if (row < n) {
                xs[XOff<COLS>(row, r16)] = x[j];  // rows past the order stay +0
            }
        });
    }
    // X(P) as the other matrix operand
    __device__ __forceinline__ f32x4 SolvedOp(int P) const
    {
        f32x4 v;
        dev::StaticFor<0, 4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            v[s] = xs[XOff<COLS>(Column(P, s), r16)];
        });
        return v;
    }
    // the operand of tile (., P) as the chain takes it: negated, -0 past the order
    __device__ __forceinline__ f32x4 ChainOp(f32x4 a, int P) const
    {
        if (Wide(P)) {
            TransposeGroups(a);
        }
        f32x4 v;
        dev::StaticFor<0, 4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            v[s] = Column(P, s) >= n ? -0.0f : -a[s];
        });
        return v;
    }
};

// x += a b in chain order.
__device__ __forceinline__ void Chain(const f32x4& a, const f32x4& b, f32x4& x)
{
    dev::StaticFor<0, 4>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        x = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], x, 0, 0, 0);
    });
}

// One triangular solve by the workgroup: in phase J the wave that owns tile J
// updates and solves it first, the others apply X(J-1) to the tiles behind it.
template <bool LOWER, bool UNIT, bool TR, int WAVES, int COLS>
__device__ __forceinline__ void SolveShared(const Tiles<LOWER, TR, COLS>& T, int wave, float (*diag)[kT][kT + 4])
{
    const int nt = T.nt;
    f32x4 nextOp{};
    f32x4 nextDiag{};
    f32x4 pre[kAheadTiles] = {};
    if (wave == 0) {
        nextDiag = T.LoadDiag(T.Tile(0));
    }
    // the first phase from `from` on whose tile the wave owns
    const auto firstOwn = [&](int from) { return from + ((wave - from) % WAVES + WAVES) % WAVES; };
    for (int ph = 0; ph < nt; ++ph) {
        const int J = T.Tile(ph);
        const int P = ph > 0 ? T.Tile(ph - 1) : 0;
        f32x4 xb{};
        if (ph > 0) {
            xb = T.SolvedOp(P);
        }
        if (ph % WAVES == wave) {
            T.StoreDiag(diag[wave & 3], nextDiag);
            f32x4 x = T.LoadX(J);
            if (ph > 0) {
                Chain(T.ChainOp(nextOp, P), xb, x);
            }
            Sync<1>();
            SolveDiag<LOWER, UNIT>(x, diag[wave & 3], T.n - kT * J, T.grp);
            T.StoreX(J, x);
        }
        if (ph > 0) {
            const int q0 = firstOwn(ph + 1);
            // two tiles at a time: their LDS round trips and chains overlap
            dev::StaticFor<0, kAheadTiles / 2>([&](auto ic) {
                constexpr int i = 2 * decltype(ic)::value;
                if (q0 + i * WAVES < nt) {
                    const bool two = q0 + (i + 1) * WAVES < nt;
                    const int I0 = T.Tile(q0 + i * WAVES);
                    const int I1 = T.Tile(two ? q0 + (i + 1) * WAVES : q0 + i * WAVES);
                    f32x4 x0 = T.LoadX(I0);
                    f32x4 x1 = T.LoadX(I1);
                    Chain(T.ChainOp(pre[i], P), xb, x0);
                    Chain(T.ChainOp(pre[i + 1], P), xb, x1);
                    T.StoreX(I0, x0);
                    if (two) {
                        T.StoreX(I1, x1);
                    }
                }
            });
            for (int q = q0 + kAheadTiles * WAVES; q < nt; q += WAVES) {
                f32x4 y = T.LoadX(T.Tile(q));
                Chain(T.ChainOp(T.LoadOp(T.Tile(q), P), P), xb, y);
                T.StoreX(T.Tile(q), y);
            }
        }
        // the next phase's operands, in flight across the barrier
        if (ph + 1 < nt) {
            if ((ph + 1) % WAVES == wave) {
                nextOp = T.LoadOp(T.Tile(ph + 1), J);
                nextDiag = T.LoadDiag(T.Tile(ph + 1));
            }
            const int q0 = firstOwn(ph + 2);
            dev::StaticFor<0, kAheadTiles>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if (q0 + i * WAVES < nt) {
                    pre[i] = T.LoadOp(T.Tile(q0 + i * WAVES), J);
                }
            });
        }
        // LDS only: the loads stay in flight
        dev::BarrierLds();
    }
}

// One triangular solve by one wave: tile J takes the products with the tiles
// before it, then its diagonal block; the operands of tile J + 1 are loaded
// while the block of tile J is solved.
template <bool LOWER, bool UNIT, bool TR>
__device__ __forceinline__ void SolveAlone(const Tiles<LOWER, TR, kT>& T, float (*diag)[kT + 4])
{
    constexpr int kRun = 8;
    f32x4 ops[kRun] = {};
    f32x4 nextDiag = T.LoadDiag(T.Tile(0));
    const auto load = [&](int ph, int q0) {
        dev::StaticFor<0, kRun>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if (q0 + i < ph) {
                ops[i] = T.LoadOp(T.Tile(ph), T.Tile(q0 + i));
            }
        });
    };
    for (int ph = 0; ph < T.nt; ++ph) {
        const int J = T.Tile(ph);
        T.StoreDiag(diag, nextDiag);
        f32x4 x = T.LoadX(J);
        for (int q0 = 0; q0 < ph; q0 += kRun) {
            dev::StaticFor<0, kRun>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if (q0 + i < ph) {
                    const int P = T.Tile(q0 + i);
                    Chain(T.ChainOp(ops[i], P), T.SolvedOp(P), x);
                }
            });
            if (q0 + kRun < ph) {
                load(ph, q0 + kRun);
            }
        }
        if (ph + 1 < T.nt) {
            load(ph + 1, 0);
            nextDiag = T.LoadDiag(T.Tile(ph + 1));
        }
        Sync<1>();
        SolveDiag<LOWER, UNIT>(x, diag, T.n - kT * J, T.grp);
        T.StoreX(J, x);
        Sync<1>();
    }
}

// Bytes of LDS of one unit (system, cols right-hand sides): unknowns,
// permutation and the traced sources of its swap groups.
__host__ __device__ constexpr int UnitBytes(int n, int cols)
{
    const int tiles = (n + kT - 1) / kT;
    const int groups = (n + kSwaps - 1) / kSwaps;
    return tiles * kT * cols * 4 + (((n + 7) & ~7) + groups * 2 * kSwaps) * 2;
}
constexpr int kDiagBytes = 4 * kT * (kT + 4) * 4;  // the diagonal blocks beside the units
static_assert(UnitBytes(kMaxTileN, kT) + kDiagBytes <= 160 * 1024, "a unit of the largest order fits in LDS");
static_assert(4 * UnitBytes(256, kT) + kDiagBytes <= 160 * 1024, "four units of one wave each fit in LDS");

// Unit u = (system u / chunks, chunk u % chunks of COLS right-hand sides).
// WAVES > 1: one unit per workgroup of WAVES waves.  WAVES == 1: one per wave,
// four waves per workgroup that never wait for each other.
// kSolveInv: C = A^-1 out of place (B = C), nrhs = n, info written per matrix.
template <SolveTileMode MODE, int WAVES, int COLS>
__global__ __launch_bounds__(WAVES == 1 ? 4 * kWave : WAVES * kWave) void SolveTileKernel(SolveTileArgs p)
{
    constexpr int kUnits = WAVES == 1 ? 4 : 1;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ __attribute__((aligned(16))) float diag[4][kT][kT + 4];
    const int n = p.n;
    const int nt = (n + kT - 1) / kT;
    const int group = dev::Uniform(static_cast<int>(threadIdx.x) / kWave);
    const int wave = WAVES == 1 ? 0 : group;
    const long long unit = static_cast<long long>(blockIdx.x) * kUnits + (WAVES == 1 ? group : 0);
    if (unit >= p.units) {
        return;  // a wave of its own: nobody waits for it
    }
    uint8_t* const mem = smem + (WAVES == 1 ? group * UnitBytes(n, COLS) : 0);
    float* xs = reinterpret_cast<float*>(mem);
    uint16_t* perm = reinterpret_cast<uint16_t*>(xs + nt * kT * COLS);
    uint16_t* from = perm + ((n + 7) & ~7);

    const int b = static_cast<int>(unit / p.chunks);
    const int chunk = static_cast<int>(unit - static_cast<long long>(b) * p.chunks);
    const int r0 = chunk * COLS;
    const int rc = min(COLS, p.nrhs - r0);
    const float* A = p.A[b];
    const auto B = dev::G(p.B[b]);
    const int t = wave * kWave + dev::LaneId();
    constexpr int kThreads = WAVES * kWave;
    if (p.ipiv != nullptr) {
        BuildPerm<WAVES>(perm, from, p.ipiv + static_cast<size_t>(b) * n, n, wave);
    }
    const auto permOf = [&](int i) { return p.ipiv != nullptr ? static_cast<int>(perm[i]) : i; };
    // rows permuted for the N and inverse solves; rows and columns past the ends are +0
    for (int i = t; i < nt * kT; i += kThreads) {
        const int src = MODE != kSolveT && i < n ? permOf(i) : i;
        float v[COLS];
        dev::StaticFor<0, COLS>([&](auto rcst) {
            constexpr int r = decltype(rcst)::value;
            if (MODE == kSolveInv) {
                v[r] = i < n && src == r0 + r ? 1.0f : 0.0f;
            } else {
                v[r] = i < n && r < rc ? B[src + static_cast<size_t>(r0 + r) * p.ldb] : 0.0f;
            }
        });
        dev::StaticFor<0, COLS>([&](auto rcst) {
            constexpr int r = decltype(rcst)::value;
            xs[XOff<COLS>(i, r)] = v[r];
        });
    }
    Sync<WAVES>();
    const bool vec = p.lda % 4 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0;
    const auto solve = [&](auto lower, auto unitDiag, auto tr) {
        constexpr bool kLower = decltype(lower)::value;
        constexpr bool kUnit = decltype(unitDiag)::value;
        constexpr bool kTr = decltype(tr)::value;
        const Tiles<kLower, kTr, COLS> T(A, p.lda, n, vec, xs);
        if constexpr (WAVES == 1) {
            SolveAlone<kLower, kUnit, kTr>(T, diag[group]);
        } else {
            SolveShared<kLower, kUnit, kTr, WAVES, COLS>(T, wave, diag);
        }
    };
    if constexpr (MODE == kSolveT) {
        // U^T y = b (lower), then L^T z = y (unit upper)
        solve(std::true_type{}, std::false_type{}, std::true_type{});
        solve(std::false_type{}, std::true_type{}, std::true_type{});
    } else {
        solve(std::true_type{}, std::true_type{}, std::false_type{});
        int zero = 0;  // the largest j + 1 with u_jj = 0, the same in every wave
        if (MODE == kSolveInv) {
            for (int j0 = 0; j0 < n; j0 += kWave) {
                const int j = j0 + dev::LaneId();
                const bool z = j < n && dev::G(A)[min(j, n - 1) * (static_cast<size_t>(p.lda) + 1)] == 0.0f;
                const uint64_t m = __builtin_amdgcn_ballot_w64(z);
                zero = m != 0 ? j0 + 64 - static_cast<int>(__builtin_clzll(m)) : zero;
            }
            if (chunk == 0 && t == 0) {
                p.info[b] = zero;
            }
        }
        if (zero == 0) {
            solve(std::false_type{}, std::false_type{}, std::false_type{});
        }
    }
    for (int i = t; i < n; i += kThreads) {
        const int row = MODE == kSolveT ? permOf(i) : i;
        dev::StaticFor<0, COLS>([&](auto rcst) {
            constexpr int r = decltype(rcst)::value;
            if (r < rc) {
                B[row + static_cast<size_t>(r0 + r) * p.ldb] = xs[XOff<COLS>(i, r)];
            }
        });
    }
}

template <SolveTileMode MODE, int WAVES, int COLS = kT>
void Launch(hipStream_t st, const SolveTileArgs& p, int batch)
{
    constexpr int kUnits = WAVES == 1 ? 4 : 1;
    const size_t lds = static_cast<size_t>(UnitBytes(p.n, COLS)) * kUnits;
    // slices keep a launch's threads below 2^32
    const int slice = (1 << 21) / p.chunks;
    for (int b0 = 0; b0 < batch; b0 += slice) {
        SolveTileArgs q = p;
        const int count = batch - b0 < slice ? batch - b0 : slice;
        q.A += b0;
        q.B += b0;
        q.ipiv = p.ipiv != nullptr ? p.ipiv + static_cast<size_t>(b0) * p.n : nullptr;
        q.info = p.info != nullptr ? p.info + b0 : nullptr;
        q.units = static_cast<long long>(count) * p.chunks;
        hipLaunchKernelGGL((SolveTileKernel<MODE, WAVES, COLS>),
                           dim3(static_cast<unsigned>((q.units + kUnits - 1) / kUnits)),
                           dim3(WAVES == 1 ? 4 * kWave : WAVES * kWave), lds, st, q);
    }
}

// Many units past order 256: up to four right-hand sides in units of four
// columns, whose LDS is a quarter, so that the registers bound the units on a
// CU and not the LDS.  N, 1 right-hand side, us with sixteen / four columns:
// order 512, 1200 systems 426 / 337; order 700, 1000 systems 613 / 552, 1200 768
// / 646 (the row-per-lane kernel before these: 386, 593 and 648).
template <SolveTileMode MODE, int WAVES>
void LaunchFew(hipStream_t st, const SolveTileArgs& p, int batch)
{
    if constexpr (MODE != kSolveInv) {
        if (p.nrhs <= kFew) {
            Launch<MODE, WAVES, kFew>(st, p, batch);
            return;
        }
    }
    Launch<MODE, WAVES>(st, p, batch);
}

}  // namespace

template <SolveTileMode MODE>
void LaunchSolveTile(hipStream_t st, int n, int nrhs, const float* const* A, int lda, const int* piv, float* const* B,
                     int ldb, int* info, int batch)
{
    const int chunks = (nrhs + kT - 1) / kT;
    const SolveTileArgs p{A, n, lda, piv, B, ldb, nrhs, chunks, info, 0};
    const long long units = static_cast<long long>(batch) * chunks;
    // A wave per unit has no barriers but one wave's latency; a workgroup per
    // unit halves the latency and wastes issue slots on waiting waves.  Order
    // 128, 8 right-hand sides, N: 256 systems 47 (wave) and 34 us (workgroup),
    // 1024: 50 and 50, 2048: 66 and 96; order 250: 1024 systems 131 and 113.
    // Past order 256 (more than 16 tiles) 16 waves have the lowest latency, and
    // fewer of them more units on a CU, up to the orders of which only one fits
    // it.  N, 1 right-hand side, us with 16 / 8 / 4 waves: order 257, 256 systems
    // 64 / 67 / 74, 2000 systems 510 / 327 / 229; order 700, 256 systems 205 /
    // 224 / 327, 1000 systems 823 / 615 / 772; order 1200, 300 systems 861 /
    // 1063 / 1819.  Up to four right-hand sides these take units of four columns.
    if (n <= 256) {
        if (units >= 1536) {
            Launch<MODE, 1>(st, p, batch);
        } else {
            Launch<MODE, 4>(st, p, batch);
        }
    } else if (units > 256 && n <= 512) {
        LaunchFew<MODE, 4>(st, p, batch);
    } else if (units > 256 && n <= 1024) {
        LaunchFew<MODE, 8>(st, p, batch);
    } else {
        Launch<MODE, 16>(st, p, batch);
    }
}

template void LaunchSolveTile<kSolveN>(hipStream_t, int, int, const float* const*, int, const int*, float* const*,
                                       int, int*, int);
template void LaunchSolveTile<kSolveT>(hipStream_t, int, int, const float* const*, int, const int*, float* const*,
                                       int, int*, int);
template void LaunchSolveTile<kSolveInv>(hipStream_t, int, int, const float* const*, int, const int*, float* const*,
                                         int, int*, int);

}  // namespace aclblas
