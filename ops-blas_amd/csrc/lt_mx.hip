// MX block-scaled GEMM behind aclblasLtMatmul: MXFP8 (E4M3FN) x MXFP8 and
// MXFP4 (E2M1) x MXFP4, row-major, D = alpha op(A) op(B) + beta C with FP32 C
// and FP32 or BF16 D.
//
// Reference: blasLt/matmul/mxfp8/arch35/matmul_mxfp8_kernel.cpp,
// blasLt/matmul/mxfp4/arch35/matmul_mxfp4_kernel.cpp and the alpha/beta
// epilogue blasLt/matmul/epilogue/arch35/epilogue_alpha_beta_kernel.cpp; the
// scale layouts are those of the reference's golden
// (test/blasLtMatmul/blasLtMatmul_golden.h:77-91).
//
// MI355X design: the MX format is native to gfx950's
// v_mfma_scale_f32_16x16x128_f8f6f4: each lane feeds 32 K elements of one row
// of its operand (row l % 16) and one E8M0 scale byte per lane, the scale of
// one 32-element K block of that row (the slot layout is at Fragment; the
// result lane holds rows 4 (l / 16) + e, column l % 16).  So one instruction
// consumes four 32-element blocks of A and of B with their scales and no
// dequantisation pass exists.
// The whole scaled product is summed in FP32 by the instruction, alpha / beta
// and the rounding to D's type are fused in the epilogue, and D is written
// once.
//
// One workgroup of four waves (2 x 2) per BT x BT tile of D (eight, 2 x 4, for
// 256 x 256); K advances 128 elements per stage, one barrier per stage.  Aligned
// operands go straight to a ring of LDS stages (LtMxDmaKernel); others through
// registers into two LDS buffers, the next stage's loads in flight while the
// matrix instructions consume this one (LtMxKernel).  An operand stored K-contiguous keeps its rows in LDS (128 bytes for
// FP8, 64 for FP4) and is read 16 bytes at a time; one stored the other way
// keeps its K rows and is read with the transposing ds_read_b64_tr_b8 / _b4, so
// nothing is transposed on the way in.  16-byte chunks are XOR-swizzled so that
// both reads are free of bank conflicts.  Loads are 16 bytes at any alignment;
// only chunks that would end past the operand are read byte by byte.  Rows or
// columns past m / n read other (valid) elements whose results are not stored;
// K blocks past k (k is a multiple of 32) read as zeros with scale 1.  A scale
// byte of 0 makes its block contribute 0, the reference golden's decoding of
// E8M0 0 (the instruction would scale by 2^-127): a stage whose scales hold a
// zero byte has those blocks' data zeroed in LDS.
//
// What bounds it: the LDS round trips at the start of a stage (its fragments
// can only be read after the barrier) against 32 matrix instructions per wave
// with 256 x 256 tiles and 16 with 128 x 128; the larger tile, whose two waves
// per SIMD also cover for each other, reaches 1.6 PFLOP/s (MXFP8: matrix cores
// busy a third of the time; 24 to 92 bytes a lane of that instance live in
// scratch).  4096^3, BF16 out, A and B K-contiguous (NT) / both row-contiguous
// (TN): MXFP8 329 -> 90 / 2537 -> 77 us, MXFP4 176 -> 67 / 1522 -> 55 us (before:
// 64 x 64 tiles, element-wise transposes, no load in flight during the
// products).  Fragments of the next
// stage held in registers during the products were slower (174 us: the
// compiler moves them through the accumulation registers).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.h"
#include "drivers.h"
#include "internal.h"
#include "lds_dma.h"

namespace aclblas {
namespace {

constexpr int kStepK = 128;     // K elements per stage (one MFMA per fragment pair)

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4Any __attribute__((aligned(1)));
typedef uint16_t u16Any __attribute__((aligned(1)));
typedef int V2i32 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) V2i32 LdsV2i32;

struct MxArgs {
    const uint8_t* A;
    const uint8_t* B;
    const uint8_t* scaleA;
    const uint8_t* scaleB;
    const float* C;
    void* D;
    long long pitchA;   // bytes between rows of A as stored
    long long pitchB;
    int m, n, k;
    int ldc, ldd;
    int tilesM, tilesN;
    int vecC, vecD;     // four consecutive elements of a row can move as one vector
    int bf16Out;
    int dma;            // the direct-to-LDS kernel may run
    float alpha, beta;
};

// Workgroup of a BT x BT tile: 2 x 2 waves, or 2 x 4 for the largest tile.
constexpr int Threads(int bt) { return bt == 256 ? 512 : 256; }
constexpr int WavesN(int bt) { return bt == 256 ? 4 : 2; }

// One operand's tile of BT rows (m or n indices).  KC: stored K-contiguous
// (element (row, kk) at row * pitch + kk, FP4 nibbles two per byte), else
// row-contiguous (at kk * pitch + row).
template <bool FP4, bool KC, int BT>
struct Operand {
    static constexpr int kThreads = Threads(BT);
    static constexpr int kRowBytes = KC ? (FP4 ? 64 : 128) : (FP4 ? BT / 2 : BT);  // an LDS row
    static constexpr int kRowChunks = kRowBytes / 16;
    static constexpr int kBytes = BT * (FP4 ? 64 : 128);                           // a stage
    static constexpr int kLoads = kBytes / 16 / kThreads;
    const uint8_t* src[kLoads];  // this thread's chunks at stage 0
    const uint8_t* end;          // past the operand's last byte
    long long step;
    int kEnd;                    // K elements
    bool inside;                 // row-contiguous: every chunk of the tile inside its row

    // swizzle key of LDS row r: rows that are read together land in distinct
    // chunks of a 256-byte window
    __device__ __forceinline__ static int Key(int r)
    {
        if (KC) {
            return FP4 ? (r >> 1) & 3 : r & 7;
        }
        return kRowChunks >= 8 ? r & 7 : (kRowChunks == 4 ? (r >> 2) & 3 : (r >> 3) & 1);
    }
    __device__ __forceinline__ static uint32_t Offset(int r, int chunk)
    {
        return static_cast<uint32_t>(r * kRowBytes + ((chunk ^ Key(r)) << 4));
    }

    __device__ __forceinline__ void Setup(const uint8_t* X, long long pitch, int row0, int rows, int k)
    {
        const int t = threadIdx.x;
        const int rowBytes = FP4 ? (rows + 1) / 2 : rows;  // row-contiguous storage
        const int byte0 = FP4 ? row0 / 2 : row0;
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const int id = t + kThreads * q;
            const int r = id / kRowChunks;
            const int c = id % kRowChunks;
            src[q] = KC ? X + static_cast<long long>(min(row0 + r, rows - 1)) * pitch + 16 * c
                        : X + static_cast<long long>(r) * pitch + byte0 + 16 * c;
        }
        step = KC ? static_cast<long long>(kRowBytes) : kStepK * pitch;
        end = KC ? nullptr : X + static_cast<long long>(k - 1) * pitch + rowBytes;
        kEnd = k;
        inside = KC || byte0 + kRowBytes <= rowBytes;
    }

    __device__ __forceinline__ void Load(int stage, u32x4 (&v)[kLoads]) const
    {
        const long long off = stage * step;
        const int left = kEnd - stage * kStepK;  // K elements from this stage on
        if (left >= kStepK && inside) {
#pragma unroll
            for (int q = 0; q < kLoads; ++q) {
                v[q] = *(const ACL_GLOBAL u32x4Any*)(src[q] + off);
            }
            return;
        }
        const int t = threadIdx.x;
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const int id = t + kThreads * q;
            const uint8_t* p = src[q] + off;
            u32x4 w = {0u, 0u, 0u, 0u};
            if (KC) {
                if ((id % kRowChunks) * (FP4 ? 32 : 16) < left) {
                    w = *(const ACL_GLOBAL u32x4Any*)p;
                }
            } else if (id / kRowChunks < left) {
                if (p + 16 <= end) {
                    w = *(const ACL_GLOBAL u32x4Any*)p;
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        if (p + i < end) {
                            w[i / 4] |= static_cast<uint32_t>(dev::LoadG<uint8_t>(p + i)) << (8 * (i % 4));
                        }
                    }
                }
            }
            v[q] = w;
        }
    }

    // The sources of a direct-to-LDS stage: a wave instruction fills 64
    // consecutive 16-byte slots, so each lane fetches the chunk that belongs in
    // its slot.  Rows past the edge, and chunks past a row's end (row-contiguous
    // rows are whole chunks then), read clamped addresses.
    __device__ __forceinline__ void SetupDma(const uint8_t* X, long long pitch, int row0, int rows)
    {
        const int t = threadIdx.x;
        const int rowBytes = FP4 ? rows / 2 : rows;
        const int byte0 = FP4 ? row0 / 2 : row0;
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const int id = t + kThreads * q;
            const int r = id / kRowChunks;
            const int c = (id % kRowChunks) ^ Key(r);
            src[q] = KC ? X + static_cast<long long>(min(row0 + r, rows - 1)) * pitch + 16 * c
                        : X + static_cast<long long>(r) * pitch + min(byte0 + 16 * c, rowBytes - 16);
        }
        step = KC ? static_cast<long long>(kRowBytes) : kStepK * pitch;
    }
    __device__ __forceinline__ void Issue(int stage, uint8_t* lds, int wave) const
    {
        const uint32_t base = dev::LdsAddr(lds);
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            dev::LdsDma16(src[q] + stage * step,
                          __builtin_amdgcn_readfirstlane(base + 1024u * (wave + kThreads / 64 * q)));
        }
    }

    __device__ __forceinline__ void Store(uint8_t* lds, const u32x4 (&v)[kLoads]) const
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const int id = t + kThreads * q;
            *reinterpret_cast<u32x4*>(lds + Offset(id / kRowChunks, id % kRowChunks)) = v[q];
        }
    }

    // A lane's operand of v_mfma_scale_f32_16x16x128_f8f6f4 for the 16 rows from
    // row0 of the tile (row0 a multiple of 16).  The instruction's K slots,
    // established on the GPU, are:
    //   FP8: the lane's bytes 0-15 are slots 16 g .. 16 g + 15 and bytes 16-31
    //        are slots 64 + 16 g .. 64 + 16 g + 15 (g = lane / 16); the scale the
    //        lane supplies covers slots 32 g .. 32 g + 31;
    //   FP4: the lane's 32 elements are slots 32 g .. 32 g + 31 and its scale
    //        covers them.
    // Slot s holds K element k0 + s.  ds_read_b64_tr_b8: in a group of 16 lanes,
    // lane 2 e + a pointing at rows 8a .. 8a + 7 of K element e gives lane i row
    // i, elements 0..7; ds_read_b64_tr_b4: lane e pointing at the 16 rows of K
    // element e gives lane i row i, elements 0..15.
    __device__ __forceinline__ static i32x8 Fragment(const uint8_t* lds, int row0, int lane)
    {
        const int g = lane >> 4;
        const int j = lane & 15;
        if constexpr (KC) {
            const int r = row0 + j;
            const u32x4 lo = *reinterpret_cast<const u32x4*>(lds + Offset(r, g));
            if constexpr (FP4) {
                return i32x8{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z),
                             static_cast<int>(lo.w), 0, 0, 0, 0};
            } else {
                const u32x4 hi = *reinterpret_cast<const u32x4*>(lds + Offset(r, 4 + g));
                return i32x8{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z),
                             static_cast<int>(lo.w), static_cast<int>(hi.x), static_cast<int>(hi.y),
                             static_cast<int>(hi.z), static_cast<int>(hi.w)};
            }
        } else if constexpr (FP4) {
            V2i32 v[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint8_t* p = lds + Offset(32 * g + 16 * h + j, row0 >> 5) + ((row0 >> 4) & 1) * 8;
                v[h] = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2i32*)p);
            }
            return i32x8{v[0].x, v[0].y, v[1].x, v[1].y, 0, 0, 0, 0};
        } else {
            V2i32 v[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int k = (h >> 1) * 64 + 16 * g + 8 * (h & 1) + (j >> 1);
                const uint8_t* p = lds + Offset(k, row0 >> 4) + 8 * (j & 1);
                v[h] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2i32*)p);
            }
            return i32x8{v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, v[3].x, v[3].y};
        }
    }
};

// Zeroes in LDS the blocks of the wave's rows (row0 .. row0 + ROWS - 1 of the
// operand's tile, one per lane) whose scale byte is 0; scales(row) gives a
// row's four.  Other waves that use the rows write the same zeros before they
// read them, so no barrier is needed; and no accumulator is live across the
// branch (one would be moved to and from the accumulation registers on every
// stage).
template <typename Op, bool FP4, bool KC, int ROWS, typename Scales>
__device__ __forceinline__ void ZeroBlocks(uint8_t* lds, int row0, int lane, Scales scales)
{
    constexpr int kSlabs = ROWS > 64 ? ROWS / 64 : 1;
    uint32_t s[kSlabs];
    uint32_t z = 0;
#pragma unroll
    for (int q = 0; q < kSlabs; ++q) {
        s[q] = scales(row0 + 64 * q + lane % min(ROWS, 64));
        z |= (s[q] - 0x01010101u) & ~s[q] & 0x80808080u;  // 0 exactly when no byte is 0
    }
    if (__builtin_amdgcn_ballot_w64(z != 0u) == 0) {
        return;
    }
    for (int e = 0; e < 4 * kSlabs; ++e) {
        const int b = e & 3;
        const int row = row0 + 64 * (e >> 2) + lane % min(ROWS, 64);
        if (((s[e >> 2] >> (8 * b)) & 0xFFu) != 0u) {
            continue;
        }
        if constexpr (KC) {
            constexpr int kChunks = FP4 ? 1 : 2;
            for (int c = 0; c < kChunks; ++c) {
                *reinterpret_cast<u32x4*>(lds + Op::Offset(row, kChunks * b + c)) = u32x4{0u, 0u, 0u, 0u};
            }
        } else if constexpr (!FP4) {
            for (int k = 32 * b; k < 32 * b + 32; ++k) {
                lds[Op::Offset(k, row >> 4) + (row & 15)] = 0;
            }
        } else {
            // the neighbouring row shares the byte
            for (int k = 32 * b; k < 32 * b + 32; ++k) {
                const uint32_t at = Op::Offset(k, row >> 5) + ((row & 31) >> 1);
                atomicAnd(reinterpret_cast<uint32_t*>(lds + (at & ~3u)),
                          ~(0xFu << (8 * (at & 3u) + 4 * (row & 1))));
            }
        }
    }
}

// The four scale bytes of a stage (K blocks 4 s .. 4 s + 3) of matrix row `row`
// (of `rows`), as two pairs.  pairsMajor: the [b / 2][rows][2] layout, else
// [rows][2 ceil(k / 64)].  Blocks past k scale by 1.
__device__ __forceinline__ uint32_t LoadScales(const uint8_t* s, bool pairsMajor, int rows, int row, int stage, int k)
{
    const int pairs = (k + 63) / 64;
    uint32_t v = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int pb = 2 * stage + h;
        const int at = min(pb, pairs - 1);
        const long long off = pairsMajor ? (static_cast<long long>(at) * rows + row) * 2
                                         : (static_cast<long long>(row) * pairs + at) * 2;
        uint32_t w = *(const ACL_GLOBAL u16Any*)(s + off);
        w = 64 * pb + 32 < k ? w : ((w & 0xFFu) | 0x7F00u);
        w = pb < pairs ? w : 0x7F7Fu;
        v |= w << (16 * h);
    }
    return v;
}

__device__ __forceinline__ uint16_t Bf16Rne(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) {
        return static_cast<uint16_t>((u >> 16) | 0x40u);
    }
    u += 0x7FFFu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

// One 2-byte value per lane to consecutive LDS dwords (zero-extended); as
// dev::LdsDma16 otherwise.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void LdsDma2(const void* g, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_ushort %0, off" : : "v"(g), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// The tile a workgroup computes: consecutive tiles on one XCD, walked in
// groups of eight tile rows that share its L2.
template <int BT>
__device__ __forceinline__ void TileOf(const MxArgs& p, int& m0, int& n0)
{
    int bid = static_cast<int>(blockIdx.x);
    if (gridDim.x % 8 == 0) {
        bid = (bid % 8) * (static_cast<int>(gridDim.x) / 8) + bid / 8;
    }
    const int perGroup = 8 * p.tilesN;
    const int firstM = bid / perGroup * 8;
    const int groupRows = min(8, p.tilesM - firstM);
    const int inGroup = bid - bid / perGroup * perGroup;
    m0 = (firstM + inGroup % groupRows) * BT;
    n0 = inGroup / groupRows * BT;
}

// alpha * acc + beta * C for a wave's kF x kF tiles at (mw, nw): the lane holds
// row r16, columns 4 g + e of each 16 x 16 tile.
template <int kFA, int kFB>
__device__ __forceinline__ void StoreTiles(const MxArgs& p, const f32x4 (&acc)[kFA][kFB], int mw, int nw, int lane)
{
    const int r16 = lane & 15;
    const int g = lane >> 4;
#pragma unroll
    for (int i = 0; i < kFA; ++i) {
        const int row = mw + 16 * i + r16;
#pragma unroll
        for (int j = 0; j < kFB; ++j) {
            const int col = nw + 16 * j + 4 * g;
            if (row >= p.m || col >= p.n) {
                continue;
            }
            const int left = min(4, p.n - col);
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = p.alpha * acc[i][j][e];
            }
            if (p.beta != 0.0f) {
                const float* c = p.C + static_cast<size_t>(row) * p.ldc + col;
                if (p.vecC != 0 && left == 4) {
                    const f32x4 cv = dev::LoadG<f32x4>(c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = fmaf(p.beta, cv[e], v[e]);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (e < left) {
                            v[e] = fmaf(p.beta, dev::LoadG<float>(c + e), v[e]);
                        }
                    }
                }
            }
            const size_t at = static_cast<size_t>(row) * p.ldd + col;
            if (p.bf16Out != 0) {
                uint16_t* d = static_cast<uint16_t*>(p.D) + at;
                const uint32_t lo = Bf16Rne(v[0]) | (static_cast<uint32_t>(Bf16Rne(v[1])) << 16);
                const uint32_t hi = Bf16Rne(v[2]) | (static_cast<uint32_t>(Bf16Rne(v[3])) << 16);
                if (p.vecD != 0 && left == 4) {
                    dev::StoreG(d, make_uint2(lo, hi));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (e < left) {
                            dev::StoreG(d + e, static_cast<uint16_t>((e < 2 ? lo : hi) >> (16 * (e & 1))));
                        }
                    }
                }
            } else {
                float* d = static_cast<float*>(p.D) + at;
                if (p.vecD != 0 && left == 4) {
                    dev::StoreG(d, f32x4{v[0], v[1], v[2], v[3]});
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (e < left) {
                            dev::StoreG(d + e, v[e]);
                        }
                    }
                }
            }
        }
    }
}

template <bool FP4, bool AK, bool BK, int BT>
__global__ __launch_bounds__(256, 2) void LtMxKernel(MxArgs p)
{
    constexpr int kFmt = FP4 ? 4 : 0;  // operand format code: 0 E4M3, 4 E2M1
    constexpr int kF = BT / 32;        // 16-row fragments per wave and operand
    using OpA = Operand<FP4, AK, BT>;
    using OpB = Operand<FP4, BK, BT>;
    __shared__ __attribute__((aligned(16))) uint8_t sA[2][OpA::kBytes];
    __shared__ __attribute__((aligned(16))) uint8_t sB[2][OpB::kBytes];
    __shared__ uint32_t sS[2][2 * BT];  // scales of A's rows, then of B's

    int m0, n0;
    TileOf<BT>(p, m0, n0);
    const int t = static_cast<int>(threadIdx.x);
    const int lane = t & 63;
    const int wave = dev::Uniform(t >> 6);
    const int wm = (wave >> 1) * (BT / 2);
    const int wn = (wave & 1) * (BT / 2);
    const int r16 = lane & 15;
    const int g = lane >> 4;

    OpA oa;
    OpB ob;
    oa.Setup(p.A, p.pitchA, m0, p.m, p.k);
    ob.Setup(p.B, p.pitchB, n0, p.n, p.k);
    // A: scales [m][2 ceil(k/64)] when stored K-contiguous, else pairs-major; B the same way
    const bool forA = t < BT;
    const int srow = forA ? min(m0 + t, p.m - 1) : min(n0 + t - BT, p.n - 1);
    const auto loadScales = [&](int stage) {
        return forA ? LoadScales(p.scaleA, !AK, p.m, srow, stage, p.k)
                    : LoadScales(p.scaleB, !BK, p.n, srow, stage, p.k);
    };

    f32x4 acc[kF][kF];
#pragma unroll
    for (int i = 0; i < kF; ++i) {
#pragma unroll
        for (int j = 0; j < kF; ++j) {
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    u32x4 va[OpA::kLoads], vb[OpB::kLoads];
    uint32_t vs = 0;
    const auto load = [&](int stage) {
        oa.Load(stage, va);
        ob.Load(stage, vb);
        if (t < 2 * BT) {
            vs = loadScales(stage);
        }
    };
    const auto store = [&](int buf) {
        oa.Store(sA[buf], va);
        ob.Store(sB[buf], vb);
        if (t < 2 * BT) {
            sS[buf][t] = vs;
        }
    };
    const int stages = (p.k + kStepK - 1) / kStepK;
    if (stages > 0) {
        load(0);
        store(0);
    }
    __syncthreads();
    for (int s = 0; s < stages; ++s) {
        const int buf = s & 1;
        if (s + 1 < stages) {
            load(s + 1);
        }
        ZeroBlocks<OpA, FP4, AK, BT / 2>(sA[buf], wm, lane, [&](int r) { return sS[buf][r]; });
        ZeroBlocks<OpB, FP4, BK, BT / 2>(sB[buf], wn, lane, [&](int r) { return sS[buf][BT + r]; });
        i32x8 b[kF];
        uint32_t sb[kF];
#pragma unroll
        for (int j = 0; j < kF; ++j) {
            b[j] = OpB::Fragment(sB[buf], wn + 16 * j, lane);
            sb[j] = sS[buf][BT + wn + 16 * j + r16] >> (8 * g);
        }
#pragma unroll
        for (int i = 0; i < kF; ++i) {
            const i32x8 a = OpA::Fragment(sA[buf], wm + 16 * i, lane);
            const uint32_t sa = sS[buf][wm + 16 * i + r16] >> (8 * g);
            // transposed product: a lane holds four consecutive columns of D
#pragma unroll
            for (int j = 0; j < kF; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                    b[j], a, acc[i][j], kFmt, kFmt, 0, static_cast<int>(sb[j]), 0, static_cast<int>(sa));
            }
        }
        if (s + 1 < stages) {
            store(buf ^ 1);
        }
        __syncthreads();
    }
    StoreTiles<kF, kF>(p, acc, m0 + wm, n0 + wn, lane);
}

// The same tile with direct-to-LDS loads: a ring of four stages, three in
// flight (two stages where the largest FP8 tile fills LDS with them).  Both operands' and the
// scales' chunks go straight to LDS; a last partial stage is loaded through
// registers with zero fill.  Needs 16-byte aligned operand rows (and whole
// chunks per row where they are row-contiguous) and 2-byte aligned scales.
template <bool FP4, bool AK, bool BK, int BT>
__global__ __launch_bounds__(Threads(BT)) void LtMxDmaKernel(MxArgs p)
{
    constexpr int kFmt = FP4 ? 4 : 0;
    constexpr int kFA = BT / 32;               // 16-row fragments per wave
    constexpr int kFB = BT / WavesN(BT) / 16;
    constexpr int kWaves = Threads(BT) / 64;
    // four stages while they fit, of the largest FP8 tile two
    constexpr int kStages = BT == 256 && !FP4 ? 2 : 4;
    using OpA = Operand<FP4, AK, BT>;
    using OpB = Operand<FP4, BK, BT>;
    // scales: [A, B][block pair of the stage][row], one pair per dword
    constexpr int kScaleLoads = 4 * BT / 64 / kWaves;
    constexpr int kPerStage = OpA::kLoads + OpB::kLoads + kScaleLoads;
    struct Stage {
        uint8_t a[OpA::kBytes];
        uint8_t b[OpB::kBytes];
        uint32_t s[2][2][BT];
    };
    __shared__ __attribute__((aligned(1024))) Stage ring[kStages];

    int m0, n0;
    TileOf<BT>(p, m0, n0);
    const int t = static_cast<int>(threadIdx.x);
    const int lane = t & 63;
    const int wave = dev::Uniform(t >> 6);
    const int wm = (wave / WavesN(BT)) * (BT / 2);
    const int wn = (wave % WavesN(BT)) * (BT / WavesN(BT));
    const int r16 = lane & 15;
    const int g = lane >> 4;
    const int nFull = p.k / kStepK;
    const int stages = (p.k + kStepK - 1) / kStepK;

    OpA oa;
    OpB ob;
    oa.SetupDma(p.A, p.pitchA, m0, p.m);
    ob.SetupDma(p.B, p.pitchB, n0, p.n);
    const int pairs = (p.k + 63) / 64;
    const uint8_t* ssrc[kScaleLoads];
    long long sstep[kScaleLoads];
#pragma unroll
    for (int y = 0; y < kScaleLoads; ++y) {
        const int idx = 64 * (wave + kWaves * y) + lane;
        const bool forA = idx < 2 * BT;
        const int h = (idx / BT) & 1;
        const bool pairsMajor = forA ? !AK : !BK;
        const int rows = forA ? p.m : p.n;
        const int row = min((forA ? m0 : n0) + idx % BT, rows - 1);
        ssrc[y] = (forA ? p.scaleA : p.scaleB) +
                  2 * (pairsMajor ? static_cast<long long>(min(h, pairs - 1)) * rows + row
                                  : static_cast<long long>(row) * pairs + min(h, pairs - 1));
        sstep[y] = pairsMajor ? 4ll * rows : 4;
    }
    const auto issue = [&](int s) {
        Stage& st = ring[s % kStages];
        if (s < nFull) {
            oa.Issue(s, st.a, wave);
            ob.Issue(s, st.b, wave);
            const uint32_t base = dev::LdsAddr(&st.s[0][0][0]);
#pragma unroll
            for (int y = 0; y < kScaleLoads; ++y) {
                LdsDma2(ssrc[y] + s * sstep[y],
                        __builtin_amdgcn_readfirstlane(base + 256u * (wave + kWaves * y)));
            }
        } else {
            OpA ta;
            OpB tb;
            ta.Setup(p.A, p.pitchA, m0, p.m, p.k);
            tb.Setup(p.B, p.pitchB, n0, p.n, p.k);
            u32x4 va[OpA::kLoads], vb[OpB::kLoads];
            ta.Load(s, va);
            tb.Load(s, vb);
            ta.Store(st.a, va);
            tb.Store(st.b, vb);
            if (t < 2 * BT) {  // 256 or 512 threads: one row each
                const bool forA = t < BT;
                const int row = forA ? min(m0 + t, p.m - 1) : min(n0 + t - BT, p.n - 1);
                const uint32_t v = forA ? LoadScales(p.scaleA, !AK, p.m, row, s, p.k)
                                        : LoadScales(p.scaleB, !BK, p.n, row, s, p.k);
                st.s[forA ? 0 : 1][0][t % BT] = v & 0xFFFFu;
                st.s[forA ? 0 : 1][1][t % BT] = v >> 16;
            }
        }
    };

    f32x4 acc[kFA][kFB];
#pragma unroll
    for (int i = 0; i < kFA; ++i) {
#pragma unroll
        for (int j = 0; j < kFB; ++j) {
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    for (int s = 0; s < kStages - 1 && s < stages; ++s) {
        issue(s);
    }
    for (int s = 0; s < stages; ++s) {
        // this wave's stages after s may stay in flight
        const int pending = kStages == 2 ? 0 : (s + 1 < nFull ? 1 : 0) + (s + 2 < nFull ? 1 : 0);
        if (pending == 2) {
            dev::WaitVmcnt<2 * kPerStage>();
        } else if (pending == 1) {
            dev::WaitVmcnt<kPerStage>();
        } else {
            dev::WaitVmcnt<0>();
        }
        dev::BarrierLds();
        Stage& st = ring[s % kStages];
        // the next loads go out before the products, which do not wait for them
        if (s + kStages - 1 < stages) {
            issue(s + kStages - 1);
        }
        ZeroBlocks<OpA, FP4, AK, BT / 2>(st.a, wm, lane,
                                         [&](int r) { return st.s[0][0][r] | (st.s[0][1][r] << 16); });
        ZeroBlocks<OpB, FP4, BK, BT / WavesN(BT)>(st.b, wn, lane,
                                                  [&](int r) { return st.s[1][0][r] | (st.s[1][1][r] << 16); });
        i32x8 b[kFB];
        uint32_t sb[kFB];
#pragma unroll
        for (int j = 0; j < kFB; ++j) {
            b[j] = OpB::Fragment(st.b, wn + 16 * j, lane);
            sb[j] = st.s[1][g >> 1][wn + 16 * j + r16] >> (8 * (g & 1));
        }
#pragma unroll
        for (int i = 0; i < kFA; ++i) {
            const i32x8 a = OpA::Fragment(st.a, wm + 16 * i, lane);
            const uint32_t sa = st.s[0][g >> 1][wm + 16 * i + r16] >> (8 * (g & 1));
#pragma unroll
            for (int j = 0; j < kFB; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                    b[j], a, acc[i][j], kFmt, kFmt, 0, static_cast<int>(sb[j]), 0, static_cast<int>(sa));
            }
        }
    }
    StoreTiles<kFA, kFB>(p, acc, m0 + wm, n0 + wn, lane);
}

template <bool FP4, bool AK, bool BK>
void Launch(hipStream_t st, MxArgs p)
{
    // Largest tiles that still give (about) every CU one: larger tiles need
    // fewer LDS bytes per product, fewer tiles leave CUs idle.  MXFP8 NT: 4096^3
    // 92 us with 256 tiles (143 with 128); 2048^3 46 us with 256 and 23 with 128
    // tiles; 1024 x 1024 x 4096 36 us with 128 and 17 with 64.  (3072^3, 144 tiles
    // of 256, takes 84 us with 128 tiles and would take 64 with 256.)
    const auto tiles = [&](int bt) {
        p.tilesM = (p.m + bt - 1) / bt;
        p.tilesN = (p.n + bt - 1) / bt;
        return static_cast<long long>(p.tilesM) * p.tilesN;
    };
    if (p.dma != 0 && tiles(256) >= 192) {
        const dim3 grid(static_cast<unsigned>(tiles(256)));
        hipLaunchKernelGGL((LtMxDmaKernel<FP4, AK, BK, 256>), grid, dim3(Threads(256)), 0, st, p);
        return;
    }
    const bool big = tiles(128) >= 256;
    const dim3 grid(static_cast<unsigned>(tiles(big ? 128 : 64)));
    if (p.dma != 0) {
        if (big) {
            hipLaunchKernelGGL((LtMxDmaKernel<FP4, AK, BK, 128>), grid, dim3(256), 0, st, p);
        } else {
            hipLaunchKernelGGL((LtMxDmaKernel<FP4, AK, BK, 64>), grid, dim3(256), 0, st, p);
        }
    } else {
        if (big) {
            hipLaunchKernelGGL((LtMxKernel<FP4, AK, BK, 128>), grid, dim3(256), 0, st, p);
        } else {
            hipLaunchKernelGGL((LtMxKernel<FP4, AK, BK, 64>), grid, dim3(256), 0, st, p);
        }
    }
}

template <bool FP4>
void LaunchTrans(hipStream_t st, bool aK, bool bK, const MxArgs& p)
{
    if (aK) {
        bK ? Launch<FP4, true, true>(st, p) : Launch<FP4, true, false>(st, p);
    } else {
        bK ? Launch<FP4, false, true>(st, p) : Launch<FP4, false, false>(st, p);
    }
}

}  // namespace

aclblasStatus_t LtMxLaunch(hipStream_t st, bool fp4, bool transA, bool transB, int m, int n, int k, float alpha,
                           const void* A, long long lda, const void* B, long long ldb, const void* scaleA,
                           const void* scaleB, float beta, const float* C, int ldc, void* D, int ldd, bool bf16Out)
{
    MxArgs p{};
    p.A = static_cast<const uint8_t*>(A);
    p.B = static_cast<const uint8_t*>(B);
    p.scaleA = static_cast<const uint8_t*>(scaleA);
    p.scaleB = static_cast<const uint8_t*>(scaleB);
    p.C = C;
    p.D = D;
    p.pitchA = lda;  // bytes per stored row (FP4: two elements per byte)
    p.pitchB = ldb;
    p.m = m;
    p.n = n;
    p.k = k;
    p.ldc = ldc;
    p.ldd = ldd;
    p.vecC = (C != nullptr && reinterpret_cast<uintptr_t>(C) % 16 == 0 && ldc % 4 == 0) ? 1 : 0;
    p.vecD = (reinterpret_cast<uintptr_t>(D) % (bf16Out ? 8 : 16) == 0 && ldd % 4 == 0) ? 1 : 0;
    p.bf16Out = bf16Out ? 1 : 0;
    // direct-to-LDS: aligned rows, and row-contiguous rows of whole 16-byte chunks
    const int rowAlign = fp4 ? 32 : 16;
    const bool alignedOps = reinterpret_cast<uintptr_t>(A) % 16 == 0 && lda % 16 == 0 &&
                            reinterpret_cast<uintptr_t>(B) % 16 == 0 && ldb % 16 == 0;
    p.dma = (alignedOps && (!transA || m % rowAlign == 0) && (transB || n % rowAlign == 0) &&
             reinterpret_cast<uintptr_t>(scaleA) % 2 == 0 && reinterpret_cast<uintptr_t>(scaleB) % 2 == 0)
                ? 1
                : 0;
    p.alpha = alpha;
    p.beta = beta;
    // A is K-contiguous when it is not transposed, B when it is
    if (fp4) {
        LaunchTrans<true>(st, !transA, transB, p);
    } else {
        LaunchTrans<false>(st, !transA, transB, p);
    }
    return LaunchStatus("aclblasLtMatmul");
}

}  // namespace aclblas
