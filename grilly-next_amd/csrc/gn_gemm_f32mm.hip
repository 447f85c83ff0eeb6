// gn_gemm_f32mm.hip — fp32 products on the fp32 matrix instruction, any size and alignment.
//
// v_mfma_f32_32x32x2_f32 multiplies and adds in fp32 (an inf stays an inf, as in an FMA chain), so
// this path keeps the semantics of scalar FMA code at up to 157 TFLOP/s.  It takes the shapes the
// six-product bf16 split (gn_gemm_f32.hip) does not (sizes that are not multiples of 4, unaligned
// operands) and those that would give that kernel a few blocks only.
//
// No LDS staging and no barrier in the main loop: a wave owns a 32 x 32 tile and reads its
// operands straight into the instruction's registers.  Lane l holds row l % 32 (of op(A), and of
// op(B)^T) and of every 8 k the four from 4 (l / 32): a k-contiguous operand is one 16-byte load per
// lane (any alignment), a k-outer one four dwords whose 32 lanes are consecutive.  The next 32 k
// are loaded while the current ones are multiplied.  The KS waves of a block share one tile and
// take every KS-th 32-k chunk; their partial sums are added in wave order through LDS.
#include <algorithm>

#include "gn_common.h"
#include "gn_gemm_dma.h"
#include "gn_mfma.h"

namespace gn {
namespace {

constexpr int CK = 32;  // k per chunk

struct Chunk {
    float4 v[CK / 8];
};

// 32 k of one operand row (the lane's four of every eight) from k0; rows are clamped by the
// caller, k past klim reads as zero (from a clamped address).
template <bool KC>
__device__ __forceinline__ void load_chunk(const float* __restrict__ P, int ld, int row, int k0, int klim,
                                           Chunk& c) {
    const int h4 = ((threadIdx.x & 63) >> 5) * 4;
    if (k0 + CK <= klim) {
#pragma unroll
        for (int s = 0; s < CK / 8; ++s) {
            const int k = k0 + 8 * s + h4;
            if (KC) {
                __builtin_memcpy(&c.v[s], P + (size_t)row * ld + k, 16);
            } else {
                const float* p = P + (size_t)k * ld + row;
                c.v[s] = make_float4(p[0], p[ld], p[2 * (size_t)ld], p[3 * (size_t)ld]);
            }
        }
        return;
    }
#pragma unroll
    for (int s = 0; s < CK / 8; ++s) {
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = k0 + 8 * s + h4 + e, kc = min(k, klim - 1);
            const float y = P[KC ? (size_t)row * ld + kc : (size_t)kc * ld + row];
            x[e] = k < klim ? y : 0.f;
        }
        c.v[s] = make_float4(x[0], x[1], x[2], x[3]);
    }
}

__device__ __forceinline__ f32x16_t mul_chunk(const Chunk& a, const Chunk& b, f32x16_t acc) {
#pragma unroll
    for (int s = 0; s < CK / 8; ++s) {
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[s].x, b.v[s].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[s].y, b.v[s].y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[s].z, b.v[s].z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[s].w, b.v[s].w, acc, 0, 0, 0);
    }
    return acc;
}

template <bool TA, bool TB, int KS>
__global__ __launch_bounds__(64 * KS) void gemm_f32mm(GemmDesc g) {
    const int tilesM = (g.M + 31) / 32, tilesN = (g.N + 31) / 32;
    const int nblk = tilesM * tilesN;
    // one contiguous range of tiles per XCD, walked eight tile rows at a time
    const int xcd = blockIdx.x & 7, per = nblk >> 3, extra = nblk & 7;
    const int pid = xcd * per + min(xcd, extra) + ((int)blockIdx.x >> 3);
    const int group_id = pid / (8 * tilesN);
    const int first_m = group_id * 8;
    const int gsize = min(tilesM - first_m, 8);
    const int in_group = pid % (8 * tilesN);
    const int m0 = (first_m + in_group % gsize) * 32, n0 = (in_group / gsize) * 32;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = min(m0 + (lane & 31), g.M - 1), col = min(n0 + (lane & 31), g.N - 1);

    const int c0 = (g.Ks[0] + CK - 1) / CK;
    const int nc = c0 + (g.nseg > 1 ? (g.Ks[1] + CK - 1) / CK : 0);
    auto load = [&](int c, Chunk& a, Chunk& b) {
        const int s = c >= c0 ? 1 : 0, k0 = (s ? c - c0 : c) * CK;
        load_chunk<!TA>(reinterpret_cast<const float*>(g.A[s]), g.lda[s], row, k0, g.Ks[s], a);
        load_chunk<TB>(reinterpret_cast<const float*>(g.B[s]), g.ldb[s], col, k0, g.Ks[s], b);
    };
    f32x16_t acc;
    zero16(acc);
    Chunk a0, b0, a1, b1;
    int c = wave;
    if (c < nc) load(c, a0, b0);
    while (c < nc) {
        if (c + KS < nc) load(c + KS, a1, b1);
        acc = mul_chunk(a0, b0, acc);
        c += KS;
        if (c >= nc) break;
        if (c + KS < nc) load(c + KS, a0, b0);
        acc = mul_chunk(a1, b1, acc);
        c += KS;
    }

    // partial tiles to LDS, then each wave finishes 1 / KS of the tile's elements
    __shared__ float sh[KS][16][64];
#pragma unroll
    for (int r = 0; r < 16; ++r) sh[wave][r][lane] = acc[r];
    __syncthreads();
    for (int r = wave; r < 16; r += KS) {
        float v = sh[0][r][lane];
#pragma unroll
        for (int w = 1; w < KS; ++w) v += sh[w][r][lane];
        const int m = m0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), n = n0 + (lane & 31);
        if (m < g.M && n < g.N) gemm_store<float, 0>(g, m, n, v);
    }
}

inline long tiles32(const GemmDesc& g) { return (long)((g.M + 31) / 32) * ((g.N + 31) / 32); }

// Eight waves per tile from 1024 tiles on (8001 x 1535 x 512: 198 -> 192 us, 2047 x 1023 x 1023: 77.7 ->
// 71.5 us against four); below, four leave more tiles in flight (512 x 1535 x 1535 43.0 -> 41.3 us,
// 163 x 88 x 1182 13.2 -> 11.3 us).
inline int split_of(const GemmDesc& g) { return tiles32(g) >= 1024 ? 8 : 4; }

template <int KS>
int launch_mm(const GemmDesc& g, int ta, int tb, hipStream_t s) {
    const unsigned grid = (unsigned)tiles32(g), nt = 64 * KS;
    if (!ta && !tb) gemm_f32mm<false, false, KS><<<grid, nt, 0, s>>>(g);
    else if (!ta && tb) gemm_f32mm<false, true, KS><<<grid, nt, 0, s>>>(g);
    else if (ta && !tb) gemm_f32mm<true, false, KS><<<grid, nt, 0, s>>>(g);
    else gemm_f32mm<true, true, KS><<<grid, nt, 0, s>>>(g);
    GN_LAUNCH_CHECK("gn_gemm (fp32)");
    return GN_OK;
}

}  // namespace

// Time model (us) of the two fp32 kernels, fitted to MI355X sweeps: the six-product split takes
// 0.72 us per 16-k stage on however few blocks and slows from ~340 blocks on; this one runs at
// 58 TFLOP/s, or 1 us per chunk of a wave where its tiles are few.  Measured (split -> here):
// 64 x 256 x 784 (one block of the split) 40.1 -> 9.2, 1000 x 512 x 784 37.7 -> 17.1, 512 x 1536 x 1536
// 73.1 -> 39.3; the split keeps 2048 x 1024 x 1024 (50.4 against 66.8) and 64 x 163840 x 1536 (283
// against 497).  Errors against 64 bits are lower here (64 x 256 x 784 4.3e-7 -> 2.5e-7: shorter
// chains of sums), and an inf operand stays an inf.  Up to K = 256 the split keeps what it takes:
// there it is within a few us (128 x 128 x 256: 16 stages), and its NaNs for infinite operands are
// what callers of those sizes know.
bool gemm_f32mm_wins(const GemmDesc& g) {
    long blocks;
    int stages;
    gemm_f32_grid(g, blocks, stages);
    const double split = 4.0 + 0.72 * stages * std::max(1.0, (double)blocks / 340.0);
    const double K = (double)g.Ks[0] + (g.nseg > 1 ? g.Ks[1] : 0);
    if (K <= 256) return false;
    const double here = 3.0 + std::max(2.0e-6 * g.M * g.N * K / 58.0, K / CK / split_of(g));
    return here < 0.9 * split;
}

// Against the scalar-FMA tiles that took odd sizes before (us): 30 x 50 x 2000 242 -> 15.0,
// 163 x 88 x 1182 150 -> 11.3, 512 x 1535 x 8001 1535 -> 215 (59 TFLOP/s), 2047 x 1023 x 1023 212 -> 71.5; errors
// 2.3 to 2.8 times lower.  What bounds it: the operand loads of each wave (a fragment is used
// for one tile), not the matrix pipe.
int gemm_f32mm_launch(const GemmDesc& g, int transA, int transB, hipStream_t s) {
    if (split_of(g) == 8) return launch_mm<8>(g, transA, transB, s);
    return launch_mm<4>(g, transA, transB, s);
}

}  // namespace gn
