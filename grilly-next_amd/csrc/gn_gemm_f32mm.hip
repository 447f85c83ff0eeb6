// gn_gemm_f32mm.hip — fp32 products on small tiles, any size and alignment.
//
// Two kernels without LDS staging or barriers: a wave owns one tile and reads its operands
// straight into the matrix instruction's registers, the next k while the current ones are
// multiplied.
//   gemm_f32seq  sizes that are not multiples of 4 and unaligned operands: v_mfma_f32_32x32x2_f32 or
//                16x16x4, whose k steps are fp32 multiply-adds in order of k (an inf stays an inf)
//   gemm_f32x6t  the six-product bf16 split of gn_gemm_f32.hip on 32 x 32 tiles, for products whose
//                128 x 128 and 64 x 256 tiles would be a few blocks
// An output's products are added in increasing k by one accumulator in both, so gemm_f32seq
// gives the bits of a scalar multiply-add loop and gemm_f32x6t those of gemm_f32x6.  Both are bound by
// their loads' latency and the split: gemm_f32x6t keeps the matrix cores 6 % busy at 512 x 768 x 1024.
#include <algorithm>

#include "gn_common.h"
#include "gn_gemm_dma.h"
#include "gn_mfma.h"

namespace gn {
namespace {

__device__ __forceinline__ void swap32(float& a, float& b) {  // {a.hi, b.lo} exchanged
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {  // odd 16-lane rows of a, even ones of b
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// block -> tile: one contiguous range of tiles per XCD, walked eight tile rows at a time
__device__ __forceinline__ void tile_of(int pid0, int tilesM, int tilesN, int& tm, int& tn) {
    const int nblk = tilesM * tilesN;
    const int xcd = pid0 & 7, per = nblk >> 3, extra = nblk & 7;
    const int pid = xcd * per + min(xcd, extra) + (pid0 >> 3);
    const int first_m = (pid / (8 * tilesN)) * 8;
    const int gsize = min(tilesM - first_m, 8), in_group = pid % (8 * tilesN);
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// 16 k of one operand row from k0 (k past klim reads as zero, from a clamped address; rows are
// clamped by the caller) as the values of the 16x16x4 (T = 16: four steps, lane group g = lane / 16
// holds k 4j + g of step j) or 32x32x2 instruction (T = 32: eight steps, half h holds k 2j + h).
template <int T, bool KC>
__device__ __forceinline__ void load_seq(const float* __restrict__ P, int ld, int row, int k0, int klim,
                                         float (&v)[T / 4]) {
    constexpr int N = T / 4, S = 64 / T;  // steps; k per step
    const int lane = threadIdx.x & 63, g = lane / T;
    if (KC && k0 + 16 <= klim) {
        const float* p = P + (size_t)row * ld + k0;
        if constexpr (T == 16) {  // group g loads k 4g .. 4g+3, then a 4 x 4 transpose over the groups
            float4 q;
            __builtin_memcpy(&q, p + 4 * g, 16);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) {  // half h loads k 8c + 4h .. +3
                float4 q;
                __builtin_memcpy(&q, p + 8 * c + 4 * g, 16);
                v[4 * c] = q.x; v[4 * c + 1] = q.y; v[4 * c + 2] = q.z; v[4 * c + 3] = q.w;
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
        // the order load_seq's fast path leaves (arrange() brings both to step order)
        const int k = k0 + (KC ? (T == 16 ? 4 * g + j : 8 * (j / 4) + 4 * g + j % 4) : S * j + g);
        const int kc = min(k, klim - 1);
        const float y = P[KC ? (size_t)row * ld + kc : (size_t)kc * ld + row];
        v[j] = k < klim ? y : 0.f;
    }
}
template <int T, bool KC>
__device__ __forceinline__ void arrange(float (&v)[T / 4]) {
    if constexpr (!KC) return;
    if constexpr (T == 16) {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
        swap16(v[0], v[1]);
        swap16(v[2], v[3]);
    } else {
#pragma unroll
        for (int c = 0; c < 8; c += 4) {  // {0|4}{1|5}{2|6}{3|7} -> {0|1}{2|3}{4|5}{6|7}
            swap32(v[c], v[c + 1]);
            swap32(v[c + 2], v[c + 3]);
            const float t = v[c + 1];
            v[c + 1] = v[c + 2];
            v[c + 2] = t;
        }
    }
}

// Block: 2 x 2 waves of T x T tiles.  FB: with the column bias of a forward Linear.
// At most four waves per SIMD: given the registers, the compiler keeps the loads of four chunks in
// flight; for eight waves it does not (512 x 10 x 256 backward 14.3 -> 17.5 us).
template <bool TA, bool TB, bool FB, int T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) void gemm_f32seq(GemmDesc g) {
    constexpr int N = T / 4;
    const int tilesM = (g.M + 2 * T - 1) / (2 * T), tilesN = (g.N + 2 * T - 1) / (2 * T);
    int tm, tn;
    tile_of(blockIdx.x, tilesM, tilesN, tm, tn);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = (2 * tm + (wave >> 1)) * T, n0 = (2 * tn + (wave & 1)) * T;
    if (m0 >= g.M || n0 >= g.N) return;
    const int row = min(m0 + lane % T, g.M - 1), col = min(n0 + lane % T, g.N - 1);
    const int c0 = (g.Ks[0] + 15) / 16, nc = c0 + (g.nseg > 1 ? (g.Ks[1] + 15) / 16 : 0);
    auto load = [&](int c, float (&a)[N], float (&b)[N]) {
        const int s = c >= c0 ? 1 : 0, k0 = (s ? c - c0 : c) * 16;
        load_seq<T, !TA>(reinterpret_cast<const float*>(g.A[s]), g.lda[s], row, k0, g.Ks[s], a);
        load_seq<T, TB>(reinterpret_cast<const float*>(g.B[s]), g.ldb[s], col, k0, g.Ks[s], b);
    };
    constexpr int R = T == 16 ? 4 : 16;
    typedef float acc_t __attribute__((ext_vector_type(R)));
    acc_t acc;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    // chunks of 16 k, D in flight
    constexpr int D = 4;
    float a[D][N], b[D][N];
#pragma unroll
    for (int d = 0; d < D; ++d) load(min(d, nc - 1), a[d], b[d]);
    for (int c = 0; c < nc; c += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (c + d < nc) {
                arrange<T, !TA>(a[d]);
                arrange<T, TB>(b[d]);
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    if constexpr (T == 16) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[d][j], b[d][j], acc, 0, 0, 0);
                    else acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[d][j], b[d][j], acc, 0, 0, 0);
                }
            }
            load(min(c + d + D, nc - 1), a[d], b[d]);
        }
    }
    const int n = n0 + lane % T;
    if (n >= g.N) return;
    if constexpr (FB) {
        const float b = g.fbias[n];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] += b;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int m = m0 + (T == 16 ? 4 * (lane >> 4) + r : 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3));
        if (m < g.M) gemm_store<float, 0>(g, m, n, acc[r]);
    }
}

template <int T>
int launch_seq(const GemmDesc& g, int ta, int tb, hipStream_t s) {
    const unsigned grid = (unsigned)(((g.M + 2 * T - 1) / (2 * T)) * (long)((g.N + 2 * T - 1) / (2 * T)));
    if (g.fbias) gemm_f32seq<false, true, true, T><<<grid, 256, 0, s>>>(g);
    else if (!ta && !tb) gemm_f32seq<false, false, false, T><<<grid, 256, 0, s>>>(g);
    else if (!ta && tb) gemm_f32seq<false, true, false, T><<<grid, 256, 0, s>>>(g);
    else if (ta && !tb) gemm_f32seq<true, false, false, T><<<grid, 256, 0, s>>>(g);
    else gemm_f32seq<true, true, false, T><<<grid, 256, 0, s>>>(g);
    GN_LAUNCH_CHECK("gn_gemm (fp32)");
    return GN_OK;
}

// k 8h .. 8h+7 of one operand row's 16-k stage (h = lane / 32); klim a multiple of 4
template <bool KC>
__device__ __forceinline__ void load8(const float* __restrict__ P, int ld, int row, int k0, int klim,
                                      float4 (&v)[2]) {
    const int kb = k0 + 8 * ((threadIdx.x & 63) >> 5);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int k = kb + 4 * i, kc = min(k, klim - 4);
        if (KC) {
            v[i] = *reinterpret_cast<const float4*>(P + (size_t)row * ld + kc);
        } else {
            const float* p = P + (size_t)kc * ld + row;
            v[i] = make_float4(p[0], p[ld], p[2 * (size_t)ld], p[3 * (size_t)ld]);
        }
    }
}
// split (zeros from klim on)
__device__ __forceinline__ void pieces(const float4 (&v)[2], int k0, int klim, bf16x8_t (&o)[3]) {
    const int kb = k0 + 8 * ((threadIdx.x & 63) >> 5);
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const bool in = kb + 4 * i < klim;
        const float x = in ? v[i].x : 0.f, y = in ? v[i].y : 0.f, z = in ? v[i].z : 0.f, t = in ? v[i].w : 0.f;
        split2(x, y, w[0][2 * i], w[1][2 * i], w[2][2 * i]);
        split2(z, t, w[0][2 * i + 1], w[1][2 * i + 1], w[2][2 * i + 1]);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) o[p] = __builtin_bit_cast(bf16x8_t, make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]));
}

// One wave, one 32 x 32 tile per block; stages of 16 k.
template <bool TA, bool TB, bool FB>
__global__ __launch_bounds__(64) void gemm_f32x6t(GemmDesc g) {
    const int tilesM = (g.M + 31) / 32, tilesN = (g.N + 31) / 32;
    int tm, tn;
    tile_of(blockIdx.x, tilesM, tilesN, tm, tn);
    const int lane = threadIdx.x;
    const int m0 = tm * 32, n0 = tn * 32;
    const int row = min(m0 + (lane & 31), g.M - 1), col = min(n0 + (lane & 31), g.N - 1);
    const int c0 = (g.Ks[0] + 15) / 16, nc = c0 + (g.nseg > 1 ? (g.Ks[1] + 15) / 16 : 0);
    auto load = [&](int c, float4 (&a)[2], float4 (&b)[2]) {
        const int s = c >= c0 ? 1 : 0, k0 = (s ? c - c0 : c) * 16;
        load8<!TA>(reinterpret_cast<const float*>(g.A[s]), g.lda[s], row, k0, g.Ks[s], a);
        load8<TB>(reinterpret_cast<const float*>(g.B[s]), g.ldb[s], col, k0, g.Ks[s], b);
    };
    f32x16_t acc;
    zero16(acc);
    constexpr int D = 4;
    float4 a[D][2], b[D][2];
#pragma unroll
    for (int d = 0; d < D; ++d) load(min(d, nc - 1), a[d], b[d]);
    for (int c = 0; c < nc; c += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (c + d < nc) {
                const int s = c + d >= c0 ? 1 : 0, k0 = (s ? c + d - c0 : c + d) * 16;
                bf16x8_t pa[3], pb[3];
                pieces(a[d], k0, g.Ks[s], pa);
                pieces(b[d], k0, g.Ks[s], pb);
                // smallest terms first, gemm_f32x6's order
                acc = mfma32(pa[2], pb[0], acc);
                acc = mfma32(pa[1], pb[1], acc);
                acc = mfma32(pa[0], pb[2], acc);
                acc = mfma32(pa[1], pb[0], acc);
                acc = mfma32(pa[0], pb[1], acc);
                acc = mfma32(pa[0], pb[0], acc);
            }
            load(min(c + d + D, nc - 1), a[d], b[d]);
        }
    }
    gemm_store_tile<float, 0, FB>(g, m0, n0, acc);
}

}  // namespace

// Time model (us) fitted to MI355X sweeps (251 products, K from 4 to 3072): gemm_f32x6 takes 0.63 us per
// 16-k stage on however few blocks and slows from ~220 blocks on, a 32 x 32 tile 0.44 us per stage up to
// ~900 tiles, and a tile's launch and store 1.4 ns (a short K of many tiles is gemm_f32x6's:
// 1536 x 1536 x 16 6.4 against 8.1, 3072 x 3072 x 16 10.6 against 17.5).
// Measured (gemm_f32x6 -> here): 64 x 256 x 784 (one block) 40 -> 20, 1000 x 512 x 784 37.6 -> 21.7,
// 512 x 1536 x 1536 73 -> 41, 200 x 4000 x 1000 46 -> 28; gemm_f32x6 keeps 2048 x 1024 x 1024 (50 against 63) and
// 64 x 163840 x 1536 (285 against 545).  Split-K products stay with gemm_f32x6 too (their planes
// add in another order, and fill the GPU).
bool gemm_f32x6t_wins(const GemmDesc& g) {
    long blocks;
    int stages, ks;
    gemm_f32_grid(g, blocks, stages, ks);
    if (ks > 1) return false;
    const double tiles = (double)((g.M + 31) / 32) * ((g.N + 31) / 32);
    const double x6 = 5.0 + 0.009 * (double)blocks + 0.63 * stages * std::max(1.0, (double)blocks / 220.0);
    return 4.2 + 0.0014 * tiles + 0.44 * stages * std::max(1.0, tiles / 900.0) < x6;
}

int gemm_f32x6t_launch(const GemmDesc& g, int transA, int transB, hipStream_t s) {
    const unsigned grid = (unsigned)(((g.M + 31) / 32) * (long)((g.N + 31) / 32));
    if (g.fbias) gemm_f32x6t<false, true, true><<<grid, 64, 0, s>>>(g);
    else if (!transA && !transB) gemm_f32x6t<false, false, false><<<grid, 64, 0, s>>>(g);
    else if (!transA && transB) gemm_f32x6t<false, true, false><<<grid, 64, 0, s>>>(g);
    else if (transA && !transB) gemm_f32x6t<true, false, false><<<grid, 64, 0, s>>>(g);
    else gemm_f32x6t<true, true, false><<<grid, 64, 0, s>>>(g);
    GN_LAUNCH_CHECK("gn_gemm (fp32 bf16x6, small tiles)");
    return GN_OK;
}

// 32 x 32 tiles where there are enough of them (512 x 1535 x 1535, 768 tiles: 72 -> 58 us against 16 x 16),
// else 16 x 16 (1182 x 163 x 88: 9.3 against 17.8).  Against the scalar-FMA tiles these sizes took before
// (us): 64 x 10 x 256 33.5 -> 7.8, 30 x 50 x 2000 241 -> 32, 163 x 88 x 1182 149 -> 17.6,
// 512 x 1535 x 8001 1604 -> 243, 2047 x 1023 x 1023 212 -> 70.  Bound by the operand loads (each fragment is
// used for one tile) and, on few tiles, by the chain of K / 4 dependent matrix instructions.
int gemm_f32seq_launch(const GemmDesc& g, int transA, int transB, hipStream_t s) {
    const long tiles = (long)((g.M + 31) / 32) * ((g.N + 31) / 32);
    return tiles >= 512 ? launch_seq<32>(g, transA, transB, s) : launch_seq<16>(g, transA, transB, s);
}

}  // namespace gn
