// gn_gemm_wave.hip — bf16 products whose large tiles would leave most of the GPU idle: few
// tokens, or a few hundred over a narrow output.
//
// A block owns a BM x BN tile (32 or 64 each way) of C and splits K over its four waves: wave w
// takes the 64-deep k-tiles w, w + 4, ...  Each wave streams its own k-tiles by LDS DMA through
// a private ring of S stages and multiplies the whole tile, so the main loop has no barrier and
// the block keeps up to 144 KB of reads in flight; the four partial tiles are added in wave
// order through LDS at the end (fp32, deterministic).  What bounds it: the DMA of a few k-tiles and the
// latency ahead of them, the matrix cores being 1-4 % busy (37 x 5632 x 2048, 16 x 768 x 32000).
#include <algorithm>

#include "gn_gemm_dma_core.h"

namespace gn {
namespace {

template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int BM, int BN, int S>
struct WaveTile {
    static constexpr int A_E = BM * BK, STAGE = (BM + BN) * BK * 2, RING = S * STAGE;
    static constexpr int NA = BM / 8, NB = BN / 8, ND = NA + NB;  // DMA instructions of a k-tile
    static constexpr int PITCH = BN + 4;
    static constexpr size_t SMEM = (size_t)4 * RING;
    static_assert(SMEM <= 160 * 1024 && (size_t)BM * (PITCH + 1) * 4 <= RING, "LDS per CU");
    static_assert((S - 1) * ND < 64, "vmcnt range");
};

// BIAS: row sums of op(A) (a weight gradient's db), from an MFMA of A against ones in the blocks
// of the first column tile.
template <bool TA, bool TB, typename CT, int BM, int BN, int EPI, int S>
__global__ __launch_bounds__(256, 1) void gemm_wave(GemmDesc g) {
    using T = WaveTile<BM, BN, S>;
    constexpr int FM = BM / 32, FN = BN / 32;
    constexpr bool BIAS = EPI == 0 && TA && !TB && sizeof(CT) == 4;
    extern __shared__ __align__(16) unsigned char smem_raw[];

    const int tilesM = (g.M + BM - 1) / BM, tilesN = (g.N + BN - 1) / BN;
    const int nblk = tilesM * tilesN;
    // one contiguous range of tiles per XCD (its L2 then holds the ranges' operands), walked
    // eight tile rows at a time
    const int xcd = blockIdx.x & 7, per = nblk >> 3, extra = nblk & 7;
    const int pid = xcd * per + min(xcd, extra) + ((int)blockIdx.x >> 3);
    constexpr int GROUP = 8;
    const int group_id = pid / (GROUP * tilesN);
    const int first_m = group_id * GROUP;
    const int gsize = min(tilesM - first_m, GROUP);
    const int in_group = pid % (GROUP * tilesN);
    const int m0 = (first_m + in_group % gsize) * BM, n0 = (in_group / gsize) * BN;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    unsigned char* ring = smem_raw + wave * T::RING;
    const uint32_t ring_a = lds_addr(ring);

    const int kt0 = (g.Ks[0] + BK - 1) / BK;
    const int KT = kt0 + (g.nseg > 1 ? (g.Ks[1] + BK - 1) / BK : 0);
    const int nt = (KT - wave + 3) >> 2;  // this wave's k-tiles: wave + 4 i, i < nt

    uint32_t voa[T::NA], vob[T::NB];
    int oseg = -1;
    auto dma = [&](int i) {
        const int t = wave + 4 * i;
        const int sg = t >= kt0 ? 1 : 0;
        const int k0 = (sg ? t - kt0 : t) * BK, klim = g.Ks[sg];
        const bf16_t* A = g.A[sg];
        const bf16_t* B = g.B[sg];
        const int lda = g.lda[sg], ldb = g.ldb[sg];
        const uint32_t base = ring_a + (uint32_t)(i % S) * T::STAGE;
        if (k0 + BK > klim) {
            stage_tail<BM, !TA, 1>(A, lda, m0, g.M, k0, klim, 0, base);
            stage_tail<BN, TB, 1>(B, ldb, n0, g.N, k0, klim, 0, base + T::A_E * 2);
            return;
        }
        if (oseg != sg) {
            oseg = sg;
            stage_offsets<BM, !TA, 1>(lda, m0, g.M, 0, voa);
            stage_offsets<BN, TB, 1>(ldb, n0, g.N, 0, vob);
        }
        const bf16_t* sa = stage_base<!TA>(A, lda, m0, k0);
        const bf16_t* sb = stage_base<TB>(B, ldb, n0, k0);
#pragma unroll
        for (int q = 0; q < T::NA; ++q) dma16s(sa, voa[q], base + 1024u * q);
#pragma unroll
        for (int q = 0; q < T::NB; ++q) dma16s(sb, vob[q], base + T::A_E * 2 + 1024u * q);
    };

    f32x16_t acc[FM][FN], rows[BIAS ? FM : 1];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) zero16(acc[i][j]);
#pragma unroll
    for (int i = 0; i < (BIAS ? FM : 1); ++i) zero16(rows[i]);
    const bool sums = BIAS && g.bias && n0 == 0;

    for (int i = 0; i < min(S, nt); ++i) dma(i);
    for (int i = 0; i < nt; ++i) {
        // tile i has landed; the younger tiles of the ring may still be in flight
        const int younger = min(nt - 1 - i, S - 1);
        if (younger >= 3 && S > 3) wait_vm<(S > 3 ? 3 : 0) * T::ND>();
        else if (younger == 2 && S > 2) wait_vm<(S > 2 ? 2 : 0) * T::ND>();
        else if (younger == 1) wait_vm<T::ND>();
        else wait_vm<0>();
        const bf16_t* sa = reinterpret_cast<const bf16_t*>(ring + (i % S) * T::STAGE);
        const bf16_t* sb = sa + T::A_E;
        bf16x8_t fa[4][FM], fb[4][FN];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int a = 0; a < FM; ++a) fa[ks][a] = frag<BM, !TA>(sa, a * 32, ks);
#pragma unroll
            for (int b = 0; b < FN; ++b) fb[ks][b] = frag<BN, TB>(sb, b * 32, ks);
        }
        // every read of the stage has returned before its refill is issued
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (i + S < nt) dma(i + S);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) acc[a][b] = mfma32(fa[ks][a], fb[ks][b], acc[a][b]);
        if constexpr (BIAS) {
            if (sums) {
                bf16x8_t one;
#pragma unroll
                for (int e = 0; e < 8; ++e) one[e] = (__bf16)1.0f;
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                    for (int a = 0; a < FM; ++a) rows[a] = mfma32(fa[ks][a], one, rows[a]);
            }
        }
    }

    // partial tiles into the waves' own rings (every DMA has landed), then summed by the block
    float* st = reinterpret_cast<float*>(ring);
    const int rq = (lane >> 5) * 4;
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                st[(a * 32 + 8 * (r >> 2) + rq + (r & 3)) * T::PITCH + b * 32 + (lane & 31)] = acc[a][b][r];
    if constexpr (BIAS) {
        if (sums && (lane & 31) == 0) {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    st[BM * T::PITCH + a * 32 + 8 * (r >> 2) + rq + (r & 3)] = rows[a][r];
        }
    }
    __syncthreads();
    const float* p0 = reinterpret_cast<const float*>(smem_raw);
    constexpr int CPR = BN / 8, WS = T::RING / 4;
#pragma unroll
    for (int c = threadIdx.x; c < BM * CPR; c += 256) {
        const int r = c / CPR, col = (c % CPR) * 8;
        const int m = m0 + r, n = n0 + col;
        const float* p = p0 + r * T::PITCH + col;
        float v[8];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float4 lo = *reinterpret_cast<const float4*>(p + w * WS);
            const float4 hi = *reinterpret_cast<const float4*>(p + w * WS + 4);
            const float u[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = w == 0 ? u[e] : v[e] + u[e];
        }
        if (m < g.M && n < g.N) store8<CT, EPI>(g, m, n, v);
    }
    if constexpr (BIAS) {
        const int m = m0 + threadIdx.x;
        if (sums && threadIdx.x < BM && m < g.M) {
            const float* p = p0 + BM * T::PITCH + threadIdx.x;
            const float v = ((p[0] + p[WS]) + p[2 * WS]) + p[3 * WS];
            float* dst = m < g.Msplit ? g.bias + m : g.bias2 + (m - g.Msplit);
            *dst = g.accumulate ? *dst + v : v;
        }
    }
}

template <bool TA, bool TB, typename CT, int BM, int BN, int EPI, int S>
int launch_wave(const GemmDesc& g, hipStream_t s) {
    using T = WaveTile<BM, BN, S>;
    static const bool ok = allow_lds(gemm_wave<TA, TB, CT, BM, BN, EPI, S>, T::SMEM);
    if (!ok) {
        set_error("gemm: cannot reserve %zu B of LDS", T::SMEM);
        return GN_E_HIP;
    }
    const int tiles = ((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    hipLaunchKernelGGL((gemm_wave<TA, TB, CT, BM, BN, EPI, S>), dim3(tiles), dim3(256), T::SMEM, s, g);
    GN_LAUNCH_CHECK("gemm (wave-split)");
    return GN_OK;
}

template <bool TA, bool TB, typename CT, int EPI>
int launch_tile(const GemmDesc& g, int shape, hipStream_t s) {
    switch (shape) {
        case 0: return launch_wave<TA, TB, CT, 64, 64, EPI, 2>(g, s);
        case 1: return launch_wave<TA, TB, CT, 64, 32, EPI, 3>(g, s);
        case 2: return launch_wave<TA, TB, CT, 32, 64, EPI, 3>(g, s);
        default: return launch_wave<TA, TB, CT, 32, 32, EPI, 4>(g, s);
    }
}

template <typename CT>
int launch_plain(const GemmDesc& g, int ta, int tb, int shape, hipStream_t s) {
    if (!ta && !tb) return launch_tile<false, false, CT, 0>(g, shape, s);
    if (!ta && tb) return launch_tile<false, true, CT, 0>(g, shape, s);
    if (ta && !tb) return launch_tile<true, false, CT, 0>(g, shape, s);
    return launch_tile<true, true, CT, 0>(g, shape, s);
}

}  // namespace

// The tile that runs g fastest here, or -1 where the large tiles do.  Time model, fitted to
// MI355X sweeps of both over M from 1 to 4096 on the FFN and decoder products: a round of
// blocks (one per CU) takes a fixed time and one step per four k-tiles; the steps are bound by
// the LDS DMA (64 x 64: 64 KB in 0.7 us = 92 GB/s per CU), so a small tile pays where
// the large ones leave CUs idle: they move half the bytes per FLOP but take 0.3-0.55 us per k-tile
// on however few CUs.  The other side is the kernel that would run instead: bf16 C the streamed
// tiles (gemm_stream_us), fp32 C and the GLU epilogue the core's.
// Measured (us, replayed; streamed tiles -> here): 64 x 5632 x 2048 13.2 -> 7.8, 64 x 2048 x 5632
// 28.9 -> 10.3, 384 x 2048 x 5632 33.4 -> 20.0, 1003 x 768 x 6144 40.9 -> 24.6, an LM head's dX 16 x 768 x
// 32000 142 -> 61, 1003 rows 175 -> 98; the streamed tiles lead at 200 x 5632 x 2048 (13.7 against 17.1),
// 768 x 2048 x 5632 (34.4 / 36.5), 1536 x 768 x 6144 (38.5 / 39.3) and 2001 x 768 x 32000 (level alone, 279
// against 342 beside its weight gradient).  fp32 C, core -> here: dW 768 x 768 over 512 rows 8.6 -> 5.8,
// over 4096 23.7 -> 17.6.  Of 240 bf16 products in that sweep the lines drawn (0.95 of the streamed
// time, 0.85 of the core's) give each the faster kernel.
int gemm_wave_shape(const GemmDesc& g, int transA, int transB, int c_dtype) {
    const bool ta = transA != 0;
    const size_t c_bytes = g.epi == 1 || c_dtype != GN_F32 ? 2 : 4;
    double best;
    if (g.epi == 0 && c_bytes == 2) {
        best = 0.95 * gemm_stream_us(g);
    } else {
        const TileChoice tc = choose_tile(g, ta, c_bytes, g.epi);
        if (tc.m_first > 0) return -1;
        best = 0.85 * tile_cost(g, ta, c_bytes, g.epi, tc.shape, tc.ksplit, tc.ksplit > 2);
    }
    static constexpr int bm[4] = {64, 64, 32, 32}, bn[4] = {64, 32, 64, 32};
    static constexpr double fixed[4] = {3.2, 1.8, 1.8, 1.6}, step[4] = {0.70, 0.52, 0.52, 0.34};
    const int steps = (k_tiles(g) + 3) / 4;
    int shape = -1;
    for (int i = 0; i < 4; ++i) {
        const long blocks = (long)((g.M + bm[i] - 1) / bm[i]) * ((g.N + bn[i] - 1) / bn[i]);
        const double f = (double)(blocks % 256) / 256.0;
        const double rounds = (double)(blocks / 256) + (f > 0 ? 0.6 + 0.4 * f : 0.0);
        // transposed operands read their fragments in two halves, fp32 tiles store twice the bytes
        const double t = rounds * (fixed[i] * (c_bytes == 4 ? 1.4 : 1.0) + steps * step[i] * (ta ? 1.4 : 1.0));
        if (t < best) { best = t; shape = i; }
    }
    return shape;
}

int gemm_wave_launch(const GemmDesc& g, int shape, int transA, int transB, int c_dtype, hipStream_t s) {
    if (g.epi == 1) return launch_tile<false, false, bf16_t, 1>(g, shape, s);
    if (c_dtype == GN_F32) return launch_plain<float>(g, transA, transB, shape, s);
    return launch_plain<bf16_t>(g, transA, transB, shape, s);
}

}  // namespace gn
