// gn_gemm_stream.hip — bf16-output products (every operand orientation) and the fp32 weight gradients
// of several rounds on blocks that stay: one per CU, each walking its share of the tiles with the
// k-tiles of all of them as one stream.
//
// A block per tile (gn_gemm_dma_core.h) spends ~11 us on its DMA prologue, pipeline fill and
// fp32-staged epilogue around the 10 us that 12 k-tiles of a 256 x 128 tile need.  Here the four
// producer waves run on into the next tile's k-tiles while the four compute waves store the
// finished one, and the store goes out through 4 KB of LDS per wave, so that a tile costs
// its k-tiles and ~3 us.  What bounds it: at 12 k-tiles the store bursts and the k-tiles about
// equally, from ~32 k-tiles on the matrix cores (63-68 % busy over 4096 x 2048 x 11264 and dW 11264 x
// 2048 x 4096) and the LDS reads that feed them.
//   us, a block per tile -> here (A k-contiguous, B row-major [N][K]; in brackets B [K][N]):
//   8192 x 32000 x 768  689 -> 447 (668 -> 464)    8192 x 3072 x 768   63 -> 42
//   2001 x 32000 x 768  152 -> 99                  8192 x  768 x 768   19 -> 15 (16 -> 14)
//   4096 x 5632 x 2048  112 -> 89  (100 -> 87)     8192 x  768 x 6144  78 -> 68 (67 -> 66)
//   8192 x 8192 x 4096  515 -> 454                 4096 x  768 x 768   10 -> 9.5
// The main loop, the order of every output's sum and its roundings are those of the core: the
// results are the same bits.
#include <algorithm>

#include "gn_gemm_dma_core.h"

namespace gn {
namespace {

// A product's operands as a producer wave keeps them: read from the kernel's arguments in one go at
// its start and held in scalar registers from then on (the empty asm keeps the compiler from
// loading them again where they are used).  Arguments read where they are needed were scalar loads
// one after the other ahead of the first DMA and, indexed by segment, between every barrier and its
// DMA, which a grid of few blocks waits for on every k-tile.  Measured (us): 64 x 768 x 3072 on 6
// streamed tiles 21.1 -> 18.2, 4096 x 768 x 3072 26.1 -> 23.9.
struct Operands {
    const bf16_t *A0, *B0, *A1, *B1;
    int lda0, ldb0, lda1, ldb1, K0, K1, M, N, nseg;
    __device__ __forceinline__ explicit Operands(const GemmDesc& g)
        : A0(g.A[0]), B0(g.B[0]), A1(g.A[1]), B1(g.B[1]), lda0(g.lda[0]), ldb0(g.ldb[0]),
          lda1(g.lda[1]), ldb1(g.ldb[1]), K0(g.Ks[0]), K1(g.Ks[1]), M(g.M), N(g.N), nseg(g.nseg) {
        asm volatile("" : "+s"(A0), "+s"(B0), "+s"(A1), "+s"(B1), "+s"(lda0), "+s"(ldb0), "+s"(lda1),
                     "+s"(ldb1), "+s"(K0), "+s"(K1), "+s"(M), "+s"(N), "+s"(nseg));
    }
};

// A producer wave's walk over the k-tiles of one output tile after another.
template <bool TA, bool TB, int BM, int BN, int NW>
struct KFeed {
    static constexpr int NDA = BM / (8 * NW), NDB = BN / (8 * NW);  // DMA instructions of a k-tile
    const Operands o;
    const int dw;  // the wave's share of a tile's DMA
    uint32_t voa[NDA], vob[NDB];
    const bf16_t *sa, *sb;  // the k-tile's origin in each operand
    int64_t da, db;         // from one k-tile to the next
    int m0, n0, left;       // left: k from here to the segment's end
    bool second;            // the segment

    __device__ __forceinline__ KFeed(const GemmDesc& g, int wave) : o(g), dw(wave) {}
    // to k = k0 of a segment
    __device__ __forceinline__ void segment(bool s1, int k0) {
        second = s1;
        const int lda = s1 ? o.lda1 : o.lda0, ldb = s1 ? o.ldb1 : o.ldb0;
        left = (s1 ? o.K1 : o.K0) - k0;
        stage_offsets<BM, !TA, NW>(lda, m0, o.M, dw, voa);
        stage_offsets<BN, TB, NW>(ldb, n0, o.N, dw, vob);
        sa = stage_base<!TA>(s1 ? o.A1 : o.A0, lda, m0, k0);
        sb = stage_base<TB>(s1 ? o.B1 : o.B0, ldb, n0, k0);
        da = TA ? (int64_t)BK * lda : BK;
        db = TB ? BK : (int64_t)BK * ldb;
    }
    // to k-tile t (over both segments) of output tile (m, n)
    __device__ __forceinline__ void start(int m, int n, int t) {
        m0 = m;
        n0 = n;
        const int kt0 = (o.K0 + BK - 1) / BK;
        segment(t >= kt0, (t < kt0 ? t : t - kt0) * BK);
    }
    // The k-tile's DMA; one that its segment's end cuts short (a ragged token count is the K of every
    // weight gradient) is filled up with zeros.
    __device__ __forceinline__ void issue(uint32_t base) {
        constexpr uint32_t B_OFF = BM * BK * 2;
        if (left >= BK) {
#pragma unroll
            for (int q = 0; q < NDA; ++q) dma16s(sa, voa[q], base + 1024u * (uint32_t)(dw * NDA + q));
#pragma unroll
            for (int q = 0; q < NDB; ++q) dma16s(sb, vob[q], base + B_OFF + 1024u * (uint32_t)(dw * NDB + q));
        } else {
            const int klim = second ? o.K1 : o.K0, k0 = klim - left;
            stage_tail<BM, !TA, NW>(second ? o.A1 : o.A0, second ? o.lda1 : o.lda0, m0, o.M, k0, klim, dw, base);
            stage_tail<BN, TB, NW>(second ? o.B1 : o.B0, second ? o.ldb1 : o.ldb0, n0, o.N, k0, klim, dw,
                                   base + B_OFF);
        }
    }
    // On to the next k-tile; false (and no move) after the product's last.
    __device__ __forceinline__ bool step() {
        if (left > BK) {
            left -= BK;
            sa += da;
            sb += db;
            return true;
        }
        if (second || o.nseg < 2) return false;
        segment(true, 0);
        return true;
    }
};

template <bool TA, bool TB, typename CT, int BM, int BN, int STAGES>
__global__ __launch_bounds__(512, 1) void gemm_stream(GemmDesc g) {
    constexpr int NW = 4;
    constexpr int A_ELEMS = BM * BK, B_ELEMS = BN * BK, STAGE_B = (A_ELEMS + B_ELEMS) * 2;
    constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 32, FN = WN / 32, NM = FM * FN;
    constexpr int RA = TA ? 2 : 1, RB = TB ? 1 : 2, NR = FM * RA + FN * RB;
    constexpr int ND = (BM + BN) / (8 * NW);  // DMA instructions of a wave per k-tile
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const uint32_t lds0 = lds_addr(smem_raw);

    const int tilesM = (g.M + BM - 1) / BM, tilesN = (g.N + BN - 1) / BN;
    const int nblk = tilesM * tilesN;
    const int ntile = (nblk - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;  // this block's
    // its i-th tile: block b runs on XCD b % 8, each XCD walks one contiguous range of the tiles,
    // GROUP tile rows at a time (gridDim.x is a multiple of 8, or a block has one tile)
    auto tile_at = [&](int i, int& m0, int& n0) __attribute__((always_inline)) {
        const int x = (int)blockIdx.x + i * (int)gridDim.x;
        const int xcd = x & 7, per = nblk >> 3, extra = nblk & 7;
        const int pid = xcd * per + min(xcd, extra) + (x >> 3);
        constexpr int GROUP = BM == 256 ? 4 : 8;
        const int first_m = (pid / (GROUP * tilesN)) * GROUP;
        const int gsize = min(tilesM - first_m, GROUP);
        const int in_group = pid % (GROUP * tilesN);
        m0 = (first_m + in_group % gsize) * BM;
        n0 = (in_group / gsize) * BN;
    };

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave >> 1) & 1, wn = wave & 1, dw = wave & 3;
    const int KT = (g.Ks[0] + BK - 1) / BK + (g.nseg > 1 ? (g.Ks[1] + BK - 1) / BK : 0);
    const int J = ntile * KT;  // k-tiles of the stream

    if (wave >= 4) {
        // producers: the compute waves' barriers, the DMA of k-tile j + STAGES after each
        KFeed<TA, TB, BM, BN, NW> feed(g, dw);
        int pi = 0, m0, n0;
        tile_at(0, m0, n0);
        feed.start(m0, n0, 0);
        auto next = [&](int slot) __attribute__((always_inline)) {
            feed.issue(lds0 + (uint32_t)(slot * STAGE_B));
            if (!feed.step() && pi + 1 < ntile) {  // past the end: the last k-tile again
                tile_at(++pi, m0, n0);
                feed.start(m0, n0, 0);
            }
        };
        static_for<STAGES>([&](auto S_) { next(decltype(S_)::value); });
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 1) * ND));
        __syncthreads();
        int slot = 0;
        for (int j = 0; j < J; ++j) {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * ND));  // k-tile j + 1 has landed
            __syncthreads();
            next(slot);
            slot = slot == STAGES - 1 ? 0 : slot + 1;
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        return;
    }

    f32x16_t acc[FM][FN];
    bf16x8_t fa[4][FM], fb[4][FN];
    auto read_one = [&](auto SET_, auto R_, const bf16_t* sa, int ks) {
        constexpr int set = decltype(SET_)::value, r = decltype(R_)::value;
        if constexpr (r < FM * RA) {
            if constexpr (r % RA == 0) fa[set][r / RA] = frag<BM, !TA>(sa, wm * WM + (r / RA) * 32, ks);
        } else {
            constexpr int rb = r - FM * RA;
            if constexpr (rb % RB == 0) fb[set][rb / RB] = frag<BN, TB>(sa + A_ELEMS, wn * WN + (rb / RB) * 32, ks);
        }
    };
    auto kstep = [&](auto CUR_, auto RSET_, auto FRONT_, const bf16_t* rsrc, int rks) {
        constexpr int cur = decltype(CUR_)::value;
        constexpr bool front = decltype(FRONT_)::value;
        static_for<NM>([&](auto Q_) {
            constexpr int q = decltype(Q_)::value;
            acc[q / FN][q % FN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[cur][q % FN], fa[cur][q / FN],
                                                                          acc[q / FN][q % FN], 0, 0, 0);
            constexpr int r0 = reads_before<NM, NR, front>(q), r1 = reads_before<NM, NR, front>(q + 1);
            static_for<NR>([&](auto R_) {
                constexpr int r = decltype(R_)::value;
                if constexpr (r >= r0 && r < r1) read_one(RSET_, R_, rsrc, rks);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using BF = std::false_type;
    using BT = std::true_type;
    auto stage_ptr = [&](int slot) { return reinterpret_cast<const bf16_t*>(smem_raw + slot * STAGE_B); };

    // Store one finished tile.  The products are transposed (op(B)'s fragment first): element r of
    // a 32 x 32 block is row lane % 32, column 8 (r / 4) + 4 (lane / 32) + r % 4, so four
    // consecutive elements are four columns of one row.  32 rows at a time go through the wave's
    // own LDS as bf16 (16-byte chunk c of row m at c ^ (m % 8)) and leave as 128-byte row segments.
    bf16_t* const C = reinterpret_cast<bf16_t*>(g.C);
    unsigned char* const st = smem_raw + STAGES * STAGE_B + wave * 4096;
    auto store = [&](auto MIX_, int m0, int n0) {
        constexpr bool MIX = decltype(MIX_)::value;  // + cbias, + C
        int ln = lane;  // opaque: its addresses are formed here, not kept across the k loop
        asm volatile("" : "+v"(ln));
        const int mr = ln & 31, nh = 4 * (ln >> 5);
        const int nw = n0 + wn * WN;
        const bool nok = nw + (ln & 7) * 8 < g.N;
        const uint32_t voff = (uint32_t)((ln >> 3) * g.ldc + (ln & 7) * 8) * 2u;
        static_for<FM>([&](auto I_) {
            constexpr int i = decltype(I_)::value;
            const int mw = m0 + wm * WM + i * 32;
            bf16_t* const Cw = C + (size_t)mw * g.ldc + nw;
            wave_lds_sync();
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[4];
#pragma unroll
                    for (int d = 0; d < 4; ++d) v[d] = acc[i][j][4 * q + d];
                    if constexpr (MIX) {
                        const int nc = j * 32 + q * 8 + nh;
                        if (g.cbias && nw + nc < g.N) {
                            const uint2 b = *reinterpret_cast<const uint2*>(g.cbias + nw + nc);
                            v[0] += __uint_as_float(b.x << 16);
                            v[1] += __uint_as_float(b.x & 0xffff0000u);
                            v[2] += __uint_as_float(b.y << 16);
                            v[3] += __uint_as_float(b.y & 0xffff0000u);
                        }
                        if (g.accumulate && nw + nc < g.N && mw + mr < g.M) {
                            const uint2 o = *reinterpret_cast<const uint2*>(Cw + (size_t)mr * g.ldc + nc);
                            v[0] += __uint_as_float(o.x << 16);
                            v[1] += __uint_as_float(o.x & 0xffff0000u);
                            v[2] += __uint_as_float(o.y << 16);
                            v[3] += __uint_as_float(o.y & 0xffff0000u);
                        }
                    }
                    *reinterpret_cast<uint2*>(st + mr * 128 + (((j * 4 + q) ^ (mr & 7)) * 16) + nh * 2) =
                        make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
                    __builtin_amdgcn_sched_barrier(0);
                }
            wave_lds_sync();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = q * 8 + (ln >> 3);
                const uint4 v = *reinterpret_cast<const uint4*>(st + r * 128 + (((ln & 7) ^ (ln >> 3)) * 16));
                char* dst = reinterpret_cast<char*>(Cw + (size_t)(q * 8) * g.ldc) + voff;
                if (mw + r < g.M && nok) *reinterpret_cast<uint4*>(dst) = v;
            }
        });
    };

    // fp32 C: one 32 x 32 block at a time, its rows 128 bytes; rows from Msplit on go to C2.
    auto store32 = [&](auto ACC_, int m0, int n0) {
        constexpr bool ACC = decltype(ACC_)::value;  // + C
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int mr = ln & 31, c8 = ln & 7, r8 = ln >> 3;
        static_for<FM>([&](auto I_) {
            constexpr int i = decltype(I_)::value;
            const int mw = m0 + wm * WM + i * 32;
            static_for<FN>([&](auto J_) {
                constexpr int j = decltype(J_)::value;
                const int n = n0 + wn * WN + j * 32 + c8 * 4;
                wave_lds_sync();
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(st + mr * 128 + (((2 * q + (ln >> 5)) ^ (mr & 7)) * 16)) =
                        make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                    acc[i][j][4 * q + 3]);
                wave_lds_sync();
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int r = q * 8 + r8, m = mw + r;
                    float4 v = *reinterpret_cast<const float4*>(st + r * 128 + ((c8 ^ r8) * 16));
                    if (m < g.M && n < g.N) {
                        float4* dst = reinterpret_cast<float4*>(
                            reinterpret_cast<float*>(m < g.Msplit ? g.C : g.C2) +
                            (size_t)(m < g.Msplit ? m : m - g.Msplit) * g.ldc + n);
                        if constexpr (ACC) {
                            const float4 o = *dst;
                            v = make_float4(v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w);
                        }
                        *dst = v;
                    }
                }
            });
        });
    };

    __syncthreads();  // k-tile 0
    static_for<NR>([&](auto R_) { read_one(I0{}, R_, stage_ptr(0), 0); });
    static_for<NR>([&](auto R_) { read_one(I1{}, R_, stage_ptr(0), 1); });
    int slot = 0;
    for (int i = 0; i < ntile; ++i) {
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b) zero16(acc[a][b]);
        for (int t = 0; t < KT; ++t) {
            const bf16_t* cur = stage_ptr(slot);
            slot = slot == STAGES - 1 ? 0 : slot + 1;
            const bf16_t* nxt = stage_ptr(slot);
            kstep(I0{}, I2{}, BF{}, cur, 2);
            kstep(I1{}, I3{}, BT{}, cur, 3);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(63) & 0xF0FFu);  // lgkmcnt(0): cur has no reader left
            __syncthreads();
            kstep(I2{}, I0{}, BF{}, nxt, 0);  // the next tile's k-tile 0 after the last
            kstep(I3{}, I1{}, BF{}, nxt, 1);
        }
        int m0, n0;
        tile_at(i, m0, n0);
        if constexpr (sizeof(CT) == 4) {
            if (g.accumulate) store32(BT{}, m0, n0);
            else store32(BF{}, m0, n0);
        } else {
            if (g.cbias || g.accumulate) store(BT{}, m0, n0);
            else store(BF{}, m0, n0);
        }
    }
}

template <bool TA, bool TB, int BM, typename CT = bf16_t>
int launch(const GemmDesc& g, int blocks, hipStream_t s) {
    constexpr int BN = 128, STAGES = 3;
    constexpr size_t smem = (size_t)STAGES * (BM + BN) * BK * sizeof(bf16_t) + 4 * 4096;  // 160 KB at 256 rows
    static_assert(smem <= 160 * 1024, "LDS per CU");
    static const bool ok = allow_lds(gemm_stream<TA, TB, CT, BM, BN, STAGES>, smem);
    if (!ok) {
        set_error("gemm: cannot reserve %zu B of LDS", smem);
        return GN_E_HIP;
    }
    const long tiles = (long)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    // beside another product a block per tile: blocks that stay would keep the other's waiting
    // (dX 4096 x 5632 x 2048 beside dW 2048 x 5632 x 4096: 190 -> 180 us, 188 -> 173 replayed)
    const unsigned grid = (unsigned)(g.beside ? tiles : std::min<long>(tiles, blocks));
    hipLaunchKernelGGL((gemm_stream<TA, TB, CT, BM, BN, STAGES>), dim3(grid), dim3(512), smem, s, g);
    GN_LAUNCH_CHECK("gemm (streamed tiles)");
    return GN_OK;
}

// compute units of the current device, rounded down to a multiple of 8 (one block each)
int stream_blocks() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        cus = 256;
    return std::max(8, cus / 8 * 8);
}

// Tile rows for g, and the time the product then takes (us, bf16 C): rounds of 256 x 128 or
// 128 x 128 tiles, whichever need less.  A round of the small ones takes 0.6 of a round of the
// large: 4.2 us + 0.29 per k-tile against 6.5 + 0.52 (up to 0.4 and 0.6 where a round fills the
// chip).  Measured, 256 -> 128 rows: 4096 x 768 x 3072 (one round either way) 33 -> 24 us, 2048^3
// 24.5 -> 20.2; 8192 x 768 x 3072 (one round against two) 39 -> 48, 2816 x 2304 x 768 14 -> 16.
int choose_rows(const GemmDesc& g, int blocks, double* us) {
    const long tn = (g.N + 127) / 128;
    const long r256 = ((g.M + 255) / 256 * tn + blocks - 1) / blocks;
    const long r128 = ((g.M + 127) / 128 * tn + blocks - 1) / blocks;
    const bool small = 0.62 * (double)r128 < (double)r256;
    *us = small ? (double)r128 * (4.2 + 0.29 * k_tiles(g)) : (double)r256 * (6.5 + 0.52 * k_tiles(g));
    return small ? 128 : 256;
}

template <int BM>
int launch_tile(const GemmDesc& g, int transA, int transB, int blocks, hipStream_t s) {
    if (!transA && !transB) return launch<false, false, BM>(g, blocks, s);
    if (!transA && transB) return launch<false, true, BM>(g, blocks, s);
    if (transA && !transB) return launch<true, false, BM>(g, blocks, s);
    return launch<true, true, BM>(g, blocks, s);
}

}  // namespace

double gemm_stream_us(const GemmDesc& g) {
    double us;
    choose_rows(g, stream_blocks(), &us);
    return us;
}

int gemm_dma_bf16(const GemmDesc& g, int transA, int transB, hipStream_t s) {
    if (g.Msplit < g.M) {
        set_error("gemm: a bf16 product has one destination");
        return GN_E_INVALID;
    }
    const int blocks = stream_blocks();
    double us;
    return choose_rows(g, blocks, &us) == 128 ? launch_tile<128>(g, transA, transB, blocks, s)
                                              : launch_tile<256>(g, transA, transB, blocks, s);
}

// Up to 1024 rows of dY and X, where a dW tile is mostly its store: this one leaves as whole row
// segments, the core's, staged per wave, in half the speed (us, register-staged 128 x 128 tiles -> core
// -> here, M x N x K of dW): 2048 x 2048 x 8 8.1 -> 14.9 -> 8.2, x 200 11.0 -> 14.4 -> 9.2, x 1003
// 25 -> 20.0 -> 14.6; 5632 x 2048 x 200 21.2 -> 31.0 -> 16.7; 4096 x 4096 x 8 16.4 -> 33.2 -> 17.2.
constexpr int kShortK = 16;  // k-tiles

// Or more than two rounds of 256 x 128 tiles, alone on the GPU.  Measured (us, a block per tile -> here,
// M x N x K of dW): 11264 x 2048 x 4096 180 -> 172, x 2048 112 -> 91; 32000 x 768 x 2001 120 -> 95;
// 8192 x 8192 x 4096 555 -> 472; the least gain just above the line (10240 x 1792 x 4096, 560 tiles,
// 153 -> 149).  Beside another product (an LM head's dX, 48 tiles over K = 32000) the core's blocks go
// on sharing the GPU: with blocks that stay the pair's pass was 522 -> 532.
bool gemm_stream_f32_wins(const GemmDesc& g, int transA, int transB) {
    if (!transA || transB || g.bias || g.cbias) return false;
    const long tiles = (long)((g.M + 255) / 256) * ((g.N + 127) / 128);
    return k_tiles(g) <= kShortK || (!g.beside && tiles > 2L * stream_blocks());
}

// Over a round of such tiles the column sums' own launch (one, ~5 us, up to these 1024 rows) costs less
// than the core's store: backward with db of 200 x 5632 x 2048 (replayed) 42.7 with the register-staged
// tiles -> 53.4 on the core -> 41 here; of 200 x 2048 x 2048, 128 tiles, 23.0 with the core's fused sums,
// which stays.
bool gemm_stream_sums_apart(const GemmDesc& g) {
    const long tiles = (long)((g.M + 255) / 256) * ((g.N + 127) / 128);
    return k_tiles(g) <= kShortK && tiles > stream_blocks() && gemm_stream_f32_wins(g, 1, 0);
}

int gemm_stream_f32(const GemmDesc& g, hipStream_t s) {
    const int blocks = stream_blocks();
    double us;
    if (k_tiles(g) <= kShortK && choose_rows(g, blocks, &us) == 128) return launch<true, false, 128, float>(g, blocks, s);
    return launch<true, false, 256, float>(g, blocks, s);
}

}  // namespace gn
