// C = alpha * A . B^T + beta * C [+ bias] [ReLU] with K split over the four waves of a workgroup: the kernel of the
// GEMMs whose 64 x 64 tiles leave most of the chip idle, or most of a tile empty.
//
// All four waves compute the same (16 TM) x (16 TN) outputs; wave w takes K-tiles w, w + 4, ... through an LDS ring of
// its own, so no wave waits for another inside the K loop (the only synchronisation is a wave's own vmcnt), and the four
// partial sums meet in LDS at the end, in a fixed order.
//
// What bounds these shapes is latency and occupancy, not a pipe: a 64 x 64 tile with K = 4136 in f32 is 55 us of one
// compute unit's matrix pipes whatever the other 200 units do.  Tiles of 32 x 32 or 16 x 16 outputs put 4 to 16 times as
// many units to work, and splitting K over the four SIMDs of a unit shortens the chain behind every output by four.
// The loads are the DMA of the other GEMM kernels (8 rows x 128 bytes of K per instruction, swizzled chunks), N and M
// are ragged (rows clamped, stores masked) and K may end in a partial K-tile (chunks past the end come from zeros).
//
// Measured (us, gemm_abt_kernel on 64 x 64 tiles / this kernel; f32 unless said otherwise): 336 x 304 x 2256 48.3 / 9.5,
// 865 x 147 x 4136 86.8 / 24.1, 700 x 700 x 4096 87.0 / 43.1, 512^3 11.6 / 5.7, 20031 x 15 x 1800 63.7 / 24.6,
// 50372 x 4 x 1208 79.1 / 43.8 (5.6 TB/s); bf16 16 x 4096 x 4096 31.3 / 5.8, 2027 x 6 x 1688 11.1 / 3.6, 52020 x 17 x 1472
// 25.3 / 25.8 (5.9 TB/s either way), 1019 x 622 x 6392 55.5 / 30.4; f16 362 x 669 x 4352 33.4 / 8.7, 1882 x 241 x 3152 27.0 / 11.6.
#include "gemm_common.h"

namespace sp {

// One K-step of a 16 x 16 fragment: 16 bytes of K per lane from either operand, B first (a lane then holds four
// consecutive output columns).  f32: the chunk holds four consecutive k of this lane group, and A and B agree on them.
template <int DT>
__device__ __forceinline__ f32x4 mma(const u32x4& b, const u32x4& a, f32x4 c) {
    if constexpr (DT == SP_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
    } else if constexpr (DT == SP_F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, b), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
    } else {
        const f32x4 vb = __builtin_bit_cast(f32x4, b), va = __builtin_bit_cast(f32x4, a);
#pragma unroll
        for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(vb[s], va[s], c, 0, 0, 0);
        return c;
    }
}

template <int DT, int TM, int TN, int NS>
__global__ __launch_bounds__(256) void gemm_wave_kernel(const void* A_first, const void* B_first, int M, int N, int K, int tiles_m,
                                                        int tiles_n, int batch, long stride_a, long stride_b, const GemmArgs g) {
    constexpr int KS = 4;                                   // waves, each with every KS-th K-tile
    constexpr int ES = DT == SP_F32 ? 4 : 2;
    constexpr int BK = ROW_BYTES / ES;
    constexpr int NIA = 2 * TM, NI = 2 * (TM + TN);         // DMA instructions per K-tile: 8 rows each
    constexpr int STAGE = NI * 8 * ROW_BYTES;
    static_assert((NS - 1) * NI < 64, "vmcnt counts to 63");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroups are dealt round-robin to the 8 XCDs: each XCD walks a contiguous range of the tiles of the whole batch,
    // along the longer side of a member's tile grid last, so that the panel its neighbours share stays in its L2.  (With
    // ranges within every member, members of one to seven tiles all began on the first XCDs: bf16 71 x (112 x 48 x 952)
    // 25.2 us, numbered through 7.4; f32 103 x (64 x 64 x 448) 16.6 / 7.8; the same tiles without a batch unchanged.)
    const unsigned tiles = (unsigned)tiles_m * (unsigned)tiles_n, all = tiles * (unsigned)batch;
    const unsigned block = blockIdx.y * tiles + blockIdx.x, xcd = block & 7u;
    unsigned t = xcd * (all / 8u) + (xcd < (all & 7u) ? xcd : (all & 7u)) + (block >> 3), member = 0;
    if (batch > 1) {
        member = t / tiles;
        t -= member * tiles;
    }
    const bool m_last = tiles_m >= tiles_n;
    const unsigned inner = m_last ? (unsigned)tiles_n : (unsigned)tiles_m;
    const unsigned hi = t / inner, lo = t - hi * inner;
    const long m0 = (long)(m_last ? hi : lo) * (16 * TM), n0 = (long)(m_last ? lo : hi) * (16 * TN);

    const long row_bytes = (long)K * ES;
    const unsigned char* pA = uniform_ptr((const unsigned char*)A_first + (long)member * stride_a + m0 * row_bytes);
    const unsigned char* pB = uniform_ptr((const unsigned char*)B_first + (long)member * stride_b + n0 * row_bytes);
    const unsigned my_lds = __builtin_amdgcn_readfirstlane((unsigned)(size_t)lds + wave * (NS * STAGE));
    const int nk = (K + BK - 1) / BK;
    const bool k_tail = K % BK != 0;
    const int r = lane >> 3;
    unsigned voff[NI];
    unsigned tail_in = 0;                                   // bit q: this lane's chunk of the last K-tile exists
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int blk = q < NIA ? q : q - NIA;
        const int kc = (lane & 7) ^ ((r ^ blk) & 7);
        const long first = q < NIA ? m0 : n0, last = (q < NIA ? M : N) - 1;
        const long row = first + blk * 8 + r < last ? first + blk * 8 + r : last;
        voff[q] = (unsigned)((row - first) * row_bytes) + kc * 16;
        if ((long)(nk - 1) * CHUNKS + kc < row_bytes / 16) tail_in |= 1u << q;
    }
    auto fetch = [&](int kt, unsigned stage) {
        const unsigned char* a = pA + (long)kt * ROW_BYTES;
        const unsigned char* b = pB + (long)kt * ROW_BYTES;
        const unsigned dst = my_lds + stage * STAGE;
        if (k_tail && kt == nk - 1) {
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                const unsigned char* inside = (q < NIA ? a : b) + voff[q];
                dma_to_lds_addr((tail_in >> q) & 1u ? inside : (const unsigned char*)kZeroChunk, dst + q * 8 * ROW_BYTES);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NI; ++q) dma_to_lds(q < NIA ? a : b, voff[q], dst + q * 8 * ROW_BYTES);
        }
    };

    // this wave's K-tiles: wave, wave + KS, ...
    const int mine = (nk - wave + KS - 1) / KS;
#pragma unroll
    for (int s = 0; s < NS; ++s)
        if (s < mine) fetch(wave + s * KS, s);

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int fi = lane & 15, fq = lane >> 4;
    const unsigned char* ring = lds + wave * (NS * STAGE);
    int stage = 0;
    for (int j = 0; j < mine; ++j) {
        // K-tile j has landed: with NS tiles under way that leaves NS - 1 behind it, near the end only "none" says it
        if (j + NS <= mine) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * NI) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned char* at = ring + stage * STAGE;
        u32x4 fa[2][TM], fb[2][TN];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int kc = 2 * fq + ks;
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[ks][i] = *reinterpret_cast<const u32x4*>(at + lds_offset(16 * i + fi, kc));
#pragma unroll
            for (int i = 0; i < TN; ++i) fb[ks][i] = *reinterpret_cast<const u32x4*>(at + NIA * 8 * ROW_BYTES + lds_offset(16 * i + fi, kc));
        }
        if (j + NS < mine) {
            // the stage is free once its fragments are in registers
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            fetch(wave + (j + NS) * KS, stage);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage = stage + 1 == NS ? 0 : stage + 1;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int jn = 0; jn < TN; ++jn) acc[i][jn] = mma<DT>(fb[ks][jn], fa[ks][i], acc[i][jn]);
    }

    // One quad of registers: C[row][col .. col + 3], the last one to three columns of a row element by element.  All
    // that is read is requested before any of it is waited for.
    constexpr int OT16 = DT == SP_BF16 ? SP_BF16 : SP_F16;
    unsigned char* const Cb = (unsigned char*)g.C + (long)member * g.stride_c;
    const bool half = g.out_dtype != SP_F32;
    auto put = [&](long row, long col, f32x4 v) {
        if (row >= M || col >= N) return;
        const long idx = row * N + col;
        const bool whole = col + 3 < N;
        float* c32 = (float*)Cb + idx;
        unsigned short* c16 = (unsigned short*)Cb + idx;
        f32x4 old = {0.f, 0.f, 0.f, 0.f}, bias = {0.f, 0.f, 0.f, 0.f};
        unsigned h[4] = {0, 0, 0, 0};
        if (whole) {
            if (g.beta != 0.f) {
                if (half) {
                    const u32x2 o = *reinterpret_cast<const u32x2_unaligned*>(c16);
                    h[0] = o.x & 0xffffu; h[1] = o.x >> 16; h[2] = o.y & 0xffffu; h[3] = o.y >> 16;
                } else {
                    old = *reinterpret_cast<const f32x4_unaligned*>(c32);
                }
            }
            if (g.bias) bias = *reinterpret_cast<const f32x4*>(g.bias + col);
        } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (col + e < N) {
                    if (g.beta != 0.f) {
                        if (half) h[e] = c16[e];
                        else old[e] = c32[e];
                    }
                    if (g.bias) bias[e] = g.bias[col + e];
                }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] *= g.alpha;
            if (g.beta != 0.f) v[e] += g.beta * (half ? half_bits_to_f32<OT16>(h[e]) : old[e]);
            v[e] += bias[e];
            if (g.relu) v[e] = fmaxf(v[e], 0.f);
        }
        if (half) {
            const u32x2 o = {pack_halves<OT16>(v[0], v[1]), pack_halves<OT16>(v[2], v[3])};
            if (whole) {
                *reinterpret_cast<u32x2_unaligned*>(c16) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (col + e < N) c16[e] = (unsigned short)(e < 2 ? o.x >> (16 * e) : o.y);
            }
        } else if (whole) {
            *reinterpret_cast<f32x4_unaligned*>(c32) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (col + e < N) c32[e] = v[e];
        }
    };
    // partial tiles: fragment f of wave w at (f * 4 + w) * 1 KiB; fragment f is then finished by wave f % 4.
    // The registers of lane l of a 16 x 16 fragment: row l % 16, columns 4 (l / 16) ...
    __syncthreads();                                    // the rings are not read any more
    f32x4* part = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jn = 0; jn < TN; ++jn) part[((i * TN + jn) * 4 + wave) * 64 + lane] = acc[i][jn];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jn = 0; jn < TN; ++jn) {
            const int f = i * TN + jn;
            if (f % 4 != wave) continue;
            const f32x4* p = part + f * 4 * 64 + lane;
            put(m0 + 16 * i + fi, n0 + 16 * jn + 4 * fq, (p[0] + p[64]) + (p[128] + p[192]));
        }
}

// ---- host side -------------------------------------------------------------------------------

template <int DT, int TM, int TN, int NS>
static int launch_wave(const GemmArgs& g, hipStream_t stream) {
    auto kernel = gemm_wave_kernel<DT, TM, TN, NS>;
    constexpr int ring = 4 * NS * 2 * (TM + TN) * 8 * ROW_BYTES, partial = TM * TN * 4096;
    constexpr int lds_bytes = ring > partial ? ring : partial;
    const int rc = ensure_dynamic_lds((const void*)kernel, lds_bytes);
    if (rc != SP_OK) return rc;
    const long blocks = (long)g.tiles_m * g.tiles_n;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (unsigned)g.batch), dim3(256), lds_bytes, stream, g.A, g.B, (int)g.M,
                       (int)g.N, (int)g.K, g.tiles_m, g.tiles_n, g.batch, g.stride_a, g.stride_b, g);
    return check_launch("sp_gemm_abt");
}

// LDS rings: two stages of 8 KiB per wave leave room for two workgroups on a compute unit, four of 4 KiB likewise; the
// larger tiles, one workgroup per unit, take all of the LDS they can use.  With more tiles than those places a ring of ONE
// stage: what a wave no longer has in flight, five workgroups (of 32 x 32; three and two of the larger tiles) on a unit
// have between them, and a workgroup's prologue and last sums hide behind the others' K loops.  (us, rings / one stage:
// f32 37 x (960 x 384 x 320), 52 tiles a unit, 130 / 104, 300 x (256 x 32 x 128), 9 a unit, 17.3 / 14.0; bf16
// 172 x (695 x 100 x 320) 69 / 43.5, 29 x (1528 x 176 x 2240) 89 / 66.  At one or two tiles a unit the rings are 5 % faster.)
template <int DT>
static int launch_wave_dtype(int tile_m, int tile_n, long cus, const GemmArgs& g, hipStream_t stream) {
    const long tiles = (long)g.tiles_m * g.tiles_n * g.batch;
    if (tile_m == 16) return launch_wave<DT, 1, 1, 4>(g, stream);
    if (tile_m == 32) return tiles > 2 * cus ? launch_wave<DT, 2, 2, 1>(g, stream) : launch_wave<DT, 2, 2, 2>(g, stream);
    if constexpr (DT != SP_F32) {
        if (tile_m == 64 && tile_n == 32) return tiles > cus ? launch_wave<DT, 4, 2, 1>(g, stream) : launch_wave<DT, 4, 2, 3>(g, stream);
        if (tile_m == 64) return tiles > cus ? launch_wave<DT, 4, 4, 1>(g, stream) : launch_wave<DT, 4, 4, 2>(g, stream);
    }
    return fail(SP_ERR_UNSUPPORTED, "sp_gemm_abt: no split-K kernel for a %d x %d tile", tile_m, tile_n);
}

int launch_gemm_wave(int dtype_in, int tile_m, int tile_n, long cus, const GemmArgs& g, hipStream_t stream) {
    switch (dtype_in) {
        case SP_F32: return launch_wave_dtype<SP_F32>(tile_m, tile_n, cus, g, stream);
        case SP_F16: return launch_wave_dtype<SP_F16>(tile_m, tile_n, cus, g, stream);
        default: return launch_wave_dtype<SP_BF16>(tile_m, tile_n, cus, g, stream);
    }
}

namespace {
struct GemmWaveKernelNames {
    GemmWaveKernelNames() {
        register_kernel("gemm_f32_split_16x16", (const void*)gemm_wave_kernel<SP_F32, 1, 1, 4>, 256);
        register_kernel("gemm_f32_split_32x32", (const void*)gemm_wave_kernel<SP_F32, 2, 2, 2>, 256);
        register_kernel("gemm_f32_split_32x32_1", (const void*)gemm_wave_kernel<SP_F32, 2, 2, 1>, 256);
        register_kernel("gemm_bf16_split_16x16", (const void*)gemm_wave_kernel<SP_BF16, 1, 1, 4>, 256);
        register_kernel("gemm_bf16_split_32x32", (const void*)gemm_wave_kernel<SP_BF16, 2, 2, 2>, 256);
        register_kernel("gemm_bf16_split_32x32_1", (const void*)gemm_wave_kernel<SP_BF16, 2, 2, 1>, 256);
        register_kernel("gemm_bf16_split_64x32", (const void*)gemm_wave_kernel<SP_BF16, 4, 2, 3>, 256);
        register_kernel("gemm_bf16_split_64x32_1", (const void*)gemm_wave_kernel<SP_BF16, 4, 2, 1>, 256);
        register_kernel("gemm_bf16_split_64x64", (const void*)gemm_wave_kernel<SP_BF16, 4, 4, 2>, 256);
        register_kernel("gemm_bf16_split_64x64_1", (const void*)gemm_wave_kernel<SP_BF16, 4, 4, 1>, 256);
    }
} gemm_wave_kernel_names;
}  // namespace

}  // namespace sp
