// C = alpha * A . B^T + beta * C [+ bias] [ReLU] for f32 A and B on the bf16 matrix pipe, without losing a bit of either.
//
// Every f32 is the exact sum of three bf16 numbers, x = h + m + l: h is x rounded to bf16, m what is left rounded to bf16, l
// the rest (8 significant bits each and two signs: 24 bits and more).  A product of two f32 is then nine products of bf16, of
// which the three smallest (m l, l m, l l) are below 2^-24 of it, of either sign, and are left out.  The other six go through
// v_mfma_f32_16x16x32_bf16, which multiplies exactly and adds in f32, 32 products to a rounding: sixteen times the rate of
// the f32 MFMA for six times the products.
//
// What this may not get wrong are numbers whose parts are no bf16: infinities and values that round to one (m would be a
// NaN), and non-zero values below 2^-110, whose l lies below the smallest bf16 (2^-133; the pipe keeps subnormal numbers).
// The loaders track the smallest non-zero magnitude, and a tile's results are looked at before they are stored: where either
// says so, the workgroup multiplies its tile again with f32 MFMAs.
//
// What bounds it: the matrix pipe at the clock its power allows.  8192 x 8192 x 4096 keeps the pipe busy for 84 % of the cycles,
// and takes 1.59 ms on zeros, 2.15 on random numbers: 255 TFLOP/s counted in f32, 1.53 PFLOP/s of bf16 (f32 MFMAs 3.70 ms,
// 149 TFLOP/s, 95 % of their peak).  Hence 16 x 16 x 32 MFMAs on two parts of 16 K each -- the 32 x 32 x 16 form needs a third
// fewer LDS reads and takes fewer cycles (1.53 ms on zeros), but more power (2.30 ms on numbers) -- and hence the split as every f32
// enters LDS, 7 vector instructions per number and workgroup, which run in the shadow of the MFMAs (split by every wave that
// reads it: as many instructions as the MFMAs leave room for).  Three stages of 16 K and one barrier each: with K-tiles of 32
// two of them would not fit 160 KiB.  The 128 wide tile is for outputs that leave units idle otherwise; alone on a unit its four
// waves have nobody to hide behind and take 1 us a K-tile, two side by side 0.6 each.
// Against float64 the sums are closer than the f32 MFMAs' (K = 512 3.4e-7 / 4.0e-7, K = 4096 1.0e-6 / 1.15e-6 of the 2-norm).
#include "gemm_tile.h"
#include "parts.h"

namespace sp {

// (A pointer made from integers has lost its address space, and a flat load counts as an LDS access as well.)
typedef const __attribute__((address_space(1))) unsigned char* global_ptr;
__device__ __forceinline__ f32x4 load_quad(const unsigned char* base, unsigned lane_offset) {
    return *reinterpret_cast<const __attribute__((address_space(1))) f32x4*>((global_ptr)base + lane_offset);
}

constexpr int PARTS_BK = 16;                       // f32 of K per stage
constexpr int PART_ROW = PARTS_BK * 2;             // bytes of one part of a row

template <int BM, int BN, int WM, int WN, bool RAGGED>
__global__ __launch_bounds__(WM* WN * 64, 2) void gemm_parts_kernel(SP_GEMM_PRELOADED, const GemmArgs g_rest) {
    SP_GEMM_TAKE_PRELOADED;
    constexpr int NW = WM * WN;
    constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
    constexpr int PART = (BM + BN) * PART_ROW, STAGE = 3 * PART;      // a stage: the h, m and l parts of all rows of A, then B
    static_assert(NW * 64 == BM + BN && BM % 64 == 0, "a wave loads 64 rows of one operand");
    static_assert(TM % 2 == 0 && TN % 2 == 0, "the A fragments alternate between two sets, the B fragments are replaced in pairs");
    constexpr int VALU_PER_MFMA = TM > 4 ? 2 : 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    tile_of_block(blockIdx.x, g.tiles_m, g.tiles_n, g.group_m, tm, tn);
    const long m0 = (long)tm * BM, n0 = (long)tn * BN, K = g.K;
    const unsigned char* const Ab = (const unsigned char*)g.A + (long)blockIdx.y * g.stride_a;
    const unsigned char* const Bb = (const unsigned char*)g.B + (long)blockIdx.y * g.stride_b;
    unsigned char* const Cb = (unsigned char*)g.C + (long)blockIdx.y * g.stride_c;
    const int nk = (int)((K + PARTS_BK - 1) / PARTS_BK);

    // ---- loader: four lanes share the 64 bytes of a row, the four loads of a lane are 16 rows apart ----
    const bool loads_a = wave * 64 < BM;
    const int quad = lane & 3;
    const unsigned char* src;
    unsigned voff[4];
    {
        long first = loads_a ? m0 + wave * 64 : n0 + (wave * 64 - BM);
        const long last = (loads_a ? g.M : g.N) - 1;
        if constexpr (RAGGED) first = first < last ? first : last;
        src = uniform_ptr((loads_a ? Ab : Bb) + first * K * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            long row = first + (lane >> 2) + 16 * i;
            if constexpr (RAGGED) row = row < last ? row : last;
            voff[i] = (unsigned)((row - first) * K * 4) + quad * 16;
        }
    }
    const bool k_tail = RAGGED && K % PARTS_BK != 0 && (nk - 1) * PARTS_BK + quad * 4 >= K;   // this lane's quad of the last K-tile is not there
    f32x4 ld[4];
    unsigned least = 0xffffffffu;                  // (parts.h)
    auto load = [&](int i, int kt) {
        const int at = kt < nk ? kt : nk - 1;      // (past the end: the last one again, into a stage that nobody reads)
        ld[i] = load_quad(src + (long)at * (PARTS_BK * 4), voff[i] - (RAGGED && k_tail && at == nk - 1 ? quad * 16 : 0));
    };
    auto load_all = [&](int kt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) load(i, kt);
    };
    // (Rows of 32 bytes, one behind the other: the sixteen lanes of a 16-byte read that LDS serves together -- 0-3, 12-15 and
    // 20-27, or 4-11, 16-19 and 28-31 -- then touch every bank once.)
    unsigned char* const wbase = lds + (wave * 64 + (lane >> 2)) * PART_ROW + quad * 8;
    // Half of the work of splitting quad i: h (and what is left), then m and l.
    u32x2 part;
    auto write_part = [&](int i, unsigned stage, int p) {
        part.x = pack_halves<SP_BF16>(ld[i][0], ld[i][1]);
        part.y = pack_halves<SP_BF16>(ld[i][2], ld[i][3]);
        *reinterpret_cast<u32x2*>(wbase + stage + p * PART + i * (16 * PART_ROW)) = part;
    };
    auto take_part = [&](int i) {
        ld[i][0] -= __uint_as_float(part.x << 16);
        ld[i][1] -= __uint_as_float(part.x & 0xffff0000u);
        ld[i][2] -= __uint_as_float(part.y << 16);
        ld[i][3] -= __uint_as_float(part.y & 0xffff0000u);
    };
    auto split_half = [&](int half, int kt, unsigned stage) {
        const int i = half >> 1;
        if ((half & 1) == 0) {
            if (RAGGED && k_tail && kt >= nk - 1) ld[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned w = parts_magnitude(ld[i][e]);
                least = w < least ? w : least;
            }
            write_part(i, stage, 0);
            take_part(i);
        } else {
            write_part(i, stage, 1);
            take_part(i);
            write_part(i, stage, 2);
        }
    };

    f32x4 acc[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    // An MFMA takes 32 products to a sum: two parts of 16 K each.  A: (h, m) and (h, l); B: (h, m), (m, h) and (l, h).
    const int fr = lane & 15, fq = lane >> 4;
    const int frag = fr * PART_ROW + (fq & 1) * 16;
    const bool second = fq >= 2;
    const unsigned afrag = (unsigned)(wm * WTM * PART_ROW + frag), bfrag = (unsigned)((BM + wn * WTN) * PART_ROW + frag);
    const unsigned abase[2] = {afrag + (second ? PART : 0), afrag + (second ? 2 * PART : 0)};
    const unsigned bbase[3] = {bfrag + (second ? PART : 0), bfrag + (second ? 0 : PART), bfrag + (second ? 0 : 2 * PART)};
    u32x4 fa[2][2], fb[TN][3];
    auto read_a = [&](unsigned stage, int i, u32x4(&f)[2]) {
#pragma unroll
        for (int p = 0; p < 2; ++p) f[p] = *reinterpret_cast<const u32x4*>(lds + abase[p] + stage + i * (16 * PART_ROW));
    };
    auto read_b = [&](unsigned stage, int j) {
#pragma unroll
        for (int p = 0; p < 3; ++p) fb[j][p] = *reinterpret_cast<const u32x4*>(lds + bbase[p] + stage + j * (16 * PART_ROW));
    };
    auto mma = [&](const u32x4(&a)[2], int i, int j, int p) {       // p: 0 h l + l h, 1 h m + m h, 2 h h + m m
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fb[j][2 - p]),
                                                            __builtin_bit_cast(bf16x8, a[p == 0 ? 1 : 0]), acc[i][j], 0, 0, 0);
    };
    // LDS answers in order, and the youngest 3 TN + 2 accesses of a step are reads of the stage after the one released: with
    // eight of them left under way every write, and every read of the released stage, is done.
    auto barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC87F);        // lgkmcnt(8); the loads of a later K-tile stay under way
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // ---- three stages: K-tile kt is multiplied from one, kt + 1 lies in the next, kt + 2 is split into the third ----
    {
        f32x4 ahead[2][4];                         // the first three K-tiles are requested together
#pragma unroll
        for (int t = 1; t < 3; ++t) {
            load_all(t);
#pragma unroll
            for (int i = 0; i < 4; ++i) ahead[t - 1][i] = ld[i];
        }
        load_all(0);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int i = 0; i < 8; ++i) split_half(i, t, t * STAGE);
#pragma unroll
            for (int i = 0; i < 4; ++i) ld[i] = ahead[t][i];
        }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);            // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < TN; ++j) read_b(0, j);
    read_a(0, 0, fa[0]);
    unsigned cur = 0, next = STAGE, into = 2 * STAGE;
    for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (i + 1 < TM) read_a(cur, i + 1, fa[(i + 1) & 1]);
            else read_a(next, 0, fa[0]);
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < TM) {
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int j = 0; j < TN; ++j) mma(fa[i & 1], i, j, p);
            } else {
#pragma unroll
                for (int j = 0; j < TN; j += 2) {    // each B fragment's successor as soon as it has done its part
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        mma(fa[i & 1], i, j, p);
                        mma(fa[i & 1], i, j + 1, p);
                    }
                    read_b(next, j);
                    read_b(next, j + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int half = (8 * i + TM - 2) / (TM - 1); half < 8 && half < (8 * (i + 1) + TM - 2) / (TM - 1); ++half) {
                split_half(half, kt + 2, into);
                if (half & 1) load(half >> 1, kt + 3);
            }
            if (i + 1 < TM) {
#pragma unroll
                for (int s = 0; s < 3 * TN; ++s) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);        // one MFMA,
                    __builtin_amdgcn_sched_group_barrier(0x2, VALU_PER_MFMA, 0);   // vector ALU in its shadow,
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);      // a write
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        barrier();
        const unsigned released = cur;
        cur = next; next = into; into = released;
    }

    // ---- what the parts cannot hold: the tile again in f32 ----
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum = __builtin_fmaf(acc[i][j][r], 0.f, sum);         // NaN if one of them is not finite
    if (__syncthreads_or(sum != 0.f || parts_tiny(least))) {
        clear();
        const unsigned char *pa[TM], *pb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const long row = m0 + wm * WTM + 16 * i + fr;
            pa[i] = Ab + (row < g.M ? row : g.M - 1) * K * 4;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const long row = n0 + wn * WTN + 16 * j + fr;
            pb[j] = Bb + (row < g.N ? row : g.N - 1) * K * 4;
        }
        for (long k = 0; k < K; k += 16) {
            const bool there = k + 4 * fq < K;               // (K is a multiple of 4)
            f32x4 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = load_quad(there ? pa[i] + (k + 4 * fq) * 4 : (const unsigned char*)kZeroChunk, 0);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = load_quad(there ? pb[j] + (k + 4 * fq) * 4 : (const unsigned char*)kZeroChunk, 0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][s], a[i][s], acc[i][j], 0, 0, 0);
        }
    }
    static_assert(NW * strip_bytes(WTN) <= 3 * STAGE, "epilogue staging must fit the stages");
    store_accumulators<SP_F32, WTM, WTN, RAGGED>(g, Cb, acc, lds + wave * strip_bytes(WTN), m0 + wm * WTM, n0 + wn * WTN, lane);
}

template <int BM, int BN, int WM, int WN, bool RAGGED>
static int launch(const GemmArgs& g, hipStream_t stream) {
    auto kernel = gemm_parts_kernel<BM, BN, WM, WN, RAGGED>;
    constexpr int lds_bytes = 9 * (BM + BN) * PART_ROW;
    const int rc = ensure_dynamic_lds((const void*)kernel, lds_bytes);
    if (rc != SP_OK) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((long)g.tiles_m * g.tiles_n), (unsigned)g.batch), dim3(WM * WN * 64), lds_bytes, stream,
                       SP_GEMM_PRELOADED_ARGS(g), g);
    return check_launch("sp_gemm_abt");
}

int launch_gemm_parts(int tile, const GemmArgs& g, hipStream_t stream) {
    if (tile == 256) return g.ragged ? launch<256, 256, 2, 4, true>(g, stream) : launch<256, 256, 2, 4, false>(g, stream);
    return g.ragged ? launch<128, 128, 2, 2, true>(g, stream) : launch<128, 128, 2, 2, false>(g, stream);
}

namespace {
struct GemmPartsKernelNames {
    GemmPartsKernelNames() {
        register_kernel("gemm_f32_parts_256x256", (const void*)gemm_parts_kernel<256, 256, 2, 4, false>, 512);
        register_kernel("gemm_f32_parts_256x256_ragged", (const void*)gemm_parts_kernel<256, 256, 2, 4, true>, 512);
        register_kernel("gemm_f32_parts_128x128", (const void*)gemm_parts_kernel<128, 128, 2, 2, false>, 256);
        register_kernel("gemm_f32_parts_128x128_ragged", (const void*)gemm_parts_kernel<128, 128, 2, 2, true>, 256);
    }
} gemm_parts_kernel_names;
}  // namespace
}  // namespace sp
