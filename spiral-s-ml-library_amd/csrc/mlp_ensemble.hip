// Fused forward of an ENSEMBLE of small f32 stacks on one shared input: member e of E computes
//     policy[e] = head(relu(x . W1[e]^T) . W2[e]^T)          x: (batch, K0), W1: (E, 64, K0), W2: (E, N, 64), all f32
// in one launch, activations never leaving registers.  This is the graph of the reference's Leduc policy
// (game/leduc/model_cem.spi:55-63: input -> matmul_ensemble_with_adjoint (E, 128, 64) -> relu ->
// matmul_ensemble_with_adjoint (E, 64, 64) -> masked_regret_matching' 3), which the graph interpreter
// (ml/layers.spi:194-240, 336-344) runs member by member, node by node.
//
// One wave per SIMD (four per workgroup, which share nothing but the load of the first layer's weights).  A wave takes the
// weights of its member into registers once -- 128 registers for the first layer, 32 per computed output for the second --
// and walks over 32-row tiles of the batch.
//   Layer 1 is v_mfma_f32_32x32x2_f32 with the WEIGHTS as the row operand, so a result tile is (features x batch rows)
// and lane (r, g) -- r = lane % 32 the batch row, g = lane / 32 -- holds features 8 a + 4 g + b (a, b = 0..3) of row
// r in register 4 a + b.  Both operands of an MFMA step take their two K-values from the lane halves g = 0, 1, and
// WHICH K-index a (step, half) pair stands for is free as long as both operands agree: step 4 j + i, half g stands
// for k = 8 j + 4 g + i, so every lane's inputs and weights are 16-byte loads.
//   Layer 2 is computed for at most 4 outputs (a masked head's valid columns, or a head that narrow), which is too
// little for the matrix pipe (a 32 x 32 tile for 3 useful rows costs a quarter of layer 1): every lane multiplies the
// 32 features of its row that it holds (after the relu) with the matching weights -- fused multiply-adds on the
// vector ALU -- and the two halves of a row are added across the lane halves.
// Sums therefore add up in another order than a row-by-row dot product; f32 throughout.  Tiles go through in pairs: the lanes
// with g = 0 run the head for their row of the first tile, the lanes with g = 1 for the second; the zeros behind the
// valid columns of a masked head are written by the whole wave, 16 bytes per lane.
#include "mlp_common.h"
#include "parts.h"
#include "gemm_dma.h"

#pragma clang fp contract(off)

namespace sp {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int EN_ROWS = 32;       // batch rows per tile
constexpr int EN_HIDDEN = 64;     // width of the hidden layer
constexpr int EN_THREADS = 256;
constexpr int EN_MAX_OUT = 4;     // computed outputs

struct EnsembleArgs {
    const float* x;
    const float* w1;
    const float* w2;
    const float* u;               // (members, batch) uniforms, or nullptr
    float* policy;                // (members, batch, n)
    int* action;                  // (members, batch), or nullptr
    long batch, tiles;
    int members, k0, n, nout, head, mask_size;
    unsigned* words;              // (members, batch) hash words of the binarize head, or nullptr
    unsigned modulo;
    unsigned per_piece;           // i / (k0 / 4) is i * per_piece >> 20 for i < 2048
    PhiloxStream ph;
};

// A member's first weight matrix, `rows` rows of K0 floats, into LDS for a workgroup of four waves: the loads in the order
// of memory, whole lines at a time and once per workgroup.  Read straight into its registers by every wave, a lane a line,
// the 32 KiB of 64 x 128 take 8 k cycles.  Microseconds of a captured launch, read straight / through LDS: 128-64-16, 8
// members of 1792 rows 13.8 / 11.6; 96-64-16, 2 of 28448 21.1 / 19.2; a hash of 200-128, 16 of 10240 32.3 / 28.7; 64-32, 7 of
// 5600 8.0 / 6.7.  Up to 32 inputs, a line or less a row, the barrier costs more: 16-64-64, 8 of 2016 6.3 / 6.7.  So it does
// for the four rows at most of a single layer under a head, up to 128 inputs: 64-64 masked to 2, 8 of 2128 4.8 / 5.6, 128-64 masked to 4,
// 2 of 984 6.7 / 6.9, but 200-64 masked to 3, 2 of 984 10.7 / 10.3.
// 16-byte piece p of row r lies at slot p ^ (r & (G - 1)) of the row, G the power of two in the pieces of a row, at most 16: lanes of
// different rows then read different banks.
constexpr bool ensemble_through_lds(int kg, int most_rows) { return kg > (most_rows > EN_MAX_OUT ? 4 : 16); }
__device__ __forceinline__ int ensemble_swizzle(int pieces) {
    const int g = pieces & -pieces;
    return (g < 16 ? g : 16) - 1;
}
__device__ __forceinline__ void ensemble_weights_to_lds(const float* w, int rows, int K0, unsigned per_piece, unsigned lds0, int wave, int lane) {
    const int pieces = K0 >> 2, mask = ensemble_swizzle(pieces);
    for (int b = wave; 64 * b < rows * pieces; b += 4) {
        const int i = 64 * b + lane, row = (int)((unsigned)i * per_piece >> 20), piece = (i - row * pieces) ^ (row & mask);
        mlp_dma((const unsigned char*)w, (unsigned)((row < rows ? row * K0 + 4 * piece : 0) * 4), __builtin_amdgcn_readfirstlane(lds0 + b * 1024));
    }
}

// KG: 8-wide groups of the input width the kernel is unrolled for; EXACT: K0 = 8 KG (else K0 < 8 KG and the groups
// past K0 are zeros); ACTION: an action per row is wanted (a uniform per row, from a tensor or a Philox stream)
template <int KG, bool EXACT, bool ACTION>
__global__ __launch_bounds__(EN_THREADS) void mlp_ensemble_kernel(const EnsembleArgs a) {
    constexpr bool LDS = ensemble_through_lds(KG, EN_HIDDEN);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int e = blockIdx.y;
    const int K0 = EXACT ? 8 * KG : a.k0;
    const int N = a.n, NOUT = a.nout;
    const int groups = K0 >> 3;
    const long batch = a.batch, tiles = a.tiles;
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    // ---- the member's weights, once ----
    f32x4 w1v[2][KG];             // [feature tile][j]: W1[e][32 t + r][8 j + 4 g .. + 3]
    if constexpr (LDS) {
        ensemble_weights_to_lds(a.w1 + (long)e * EN_HIDDEN * K0, EN_HIDDEN, K0, a.per_piece, (unsigned)(size_t)lds, wave, lane);
    } else {
        const float* w1 = a.w1 + (long)e * EN_HIDDEN * K0;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < KG; ++j) {
                const int jj = EXACT || j < groups ? j : 0;
                const f32x4 v = *reinterpret_cast<const f32x4*>(w1 + (long)(32 * t + r) * K0 + 8 * jj + 4 * g);
                w1v[t][j] = EXACT || j < groups ? v : zero4;
            }
    }
    f32x4 w2v[EN_MAX_OUT][2][4];  // [output][t][a]: W2[e][o][32 t + 8 a + 4 g .. + 3]: the features this lane half holds
    {
        const float* w2 = a.w2 + (long)e * N * EN_HIDDEN;
#pragma unroll
        for (int o = 0; o < EN_MAX_OUT; ++o)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(w2 + (long)(o < NOUT ? o : 0) * EN_HIDDEN + 32 * t + 8 * a4 + 4 * g);
                    w2v[o][t][a4] = o < NOUT ? v : zero4;
                }
    }

    // inputs of a tile: lane (r, g) takes x[row0 + r][8 j + 4 g .. + 3]; rows past the batch read the last row (their
    // results are not stored), groups past K0 read group 0 and count as zeros
    auto x_row = [&](long tile) {
        long row = tile * EN_ROWS + r;
        row = row < batch ? row : batch - 1;
        return a.x + row * K0 + 4 * g;
    };
    auto load_piece = [&](const float* xr, int j) { return *reinterpret_cast<const f32x4*>(xr + 8 * (EXACT || j < groups ? j : 0)); };

    const long stride = (long)gridDim.x * 4;
    long tile = (long)blockIdx.x * 4 + wave;
    if constexpr (!LDS) {
        if (tile >= tiles) return;
    }
    f32x4 xv[KG];
    {
        const float* xr = x_row(LDS && tile >= tiles ? 0 : tile);
#pragma unroll
        for (int j = 0; j < KG; ++j) xv[j] = load_piece(xr, j);
    }
    if constexpr (LDS) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tile >= tiles) return;
        const int pieces = K0 >> 2, swizzle = r & ensemble_swizzle(pieces);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < KG; ++j) {
                const int jj = EXACT || j < groups ? j : 0;
                const f32x4 v = *reinterpret_cast<const f32x4*>(lds + ((32 * t + r) * pieces + ((2 * jj + g) ^ swizzle)) * 16);
                w1v[t][j] = EXACT || j < groups ? v : zero4;
            }
    }
    const HeadOut out = HeadOut{a.policy, ACTION ? a.action : nullptr, nullptr, a.head, N};
    const int limit = a.mask_size > 0 ? a.mask_size : NOUT;
    const bool wave_fill = N > NOUT && (N & 3) == 0;
    const int s4 = N >> 2, c0 = (NOUT + 3) >> 2;

    // The zeros behind the valid columns of a masked head are written by the whole wave, 16 bytes per lane: lane l takes
    // pieces l, l + 64, ... of a tile's 32 s4 pieces.  64-wide rows (16 pieces): a lane's pieces are 1 KiB apart, all in
    // one column -- eight stores in a straight line; other widths walk (row and column of a piece advance by fixed
    // steps: no division inside the walk).
    const int fill_r0 = wave_fill ? lane / s4 : 0, fill_c0 = wave_fill ? lane - fill_r0 * s4 : 0;
    const int fill_dr = wave_fill ? 64 / s4 : 0, fill_dc = wave_fill ? 64 - fill_dr * s4 : 0;
    auto fill_zeros = [&](long t) {
        const long row0 = t * EN_ROWS;
        float* block = a.policy + ((long)e * batch + row0) * N;
        const int rows_here = batch - row0 < EN_ROWS ? (int)(batch - row0) : EN_ROWS;
        if (s4 == 16 && rows_here == EN_ROWS) {
            if (fill_c0 >= c0) {
                f32x4* mine = reinterpret_cast<f32x4*>(block) + lane;
#pragma unroll
                for (int k = 0; k < 8; ++k) mine[64 * k] = zero4;
            }
        } else {
            int rr = fill_r0, c = fill_c0;
            for (int idx = lane; idx < EN_ROWS * s4; idx += 64) {
                if (c >= c0 && rr < rows_here) *reinterpret_cast<f32x4*>(block + rr * N + 4 * c) = zero4;
                rr += fill_dr;
                c += fill_dc;
                if (c >= s4) {
                    c -= s4;
                    ++rr;
                }
            }
        }
    };

    // Both layers of one tile; the outputs of row r end up in BOTH lanes (r, 0) and (r, 1).
    auto forward = [&](long next_tile, float (&p)[4]) {
        // ---- layer 1: (64 features x 32 rows) += W1 . x^T, two K-values per step.  A register of inputs is asked for
        //      the NEXT tile's values as soon as this tile's MFMAs have read it: they arrive a whole tile ahead. ----
        const float* const xr_next = x_row(next_tile);
        f32x16 acc[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
#pragma unroll
        for (int j = 0; j < KG; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(w1v[t][j][i], xv[j][i], acc[t], 0, 0, 0);
            xv[j] = load_piece(xr_next, j);
            __builtin_amdgcn_sched_barrier(0);      // (keeps every load behind the MFMAs that free its register)
        }
        // ---- relu; layer 2: this lane's 32 features of its row against the matching weights, then the other half's ----
#pragma unroll
        for (int o = 0; o < EN_MAX_OUT; ++o) {
            p[o] = 0.f;
            if (o >= NOUT) continue;                           // (uniform)
            float s0 = 0.f, s1 = 0.f;                          // (two chains: an FMA need not wait for the one before)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    s0 = __builtin_fmaf(w2v[o][t][i >> 2][i & 3], fmaxf(acc[t][i], 0.f), s0);
                    s1 = __builtin_fmaf(w2v[o][t][(i + 1) >> 2][(i + 1) & 3], fmaxf(acc[t][i + 1], 0.f), s1);
                }
            const float mine = s0 + s1;
            p[o] = mine + __shfl_xor(mine, 32);
        }
    };

    // Tiles go through in pairs and the heads of a pair run together -- lanes (r, 0) finish row r of the first tile,
    // lanes (r, 1) row r of the second: the head is a chain of dependent instructions that costs the same for 64 lanes
    // as for 32, and vector-ALU work does not hide behind f32 MFMAs.
    for (; tile < tiles; tile += 2 * stride) {
        const long tile_b = tile + stride;
        const bool has_b = tile_b < tiles;                      // (uniform)
        float p[4] = {0.f, 0.f, 0.f, 0.f};                     // of this lane's row: the first tile's for g = 0, the second's for g = 1
#pragma unroll 1
        for (int half = 0; half < (has_b ? 2 : 1); ++half) {
            const long after = tile + (half + 1) * stride;      // the tile whose inputs are requested meanwhile
            float ph[4];
            forward(after < tiles ? after : tile, ph);
#pragma unroll
            for (int n = 0; n < 4; ++n) p[n] = g == half ? ph[n] : p[n];
        }
        int fill_end = 1 << 30;
        if (wave_fill) {
            fill_end = 4 * c0;
            fill_zeros(tile);
            if (has_b) fill_zeros(tile_b);
        }
        const long my_tile = g == 0 ? tile : tile_b;
        const long my_row = my_tile * EN_ROWS + r;
        if ((g == 0 || has_b) && my_row < batch) {
            const long grow = (long)e * batch + my_row;
            float u = 1.f;
            if constexpr (ACTION) u = a.u != nullptr ? a.u[grow] : reference_row_uniform(a.ph, grow);
            head_row4_any(a.head, out, p, grow, NOUT, limit, u, fill_end);
        }
    }
}

// The same on the bf16 matrix pipe, every f32 as three bf16 parts (parts.h): sixteen times the rate of the f32 MFMAs for the eight
// products of parts that count, and next to 16-bit MFMAs vector instructions hide.
// Two waves per SIMD: wave w and w + 4 of a workgroup take the two halves of one member's hidden layer, in 12 KS registers as
// parts.  A workgroup has four members and walks over tiles of 32 batch rows, a tile a round; the inputs of a round are split
// once per workgroup, every wave its share, into LDS, in the order the fragments of v_mfma_f32_32x32x16_bf16 are read.  Under
// the products of round n run the split of the inputs of round n + 1 and the second layer of round n - 1; in front of every
// second round one wave of a pair, in turn, does the heads of rounds n - 4 and n - 3, next to the other's products, and behind
// the barrier both store the rows of round n - 4.  Three buffers of inputs, so that the one barrier of a round can stand in its
// middle: nobody waits at a round's ends.  Second layer and head are those of the kernel above, in f32.
// A round has three sums: `large` of the products h h, which come from zero for each step of 16 inputs and are added by the vector
// ALU (three MFMAs later), and `small` of the other seven; both in `done` at its end.
// What bounds it: 32 x 65536 rows of 128 inputs take 250 to 260 us (f32 MFMAs 335 to 360), 65 rounds of 6.8 k cycles at 1.75 GHz; the matrix pipe is
// busy for 4.1 k of a round, beside it 410 vector instructions per wave and round, in part, and what waves
// wait for LDS and each other.  (Six products in one sum, without the additions, took 210 us and lost bits, see parts.h.  Taken
// back on the way there: one wave per SIMD with both halves 248 us, heads in front of a barrier at the round's end 240, zeros and
// probabilities of a row stored apart 257, fragments two steps ahead instead of one 230, stores past the caches 228.)
// With sampling (ACTION) 52 to 70 scalar registers live in lanes of vector registers: 264 us of 254 without.
// Rows of inputs, or weights of a member, that parts cannot hold (parts.h) take f32 MFMAs: a round is multiplied twice then, and
// the rows keep what is theirs, so a row's result depends on itself alone.  That product is read from memory as it goes: with an
// input above 2^60 in every tile the call above takes 735 us (the f32 kernel 366); tiny inputs and weights cost nothing.
typedef const __attribute__((address_space(1))) f32x4* global_f32x4;
constexpr int EP_THREADS = 512;
typedef unsigned u32x2_parts __attribute__((ext_vector_type(2)));

template <int KS, int NO, bool ACTION>
__global__ __launch_bounds__(EP_THREADS, 2) void mlp_ensemble_parts_kernel(const EnsembleArgs a) {
    constexpr int BUFFER = KS * 3072, RAW_AT = 3 * BUFFER, W2_AT = RAW_AT + 8 * 6144, SUMS_AT = W2_AT + 4096, PROBS_AT = SUMS_AT + 16384, FLAGS_AT = PROBS_AT + 16384 / 2;
    static_assert(KS == 2 || KS == 4 || KS == 8, "steps of 16 inputs, at most one for each wave to split");
    // the barrier stands in front of this step (with two steps: behind them); a wave's share of the next inputs is split before
    // it, and all of the second layer
    constexpr int BARRIER = KS == 2 ? 2 : KS / 2, FEATURES = 16 / BARRIER, SPLIT = KS == 8 ? 1 : 0;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int half = wave >> 2, pair = wave & 3;
    const int K0 = a.k0, N = a.n, NOUT = a.nout;
    const long batch = a.batch;
    const int tiles = (int)a.tiles;                    // (the launcher sees to it that they fit)
    const bool active = (int)blockIdx.y * 4 + pair < a.members;
    const int e = active ? (int)blockIdx.y * 4 + pair : a.members - 1;
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

    auto load8 = [&](const float* row, int s, f32x4 (&v)[2]) {      // k = 16 s + 8 g .. + 7 of a row of x or W1
        const int k = 16 * s + 8 * g;
        const bool there = k < K0;                                  // (K0 is a multiple of 8)
        const global_f32x4 at = (global_f32x4)(row + (there ? k : 0));
        v[0] = at[0];
        v[1] = at[1];
        return there;
    };

    // ---- inputs: this wave's share of a round is step `wave` of its tile (with fewer steps than waves some do the same),
    //      32 bytes a lane, by DMA into a ring of three ----
    const int my_step = wave % KS;
    const bool there = 16 * my_step + 8 * g < K0;      // (K0 is a multiple of 8)
    const int stride = gridDim.x, mine = (tiles - (int)blockIdx.x + stride - 1) / stride;      // rounds: tiles blockIdx.x + n stride (at least one)
    auto tile_at = [&](int n) { return (int)blockIdx.x + (n < mine ? n : 0) * stride; };
    const unsigned raw_at = RAW_AT + wave * 6144;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)lds);
    auto fetch_share = [&](int n, unsigned slot) {
        long row = (long)tile_at(n) * EN_ROWS + r;
        row = row < batch ? row : batch - 1;
        const unsigned char* const at = there ? (const unsigned char*)(a.x + row * K0 + 16 * my_step + 8 * g) : (const unsigned char*)kZeroChunk;
        dma_to_lds_addr(at, lds0 + raw_at + slot * 2048);
        dma_to_lds_addr(there ? at + 16 : at, lds0 + raw_at + slot * 2048 + 1024);
    };
    // one twelfth of splitting it: part i of numbers 2 d and 2 d + 1
    f32x4 raw[2];
    auto read_share = [&](unsigned slot) {
        raw[0] = *reinterpret_cast<const f32x4*>(lds + raw_at + slot * 2048 + lane * 16);
        raw[1] = *reinterpret_cast<const f32x4*>(lds + raw_at + slot * 2048 + 1024 + lane * 16);
    };
    u32x2_parts split_to[3];
    float two[2], most = 0.f;
    auto split_slice = [&](unsigned buffer, int slice) {
        const int d = slice / 3, i = slice % 3;
        if (i == 0) {
            two[0] = raw[d >> 1][2 * (d & 1)];
            two[1] = raw[d >> 1][2 * (d & 1) + 1];
            most = parts_most(most, two[0], two[1]);
            two[0] *= PARTS_X_SCALE;
            two[1] *= PARTS_X_SCALE;
        }
        split_to[i][d & 1] = take_parts(two[0], two[1]);
        if (i < 2) asm volatile("" : "+v"(two[0]), "+v"(two[1]));
        if (slice % 6 == 5) {
            unsigned char* const at = lds + buffer * BUFFER + my_step * 3072 + lane * 16 + (d >> 1) * 8;
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<u32x2_parts*>(at + k * 1024) = split_to[k];
        }
    };
    unsigned* const flags = reinterpret_cast<unsigned*>(lds + FLAGS_AT);     // [buffer][wave]: bit r: inputs of row r that parts cannot hold
    auto raise_flag = [&](unsigned buffer) {
        const unsigned long long bad = __ballot(most > PARTS_MOST);
        flags[buffer * 8 + wave] = (unsigned)(bad | bad >> 32);        // (every lane the same)
        most = 0.f;
    };
    fetch_share(0, 0);
    fetch_share(1, 1);
    fetch_share(2, 2);

    // ---- this half of the member's hidden layer, once ----
    parts_u32x4 w1[KS][3];
    bool w_bad, w_small = false;
    for (;;) {
        PartsWeights range;
        const float* const w = a.w1 + ((long)e * EN_HIDDEN + 32 * half + r) * K0;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            f32x4 v[2];
            if (!load8(w, s, v)) v[0] = v[1] = zero4;
#pragma unroll
            for (int k = 0; k < 8; ++k) range.take(v[k >> 2][k & 3]);
            split_parts(v, w_small ? PARTS_W_SCALE_SMALL : PARTS_W_SCALE, w1[s]);
        }
        const bool small = __any(range.small());
        w_bad = __any(range.wide()) || (small && __any(range.large()));
        if (!small || w_bad || w_small) break;
        w_small = true;                                // (once more, with the other scale)
    }
    // W2[e][o][32 half + 8 a4 + 4 g ..] at (o * 4 + a4) * 2 + g of the wave's 512 bytes, rows past NOUT are zeros
    f32x4* const w2 = reinterpret_cast<f32x4*>(lds + W2_AT + wave * 512);
    if (lane < 32) {
        const int o = lane >> 3, rest = lane & 7;
        const f32x4 v = *(global_f32x4)(a.w2 + ((long)e * N + (o < NOUT ? o : 0)) * EN_HIDDEN + 32 * half + 4 * rest);
        w2[lane] = o < NOUT ? v : zero4;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    read_share(0);
#pragma unroll
    for (int i = 0; i < 12; ++i) split_slice(0, i);
    raise_flag(0);
    __syncthreads();

    // ---- heads of rounds n and, for the lanes with g = 1, n + 1: the chain costs the same for 64 lanes as for 32 ----
    // sums: [round % 4][pair][half][output][row]
    float* const sums = reinterpret_cast<float*>(lds + SUMS_AT) + pair * 256;
    const int limit = a.mask_size > 0 ? a.mask_size : NOUT, s4 = N >> 2;
    const bool quads = (N & 3) == 0;
    float* const policy = a.policy + (long)e * batch * N;
    f32x4* const probs = reinterpret_cast<f32x4*>(lds + PROBS_AT) + pair * 32;         // [round % 4][pair][row], the first four columns
    auto heads = [&](int n, bool both) {
        if (!active) return;
        const int j = n + (both ? g : 0);
        const float* const at = sums + (j & 3) * 1024 + r;
        float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int o = 0; o < NO; ++o) p[o] = o < NOUT ? at[32 * o] + at[128 + 32 * o] : 0.f;
        switch (a.head) {
            case SP_HEAD_SOFTMAX: head_values4<SP_HEAD_SOFTMAX>(p, limit); break;
            case SP_HEAD_REGRET_MATCHING: head_values4<SP_HEAD_REGRET_MATCHING>(p, limit); break;
            case SP_HEAD_SOFTMAX_RM: head_values4<SP_HEAD_SOFTMAX_RM>(p, limit); break;
            default: break;
        }
        if (quads) probs[(j & 3) * 128 + r] = f32x4{p[0], 1 < NOUT ? p[1] : 0.f, 2 < NOUT ? p[2] : 0.f, 3 < NOUT ? p[3] : 0.f};
        const long row = ((long)blockIdx.x + (long)j * stride) * EN_ROWS + r;
        if (g == 1 && !both || row >= batch) return;
        if (!quads) {
            float* const to = policy + row * N;
#pragma unroll
            for (int o = 0; o < 4; ++o)
                if (o < NOUT) to[o] = p[o];
            for (int c = NOUT; c < N; ++c) to[c] = 0.f;
        }
        if constexpr (ACTION) {
            const long grow = (long)e * batch + row;
            a.action[grow] = head_pick4(p, a.u != nullptr ? a.u[grow] : reference_row_uniform(a.ph, grow));
        }
    };
    // Rows leave whole, 16 bytes per lane, in four stores from each wave of a pair for its 16 rows of a tile (lines that are written
    // in two pieces leave the L2 in two).  Rows past the tile or the batch are the last one once more: every lane stores every time,
    // so the counter of outstanding accesses runs at a known pace.
    const bool rows_out = quads && active;
    const int shift = (s4 & (s4 - 1)) == 0 ? 31 - __builtin_clz(s4) : -1;
    auto store_quarter = [&](int n, int q) {
        if (!rows_out) return;
        int piece = lane + 64 * q;
        asm volatile("" : "+v"(piece));                // (computed here: kept, the four of them are registers that are not there)
        const int rr0 = shift >= 0 ? piece >> shift : piece / s4, c = piece - rr0 * s4;
        const long tile0 = (long)tile_at(n) * EN_ROWS, left = batch - 1 - tile0;
        const int first = 16 * half + (rr0 < 15 ? rr0 : 15), rr = first < left ? first : (int)left;
        const f32x4 v = probs[(n & 3) * 128 + rr];
        *reinterpret_cast<f32x4*>(policy + tile0 * N + (rr * N + 4 * c)) = c == 0 ? v : zero4;
    };

    f32x16 done, large, small, these;                  // a round's results; the sums on their way there (parts.h)
    auto clear = [&](f32x16& c) {
#pragma unroll
        for (int i = 0; i < 16; ++i) c[i] = 0.f;
    };
    clear(done);
    parts_u32x4 xf[2][3];
    auto read_step = [&](unsigned buffer, int s, int i) {
        xf[s & 1][i] = *reinterpret_cast<const parts_u32x4*>(lds + buffer * BUFFER + s * 3072 + i * 1024 + lane * 16);
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) read_step(0, 0, i);
    unsigned now = 0, next = 1;                        // the buffers of this round's inputs and of the next one's
    // W2 of G features at a time (four outputs of four features are registers that are not there)
    constexpr int G = NO == 4 ? 2 : 4;
    typedef float weights_of __attribute__((ext_vector_type(G)));
    weights_of wv[NO];
    auto second_weights = [&](int f) {                 // of features f .. f + G - 1 of the 16 that this lane holds
#pragma unroll
        for (int o = 0; o < NO; ++o) wv[o] = *reinterpret_cast<const weights_of*>((const float*)(w2 + (o * 4 + (f >> 2)) * 2 + g) + (f & 3));
    };
    second_weights(0);
    // Round n: its products; the second layer of the round before it from `done`; the inputs of the next.
    auto work = [&](int n) {
        // The inputs of round n + 1 have landed: behind them came those of round n + 2 and, from round 4 on, four
        // stores of each of the last two rounds (a head's store more, and the wait is for a little more).
        if (rows_out && n >= 6) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        if (SPLIT == 0) read_share(next);
        if ((n & 1) == 0 && n >= 4 && ((n >> 1) & 1) == half) heads(n - 4, true);
        float s2[NO][2];
#pragma unroll
        for (int o = 0; o < NO; ++o) s2[o][0] = s2[o][1] = 0.f;
        auto second = [&](int f) {
            const float y = vmax(done[f], 0.f);
#pragma unroll
            for (int o = 0; o < NO; ++o) {
                s2[o][f & 1] = __builtin_fmaf(wv[o][f % G], y, s2[o][f & 1]);
                asm volatile("" : "+v"(s2[o][f & 1]));              // (here, and not where the sums are used)
            }
            if (f % G == G - 1) second_weights((f + 1) % 16);
        };
        auto put_sum = [&](int o, bool write) {
            if (!write) {
                s2[o][0] = s2[o][0] + s2[o][1];
                s2[o][0] += __shfl_xor(s2[o][0], 32);
            } else if (g == 0) {
                sums[((n - 1) & 3) * 1024 + half * 128 + r + 32 * o] = s2[o][0];
            }
        };
        auto barrier = [&]() {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F);                     // lgkmcnt(0): loads and stores stay under way
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        parts_u32x4 flag[2];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (s == BARRIER) barrier();
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const parts_u32x4 w = w1[s][PARTS_W[m]], x = xf[s & 1][PARTS_X[m]];
                if (m == 0 && s == 0) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(large) : "v"(w), "v"(x));
                else if (m == 0) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(these) : "v"(w), "v"(x));
                else if (m == 1 && s == 0) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(small) : "v"(w), "v"(x));
                else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(small) : "v"(w), "v"(x));
                // in the shadow of this MFMA:
                if (m < 3 && s + 1 < KS) read_step(now, s + 1, m);
                if (m < 3 && s + 1 == KS && BARRIER < KS) read_step(next, 0, m);
                if (s > 0 && m >= 4) {                              // (three MFMAs behind the one that they come from)
#pragma unroll
                    for (int i = 4 * (m - 4); i < 4 * (m - 3); ++i) large[i] += these[i];
                    asm volatile("" : "+v"(large));                 // (here, and not where the sums are used)
                }
                if (s < BARRIER)
#pragma unroll
                    for (int f = s * FEATURES + m * FEATURES / 8; f < s * FEATURES + (m + 1) * FEATURES / 8; ++f) second(f);
                if (s + 1 == SPLIT && m == 4) read_share(next);
                if (s == SPLIT || s == SPLIT + 1) {
                    const int slice = (s - SPLIT) * 8 + m;
                    if (slice < 12) split_slice(next, slice);
                    else if (slice == 12) raise_flag(next);
                }
                if (s == 0 && m == 5) fetch_share(n + 3, now);
                if (s + 1 == KS && m >= 4 && m < 6) flag[m - 4] = *reinterpret_cast<const parts_u32x4*>(flags + now * 8 + (m - 4) * 4);
                constexpr int APART = BARRIER < KS ? 8 * (KS - BARRIER) / 4 : 1;
                if (s >= BARRIER && ((s - BARRIER) * 8 + m) % APART == 1 && n >= 4) store_quarter(n - 4, ((s - BARRIER) * 8 + m) / APART);
                if (s == BARRIER && m < NO) put_sum(m, false);
                if (s == BARRIER + 1 && m < NO) put_sum(m, true);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (BARRIER + 1 >= KS) {
#pragma unroll
            for (int o = 0; o < NO; ++o) {
                if (BARRIER >= KS) put_sum(o, false);
                put_sum(o, true);
            }
        }
        if constexpr (BARRIER >= KS) {
            barrier();
#pragma unroll
            for (int i = 0; i < 3; ++i) read_step(next, 0, i);
            if (n >= 4)
#pragma unroll
                for (int q = 0; q < 4; ++q) store_quarter(n - 4, q);
        }
        // (what the compiler cannot see is that `small` comes from MFMAs: the last is eight passes)
        asm volatile("s_nop 15\n\ts_nop 3" : "+v"(small));
#pragma unroll
        for (int i = 0; i < 16; ++i) done[i] = large[i] + small[i];
        if (w_small) {
#pragma unroll
            for (int i = 0; i < 16; ++i) done[i] *= PARTS_UNSCALE_SMALL;
        }
        const parts_u32x4 both = flag[0] | flag[1];
        const unsigned bad = both.x | both.y | both.z | both.w;
        if (w_bad || __any(bad != 0)) {                             // rows that parts cannot hold, and no others, take their f32 sums
            clear(these);
            long row = (long)tile_at(n) * EN_ROWS + r;
            row = row < batch ? row : batch - 1;
            for (int s = 0; s < (K0 + 15) / 16; ++s) {
                f32x4 xv[2], wv1[2];
                if (!load8(a.x + row * K0, s, xv)) xv[0] = xv[1] = zero4;
                if (!load8(a.w1 + ((long)e * EN_HIDDEN + 32 * half + r) * K0, s, wv1)) wv1[0] = wv1[1] = zero4;
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        asm volatile("s_nop 3\n\tv_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+v"(these) : "v"(wv1[c][i]), "v"(xv[c][i]));
            }
            asm volatile("s_nop 15\n\ts_nop 15" : "+v"(these));
            const bool mine = w_bad || ((bad >> r) & 1) != 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) done[i] = mine ? these[i] : done[i];
        }
        now = next;
        next = next == 2 ? 0 : next + 1;
    };
    for (int n = 0; n <= mine; ++n) work(n);          // (one round more than there are: its products are not used)
    // what the rounds did not get to: the last two (or one, if it has no partner), and with an odd last round the two before it
    __syncthreads();
    const int last = (mine - 1) & ~1;                // the even round of the last pair
    if (half == 0) heads(last, last + 1 < mine);
    else if (last >= 2 && last + 2 > mine) heads(last - 2, true);
    __syncthreads();
    for (int n = mine > 3 ? mine - 3 : 0; n < mine; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) store_quarter(n, q);
}

// ONE ensemble layer and its head: policy[e] = head(x . W[e]^T) for a head of at most 4 computed outputs, or
// word[e][r] = (OR over j < 32 of (not (y[r][j] <= 0)) << j) mod modulo with y = x . W[e]^T -- the graphs of the
// reference's other agents (game/nl_hu_holdem/model_cem.spi:84-100: matmul_ensemble_with_adjoint -> masked regret
// matching; game/leduc/model_cfr.spi:56-61 and game/nl_hu_holdem/model_cfr.spi:82-88: matmul_ensemble -> binarize,
// ml/primitives.spi:817-821).  Either head needs at most the first 32 output columns, so the layer is ONE 32 x 32
// MFMA tile per 32 batch rows (the weights' rows past the needed columns are zeros) instead of the full product, and the
// (members x batch x outputs) activations are never written.  Same walk, same operand mapping and the same input
// prefetch as the first layer of the kernel above; lane (r, g) ends up with outputs 8 a + 4 g + b of row r.
// MODE 0: policy, 1: policy and action, 2: binarize.
template <int KG, bool EXACT, int MODE>
__global__ __launch_bounds__(EN_THREADS) void ensemble_layer_kernel(const EnsembleArgs a) {
    constexpr bool LDS = ensemble_through_lds(KG, MODE == 2 ? 32 : EN_MAX_OUT);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int e = blockIdx.y;
    const int K0 = EXACT ? 8 * KG : a.k0;
    const int N = a.n, NOUT = a.nout;                        // NOUT: rows of W that are read (<= 32)
    const int groups = K0 >> 3;
    const long batch = a.batch, tiles = a.tiles;
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    f32x4 wv[KG];                                            // W[e][r][8 j + 4 g .. + 3], rows past NOUT are zeros
    if constexpr (LDS) {
        ensemble_weights_to_lds(a.w1 + (long)e * N * K0, NOUT, K0, a.per_piece, (unsigned)(size_t)lds, wave, lane);
    } else {
        const float* w = a.w1 + ((long)e * N + (r < NOUT ? r : 0)) * K0 + 4 * g;
#pragma unroll
        for (int j = 0; j < KG; ++j) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(w + 8 * (EXACT || j < groups ? j : 0));
            wv[j] = (EXACT || j < groups) && r < NOUT ? v : zero4;
        }
    }
    auto x_row = [&](long tile) {
        long row = tile * EN_ROWS + r;
        row = row < batch ? row : batch - 1;
        return a.x + row * K0 + 4 * g;
    };
    auto load_piece = [&](const float* xr, int j) { return *reinterpret_cast<const f32x4*>(xr + 8 * (EXACT || j < groups ? j : 0)); };

    const long stride = (long)gridDim.x * 4;
    long tile = (long)blockIdx.x * 4 + wave;
    if constexpr (!LDS) {
        if (tile >= tiles) return;
    }
    f32x4 xv[KG];
    {
        const float* xr = x_row(LDS && tile >= tiles ? 0 : tile);
#pragma unroll
        for (int j = 0; j < KG; ++j) xv[j] = load_piece(xr, j);
    }
    if constexpr (LDS) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tile >= tiles) return;
        const int pieces = K0 >> 2, row = r < NOUT ? r : 0, swizzle = row & ensemble_swizzle(pieces);
#pragma unroll
        for (int j = 0; j < KG; ++j) {
            const int jj = EXACT || j < groups ? j : 0;
            const f32x4 v = *reinterpret_cast<const f32x4*>(lds + (row * pieces + ((2 * jj + g) ^ swizzle)) * 16);
            wv[j] = (EXACT || j < groups) && r < NOUT ? v : zero4;
        }
    }
    const HeadOut out = HeadOut{a.policy, MODE == 1 ? a.action : nullptr, nullptr, a.head, N};
    const int limit = a.mask_size > 0 ? a.mask_size : NOUT;
    const bool wave_fill = MODE != 2 && N > NOUT && (N & 3) == 0;
    const int s4 = N >> 2, c0 = (NOUT + 3) >> 2;
    const int fill_r0 = wave_fill ? lane / s4 : 0, fill_c0 = wave_fill ? lane - fill_r0 * s4 : 0;
    const int fill_dr = wave_fill ? 64 / s4 : 0, fill_dc = wave_fill ? 64 - fill_dr * s4 : 0;

    for (; tile < tiles; tile += stride) {
        const long next = tile + stride;
        const float* const xr_next = x_row(next < tiles ? next : tile);
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int j = 0; j < KG; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[j][i], xv[j][i], acc, 0, 0, 0);
            xv[j] = load_piece(xr_next, j);
            __builtin_amdgcn_sched_barrier(0);      // (left alone, the scheduler sinks the loads to the end of the tile,
                                                    //  and the next tile then starts by waiting for all of them)
        }
        const long row0 = tile * EN_ROWS;
        const long first = (long)e * batch + row0;              // row of the stacked (members x batch) outputs
        if constexpr (MODE == 2) {
            unsigned word = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                word |= (acc[i] <= 0.f ? 0u : 1u) << (8 * (i >> 2) + 4 * g + (i & 3));
            word |= (unsigned)__shfl_xor((int)word, 32);
            if (g == 0 && row0 + r < batch) a.words[first + r] = word % a.modulo;
        } else {
            float u = 1.f;
            if constexpr (MODE == 1) {
                const long row = first + (row0 + r < batch ? r : 0);
                u = a.u != nullptr ? a.u[row] : reference_row_uniform(a.ph, row);
            }
            int fill_end = 1 << 30;
            if (wave_fill) {
                fill_end = 4 * c0;
                float* block = a.policy + first * N;
                const int rows_here = batch - row0 < EN_ROWS ? (int)(batch - row0) : EN_ROWS;
                if (s4 == 16 && rows_here == EN_ROWS) {
                    if (fill_c0 >= c0) {
                        f32x4* mine = reinterpret_cast<f32x4*>(block) + lane;
#pragma unroll
                        for (int k = 0; k < 8; ++k) mine[64 * k] = zero4;
                    }
                } else {
                    int rr = fill_r0, c = fill_c0;
                    for (int idx = lane; idx < EN_ROWS * s4; idx += 64) {
                        if (c >= c0 && rr < rows_here) *reinterpret_cast<f32x4*>(block + rr * N + 4 * c) = zero4;
                        rr += fill_dr;
                        c += fill_dc;
                        if (c >= s4) {
                            c -= s4;
                            ++rr;
                        }
                    }
                }
            }
            const float p[4] = {acc[0], acc[1], acc[2], acc[3]};
            if (g == 0 && row0 + r < batch) head_row4_any(a.head, out, p, first + r, NOUT, limit, u, fill_end);
        }
    }
}

}  // namespace sp

using namespace sp;

template <int KG>
static const void* pick_ensemble_kernel_kg(bool exact, bool action) {
    if (exact) return action ? (const void*)mlp_ensemble_kernel<KG, true, true> : (const void*)mlp_ensemble_kernel<KG, true, false>;
    return action ? (const void*)mlp_ensemble_kernel<KG, false, true> : (const void*)mlp_ensemble_kernel<KG, false, false>;
}
// One workgroup (4 waves, one per SIMD) per compute unit while the members leave room for that: a wave then keeps its
// member's weights for all its tiles.
static long ensemble_blocks(long members, long tiles) {
    const long gx = (device_cu_count() + members - 1) / members, most = (tiles + 3) / 4;
    return gx < most ? gx : most;
}
// Rounds per workgroup on the bf16 pipe: four members a workgroup, one workgroup per unit.
static long ensemble_parts_blocks(long members, long tiles) {
    const long blocks = device_cu_count() / ((members + 3) / 4);
    return blocks < 1 ? 1 : blocks < tiles ? blocks : tiles;
}
// Which kernel takes two layers: the faster by what their rounds take.  The one on the bf16 pipe has rounds of a tile of four
// members, a workgroup a unit, the f32 one of a tile on each of a unit's four SIMDs; either is a start and so much for each round
// of the unit with the most.  Fitted on 350 calls of 2 to 1200 members, 16 to 131072 rows, with and without sampling, to 10 and
// 17 % (ninety of a hundred); on 450 others none that it sends to the bf16 pipe is more than 1 % slower there than in f32, and it is 2 %
// behind the faster one on the geometric mean.  (Us, f32 / bf16 pipe, taken first: 128 inputs, 17 x 32 rows 8.7 / 14.2,
// 9 x 6144 26.2 / 22.3, 3 x 65536 70 / 42, 516 x 2048 259 / 191; 32 inputs, 1028 x 2048 191 / 248, 516 x 2048 117 / 122,
// 5 x 65536 49 / 40, 33 x 8192 45 / 28.)  Below three members the bf16 pipe has half of its waves idle.
static bool ensemble_takes_parts(long members, long batch, int k0) {
    const long tiles = (batch + EN_ROWS - 1) / EN_ROWS, cus = device_cu_count();
    if (members < 3 || tiles > 2147480000l) return false;
    const long groups = (members + 3) / 4, blocks = ensemble_parts_blocks(members, tiles);
    const long parts = (groups * blocks + cus - 1) / cus * ((tiles + blocks - 1) / blocks);
    const long gx = ensemble_blocks(members, tiles);
    const long f32 = (members * gx + cus - 1) / cus * ((tiles + 4 * gx - 1) / (4 * gx));
    const float start[3][2] = {{6.2f, 3.7f}, {8.4f, 4.2f}, {11.5f, 6.1f}}, round[3][2] = {{2.f, 2.44f}, {2.45f, 3.55f}, {3.36f, 5.8f}};
    const int k = k0 <= 32 ? 0 : k0 <= 64 ? 1 : 2;                       // 32, 64 or 128 inputs
    return start[k][0] + round[k][0] * (float)parts < 0.9f * (start[k][1] + round[k][1] * (float)f32);
}

template <int KS>
static int launch_ensemble_parts(EnsembleArgs& a, hipStream_t stream, const char* what) {
    const bool action = a.action != nullptr;
    const void* kernel = a.nout <= 3 ? (action ? (const void*)mlp_ensemble_parts_kernel<KS, 3, true> : (const void*)mlp_ensemble_parts_kernel<KS, 3, false>)
                                     : (action ? (const void*)mlp_ensemble_parts_kernel<KS, 4, true> : (const void*)mlp_ensemble_parts_kernel<KS, 4, false>);
    const int lds_bytes = 3 * KS * 3072 + 8 * 6144 + 4096 + 16384 + 8192 + 128;
    const int rc = ensure_dynamic_lds(kernel, lds_bytes);
    if (rc != SP_OK) return rc;
    a.tiles = (a.batch + EN_ROWS - 1) / EN_ROWS;
    const long groups = (a.members + 3) / 4, gx = ensemble_parts_blocks(a.members, a.tiles);
    void* args[] = {(void*)&a};
    const hipError_t err = hipLaunchKernel(kernel, dim3((unsigned)gx, (unsigned)groups), dim3(EP_THREADS), args, lds_bytes, stream);
    if (err != hipSuccess) return fail(SP_ERR_DEVICE, "%s: launch failed: %s", what, hipGetErrorString(err));
    return check_launch(what);
}
static const void* pick_ensemble_kernel(int kg, bool exact, bool action) {
    return kg == 4 ? pick_ensemble_kernel_kg<4>(exact, action) : kg == 8 ? pick_ensemble_kernel_kg<8>(exact, action)
                                                                         : pick_ensemble_kernel_kg<16>(exact, action);
}

template <int KG, int MODE>
static const void* pick_layer_kernel_kg(bool exact) {
    return exact ? (const void*)ensemble_layer_kernel<KG, true, MODE> : (const void*)ensemble_layer_kernel<KG, false, MODE>;
}
template <int MODE>
static const void* pick_layer_kernel(int kg, bool exact) {
    return kg == 4 ? pick_layer_kernel_kg<4, MODE>(exact) : kg == 8 ? pick_layer_kernel_kg<8, MODE>(exact)
         : kg == 16 ? pick_layer_kernel_kg<16, MODE>(exact) : pick_layer_kernel_kg<32, MODE>(exact);
}

static int ensemble_launch(const void* kernel, EnsembleArgs& a, hipStream_t stream, const char* what) {
    a.tiles = (a.batch + EN_ROWS - 1) / EN_ROWS;
    const int pieces = a.k0 / 4, rows = a.w2 != nullptr ? EN_HIDDEN : a.nout, most_rows = a.w2 != nullptr ? EN_HIDDEN : a.words != nullptr ? 32 : EN_MAX_OUT;
    a.per_piece = ((1u << 20) + (unsigned)pieces - 1u) / (unsigned)pieces;
    const int lds_bytes = ensemble_through_lds((a.k0 + 7) / 8, most_rows) ? (rows * pieces + 63) / 64 * 1024 : 0;
    void* args[] = {(void*)&a};
    hipError_t err = hipLaunchKernel(kernel, dim3((unsigned)ensemble_blocks(a.members, a.tiles), (unsigned)a.members), dim3(EN_THREADS), args, lds_bytes, stream);
    if (err != hipSuccess) return fail(SP_ERR_DEVICE, "%s: launch failed: %s", what, hipGetErrorString(err));
    return check_launch(what);
}

// Reference role: the body of `graph_run_host model {ensemble}` (ml/layers.spi:336-344) for a graph of the shape
// input -> matmul_ensemble -> relu -> matmul_ensemble -> head (game/leduc/model_cem.spi:55-63) or
// input -> matmul_ensemble -> head (game/nl_hu_holdem/model_cem.spi:84-100).
extern "C" int sp_mlp_forward_ensemble(int dtype, const void* x, int32_t n_layers, const void* const* weights,
                                       const int32_t* dims, int32_t members, const float* u, const sp_philox_t* philox,
                                       float* policy_out, int32_t* action_out, int64_t batch, int32_t head,
                                       int32_t mask_size, void* stream) {
    SP_REQUIRE_PTR(x);
    SP_REQUIRE_PTR(policy_out);
    SP_OPTIONAL_PTR(u); SP_OPTIONAL_PTR(action_out);
    if (weights == nullptr || dims == nullptr) return fail(SP_ERR_NULL, "sp_mlp_forward_ensemble: weights/dims is NULL");
    if (dtype != SP_F32) return fail(SP_ERR_DTYPE, "sp_mlp_forward_ensemble: dtype must be f32");
    if (n_layers != 1 && n_layers != 2) return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: one or two layers, got %d", n_layers);
    if (members <= 0 || members > 65535) return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: members must be in [1, 65535]");
    if (batch <= 0 || batch > (1ll << 40) / members) return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: batch must be positive (and members x batch below 2^40)");
    if (head < SP_HEAD_NONE || head > SP_HEAD_SOFTMAX_RM) return fail(SP_ERR_ARG, "sp_mlp_forward_ensemble: unknown head %d", head);
    if (action_out != nullptr && u == nullptr && philox == nullptr)
        return fail(SP_ERR_NULL, "sp_mlp_forward_ensemble: action requested but u and philox are NULL");
    if (u != nullptr && philox != nullptr) return fail(SP_ERR_ARG, "sp_mlp_forward_ensemble: at most one of u and philox may be given");
    const int k0 = dims[0], n = dims[n_layers];
    const int k_max = n_layers == 2 ? 128 : 256;
    if (k0 < 8 || k0 % 8 != 0 || k0 > k_max)
        return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: input width %d must be a multiple of 8 in [8, %d]", k0, k_max);
    if (n_layers == 2 && dims[1] != EN_HIDDEN)
        return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: hidden width must be %d, got %d", EN_HIDDEN, dims[1]);
    if (n <= 0 || n > MLP_MAX_OUT) return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: output width %d must be in [1, %d]", n, MLP_MAX_OUT);
    if (mask_size < 0 || mask_size > n) return fail(SP_ERR_ARG, "sp_mlp_forward_ensemble: mask_size must be in [0, %d], got %d", n, mask_size);
    // a masked head gives probability zero to the columns past the mask: only the valid ones are computed
    const int nout = head != SP_HEAD_NONE && mask_size > 0 ? mask_size : n;
    if (nout > EN_MAX_OUT)
        return fail(SP_ERR_SHAPE, "sp_mlp_forward_ensemble: at most 4 computed outputs (the head's width, or its mask), got %d", nout);
    for (int i = 0; i < n_layers; ++i) {
        if (weights[i] == nullptr) return fail(SP_ERR_NULL, "sp_mlp_forward_ensemble: weights[%d] is NULL", i);
        if (!aligned16(weights[i])) return fail(SP_ERR_ALIGN, "sp_mlp_forward_ensemble: weights[%d] is not 16-byte aligned", i);
    }
    if (!aligned16(x)) return fail(SP_ERR_ALIGN, "sp_mlp_forward_ensemble: x is not 16-byte aligned");
    if (n % 4 == 0 && !aligned16(policy_out)) return fail(SP_ERR_ALIGN, "sp_mlp_forward_ensemble: policy_out is not 16-byte aligned");
    EnsembleArgs a{};
    a.ph.philox_mode = -1;
    int rc = mlp_set_philox(a.ph, philox, (int64_t)members * batch, n, __func__);
    if (rc != SP_OK) return rc;
    rc = require_gfx950(__func__);
    if (rc != SP_OK) return rc;
    a.x = (const float*)x; a.w1 = (const float*)weights[0]; a.w2 = n_layers == 2 ? (const float*)weights[1] : nullptr; a.u = u;
    a.policy = policy_out; a.action = action_out; a.batch = batch; a.members = members; a.k0 = k0; a.n = n; a.nout = nout;
    a.head = head; a.mask_size = mask_size;
    const int kg = k0 <= 32 ? 4 : k0 <= 64 ? 8 : k0 <= 128 ? 16 : 32;
    if (n_layers == 2 && ensemble_takes_parts(a.members, batch, k0)) {
        return kg == 4 ? launch_ensemble_parts<2>(a, (hipStream_t)stream, __func__) : kg == 8 ? launch_ensemble_parts<4>(a, (hipStream_t)stream, __func__)
                                                                                               : launch_ensemble_parts<8>(a, (hipStream_t)stream, __func__);
    }
    const void* kernel = n_layers == 2 ? pick_ensemble_kernel(kg, k0 == 8 * kg, action_out != nullptr)
                       : action_out != nullptr ? pick_layer_kernel<1>(kg, k0 == 8 * kg) : pick_layer_kernel<0>(kg, k0 == 8 * kg);
    return ensemble_launch(kernel, a, (hipStream_t)stream, __func__);
}

// Reference role: `graph_run_host model {ensemble}` for input -> matmul_ensemble -> binarize' (game/leduc/model_cfr.spi:56-61,
// game/nl_hu_holdem/model_cfr.spi:82-88; ml/layers.spi:439-446, ml/primitives.spi:817-821).
extern "C" int sp_ensemble_binarize(int dtype, const void* x, const void* weights, uint32_t* out, int32_t members,
                                    int64_t batch, int32_t k0, int32_t n, uint32_t modulo, void* stream) {
    SP_REQUIRE_PTR(x);
    SP_REQUIRE_PTR(weights);
    SP_REQUIRE_PTR(out);
    if (dtype != SP_F32) return fail(SP_ERR_DTYPE, "sp_ensemble_binarize: dtype must be f32");
    if (members <= 0 || members > 65535) return fail(SP_ERR_SHAPE, "sp_ensemble_binarize: members must be in [1, 65535]");
    if (batch <= 0 || batch > (1ll << 40) / members) return fail(SP_ERR_SHAPE, "sp_ensemble_binarize: batch must be positive (and members x batch below 2^40)");
    if (k0 < 8 || k0 % 8 != 0 || k0 > 256)
        return fail(SP_ERR_SHAPE, "sp_ensemble_binarize: input width %d must be a multiple of 8 in [8, 256]", k0);
    if (n <= 0) return fail(SP_ERR_SHAPE, "sp_ensemble_binarize: output width must be positive");
    if (modulo == 0) return fail(SP_ERR_ARG, "sp_ensemble_binarize: modulo must be positive");
    if (!aligned16(x) || !aligned16(weights)) return fail(SP_ERR_ALIGN, "sp_ensemble_binarize: x / weights not 16-byte aligned");
    int rc = require_gfx950(__func__);
    if (rc != SP_OK) return rc;
    EnsembleArgs a{};
    a.ph.philox_mode = -1;
    a.x = (const float*)x; a.w1 = (const float*)weights; a.batch = batch; a.members = members; a.k0 = k0; a.n = n;
    a.nout = n < 32 ? n : 32;          // the device's 32-bit shift drops the columns from 32 on
    a.words = out; a.modulo = modulo;
    const int kg = k0 <= 32 ? 4 : k0 <= 64 ? 8 : k0 <= 128 ? 16 : 32;
    return ensemble_launch(pick_layer_kernel<2>(kg, k0 == 8 * kg), a, (hipStream_t)stream, __func__);
}

namespace {
struct MlpEnsembleKernelNames {
    MlpEnsembleKernelNames() {
        register_kernel("mlp_forward_ensemble", (const void*)mlp_ensemble_kernel<16, true, false>, EN_THREADS);
        register_kernel("mlp_forward_ensemble_parts", (const void*)mlp_ensemble_parts_kernel<8, 3, false>, EP_THREADS);
        register_kernel("mlp_forward_ensemble_parts_action", (const void*)mlp_ensemble_parts_kernel<8, 4, true>, EP_THREADS);
    }
} mlp_ensemble_kernel_names;
}  // namespace
