// Fused forward of a stack of small f32 layers -- matmul [-> ln_l2] [-> relu | tanh | sigmoid] -> ... -> matmul -> row head
// [-> sampling] -- for one model or for every member of an ensemble on one shared input, in one launch.  These are the graphs
// of ml/layers.spi test3 - test5 (:564-665), which the interpreter (:194-240, 336-344) runs node by node.
//
// A wave owns 16 batch rows and takes them through the whole stack; the activations never leave its registers.  The product
// is v_mfma_f32_16x16x4 with the WEIGHTS as the row operand, so lane (r, q) -- r = lane % 16 the batch row, q = lane / 16 --
// ends up with features 16 t + 4 q + i of row r in register i of tile t.  Which K-index an MFMA step takes from lane group q
// is free as long as both operands agree: step i of K-block j stands for k = 16 j + 4 q + i, so a layer's result registers
// ARE the next layer's second operand.  The norm of a row is 4 registers x tiles and two cross-lane adds.
//   The weights of all layers sit in LDS in the order they are consumed (one 1 KiB block per 16 x 16 of W,
// lane l's 16 bytes at 16 l: conflict-free reads, and the DMA's natural layout), so the walk over a stack is one
// pointer that advances by 1 KiB per four MFMAs.  Features and K past a layer's widths are zeros.
//   The logits cross LDS once more, from the feature-major registers into one row per 16 lanes: the head and the sampling
// are the row primitives' own operations in their order, and the stores are whole rows.
//
// What bounds it: the f32 matrix pipe, 32 cycles per MFMA and SIMD (a 64-64-64-64 stack is 6144 of them for 16 rows), and the
// vector ALU, whose instructions do not hide behind f32 MFMAs whichever wave they come from (800 instructions, 3200 cycles, per
// 16 rows of that stack with ln_l2, relu, softmax and sampling).  Hence the products in a straight line where a layer is full,
// the uniforms of four tiles in one go, one reciprocal per norm.  16-row tiles because a batch of 16384 rows is then one
// tile per SIMD.
// Measured, that stack over 16384 rows (node by node / every layer through part_product, a draw per tile / this kernel, us):
// one model 32.8 / 13.8 / 9.9, 16 members 206 / 87 / 68.8 (the matrix pipe alone: 41).
//   Few rows: stack_features_kernel, below.
//   PARTS: the same with the products in three bf16 parts (parts.h), 192 MFMAs of 16 cycles for 16 rows instead of 192 of 32, and
// 400 vector instructions more, in part beside them: 16 members of 16384 rows 68 -> 56 us, of 57344 228 -> 190.  Bound by the
// vector ALU and the 7 us in which a workgroup's sixteen waves start together, with the same phases; a raised priority for waves
// in their products changed nothing.  Sixteen waves because their norms and heads hide behind each other's products (with six
// products instead of eight: sixteen waves 52.5 and 157, eight 63.6 and 186).  128 registers a lane are just enough: what the head,
// the draws and the f32 product need of addresses is computed where it is used.  (Kept over the loop, they were up to 30 registers
// in memory.)  The sums are closer to float64 than the f32 pipe's: error of the probabilities 0.41 to 1.00 of that, whatever
// the inputs (N(0, 1), uniform, 0 and 1, relu, one to eight non-zero numbers a row).
#include "mlp_common.h"
#include "row_common.h"
#include "gemm_dma.h"
#include "parts.h"

#pragma clang fp contract(off)

namespace sp {

constexpr int ST_ROWS = 16;            // batch rows per tile
constexpr int ST_MAX_LAYERS = 8;
constexpr int ST_MAX_WIDTH = 128;
constexpr int ST_MAX_OUT = 64;
constexpr int ST_MAX_THREADS = 512;
constexpr int ST_PARTS_THREADS = 1024;
constexpr int ST_BLOCK = 1024;         // bytes of a 16 x 16 block of weights
constexpr int ST_PARTS_UNIT = 3072;    // 16 features and 32 of K as three parts
constexpr int ST_SCRATCH = ST_ROWS * ST_MAX_OUT * 4;   // per wave: the logits on their way into rows
constexpr int ST_LDS = 160 * 1024;

struct StackArgs {
    const float* x;
    const float* u;                    // (members, batch) uniforms, or nullptr
    float* policy;                     // (members, batch, n)
    int* action;                       // (members, batch), or nullptr
    const float* w[ST_MAX_LAYERS];     // (members, dims[l + 1], dims[l])
    int dims[ST_MAX_LAYERS + 1];       // the last one: the computed outputs (a mask leaves only its own)
    int acts[ST_MAX_LAYERS];           // sp_map_op, plus SP_STACK_LN_L2
    unsigned per_kt[ST_MAX_LAYERS];    // of kt = 16 wide blocks of a layer's inputs: b / kt is b * per_kt >> 16 for b <= 64
    int n_layers, n, mask_size;        // n: output width; mask_size: the valid columns of the head
    int w_bytes;                       // weights in LDS
    int batch, tiles;
    long out_stride;                   // floats between two members' weights of the last layer
    PhiloxStream ph;
};

template <int HT, typename F>
__device__ __forceinline__ void map_tiles(f32x4 (&y)[HT], int nt, F f) {
#pragma unroll
    for (int t = 0; t < HT; ++t) {
        if (t < nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) y[t][i] = f(y[t][i]);
        __builtin_amdgcn_sched_barrier(0);      // (a tile at a time: registers)
    }
}

// y (NT tiles of features) = W . x for the weights at wp, K-blocks outermost; advances wp behind them.
// A full layer is a straight line, the weights of one K-block read ahead of the products of the one before.
template <int KT, int NT>
__device__ __forceinline__ void full_product(const unsigned char*& wp, const f32x4 (&x)[KT], f32x4 (&y)[NT]) {
    f32x4 w[2][NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        y[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        w[0][t] = *reinterpret_cast<const f32x4*>(wp + t * ST_BLOCK);
    }
#pragma unroll
    for (int j = 0; j < KT; ++j) {
        __builtin_amdgcn_sched_barrier(0);      // (else every load of the layer moves up here: registers)
        if (j + 1 < KT) {
#pragma unroll
            for (int t = 0; t < NT; ++t) w[(j + 1) & 1][t] = *reinterpret_cast<const f32x4*>(wp + ((j + 1) * NT + t) * ST_BLOCK);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) y[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j & 1][t][i], x[j][i], y[t], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    wp += KT * NT * ST_BLOCK;
}

// The same for kt <= KT blocks of K and nt <= NT tiles of features: groups of four tiles as above, then of two and of one (the sums of a
// group are chains which the matrix pipe takes in turn), the weights one block ahead (behind the last block of the stack lies the
// scratch: read, not used).
template <int G, int KT, int NT>
__device__ __forceinline__ void group_product(const unsigned char*& wp, const f32x4 (&x)[KT], f32x4 (&y)[NT], int t0, int kt) {
    f32x4 w[G];
#pragma unroll
    for (int t = 0; t < G; ++t) {
        y[t0 + t] = f32x4{0.f, 0.f, 0.f, 0.f};
        w[t] = *reinterpret_cast<const f32x4*>(wp + t * ST_BLOCK);
    }
#pragma unroll
    for (int j = 0; j < KT; ++j)
        if (j < kt) {
            wp += G * ST_BLOCK;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < G; ++t) {
                    y[t0 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t][i], x[j][i], y[t0 + t], 0, 0, 0);
                    if (i == 3) w[t] = *reinterpret_cast<const f32x4*>(wp + t * ST_BLOCK);      // (the next block's, in time for its first use)
                }
            __builtin_amdgcn_sched_barrier(0);
        }
}
template <int KT, int NT>
__device__ __forceinline__ void part_product(const unsigned char*& wp, const f32x4 (&x)[KT], f32x4 (&y)[NT], int kt, int nt) {
#pragma unroll
    for (int g = 0; g < NT; g += 4) {
        if (g + 4 <= nt) {
            group_product<4>(wp, x, y, g, kt);
        } else {
#pragma unroll
            for (int t = g; t < g + 4; ++t) y[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (g < nt) {
                if (nt & 2) group_product<2>(wp, x, y, g, kt);
                if (nt & 1) {
                    if (nt & 2) group_product<1>(wp, x, y, g + 2, kt);
                    else group_product<1>(wp, x, y, g, kt);
                }
            }
        }
    }
}

// ---- the products on the bf16 matrix pipe: both operands as three bf16 parts (parts.h), eight of the nine products, each of
// 32 of K in one v_mfma_f32_16x16x32_bf16.  Lane group q holds k = 32 j + 4 q + i and 32 j + 16 + 4 q + i, so that a layer's
// results are here, too, the next one's operand.
typedef __bf16 stack_bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void stack_parts(f32x4 v, f32x4 w, float scale, parts_u32x4 (&p)[3]) {
    const parts_f32x4 both[2] = {{v[0], v[1], v[2], v[3]}, {w[0], w[1], w[2], w[3]}};
    split_parts(both, scale, p);
}
__device__ __forceinline__ f32x4 parts_mfma(parts_u32x4 w, parts_u32x4 x, f32x4 y) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(stack_bf16x8, w), __builtin_bit_cast(stack_bf16x8, x), y, 0, 0, 0);
}

// A full layer, the weights of a tile of features and 32 of K read ahead of the products of the one before.
__device__ __forceinline__ void parts_product(const unsigned char*& wp, const parts_u32x4 (&x)[2][3], f32x4 (&y)[4]) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    parts_u32x4 w[2][3];
    f32x4 large = zero, small = zero;
#pragma unroll
    for (int s = 0; s <= 8; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        if (s < 8) {
#pragma unroll
            for (int i = 0; i < 3; ++i) w[s & 1][i] = *reinterpret_cast<const parts_u32x4*>(wp + s * ST_PARTS_UNIT + i * 1024);
        }
        if (s > 0) {
            const int t = (s - 1) >> 1, j = (s - 1) & 1, now = (s - 1) & 1;
            const f32x4 these = parts_mfma(w[now][0], x[j][0], zero);
            if (j == 0) small = zero;
#pragma unroll
            for (int p = 1; p < 8; ++p) small = parts_mfma(w[now][PARTS_W[p]], x[j][PARTS_X[p]], small);
            if (j == 0) large = these;
            else y[t] = (large + these) + small;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    wp += 8 * ST_PARTS_UNIT;
}

// The product of rows that parts cannot hold (16 members of 16384 rows with one in every tile 95 us, without 68, f32 75, host
// included), in f32 from the weights where they are, into the wave's scratch (a lane's own
// 16 bytes of each tile of features).
template <int HT>
__device__ __forceinline__ void wide_product(const float* W, int K, int F, const f32x4 (&x)[HT], unsigned char* scratch, int r, int q) {
    for (int t = 0; 16 * t < F; ++t) {
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < HT; ++j) {
            const int row = 16 * t + r, col = 16 * j + 4 * q;
            f32x4 w = {0.f, 0.f, 0.f, 0.f};
            if (row < F && col < K) w = *reinterpret_cast<const f32x4*>(W + (long)row * K + col);
            if (16 * j < K)
#pragma unroll
                for (int i = 0; i < 4; ++i) y = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[j][i], y, 0, 0, 0);
        }
        *reinterpret_cast<f32x4*>(scratch + t * 1024 + (q * 16 + r) * 16) = y;
    }
}

// The head of a row in 16 lanes, lane lq with columns 4 lq .. in v (used up): softmax or regret matching of its first `limit` columns.
template <bool REGRET>
__device__ __forceinline__ void stack_head(f32x4& v, int lq, int limit, float (&p)[4]) {
    // columns past the head's width, or its mask, enter as -inf (an exact 0 after the exponential) or 0
    if (limit < ST_MAX_OUT) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (4 * lq + k >= limit) v[k] = -__builtin_inff();
    }
    if constexpr (REGRET) {
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = 4 * lq + k < limit ? fmaxf(v[k], 0.f) : 0.f;
        const float s = group_reduce<16>(sum4(p), [](float m, float n) { return m + n; });
        const float inv_len = 1.f / (float)limit;
        const RowDivisor over_s(s);
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = 4 * lq + k < limit ? (s != 0.f ? over_s(p[k]) : inv_len) : 0.f;
    } else {
        const float m = group_max<16>(vmax(vmax(v[0], v[1]), vmax(v[2], v[3])));
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = fast_exp(v[k] - m);
        const float s = group_reduce<16>(sum4(p), [](float m, float n) { return m + n; });
        const float inv = 1.f / s;
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = p[k] * inv;
    }
}

// local_discrete_sampling (ml/primitives.spi:782-798) of such a row.
__device__ __forceinline__ int stack_pick(const float (&p)[4], int lq, float u) {
    const float incl = group_inclusive_scan<16>(sum4(p), lq);
    float run = dpp_move<0x138>(incl);
    if (lq == 0) run = 0.f;
    float c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        run = run + p[k];
        c[k] = run;
    }
    const float m = group_max<16>(sum4(p) > 0.f ? c[3] : -__builtin_inff());
    const float thr = u * m;
    int pick = 2147483647;
#pragma unroll
    for (int k = 3; k >= 0; --k)
        if (p[k] > 0.f && c[k] >= thr) pick = 4 * lq + k;
    return group_reduce<16>(pick, [](int m, int n) { return m < n ? m : n; });
}

// HT: 16-wide tiles of the widest layer (4 or 8).  PARTS: products in bf16 parts (FULL, and as many outputs).  FULL: the input and every hidden layer have exactly that many.  REGRET:
// regret matching instead of softmax as the head (of mask_size columns, either).
template <int HT, bool REGRET, bool FULL, bool PARTS = false>
__global__ __launch_bounds__(PARTS ? ST_PARTS_THREADS : ST_MAX_THREADS, HT == 4 ? 4 : 2) void mlp_stack_kernel(const StackArgs a) {
    static_assert(!PARTS || HT == 4, "the scratch holds one product of 64 features");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int e = blockIdx.y;
    const int layers = a.n_layers, k0 = a.dims[0], kt0 = (k0 + 15) >> 4;

    auto load_x = [&](int tile, f32x4 (&x)[HT]) {
        int row = tile * ST_ROWS + r;
        row = row < a.batch ? row : a.batch - 1;
        const float* xr = a.x + (long)row * k0 + 4 * q;
        // (a load that only some lanes take part in is waited for where the others go on.  Up to eight of them: at most the last one is of
        // that kind, 108-64-32, 48 rows, 5 k cycles for the inputs otherwise.  Up to four: the branches cost more, 32-16-64 relu, 7280 rows x 16
        // 12.7 us without them, 13.5 with, 60-16-16-4 17024 rows 8.0, 8.4 -- but where every block is whole.)
        constexpr bool WHOLE = !PARTS && (HT == 8 || FULL);
        if (!PARTS && k0 < 16) {
#pragma unroll
            for (int j = 0; j < HT; ++j) x[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (4 * q < k0) x[0] = *reinterpret_cast<const f32x4*>(xr);
            return;
        }
#pragma unroll
        for (int j = 0; j < HT; ++j) {
            if (WHOLE && 16 * j + 16 <= k0) {
                x[j] = *reinterpret_cast<const f32x4*>(xr + 16 * j);
            } else {
                x[j] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (j < kt0 && 16 * j + 4 * q < k0) x[j] = *reinterpret_cast<const f32x4*>(xr + 16 * j);
            }
        }
    };
    int tile = blockIdx.x * waves + wave;
    f32x4 x[HT];
    load_x(tile < a.tiles ? tile : 0, x);

    const int stride = gridDim.x * waves;
    // The uniforms of four tiles at once, lane group q those of tile q from here: a draw is 250 vector instructions.
    auto draw = [&](int tile) {
        int rr = r, qq = q;
        if constexpr (PARTS) asm volatile("" : "+v"(rr), "+v"(qq));      // (see wide_product)
        const long at = (long)(tile + (long)qq * stride) * ST_ROWS + rr;
        const int row = at < a.batch ? (int)at : a.batch - 1;
        if (a.ph.philox_mode < 0) return a.u[(long)e * a.batch + row];
        if (a.ph.member_rows > 0) return run_row_uniform<unsigned>(a.ph, row, a.ph.draw_offset + (unsigned long long)e * a.ph.member_draws);
        return run_row_uniform<unsigned>(a.ph, (unsigned)e * a.batch + row, a.ph.draw_offset);
    };
    float u4 = 1.f;
    // ---- the member's weights, once per workgroup ----
    const unsigned lds0 = (unsigned)(size_t)lds;
    bool weights_wide = false, weights_small = false;
    auto weights_of = [&](int l) { return a.w[l] + (long)e * (l + 1 < layers ? (long)a.dims[l] * a.dims[l + 1] : a.out_stride); };
    if constexpr (!PARTS) {
        unsigned dst = lds0;
        for (int l = 0; l < layers; ++l) {
            const int K = a.dims[l], F = a.dims[l + 1], kt = (K + 15) >> 4, nt = (F + 15) >> 4;
            const float* W = weights_of(l);
            // in the order the products read them: full_product's tiles in one group, part_product's in fours, two and one
            const bool full = FULL && (l + 1 < layers || nt == ST_MAX_OUT / 16);
            const unsigned mine = (unsigned)(r * K + 4 * q) * 4;
            const int whole = full ? nt : nt & ~3, log_group = full && nt == 8 ? 3 : 2;       // tiles in groups (of 8 or 4)
            const unsigned per_kt = a.per_kt[l];
            for (int b = wave; b < kt * nt; b += waves) {
                int tile, block;
                if (!FULL && nt == 1) {
                    tile = 0;
                    block = b;
                } else if (b < kt * whole) {
                    const int turn = b >> log_group, group = (int)((unsigned)turn * per_kt >> 16);
                    tile = (group << log_group) + (b & ((1 << log_group) - 1));
                    block = turn - group * kt;
                } else {                                  // a group of two, if nt has one, and the last tile
                    const int over = b - kt * whole, two = nt & 2;
                    tile = over < kt * two ? whole + (over & 1) : whole + two;
                    block = over < kt * two ? over >> 1 : over - kt * two;
                }
                const int row = 16 * tile, col = 16 * block;
                const unsigned to = __builtin_amdgcn_readfirstlane(dst + b * ST_BLOCK);
                const unsigned char* const at = (const unsigned char*)(W + row * K + col);
                if (row + 16 <= F && col + 16 <= K) mlp_dma(at, mine, to);
                else dma_to_lds_addr(row + r < F && col + 4 * q < K ? at + mine : (const unsigned char*)kZeroChunk, to);
            }
            dst += kt * nt * ST_BLOCK;
        }
        if (tile >= a.tiles) {                           // (a wave with rows: in front of its first products)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
    } else {
        // units (layer, tile of features, 32 of K) wave, wave + waves, ... of the whole stack, two of them in flight
        const int units = 8 * layers;
        int* const flags = reinterpret_cast<int*>(lds + a.w_bytes);       // (the scratch, not in use yet)
        for (;;) {
            PartsWeights range;
            for (int n0 = wave; n0 < units; n0 += 2 * waves) {
                f32x4 v[2][2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int n = n0 + i * waves < units ? n0 + i * waves : n0, l = n >> 3, K = a.dims[l];
                    const int row = 16 * ((n >> 1) & 3) + r, col = 32 * (n & 1) + 4 * q;
                    const float* const at = weights_of(l) + (long)row * K + col;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        v[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
                        if (row < a.dims[l + 1] && col + 16 * h < K) v[i][h] = *reinterpret_cast<const f32x4*>(at + 16 * h);
                    }
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (i == 1 && n0 + waves >= units) break;
                    parts_u32x4 p[3];
#pragma unroll
                    for (int k = 0; k < 8; ++k) range.take(v[i][k >> 2][k & 3]);
                    stack_parts(v[i][0], v[i][1], weights_small ? PARTS_W_SCALE_SMALL : PARTS_W_SCALE, p);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        *reinterpret_cast<parts_u32x4*>(lds + (n0 + i * waves) * ST_PARTS_UNIT + k * 1024 + lane * 16) = p[k];
                }
            }
            flags[wave] = (__any(range.small()) ? 1 : 0) | (__any(range.large()) ? 2 : 0) | (__any(range.wide()) ? 4 : 0);      // every lane the same
            __syncthreads();
            int any = 0;
            for (int w = 0; w < waves; ++w) any |= flags[w];
            any = __builtin_amdgcn_readfirstlane(any);
            __syncthreads();
            weights_wide = (any & 4) != 0 || (any & 3) == 3;
            if ((any & 1) == 0 || weights_wide || weights_small) break;
            weights_small = true;                      // (once more, with the other scale)
        }
    }
#pragma unroll
    for (int j = 0; j < HT; ++j) asm volatile("" : "+v"(x[j]));       // (the compiler's own wait for the first inputs: here, not in the loop)
    unsigned char* const scratch = lds + a.w_bytes + wave * ST_SCRATCH;

    float* const policy = a.policy + (long)e * a.batch * a.n;
    int* const action = a.action + (long)e * a.batch;       // (only used where a.action is not null)
    for (int turn = 0; tile < a.tiles; tile += stride, ++turn) {
        if (a.action != nullptr && (turn & 3) == 0) u4 = draw(tile);
        if constexpr (!PARTS) {
            if (turn == 0) {                             // the draw runs while the weights are on their way
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
            }
        }
        const unsigned char* wp = lds + lane * 16;
        f32x4 xn[HT];
        load_x(tile + stride < a.tiles ? tile + stride : tile, xn);
        // rows with numbers that parts cannot hold get the f32 product: the others' sums are theirs alone either way
        auto product_of_parts = [&](int l, f32x4 (&y)[HT]) {
          if constexpr (PARTS) {
            float most = 0.f;
            parts_u32x4 xp[2][3];
#pragma unroll
            for (int j = 0; j < HT; ++j) most = parts_most(parts_most(most, x[j][0], x[j][1]), x[j][2], x[j][3]);
            const unsigned long long lanes = __ballot(most > PARTS_MOST || weights_wide);
            if (lanes != 0) {
                int row = r, group = q;
                asm volatile("" : "+v"(row), "+v"(group));      // (addresses are computed here: kept, they are registers that are not there)
                wide_product<HT>(weights_of(l), a.dims[l], a.dims[l + 1], x, scratch, row, group);
            }
            stack_parts(x[0], x[1], PARTS_X_SCALE, xp[0]);
            stack_parts(x[2], x[3], PARTS_X_SCALE, xp[1]);
            parts_product(wp, xp, y);
            if (weights_small) {
#pragma unroll
                for (int t = 0; t < HT; ++t) y[t] *= PARTS_UNSCALE_SMALL;
            }
            if (lanes != 0) {
                const bool mine = (((lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) >> r) & 1) != 0;
#pragma unroll
                for (int t = 0; t < HT; ++t)
                    if (mine && 16 * t < a.dims[l + 1]) y[t] = *reinterpret_cast<const f32x4*>(scratch + t * 1024 + lane * 16);
            }
          }
        };
        for (int l = 0; l + 1 < layers; ++l) {
            const int nt = a.dims[l + 1] >> 4;
            f32x4 y[HT];
            if constexpr (PARTS) product_of_parts(l, y);
            else if constexpr (FULL) full_product<HT, HT>(wp, x, y);
            else part_product<HT, HT>(wp, x, y, (a.dims[l] + 15) >> 4, nt);
            const int act = a.acts[l];
            if (act & SP_STACK_LN_L2) {       // local_ln_l2 (ml/primitives.spi:701-703)
                float s0 = 0.f, s1 = 0.f;
#pragma unroll
                for (int t = 0; t < HT; ++t) {
                    s0 = __builtin_fmaf(y[t][0], y[t][0], s0);
                    s1 = __builtin_fmaf(y[t][1], y[t][1], s1);
                    s0 = __builtin_fmaf(y[t][2], y[t][2], s0);
                    s1 = __builtin_fmaf(y[t][3], y[t][3], s1);
                }
                float s = s0 + s1;
                s += __shfl_xor(s, 16);
                s += __shfl_xor(s, 32);
                const RowDivisor over_s(s);
                // (no row of the wave is zero or needs the scale, as nearly always: the same quotients by one multiplication)
                if (__all(s != 0.f && over_s.scale == 1.f)) map_tiles<HT>(y, FULL ? HT : nt, [&](float v) { return v * over_s.inv; });
                else map_tiles<HT>(y, FULL ? HT : nt, [&](float v) { return s != 0.f ? over_s(v) : 0.f; });
            }
            const int map = act & ~SP_STACK_LN_L2;
            if (map == SP_MAP_RELU) map_tiles<HT>(y, FULL ? HT : nt, [](float v) { return fmaxf(v, 0.f); });
            else if (map == SP_MAP_TANH) map_tiles<HT>(y, FULL ? HT : nt, [](float v) { return tanhf(v); });
            else if (map == SP_MAP_SIGMOID) map_tiles<HT>(y, FULL ? HT : nt, [](float v) { return 1.f / (1.f + expf(-v)); });
#pragma unroll
            for (int t = 0; t < HT; ++t) x[t] = y[t];
        }
        f32x4 logits[ST_MAX_OUT / 16];
        const int nt = (a.dims[layers] + 15) >> 4;
        if constexpr (PARTS) product_of_parts(layers - 1, logits);
        else if (FULL && nt == ST_MAX_OUT / 16) full_product<HT, ST_MAX_OUT / 16>(wp, x, logits);
        else part_product<HT, ST_MAX_OUT / 16>(wp, x, logits, (a.dims[layers - 1] + 15) >> 4, nt);

        // ---- logits into rows: quad c of row r at slot c ^ r of its 256 bytes ----
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t < nt) *reinterpret_cast<f32x4*>(scratch + r * 256 + (((4 * t + q) ^ r) & 15) * 16) = logits[t];
        // the next tile's inputs are waited for here, in front of the stores: the counter of outstanding accesses runs in
        // order, and behind them that wait would be one for the stores
#pragma unroll
        for (int j = 0; j < HT; ++j) {
            x[j] = xn[j];
            asm volatile("" : "+v"(x[j]));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // ---- the head and the sampling: lane l of 16 holds columns 4 l .. of its row, as in the row primitives ----
        int lq = r, hq = q;                       // (lane % 16 again: here the column quad)
        if constexpr (PARTS) asm volatile("" : "+v"(lq), "+v"(hq));      // (see wide_product)
        const int limit = a.mask_size;
        const int rows_here = a.batch - tile * ST_ROWS;
        float* const tile_policy = policy + (long)tile * (ST_ROWS * a.n);
#pragma unroll
        for (int pass = 0; pass < 4; ++pass) {
            const int rr = 4 * pass + hq;
            f32x4 v = *reinterpret_cast<const f32x4*>(scratch + rr * 256 + ((lq ^ rr) & 15) * 16);
            float p[4];
            stack_head<REGRET>(v, lq, limit, p);
            const bool row_ok = rr < rows_here;
            if (row_ok && 4 * lq < a.n)
                store16_through(reinterpret_cast<f32x4*>(tile_policy + rr * a.n + 4 * lq), f32x4{p[0], p[1], p[2], p[3]});
            if (a.action != nullptr) {
                const int pick = stack_pick(p, lq, __shfl(u4, rr + 16 * (turn & 3)));
                if (row_ok && lq == 0) action[tile * ST_ROWS + rr] = pick;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ---- few rows: the waves of a workgroup share a layer's features ------------------------------------------------------------------
// Where there is a tile of 16 rows per unit or two, latency is all there is: the chain of loads, products and barriers behind a row,
// and the instructions themselves, which a launch fetches cold at about a byte a cycle.  A workgroup takes R x 16 rows of one member;
// wave w computes the tiles w, w + waves, ... of 16 features of every layer, each in one rolled loop over units of 32 K-values whose
// weights it streams through a ring of its own, and the activations cross LDS (a barrier a layer; one more where rows are normalised,
// by the waves of the row tiles).  Inputs, uniforms and as many weights as the ring holds are asked for at once; the draws run
// meanwhile.  Every sum, norm and head has the operations and the order of the kernel above.
// LDS: [two buffers of activations][uniforms][a wave's ring].  A buffer is `planes` planes of 64 columns; row r of a plane is 256 bytes,
// its 16-byte piece p in slot p ^ (r & 15), and so are the rows of logits.  A unit is 16 rows of 128 bytes, piece p of row i in slot
// p ^ 2 ((i >> 1) & 3): no bank conflicts in either (16 lanes of a ds_read_b128: rows 0-3 and 12-15 of one lane group with rows 4-11
// of the next).
constexpr int SF_UNIT = 2048, SF_UNIFORMS = 2048, SF_MAX_THREADS = 512, SF_SLOTS = 16;

template <int R, bool REGRET>
__global__ __launch_bounds__(SF_MAX_THREADS) void stack_features_kernel(const float* x_first, const float* w0_first, const float* w1_first,
                                                                        const float* w2_first, unsigned long long widths, int batch, unsigned counts,
                                                                        int slots, unsigned acts, const StackArgs a) {
    constexpr int PLANE = R * ST_ROWS * 256;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int e = blockIdx.y;
    const int NL = (int)(counts & 15u), N = (int)(counts >> 4 & 0xffu), waves = (int)(counts >> 12 & 15u), planes = (int)(counts >> 16 & 3u), n = (int)(counts >> 18);
    const int acts_bytes = planes * PLANE;
    const int row0 = blockIdx.x * (ST_ROWS * R);
    const unsigned lds0 = (unsigned)(size_t)lds;
    auto width = [&](int l) { return (int)((unsigned)(widths >> (8 * l)) & 0xffu) << 2; };
    auto outputs_of = [&](int l) { return l + 1 < NL ? width(l + 1) : N; };
    const int K0 = width(0);

    // ---- inputs: four rows of a plane per instruction, zeros past the batch and past K0 ----
#pragma unroll 1
    for (int b = wave; b < (K0 > 64 ? 8 * R : 4 * R); b += waves) {
        const int plane = b >= 4 * R ? 1 : 0, row = 4 * (b - plane * 4 * R) + (lane >> 4);
        const int col = 4 * (16 * plane + ((lane & 15) ^ (row & 15)));
        const bool inside = row0 + row < batch && col < K0;
        const unsigned char* at = (const unsigned char*)(x_first + (long)(row0 + row) * K0 + col);
        dma_to_lds_addr(inside ? at : (const unsigned char*)kZeroChunk, lds0 + b * 1024);
    }
    // the head's rows: with one row tile four waves take four rows each, else wave w the rows of tile w
    const int head_tile = R == 1 ? 0 : wave;
    const bool head_wave = R == 1 ? wave < 4 : wave < R;
    const int my_row = row0 + ST_ROWS * head_tile + r;
    const bool explicit_u = a.action != nullptr && a.ph.philox_mode < 0;
    if (explicit_u && head_wave) {
        const float* at = a.u + (long)e * batch + (my_row < batch ? my_row : batch - 1);
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(at), "s"(lds0 + 2 * acts_bytes + wave * 256) : "memory", "m0");
    }

    // ---- the stream of this wave's weights ----
    const int ring_bytes = slots * SF_UNIT, ring_at = 2 * acts_bytes + SF_UNIFORMS + wave * ring_bytes;
    const int r8 = lane >> 3, piece = (lane & 7) ^ (((r8 >> 1) & 3) << 1);
    int f_layer = 0, f_tile = wave, f_k = 0, f_slot = 0, issued = 0;
    auto member_of = [&](int l) { return (long)e * (width(l) * (l + 1 < NL ? width(l + 1) : n)); };
    const float* f_base = w0_first + member_of(0);
    auto next_unit = [&]() {                            // (layer, tile) to fetch from, past the layers that have none for this wave
        while (f_layer < NL && 16 * f_tile >= outputs_of(f_layer)) {
            ++f_layer;
            f_tile = wave;
            f_base = (f_layer == 1 ? w1_first : f_layer == 2 ? w2_first : a.w[f_layer & (ST_MAX_LAYERS - 1)]) + member_of(f_layer);
        }
    };
    next_unit();
    auto issue_unit = [&]() {
        const int K = width(f_layer), F = outputs_of(f_layer);
        const int k = f_k + 4 * piece, row = 16 * f_tile + r8;
        const unsigned char* at = (const unsigned char*)(f_base + (long)row * K + k);
        const bool k_inside = k < K;
        dma_to_lds_addr(k_inside && row < F ? at : (const unsigned char*)kZeroChunk, lds0 + ring_at + f_slot);
        dma_to_lds_addr(k_inside && row + 8 < F ? at + 32l * K : (const unsigned char*)kZeroChunk, lds0 + ring_at + f_slot + 1024);
        f_slot = f_slot + SF_UNIT == ring_bytes ? 0 : f_slot + SF_UNIT;
        ++issued;
        f_k += 32;
        if (f_k >= K) {
            f_k = 0;
            f_tile += waves;
            next_unit();
        }
    };
    int x_at[4], w_at[2];                               // the 16 wide blocks of a plane, and of a unit
#pragma unroll
    for (int b = 0; b < 4; ++b) x_at[b] = r * 256 + (((4 * b + q) ^ r) << 4);
#pragma unroll
    for (int b = 0; b < 2; ++b) w_at[b] = ring_at + r * 128 + (((4 * b + q) ^ (((r >> 1) & 3) << 1)) << 4);
    // all slots but two: those behind the units being multiplied are filled next, under their products
#pragma unroll 1
    for (int s = 2; s < slots && f_layer < NL; ++s) issue_unit();
    float uniform = 1.f;
    if (a.action != nullptr && head_wave && a.ph.philox_mode >= 0) {
        const int row = my_row < batch ? my_row : batch - 1;
        if (a.ph.member_rows > 0) uniform = run_row_uniform<unsigned>(a.ph, row, a.ph.draw_offset + (unsigned long long)e * a.ph.member_draws);
        else uniform = run_row_uniform<unsigned>(a.ph, (unsigned)e * batch + row, a.ph.draw_offset);
    }
    // the oldest loads first: at most `young` units that were asked for later may be outstanding
    auto wait_units = [&](int young) {
        if (young >= 12) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
        else if (young >= 6) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
        else if (young >= 3) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        else if (young >= 1) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    wait_units(issued);                                 // this wave's inputs have landed
    asm volatile("s_barrier" ::: "memory");

    int buffer = 0, c_slot = 0, consumed = 0;
#pragma unroll 1
    for (int layer = 0; layer < NL; ++layer) {
        const int K = width(layer), F = outputs_of(layer);
        const unsigned act = acts >> (4 * layer) & 15u;
        const int map = (int)(act & 3u);              // of the last layer: none
        auto mapped = [&](f32x4& y) {
            if (map == SP_MAP_RELU) {
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = fmaxf(y[i], 0.f);
            } else if (map != SP_MAP_COPY) {
#pragma unroll 1
                for (int i = 0; i < 4; ++i) {            // (rolled: one copy of the function)
                    float v = y[0];
                    if (map == SP_MAP_TANH) v = tanhf(v);
                    else v = 1.f / (1.f + expf(-v));
                    y = f32x4{y[1], y[2], y[3], v};
                }
            }
        };
        const int to = acts_bytes - buffer;             // the other buffer
#pragma unroll 1
        for (int t = wave; 16 * t < F; t += waves) {
            f32x4 y[R];
#pragma unroll
            for (int rt = 0; rt < R; ++rt) y[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int k = 0; k < K; k += 64) {
                const int units = k + 32 < K ? 2 : 1;
                wait_units(issued - consumed - units);
                const unsigned char* const acts_at = lds + buffer + (k >> 6) * PLANE;
                f32x4 x[4][R], w[4];
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    if (b < 2 || units == 2) {
                        w[b] = *reinterpret_cast<const f32x4*>(lds + w_at[b & 1] + c_slot);
                        if (b & 1) c_slot = c_slot + SF_UNIT == ring_bytes ? 0 : c_slot + SF_UNIT;
#pragma unroll
                        for (int rt = 0; rt < R; ++rt) x[b][rt] = *reinterpret_cast<const f32x4*>(acts_at + x_at[b] + rt * 4096);
                    }
                consumed += units;
                for (int u = 0; u < units && f_layer < NL; ++u) issue_unit();      // into the slots of the units before these
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    if (k + 16 * b < K)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int rt = 0; rt < R; ++rt) y[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][i], x[b][rt][i], y[rt], 0, 0, 0);
            }
            // lane (r, q): features 16 t + 4 q .. + 3 of batch row r
            const int at = to + (t >> 2) * PLANE + r * 256 + (((4 * (t & 3) + q) ^ r) << 4);
#pragma unroll
            for (int rt = 0; rt < R; ++rt) {
                if (!(act & 8u)) mapped(y[rt]);
                *reinterpret_cast<f32x4*>(lds + at + rt * 4096) = y[rt];
            }
        }
        buffer = to;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (act & 8u) {                                  // local_ln_l2 (ml/primitives.spi:701-703) of the rows of tile `wave`
            if (wave < R) {
                unsigned char* const rows = lds + buffer + wave * 4096;
                f32x4 y[ST_MAX_WIDTH / 16];
                float s0 = 0.f, s1 = 0.f;
#pragma unroll
                for (int t = 0; t < ST_MAX_WIDTH / 16; ++t)
                    if (16 * t < F) y[t] = *reinterpret_cast<const f32x4*>(rows + (t >> 2) * PLANE + x_at[t & 3]);
#pragma unroll
                for (int t = 0; t < ST_MAX_WIDTH / 16; ++t)
                    if (16 * t < F) {
                        s0 = __builtin_fmaf(y[t][0], y[t][0], s0);
                        s1 = __builtin_fmaf(y[t][1], y[t][1], s1);
                        s0 = __builtin_fmaf(y[t][2], y[t][2], s0);
                        s1 = __builtin_fmaf(y[t][3], y[t][3], s1);
                    }
                float s = s0 + s1;
                s += __shfl_xor(s, 16);
                s += __shfl_xor(s, 32);
                const RowDivisor over_s(s);
#pragma unroll
                for (int t = 0; t < ST_MAX_WIDTH / 16; ++t)
                    if (16 * t < F) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) y[t][i] = s != 0.f ? over_s(y[t][i]) : 0.f;
                        mapped(y[t]);
                        *reinterpret_cast<f32x4*>(rows + (t >> 2) * PLANE + x_at[t & 3]) = y[t];
                    }
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    }
    if (!head_wave) return;
    if (explicit_u) uniform = *reinterpret_cast<const float*>(lds + 2 * acts_bytes + wave * 256 + lane * 4);

    // ---- the head and the sampling, four rows at a time: lane l of 16 holds columns 4 l .. of its row, as in the row primitives ----
    const int limit = a.mask_size;
    const unsigned char* const logits = lds + buffer + head_tile * 4096;
    float* const policy = a.policy + (long)e * batch * n;
#pragma unroll 1
    for (int pass = R == 1 ? wave : 0; pass < (R == 1 ? wave + 1 : 4); ++pass) {
        const int rr = 4 * pass + q, row = row0 + ST_ROWS * head_tile + rr;
        f32x4 v = *reinterpret_cast<const f32x4*>(logits + rr * 256 + ((r ^ rr) & 15) * 16);
        float p[4];
        stack_head<REGRET>(v, r, limit, p);
        const bool row_ok = row < batch;
        if (row_ok && 4 * r < n) store16_through(reinterpret_cast<f32x4*>(policy + (long)row * n + 4 * r), f32x4{p[0], p[1], p[2], p[3]});
        if (a.action != nullptr) {
            const int pick = stack_pick(p, r, __shfl(uniform, rr));
            if (row_ok && r == 0) a.action[(long)e * batch + row] = pick;
        }
    }
}

}  // namespace sp

using namespace sp;

template <int HT, bool FULL, bool PARTS = false>
static const void* pick_stack_kernel(bool regret) {
    return regret ? (const void*)mlp_stack_kernel<HT, true, FULL, PARTS> : (const void*)mlp_stack_kernel<HT, false, FULL, PARTS>;
}

// Bytes of LDS the weights take; computed: the outputs that a mask leaves.
static long stack_weight_bytes(int n_layers, const int32_t* dims, int computed) {
    long blocks = 0;
    for (int l = 0; l < n_layers; ++l) blocks += (long)((dims[l] + 15) / 16) * (((l + 1 < n_layers ? dims[l + 1] : computed) + 15) / 16);
    return blocks * ST_BLOCK;
}

// The sizes and the head of a call: what sp_stack_forward_takes answers for and sp_stack_forward_f32 checks.
static bool head_is_masked(int head_op) { return head_op == SP_ROW_MASKED_SOFTMAX || head_op == SP_ROW_MASKED_REGRET_MATCHING; }
static bool head_is_regret(int head_op) { return head_op == SP_ROW_REGRET_MATCHING || head_op == SP_ROW_MASKED_REGRET_MATCHING; }
static int check_stack_sizes(const char* fn, int n_layers, const int32_t* dims, int members, int64_t batch, int head_op, int mask_size) {
    if (n_layers < 1 || n_layers > ST_MAX_LAYERS) return fail(SP_ERR_SHAPE, "%s: 1 to %d layers, got %d", fn, ST_MAX_LAYERS, n_layers);
    if (members <= 0 || members > 65535) return fail(SP_ERR_SHAPE, "%s: members must be in [1, 65535]", fn);
    if (batch <= 0 || batch >= (1ll << 31) / members - ST_ROWS) return fail(SP_ERR_SHAPE, "%s: batch must be positive and members x batch below 2^31", fn);
    if (!head_is_regret(head_op) && head_op != SP_ROW_SOFTMAX && head_op != SP_ROW_MASKED_SOFTMAX) return fail(SP_ERR_ARG, "%s: unknown head %d", fn, head_op);
    const int n = dims[n_layers];
    if (dims[0] < 4 || dims[0] % 4 != 0 || dims[0] > ST_MAX_WIDTH)
        return fail(SP_ERR_SHAPE, "%s: input width %d must be a multiple of 4 in [4, %d]", fn, dims[0], ST_MAX_WIDTH);
    for (int l = 1; l < n_layers; ++l)
        if (dims[l] < 16 || dims[l] % 16 != 0 || dims[l] > ST_MAX_WIDTH)
            return fail(SP_ERR_SHAPE, "%s: hidden width %d must be a multiple of 16 in [16, %d]", fn, dims[l], ST_MAX_WIDTH);
    if (n < 4 || n % 4 != 0 || n > ST_MAX_OUT)
        return fail(SP_ERR_SHAPE, "%s: output width %d must be a multiple of 4 in [4, %d]", fn, n, ST_MAX_OUT);
    if (head_is_masked(head_op) && (mask_size <= 0 || mask_size > n)) return fail(SP_ERR_ARG, "%s: mask_size must be in [1, %d], got %d", fn, n, mask_size);
    const long w_bytes = stack_weight_bytes(n_layers, dims, head_is_masked(head_op) ? mask_size : n);
    if (w_bytes > ST_LDS - 4 * ST_SCRATCH) return fail(SP_ERR_UNSUPPORTED, "%s: %ld bytes of weights exceed the LDS", fn, w_bytes);
    return SP_OK;
}

extern "C" int sp_stack_forward_takes(int32_t n_layers, const int32_t* dims, int32_t members, int64_t batch, int32_t head_op, int32_t mask_size) {
    if (dims == nullptr) return fail(SP_ERR_NULL, "sp_stack_forward_takes: dims is NULL");
    return check_stack_sizes(__func__, n_layers, dims, members, batch, head_op, mask_size);
}

// Reference role: the body of `graph_run_host model` (ml/layers.spi:336-344) for the chains named at the top.
extern "C" int sp_stack_forward_f32(const void* x, int32_t n_layers, const void* const* weights, const int32_t* dims,
                                    const int32_t* acts, int32_t members, const float* u, const sp_philox_t* philox,
                                    float* policy_out, int32_t* action_out, int64_t batch, int32_t head_op, int32_t mask_size,
                                    void* stream) {
    SP_REQUIRE_PTR(x);
    SP_REQUIRE_PTR(policy_out);
    SP_OPTIONAL_PTR(u); SP_OPTIONAL_PTR(action_out);
    if (weights == nullptr || dims == nullptr || (acts == nullptr && n_layers != 1)) return fail(SP_ERR_NULL, "sp_stack_forward_f32: weights/dims/acts is NULL");
    int rc = check_stack_sizes(__func__, n_layers, dims, members, batch, head_op, mask_size);
    if (rc != SP_OK) return rc;
    if (action_out != nullptr && u == nullptr && philox == nullptr)
        return fail(SP_ERR_NULL, "sp_stack_forward_f32: action requested but u and philox are NULL");
    if (u != nullptr && philox != nullptr) return fail(SP_ERR_ARG, "sp_stack_forward_f32: at most one of u and philox may be given");
    const int n = dims[n_layers];
    const bool masked = head_is_masked(head_op), regret = head_is_regret(head_op);
    StackArgs a{};
    int widest = 0;
    for (int l = 0; l < n_layers; ++l) {
        if (weights[l] == nullptr) return fail(SP_ERR_NULL, "sp_stack_forward_f32: weights[%d] is NULL", l);
        if (!aligned16(weights[l])) return fail(SP_ERR_ALIGN, "sp_stack_forward_f32: weights[%d] is not 16-byte aligned", l);
        if (l + 1 < n_layers) {                            // (behind the last layer stands the head)
            const int map = acts[l] & ~SP_STACK_LN_L2;
            if (map != SP_MAP_COPY && map != SP_MAP_RELU && map != SP_MAP_TANH && map != SP_MAP_SIGMOID)
                return fail(SP_ERR_ARG, "sp_stack_forward_f32: unknown activation %d of layer %d", acts[l], l);
            a.acts[l] = acts[l];
        }
        a.w[l] = (const float*)weights[l];
        a.dims[l] = dims[l];
        const unsigned kt = (unsigned)(dims[l] + 15) / 16;
        a.per_kt[l] = (65536 + kt - 1) / kt;
        if (dims[l] > widest) widest = dims[l];
    }
    a.ph.philox_mode = -1;
    rc = mlp_set_philox(a.ph, philox, (int64_t)members * batch, n, __func__);
    if (rc != SP_OK) return rc;
    if (philox != nullptr && philox->member_rows > 0 && philox->member_rows != batch)
        return fail(SP_ERR_ARG, "sp_stack_forward_f32: member_rows must be the batch");
    a.mask_size = masked ? mask_size : n;
    a.dims[n_layers] = a.mask_size;
    a.out_stride = (long)n * dims[n_layers - 1];
    long w_bytes = stack_weight_bytes(n_layers, dims, a.mask_size);
    rc = require_gfx950(__func__);
    if (rc != SP_OK) return rc;
    a.x = (const float*)x; a.u = u; a.policy = policy_out; a.action = action_out;
    a.n_layers = n_layers; a.n = n; a.batch = (int)batch;
    a.tiles = (int)((batch + ST_ROWS - 1) / ST_ROWS);
    const int ht = widest <= 64 ? 4 : 8;
    const long cus = device_cu_count(), tiles = (long)a.tiles * members;
    {
        // A tile of rows per unit at most: the waves share its features; two where layers are wider than 64, as they leave the other kernel
        // one workgroup a unit.  Us of a captured launch, that kernel / so: 108-64-32 48 rows 9.7 / 6.9, 124-64-32 tanh 1680 rows 10.9 / 6.8,
        // 4-16-4 48 rows 5.7 / 4.5, 64-64-64-64 ln_l2 relu 4096 rows 10.3 / 8.5, 128-128-64 48 rows x 4 13.6 / 7.2, 4096 rows 14.0 / 8.9;
        // two tiles: 128-128-64 8192 rows 14.1 / 10.3, 128-96-64 12.6 / 10.0, 80-128-64 tanh 6656 rows 15.3 / 10.3, but 64-64-64-64
        // 10.5 / 10.9, 100-16-32 7.7 / 7.8; four tiles 64-64-64-64 16384 rows 10.8 / 12.9.
        const int rt = tiles <= cus ? 1 : tiles <= 2 * cus && widest > 64 ? 2 : 0;
        if (rt > 0) {
            unsigned long long widths = 0;
            int most_tiles = (a.mask_size + 15) / 16, units = 0;
            for (int l = 0; l < n_layers; ++l) {
                widths |= (unsigned long long)(dims[l] / 4) << (8 * l);
                if (l > 0 && dims[l] / 16 > most_tiles) most_tiles = dims[l] / 16;
            }
            const int waves = most_tiles < 4 ? 4 : most_tiles > 8 ? 8 : most_tiles;
            for (int l = 0; l < n_layers; ++l) units += (dims[l] + 31) / 32 * ((((l + 1 < n_layers ? dims[l + 1] : a.mask_size) + 15) / 16 + waves - 1) / waves);
            const int planes = widest > 64 ? 2 : 1, ring_at = 2 * planes * rt * ST_ROWS * 256 + SF_UNIFORMS;
            int slots = (ST_LDS - ring_at) / (waves * SF_UNIT);
            slots = slots < SF_SLOTS ? slots : SF_SLOTS;
            slots = units + 2 < slots ? units + 2 : slots;
            unsigned counts = (unsigned)n_layers | (unsigned)a.mask_size << 4 | (unsigned)waves << 12 | (unsigned)planes << 16 | (unsigned)n << 18, acts_bits = 0;
            for (int l = 0; l + 1 < n_layers; ++l) acts_bits |= (unsigned)((acts[l] & 3) | (acts[l] & SP_STACK_LN_L2 ? 8 : 0)) << (4 * l);
            const void* kernel = rt == 1 ? (regret ? (const void*)stack_features_kernel<1, true> : (const void*)stack_features_kernel<1, false>)
                                         : (regret ? (const void*)stack_features_kernel<2, true> : (const void*)stack_features_kernel<2, false>);
            rc = ensure_dynamic_lds(kernel, ST_LDS);
            if (rc != SP_OK) return rc;
            const float *x_first = a.x, *w0 = a.w[0], *w1 = a.w[n_layers > 1 ? 1 : 0], *w2 = a.w[n_layers > 2 ? 2 : 0];
            void* args[] = {(void*)&x_first, (void*)&w0, (void*)&w1, (void*)&w2, (void*)&widths, (void*)&a.batch, (void*)&counts, (void*)&slots, (void*)&acts_bits, (void*)&a};
            const hipError_t err = hipLaunchKernel(kernel, dim3((unsigned)((a.tiles + rt - 1) / rt), (unsigned)members), dim3(64 * waves), args,
                                                   ring_at + waves * slots * SF_UNIT, (hipStream_t)stream);
            if (err != hipSuccess) return fail(SP_ERR_DEVICE, "sp_stack_forward_f32: launch failed: %s", hipGetErrorString(err));
            return check_launch(__func__);
        }
    }
    bool full = true;
    for (int l = 0; l < n_layers; ++l) full = full && (dims[l] + 15) / 16 == ht;
    // workgroups of a member, tiles of a wave (no more workgroups than give those), rounds of workgroups
    struct Launch { long gx, each, rounds; };
    auto launch_of = [&](long gx, long waves, long at_once) {
        const long most = (a.tiles + waves - 1) / waves;
        if (gx > most) gx = most;
        const long each = (a.tiles + gx * waves - 1) / (gx * waves);
        gx = (a.tiles + each * waves - 1) / (each * waves);
        return Launch{gx, each, (members * gx + at_once - 1) / at_once};
    };
    // Four waves a workgroup while that is one tile per SIMD; beyond it eight, so that one wave's norms and head run beside
    // another's products, and as many workgroups per unit as the LDS holds (at most two).
    int waves = tiles > 4 * cus && w_bytes + 8 * ST_SCRATCH <= ST_LDS ? 8 : 4;
    int lds_bytes = (int)w_bytes + waves * ST_SCRATCH;
    const int resident = 2 * lds_bytes <= ST_LDS ? 2 : 1;
    Launch at = launch_of((cus * resident + members - 1) / members, waves, cus * resident);
    // Full 64 wide stacks in bf16 parts, sixteen waves in one workgroup per unit, a member's, from a tile for every wave of every unit
    // up (one layer: two, its product is less of the work).  Splitting the weights takes a few us a workgroup: with more members than
    // units each has two tiles a wave at least.  A turn of the unit's sixteen waves takes 1.5 to 1.8 times one of eight in f32 (four
    // layers less, their f32 weights leave room for one workgroup a unit); so either seven tenths of the turns of all rounds have a
    // tile, or f32 has 2.2 times the turns, 2 if both have one round of workgroups (f32's last round gets by with less).  Of 800 calls
    // of 1 to 600 members, one to four layers, with and without ln_l2, none that this takes is slower than in f32.  Us, f32 / parts,
    // 64-64-64-64: 65536 rows 21.5 / 18.9, 131072 37.0 / 31.2, 16 members of 16384 70 / 57, of 57344 231 / 187, 512 of 1000 127 /
    // 111; 64-64-64: 65536 rows 16.5 / 15.7, 131072 27.4 / 24.7, 200 members of 2000 96 / 74, but 300 of 762 54.7 / 62.5, 129 of 2000
    // 71 / 73; 64-64: 131072 rows 18.7 / 17.7, 4 members of 50000 32.5 / 28.8.
    constexpr int PARTS_WAVES = ST_PARTS_THREADS / 64;
    const long w_parts = (long)n_layers * 8 * ST_PARTS_UNIT;
    const Launch at_parts = launch_of(cus < members ? 1 : cus / members, PARTS_WAVES, cus);
    const long turns = at_parts.rounds * at_parts.each, turns_f32 = at.rounds * at.each * (waves * resident / 8);
    const bool parts = full && ht == 4 && (a.mask_size + 15) / 16 == 4 && w_parts + PARTS_WAVES * ST_SCRATCH <= ST_LDS &&
                       tiles >= (n_layers > 1 ? 1 : 2) * PARTS_WAVES * cus && (members <= cus || a.tiles >= 2 * PARTS_WAVES) &&
                       (n_layers == 4 || 10 * tiles >= 7 * turns * PARTS_WAVES * cus || 5 * turns_f32 >= 11 * turns ||
                        (at.rounds == 1 && at_parts.rounds == 1 && turns_f32 >= 2 * turns));
    if (parts) {
        w_bytes = w_parts;
        waves = PARTS_WAVES;
        lds_bytes = (int)w_bytes + waves * ST_SCRATCH;
        at = at_parts;
    }
    a.w_bytes = (int)w_bytes;
    const void* kernel = parts ? pick_stack_kernel<4, true, true>(regret)
                       : ht == 4 ? (full ? pick_stack_kernel<4, true>(regret) : pick_stack_kernel<4, false>(regret))
                                 : (full ? pick_stack_kernel<8, true>(regret) : pick_stack_kernel<8, false>(regret));
    rc = ensure_dynamic_lds(kernel, ST_LDS);
    if (rc != SP_OK) return rc;
    void* args[] = {(void*)&a};
    const hipError_t err = hipLaunchKernel(kernel, dim3((unsigned)at.gx, (unsigned)members), dim3(64 * waves), args, lds_bytes, (hipStream_t)stream);
    if (err != hipSuccess) return fail(SP_ERR_DEVICE, "sp_stack_forward_f32: launch failed: %s", hipGetErrorString(err));
    return check_launch(__func__);
}

namespace {
struct MlpStackKernelNames {
    MlpStackKernelNames() {
        register_kernel("stack_forward_f32_few", (const void*)stack_features_kernel<1, false>, SF_MAX_THREADS);
        register_kernel("stack_forward_f32_few_regret", (const void*)stack_features_kernel<1, true>, SF_MAX_THREADS);
        register_kernel("stack_forward_f32_few_2", (const void*)stack_features_kernel<2, false>, SF_MAX_THREADS);
        register_kernel("stack_forward_f32", (const void*)mlp_stack_kernel<4, false, true>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_regret", (const void*)mlp_stack_kernel<4, true, true>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_parts", (const void*)mlp_stack_kernel<4, false, true, true>, ST_PARTS_THREADS);
        register_kernel("stack_forward_f32_parts_regret", (const void*)mlp_stack_kernel<4, true, true, true>, ST_PARTS_THREADS);
        register_kernel("stack_forward_f32_part", (const void*)mlp_stack_kernel<4, false, false>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_part_regret", (const void*)mlp_stack_kernel<4, true, false>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_128", (const void*)mlp_stack_kernel<8, false, true>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_128_regret", (const void*)mlp_stack_kernel<8, true, true>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_128_part", (const void*)mlp_stack_kernel<8, false, false>, ST_MAX_THREADS);
        register_kernel("stack_forward_f32_128_part_regret", (const void*)mlp_stack_kernel<8, true, false>, ST_MAX_THREADS);
    }
} mlp_stack_kernel_names;
}  // namespace
