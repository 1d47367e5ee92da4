// Fused forward of 16-bit stacks of any hidden width (multiples of 32 up to 256) under any head of up to 64 outputs: the stacks
// that the kernels for 256 wide layers and narrow heads (mlp.hip, mlp_packed.hip, mlp_resident.hip, mlp_pipe.hip) do not take.
//
// Three kernels, by how much work there is: up to 64 rows per compute unit the first, beyond that the second (beyond 128 where the weights
// exceed the LDS; the third up to there).  bf16, us of a captured launch, first / second: 64-128-128-4 4096 rows 5.5 / 8.1, 16384 6.4 / 8.3, 65536 21 / 8.7;
// 192-96-64-64 masked to 3, 10061 rows 7.1 / 11.3; 64-192-192-192-4 16384 rows 10.2 / 19, 65536 35 / 20.
//   mlp_features_kernel: a workgroup of eight or sixteen waves takes R x 16 rows through the stack.  The waves share out a layer's tiles of 16
// output features; each streams the weights of its own features through a ring in LDS that nobody else reads, so weights need no
// barrier, and the activations cross LDS between layers (one barrier a layer, two buffers).  The last layer and the head of row
// tile w are wave w's.  Everything comes in by DMA: inputs, uniforms and as many weights as the ring holds are asked for in the
// first few hundred cycles, and a step waits for its own weights alone.  This is the form for few rows, where latency is all
// there is.
//   mlp_rows_kernel: all weights of the stack in LDS, loaded once per workgroup; a wave takes 32 rows at a time through the stack
// with the activations in its registers, no barrier behind the first.  Weights that do not fit stream through a ring, for all waves alike.
// Workgroups of four waves up to 128 rows per compute unit, so that twice as many units have one (us, eight waves / four: 256-256-16 24620
// rows 20.0 / 16.6, 128-64-64 masked to 3 9.2 / 8.3, 64-192-24 11.0 / 10.1, 32-64-64-64-10 11.0 / 10.6).
//   mlp_round_kernel: from 64 to 128 rows per compute unit what does not fit, under up to 32 outputs, and some short stacks.
//
// Against one kernel of 16 rows a wave with all weights through a ring (us, before / now): 128-64-64 masked to 3, 64 rows 8.9 / 4.2;
// 80-192-192-192-24, 115 rows 19.4 / 9.4; 80-128-128-128-64-4, 614 rows 16.3 / 7.5; 64-128-128-64, 4096 rows 17.5 / 7.6; 64-128-128-4,
// 65536 rows 20.5 / 8.7 and 400000 120 / 40; 256-64-64-64-128-64, 178588 rows 147 / 64; 64-192-192-192-4, 65536 rows 32 / 20;
// 128-192-192-192-192-4, 400000 rows 267 / 181; 128-64-64 masked to 3, 524288 rows 133 / 78 (3.5 TB/s).
//
// Both multiply with v_mfma_f32_16x16x32, weights first, k-steps of 32 in ascending order, lane group q holding k = 32 s + 8 q ..
// + 7: an output's products add up in the same order in both, and in every other kernel of these stacks.
#include "mlp_common.h"
#include "gemm_dma.h"

#pragma clang fp contract(off)

namespace sp {

constexpr int AN_UNIT = 2048;                  // 16 rows of weights x 64 of K
constexpr int AN_LDS = 160 * 1024;

// Widths of a stack in one scalar: byte l holds dims[l] / 16 of layer l's input.
__device__ __forceinline__ int any_width(unsigned long long widths, int l) { return (int)((unsigned)(widths >> (8 * l)) & 0xffu) << 4; }

template <int DT>
__device__ __forceinline__ f32x4 any_mfma(const u32x4& w, const u32x4& x, const f32x4& c) {
    if constexpr (DT == SP_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
}

// relu is max(0, x), a NaN becomes 0.  The matrix pipe's own NaNs have the sign set, whatever went in, and pack_relu2, which compares
// rounded values as integers, makes them 0; one that a bias brings may have it clear, so sums with a bias pass an f32 maximum first.  (That
// maximum for every sum costs 1 to 3 % without a bias: 64-192-192-192-4, 65536 rows.)  Stacks whose hidden layers are all 256 wide
// (AN_ALL_256, in the layer count that a kernel is given) do without, as in the kernels that take the others of them: there a bias that is
// a NaN stays one, and what a head of up to 16 outputs leaves past its mask are zeros, in a row of NaNs, too.
constexpr unsigned AN_ALL_256 = 0x80;
__device__ __forceinline__ float any_biased(float sum, float bias) {
    float r;
    asm("v_add_f32 %0, %1, %2" : "=v"(r) : "v"(sum), "v"(bias));       // (the sum first: of two NaNs it is the one that stays)
    return r;
}
__device__ __forceinline__ void any_max0(f32x4& v) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float m;
        asm("v_max_f32 %0, 0, %1" : "=v"(m) : "v"(v[r]));
        v[r] = m;
    }
}

// The last layer's outputs as the matrix pipe leaves them when the weight rows of a pair of tiles are fed in the order 32 u + 8 (i / 4)
// + i % 4 (even tile) and + 4 (odd tile): lane (j, q) holds columns 32 u + 8 q .. + 7 of batch row j.
//   The head of those 16 rows, all 64 lanes at work: the formulas and the order of every sum are head_row's (mlp_common.h) -- sums
// run through the columns one after the other, from lane group to lane group.  `n`: computed outputs; `stride`: the row's width, of
// which the columns from n on lie past the mask.
template <int P>
__device__ __forceinline__ float any_running_sum(const float (&p)[P][8], int n, int j, int q, float (*cdf)[8]) {
    float carry = 0.f;
#pragma unroll
    for (int u = 0; u < P; ++u) {
#pragma unroll 1
        for (int s = 0; s < 4; ++s) {
            if (32 * u + 8 * s >= n) break;                       // (uniform)
            float run = carry;
            if (cdf == nullptr) {
#pragma unroll
                for (int k = 0; k < 8; ++k) run = run + p[u][k];
            } else if (q == s) {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    run = run + p[u][k];
                    cdf[u][k] = run;
                }
            }
            carry = __shfl(run, j + 16 * s);
        }
    }
    return carry;
}

template <int P>
__device__ __forceinline__ void any_head(const HeadOut& o, const f32x4 (&v)[2 * P], long row, bool row_ok, int j, int q, int n, int limit, float uniform, bool all_256) {
    const float NEG_INF = -__builtin_inff();
    const int stride = o.stride;
    const bool whole = (stride & 3) == 0;
    float p[P][8], past = 0.f;                      // past: of the columns that no lane holds
    auto store_row = [&](float* out) {
        float* const at = out + row * stride;
        if (!row_ok) return;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int col = 32 * u + 8 * q + 4 * h;
                float4 piece = make_float4(past, past, past, past);
                if (u < P) piece = make_float4(p[u < P ? u : 0][4 * h], p[u < P ? u : 0][4 * h + 1], p[u < P ? u : 0][4 * h + 2], p[u < P ? u : 0][4 * h + 3]);
                if (whole) {
                    if (col < stride) *reinterpret_cast<float4*>(at + col) = piece;
                } else {
                    if (col < stride) at[col] = piece.x;
                    if (col + 1 < stride) at[col + 1] = piece.y;
                    if (col + 2 < stride) at[col + 2] = piece.z;
                    if (col + 3 < stride) at[col + 3] = piece.w;
                }
            }
    };
#pragma unroll
    for (int u = 0; u < P; ++u)
#pragma unroll
        for (int k = 0; k < 8; ++k) p[u][k] = 32 * u + 8 * q + k < n ? v[2 * u + (k >> 2)][k & 3] : 0.f;
    if (o.logits != nullptr) store_row(o.logits);      // (then n is the row's width)
    if (o.head == SP_HEAD_SOFTMAX || o.head == SP_HEAD_SOFTMAX_RM) {
        float m = NEG_INF;
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                p[u][k] = 32 * u + 8 * q + k < limit ? p[u][k] : NEG_INF;
                m = fmaxf(m, p[u][k]);
            }
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) p[u][k] = __builtin_amdgcn_exp2f((p[u][k] - m) * 1.44269504088896340736f);
        const float inv = __builtin_amdgcn_rcpf(any_running_sum<P>(p, n, j, q, nullptr));
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) p[u][k] = p[u][k] * inv;
        past = __builtin_amdgcn_exp2f((NEG_INF - m) * 1.44269504088896340736f) * inv;
    }
    if (o.head == SP_HEAD_REGRET_MATCHING || o.head == SP_HEAD_SOFTMAX_RM) {
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) p[u][k] = 32 * u + 8 * q + k < limit ? fmaxf(p[u][k], 0.f) : 0.f;
        const float s = any_running_sum<P>(p, n, j, q, nullptr);
        const float inv_len = __builtin_amdgcn_rcpf((float)limit);
        const float inv = s != 0.f ? __builtin_amdgcn_rcpf(s) : 0.f;
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) p[u][k] = s != 0.f ? p[u][k] * inv : (32 * u + 8 * q + k < limit ? inv_len : 0.f);
        past = 0.f * inv;
    }
    if (all_256 && n <= 16) {
        past = 0.f;
        int qz = q;
        asm volatile("" : "+v"(qz));                    // (comparisons of its own: those above would be kept for it, two registers each)
#pragma unroll
        for (int k = 0; k < 8; ++k) p[0][k] = 8 * qz + k < n ? p[0][k] : 0.f;
    }
    store_row(o.policy);
    if (o.action != nullptr) {
        float cdf[P][8];
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) cdf[u][k] = 0.f;
        any_running_sum<P>(p, n, j, q, cdf);
        float m = NEG_INF;
#pragma unroll
        for (int u = 0; u < P; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (p[u][k] > 0.f) m = fmaxf(m, cdf[u][k]);
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        const float thr = uniform * m;
        int pick = INT_MAX_;
#pragma unroll
        for (int u = P - 1; u >= 0; --u)
#pragma unroll
            for (int k = 7; k >= 0; --k)
                if (p[u][k] > 0.f && cdf[u][k] >= thr) pick = 32 * u + 8 * q + k;
        int other = __shfl_xor(pick, 16);
        pick = other < pick ? other : pick;
        other = __shfl_xor(pick, 32);
        pick = other < pick ? other : pick;
        if (row_ok && q == 0) o.action[row] = pick;
    }
}

// At most four outputs, all of them in every lane of a row: the same formulas.  store(out): the row's p and `past` behind it.
template <typename Store>
__device__ __forceinline__ void any_head4(const HeadOut& o, float (&p)[4], float& past, int n, int limit, bool all_256, const Store& store) {
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = k < n ? p[k] : 0.f;
    past = 0.f;
    if (o.logits != nullptr) store(o.logits);          // (then n is the row's width)
    if (o.head == SP_HEAD_SOFTMAX || o.head == SP_HEAD_SOFTMAX_RM) {
        float m = -__builtin_inff();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            p[k] = k < limit ? p[k] : -__builtin_inff();
            m = fmaxf(m, p[k]);
        }
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            p[k] = __builtin_amdgcn_exp2f((p[k] - m) * 1.44269504088896340736f);
            s = s + p[k];
        }
        const float inv = __builtin_amdgcn_rcpf(s);
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = p[k] * inv;
        past = __builtin_amdgcn_exp2f((-__builtin_inff() - m) * 1.44269504088896340736f) * inv;
    }
    if (o.head == SP_HEAD_REGRET_MATCHING || o.head == SP_HEAD_SOFTMAX_RM) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            p[k] = k < limit ? fmaxf(p[k], 0.f) : 0.f;
            s = s + p[k];
        }
        const float inv_len = __builtin_amdgcn_rcpf((float)limit);
        const float inv = s != 0.f ? __builtin_amdgcn_rcpf(s) : 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = s != 0.f ? p[k] * inv : (k < limit ? inv_len : 0.f);
        past = 0.f * inv;
    }
    if (all_256) past = 0.f;
    store(o.policy);
}

// ---- the waves share a layer's features -------------------------------------------------------------------------------------------
// What bounds it is latency: the chain of loads, products and barriers behind a row, and the instructions themselves, which a launch
// fetches cold at about a byte a cycle.  Hence one loop over units for every layer, the last among them, and nothing unrolled.
// LDS: [two buffers of activations][uniforms, 256 bytes a wave][a wave's ring of `slots` units].  A buffer of activations is two
// planes of 128 columns; row r of a plane is 256 bytes, its 16-byte piece p in slot p ^ (r & 15).  The last layer's outputs are rows of
// 64 floats in one of them, in the same way.  A unit is 16 rows of 64 K-values, 128 bytes each, piece p of row i in slot
// p ^ 2 ((i >> 1) & 3): both are read without bank conflicts (16 lanes of a ds_read_b128: rows 0-3 and 12-15 of one lane group with
// rows 4-11 of the next).
template <int R>
struct AnyFeatures {
    static constexpr int PLANE = R * 16 * 256, ACTS = 2 * PLANE, UNIFORMS_AT = 2 * ACTS, RING_AT = UNIFORMS_AT + 2048;
};
constexpr int AN_FEATURES_THREADS = 1024, AN_SLOTS = 16;

template <int DT, int R>
__global__ __launch_bounds__(AN_FEATURES_THREADS) void mlp_features_kernel(const void* x_first, const void* w0_first, const void* w1_first,
                                                                           unsigned long long widths, long batch, const float* u_first, unsigned counts,
                                                                           int slots, const MlpArgs a) {
    typedef AnyFeatures<R> L;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, q = lane >> 4;
    const bool all_256 = counts & AN_ALL_256;
    const int NL = (int)(counts & 0x7fu), N = (int)(counts >> 8 & 0xffu), waves = (int)(counts >> 16);
    const long row0 = (long)blockIdx.x * (16 * R);
    const unsigned lds0 = (unsigned)(size_t)lds;
    const int K0 = any_width(widths, 0);

    // ---- inputs: four rows of a plane per instruction, zeros past the batch and past K0 ----
#pragma unroll 1
    for (int b = wave; b < (K0 > 128 ? 8 * R : 4 * R); b += waves) {
        const int plane = b >= 4 * R ? 1 : 0, r = 4 * (b - plane * 4 * R) + (lane >> 4);
        const int col = 8 * (16 * plane + ((lane & 15) ^ (r & 15)));
        const bool inside = row0 + r < batch && col < K0;
        const unsigned char* at = (const unsigned char*)x_first + ((row0 + r) * K0 + col) * 2;
        dma_to_lds_addr(inside ? at : (const unsigned char*)kZeroChunk, lds0 + b * 1024);
    }
    const long my_row = row0 + 16 * wave + j;          // of the head
    if (u_first != nullptr && wave < R) {
        const float* at = u_first + (my_row < batch ? my_row : batch - 1);
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(at), "s"(lds0 + L::UNIFORMS_AT + wave * 256) : "memory", "m0");
    }

    // ---- the stream of this wave's weights: tiles wave, wave + waves, ... of 16 features of every layer, K inside ----
    auto outputs_of = [&](int l) { return l + 1 < NL ? any_width(widths, l + 1) : N; };
    const int r8 = lane >> 3, piece = (lane & 7) ^ (((r8 >> 1) & 3) << 1);
    const unsigned ring0 = lds0 + L::RING_AT + wave * slots * AN_UNIT;
    const int ring_bytes = slots * AN_UNIT;
    int f_layer = 0, f_tile = wave, f_k = 0, f_slot = 0, issued = 0;
    const unsigned char* f_base = (const unsigned char*)w0_first;
    auto next_unit = [&]() {                            // (layer, tile) to fetch from, past the layers that have none for this wave
        while (f_layer < NL && 16 * f_tile >= outputs_of(f_layer)) {
            ++f_layer;
            f_tile = wave;
            f_base = (const unsigned char*)(f_layer == 1 ? w1_first : a.w[f_layer & (MLP_MAX_LAYERS - 1)]);
        }
    };
    next_unit();
    auto issue_unit = [&]() {
        const int K = any_width(widths, f_layer), most = outputs_of(f_layer) - 1;
        int k = f_k + piece * 8, ra = 16 * f_tile + r8, rb = ra + 8;
        k = k <= K - 8 ? k : K - 8;                      // past K: meets zeros, or is not read
        ra = ra < most ? ra : most;                      // past the outputs: results that nobody reads
        rb = rb < most ? rb : most;
        mlp_dma(f_base, (unsigned)((ra * K + k) * 2), ring0 + f_slot);
        mlp_dma(f_base, (unsigned)((rb * K + k) * 2), ring0 + f_slot + 1024);
        f_slot = f_slot + AN_UNIT == ring_bytes ? 0 : f_slot + AN_UNIT;
        ++issued;
        f_k += 64;
        if (f_k >= K) {
            f_k = 0;
            f_tile += waves;
            next_unit();
        }
    };
    float uniform = 1.f;
    const HeadOut out = head_out(a);
    const int mask_size = a.mask_size, ph_mode = a.ph.philox_mode;
    int a_at[2], w_at[2];                                // fragments of the two k-steps of a unit
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        a_at[ks] = j * 256 + (((4 * ks + q) ^ j) << 4);
        w_at[ks] = L::RING_AT + wave * ring_bytes + j * 128 + (((4 * ks + q) ^ (((j >> 1) & 3) << 1)) << 4);
    }
    // all slots but one: the one behind the unit being multiplied is filled next, under its products
#pragma unroll 1
    for (int s = 1; s < slots && f_layer < NL; ++s) issue_unit();
    if (wave < R && ph_mode >= 0) uniform = reference_row_uniform(a.ph, my_row < batch ? my_row : 0);

    // the oldest loads first: at most `young` units that were asked for later may be outstanding
    auto wait_units = [&](int young) {
        if (young >= 12) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
        else if (young >= 6) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
        else if (young >= 3) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        else if (young >= 1) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    wait_units(issued);                                  // this wave's inputs have landed
    asm volatile("s_barrier" ::: "memory");
    int buffer = 0, c_slot = 0, consumed = 0;
#pragma unroll 1
    for (int layer = 0; layer < NL; ++layer) {
        const int K = any_width(widths, layer), F = outputs_of(layer);
        const bool last = layer + 1 == NL;
#pragma unroll 1
        for (int t = wave; 16 * t < F; t += waves) {
            f32x4 acc[R];
#pragma unroll
            for (int rt = 0; rt < R; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int k = 0; k < K; k += 64) {
                wait_units(issued - consumed - 1);
                const unsigned char* const acts = lds + buffer + (k >> 7) * L::PLANE;
                const int odd = (k & 64) << 1;
                u32x4 x[2][R], w[2];
                const bool two = k + 32 < K;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) w[ks] = *reinterpret_cast<const u32x4*>(lds + w_at[ks] + c_slot);
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int rt = 0; rt < R; ++rt) x[ks][rt] = *reinterpret_cast<const u32x4*>(acts + (a_at[ks] ^ odd) + rt * 4096);
                ++consumed;
                c_slot = c_slot + AN_UNIT == ring_bytes ? 0 : c_slot + AN_UNIT;
                if (f_layer < NL) issue_unit();          // into the slot of the unit before this one
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int rt = 0; rt < R; ++rt) acc[rt] = any_mfma<DT>(w[0], x[0][rt], acc[rt]);
                if (two)                                 // (else the second half of the unit lies past K)
#pragma unroll
                    for (int rt = 0; rt < R; ++rt) acc[rt] = any_mfma<DT>(w[1], x[1][rt], acc[rt]);
            }
            // lane (j, q): features 16 t + 4 q .. + 3 of batch row j
            const float* const bias = a.b[layer];
            if (bias != nullptr) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = 16 * t + 4 * q + r;
                    const float b = bias[n < F ? n : F - 1];
#pragma unroll
                    for (int rt = 0; rt < R; ++rt) acc[rt][r] = any_biased(acc[rt][r], b);
                }
                if (!last && !all_256)
#pragma unroll
                    for (int rt = 0; rt < R; ++rt) any_max0(acc[rt]);
            }
            unsigned char* const to = lds + (buffer ^ L::ACTS) + j * 256;
            if (!last) {
                const int at = (t >> 3) * L::PLANE + ((((2 * t & 15) + (q >> 1)) ^ j) << 4) + (q & 1) * 8;
#pragma unroll
                for (int rt = 0; rt < R; ++rt)
                    *reinterpret_cast<u32x2*>(to + at + rt * 4096) = u32x2{pack_relu2<DT>(acc[rt][0], acc[rt][1]), pack_relu2<DT>(acc[rt][2], acc[rt][3])};
            } else {
                const int at = ((4 * t + q) ^ j) << 4;
#pragma unroll
                for (int rt = 0; rt < R; ++rt) *reinterpret_cast<f32x4*>(to + at + rt * 4096) = acc[rt];
            }
        }
        buffer ^= L::ACTS;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if (wave >= R) return;
    const unsigned char* const rows = lds + buffer + (16 * wave + j) * 256;
    auto outputs = [&](int c) { return *reinterpret_cast<const f32x4*>(rows + ((c ^ j) << 4)); };       // columns 4 c .. + 3
    if (u_first != nullptr) uniform = *reinterpret_cast<const float*>(lds + L::UNIFORMS_AT + wave * 256 + lane * 4);
    const int limit = mask_size > 0 ? mask_size : N;
    const bool row_ok = my_row < batch;
    if (N <= 4) {
        const f32x4 v = outputs(0);
        float p[4] = {v[0], v[1], v[2], v[3]}, past;
        any_head4(out, p, past, N, limit, all_256, [&](float* to) {      // the four lanes of a row share its pieces
            const int stride = out.stride;
            float* const at = to + my_row * stride;
            if (!row_ok) return;
            if ((stride & 3) == 0) {
#pragma unroll 1
                for (int c = 4 * q; c < stride; c += 16)
                    *reinterpret_cast<float4*>(at + c) = c > 0 ? make_float4(past, past, past, past) : make_float4(p[0], N > 1 ? p[1] : past, N > 2 ? p[2] : past, N > 3 ? p[3] : past);
            } else {
#pragma unroll 1
                for (int c = q; c < stride; c += 4) at[c] = c < N ? (c == 0 ? p[0] : c == 1 ? p[1] : c == 2 ? p[2] : p[3]) : past;
            }
        });
        if (out.action != nullptr && row_ok && q == 0) out.action[my_row] = head_pick4(p, uniform);
    } else if (N <= 32) {
        const f32x4 v[2] = {outputs(2 * q), outputs(2 * q + 1)};
        any_head<1>(out, v, my_row, row_ok, j, q, N, limit, uniform, all_256);
    } else {
        const f32x4 v[4] = {outputs(2 * q), outputs(2 * q + 1), outputs(8 + 2 * q), outputs(9 + 2 * q)};
        any_head<2>(out, v, my_row, row_ok, j, q, N, limit, uniform, false);
    }
}

// ---- the waves share the rows -----------------------------------------------------------------------------------------------------
// What bounds it: the vector ALU and latency, of two waves per SIMD (their registers hold 32 rows of activations and sums): per 32 rows
// of 64-128-128-4 11 k cycles, of which the products take 6 k and the matrix pipe is busy for 1.9 k; under 64 outputs the head is half of it.
// (Three waves per SIMD spill: 256-64-64-64-128-64 64 -> 72 us; the next rows' inputs in registers of their own, too: 57 -> 70.)
// Weights in LDS in groups of 32 rows x 64 of K (4 KiB): 128-byte rows, piece p of row r in slot p ^ mlp_swz(r).  All of the stack's, once;
// or (STREAM), where they do not fit, a ring of four stages of one 64 wide step of K each, three steps ahead of the products and on
// into the next rows, one barrier a step.  HT: 16-wide tiles of the widest hidden layer (8 or 16).
constexpr int AN_GROUP = 4096, AN_ROWS = 32, AN_STAGE = 8 * AN_GROUP;

template <int DT, int HT, bool STREAM, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void mlp_rows_kernel(unsigned long long widths, unsigned counts, const MlpArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, q = lane >> 4;
    const bool all_256 = HT == 16 && (counts & AN_ALL_256);
    const int NL = (int)(counts & 0x7fu);
    const unsigned lds0 = (unsigned)(size_t)lds;
    const long tiles = (a.batch + AN_ROWS - 1) / AN_ROWS, step = (long)gridDim.x * WAVES;
    const int r8 = lane >> 3;
    int f_layer = 0, f_k = 0, f_stage = 0;                // the next step of K to fetch
    long f_tile = (long)blockIdx.x * WAVES;            // (of wave 0: the waves go through the same steps)
    // one 64 wide step of K of a layer, this wave's share of its 4 gn instructions; returns their number
    auto fetch_step = [&](unsigned at) {
        const int K = any_width(widths, f_layer), F = f_layer + 1 < NL ? any_width(widths, f_layer + 1) : (int)(counts >> 8);
        const unsigned char* const W = (const unsigned char*)a.w[f_layer];
        const int instructions = 4 * ((F + 31) >> 5);
        int count = 0;
        for (int b = wave; b < instructions; b += WAVES) {
            const int r = 8 * b + r8;                     // instruction b fetches rows 8 b .. + 7
            int k = 64 * f_k + 8 * ((lane & 7) ^ mlp_swz(r));
            k = k <= K - 8 ? k : K - 8;                   // past K: meets zeros, or is not read
            const int row = r < F ? r : F - 1;            // past the outputs: results that nobody reads
            mlp_dma(W, (unsigned)((row * K + k) * 2), at + b * 1024);
            ++count;
        }
        if (64 * ++f_k >= K) {
            f_k = 0;
            ++f_layer;
        }
        return count;
    };
    int ahead[3] = {0, 0, 0};                             // STREAM: instructions of this wave for the three steps in flight
    auto fetch_next = [&]() {
        ahead[0] = ahead[1];
        ahead[1] = ahead[2];
        ahead[2] = 0;
        if (f_tile >= tiles) return;
        ahead[2] = fetch_step(lds0 + f_stage * AN_STAGE);
        f_stage = (f_stage + 1) & 3;
        if (f_layer == NL) {
            f_layer = 0;
            f_tile += step;
        }
    };
    if constexpr (STREAM) {
        for (int i = 0; i < 3; ++i) fetch_next();
    } else {
        unsigned at = lds0;
        while (f_layer < NL) {
            const int F = f_layer + 1 < NL ? any_width(widths, f_layer + 1) : (int)(counts >> 8);
            fetch_step(at);
            at += ((F + 31) >> 5) * AN_GROUP;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    // lane j feeds weight row 8 (j / 4) + j % 4 of a group to the even tile and + 4 to the odd one
    const int n0 = 8 * (j >> 2) + (j & 3);
    int w_at[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) w_at[ks] = n0 * 128 + (((4 * ks + q) ^ mlp_swz(n0)) << 4);
    int stage = 0;
    const unsigned char* wp = lds;                        // the group being multiplied
    // A 64 wide step of K is about to be multiplied: it has landed, everywhere.
    auto begin_step = [&]() {
        if constexpr (STREAM) {
            const int young = ahead[1] + ahead[2];        // what may be outstanding was asked for later
            if (young >= 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
            else if (young >= 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
            else if (young >= 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else if (young >= 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
            else if (young >= 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else if (young >= 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            fetch_next();                                 // into the stage that every wave has read before this barrier
            wp = lds + stage * AN_STAGE;
            stage = (stage + 1) & 3;
        }
    };
    // acc[rt][t] = W . x for gn <= TILES / 2 pairs of tiles of features
    auto products = [&](int K, int gn, auto& acc, const auto& x, auto STEPS_, auto TILES_) {
        constexpr int STEPS = decltype(STEPS_)::value, TILES = decltype(TILES_)::value;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int t = 0; t < TILES; ++t) acc[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < STEPS; ++c)
            if (64 * c < K) {
                begin_step();
                const bool two = 64 * c + 32 < K;
#pragma unroll
                for (int u = 0; u < TILES / 2; ++u)
                    if (u < gn) {
                        u32x4 w[2][2];                    // [tile][k-step]
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                            for (int t = 0; t < 2; ++t) w[t][ks] = *reinterpret_cast<const u32x4*>(wp + w_at[ks] + t * 512);
                        wp += AN_GROUP;
#pragma unroll
                        for (int t = 0; t < 2; ++t)
#pragma unroll
                            for (int rt = 0; rt < 2; ++rt) acc[rt][2 * u + t] = any_mfma<DT>(w[t][0], x[rt][2 * c], acc[rt][2 * u + t]);
                        if (two)
#pragma unroll
                            for (int t = 0; t < 2; ++t)
#pragma unroll
                                for (int rt = 0; rt < 2; ++rt) acc[rt][2 * u + t] = any_mfma<DT>(w[t][1], x[rt][2 * c + 1], acc[rt][2 * u + t]);
                    }
            }
    };
    // At most four outputs: weight row i % 4 for row i of the product, so that every lane of a batch row gets all of them.
    const int r4 = j & 3;
    int w4_at[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) w4_at[ks] = r4 * 128 + (((4 * ks + q) ^ mlp_swz(r4)) << 4);
    auto products4 = [&](int K, f32x4 (&acc)[2][4], const auto& x, auto STEPS_) {
        constexpr int STEPS = decltype(STEPS_)::value;
        acc[0][0] = acc[1][0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < STEPS; ++c)
            if (64 * c < K) {
                begin_step();
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
                    if (ks == 0 || 64 * c + 32 < K) {
                        const u32x4 w = *reinterpret_cast<const u32x4*>(wp + w4_at[ks]);
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) acc[rt][0] = any_mfma<DT>(w, x[rt][2 * c + ks], acc[rt][0]);
                    }
                wp += AN_GROUP;
            }
    };
    auto load_inputs = [&](long tile, int K0, u32x4 (&x)[2][8]) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            long row = tile * AN_ROWS + 16 * rt + j;
            row = row < a.batch ? row : a.batch - 1;
            const unsigned char* const xr = (const unsigned char*)a.x + (row * K0 + 8 * q) * 2;
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (32 * s + 16 < K0) x[rt][s] = *reinterpret_cast<const u32x4*>(xr + 64 * s);
                else if (32 * s < K0) x[rt][s] = *reinterpret_cast<const u32x4*>(q < 2 ? xr + 64 * s : (const unsigned char*)kZeroChunk);     // K ends in mid-step: zeros
        }
    };
    for (long tile = (long)blockIdx.x * WAVES + wave; STREAM ? tile - wave < tiles : tile < tiles; tile += step) {
        int K0 = any_width(widths, 0), N = (int)(counts >> 8);
        asm volatile("" : "+s"(K0), "+s"(N));             // (or every comparison with them is kept over the loop)
        const long row0 = tile * AN_ROWS;
        u32x4 act[2][8];
        load_inputs(tile, K0, act);
        if (!STREAM) wp = lds;
        f32x4 y[2][4];
#pragma unroll 1
        for (int layer = 0; layer + 1 < NL; ++layer) {
            const int K = any_width(widths, layer), gn = any_width(widths, layer + 1) >> 5;
            f32x4 acc[2][HT];
            products(K, gn, acc, act, IC<4>{}, IC<HT>{});
            const float* bias = a.b[layer];
            if (bias != nullptr) {
#pragma unroll
                for (int t = 0; t < HT; ++t)
                    if (t < 2 * gn)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float b = bias[32 * (t >> 1) + 4 * (t & 1) + 8 * q + r];
                            acc[0][t][r] = any_biased(acc[0][t][r], b);
                            acc[1][t][r] = any_biased(acc[1][t][r], b);
                        }
                if (!all_256)
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                        for (int t = 0; t < HT; ++t) any_max0(acc[rt][t]);
            }
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int s = 0; s < HT / 2; ++s) {
                    const f32x4 lo = acc[rt][2 * s], hi = acc[rt][2 * s + 1];
                    act[rt][s] = u32x4{pack_relu2<DT>(lo[0], lo[1]), pack_relu2<DT>(lo[2], lo[3]), pack_relu2<DT>(hi[0], hi[1]), pack_relu2<DT>(hi[2], hi[3])};
                }
        }
        const long my_row = row0 + 16 * (q >> 1) + j;     // of a head of few outputs, and of the uniform
        float uniform = 1.f;
        if (a.u != nullptr) uniform = a.u[my_row < a.batch ? my_row : a.batch - 1];
        const int KL = any_width(widths, NL - 1);
        if (N <= 4) products4(KL, y, act, IC<4>{});
        else products(KL, (N + 31) >> 5, y, act, IC<4>{}, IC<4>{});
        const HeadOut out = head_out(a);
        const int limit = a.mask_size > 0 ? a.mask_size : N;
        const float* bias = a.b[NL - 1];
        if (N <= 4) {                                     // both tiles at once: lanes 0..31 the first's rows, two each, the others the second's
            float p[4], past;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                p[k] = q < 2 ? y[0][0][k] : y[1][0][k];
                if (bias != nullptr) p[k] += bias[k < N ? k : N - 1];
            }
            if (a.ph.philox_mode >= 0) uniform = reference_row_uniform(a.ph, my_row < a.batch ? my_row : 0);
            any_head4(out, p, past, N, limit, all_256, [&](float* to) {
                // the 32 rows are one block: whole waves write it, 16 bytes or one column per lane (row r's p: lane r % 16 + 32 (r / 16))
                const int stride = out.stride, piece = (stride & 3) == 0 ? 4 : 1, per_row = stride / piece;
                int r = lane / per_row, c = lane - r * per_row;
                const int dr = 64 / per_row, dc = 64 - dr * per_row;
                float* at = to + row0 * stride + lane * piece;
#pragma unroll 1
                for (int i = 0; 2 * i < per_row; ++i) {                         // (every lane takes part in every turn: rows are read from all of them)
                    const int from = (r & 15) + ((r & 16) << 1);
                    const float rest = __shfl(past, from), p0 = __shfl(p[0], from), p1 = __shfl(p[1], from), p2 = __shfl(p[2], from), p3 = __shfl(p[3], from);
                    if (r < AN_ROWS && row0 + r < a.batch) {
                        if (piece == 4) *reinterpret_cast<float4*>(at) = c > 0 ? make_float4(rest, rest, rest, rest) : make_float4(p0, N > 1 ? p1 : rest, N > 2 ? p2 : rest, N > 3 ? p3 : rest);
                        else *at = c < N ? (c == 0 ? p0 : c == 1 ? p1 : c == 2 ? p2 : p3) : rest;
                    }
                    at += 64 * piece;
                    r += dr;
                    c += dc;
                    if (c >= per_row) {
                        c -= per_row;
                        ++r;
                    }
                }
            });
            if (out.action != nullptr && (q & 1) == 0 && my_row < a.batch) out.action[my_row] = head_pick4(p, uniform);
            continue;
        }
#pragma unroll 1
        for (int rt = 0; rt < 2; ++rt) {
            const long row = row0 + 16 * rt + j;
            const bool ok = row < a.batch;
            int qh = q;
            asm volatile("" : "+v"(qh));                  // (the same: two scalar registers a comparison)
            float u = __shfl(uniform, 32 * rt + j);
            if (a.ph.philox_mode >= 0) u = reference_row_uniform(a.ph, ok ? row : 0);
            f32x4 mine[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                mine[t] = rt == 0 ? y[0][t] : y[1][t];
                if (bias != nullptr)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int n = 32 * (t >> 1) + 8 * q + 4 * (t & 1) + r;
                        mine[t][r] += bias[n < N ? n : N - 1];
                    }
            }
            if (N <= 32) {
                const f32x4 v[2] = {mine[0], mine[1]};
                any_head<1>(out, v, row, ok, j, qh, N, limit, u, all_256);
            } else {
                any_head<2>(out, mine, row, ok, j, qh, N, limit, u, false);
            }
        }
    }
}

// ---- 65 to 128 rows per compute unit, mostly of stacks that do not fit the LDS: a round of workgroups of 128 rows -----------------------
// Eight waves, 16 batch rows per wave: every wave pushes its rows through ALL layers with the activations in its registers, as in the
// kernel of 256 wide layers (mlp.hip), whose weight stream -- chunks of 64 K-columns through a ring of four LDS stages, three
// ahead, one barrier a chunk -- this is for any hidden width.  Two rounds of mlp_features_kernel, or four waves of 32 rows a unit, take longer
// (us, this / mlp_features_kernel / mlp_rows_kernel, 24620 rows: 48-256-256-32-64 masked to 4 18.1 / 20.0 / 20.5, 64-256-256-128-6 18.0 / 22.3 /
// 23.8, 128-192-192-192-4 18.7 / 19.7 / 20.3, 128-128-128-128-128-128-128-20 23.5 / 24.0 / 23.5); more than 32 computed outputs, whose head is a chain
// of one lane's own here, do not gain (256-224-256-256-64 33.9 / 31.5 / 36.2).  So do, where weights fit, stacks of up to two hidden layers under
// five to sixteen outputs, whose head is a large part (this / mlp_rows_kernel, 27000 rows: 128-192-10 10.8 / 12.0, 256-192-10 14.6 / 15.3, 32-64-64-10
// 9.1 / 9.6; the other way 256-224-16 16.5 / 15.5, and with three hidden layers 192-96-96-96-6 15.4 / 13.8).
constexpr int AN_ROUND_WAVES = 8, AN_ROUND_ROWS = 16 * AN_ROUND_WAVES, AN_ROUND_OUT = 32;
constexpr int AN_ROUND_LDS = MLP_STAGES * MLP_STAGE_BYTES + 1024;     // the ring, and what the loads that keep the count go to

template <int DT>
__global__ __launch_bounds__(AN_ROUND_WAVES * 64) void mlp_round_kernel(const MlpArgs a) {
    constexpr int NW = AN_ROUND_WAVES, MLP_ROWS = AN_ROUND_ROWS;
    constexpr int MLP_DMA_PER_WAVE = MLP_MAX_DIM / 8 / NW;         // of 1 KiB, in a full chunk
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15;       // batch row inside the wave's 16-row tile; weight row inside a 16-row tile
    const int q = lane >> 4;       // which 8 of the 32 K-values of an MFMA step this lane feeds
    const long row = (long)blockIdx.x * MLP_ROWS + wave * 16 + j;
    const bool row_ok = row < a.batch;
    const unsigned lds_base = (unsigned)(size_t)lds;
    const unsigned dummy_dst = lds_base + MLP_STAGES * MLP_STAGE_BYTES;

    // ---- weight chunk pipeline: chunk = (layer, 64-column slab c) ----
    int pf_layer = 0, pf_c = 0;    // next chunk to fetch
    int pf_stage = 0;
    auto fetch_next_chunk = [&]() {
        const bool live = pf_layer < a.n_layers;
        const int layer = live ? pf_layer : 0;
        const int K = a.dims[layer], N = a.dims[layer + 1];
        const unsigned char* W = (const unsigned char*)a.w[layer];
        const int n_instr = live ? (N + 7) / 8 : 0;            // 8 weight rows (128 bytes each) per instruction
#pragma unroll
        for (int m = 0; m < MLP_DMA_PER_WAVE; ++m) {
            const int ii = wave + NW * m;
            if (ii < n_instr) {
                int n = ii * 8 + (lane >> 3);
                const int piece = (lane & 7) ^ mlp_swz(n);        // the K piece that belongs in LDS slot lane & 7
                n = n < N ? n : N - 1;                             // rows past N: any valid row, never used
                int k = pf_c * 64 + piece * 8;
                k = k <= K - 8 ? k : K - 8;                        // pieces past K: multiplied by zero activations
                mlp_dma(W, (unsigned)((n * K + k) * 2), lds_base + pf_stage * MLP_STAGE_BYTES + ii * 1024);
            } else {
                mlp_dma((const unsigned char*)a.w[0], 0u, dummy_dst);  // keeps the per-chunk DMA count fixed
            }
        }
        if (live) {
            ++pf_c;
            if (pf_c * 64 >= K) { pf_c = 0; ++pf_layer; }
        }
        pf_stage = (pf_stage + 1) & (MLP_STAGES - 1);
    };
    fetch_next_chunk();
    fetch_next_chunk();
    fetch_next_chunk();

    // ---- the wave's input rows as MFMA operand fragments: for step s (32 K-values) lane (j, q)
    //      holds x[row][32 s + 8 q .. + 7] ----
    u32x4 act[MLP_MAX_DIM / 32];
    {
        const int K0 = a.dims[0];
        const unsigned char* xr = (const unsigned char*)a.x + row * K0 * 2;
#pragma unroll
        for (int s = 0; s < MLP_MAX_DIM / 32; ++s) {
            u32x4 v = {0u, 0u, 0u, 0u};
            if (row_ok && 32 * s + 8 * q < K0) v = *reinterpret_cast<const u32x4*>(xr + (32 * s + 8 * q) * 2);
            act[s] = v;
        }
    }

    f32x4 acc[MLP_MAX_DIM / 16];
    int stage = 0;
    // LDS byte offset of this lane's 16-byte weight piece for the first tile of a chunk: lane j feeds
    // weight row n0 = 8 (j / 4) + j % 4 of the 32-row group, K piece 4 sp + q (sp = which 32-wide step
    // of the chunk).  Tile t adds (t / 2) * 32 + (t % 2) * 4 rows, which leaves swz() unchanged.
    const int n0 = 8 * (j >> 2) + (j & 3);
    unsigned frag_off[2];
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) frag_off[sp] = (unsigned)(n0 * 128 + (((4 * sp + q) ^ mlp_swz(n0)) << 4));
    auto tile_off = [](int t) { return ((t >> 1) * 32 + (t & 1) * 4) * 128; };
    auto tile_col = [&](int t) { return 32 * (t >> 1) + 4 * (t & 1) + 8 * q; };  // first of this lane's 4 columns
    // per-wave f32 staging of the last layer's outputs; it reuses the first weight stage once every
    // wave is done with the weights
    float* head_rows = reinterpret_cast<float*>(lds) + wave * 16 * MLP_MAX_OUT;
    static_assert(NW * 16 * MLP_MAX_OUT * 4 <= MLP_STAGE_BYTES, "head staging must fit one weight stage");

    for (int layer = 0; layer < a.n_layers; ++layer) {
        const int K = a.dims[layer], N = a.dims[layer + 1];
        const int nt = 2 * ((N + 31) / 32);   // output tiles come in pairs covering 32 columns
        const bool last = layer + 1 == a.n_layers;
#pragma unroll
        for (int t = 0; t < MLP_MAX_DIM / 16; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
        for (int c = 0; c < MLP_MAX_DIM / 64; ++c) {
            if (c * 64 < K) {
                // the two newer chunks may still be in flight; everything older has landed
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * MLP_DMA_PER_WAVE) : "memory");
                __syncthreads();
                fetch_next_chunk();   // into the stage every wave finished reading before this barrier
                const unsigned char* st = lds + stage * MLP_STAGE_BYTES;
                // Output tiles are walked in groups of 4 (64 columns) with one uniform branch per
                // group, so that the 8 or 16 LDS reads and the MFMAs of a group form one straight
                // line the scheduler can overlap.  A partly filled last group multiplies whatever
                // the stage holds past row N; those columns are never used.
                const bool two_steps = c * 64 + 32 < K;
                auto mma = [&](int t, int sp, const u32x4& w) {
                    // weights are the first operand: the result fragment is (n, batch row)
                    if constexpr (DT == SP_F16)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, act[2 * c + sp]), acc[t], 0, 0, 0);
                    else
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, act[2 * c + sp]), acc[t], 0, 0, 0);
                };
                auto read = [&](int t, int sp) {
                    return *reinterpret_cast<const u32x4*>(st + frag_off[sp] + tile_off(t));
                };
                if (nt == MLP_MAX_DIM / 16 && two_steps) {
                    // full-width chunk: 8 groups of (4 tiles, one 32-wide step), software pipelined by
                    // hand: the weight pieces of group g + 2 are requested before the MFMAs of group g
                    // (with one wave per SIMD nothing else hides the LDS latency)
                    u32x4 w[3][4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) w[0][t] = read(t, 0);
#pragma unroll
                    for (int t = 0; t < 4; ++t) w[1][t] = read(t, 1);
#pragma unroll
                    for (int g = 0; g < 8; ++g) {
                        if (g + 2 < 8) {
#pragma unroll
                            for (int t = 0; t < 4; ++t) w[(g + 2) % 3][t] = read(((g + 2) >> 1) * 4 + t, (g + 2) & 1);
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int t = 0; t < 4; ++t) mma((g >> 1) * 4 + t, g & 1, w[g % 3][t]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
#pragma unroll
                    for (int g4 = 0; g4 < MLP_MAX_DIM / 64; ++g4) {
                        if (g4 * 4 < nt) {
                            u32x4 w0[4], w1[4];
#pragma unroll
                            for (int t = 0; t < 4; ++t) w0[t] = read(g4 * 4 + t, 0);
                            if (two_steps) {
#pragma unroll
                                for (int t = 0; t < 4; ++t) w1[t] = read(g4 * 4 + t, 1);
                            }
#pragma unroll
                            for (int t = 0; t < 4; ++t) mma(g4 * 4 + t, 0, w0[t]);
                            if (two_steps) {
#pragma unroll
                                for (int t = 0; t < 4; ++t) mma(g4 * 4 + t, 1, w1[t]);
                            }
                        }
                    }
                }
                stage = (stage + 1) & (MLP_STAGES - 1);
            }
        }

        // ---- layer epilogue: in tile t lane (j, q) holds columns tile_col(t) + 0..3 of batch row j;
        //      tiles 2 s and 2 s + 1 together give it columns 32 s + 8 q .. + 7 ----
        const float* bias = a.b[layer];
#pragma unroll
        for (int t = 0; t < MLP_MAX_DIM / 16; ++t) {
            if (t < nt && bias != nullptr) {
                const int n = tile_col(t);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < N) acc[t][r] += bias[n + r];
            }
        }
        if (!last) {
#pragma unroll
            for (int s = 0; s < MLP_MAX_DIM / 32; ++s) {
                u32x4 v = {0u, 0u, 0u, 0u};
                if (32 * s < N) {
                    const f32x4 lo = acc[2 * s], hi = acc[2 * s + 1];
                    v.x = relu_pack2<DT>(lo[0], lo[1]);
                    v.y = relu_pack2<DT>(lo[2], lo[3]);
                    v.z = relu_pack2<DT>(hi[0], hi[1]);
                    v.w = relu_pack2<DT>(hi[2], hi[3]);
                }
                act[s] = v;
            }
        } else {
            __syncthreads();   // all waves have read their last weight chunk: the stage can be reused
#pragma unroll
            for (int t = 0; t < AN_ROUND_OUT / 16; ++t) {
                if (t < nt) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) head_rows[j * MLP_MAX_OUT + tile_col(t) + r] = acc[t][r];
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // drain the dummy DMAs before the LDS is released

    // ---- head: lanes 0..15 of every wave own one batch row each (the staging is wave private) ----
    const int N = a.dims[a.n_layers];
    const int limit = a.mask_size > 0 ? a.mask_size : N;
    float past = 0.f;
    if (lane < 16 && row_ok) {
        float* p = head_rows + lane * MLP_MAX_OUT;   // this row's outputs
        const float u = a.ph.philox_mode >= 0 ? reference_row_uniform(a.ph, row) : a.action != nullptr ? a.u[row] : 1.f;
        // narrow heads run in registers, at the smallest width that holds them: the head is a chain of this lane's own (batch
        // 64, us, always 64 columns / these widths: 64-64-64-10 14.9 / 10.0, 64-96-96-16 16.7 / 11.8, 128-64-24 14.1 / 10.2)
        if (N <= 8) head_row<8>(head_out(a), p, row, N, limit, u, N, &past);
        else if (N <= 16) head_row<16>(head_out(a), p, row, N, limit, u);
        else head_row<AN_ROUND_OUT>(head_out(a), p, row, N, limit, u);
    }
    if (a.out_stride > N) {
        // a masked head computed for its valid columns only (N < 8): the wave fills the rest of its 16 policy rows, 16 bytes
        // per lane where rows are whole pieces, the columns in front of the first whole piece by the row's own lane
        const int stride = a.out_stride, s4 = stride >> 2, c0 = stride % 4 == 0 ? (N + 3) >> 2 : s4 + 1;
        if (lane < 16 && row_ok)
            for (int c = N; c < stride && c < 4 * c0; ++c) a.policy[row * stride + c] = past;
        if (c0 < s4) {
            const long first = (long)blockIdx.x * MLP_ROWS + wave * 16;
            int r = lane / s4, c = lane - r * s4;
            const int dr = 64 / s4, dc = 64 - dr * s4;
            for (int idx = lane; idx < 16 * s4; idx += 64) {      // (16 s4 is a multiple of 16: the lanes of the rows stay in)
                const float v = __shfl(past, r);
                if (c >= c0 && first + r < a.batch) *reinterpret_cast<float4*>(a.policy + (first + r) * stride + 4 * c) = make_float4(v, v, v, v);
                r += dr;
                c += dc;
                if (c >= s4) {
                    c -= s4;
                    ++r;
                }
            }
        }
    }
}

// ---- host -------------------------------------------------------------------------------------------------------------------------
template <int DT>
static const void* pick_features_kernel(int r) {
    return r == 1 ? (const void*)mlp_features_kernel<DT, 1> : r == 2 ? (const void*)mlp_features_kernel<DT, 2> : (const void*)mlp_features_kernel<DT, 4>;
}

template <int DT, int WAVES>
static const void* pick_rows_kernel_waves(int widest, bool stream_weights) {
    if (widest <= 128) return stream_weights ? (const void*)mlp_rows_kernel<DT, 8, true, WAVES> : (const void*)mlp_rows_kernel<DT, 8, false, WAVES>;
    return stream_weights ? (const void*)mlp_rows_kernel<DT, 16, true, WAVES> : (const void*)mlp_rows_kernel<DT, 16, false, WAVES>;
}
template <int DT>
static const void* pick_rows_kernel(int widest, bool stream_weights, int waves) {
    return waves == 4 ? pick_rows_kernel_waves<DT, 4>(widest, stream_weights) : pick_rows_kernel_waves<DT, 8>(widest, stream_weights);
}

int mlp_any_launch(int dtype, const MlpArgs& a, hipStream_t stream, const char* what) {
    const int NL = a.n_layers, N = a.dims[NL];
    unsigned long long widths = 0;
    long group_bytes = 0;
    for (int l = 0; l < NL; ++l) {
        widths |= (unsigned long long)(a.dims[l] / 16) << (8 * l);
        const long gk = (a.dims[l] + 63) / 64;
        group_bytes += gk * ((a.dims[l + 1] + 31) / 32) * AN_GROUP;
    }
    const long cus = device_cu_count();
    int widest = 32;
    bool all_256 = NL > 1;
    for (int l = 1; l < NL; ++l) {
        widest = a.dims[l] > widest ? a.dims[l] : widest;
        all_256 = all_256 && a.dims[l] == 256;
    }
    unsigned counts = (unsigned)NL | (all_256 ? AN_ALL_256 : 0u) | (unsigned)N << 8;
    const bool stream_weights = group_bytes > AN_LDS;
    // of a masked head with at most seven valid columns only those are computed here, else all (what lies past them needs one of its own)
    const int outputs = N <= 7 ? N : a.out_stride;
    const bool short_stack = NL <= 3 && outputs > 4 && outputs <= 16;
    if ((stream_weights || short_stack) && !all_256 && outputs <= AN_ROUND_OUT && a.batch > 64 * cus && a.batch <= AN_ROUND_ROWS * cus) {
        const void* kernel = dtype == SP_F16 ? (const void*)mlp_round_kernel<SP_F16> : (const void*)mlp_round_kernel<SP_BF16>;
        int rc = ensure_dynamic_lds(kernel, AN_ROUND_LDS);
        if (rc != SP_OK) return rc;
        MlpArgs whole = a;
        whole.dims[NL] = outputs;
        void* args[] = {(void*)&whole};
        const hipError_t e = hipLaunchKernel(kernel, dim3((unsigned)((a.batch + AN_ROUND_ROWS - 1) / AN_ROUND_ROWS)), dim3(64 * AN_ROUND_WAVES), args, AN_ROUND_LDS, stream);
        if (e != hipSuccess) return fail(SP_ERR_DEVICE, "%s: launch failed: %s", what, hipGetErrorString(e));
        return check_launch(what);
    }
    if (a.batch > (stream_weights ? 128 : 64) * cus) {
        const long tiles = (a.batch + AN_ROWS - 1) / AN_ROWS, per_block = tiles <= 4 * cus ? 4 : 8;
        const void* kernel = dtype == SP_F16 ? pick_rows_kernel<SP_F16>(widest, stream_weights, (int)per_block) : pick_rows_kernel<SP_BF16>(widest, stream_weights, (int)per_block);
        int rc = ensure_dynamic_lds(kernel, AN_LDS);
        if (rc != SP_OK) return rc;
        const long most = (tiles + per_block - 1) / per_block, blocks = most < cus ? most : cus;
        void* args[] = {(void*)&widths, (void*)&counts, (void*)&a};
        const hipError_t e = hipLaunchKernel(kernel, dim3((unsigned)blocks), dim3(64 * per_block), args, stream_weights ? 4 * AN_STAGE : (size_t)group_bytes, stream);
        if (e != hipSuccess) return fail(SP_ERR_DEVICE, "%s: launch failed: %s", what, hipGetErrorString(e));
        return check_launch(what);
    }
    // rows of a workgroup: as few as leave one workgroup per compute unit
    const int r = a.batch <= 16 * cus ? 1 : a.batch <= 32 * cus ? 2 : 4;
    const void* kernel = dtype == SP_F16 ? pick_features_kernel<SP_F16>(r) : pick_features_kernel<SP_BF16>(r);
    int rc = ensure_dynamic_lds(kernel, AN_LDS);
    if (rc != SP_OK) return rc;
    // (us, 4 / 8 / 16 waves, one workgroup per compute unit: 80-192-192-192-24 12.0 / 10.1 / 9.4, 64-128-128-4 6.3 / 5.5 / 5.8, 128-64-64
    // 4.2 / 4.2 / 4.4; of 64 rows each 64-192-192-192-4 13.6 / 11.1 / 10.2, 192-96-64-64 8.8 / 7.1 / 7.4)
    const int waves = widest >= 160 ? 16 : 8;
    const int ring_at = r == 1 ? AnyFeatures<1>::RING_AT : r == 2 ? AnyFeatures<2>::RING_AT : AnyFeatures<4>::RING_AT;
    int units = 0;                                        // of wave 0, the busiest
    for (int l = 0; l < NL; ++l) units += (a.dims[l] + 63) / 64 * (((a.dims[l + 1] + 15) / 16 + waves - 1) / waves);
    int slots = (AN_LDS - ring_at) / (waves * AN_UNIT);
    slots = slots < AN_SLOTS ? slots : AN_SLOTS;
    slots = units + 1 < slots ? units + 1 : slots;
    counts |= (unsigned)waves << 16;
    const int lds_bytes = ring_at + waves * slots * AN_UNIT;
    const long blocks = (a.batch + 16 * r - 1) / (16 * r);
    const void *x = a.x, *w0 = a.w[0], *w1 = NL > 1 ? a.w[1] : a.w[0];
    long batch = a.batch;
    void* args[] = {(void*)&x, (void*)&w0, (void*)&w1, (void*)&widths, (void*)&batch, (void*)&a.u, (void*)&counts, (void*)&slots, (void*)&a};
    const hipError_t e = hipLaunchKernel(kernel, dim3((unsigned)blocks), dim3(64 * waves), args, lds_bytes, stream);
    if (e != hipSuccess) return fail(SP_ERR_DEVICE, "%s: launch failed: %s", what, hipGetErrorString(e));
    return check_launch(what);
}

namespace {
struct MlpAnyKernelNames {
    MlpAnyKernelNames() {
        register_kernel("mlp_forward", (const void*)mlp_features_kernel<SP_F16, 1>, AN_FEATURES_THREADS);
        register_kernel("mlp_forward_64_rows", (const void*)mlp_features_kernel<SP_F16, 4>, AN_FEATURES_THREADS);
        register_kernel("mlp_forward_wide", (const void*)mlp_rows_kernel<SP_F16, 16, false, 8>, 512);
        register_kernel("mlp_forward_wide_4w", (const void*)mlp_rows_kernel<SP_F16, 16, false, 4>, 256);
        register_kernel("mlp_forward_wide_stream", (const void*)mlp_rows_kernel<SP_F16, 16, true, 8>, 512);
        register_kernel("mlp_forward_wide_128", (const void*)mlp_rows_kernel<SP_F16, 8, false, 8>, 512);
        register_kernel("mlp_forward_round", (const void*)mlp_round_kernel<SP_F16>, AN_ROUND_WAVES * 64);
    }
} mlp_any_kernel_names;
}  // namespace

}  // namespace sp
