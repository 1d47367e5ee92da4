// What the GEMM kernels share: arguments, the swizzled LDS tile, the DMA loads and the stores of C.
#pragma once
#include "common.h"
#include "gemm_dma.h"
#include <type_traits>

namespace sp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

struct GemmArgs {
    const void* A;
    const void* B;
    void* C;
    const float* bias;
    long M, N, K;
    float alpha, beta;
    int relu;
    int out_dtype;
    int tiles_m, tiles_n;
    long stride_a, stride_b, stride_c;   // bytes between the matrices of a batch (0: shared)
    int batch;
    int group_m;   // tile rows per group of the block -> tile walk (4: an XCD's 32 concurrent tiles form a 4 x 8 patch)
    int ragged;    // M or N is not a multiple of the tile: tiles_m / tiles_n are rounded up
    int k_rotate;  // workgroup t starts its K loop at K-tile (t * k_rotate) % nk and wraps around (0: everyone at 0)
    int store_policy;   // of the stores of C when beta == 0: ST_THROUGH or ST_STREAM, of ragged tiles also ST_PLAIN (with beta != 0 C is read here: ST_PLAIN)
    int phase_groups;   // persistent four-wave kernel: workgroup w starts ((w / 8) % phase_groups) * phase_skew
    int phase_skew;     // sleeps of ~2048 cycles late (0 / 1 groups: everybody at once)
};

// The tiled kernels take the fields their first fetches need (operand addresses, K, batch strides, the tile grid) once
// more as leading scalar parameters: the library is built with kernel-argument preloading, which hands the first
// dwords of scalar parameters to a wave in registers when it starts (a struct is not preloaded), so the first
// fetches do not wait for a scalar load from the argument block (~900 cycles).
#define SP_GEMM_PRELOADED const void *A_first, const void *B_first, long K_first, long stride_a_first, long stride_b_first, \
                          int tiles_m_first, int tiles_n_first, int group_m_first
#define SP_GEMM_PRELOADED_ARGS(g) (g).A, (g).B, (g).K, (g).stride_a, (g).stride_b, (g).tiles_m, (g).tiles_n, (g).group_m
__device__ __forceinline__ GemmArgs with_preloaded(const GemmArgs& g0, SP_GEMM_PRELOADED) {
    GemmArgs g = g0;
    g.A = A_first; g.B = B_first; g.K = K_first; g.stride_a = stride_a_first; g.stride_b = stride_b_first;
    g.tiles_m = tiles_m_first; g.tiles_n = tiles_n_first; g.group_m = group_m_first;
    return g;
}
#define SP_GEMM_TAKE_PRELOADED                                                                                          \
    const GemmArgs g = with_preloaded(g_rest, A_first, B_first, K_first, stride_a_first, stride_b_first, tiles_m_first, \
                                      tiles_n_first, group_m_first)

constexpr int ROW_BYTES = 128;  // bytes of K per LDS row and K-tile
constexpr int CHUNKS = 8;       // 16-byte chunks per LDS row

// 16-byte chunk `kc` of LDS row `row` lives at chunk slot kc ^ swz(row): any 8 consecutive rows
// read at the same kc touch 8 different slots, and rows r, r+8 land in different 128-byte halves.
__device__ __forceinline__ int lds_offset(int row, int kc) {
    return row * ROW_BYTES + (((kc ^ row ^ (row >> 3)) & 7) << 4);
}

template <int T>
__device__ __forceinline__ float half_bits_to_f32(unsigned bits) {
    if constexpr (T == SP_BF16) return __uint_as_float(bits << 16);
    else return (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
}

__device__ __forceinline__ unsigned short f32_to_bf16_rne(float x) {
    unsigned u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

// Two f32 values rounded to nearest even and packed into one register (v_cvt_pk_{f16,bf16}_f32).
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int T>
__device__ __forceinline__ unsigned pack_halves(float a, float b) {
    if constexpr (T == SP_BF16) return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
    else return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, f16x2));
}

// A store of C with a cache policy.  ST_PLAIN: the compiler's store (write-back in the XCD's L2).  ST_THROUGH
// (sc1): written through the L2 as it is issued, instead of leaving the L2 in bursts when lines are evicted or the
// kernel ends -- the C of a GEMM is written once and read by nobody in this launch.  ST_STREAM (nt): streaming, for
// outputs that should not take room in the caches from operands that are read again.  The host picks one per launch
// (`store_policy`).  Measured (bf16, f32 C, us, plain / through / stream): 65536 x 256 x 256 20.8 / 18.0 / 20.7;
// 131072 x 256 x 256 36.5 / 33.3 / 37.3; 65536 x 256 x 2048 76.0 / 75.2 / 65.0; 8192^3 731 / 730 / 689;
// 16384 x 4096 x 4096 383 / 390 / 364; 65536 x 2048 x 512 178 / 177 / 158; 65536 x 1024 x 512 91 / 91 / 96;
// 8192 x 8192 x 1024 123 / 128 / 132; 4096^3 92.6 / 91.8 / 92.2.
enum { ST_PLAIN = 0, ST_THROUGH = 1, ST_STREAM = 2 };
// ALIGN: what the address is known to be aligned to (the attribute of a typedef is lost where that type is a template
// argument, so it is put on inside).
template <int ALIGN, typename V>
__device__ __forceinline__ V load_aligned(const void* p) {
    typedef V W __attribute__((aligned(ALIGN)));
    static_assert(alignof(W) == ALIGN, "alignment lost");
    return *reinterpret_cast<const W*>(p);
}
template <int POLICY, int ALIGN, typename V>
__device__ __forceinline__ void store_c(void* p, V v) {
    typedef V W __attribute__((aligned(ALIGN)));
    static_assert(alignof(W) == ALIGN, "alignment lost");
    static_assert(sizeof(V) == 16 || sizeof(V) == 8, "16- or 8-byte pieces of C");
    if constexpr (POLICY == ST_STREAM) __builtin_nontemporal_store(v, reinterpret_cast<W*>(p));
    else if constexpr (POLICY == ST_PLAIN) *reinterpret_cast<W*>(p) = v;
    else if constexpr (sizeof(V) == 16) store16_through((V*)p, v);
    else asm volatile("global_store_dwordx2 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory");
}

// Four consecutive columns of a row of C whose width need not be a multiple of 4: the same 16- and 8-byte accesses at
// element alignment (the memory pipe takes them at any element boundary), and single elements for the last few columns
// of a row.  v = alpha * sum goes in; beta * C, bias and ReLU are applied here.
typedef f32x4 f32x4_unaligned __attribute__((aligned(4)));
typedef u32x2 u32x2_unaligned __attribute__((aligned(2)));
__device__ __forceinline__ void store_element(unsigned char* C, int out_dtype, long idx, float r, float beta, float bias, int relu) {
    if (out_dtype == SP_F32) {
        float* c = (float*)C + idx;
        if (beta != 0.f) r += beta * *c;
        r += bias;
        *c = relu ? fmaxf(r, 0.f) : r;
    } else {
        unsigned short* c = (unsigned short*)C + idx;
        if (beta != 0.f) r += beta * (out_dtype == SP_BF16 ? half_bits_to_f32<SP_BF16>(*c) : half_bits_to_f32<SP_F16>(*c));
        r += bias;
        if (relu) r = fmaxf(r, 0.f);
        *c = (unsigned short)(out_dtype == SP_BF16 ? pack_halves<SP_BF16>(r, 0.f) : pack_halves<SP_F16>(r, 0.f));
    }
}

// One wave-wide DMA: every lane copies 16 bytes from global memory (uniform base + per-lane
// 32-bit offset) to LDS byte m0 + 16 * lane.  Completion is tracked by vmcnt; the instruction is
// issued from inline assembly so that the tile in flight does not make the compiler wait before
// LDS reads of the tile being multiplied (it cannot tell the two buffers apart).
__device__ __forceinline__ void dma_to_lds(const unsigned char* base, unsigned lane_offset, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_offset), "s"(base), "s"(lds_addr)
                 : "memory", "m0");
}

__device__ __forceinline__ const unsigned char* uniform_ptr(const unsigned char* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (const unsigned char*)(((unsigned long long)hi << 32) | lo);
}

// The split-K kernel of gemm_wave.hip on a tile of its menu (16 x 16, 32 x 32; 16-bit inputs also 64 x 32, 64 x 64), with
// tiles_m / tiles_n set for that tile, rows of at most 32 MiB (per-lane byte offsets of up to 63 rows in 32 bits) and fewer
// than 2^32 tiles in the batch; cus: the compute units of the device.
int launch_gemm_wave(int dtype_in, int tile_m, int tile_n, long cus, const GemmArgs& g, hipStream_t stream);
constexpr long kWaveMaxRowBytes = 1l << 25;

}  // namespace sp
