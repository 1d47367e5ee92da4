// What the workgroup-tile kernels with 32 x 32 MFMAs share: the walk over the tiles and the stores of a wave's accumulators.
#pragma once
#include "gemm_common.h"

namespace sp {

// Map the linear workgroup id to an output tile.  Workgroups are dealt round-robin to the 8 XCDs
// (each with a private L2), so id % 8 selects the XCD; each XCD gets a contiguous range of the
// tile sequence, and the sequence walks the tile grid in column-major groups of GROUP_M tile rows
// so that an XCD's concurrent tiles share A and B panels.
__device__ __forceinline__ void tile_of_block(int pid, int tiles_m, int tiles_n, int GROUP_M, int& tm, int& tn) {
    constexpr int XCDS = 8;
    const int n = tiles_m * tiles_n;
    const int xcd = pid % XCDS;
    const int idx = pid / XCDS;
    const int base = n / XCDS, rem = n % XCDS;
    const int t = xcd * base + (xcd < rem ? xcd : rem) + idx;
    const int group_size = GROUP_M * tiles_n;
    const int g = t / group_size;
    const int first_m = g * GROUP_M;
    const int gsz = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
    const int in_group = t % group_size;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

constexpr int strip_columns(int wave_columns) { return wave_columns < 64 ? wave_columns : 64; }
constexpr int strip_bytes(int wave_columns) { return 32 * (strip_columns(wave_columns) * 4 + 16); }

// Where the accumulators of MFMAs with B as the first operand hold the outputs of a strip of 32 rows (number i of the wave tile)
// and 32 SF columns (number js): at(row, column, four consecutive columns) for every quad of registers.
template <int SF, int TM, int TN, typename F>
__device__ __forceinline__ void strip_quads(const f32x16 (&acc)[TM][TN], int i, int js, int lane, F at) {      // 32 x 32 MFMAs
#pragma unroll
    for (int jj = 0; jj < SF; ++jj)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
            const f32x16& c16 = acc[i][js * SF + jj];
            at(lane & 31, jj * 32 + gq * 8 + (lane >> 5) * 4, f32x4{c16[4 * gq], c16[4 * gq + 1], c16[4 * gq + 2], c16[4 * gq + 3]});
        }
}
template <int SF, int TM, int TN, typename F>
__device__ __forceinline__ void strip_quads(const f32x4 (&acc)[TM][TN], int i, int js, int lane, F at) {       // 16 x 16 MFMAs
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int jj = 0; jj < 2 * SF; ++jj) at(16 * ii + (lane & 15), 16 * jj + 4 * (lane >> 4), acc[2 * i + ii][js * 2 * SF + jj]);
}

// The end of a tile: a wave transposes its accumulators (WTM x WTN outputs from (m_first, n_first) on) through a private LDS
// strip of 32 rows x up to 64 columns, so that C is written (and, for beta != 0, read) as whole row segments: 16 bytes per lane,
// up to 256 contiguous bytes per row.
template <int OT, int WTM, int WTN, bool RAGGED, typename ACC>
__device__ __forceinline__ void store_accumulators(const GemmArgs& g, unsigned char* Cb, const ACC& acc, unsigned char* stg,
                                                   long m_first, long n_first, int lane) {
    constexpr int TM = WTM / 32, TN = WTN / 32;
    constexpr int SW = strip_columns(TN * 32);     // columns per strip
    constexpr int SF = SW / 32;                    // fragments per strip
    constexpr int EPI_STRIDE = SW * 4 + 16;        // bytes; the pad keeps the 16-byte column writes conflict free
    constexpr int LPR = SW / 4;                    // lanes per output row
    constexpr int RPP = 64 / LPR;                  // rows per pass
    const int er = lane / LPR, ec = (lane % LPR) * 4;
    const float alpha = g.alpha, beta = g.beta;
    const long row_step = (long)RPP * g.N;
    // The options are compile-time inside the loops: a branch per output row would split them into blocks of one
    // LDS read -> one store each, with every latency exposed.
    auto write_tile = [&](auto BETA_, auto RELU_, auto POLICY_) {
        constexpr bool HAS_BETA = decltype(BETA_)::value, RELU = decltype(RELU_)::value;
        constexpr int POLICY = decltype(POLICY_)::value;
        auto finish = [&](f32x4 v, const f32x4& old, const f32x4& bias) {
            v = v * alpha;
            if constexpr (HAS_BETA) v += beta * old;
            v += bias;
            if constexpr (RELU) { v.x = fmaxf(v.x, 0.f); v.y = fmaxf(v.y, 0.f); v.z = fmaxf(v.z, 0.f); v.w = fmaxf(v.w, 0.f); }
            return v;
        };
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int js = 0; js < TN / SF; ++js) {
                const long col = n_first + js * SW + ec;
                const bool col_ok = !RAGGED || col + 3 < g.N;          // all four columns of this lane
                f32x4 bias4 = {0.f, 0.f, 0.f, 0.f};
                if (g.bias && col_ok) bias4 = *reinterpret_cast<const f32x4*>(g.bias + col);
                strip_quads<SF>(acc, i, js, lane, [&](int row, int c, const f32x4& v) {
                    *reinterpret_cast<f32x4*>(stg + row * EPI_STRIDE + c * 4) = v;
                });
                const long row_first = m_first + i * 32 + er;
                long idx = row_first * g.N + col;     // advanced by RPP rows per pass
                // one 4-column piece: what C held there, and the store
                constexpr int AT32 = RAGGED ? 4 : 16, AT16 = RAGGED ? 2 : 8;      // ragged rows begin at any element
                auto read_old = [&](long at) {
                    if constexpr (OT == SP_F32) {
                        return load_aligned<AT32, f32x4>((const float*)Cb + at);
                    } else {
                        const u32x2 o = load_aligned<AT16, u32x2>((const unsigned short*)Cb + at);
                        return f32x4{half_bits_to_f32<OT>(o.x & 0xffffu), half_bits_to_f32<OT>(o.x >> 16),
                                     half_bits_to_f32<OT>(o.y & 0xffffu), half_bits_to_f32<OT>(o.y >> 16)};
                    }
                };
                auto write = [&](long at, const f32x4& r) {
                    if constexpr (OT == SP_F32) {
                        store_c<POLICY, AT32>((float*)Cb + at, r);
                    } else {
                        u32x2 o;
                        o.x = pack_halves<OT>(r.x, r.y);
                        o.y = pack_halves<OT>(r.z, r.w);
                        store_c<POLICY, AT16>((unsigned short*)Cb + at, o);
                    }
                };
                constexpr int PASSES = 32 / RPP;
                if constexpr (RAGGED) {
                    // The masks split every pass into blocks of its own, so nothing may wait inside them: all of LDS (and
                    // of the old C) is read first, then everything is stored (63 x 223 x 24 f32 with beta: one read, one
                    // store per pass 7.4 us, this form 4.4).
                    f32x4 v[PASSES], old[PASSES];
                    const long rows_left = g.M - row_first;
#pragma unroll
                    for (int p = 0; p < PASSES; ++p) {
                        v[p] = *reinterpret_cast<const f32x4*>(stg + (p * RPP + er) * EPI_STRIDE + ec * 4);
                        if constexpr (HAS_BETA) {
                            old[p] = f32x4{0.f, 0.f, 0.f, 0.f};
                            if (col_ok && p * RPP < rows_left) old[p] = read_old(idx + p * row_step);
                        }
                    }
                    const bool row_end = g.N % 4 != 0 && n_first + js * SW < g.N && g.N < n_first + (js + 1) * SW;
                    if (row_end) {                       // the last one to three columns of this strip's 32 rows
                        const int first = (int)(g.N / 4 * 4 - (n_first + js * SW)), count = (int)(g.N % 4);
                        const long row = m_first + i * 32 + (lane & 31);
                        for (int e = lane >> 5; e < count && row < g.M; e += 2) {
                            const long c = n_first + js * SW + first + e;
                            const float sum = *reinterpret_cast<const float*>(stg + (lane & 31) * EPI_STRIDE + (first + e) * 4);
                            store_element(Cb, OT, row * g.N + c, sum * alpha, HAS_BETA ? beta : 0.f, g.bias ? g.bias[c] : 0.f, RELU);
                        }
                    }
#pragma unroll
                    for (int p = 0; p < PASSES; ++p)
                        if (col_ok && p * RPP < rows_left)
                            write(idx + p * row_step, finish(v[p], HAS_BETA ? old[p] : f32x4{0.f, 0.f, 0.f, 0.f}, bias4));
                } else {
#pragma unroll
                    for (int p = 0; p < PASSES; ++p, idx += row_step) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(stg + (p * RPP + er) * EPI_STRIDE + ec * 4);
                        f32x4 old = {0.f, 0.f, 0.f, 0.f};
                        if constexpr (HAS_BETA) old = read_old(idx);
                        write(idx, finish(v, old, bias4));
                    }
                }
            }
        }
    };
    typedef std::integral_constant<int, ST_PLAIN> plain_t;
    typedef std::integral_constant<int, ST_THROUGH> through_t;
    typedef std::integral_constant<int, ST_STREAM> stream_t;
    if (beta != 0.f) {
        if (g.relu) write_tile(std::true_type{}, std::true_type{}, plain_t{});
        else write_tile(std::true_type{}, std::false_type{}, plain_t{});
    } else if (g.store_policy == ST_STREAM) {
        if (g.relu) write_tile(std::false_type{}, std::true_type{}, stream_t{});
        else write_tile(std::false_type{}, std::false_type{}, stream_t{});
    } else {
        typedef std::conditional_t<RAGGED, plain_t, through_t> other_t;      // (see where the policy is picked)
        if (g.relu) write_tile(std::false_type{}, std::true_type{}, other_t{});
        else write_tile(std::false_type{}, std::false_type{}, other_t{});
    }
}

}  // namespace sp
