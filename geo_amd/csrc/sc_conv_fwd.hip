// SC convolution forward: AND / OR / popcount over bit-packed streams (gfx950).
//
//   y[n,co,a,b] = sum_{v<H} sum_{p<P} ( popc( OR_{ci,u} A[n,p,ci,a+u,b+v] & WP[p,v,ci*W+u,co] )
//                                      - popc( OR_{ci,u} A[n,p,ci,a+u,b+v] & WN[p,v,ci*W+u,co] ) )
// (sc.cpp:12-259 with the im2col of sc.cpp:440-452 folded into the addressing).
//
// Mapping.  One wave of 64 lanes per workgroup.  Lanes run over output positions: lane
// slot = (item n, row group a/R, column b) flattened, so a wave may span items.  Every
// lane keeps R consecutive rows x 16 output channels x 2 rails of OR accumulators in
// VGPRs.  The 32 weight words of one (pack, kernel row, OR-group member, c_out tile) are
// the same for all lanes: they are read with scalar loads and enter v_and_or_b32 as its
// SGPR operand, so the inner loop is one VALU instruction per (activation word, weight
// word) pair.  A kernel row's popcounts are folded into int32 sums with v_bcnt_u32_b32.
// Consecutive workgroups take the c_out tiles of the same positions.
#include "sc_common.h"

#include <cmath>
#include <type_traits>

namespace geo_sc {

namespace {

struct FwdParams {
    const uint32_t* __restrict__ act;  // [n][P][c_in][wi][hi], or [P][c_in][wi][hi][n] with ROWS_IN_N
    const uint32_t* __restrict__ wgt;  // [P][h_k][k_or][n_cotile][2][16]
    const uint32_t* __restrict__ wgt_rail;      // [n_cotile][line][16]: the non-zero rail's words
    const uint32_t* __restrict__ wgt_rail_idx;  // [n_cotile][line][8]: a 16-bit field per word
    const uint32_t* __restrict__ wgt_right;      // the packed lines' right halves by themselves, or null
    const uint32_t* __restrict__ wgt_right_idx;  // and their fields
    size_t rail_lines;                          // lines per c_out tile: P * lines per pack
    int32_t* __restrict__ y;           // [n][c_out][wo][ho]
    int n, c_in, wi, hi, c_out, w_k, h_k, packs;
    int wo, ho, n_cotile;
    int row_groups;        // ceil(wo / R), or ceil(n / R) when the rows of a lane are batch items
    long long slots;       // lane slots: n * row_groups * ho, or row_groups * ho
    unsigned act_plane;    // c_in * wi * hi
    int pv_per_block;      // (pack, add group) pairs per blockIdx.y
    // accumulation structure (split kernel): add groups (outer, inner), OR channels in all and
    // per outer group, and the activation strides of an inner add step / an OR channel step
    int add_outer, add_inner, or_ch_total, or_ch_per_group;
    unsigned add_stride, or_stride;
    int or_rows;  // kernel rows OR-ed together before the popcount (1, or h_k for the full OR)
    int or_shares, pairs_per_slot;  // k_conv_fwd_tile_rail: waves per OR group, pairs one after the other
};

// acc |= a & w with w wave-uniform: a single v_and_or_b32 whose first source is the SGPR.
// Written as an instruction because the compiler otherwise re-associates chains of these
// into v_and + v_and + v_or3 (three instructions per two pairs instead of two).
__device__ __forceinline__ void and_or(uint32_t& acc, uint32_t a, uint32_t w_uniform)
{
    asm("v_and_or_b32 %0, %1, %2, %0" : "+v"(acc) : "s"(w_uniform), "v"(a));
}

// OR-accumulate CU consecutive input channels: per channel NW activation words per lane and
// WK weight lines per wave.  word(r, u) is the activation word row r meets at kernel tap u.
template <int R, int WK, int CU, int NW, bool ROWS_IN_N>
__device__ __forceinline__ void or_channels(uint32_t (&orp)[R][kCoTile], uint32_t (&orn)[R][kCoTile],
                                            const uint32_t*& ap, const uint32_t*& wp, const unsigned (&off)[NW],
                                            unsigned ch_stride, unsigned k_stride)
{
    constexpr int C = kCoTile;
    uint32_t aw[CU][NW];
#pragma unroll
    for (int cu = 0; cu < CU; cu++)
#pragma unroll
        for (int j = 0; j < NW; j++) aw[cu][j] = ap[cu * ch_stride + off[j]];
#pragma unroll
    for (int cu = 0; cu < CU; cu++)
#pragma unroll
        for (int u = 0; u < WK; u++) {
            uint32_t wv[2 * C];
#pragma unroll
            for (int c = 0; c < 2 * C; c++) wv[c] = wp[c];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint32_t a = aw[cu][ROWS_IN_N ? r * WK + u : r + u];
#pragma unroll
                for (int c = 0; c < C; c++) {
                    and_or(orp[r][c], a, wv[c]);
                    and_or(orn[r][c], a, wv[C + c]);
                }
            }
            wp += k_stride;
        }
    ap += CU * ch_stride;
}

// Template parameters:
//   R   rows of accumulators per lane.  ROWS_IN_N == false: R consecutive output rows a
//       (dim 2) of one item; the WK kernel taps slide over R+WK-1 activation words, so each
//       word is loaded once per channel.  ROWS_IN_N == true (outputs with a single row, e.g.
//       the SC-linear mapping): R consecutive batch items.
//   WK  kernel extent in dim 2 (0: run-time extent, R == 1).
//   CU  input channels per loop trip, chosen so that a trip holds ~192 and-or instructions.
template <int R, int WK, int CU, bool ROWS_IN_N>
__global__ __launch_bounds__(64) void k_conv_fwd(FwdParams q)
{
    constexpr int C = kCoTile;
    static_assert(WK > 0 || (R == 1 && !ROWS_IN_N), "run-time kernel extent handles one row per lane");
    const int cot = blockIdx.x % q.n_cotile;
    const long long slot0 = (long long)(blockIdx.x / q.n_cotile) * 64 + threadIdx.x;
    const bool live = slot0 < q.slots;
    const long long slot = live ? slot0 : 0;
    // lane slot -> (first item n, first output row a0, output column b).  With ROWS_IN_N the
    // R rows of a lane are items n and n + row_groups, consecutive lanes are consecutive
    // items, and the activation streams are stored item-innermost.
    const int b = ROWS_IN_N ? (int)(slot / q.row_groups) : (int)(slot % q.ho);
    const long long t = slot / q.ho;
    const int a0 = ROWS_IN_N ? 0 : (int)(t % q.row_groups) * R;
    const long long n = ROWS_IN_N ? slot % q.row_groups : t / q.row_groups;
    const unsigned item_stride = (unsigned)q.packs * q.act_plane;

    constexpr int NW = WK == 0 ? 1 : (ROWS_IN_N ? R * WK : R + WK - 1);
    // word offsets inside one channel plane.  Rows past the end (partial last group) are
    // clamped to valid ones: they only feed outputs that are never stored.
    unsigned off[NW];
    if constexpr (WK > 0) {
#pragma unroll
        for (int j = 0; j < NW; j++) {
            if (ROWS_IN_N) {
                const int r = j / WK, u = j % WK;
                off[j] = (n + (long long)r * q.row_groups < q.n ? (unsigned)r * q.row_groups : 0u) +
                         (unsigned)u * q.hi * q.n;
            } else {
                const int row = a0 + j < q.wi ? a0 + j : q.wi - 1;
                off[j] = (unsigned)row * q.hi;
            }
        }
    } else {
        off[0] = 0;
    }
    // strides (words) of one pack, one kernel row step, one channel
    const size_t pack_stride = ROWS_IN_N ? (size_t)q.act_plane * q.n : (size_t)q.act_plane;
    const unsigned v_stride = ROWS_IN_N ? (unsigned)q.n : 1u;
    const unsigned ch_stride = ROWS_IN_N ? (unsigned)q.wi * q.hi * q.n : (unsigned)q.wi * q.hi;
    const uint32_t* act_n = ROWS_IN_N ? q.act + (size_t)b * q.n + n : q.act + (size_t)n * item_stride + b;
    const int k_or = q.c_in * q.w_k;
    const unsigned k_stride = (unsigned)q.n_cotile * 2 * C;

    int sum[R][C];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int c = 0; c < C; c++) sum[r][c] = 0;

    for (int p = 0; p < q.packs; p++) {
        for (int v = 0; v < q.h_k; v++) {
            uint32_t orp[R][C], orn[R][C];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < C; c++) orp[r][c] = orn[r][c] = 0u;

            const uint32_t* ap = act_n + (size_t)p * pack_stride + (size_t)v * v_stride;
            const uint32_t* wp = q.wgt + ((size_t)(p * q.h_k + v) * k_or * q.n_cotile + cot) * (2 * C);

            if constexpr (WK > 0) {
                int ci = 0;
                for (; ci + CU <= q.c_in; ci += CU)
                    or_channels<R, WK, CU, NW, ROWS_IN_N>(orp, orn, ap, wp, off, ch_stride, k_stride);
                if constexpr (CU > 1)
                    for (; ci < q.c_in; ci++)
                        or_channels<R, WK, 1, NW, ROWS_IN_N>(orp, orn, ap, wp, off, ch_stride, k_stride);
            } else {
                for (int ci = 0; ci < q.c_in; ci++) {
                    for (int u = 0; u < q.w_k; u++) {
                        uint32_t wv[2 * C];
#pragma unroll
                        for (int c = 0; c < 2 * C; c++) wv[c] = wp[c];
                        int row = a0 + u;
                        row = row < q.wi ? row : q.wi - 1;
                        const uint32_t aw = ap[(unsigned)row * q.hi];
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            and_or(orp[0][c], aw, wv[c]);
                            and_or(orn[0][c], aw, wv[C + c]);
                        }
                        wp += k_stride;
                    }
                    ap += ch_stride;
                }
            }
            // binary add across kernel rows and packs: v_bcnt_u32_b32 folds the add
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < C; c++) sum[r][c] += __popc(orp[r][c]) - __popc(orn[r][c]);
        }
    }

    if (!live) return;
    const size_t out_plane = (size_t)q.wo * q.ho;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int co = cot * C + c;
        if (co >= q.c_out) break;
        int32_t* yo = q.y + ((size_t)n * q.c_out + co) * out_plane + (size_t)a0 * q.ho + b;
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (ROWS_IN_N) {
                if (n + (long long)r * q.row_groups < q.n)
                    yo[(size_t)r * q.row_groups * q.c_out * out_plane] = sum[r][c];
            } else {
                if (a0 + r < q.wo) yo[(size_t)r * q.ho] = sum[r][c];
            }
        }
    }
}

// The same kernel for launches that are split over blockIdx.y: each workgroup sums a
// contiguous range of (pack, add group) pairs and adds its partial result to y with integer
// atomics (y is zeroed first).  Used for small layers that would otherwise leave most of the
// GPU idle, and for the accumulation modes other than "OR over (c_in, w_k), add over h_k":
// the add groups are (outer, inner) pairs, an outer group owning a range of OR channels
//   Y : outer 1,              inner kernel rows,     OR channels = input channels
//   YZ: outer channel groups, inner kernel rows,     OR channels = the group's input channels
//   Z : outer 1,              inner input channels,  OR channels = kernel rows
//   FULL: one group per pack; the OR runs over the input channels of or_rows = h_k kernel rows
// (sc_cuda_kernel.cu:176-349, :1351-1366), expressed through the two activation strides in FwdParams; the
// weight lines arrive in exactly the order the loop consumes them.
// Template parameters:
//   R   rows of accumulators per lane.  ROWS_IN_N == false: R consecutive output rows a
//       (dim 2) of one item; the WK kernel taps slide over R+WK-1 activation words, so each
//       word is loaded once per channel.  ROWS_IN_N == true (outputs with a single row, e.g.
//       the SC-linear mapping): R consecutive batch items.
//   WK  kernel extent in dim 2 (0: run-time extent, R == 1).
//   CU  input channels per loop trip, chosen so that a trip holds ~192 and-or instructions.
template <int R, int WK, int CU, bool ROWS_IN_N>
__global__ __launch_bounds__(64) void k_conv_fwd_split(FwdParams q)
{
    constexpr int C = kCoTile;
    static_assert(WK > 0 || (R == 1 && !ROWS_IN_N), "run-time kernel extent handles one row per lane");
    const int cot = blockIdx.x % q.n_cotile;
    const long long slot0 = (long long)(blockIdx.x / q.n_cotile) * 64 + threadIdx.x;
    const bool live = slot0 < q.slots;
    const long long slot = live ? slot0 : 0;
    // lane slot -> (first item n, first output row a0, output column b).  With ROWS_IN_N the
    // R rows of a lane are items n and n + row_groups, consecutive lanes are consecutive
    // items, and the activation streams are stored item-innermost.
    const int b = ROWS_IN_N ? (int)(slot / q.row_groups) : (int)(slot % q.ho);
    const long long t = slot / q.ho;
    const int a0 = ROWS_IN_N ? 0 : (int)(t % q.row_groups) * R;
    const long long n = ROWS_IN_N ? slot % q.row_groups : t / q.row_groups;
    const unsigned item_stride = (unsigned)q.packs * q.act_plane;

    constexpr int NW = WK == 0 ? 1 : (ROWS_IN_N ? R * WK : R + WK - 1);
    // word offsets inside one channel plane.  Rows past the end (partial last group) are
    // clamped to valid ones: they only feed outputs that are never stored.
    unsigned off[NW];
    if constexpr (WK > 0) {
#pragma unroll
        for (int j = 0; j < NW; j++) {
            if (ROWS_IN_N) {
                const int r = j / WK, u = j % WK;
                off[j] = (n + (long long)r * q.row_groups < q.n ? (unsigned)r * q.row_groups : 0u) +
                         (unsigned)u * q.hi * q.n;
            } else {
                const int row = a0 + j < q.wi ? a0 + j : q.wi - 1;
                off[j] = (unsigned)row * q.hi;
            }
        }
    } else {
        off[0] = 0;
    }
    // strides (words) of one pack, one kernel row step, one channel
    const size_t pack_stride = ROWS_IN_N ? (size_t)q.act_plane * q.n : (size_t)q.act_plane;
    const unsigned v_stride = ROWS_IN_N ? (unsigned)q.n : 1u;
    const unsigned ch_stride = ROWS_IN_N ? (unsigned)q.wi * q.hi * q.n : (unsigned)q.wi * q.hi;
    const uint32_t* act_n = ROWS_IN_N ? q.act + (size_t)b * q.n + n : q.act + (size_t)n * item_stride + b;
    const unsigned k_stride = (unsigned)q.n_cotile * 2 * C;

    int sum[R][C];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int c = 0; c < C; c++) sum[r][c] = 0;

    // (pack, add group) pairs are independent partial sums: blockIdx.y takes a contiguous
    // range of them when the launch is split to fill the GPU
    const int groups = q.add_outer * q.add_inner;
    const int pv_begin = blockIdx.y * q.pv_per_block;
    const int pv_end = min(q.packs * groups, pv_begin + q.pv_per_block);
    const unsigned add_stride = ROWS_IN_N ? v_stride : q.add_stride;
    const unsigned or_stride = ROWS_IN_N ? ch_stride : q.or_stride;
    const size_t lines_per_pack = (size_t)q.or_rows * q.add_inner * q.or_ch_total * q.w_k;
    {
        for (int pv = pv_begin; pv < pv_end; pv++) {
            const int p = pv / groups, g = pv - p * groups;
            const int go = g / q.add_inner, gi = g - go * q.add_inner;
            const int ch0 = go * q.or_ch_per_group;
            const int chs = min(q.or_ch_per_group, q.or_ch_total - ch0);
            uint32_t orp[R][C], orn[R][C];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < C; c++) orp[r][c] = orn[r][c] = 0u;

            const uint32_t* ap0 = act_n + (size_t)p * pack_stride + (size_t)gi * add_stride + (size_t)ch0 * or_stride;
            const size_t line = p * lines_per_pack + (size_t)ch0 * q.add_inner * q.w_k + (size_t)gi * chs * q.w_k;
            const uint32_t* wp = q.wgt + (line * q.n_cotile + cot) * (2 * C);

            for (int row = 0; row < q.or_rows; row++) {
                const uint32_t* ap = ap0 + row;  // next kernel row: one word further (never with ROWS_IN_N)
                if constexpr (WK > 0) {
                    int ci = 0;
                    for (; ci + CU <= chs; ci += CU)
                        or_channels<R, WK, CU, NW, ROWS_IN_N>(orp, orn, ap, wp, off, or_stride, k_stride);
                    if constexpr (CU > 1)
                        for (; ci < chs; ci++)
                            or_channels<R, WK, 1, NW, ROWS_IN_N>(orp, orn, ap, wp, off, or_stride, k_stride);
                } else {
                    for (int ci = 0; ci < chs; ci++) {
                        for (int u = 0; u < q.w_k; u++) {
                            uint32_t wv[2 * C];
#pragma unroll
                            for (int c = 0; c < 2 * C; c++) wv[c] = wp[c];
                            int arow = a0 + u;
                            arow = arow < q.wi ? arow : q.wi - 1;
                            const uint32_t aw = ap[(unsigned)arow * q.hi];
#pragma unroll
                            for (int c = 0; c < C; c++) {
                                and_or(orp[0][c], aw, wv[c]);
                                and_or(orn[0][c], aw, wv[C + c]);
                            }
                            wp += k_stride;
                        }
                        ap += or_stride;
                    }
                }
            }
            // binary add across kernel rows and packs: v_bcnt_u32_b32 folds the add
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < C; c++) sum[r][c] += __popc(orp[r][c]) - __popc(orn[r][c]);
        }
    }

    if (!live) return;
    const size_t out_plane = (size_t)q.wo * q.ho;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int co = cot * C + c;
        if (co >= q.c_out) break;
        int32_t* yo = q.y + ((size_t)n * q.c_out + co) * out_plane + (size_t)a0 * q.ho + b;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const bool row_ok = ROWS_IN_N ? n + (long long)r * q.row_groups < q.n : a0 + r < q.wo;
            int32_t* dst = yo + (ROWS_IN_N ? (size_t)r * q.row_groups * q.c_out * out_plane : (size_t)r * q.ho);
            if (!row_ok) continue;
            atomicAdd(dst, sum[r][c]);  // integer adds: order does not matter
        }
    }
}

// Layers with few output positions and large OR groups (classifier layers: 64 x 4 x 4 -> 10 at
// batch 256 has 2560 outputs of 1024 products each): one wave per (R output positions, c_out tile,
// pack, add group); the lanes run over the members of the OR group, each with its own weight
// line in VGPRs (read once for all R positions), and the R x 32 partial OR words are combined across the
// wave by halving: in the step of lane bit k every lane hands the half of its words that its partner
// keeps to that partner, so with R = 2 32 + 16 + 8 + 4 + 2 + 1 shuffles leave one finished word per lane (bit 5:
// position, bit 4: rail, bits 3 - 0: channel) where a full xor reduction of every word takes 64 x 6.  With R = 1 the
// two half waves are ORed first (32 shuffles) and then hold the same words.
// Results are added into the zeroed y with integer atomics.  Activation layout [n][P][c_in][wi][hi].
// Bound by the latency of a wave's loads and shuffles, so with few waves R = 1 (see thin_positions).  64 x 4 x 4 -> 10,
// against one position and a full reduction per wave: batch 256, L 64: 15.9 -> 10.7 us, L 128: 24.2 -> 14.7 (R = 2); one
// image, L 128: 7.6 -> 6.4 (7.9 with R = 2), batch 16: 8.1 -> 7.0 (8.3).
template <int R>
__global__ __launch_bounds__(64) void k_conv_fwd_thin(FwdParams q, long long positions)
{
    constexpr int C = kCoTile;
    const int lane = threadIdx.x;
    const int cot = blockIdx.x % q.n_cotile;
    const long long m0 = (long long)(blockIdx.x / q.n_cotile) * R;
    const int groups = q.add_outer * q.add_inner;
    const int p = blockIdx.y / groups, g = blockIdx.y - p * groups;
    const int go = g / q.add_inner, gi = g - go * q.add_inner;
    const int ch0 = go * q.or_ch_per_group;
    const int chs = min(q.or_ch_per_group, q.or_ch_total - ch0);
    const int members = q.or_rows * chs * q.w_k;
    const size_t lines_per_pack = (size_t)q.or_rows * q.add_inner * q.or_ch_total * q.w_k;
    const size_t line0 = p * lines_per_pack + (size_t)ch0 * q.add_inner * q.w_k + (size_t)gi * chs * q.w_k;
    const uint32_t* ap0[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const long long m = m0 + r < positions ? m0 + r : m0;  // a position past the end is never stored
        const int b = (int)(m % q.ho);
        const long long t = m / q.ho;
        const int a = (int)(t % q.wo);
        const long long n = t / q.wo;
        ap0[r] = q.act + ((size_t)n * q.packs + p) * q.act_plane + (size_t)gi * q.add_stride +
                 (size_t)ch0 * q.or_stride + (size_t)a * q.hi + b;
    }

    uint32_t acc[R * 2 * C];  // [position][rail][channel]
#pragma unroll
    for (int i = 0; i < R * 2 * C; i++) acc[i] = 0u;
    for (int j = lane; j < members; j += 64) {
        // member j = (kernel row of the OR, channel of the group, tap u), u fastest
        const int u = j % q.w_k, t2 = j / q.w_k;
        const int ch = t2 % chs, row = t2 / chs;
        const size_t off = (size_t)ch * q.or_stride + (size_t)u * q.hi + row;
        uint32_t aw[R];
#pragma unroll
        for (int r = 0; r < R; r++) aw[r] = ap0[r][off];
        const uint4* wl = reinterpret_cast<const uint4*>(q.wgt + ((line0 + j) * q.n_cotile + cot) * (2 * C));
        uint32_t wv[2 * C];
#pragma unroll
        for (int v4 = 0; v4 < 2 * C / 4; v4++) {
            const uint4 w4 = wl[v4];
            wv[4 * v4] = w4.x;
            wv[4 * v4 + 1] = w4.y;
            wv[4 * v4 + 2] = w4.z;
            wv[4 * v4 + 3] = w4.w;
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 2 * C; c++) acc[r * 2 * C + c] |= aw[r] & wv[c];
    }
    // (a lambda per step: as a loop over `half` the compiler does not unroll it for R = 1 and indexes at run time)
    auto halve = [&](auto half_tag) {
        constexpr int half = decltype(half_tag)::value;
        const bool upper = (lane & half) != 0;
#pragma unroll
        for (int i = 0; i < half; i++) {
            const uint32_t keep = upper ? acc[i + half] : acc[i], give = upper ? acc[i] : acc[i + half];
            acc[i] = keep | (uint32_t)__shfl_xor((int)give, half);
        }
    };
    static_assert(R * 2 * C == 64 || R * 2 * C == 32, "a finished word per lane, or per pair of lanes");
    if constexpr (R == 2) {
        halve(std::integral_constant<int, 32>());
    } else {
#pragma unroll
        for (int i = 0; i < 2 * C; i++) acc[i] |= (uint32_t)__shfl_xor((int)acc[i], 32);
    }
    halve(std::integral_constant<int, 16>());
    halve(std::integral_constant<int, 8>());
    halve(std::integral_constant<int, 4>());
    halve(std::integral_constant<int, 2>());
    halve(std::integral_constant<int, 1>());
    const int mine = __popc(acc[0]);
    const int other = __shfl_xor(mine, C);  // the channel's other rail
    const long long m = m0 + (lane >> 5);
    const int co = cot * C + (lane & (C - 1));
    if ((lane & C) || lane >= 32 * R || m >= positions || co >= q.c_out) return;
    const int b = (int)(m % q.ho);
    const long long t = m / q.ho;
    const int a = (int)(t % q.wo);
    const long long n = t / q.wo;
    atomicAdd(q.y + (((size_t)n * q.c_out + co) * q.wo + a) * q.ho + b, mine - other);
}

// ---------------------------------------------------------------------------------------------
// Rail-skipping kernel for the plain y-mode launches.
//
// A weight has at most one non-zero code (wp = code of clamp(w, 0, .), wn = code of -clamp(w, ., 0),
// sc.cpp:301-304), and a zero code gives an all-zero stream: of the two v_and_or_b32 that
// k_conv_fwd issues per (activation word, weight), one always ORs zeros.  Which one is uniform
// over the wave but varies per (member, channel), so it cannot select a register at compile time;
// gfx9's VGPR index mode can at run time: with s_set_gpr_idx_on(SRC2, DST) the accumulator operand of
// every following VALU instruction is offset by M0[7:0], one M0 update per (member,
// channel) points the same two v_and_or_b32 (two rows) at the channel's positive or negative
// accumulators.  The scalar instructions issue beside the vector ones (measured: one index update
// per v_and_or_b32 leaves the vector rate unchanged), so the kernel executes half of k_conv_fwd's
// vector instructions.
//
// The 64 OR accumulators sit in fixed registers v[64:127]: P[c][r] = v[64 + 2 c + r],
// N[c][r] = v[96 + 2 c + r].  The index of a channel is 2 c (positive rail or zero weight) or
// 32 + 2 c (negative rail); the asm blocks name v64 / v65 and the index does the rest.  The index
// arrives as a ready-made 16-bit M0 value per channel (index and the two operand enables), so one
// scalar instruction per channel moves it into M0 (s_and_b32 / s_lshr_b32 on a word that holds two
// of them; same effect as s_set_gpr_idx_idx, without a separate shift).  The
// compiler sees the four 16-register vectors as read and written by every block and keeps them
// in place.  Index mode is switched off at the end of every block: compiler-generated vector
// instructions in between must not be indexed.
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));

// M0 of a channel from its 16-bit field: index in bits 7:0, the SRC2 and DST enables in bits 15:12
#define GEO_SC_RAIL_LO(I) "s_and_b32 m0, %[" I "], 0xffff\n"
#define GEO_SC_RAIL_HI(I) "s_lshr_b32 m0, %[" I "], 16\n"
#define GEO_SC_RAIL_OPERANDS                                                                                           \
    [w0] "s"(w[0]), [w1] "s"(w[1]), [w2] "s"(w[2]), [w3] "s"(w[3]), [w4] "s"(w[4]), [w5] "s"(w[5]), [w6] "s"(w[6]),     \
        [w7] "s"(w[7]), [w8] "s"(w[8]), [w9] "s"(w[9]), [w10] "s"(w[10]), [w11] "s"(w[11]), [w12] "s"(w[12]),           \
        [w13] "s"(w[13]), [w14] "s"(w[14]), [w15] "s"(w[15]), [i0] "s"(ix[0]), [i1] "s"(ix[1]), [i2] "s"(ix[2]),        \
        [i3] "s"(ix[3]), [i4] "s"(ix[4]), [i5] "s"(ix[5]), [i6] "s"(ix[6]), [i7] "s"(ix[7]), [a0] "v"(a0), [a1] "v"(a1)
// 16 channels x PAIR, the M0 update of every channel but the first in front of its pair
#define GEO_SC_RAIL_16(PAIR)                                                                                           \
    PAIR("w0", "") PAIR("w1", GEO_SC_RAIL_HI("i0")) PAIR("w2", GEO_SC_RAIL_LO("i1")) PAIR("w3", GEO_SC_RAIL_HI("i1"))   \
    PAIR("w4", GEO_SC_RAIL_LO("i2")) PAIR("w5", GEO_SC_RAIL_HI("i2")) PAIR("w6", GEO_SC_RAIL_LO("i3"))                  \
    PAIR("w7", GEO_SC_RAIL_HI("i3")) PAIR("w8", GEO_SC_RAIL_LO("i4")) PAIR("w9", GEO_SC_RAIL_HI("i4"))                  \
    PAIR("w10", GEO_SC_RAIL_LO("i5")) PAIR("w11", GEO_SC_RAIL_HI("i5")) PAIR("w12", GEO_SC_RAIL_LO("i6"))               \
    PAIR("w13", GEO_SC_RAIL_HI("i6")) PAIR("w14", GEO_SC_RAIL_LO("i7")) PAIR("w15", GEO_SC_RAIL_HI("i7"))

// Defines, for accumulators pinned at v[B0 : B0 + 63] (V0 = "vB0", V1 = "v(B0 + 1)" name the first pair):
//  LINE : one weight line (16 channels) against the two activation words of the lane's two rows;
//  FIRST: the first weight line of an OR group, which assigns instead of accumulating and clears the channel's
//         other rail (index ^ 32), so that the 64 accumulators need no zeroing pass.  v_and_b32 and v_mov_b32
//         are two-operand instructions, which issue at twice the rate of v_and_or_b32: the line costs what an
//         accumulating line costs.
// Not volatile: every effect goes through the operands, and a volatile asm would count as a possible store,
// after which the compiler no longer reads the weight lines with scalar loads.
#define GEO_SC_DEFINE_RAIL_LINES(LINE, FIRST, V0, V1, RP0, RP1, RN0, RN1)                                              \
    __device__ __forceinline__ void LINE(u32x16& p0, u32x16& p1, u32x16& n0, u32x16& n1, const uint32_t (&w)[kCoTile],  \
                                         const uint32_t (&ix)[kCoTile / 2], uint32_t a0, uint32_t a1)                  \
    {                                                                                                                  \
        asm("s_set_gpr_idx_on %[i0], gpr_idx(SRC2,DST)\n" GEO_SC_RAIL_16(GEO_SC_RAIL_PAIR_##LINE) "s_set_gpr_idx_off\n" \
            : "+{" RP0 "}"(p0), "+{" RP1 "}"(p1), "+{" RN0 "}"(n0), "+{" RN1 "}"(n1)                                   \
            : GEO_SC_RAIL_OPERANDS                                                                                     \
            : "m0", "scc");                                                                                            \
    }                                                                                                                  \
    __device__ __forceinline__ void FIRST(u32x16& p0, u32x16& p1, u32x16& n0, u32x16& n1, const uint32_t (&w)[kCoTile], \
                                          const uint32_t (&ix)[kCoTile / 2], uint32_t a0, uint32_t a1)                 \
    {                                                                                                                  \
        asm("s_set_gpr_idx_on %[i0], gpr_idx(SRC2,DST)\n" GEO_SC_RAIL_16(GEO_SC_RAIL_PAIR_##FIRST) "s_set_gpr_idx_off\n" \
            : "={" RP0 "}"(p0), "={" RP1 "}"(p1), "={" RN0 "}"(n0), "={" RN1 "}"(n1)                                   \
            : GEO_SC_RAIL_OPERANDS                                                                                     \
            : "m0", "scc");                                                                                            \
    }

// accumulators at v[64:127]: the kernels with four waves per SIMD
#define GEO_SC_RAIL_PAIR_rail_line(W, SET)                                                                             \
    SET "v_and_or_b32 v64, %[" W "], %[a0], v64\n"                                                                     \
        "v_and_or_b32 v65, %[" W "], %[a1], v65\n"
#define GEO_SC_RAIL_PAIR_rail_line_first(W, SET)                                                                       \
    SET "v_and_b32 v64, %[" W "], %[a0]\n"                                                                            \
        "v_and_b32 v65, %[" W "], %[a1]\n"                                                                            \
        "s_xor_b32 m0, m0, 32\n"                                                                                      \
        "v_mov_b32 v64, 0\n"                                                                                          \
        "v_mov_b32 v65, 0\n"
GEO_SC_DEFINE_RAIL_LINES(rail_line, rail_line_first, "v64", "v65", "v[64:79]", "v[80:95]", "v[96:111]", "v[112:127]")
// accumulators at v[32:95]: the kernel with five waves per SIMD (96 registers in all)
#define GEO_SC_RAIL_PAIR_rail_line_lo(W, SET)                                                                          \
    SET "v_and_or_b32 v32, %[" W "], %[a0], v32\n"                                                                     \
        "v_and_or_b32 v33, %[" W "], %[a1], v33\n"
#define GEO_SC_RAIL_PAIR_rail_line_first_lo(W, SET)                                                                    \
    SET "v_and_b32 v32, %[" W "], %[a0]\n"                                                                            \
        "v_and_b32 v33, %[" W "], %[a1]\n"                                                                            \
        "s_xor_b32 m0, m0, 32\n"                                                                                      \
        "v_mov_b32 v32, 0\n"                                                                                          \
        "v_mov_b32 v33, 0\n"
GEO_SC_DEFINE_RAIL_LINES(rail_line_lo, rail_line_first_lo, "v32", "v33", "v[32:47]", "v[48:63]", "v[64:79]", "v[80:95]")
#undef GEO_SC_DEFINE_RAIL_LINES
#undef GEO_SC_RAIL_16
#undef GEO_SC_RAIL_OPERANDS
#undef GEO_SC_RAIL_LO
#undef GEO_SC_RAIL_HI

// sum += popcount(pos) - popcount(neg) in three instructions (the compiler's form takes four)
__device__ __forceinline__ void popc_diff(int& sum, uint32_t pos, uint32_t neg)
{
    uint32_t t;
    asm("v_bcnt_u32_b32 %0, %1, %0" : "+v"(sum) : "v"(pos));
    asm("v_bcnt_u32_b32 %0, %1, 0" : "=v"(t) : "v"(neg));
    sum -= (int)t;
}
static_assert(kCoTile == 16, "rail_line is written for tiles of 16 output channels");

// Weight lines as constant memory (no launch that reads them writes them): where LDS atomics and barriers sit
// in the same loop the compiler reads a plain global pointer with vector loads.
typedef const __attribute__((address_space(4))) uint32_t* ConstWords;

// The packed lines of a c_out tile from line `line` on: 16 words and 16 fields of 16 bits each.
struct RailLines {
    ConstWords w, f;
    __device__ __forceinline__ RailLines(const FwdParams& q, int cot, size_t line)
    {
        const size_t at = (size_t)cot * q.rail_lines + line;
        w = (ConstWords)(q.wgt_rail + at * kCoTile);
        f = (ConstWords)(q.wgt_rail_idx + at * (kCoTile / 2));
    }
    template <int N>
    __device__ __forceinline__ void load(uint32_t (&wv)[N][kCoTile], uint32_t (&iv)[N][kCoTile / 2]) const
    {
#pragma unroll
        for (int l = 0; l < N; l++) {
#pragma unroll
            for (int c = 0; c < kCoTile; c++) wv[l][c] = w[l * kCoTile + c];
#pragma unroll
            for (int c = 0; c < kCoTile / 2; c++) iv[l][c] = f[l * (kCoTile / 2) + c];
        }
    }
    __device__ __forceinline__ void advance(int lines)
    {
        w += lines * kCoTile;
        f += lines * (kCoTile / 2);
    }
};

// Two output rows per lane (R = 2), position-major activation streams, kernel extent WK in dim 2.
// Same lane -> position mapping, grid and result as k_conv_fwd<2, WK, 1, false>.
// CU: input channels per loop trip (their loads are issued together: 2 for 1-wide kernels, so that a
// trip holds 64 vector instructions behind one wait instead of 32).
template <int WK, int CU>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_conv_fwd_rail(FwdParams q)
{
    constexpr int C = kCoTile, R = 2, NW = R + WK - 1;
    const int cot = blockIdx.x % q.n_cotile;
    const long long slot0 = (long long)(blockIdx.x / q.n_cotile) * 64 + threadIdx.x;
    const bool live = slot0 < q.slots;
    const long long slot = live ? slot0 : 0;
    const int b = (int)(slot % q.ho);
    const long long t = slot / q.ho;
    const int a0 = (int)(t % q.row_groups) * R;
    const long long n = t / q.row_groups;
    const unsigned item_stride = (unsigned)q.packs * q.act_plane;
    // word offsets inside one channel plane; rows past the end (partial last group) are clamped to
    // valid ones: they only feed outputs that are never stored
    unsigned off[NW];
#pragma unroll
    for (int j = 0; j < NW; j++) {
        const int row = a0 + j < q.wi ? a0 + j : q.wi - 1;
        off[j] = (unsigned)row * q.hi;
    }
    const unsigned ch_stride = (unsigned)q.wi * q.hi;
    const uint32_t* act_n = q.act + (size_t)n * item_stride + b;
    const int k_or = q.c_in * q.w_k;

    int sum[2 * C];  // [2 c + r]
#pragma unroll
    for (int i = 0; i < 2 * C; i++) sum[i] = 0;

    for (int p = 0; p < q.packs; p++) {
        for (int v = 0; v < q.h_k; v++) {
            u32x16 p0 = 0u, p1 = 0u, n0 = 0u, n1 = 0u;
            const uint32_t* ap = act_n + (size_t)p * q.act_plane + v;
            RailLines rl(q, cot, (size_t)(p * q.h_k + v) * k_or);
            auto channels = [&](auto cu_tag) {
                constexpr int N = decltype(cu_tag)::value;
                uint32_t aw[N][NW];
#pragma unroll
                for (int cu = 0; cu < N; cu++)
#pragma unroll
                    for (int j = 0; j < NW; j++) aw[cu][j] = ap[cu * ch_stride + off[j]];
                uint32_t wv[N * WK][C], iv[N * WK][C / 2];
                rl.load(wv, iv);
#pragma unroll
                for (int cu = 0; cu < N; cu++)
#pragma unroll
                    for (int u = 0; u < WK; u++)
                        rail_line(p0, p1, n0, n1, wv[cu * WK + u], iv[cu * WK + u], aw[cu][u], aw[cu][u + 1]);
                rl.advance(N * WK);
                ap += N * ch_stride;
            };
            int ci = 0;
            for (; ci + CU <= q.c_in; ci += CU) channels(std::integral_constant<int, CU>());
            if constexpr (CU > 1)
                for (; ci < q.c_in; ci++) channels(std::integral_constant<int, 1>());
            // binary add across kernel rows and packs: v_bcnt_u32_b32 folds the add
#pragma unroll
            for (int i = 0; i < C; i++) {
                sum[i] += __popc(p0[i]) - __popc(n0[i]);
                sum[C + i] += __popc(p1[i]) - __popc(n1[i]);
            }
        }
    }

    if (!live) return;
    const size_t out_plane = (size_t)q.wo * q.ho;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int co = cot * C + c;
        if (co >= q.c_out) break;
        int32_t* yo = q.y + ((size_t)n * q.c_out + co) * out_plane + (size_t)a0 * q.ho + b;
#pragma unroll
        for (int r = 0; r < R; r++)
            if (a0 + r < q.wo) yo[(size_t)r * q.ho] = sum[2 * c + r];
    }
}

// The rail-skipping form of k_conv_fwd_split<2, WK, 1, false>: launches split over blockIdx.y and
// the accumulation modes other than y, position-major activation streams, two output rows per lane.
// Partial sums are added to the zeroed y with integer atomics.
// The add groups of the other modes are short (z mode: 9 lines of a 3 x 3 kernel), so what happens
// per group is kept scalar and small: the (pack, outer, inner) group counters advance by increments (no
// divisions), the weight lines of a c_out tile follow each other in loop order (both pointers only
// advance), and the activation words come through buffer loads (resource over the stream buffer, one
// 32-bit byte offset per lane and row, the group's and channel's offset as the scalar operand).
template <int WK, int CU>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_conv_fwd_split_rail(FwdParams q)
{
    constexpr int C = kCoTile, R = 2, NW = R + WK - 1;
    const int cot = blockIdx.x % q.n_cotile;
    const long long slot0 = (long long)(blockIdx.x / q.n_cotile) * 64 + threadIdx.x;
    const bool live = slot0 < q.slots;
    const long long slot = live ? slot0 : 0;
    const int b = (int)(slot % q.ho);
    const long long t = slot / q.ho;
    const int a0 = (int)(t % q.row_groups) * R;
    const long long n = t / q.row_groups;
    const unsigned item_stride = (unsigned)q.packs * q.act_plane;
    // byte offsets of the lane's rows in the stream buffer (the launcher keeps the buffer under 4 GB);
    // rows past the end (partial last group) are clamped to valid ones: they only feed outputs that are
    // never stored
    unsigned voff[NW];
#pragma unroll
    for (int j = 0; j < NW; j++) {
        const int row = a0 + j < q.wi ? a0 + j : q.wi - 1;
        voff[j] = 4u * ((unsigned)n * item_stride + (unsigned)b + (unsigned)row * q.hi);
    }
    const __amdgpu_buffer_rsrc_t act = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(q.act), 0, (int)(4u * (unsigned)q.n * item_stride), 0x00020000);
    const unsigned plane_b = 4u * q.act_plane, add_b = 4u * q.add_stride, or_b = 4u * q.or_stride;

    int sum[2 * C];  // [2 c + r]
#pragma unroll
    for (int i = 0; i < 2 * C; i++) sum[i] = 0;

    const int groups = q.add_outer * q.add_inner;
    const int pv_begin = blockIdx.y * q.pv_per_block;
    const int pv_end = min(q.packs * groups, pv_begin + q.pv_per_block);
    const size_t lines_per_pack = (size_t)q.or_rows * q.add_inner * q.or_ch_total * q.w_k;
    // group counters of pv_begin; the loop advances them
    int p = pv_begin / groups;
    int go = (pv_begin - p * groups) / q.add_inner;
    int gi = pv_begin - p * groups - go * q.add_inner;
    const int ch_first = go * q.or_ch_per_group;
    RailLines rl(q, cot, p * lines_per_pack + (size_t)ch_first * q.add_inner * q.w_k +
                             (size_t)gi * min(q.or_ch_per_group, q.or_ch_total - ch_first) * q.w_k);
    for (int pv = pv_begin; pv < pv_end; pv++) {
        const int ch0 = go * q.or_ch_per_group;
        const int chs = min(q.or_ch_per_group, q.or_ch_total - ch0);
        u32x16 p0, p1, n0, n1;  // written by the group's first line
        bool first = true;
        const unsigned group_off = (unsigned)p * plane_b + (unsigned)gi * add_b + (unsigned)ch0 * or_b;
        for (int row = 0; row < q.or_rows; row++) {
            unsigned ch_off = group_off + 4u * (unsigned)row;  // next kernel row: one word further
            auto channels_of = [&](auto cu_tag, auto first_tag) {
                constexpr int N = decltype(cu_tag)::value;
                constexpr bool FIRST = decltype(first_tag)::value;
                uint32_t aw[N][NW];
#pragma unroll
                for (int cu = 0; cu < N; cu++)
#pragma unroll
                    for (int j = 0; j < NW; j++)
                        aw[cu][j] = __builtin_amdgcn_raw_buffer_load_b32(act, (int)voff[j],
                                                                         (int)(ch_off + (unsigned)cu * or_b), 0);
                uint32_t wv[N * WK][C], iv[N * WK][C / 2];
                rl.load(wv, iv);
#pragma unroll
                for (int cu = 0; cu < N; cu++)
#pragma unroll
                    for (int u = 0; u < WK; u++) {
                        if (FIRST && cu == 0 && u == 0)
                            rail_line_first(p0, p1, n0, n1, wv[0], iv[0], aw[0][0], aw[0][1]);
                        else
                            rail_line(p0, p1, n0, n1, wv[cu * WK + u], iv[cu * WK + u], aw[cu][u], aw[cu][u + 1]);
                    }
                rl.advance(N * WK);
                ch_off += (unsigned)N * or_b;
            };
            auto channels = [&](auto cu_tag) {
                if (first)
                    channels_of(cu_tag, std::true_type());
                else
                    channels_of(cu_tag, std::false_type());
                first = false;
            };
            int ci = 0;
            for (; ci + CU <= chs; ci += CU) channels(std::integral_constant<int, CU>());
            if constexpr (CU > 1)
                for (; ci < chs; ci++) channels(std::integral_constant<int, 1>());
        }
#pragma unroll
        for (int i = 0; i < C; i++) {
            popc_diff(sum[i], p0[i], n0[i]);
            popc_diff(sum[C + i], p1[i], n1[i]);
        }
        // next group: inner add group, then outer, then pack
        if (++gi == q.add_inner) {
            gi = 0;
            if (++go == q.add_outer) {
                go = 0;
                p++;
            }
        }
    }

    if (!live) return;
    const size_t out_plane = (size_t)q.wo * q.ho;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int co = cot * C + c;
        if (co >= q.c_out) break;
        int32_t* yo = q.y + ((size_t)n * q.c_out + co) * out_plane + (size_t)a0 * q.ho + b;
#pragma unroll
        for (int r = 0; r < R; r++)
            if (a0 + r < q.wo) atomicAdd(yo + (size_t)r * q.ho, sum[2 * c + r]);  // integer adds: order does not matter
    }
}

// The five-wave kernels (accumulators at v[32:95], 96 registers): launches in which a wave keeps no running sums.
// A lane's position and the byte offsets of its rows in the stream buffer (the launcher keeps the buffer under
// 4 GB); rows past the end (partial last group) are clamped to valid ones: they only feed outputs that are never
// stored.
template <int NW>
struct PairLane {
    bool live;
    int a0, b;
    long long n;
    unsigned voff[NW];
    __device__ __forceinline__ PairLane(const FwdParams& q, long long slot0)
    {
        live = slot0 < q.slots;
        const long long slot = live ? slot0 : 0;
        b = (int)(slot % q.ho);
        const long long t = slot / q.ho;
        a0 = (int)(t % q.row_groups) * 2;
        n = t / q.row_groups;
#pragma unroll
        for (int j = 0; j < NW; j++) {
            const int row = a0 + j < q.wi ? a0 + j : q.wi - 1;
            voff[j] = 4u * ((unsigned)n * (unsigned)q.packs * q.act_plane + (unsigned)b + (unsigned)row * q.hi);
        }
    }
};

// ---- the OR of consecutive channels of an add group, as one asm block for 3- and 5-wide kernels ----
// How many of a line's words are zero is a property of the weights: streams of a small code are mostly zero words (the initial
// weights of a 64-channel layer at L 256: two thirds), and so are the channels that pad the last tile.  The channels
// of a group go through one of three loops, picked by the zero words of the group's first lines:
//   DENSE (fewer than kSkipZeros per line)  every word of a line;
//   SKIP                                    a jump over the line's zero words, which its packing has put in front;
//   HALF  (kHalfZeros or more)              only the right halves of the lines (slots 8 - 15) are loaded, so that two
//                                           stages of lines fit the scalar registers and one is in flight while the other is
//                                           ORed; the left half of a line with more than eight words is loaded where it is met.
//                                           Where many of them need it the rest of the group changes loops (GEO_SC_FALL_IF).
// What bounds them: DENSE the issue of v_and_or_b32; HALF the scalar instructions, one per SIMD and four cycles like
// the vector ones, of which a line takes one per word and four for its jump.
// One block with its loads and waits inside, registers assigned by hand: scalar loads return out of order, so only
// lgkmcnt(0) says that a line has arrived and the next stage's loads must be issued behind that wait, an order that the
// compiler does not keep; and 64 pinned accumulators that live across its branches it spills.
// Scalar registers (s32 is the compiler's): DENSE and SKIP: words of three lines in s[36:51], s[52:67], s[68:83], their fields
// in s[84:91], s[92:99], s[24:31].  HALF: words of stage A's three lines in s[36:59], of stage B's in s[60:83], fields in
// s[84:95] and s[96:99], s[24:31].  SKIP and HALF: the addresses that the lines' jumps start from in s[18:23] (low) and vcc_hi (high).
// s33, s34: temporary; s35: the zero words of the first lines.
// Index mode stays on between the loads of a channel and the next one's: nothing but the slots' vector instructions is issued.
#define GEO_SC_SLOT(SET, W, I, X0, X1)                                                                                 \
    SET "v_and_or_b32 v32, s[" #W "+" #I "], %[" X0 "], v32\n"                                                         \
        "v_and_or_b32 v33, s[" #W "+" #I "], %[" X1 "], v33\n"
#define GEO_SC_SLOT_FIRST(SET, W, I, X0, X1)                                                                           \
    SET "v_and_b32 v32, s[" #W "+" #I "], %[" X0 "]\n"                                                                 \
        "v_and_b32 v33, s[" #W "+" #I "], %[" X1 "]\n"                                                                 \
        "s_xor_b32 m0, m0, 32\n"                                                                                       \
        "v_mov_b32 v32, 0\n"                                                                                           \
        "v_mov_b32 v33, 0\n"
#define GEO_SC_M0_LO(F, J) "s_mov_b32 m0, s[" #F "+" #J "]\n"
#define GEO_SC_M0_HI(F, J) "s_lshr_b32 m0, s[" #F "+" #J "], 16\n"
#define GEO_SC_EIGHT(SLOT, W, F, X0, X1) SLOT(GEO_SC_M0_LO(F, 0), W, 0, X0, X1) GEO_SC_SEVEN(SLOT, W, F, X0, X1)
#define GEO_SC_SEVEN(SLOT, W, F, X0, X1) SLOT(GEO_SC_M0_HI(F, 0), W, 1, X0, X1)                                        \
    SLOT(GEO_SC_M0_LO(F, 1), W, 2, X0, X1) SLOT(GEO_SC_M0_HI(F, 1), W, 3, X0, X1)                                      \
    SLOT(GEO_SC_M0_LO(F, 2), W, 4, X0, X1) SLOT(GEO_SC_M0_HI(F, 2), W, 5, X0, X1)                                      \
    SLOT(GEO_SC_M0_LO(F, 3), W, 6, X0, X1) SLOT(GEO_SC_M0_HI(F, 3), W, 7, X0, X1)
#define GEO_SC_INDEX_ON "s_set_gpr_idx_on 0, gpr_idx(SRC2,DST)\n"
#define GEO_SC_INDEX_OFF "s_set_gpr_idx_off\n"
// Over zero words: a slot is 20 bytes of code.  A jump takes BITS bits of a field, as many as there are places behind it: whatever a
// buffer holds, it lands on one of them.  s_getpc_b64 gives the address of the s_add_u32, three words in front of place 0.
#define GEO_SC_JUMP(F, BITS)                                                                                           \
    "s_bfe_u32 s33, s[" #F "+0], " #BITS "<<16|8\n"                                                                    \
    "s_mulk_i32 s33, 20\n"                                                                                             \
    "s_addk_i32 s33, 12\n"                                                                                             \
    "s_getpc_b64 s[34:35]\n"                                                                                           \
    "s_add_u32 s34, s34, s33\n"                                                                                        \
    "s_addc_u32 s35, s35, 0\n"                                                                                         \
    "s_setpc_b64 s[34:35]\n"
// the same over eight places with the address of place 0 in BASE and vcc_hi (GEO_SC_BASE; no carry between the places)
#define GEO_SC_JUMP_FROM(BASE, F)                                                                                      \
    "s_bfe_u32 s33, s[" #F "+0], 3<<16|8\n"                                                                            \
    "s_lshl4_add_u32 vcc_lo, s33, " BASE "\n"                                                                          \
    "s_lshl2_add_u32 vcc_lo, s33, vcc_lo\n"                                                                            \
    "s_setpc_b64 vcc\n"
#define GEO_SC_WHOLE(W, F, X0, X1) GEO_SC_EIGHT(GEO_SC_SLOT, W, F, X0, X1) GEO_SC_EIGHT(GEO_SC_SLOT, W + 8, F + 4, X0, X1)
#define GEO_SC_FIRST(W, F, X0, X1)                                                                                     \
    GEO_SC_EIGHT(GEO_SC_SLOT_FIRST, W, F, X0, X1) GEO_SC_EIGHT(GEO_SC_SLOT_FIRST, W + 8, F + 4, X0, X1)
// A line of the loops DENSE and SKIP, the I-th of its channel; X: "x" or "y", the channel's words.  SKIP: past the jump where no word
// is zero (64 -> 64 at 28 x 28, batch 64, L 128, 12 words in the first channel's lines and 16 in the others': 296 us, 323 with a jump
// at every line); s18 + I and vcc_hi hold the address of the line's first slot in the loop's copy for x (GEO_SC_SKIP_BASES).
#define GEO_SC_DENSE(X, I, W, F, X0, X1) GEO_SC_WHOLE(W, F, X0, X1)
#define GEO_SC_SKIP(X, I, W, F, X0, X1)                                                                                \
    "s_bfe_u32 s33, s[" #F "+0], 4<<16|8\n"                                                                            \
    "s_cbranch_scc0 .Lsc_s" X #I "_%=\n"                                                                               \
    "s_lshl4_add_u32 vcc_lo, s33, s[18+" #I "]\n"                                                                      \
    "s_lshl2_add_u32 vcc_lo, s33, vcc_lo\n"                                                                            \
    ".ifnc " X ",x\n"                                                                                                  \
    "s_add_u32 vcc_lo, vcc_lo, .Lsc_sy" #I "_%=-.Lsc_sx" #I "_%=\n"                                                    \
    ".endif\n"                                                                                                         \
    "s_setpc_b64 vcc\n"                                                                                                \
    ".Lsc_s" X #I "_%=:\n" GEO_SC_WHOLE(W, F, X0, X1)
// A line's right half behind a jump, slots 9 to 15 at places 1 to 7.  Place 0, as long as a slot, leaves for a copy of the eight slots
// (GEO_SC_LEFT, out of line) behind which the left half is loaded if it holds words.
#define GEO_SC_RIGHT(LABEL, SEVEN)                                                                                     \
    ".Lsc_" LABEL "_%=:\n"                                                                                             \
    "s_branch .Lsc_" LABEL "_left_%=\n"                                                                                \
    "s_nop 0\ns_nop 0\ns_nop 0\ns_nop 0\n" SEVEN ".Lsc_" LABEL "_done_%=:\n"
// (three words that no wave comes to: a line's code is 192 bytes, and the loop begins at a multiple of 32; without, 0.5 % more)
#define GEO_SC_HALF(LABEL, BASE, W, F, X0, X1)                                                                         \
    GEO_SC_JUMP_FROM(BASE, F) "s_nop 0\ns_nop 0\ns_nop 0\n" GEO_SC_RIGHT(LABEL, GEO_SC_SEVEN(GEO_SC_SLOT, W, F, X0, X1))
#define GEO_SC_BASE(LABEL, BASE) "s_add_u32 " BASE ", vcc_lo, .Lsc_" LABEL "_%=-.Lsc_pc_%=\n"
// line L of its channel, of eight words or more; AFTER: behind its left half
#define GEO_SC_LEFT(LABEL, BASE, W, F, X0, X1, L, AFTER)                                                               \
    ".Lsc_" LABEL "_left_%=:\n" GEO_SC_EIGHT(GEO_SC_SLOT, W, F, X0, X1)                                                \
    "s_bitcmp1_b32 s[" #F "+0], 11\n"                                                                                  \
    "s_cbranch_scc0 .Lsc_" LABEL "_done_%=\n"                                                                          \
    "s_lshr_b32 s33, %[wo], 1\n"                                                                                       \
    "s_load_dwordx8 s[" #W ":" #W "+7], %[wp], %[wo] offset:64*" #L "\n"                                               \
    "s_load_dwordx4 s[" #F ":" #F "+3], %[ip], s33 offset:32*" #L "\n"                                                 \
    "s_waitcnt lgkmcnt(0)\n"                                                                                           \
    "s_bfe_u32 s33, s[" #F "+0], 3<<16|8\n"                                                                            \
    "s_lshl4_add_u32 vcc_lo, s33, " BASE "\n"                                                                          \
    "s_lshl2_add_u32 vcc_lo, s33, vcc_lo\n"                                                                            \
    "s_add_u32 vcc_lo, vcc_lo, .Lsc_" LABEL "_half_%=-.Lsc_" LABEL "_%=\n"                                             \
    "s_setpc_b64 vcc\n"                                                                                                \
    ".Lsc_" LABEL "_half_%=:\n" GEO_SC_EIGHT(GEO_SC_SLOT, W, F, X0, X1)                                                \
    AFTER                                                                                                              \
    "s_branch .Lsc_" LABEL "_done_%=\n"
// The first lines can be emptier than the rest of the group.  A level rises by 4 with each line of stage B that needs its left half,
// falls by DECAY with each channel (by two for each line of stage B) and not below 0; above 10 the next channels go through another
// loop, DENSE where the stage's last line has fewer than kSkipZeros zero words.  %[cnt]: the level, less DECAY for each channel
// that is left.  A first channel without words in front of full ones, 64 -> 64 at 28 x 28, batch 64, L 128: 289 us, 370 in HALF to
// the end, 294 before any words were skipped.
#define GEO_SC_RISE "s_addk_i32 %[cnt], 4\n"
#define GEO_SC_FALL_IF(DECAY)                                                                                          \
    "s_mul_i32 s33, %[left], " #DECAY "\n"                                                                             \
    "s_add_i32 %[cnt], %[cnt], s33\n"                                                                                  \
    "s_max_i32 %[cnt], %[cnt], 0\n"                                                                                    \
    "s_addk_i32 %[cnt], 4\n"                                                                                           \
    "s_cmp_gt_i32 %[cnt], 10\n"                                                                                        \
    "s_cbranch_scc1 .Lsc_fall_%=\n"                                                                                    \
    "s_sub_i32 %[cnt], %[cnt], s33\n"
// 0 at the first channel of stage B
#define GEO_SC_FALL_COUNT(DECAY, CHANNELS)                                                                             \
    "s_sub_u32 %[cnt], " #CHANNELS ", %[left]\n"                                                                       \
    "s_mul_i32 %[cnt], %[cnt], " #DECAY "\n"
// B: bytes of a channel's lines; F: the first field of the last line's left half; the next channel's words are on their way
#define GEO_SC_FALL(B, F, TO_DENSE, TO_SKIP)                                                                           \
    ".Lsc_fall_%=:\n"                                                                                                  \
    "s_addk_i32 %[wo], " #B "\n" GEO_SC_NEXT_OR_END                                                                    \
    "s_waitcnt lgkmcnt(0)\n"                                                                                           \
    "s_bfe_u32 s34, s[" #F "+0], 3<<16|8\n" GEO_SC_LOADS_FULL                                                          \
    "s_cmp_lt_u32 s34, %[zskip]/3\n"                                                                                   \
    "s_cbranch_scc1 " TO_DENSE "\n"                                                                                    \
    "s_branch " TO_SKIP "\n"
// loads of line L of the channel AT bytes behind %[wo] (in the words; half of it in the fields, s33)
#define GEO_SC_FIELD_OFFSET "s_lshr_b32 s33, %[wo], 1\n"
#define GEO_SC_LOAD(W, F, L)                                                                                           \
    "s_load_dwordx16 s[" #W ":" #W "+15], %[wp], %[wo] offset:64*" #L "\n"                                             \
    "s_load_dwordx8 s[" #F ":" #F "+7], %[ip], s33 offset:32*" #L "\n"
#define GEO_SC_LOAD_HALF(W, F, L, AT)                                                                                  \
    "s_load_dwordx8 s[" #W ":" #W "+7], %[wp], %[wo] offset:" #AT "+64*" #L "+32\n"                                    \
    "s_load_dwordx4 s[" #F ":" #F "+3], %[ip], s33 offset:" #AT "/2+32*" #L "+16\n"
// (the next channel's line: not behind the last one)
#define GEO_SC_LOAD_NEXT(W, F, L)                                                                                      \
    "s_cmp_lt_u32 %[left], 2\n"                                                                                        \
    "s_cbranch_scc1 1f\n"                                                                                              \
    GEO_SC_FIELD_OFFSET GEO_SC_LOAD(W, F, L) "1:\n"
#define GEO_SC_WAIT_ALL "s_waitcnt vmcnt(0) lgkmcnt(0)\n"
#define GEO_SC_WAIT_LINES "s_waitcnt lgkmcnt(0)\n"
#define GEO_SC_FETCH(X, V) "buffer_load_dword %[" X "], %[" V "], %[act], %[co] offen\n"
#define GEO_SC_FETCH4(X) GEO_SC_FETCH(X "0", "v0") GEO_SC_FETCH(X "1", "v1") GEO_SC_FETCH(X "2", "v2") GEO_SC_FETCH(X "3", "v3")
#define GEO_SC_FETCH6(X) GEO_SC_FETCH4(X) GEO_SC_FETCH(X "4", "v4") GEO_SC_FETCH(X "5", "v5")
// to the next channel and its activation words, if there is one; B: bytes of a channel's lines
#define GEO_SC_AHEAD(B, FETCHES)                                                                                       \
    "s_cmp_lt_u32 %[left], 2\n"                                                                                        \
    "s_cbranch_scc1 1f\n"                                                                                              \
    "s_add_u32 %[co], %[co], %[orb]\n"                                                                                 \
    "s_addk_i32 %[wo], " #B "\n"                                                                                       \
    FETCHES "1:\n"
#define GEO_SC_NEXT_OR_END                                                                                             \
    "s_sub_u32 %[left], %[left], 1\n"                                                                                  \
    "s_cmp_eq_u32 %[left], 0\n"                                                                                        \
    "s_cbranch_scc1 99f\n"
// One channel with its words in X, the next one's to Y.
#define GEO_SC_CHANNEL3(LINE, X, Y)                                                                                    \
    GEO_SC_WAIT_ALL GEO_SC_INDEX_OFF GEO_SC_AHEAD(192, GEO_SC_FETCH4(Y)) GEO_SC_INDEX_ON                               \
    LINE(X, 0, 36, 84, X "0", X "1") GEO_SC_LOAD_NEXT(36, 84, 0)                                                       \
    LINE(X, 1, 52, 92, X "1", X "2") GEO_SC_LOAD_NEXT(52, 92, 1)                                                       \
    LINE(X, 2, 68, 24, X "2", X "3") GEO_SC_LOAD_NEXT(68, 24, 2)                                                       \
    GEO_SC_NEXT_OR_END
// (lines 3 and 4 take the place of lines 0 and 1)
#define GEO_SC_CHANNEL5(LINE, X, Y)                                                                                    \
    GEO_SC_WAIT_ALL GEO_SC_INDEX_ON                                                                                    \
    LINE(X, 0, 36, 84, X "0", X "1") GEO_SC_FIELD_OFFSET GEO_SC_LOAD(36, 84, 3)                                        \
    LINE(X, 1, 52, 92, X "1", X "2") GEO_SC_FIELD_OFFSET GEO_SC_LOAD(52, 92, 4)                                        \
    GEO_SC_INDEX_OFF GEO_SC_AHEAD(320, GEO_SC_FETCH6(Y)) GEO_SC_INDEX_ON                                               \
    LINE(X, 2, 68, 24, X "2", X "3") GEO_SC_LOAD_NEXT(68, 24, 2)                                                       \
    GEO_SC_WAIT_LINES                                                                                                  \
    LINE(X, 3, 36, 84, X "3", X "4") GEO_SC_LOAD_NEXT(36, 84, 0)                                                       \
    LINE(X, 4, 52, 92, X "4", X "5") GEO_SC_LOAD_NEXT(52, 92, 1)                                                       \
    GEO_SC_NEXT_OR_END
// the first channel's first line
#define GEO_SC_LINE0                                                                                                   \
    "s_cmp_lg_u32 %[cnt], 0\n"                                                                                         \
    "s_cbranch_scc1 3f\n"                                                                                              \
    GEO_SC_FIRST(36, 84, "x0", "x1")                                                                                   \
    "s_branch 4f\n"                                                                                                    \
    "3:\n" GEO_SC_WHOLE(36, 84, "x0", "x1") "4:\n"
// the first channel in front of DENSE and SKIP: the next one's loads go out as in the loops
#define GEO_SC_FIRST_CHANNEL3                                                                                          \
    GEO_SC_AHEAD(192, GEO_SC_FETCH4("y")) GEO_SC_INDEX_ON                                                              \
    GEO_SC_LINE0 GEO_SC_LOAD_NEXT(36, 84, 0)                                                                           \
    GEO_SC_WHOLE(52, 92, "x1", "x2") GEO_SC_LOAD_NEXT(52, 92, 1)                                                       \
    GEO_SC_WHOLE(68, 24, "x2", "x3") GEO_SC_LOAD_NEXT(68, 24, 2)                                                       \
    GEO_SC_NEXT_OR_END
#define GEO_SC_FIRST_CHANNEL5                                                                                          \
    GEO_SC_INDEX_ON GEO_SC_LINE0 GEO_SC_FIELD_OFFSET GEO_SC_LOAD(36, 84, 3)                                            \
    GEO_SC_WHOLE(52, 92, "x1", "x2") GEO_SC_FIELD_OFFSET GEO_SC_LOAD(52, 92, 4)                                        \
    GEO_SC_INDEX_OFF GEO_SC_AHEAD(320, GEO_SC_FETCH6("y")) GEO_SC_INDEX_ON                                             \
    GEO_SC_WHOLE(68, 24, "x2", "x3") GEO_SC_LOAD_NEXT(68, 24, 2)                                                       \
    GEO_SC_WAIT_LINES                                                                                                  \
    GEO_SC_WHOLE(36, 84, "x3", "x4") GEO_SC_LOAD_NEXT(36, 84, 0)                                                       \
    GEO_SC_WHOLE(52, 92, "x4", "x5") GEO_SC_LOAD_NEXT(52, 92, 1)                                                       \
    GEO_SC_NEXT_OR_END
// the first lines' zero words (bits 11:8 of the first field word) pick the loop for the channels behind the first
#define GEO_SC_COUNT_ZEROS                                                                                             \
    "s_bfe_u32 s35, s84, 0x40008\n"                                                                                    \
    "s_bfe_u32 s33, s92, 0x40008\n"                                                                                    \
    "s_add_u32 s35, s35, s33\n"                                                                                        \
    "s_bfe_u32 s33, s24, 0x40008\n"                                                                                    \
    "s_add_u32 s35, s35, s33\n"
#define GEO_SC_LOADS_FULL GEO_SC_FIELD_OFFSET GEO_SC_LOAD(36, 84, 0) GEO_SC_LOAD(52, 92, 1) GEO_SC_LOAD(68, 24, 2)
#define GEO_SC_LOADS_HALF_A(AT)                                                                                        \
    GEO_SC_LOAD_HALF(36, 84, 0, AT) GEO_SC_LOAD_HALF(44, 88, 1, AT) GEO_SC_LOAD_HALF(52, 92, 2, AT)
// The addresses that SKIP's jumps start from, where the code from here to 99 lies in one 4 GB, otherwise to DENSE; AT: a label's name.
#define GEO_SC_SKIP_BASES(AT, DENSE, BASES)                                                                            \
    "s_getpc_b64 vcc\n"                                                                                                \
    ".Lsc_pc" AT "_%=:\n"                                                                                              \
    "s_add_u32 s33, vcc_lo, 99f-.Lsc_pc" AT "_%=\n"                                                                    \
    "s_cbranch_scc1 " DENSE "\n" BASES
#define GEO_SC_SKIP_BASE(AT, I) "s_add_u32 s[18+" #I "], vcc_lo, .Lsc_sx" #I "_%=-.Lsc_pc" AT "_%=\n"
#define GEO_SC_SKIP_BASES3(AT, DENSE)                                                                                  \
    GEO_SC_SKIP_BASES(AT, DENSE, GEO_SC_SKIP_BASE(AT, 0) GEO_SC_SKIP_BASE(AT, 1) GEO_SC_SKIP_BASE(AT, 2))
#define GEO_SC_SKIP_BASES5(AT, DENSE)                                                                                  \
    GEO_SC_SKIP_BASES(AT, DENSE, GEO_SC_SKIP_BASE(AT, 0) GEO_SC_SKIP_BASE(AT, 1) GEO_SC_SKIP_BASE(AT, 2)               \
                      GEO_SC_SKIP_BASE(AT, 3) GEO_SC_SKIP_BASE(AT, 4))
// The first channel (its first line assigns where `row` is 0), then a loop; each has the channel's words in x or y in turn.
// The order of the code keeps a short DENSE group to one jump, which is under way with its first loads: an instruction fetch
// from a place that no wave of the CU has been to takes longer than a line.
#define GEO_SC_OR_CHANNELS(B, FETCHES, FIRST_CHANNEL, REST_OF_FIRST, CHANNEL, SKIP_BASES, BASES, FALL_COUNT, HALF_LOOP, LEFT_HALVES) \
    "s_nop 4\n" /* the compiler may have written an operand of the loads with a vector instruction just before */      \
    GEO_SC_LOADS_FULL FETCHES                                                                                          \
    "s_branch 7f\n"                                                                                                    \
    /* SKIP, entered at 20 with nothing loaded but the words on their way to x, at 23 and 24 with all on its way, words to x or y */ \
    "24:\n" SKIP_BASES("y", "12f") "s_branch 22f\n"                                                                    \
    "20:\n" GEO_SC_LOADS_FULL                                                                                          \
    "23:\n" SKIP_BASES("x", "13f")                                                                                     \
    "21:\n" CHANNEL(GEO_SC_SKIP, "x", "y") "22:\n" CHANNEL(GEO_SC_SKIP, "y", "x") "s_branch 21b\n"                     \
    /* HALF: its first channel, too, takes whole lines */                                                              \
    "5:\n" GEO_SC_INDEX_ON GEO_SC_LINE0                                                                                \
    GEO_SC_WHOLE(52, 92, "x1", "x2") GEO_SC_WHOLE(68, 24, "x2", "x3") REST_OF_FIRST                                    \
    GEO_SC_NEXT_OR_END GEO_SC_INDEX_OFF                                                                                \
    "s_add_u32 %[co], %[co], %[orb]\n"                                                                                 \
    "s_addk_i32 %[wo], " #B "\n"                                                                                       \
    FETCHES                                                                                                            \
    "s_getpc_b64 vcc\n"                                                                                                \
    ".Lsc_pc_%=:\n"                                                                                                    \
    /* all slots between here and 99 in one 4 GB: a carry takes the other loop */                                      \
    "s_add_u32 s33, vcc_lo, 99f-.Lsc_pc_%=\n"                                                                          \
    "s_cbranch_scc1 20b\n"                                                                                             \
    GEO_SC_FIELD_OFFSET GEO_SC_LOADS_HALF_A(0) BASES FALL_COUNT                                                        \
    ".p2align 5\n31:\n" HALF_LOOP LEFT_HALVES                                                                          \
    "7:\n" GEO_SC_WAIT_ALL GEO_SC_COUNT_ZEROS                                                                          \
    "s_cmp_ge_u32 s35, %[zhalf]\n"                                                                                     \
    "s_cbranch_scc1 5b\n"                                                                                              \
    FIRST_CHANNEL                                                                                                      \
    "s_cmp_ge_u32 s35, %[zskip]\n"                                                                                     \
    "s_cbranch_scc1 24b\n"                                                                                             \
    "12:\n" CHANNEL(GEO_SC_DENSE, "y", "x") "13:\n" CHANNEL(GEO_SC_DENSE, "x", "y") "s_branch 12b\n"                   \
    "99:\n" GEO_SC_INDEX_OFF
#define GEO_SC_OR_OPERANDS                                                                                             \
    [wp] "s"(wp), [ip] "s"(ip), [act] "s"(act), [orb] "s"(or_b), [zskip] "n"(3 * kSkipZeros),                          \
        [zhalf] "n"(3 * kHalfZeros), [v0] "v"(voff[0]), [v1] "v"(voff[1]), [v2] "v"(voff[2]), [v3] "v"(voff[3])
#define GEO_SC_OR_CLOBBERS                                                                                             \
    "m0", "scc", "vcc", "memory", "s18", "s19", "s20", "s21", "s22", "s23", "s24", "s25", "s26", "s27", "s28",         \
    "s29", "s30", "s31", "s33", "s34", "s35", "s36", "s37", "s38", "s39", "s40", "s41", "s42", "s43", "s44",           \
    "s45", "s46", "s47", "s48", "s49", "s50", "s51", "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59",           \
    "s60", "s61", "s62", "s63", "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74",           \
    "s75", "s76", "s77", "s78", "s79", "s80", "s81", "s82", "s83", "s84", "s85", "s86", "s87", "s88", "s89",           \
    "s90", "s91", "s92", "s93", "s94", "s95", "s96", "s97", "s98", "s99"
// Mean zero words per line from which the loops are taken.  SKIP from 1, 2 or 3 on: uniform weights (one line in three has a zero
// word), 128 -> 128 at 16 x 16, batch 256, L 128 1.135 / 1.129 / 1.127 ms; initial weights widened threefold, 64 -> 64 at 32 x 32, batch
// 128, L 128 478 / 486 / 508 us.  HALF from 6, 7 or 8 on: 64 -> 64 at 56 x 56, 30 items, L 256, initial weights 509 / 510 / 511 us, widened
// twofold 674 / 664 / 659.
constexpr int kSkipZeros = 2, kHalfZeros = 7;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// chs >= 1 channels, the first at byte offset ch_off of the stream buffer `act`, or_b bytes apart; wp, ip: their lines.
// row 0: the accumulators are assigned, otherwise added to.
__device__ __forceinline__ void or_channels_rail(const u32x4& act, const unsigned (&voff)[4], unsigned ch_off, unsigned or_b,
                                                 ConstWords wp, ConstWords ip, int chs, int row, u32x16& p0, u32x16& p1,
                                                 u32x16& n0, u32x16& n1)
{
    uint32_t x0, x1, x2, x3, y0, y1, y2, y3;
    unsigned wo = 0, left = (unsigned)chs;
// even channels in stage A, odd ones in stage B; the next channel's lines to the other stage
#define GEO_SC_HALF_CHANNEL3(LOADS, FETCHES)                                                                           \
    GEO_SC_WAIT_ALL GEO_SC_INDEX_OFF                                                                                   \
    "s_cmp_lt_u32 %[left], 2\n"                                                                                        \
    "s_cbranch_scc1 1f\n"                                                                                              \
    "s_add_u32 %[co], %[co], %[orb]\n"                                                                                 \
    GEO_SC_FIELD_OFFSET LOADS FETCHES                                                                                  \
    "1:\n" GEO_SC_INDEX_ON
    asm volatile(
        GEO_SC_OR_CHANNELS(192, GEO_SC_FETCH4("x"), GEO_SC_FIRST_CHANNEL3, "", GEO_SC_CHANNEL3, GEO_SC_SKIP_BASES3,
            GEO_SC_BASE("a0", "s18") GEO_SC_BASE("a1", "s19") GEO_SC_BASE("a2", "s20")
            GEO_SC_BASE("b0", "s21") GEO_SC_BASE("b1", "s22") GEO_SC_BASE("b2", "s23"), GEO_SC_FALL_COUNT(3, 1),
            GEO_SC_HALF_CHANNEL3(GEO_SC_LOAD_HALF(60, 96, 0, 192) GEO_SC_LOAD_HALF(68, 24, 1, 192)
                                 GEO_SC_LOAD_HALF(76, 28, 2, 192), GEO_SC_FETCH4("y"))
            GEO_SC_HALF("a0", "s18", 36, 84, "x0", "x1") GEO_SC_HALF("a1", "s19", 44, 88, "x1", "x2")
            GEO_SC_HALF("a2", "s20", 52, 92, "x2", "x3")
            "s_addk_i32 %[wo], 192\n" GEO_SC_NEXT_OR_END
            GEO_SC_HALF_CHANNEL3(GEO_SC_LOADS_HALF_A(192), GEO_SC_FETCH4("x"))
            GEO_SC_HALF("b0", "s21", 60, 96, "y0", "y1") GEO_SC_HALF("b1", "s22", 68, 24, "y1", "y2")
            GEO_SC_HALF("b2", "s23", 76, 28, "y2", "y3")
            "s_addk_i32 %[wo], 192\n" GEO_SC_NEXT_OR_END
            "s_branch 31b\n",
            GEO_SC_LEFT("a0", "s18", 36, 84, "x0", "x1", 0, "") GEO_SC_LEFT("a1", "s19", 44, 88, "x1", "x2", 1, "")
            GEO_SC_LEFT("a2", "s20", 52, 92, "x2", "x3", 2, "") GEO_SC_LEFT("b0", "s21", 60, 96, "y0", "y1", 0, GEO_SC_RISE)
            GEO_SC_LEFT("b1", "s22", 68, 24, "y1", "y2", 1, GEO_SC_RISE) GEO_SC_LEFT("b2", "s23", 76, 28, "y2", "y3", 2, GEO_SC_FALL_IF(3))
            GEO_SC_FALL(192, 28, "13f", "23b"))
        : "+{v[32:47]}"(p0), "+{v[48:63]}"(p1), "+{v[64:79]}"(n0), "+{v[80:95]}"(n1), [x0] "=&v"(x0), [x1] "=&v"(x1),
          [x2] "=&v"(x2), [x3] "=&v"(x3), [y0] "=&v"(y0), [y1] "=&v"(y1), [y2] "=&v"(y2), [y3] "=&v"(y3),
          [co] "+&s"(ch_off), [wo] "+&s"(wo), [left] "+&s"(left), [cnt] "+&s"(row)
        : GEO_SC_OR_OPERANDS
        : GEO_SC_OR_CLOBBERS);
}

__device__ __forceinline__ void or_channels_rail(const u32x4& act, const unsigned (&voff)[6], unsigned ch_off, unsigned or_b,
                                                 ConstWords wp, ConstWords ip, int chs, int row, u32x16& p0, u32x16& p1,
                                                 u32x16& n0, u32x16& n1)
{
    uint32_t x0, x1, x2, x3, x4, x5, y0, y1, y2, y3, y4, y5;
    unsigned wo = 0, left = (unsigned)chs;
    // HALF: lines 0 - 2 of a channel in stage A, lines 3 and 4 in stage B; the channel's words in x, the next one's to y
    asm volatile(
        GEO_SC_OR_CHANNELS(320, GEO_SC_FETCH6("x"), GEO_SC_FIRST_CHANNEL5,
            GEO_SC_FIELD_OFFSET GEO_SC_LOAD(36, 84, 3) GEO_SC_LOAD(52, 92, 4) GEO_SC_WAIT_LINES
            GEO_SC_WHOLE(36, 84, "x3", "x4") GEO_SC_WHOLE(52, 92, "x4", "x5"),
            GEO_SC_CHANNEL5, GEO_SC_SKIP_BASES5,
            GEO_SC_BASE("a0", "s18") GEO_SC_BASE("a1", "s19") GEO_SC_BASE("a2", "s20")
            GEO_SC_BASE("b0", "s21") GEO_SC_BASE("b1", "s22"), GEO_SC_FALL_COUNT(4, 0),
            GEO_SC_WAIT_ALL
            GEO_SC_FIELD_OFFSET GEO_SC_LOAD_HALF(60, 96, 3, 0) GEO_SC_LOAD_HALF(68, 24, 4, 0)
            "s_cmp_lt_u32 %[left], 2\n"
            "s_cbranch_scc1 1f\n"
            "s_add_u32 %[co], %[co], %[orb]\n"
            GEO_SC_FETCH6("y")
            "1:\n" GEO_SC_INDEX_ON
            GEO_SC_HALF("a0", "s18", 36, 84, "x0", "x1") GEO_SC_HALF("a1", "s19", 44, 88, "x1", "x2")
            GEO_SC_HALF("a2", "s20", 52, 92, "x2", "x3")
            GEO_SC_WAIT_LINES
            "s_cmp_lt_u32 %[left], 2\n"
            "s_cbranch_scc1 1f\n"
            GEO_SC_FIELD_OFFSET GEO_SC_LOADS_HALF_A(320)
            "1:\n"
            GEO_SC_HALF("b0", "s21", 60, 96, "x3", "x4") GEO_SC_HALF("b1", "s22", 68, 24, "x4", "x5")
            "s_addk_i32 %[wo], 320\n" GEO_SC_NEXT_OR_END
            GEO_SC_INDEX_OFF
            "s_waitcnt vmcnt(0)\n"
            "v_mov_b32 %[x0], %[y0]\n"
            "v_mov_b32 %[x1], %[y1]\n"
            "v_mov_b32 %[x2], %[y2]\n"
            "v_mov_b32 %[x3], %[y3]\n"
            "v_mov_b32 %[x4], %[y4]\n"
            "v_mov_b32 %[x5], %[y5]\n"
            "s_branch 31b\n",
            GEO_SC_LEFT("a0", "s18", 36, 84, "x0", "x1", 0, "") GEO_SC_LEFT("a1", "s19", 44, 88, "x1", "x2", 1, "")
            GEO_SC_LEFT("a2", "s20", 52, 92, "x2", "x3", 2, "") GEO_SC_LEFT("b0", "s21", 60, 96, "x3", "x4", 3, GEO_SC_RISE)
            GEO_SC_LEFT("b1", "s22", 68, 24, "x4", "x5", 4, GEO_SC_FALL_IF(4))
            GEO_SC_FALL(320, 24, "12f", "24b"))
        : "+{v[32:47]}"(p0), "+{v[48:63]}"(p1), "+{v[64:79]}"(n0), "+{v[80:95]}"(n1), [x0] "=&v"(x0), [x1] "=&v"(x1),
          [x2] "=&v"(x2), [x3] "=&v"(x3), [x4] "=&v"(x4), [x5] "=&v"(x5), [y0] "=&v"(y0), [y1] "=&v"(y1), [y2] "=&v"(y2),
          [y3] "=&v"(y3), [y4] "=&v"(y4), [y5] "=&v"(y5), [co] "+&s"(ch_off), [wo] "+&s"(wo), [left] "+&s"(left), [cnt] "+&s"(row)
        : GEO_SC_OR_OPERANDS, [v4] "v"(voff[4]), [v5] "v"(voff[5])
        : GEO_SC_OR_CLOBBERS);
}

// The HALF way for a group of 16 one-wide lines (the linear layer in OR groups of 16), unrolled, accumulators at v[64:127],
// cleared by the caller.  Stages of three lines, the last of one: lines A, A + 1, A + 2 in the registers of stage A or B, their
// activation words in x or y (two items per lane).
#define GEO_SC_SLOT64(SET, W, I, X0, X1)                                                                               \
    SET "v_and_or_b32 v64, s[" #W "+" #I "], %[" X0 "], v64\n"                                                          \
        "v_and_or_b32 v65, s[" #W "+" #I "], %[" X1 "], v65\n"
// Loads.  %[wp], %[ip]: the group's right halves by themselves, 32 bytes per line of the words and 16 of the fields; %[wl],
// %[il]: its whole lines.  The scalar cache's misses bound this loop (four waves of a SIMD with a line sequence of their own
// each): of whole lines, half of every 64 bytes unused, the 4096 x 4096 layer at batch 1024 takes 2.33 ms, of these 1.4.
#define GEO_SC_X16(W, BASE, AT) "s_load_dwordx16 s[" #W ":" #W "+15], %[" BASE "], " #AT "\n"
#define GEO_SC_X8(W, BASE, AT) "s_load_dwordx8 s[" #W ":" #W "+7], %[" BASE "], " #AT "\n"
#define GEO_SC_X4(W, BASE, AT) "s_load_dwordx4 s[" #W ":" #W "+3], %[" BASE "], " #AT "\n"
// three lines from line L on, to stage A or B
#define GEO_SC_HALVES_A(L)                                                                                             \
    GEO_SC_X16(36, "wp", 32*L) GEO_SC_X8(52, "wp", 32*L+64) GEO_SC_X8(84, "ip", 16*L) GEO_SC_X4(92, "ip", 16*L+32)
#define GEO_SC_HALVES_B(L)                                                                                             \
    GEO_SC_X16(60, "wp", 32*L) GEO_SC_X8(76, "wp", 32*L+64) GEO_SC_X4(96, "ip", 16*L) GEO_SC_X8(24, "ip", 16*L+16)
#define GEO_SC_HALF16(LABEL, W, F, X0, X1)                                                                             \
    GEO_SC_JUMP(F, 3) GEO_SC_RIGHT(LABEL, GEO_SC_SEVEN(GEO_SC_SLOT64, W, F, X0, X1))
#define GEO_SC_LEFT16(LABEL, W, F, X0, X1, L)                                                                          \
    ".Lsc_" LABEL "_left_%=:\n" GEO_SC_EIGHT(GEO_SC_SLOT64, W, F, X0, X1)                                              \
    "s_bitcmp1_b32 s[" #F "+0], 11\n"                                                                                  \
    "s_cbranch_scc0 .Lsc_" LABEL "_done_%=\n"                                                                          \
    "s_load_dwordx8 s[" #W ":" #W "+7], %[wl], 64*" #L "\n"                                                            \
    "s_load_dwordx4 s[" #F ":" #F "+3], %[il], 32*" #L "\n"                                                            \
    "s_waitcnt lgkmcnt(0)\n"                                                                                           \
    GEO_SC_JUMP(F, 3) GEO_SC_EIGHT(GEO_SC_SLOT64, W, F, X0, X1)                                                        \
    "s_branch .Lsc_" LABEL "_done_%=\n"
// N + 0, N + 1, N + 2 name the lines' labels
#define GEO_SC_LINES16_A(N)                                                                                            \
    GEO_SC_INDEX_ON GEO_SC_HALF16(#N "p0", 36, 84, "x0", "x1") GEO_SC_HALF16(#N "p1", 44, 88, "x2", "x3")              \
    GEO_SC_HALF16(#N "p2", 52, 92, "x4", "x5") GEO_SC_INDEX_OFF
#define GEO_SC_LINES16_B(N)                                                                                            \
    GEO_SC_INDEX_ON GEO_SC_HALF16(#N "p0", 60, 96, "y0", "y1") GEO_SC_HALF16(#N "p1", 68, 24, "y2", "y3")              \
    GEO_SC_HALF16(#N "p2", 76, 28, "y4", "y5") GEO_SC_INDEX_OFF
#define GEO_SC_LEFT16_A(N)                                                                                             \
    GEO_SC_LEFT16(#N "p0", 36, 84, "x0", "x1", N) GEO_SC_LEFT16(#N "p1", 44, 88, "x2", "x3", (N + 1))                  \
    GEO_SC_LEFT16(#N "p2", 52, 92, "x4", "x5", (N + 2))
#define GEO_SC_LEFT16_B(N)                                                                                             \
    GEO_SC_LEFT16(#N "p0", 60, 96, "y0", "y1", N) GEO_SC_LEFT16(#N "p1", 68, 24, "y2", "y3", (N + 1))                  \
    GEO_SC_LEFT16(#N "p2", 76, 28, "y4", "y5", (N + 2))
// FX(N), FY(N): the activation words of lines N, N + 1, N + 2 to x and y; FY1(N): of line N
#define GEO_SC_LINES16(WAIT, FX, FY, FY1)                                                                              \
    "s_nop 4\n" GEO_SC_HALVES_A(0) FX(0)                                                                               \
    WAIT GEO_SC_HALVES_B(3) FY(3) GEO_SC_LINES16_A(0)                                                                 \
    WAIT GEO_SC_HALVES_A(6) FX(6) GEO_SC_LINES16_B(3)                                                                 \
    WAIT GEO_SC_HALVES_B(9) FY(9) GEO_SC_LINES16_A(6)                                                                 \
    WAIT GEO_SC_HALVES_A(12) FX(12) GEO_SC_LINES16_B(9)                                                               \
    WAIT GEO_SC_X8(60, "wp", 480) GEO_SC_X4(96, "ip", 240) FY1(15) GEO_SC_LINES16_A(12)                             \
    WAIT GEO_SC_INDEX_ON GEO_SC_HALF16("15p0", 60, 96, "y0", "y1")                                                     \
    "s_branch 99f\n"                                                                                                   \
    GEO_SC_LEFT16_A(0) GEO_SC_LEFT16_B(3) GEO_SC_LEFT16_A(6) GEO_SC_LEFT16_B(9) GEO_SC_LEFT16_A(12)                    \
    GEO_SC_LEFT16("15p0", 60, 96, "y0", "y1", 15)                                                                      \
    "99:\n" GEO_SC_INDEX_OFF

// OR of one (pack, add group) pair over share `share` of `shares` of the group's channels, assigned to the
// accumulators; false where the share has no channels (nothing is assigned then).
template <int WK, int CU>
__device__ __forceinline__ bool or_pair(const FwdParams& q, __amdgpu_buffer_rsrc_t act, const unsigned (&voff)[WK + 1],
                                        int cot, int pv, int share, int shares, u32x16& p0, u32x16& p1, u32x16& n0,
                                        u32x16& n1)
{
    constexpr int C = kCoTile, NW = WK + 1;
    const unsigned plane_b = 4u * q.act_plane, add_b = 4u * q.add_stride, or_b = 4u * q.or_stride;
    const int groups = q.add_outer * q.add_inner;
    const int p = pv / groups;
    const int go = (pv - p * groups) / q.add_inner;
    const int gi = pv - p * groups - go * q.add_inner;
    const int ch0 = go * q.or_ch_per_group;
    const int chs = min(q.or_ch_per_group, q.or_ch_total - ch0);
    const int chunk = (chs + shares - 1) / shares;
    const int c_begin = min(chs, chunk * share), c_end = min(chs, chunk * (share + 1));
    if (c_begin == c_end) return false;
    // the buffer resource as words, for the asm blocks
    const unsigned long long act_base = (unsigned long long)q.act;
    const u32x4 act_words = {(uint32_t)act_base, (uint32_t)(act_base >> 32), 4u * (unsigned)q.n * (unsigned)q.packs * q.act_plane,
                             0x00020000u};
    const size_t lines_per_pack = (size_t)q.or_rows * q.add_inner * q.or_ch_total * q.w_k;
    const size_t line = p * lines_per_pack + (size_t)ch0 * q.add_inner * q.w_k + (size_t)gi * chs * q.w_k;
    bool first = true;
    const unsigned group_off = (unsigned)p * plane_b + (unsigned)gi * add_b + (unsigned)(ch0 + c_begin) * or_b;
    for (int row = 0; row < q.or_rows; row++) {
        RailLines rl(q, cot, line + ((size_t)row * chs + c_begin) * WK);
        unsigned ch_off = group_off + 4u * (unsigned)row;  // next kernel row: one word further
        if constexpr (WK == 3 || WK == 5) {
            or_channels_rail(act_words, voff, ch_off, or_b, rl.w, rl.f, c_end - c_begin, row, p0, p1, n0, n1);
            continue;
        }
        auto channels_of = [&](auto cu_tag, auto first_tag) {
            constexpr int N = decltype(cu_tag)::value;
            constexpr bool FIRST = decltype(first_tag)::value;
            uint32_t aw[N][NW];
#pragma unroll
            for (int cu = 0; cu < N; cu++)
#pragma unroll
                for (int j = 0; j < NW; j++)
                    aw[cu][j] = __builtin_amdgcn_raw_buffer_load_b32(act, (int)voff[j], (int)(ch_off + (unsigned)cu * or_b), 0);
            uint32_t wv[N * WK][C], iv[N * WK][C / 2];
            rl.load(wv, iv);
#pragma unroll
            for (int cu = 0; cu < N; cu++)
#pragma unroll
                for (int u = 0; u < WK; u++) {
                    if (FIRST && cu == 0 && u == 0)
                        rail_line_first_lo(p0, p1, n0, n1, wv[0], iv[0], aw[0][0], aw[0][1]);
                    else
                        rail_line_lo(p0, p1, n0, n1, wv[cu * WK + u], iv[cu * WK + u], aw[cu][u], aw[cu][u + 1]);
                }
            rl.advance(N * WK);
            ch_off += (unsigned)N * or_b;
        };
        auto channels = [&](auto cu_tag) {
            if (first)
                channels_of(cu_tag, std::true_type());
            else
                channels_of(cu_tag, std::false_type());
            first = false;
        };
        int ci = c_begin;
        for (; ci + CU <= c_end; ci += CU) channels(std::integral_constant<int, CU>());
        if constexpr (CU > 1)
            for (; ci < c_end; ci++) channels(std::integral_constant<int, 1>());
    }
    return true;
}

// k_conv_fwd_split_rail for launches in which every wave sums exactly one (pack, add group) pair (blockIdx.y =
// the pair) and which are more than a round of waves.  Without running sums a wave needs 96 registers instead of
// 128 - the 64 accumulators sit at v[32:95], the counts go from the popcounts straight into the atomics - so
// five waves fit a SIMD instead of four.
// Two waves per workgroup, each with a tile of its own: a CU takes at most 16 workgroups, which single-wave
// workgroups would hit at four waves per SIMD.
constexpr int kPairWaves = 2;
template <int WK, int CU>
__global__ __launch_bounds__(64 * kPairWaves) __attribute__((amdgpu_waves_per_eu(5, 5)))
void k_conv_fwd_pair_rail(FwdParams q, unsigned n_tiles)
{
    constexpr int C = kCoTile;
    const int wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned tile = blockIdx.x * kPairWaves + wave_in_wg;
    if (tile >= n_tiles) return;
    const int cot = tile % q.n_cotile;
    const PairLane<WK + 1> at(q, (long long)(tile / q.n_cotile) * 64 + (threadIdx.x & 63));
    const __amdgpu_buffer_rsrc_t act = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(q.act), 0, (int)(4u * (unsigned)q.n * (unsigned)q.packs * q.act_plane), 0x00020000);
    u32x16 p0, p1, n0, n1;  // written by the group's first line
    or_pair<WK, CU>(q, act, at.voff, cot, blockIdx.y, 0, 1, p0, p1, n0, n1);
    if (!at.live) return;
    const size_t out_plane = (size_t)q.wo * q.ho;
    int32_t* yo = q.y + ((size_t)at.n * q.c_out + (size_t)cot * C) * out_plane + (size_t)at.a0 * q.ho + at.b;
    const bool row1 = at.a0 + 1 < q.wo;
    // accumulator (channel c, row r) is element 2 c + r of the 32: p0 / n0 hold channels 0 - 7, p1 / n1 8 - 15
#pragma unroll
    for (int c = 0; c < C; c++) {
        if (cot * C + c >= q.c_out) break;
        const u32x16& pv16 = c < C / 2 ? p0 : p1;
        const u32x16& nv16 = c < C / 2 ? n0 : n1;
        const int e = 2 * (c % (C / 2));
        atomicAdd(yo + (size_t)c * out_plane, __popc(pv16[e]) - __popc(nv16[e]));  // integer adds: order does not matter
        if (row1) atomicAdd(yo + (size_t)c * out_plane + q.ho, __popc(pv16[e + 1]) - __popc(nv16[e + 1]));
    }
}

// The kernel of most launches: a workgroup owns one tile (64 lane slots x 16 channels) and works on
// blockDim / (64 or_shares) pairs at a time, `or_shares` waves to a pair, `pairs_per_slot` pairs one after the other.
// Bound by the issue rate of v_and_or_b32 where the launch fills the GPU; what decides then is the number of
// waves a SIMD can choose from, as every wave waits for its channel's words and weight lines before it can issue
// their 96 and-ors (3 lines): the counts are summed in LDS (ds_add_u32) instead of in 32 registers, so
// that five waves fit a SIMD.  128 -> 128 channels, 3 x 3, 16 x 16, batch 256, L 128: 1.13 ms; with the sums in
// registers (four waves) 1.38, and 1.29 with the activation words of four c_out tiles staged through LDS besides,
// which this kernel replaced; 64 -> 64 at 56 x 56, L 256, batch 30: 0.95 -> 0.87.
// or_shares > 1, for launches with too few (tile, pair) waves: an OR can be cut anywhere, so every wave of a pair
// takes a share of the channels and the partial words meet in LDS (ds_or_b32).  512 -> 512 channels, L 128:
// 4 x 4 images, batch 50: 474 -> 300 us, batch 128: 924 -> 605; 2 x 2, batch 50: 1760 -> 190 (where lanes ran
// over the members); 32 -> 32, 5 x 5, 16 x 16, one image: 27 -> 12.
// With one row of blocks the sums are stored (no zeroing launch, no global atomics); with more they are added to
// the zeroed y.
// Dynamic LDS: 32 x 64 sums, and with or_shares > 1 a 64 x 64 OR buffer per pair in flight.
constexpr int kTileWaves = 16;
template <int WK, int CU>
__global__ __launch_bounds__(64 * kTileWaves) __attribute__((amdgpu_waves_per_eu(5, 5)))
void k_conv_fwd_tile_rail(FwdParams q)
{
    constexpr int C = kCoTile;
    // all cache lines of the arguments in one round of loads, where the compiler's order takes four (see k_weight_streams):
    // 9.26 -> 9.08 us in a graph, 3 -> 32 channels, 3 x 3, 32 x 32, batch 32, L 64
    asm volatile("" ::"s"(q.act), "s"(q.wgt_rail), "s"(q.n), "s"(q.n_cotile), "s"(q.act_plane), "s"(q.or_stride), "s"(q.or_shares));
    extern __shared__ uint32_t tile_lds[];
    int* red = reinterpret_cast<int*>(tile_lds);  // [2 c + r][lane]
    uint32_t* orb = tile_lds + 2 * C * 64;        // [pair][rail][2 c + r][lane]
    const int waves = blockDim.x >> 6, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int shares = q.or_shares, in_flight = waves / shares;
    const int mine = wave / shares, share = wave - mine * shares;
    const int lds_words = 2 * C * 64 + (shares > 1 ? in_flight * 4 * C * 64 : 0);
    for (int i = threadIdx.x; i < lds_words; i += blockDim.x) tile_lds[i] = 0;
    __syncthreads();
    const int cot = blockIdx.x % q.n_cotile;
    const PairLane<WK + 1> at(q, (long long)(blockIdx.x / q.n_cotile) * 64 + lane);
    const __amdgpu_buffer_rsrc_t act = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(q.act), 0, (int)(4u * (unsigned)q.n * (unsigned)q.packs * q.act_plane), 0x00020000);
    const int pairs = q.packs * q.add_outer * q.add_inner;
    for (int it = 0; it < q.pairs_per_slot; it++) {
        const int pv = (blockIdx.y * q.pairs_per_slot + it) * in_flight + mine;
        u32x16 p0, p1, n0, n1;  // written by the group's first line
        if (pv < pairs && or_pair<WK, CU>(q, act, at.voff, cot, pv, share, shares, p0, p1, n0, n1)) {
            if (shares == 1) {
#pragma unroll
                for (int e = 0; e < C; e++) {  // results unused: ds_add_u32
                    atomicAdd(&red[e * 64 + lane], __popc(p0[e]) - __popc(n0[e]));
                    atomicAdd(&red[(C + e) * 64 + lane], __popc(p1[e]) - __popc(n1[e]));
                }
            } else {
                uint32_t* o = orb + mine * (4 * C * 64) + lane;
#pragma unroll
                for (int e = 0; e < C; e++) {
                    atomicOr(o + e * 64, p0[e]);
                    atomicOr(o + (C + e) * 64, p1[e]);
                    atomicOr(o + (2 * C + e) * 64, n0[e]);
                    atomicOr(o + (3 * C + e) * 64, n1[e]);
                }
            }
        }
        if (shares > 1) {
            __syncthreads();
            // element e of the 32 belongs to one wave: it counts, sums and clears for the next pairs
            for (int e = wave; e < 2 * C; e += waves) {
                int d = red[e * 64 + lane];
                for (int s = 0; s < in_flight; s++) {
                    uint32_t* o = orb + s * (4 * C * 64) + e * 64 + lane;
                    d += __popc(o[0]) - __popc(o[2 * C * 64]);
                    o[0] = 0;
                    o[2 * C * 64] = 0;
                }
                red[e * 64 + lane] = d;
            }
            if (it + 1 < q.pairs_per_slot) __syncthreads();
        }
    }
    __syncthreads();
    if (!at.live) return;
    const size_t out_plane = (size_t)q.wo * q.ho;
    int32_t* yo = q.y + ((size_t)at.n * q.c_out + (size_t)cot * C) * out_plane + (size_t)at.a0 * q.ho + at.b;
    for (int e = wave; e < 2 * C; e += waves) {
        const int c = e >> 1, r = e & 1;
        if (cot * C + c >= q.c_out || at.a0 + r >= q.wo) continue;
        int32_t* dst = yo + (size_t)c * out_plane + (size_t)r * q.ho;
        if (gridDim.y == 1)
            *dst = red[e * 64 + lane];
        else
            atomicAdd(dst, red[e * 64 + lane]);  // integer adds: order does not matter
    }
}

// The rail-skipping kernel for item-innermost activation streams (y mode, outputs with a single row: the
// SC-linear mapping, classifier layers) as a workgroup of S waves that share 128 items x 16 channels:
// every wave sums a contiguous range of (pack, kernel row) groups, the partial sums meet in LDS
// (ds_add_u32), and the workgroup stores the finished counts, channel fastest, so that the 16 channels of
// an item leave as one 64-byte run when the output has a single position (y is then (N, Cout)).  No
// zeroing pass over y, no global atomics.
// Everything that moves between groups is scalar: the activation words are read with buffer loads
// (resource over the whole stream buffer, per-lane byte offset of the lane's two items, the line's
// offset as the scalar operand), the rail-packed weight lines of a c_out tile follow each other in the
// order of the loop, so the two weight pointers only ever advance.
// Weight lines are a stream without reuse inside a wave (the 4096 x 4096 layer: 403 MB for 256 c_out
// tiles): every kTouchGroups groups the wave touches the lines of the groups after those with one vector
// load per 128 bytes, so that the scalar loads that follow find them in L2.
constexpr int kTouchGroups = 4;
template <int WK, int CU, int S>
__global__ __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_conv_fwd_items_rail_wg(FwdParams q)
{
    constexpr int C = kCoTile, R = 2;
    __shared__ int red[R * 64 * C];  // [r][lane][c]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int cot = blockIdx.x % q.n_cotile;
    const long long slot_first = (long long)(blockIdx.x / q.n_cotile) * 64;  // always a live slot
    const long long slot0 = slot_first + lane;
    const bool live = slot0 < q.slots;
    const long long slot = live ? slot0 : slot_first;
    const int b = (int)(slot / q.row_groups);
    const long long n = slot % q.row_groups;
    // lane offsets (bytes) of the two items inside a line's words; an item past the end is clamped to
    // the first one: it only feeds an output that is never stored
    unsigned loff[R];
#pragma unroll
    for (int j = 0; j < R; j++)
        loff[j] = 4u * ((unsigned)b * q.n + (unsigned)n +
                        (n + (long long)j * q.row_groups < q.n ? (unsigned)j * q.row_groups : 0u));
    // byte strides inside the stream buffer [P][c_in][wi][hi][n] (the launcher keeps it under 4 GB)
    const unsigned pack_b = 4u * q.act_plane * (unsigned)q.n;
    const unsigned tap_b = 4u * (unsigned)q.hi * q.n;
    const unsigned row_b = 4u * (unsigned)q.n;
    const unsigned ch_b = 4u * (unsigned)q.wi * q.hi * q.n;
    const __amdgpu_buffer_rsrc_t act = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(q.act), 0,
                                                                          (int)(pack_b * (unsigned)q.packs), 0x00020000);

    int sum[2 * C];  // [2 c + r]
#pragma unroll
    for (int i = 0; i < 2 * C; i++) sum[i] = 0;

    const int k_or = q.c_in * WK;
    const int pv_begin = wave * q.pv_per_block;
    const int pv_end = min(q.packs * q.h_k, pv_begin + q.pv_per_block);
    int v = pv_begin % q.h_k;
    unsigned group_off = (unsigned)(pv_begin / q.h_k) * pack_b + (unsigned)v * row_b;
    RailLines rl(q, cot, (size_t)pv_begin * k_or);
    uint32_t touched = 0;  // used by nothing but the empty asm below, which keeps the loads
    for (int pv = pv_begin; pv < pv_end; pv++) {
        u32x16 p0, p1, n0, n1;  // written by the group's first line
        bool first = true;
        if (((pv - pv_begin) & (kTouchGroups - 1)) == 0) {
            // the lines of groups pv + kTouchGroups .. pv + 2 kTouchGroups - 1: one lane per 128 bytes,
            // first of the words, then of the fields
            asm volatile("" ::"v"(touched));  // the previous touch has long arrived: no wait in practice
            const size_t line = (size_t)(pv + kTouchGroups) * k_or;
            const int w_lanes = kTouchGroups * k_or * C / 32;  // 128-byte pieces of the words
            const bool field = lane >= w_lanes;
            const size_t at = min(line * C + (size_t)(field ? lane - w_lanes : lane) * (field ? 64 : 32), q.rail_lines * C - 2);
            touched = field ? q.wgt_rail_idx[((size_t)cot * q.rail_lines * C + at) / 2]
                            : q.wgt_rail[(size_t)cot * q.rail_lines * C + at];
        }
        unsigned ch_off = group_off;
        auto channels_of = [&](auto cu_tag, auto first_tag) {
            constexpr int N = decltype(cu_tag)::value;
            constexpr bool FIRST = decltype(first_tag)::value;
            uint32_t aw[N][WK][R];
#pragma unroll
            for (int cu = 0; cu < N; cu++)
#pragma unroll
                for (int u = 0; u < WK; u++)
#pragma unroll
                    for (int j = 0; j < R; j++)
                        aw[cu][u][j] = __builtin_amdgcn_raw_buffer_load_b32(
                            act, (int)loff[j], (int)(ch_off + (unsigned)cu * ch_b + (unsigned)u * tap_b), 0);
            uint32_t wv[N * WK][C], iv[N * WK][C / 2];
            rl.load(wv, iv);
#pragma unroll
            for (int cu = 0; cu < N; cu++)
#pragma unroll
                for (int u = 0; u < WK; u++) {
                    if (FIRST && cu == 0 && u == 0)
                        rail_line_first(p0, p1, n0, n1, wv[0], iv[0], aw[0][0][0], aw[0][0][1]);
                    else
                        rail_line(p0, p1, n0, n1, wv[cu * WK + u], iv[cu * WK + u], aw[cu][u][0], aw[cu][u][1]);
                }
            rl.advance(N * WK);
            ch_off += (unsigned)N * ch_b;
        };
        auto channels = [&](auto cu_tag) {
            if (first)
                channels_of(cu_tag, std::true_type());
            else
                channels_of(cu_tag, std::false_type());
            first = false;
        };
        // trips of CU channels, the remainder in trips of two where that avoids a trip of one (16
        // channels with CU = 3: 3 3 3 3 2 2)
        int left = q.c_in;
        if constexpr (CU > 2) {
            while (left >= CU + 2 || left == CU) {
                channels(std::integral_constant<int, CU>());
                left -= CU;
            }
        }
        if constexpr (CU > 1) {
            for (; left >= 2; left -= 2) channels(std::integral_constant<int, 2>());
        }
        for (; left > 0; left--) channels(std::integral_constant<int, 1>());
#pragma unroll
        for (int i = 0; i < C; i++) {
            popc_diff(sum[i], p0[i], n0[i]);
            popc_diff(sum[C + i], p1[i], n1[i]);
        }
        // next (pack, kernel row): one row further, or the first row of the next pack
        group_off += row_b;
        if (++v == q.h_k) {
            v = 0;
            group_off += pack_b - (unsigned)q.h_k * row_b;
        }
    }
    asm volatile("" ::"v"(touched));
    // partial sums of the S waves meet in LDS: wave 0 writes, the others add
    if (wave == 0) {
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int r = 0; r < R; r++) red[(r * 64 + lane) * C + c] = sum[2 * c + r];
    }
    __syncthreads();
    if (wave != 0 && pv_begin < pv_end) {
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int r = 0; r < R; r++) atomicAdd(&red[(r * 64 + lane) * C + c], sum[2 * c + r]);
    }
    __syncthreads();
    const size_t out_plane = (size_t)q.wo * q.ho;
    for (int e = threadIdx.x; e < R * 64 * C; e += 64 * S) {
        const int c = e % C, sl = (e / C) % 64, r = e / (C * 64);
        const long long s_out = slot_first + sl;
        const int co = cot * C + c;
        if (s_out >= q.slots || co >= q.c_out) continue;
        const long long item = s_out % q.row_groups + (long long)r * q.row_groups;
        if (item >= q.n) continue;
        q.y[((size_t)item * q.c_out + co) * out_plane + (size_t)(s_out / q.row_groups)] = red[e];
    }
}

// The item-innermost kernel for OR groups of LPG = 16 one-wide lines (the SC-linear mapping with groups of
// 16 inputs), as one workgroup of 16 waves per (128 items, 8 c_out tiles): wave = (c_out tile, half of
// the (pack, kernel row) groups).  The eight waves of a half read the same activation words: per group
// every wave sends two of the 16 lines straight to LDS (one dword per lane and transfer, in the order of the lanes),
// and all read a line back with one ds_read2st64_b32: an eighth of the vector loads, and what a wave waits for in
// front of a line's 32 vector instructions is LDS and the scalar cache.  Groups are double-buffered: the transfers
// of group t + 1 are under way while group t is computed, and one barrier per group stands behind both.  The
// two halves add their sums in LDS and the workgroup stores 128 items x 128
// channels, 512-byte runs per item.  With 8 position tiles x 32 tile groups (4096 x 4096 at batch 1024)
// that is 256 workgroups, one per CU, in a single round.
// The 256 workgroups walk their weight streams in step (768 KB of lines per group and L2, 384 KB of right halves): a touch two
// groups ahead is still in L2 when its lines are read (every word: 1, 2 or 4 groups ahead 2.99 / 2.92 / 3.26 ms; right halves, with the
// generators: 1.65 / 1.60 / 1.79).
// Mostly empty lines (sampled over the workgroup's tiles) take their right halves only, ahead of their use, from the
// copy that the whole-op forward keeps of them: 4096 x 4096 at batch 1024, initial weights, 0.77 of the words zero: 1.4 ms, 2.33 with halves
// of whole lines, 2.92 with every word.
constexpr int kLinTouchGroups = 2;
// The lane's number, formed anew where it is used: the kernel below fills its 128 registers, and a value that is kept across its
// loops goes to scratch memory, whose loads wait for every load in flight.
__device__ __forceinline__ int fresh_lane()
{
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\nv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
}
// lds: the byte address of the lane's words of line 0, the second item's 256 bytes further, lines 512 bytes apart (x at v[52:57], y at v[58:63])
#define GEO_SC_LDS_FETCH1(V, N) "ds_read2st64_b32 v[" V "], %[lds] offset0:2*(" #N ") offset1:2*(" #N ")+1\n"
#define GEO_SC_LDS_FETCH_X(N)                                                                                          \
    GEO_SC_LDS_FETCH1("52:53", N) GEO_SC_LDS_FETCH1("54:55", N + 1) GEO_SC_LDS_FETCH1("56:57", N + 2)
#define GEO_SC_LDS_FETCH_Y(N)                                                                                          \
    GEO_SC_LDS_FETCH1("58:59", N) GEO_SC_LDS_FETCH1("60:61", N + 1) GEO_SC_LDS_FETCH1("62:63", N + 2)
#define GEO_SC_LDS_FETCH_Y1(N) GEO_SC_LDS_FETCH1("58:59", N)
__device__ __forceinline__ void or_lines16_lds(uint32_t lds, ConstWords wp, ConstWords ip, ConstWords wl, ConstWords il, u32x16& p0, u32x16& p1,
                                               u32x16& n0, u32x16& n1)
{
    uint32_t x0, x1, x2, x3, x4, x5, y0, y1, y2, y3, y4, y5;
    asm volatile(GEO_SC_LINES16(GEO_SC_WAIT_LINES, GEO_SC_LDS_FETCH_X, GEO_SC_LDS_FETCH_Y, GEO_SC_LDS_FETCH_Y1)
                 : "+{v[64:79]}"(p0), "+{v[80:95]}"(p1), "+{v[96:111]}"(n0), "+{v[112:127]}"(n1), [x0] "=&{v52}"(x0),
                   [x1] "=&{v53}"(x1), [x2] "=&{v54}"(x2), [x3] "=&{v55}"(x3), [x4] "=&{v56}"(x4), [x5] "=&{v57}"(x5),
                   [y0] "=&{v58}"(y0), [y1] "=&{v59}"(y1), [y2] "=&{v60}"(y2), [y3] "=&{v61}"(y3), [y4] "=&{v62}"(y4),
                   [y5] "=&{v63}"(y5)
                 : [wp] "s"(wp), [ip] "s"(ip), [wl] "s"(wl), [il] "s"(il), [lds] "v"(lds)
                 : GEO_SC_OR_CLOBBERS);
}
// The lane's two words of consecutive lines from byte address `lds` on.  In front of a plain read the compiler waits for every
// transfer to LDS that is under way, the next group's among them, as it cannot tell the two buffers apart: 4096 x 4096 at batch
// 1024 with every word 3.02 ms instead of 2.92.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void lds_lines(uint32_t (&aw)[3][2], uint32_t lds)
{
    u32x2 a, b, c;
    asm volatile("ds_read2st64_b32 %0, %3 offset1:1\n"
                 "ds_read2st64_b32 %1, %3 offset0:2 offset1:3\n"
                 "ds_read2st64_b32 %2, %3 offset0:4 offset1:5\n"
                 "s_waitcnt lgkmcnt(0)" : "=&v"(a), "=&v"(b), "=&v"(c) : "v"(lds) : "memory");
    aw[0][0] = a.x, aw[0][1] = a.y, aw[1][0] = b.x, aw[1][1] = b.y, aw[2][0] = c.x, aw[2][1] = c.y;
}
__device__ __forceinline__ void lds_lines(uint32_t (&aw)[2][2], uint32_t lds)
{
    u32x2 a, b;
    asm volatile("ds_read2st64_b32 %0, %2 offset1:1\n"
                 "ds_read2st64_b32 %1, %2 offset0:2 offset1:3\n"
                 "s_waitcnt lgkmcnt(0)" : "=&v"(a), "=&v"(b) : "v"(lds) : "memory");
    aw[0][0] = a.x, aw[0][1] = a.y, aw[1][0] = b.x, aw[1][1] = b.y;
}
__global__ __launch_bounds__(64 * kLinTiles * kLinHalves) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_conv_fwd_items_rail_lds(FwdParams q)
{
    constexpr int C = kCoTile, R = 2, LPG = kLinLines, NWV = kLinTiles, G = kLinHalves, LPW = LPG / NWV;
    __shared__ uint32_t stage[G][2][LPG][R][64];     // 32 KB
    __shared__ int red[NWV][R * 64 * C];             // 64 KB
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int cw = wave_all % NWV, half = wave_all / NWV;
    const int cot_groups = q.n_cotile / NWV;
    const int cot = (blockIdx.x % cot_groups) * NWV + cw;
    const long long slot_first = (long long)(blockIdx.x / cot_groups) * 64;  // always a live slot
    const long long slot0 = slot_first + lane;
    const long long slot = slot0 < q.slots ? slot0 : slot_first;
    const int b = (int)(slot / q.row_groups);
    const long long n = slot % q.row_groups;
    // lane's byte offset inside a line's words, and which lanes have a second item (others read the first one's words twice: they
    // only feed an output that is never stored)
    const unsigned loff = 4u * ((unsigned)b * q.n + (unsigned)n);
    const unsigned long long second = __ballot(n + (long long)q.row_groups < q.n);
    const unsigned pack_b = 4u * q.act_plane * (unsigned)q.n;
    const unsigned row_b = 4u * (unsigned)q.n;
    const unsigned ch_b = 4u * (unsigned)q.wi * q.hi * q.n;
    const __amdgpu_buffer_rsrc_t act = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(q.act), 0,
                                                                          (int)(pack_b * (unsigned)q.packs), 0x00020000);
    int sum[2 * C];  // [2 c + r]
#pragma unroll
    for (int i = 0; i < 2 * C; i++) sum[i] = 0;

    // this half's groups (the launcher makes the halves equal: every wave meets every barrier)
    const int pv_begin = half * q.pv_per_block;
    const int n_groups = q.pv_per_block;
    int v = pv_begin % q.h_k;
    unsigned group_off = (unsigned)(pv_begin / q.h_k) * pack_b + (unsigned)v * row_b;
    RailLines rl(q, cot, (size_t)pv_begin * LPG);
    const size_t right_at = ((size_t)cot * q.rail_lines + (size_t)pv_begin * LPG) * (C / 2);
    ConstWords right_w = (ConstWords)(q.wgt_right + right_at), right_f = (ConstWords)(q.wgt_right_idx + right_at / 2);
    // The touched values are used by nothing but the empty asm below, which keeps the loads.
    uint32_t touched_w = 0, touched_f = 0;

    // this wave's lines of a group, cw + NWV * i, straight into LDS (a lane's word lands at its dword): 4 registers that
    // hold the words until they are written otherwise cost the loops below their last free ones
    typedef __attribute__((address_space(3))) uint32_t* LdsWords;
    const uint32_t stage_lds = (uint32_t)(uintptr_t)(LdsWords)&stage[half][0][0][0][0];
    auto fetch = [&](unsigned goff, int buf) {
        const unsigned loff1 = loff + (__builtin_amdgcn_inverse_ballot_w64(second) ? 4u * (unsigned)q.row_groups : 0u);
#pragma unroll
        for (int i = 0; i < LPW; i++) {
            const unsigned so = goff + (unsigned)(cw + NWV * i) * ch_b;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(act, (LdsWords)&stage[half][buf][cw + NWV * i][0][0], 4, (int)loff, (int)so, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(act, (LdsWords)&stage[half][buf][cw + NWV * i][1][0], 4, (int)loff1, (int)so, 0, 0);
        }
    };
    // the words are in LDS before any wave passes the barrier
    auto arrive = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    auto next_group = [&]() {
        group_off += row_b;
        if (++v == q.h_k) {
            v = 0;
            group_off += pack_b - (unsigned)q.h_k * row_b;
        }
    };
    // Right halves only where few of 128 lines, sixteen of each of the workgroup's tiles, spread over members, rows and packs, need
    // their left half, and no tile's: the waves meet at barriers, so that they take one choice, and a tile of full lines holds up the
    // others.  1024 items, 4096 outputs, 64 groups of 16, against every word's loop: a fifth of all lines full 0.89 of its time, two in
    // five 1.04, all 1.44; all lines of one tile in eight 1.27.
    bool half_lines = false;
    if (q.wgt_right) {
        const int first_tile = (blockIdx.x % cot_groups) * NWV;
        unsigned long long full[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const unsigned i = (unsigned)(64 * k + lane);
            const size_t line = min((size_t)i * q.rail_lines / 128 + (2 * (i / NWV) + i) % LPG, q.rail_lines - 1);
            const size_t at = (size_t)(first_tile + i % NWV) * q.rail_lines + line;
            full[k] = __ballot((q.wgt_rail_idx[at * (C / 2)] >> 11 & 1u) == 0);  // bits 11:8: the line's zero words
        }
        half_lines = __popcll(full[0]) + __popcll(full[1]) <= 48;
#pragma unroll
        for (int t = 0; t < NWV; t++) {
            const unsigned long long tile = 0x0101010101010101ull << t;
            half_lines &= __popcll(full[0] & tile) + __popcll(full[1] & tile) < 11;
        }
    }
    static_assert(NWV == 8, "every eighth sample is of the same tile");
    fetch(group_off, 0);
    arrive();
    auto walk = [&](auto half_tag) {
    constexpr bool HALF = decltype(half_tag)::value;
    for (int t = 0; t < n_groups; t++) {
        const int buf = t & 1;
        const bool more = t + 1 < n_groups;
        next_group();
        const bool touch = (t & (kLinTouchGroups - 1)) == 0;
        if (touch) asm volatile("" ::"v"(touched_w), "v"(touched_f));  // the previous touch, long there: no wait behind the fetch
        if (more) fetch(group_off, buf ^ 1);
        if (touch) {
            // a lane's 128 bytes of two groups' words and 64 of their fields; further lanes repeat the last
            constexpr int W = HALF ? C / 2 : C;
            const size_t line = (size_t)cot * q.rail_lines +
                                min((size_t)(pv_begin + t + kLinTouchGroups) * LPG, q.rail_lines - kLinTouchGroups * LPG);
            const unsigned piece = 32u * (unsigned)min(fresh_lane(), kLinTouchGroups * LPG * W / 32 - 1);
            touched_w = ((ConstWords)((HALF ? q.wgt_right : q.wgt_rail) + line * W))[piece];
            touched_f = ((ConstWords)((HALF ? q.wgt_right_idx : q.wgt_rail_idx) + line * (W / 2)))[piece >> 1];
        }
        u32x16 p0, p1, n0, n1;  // written by the group's first line
        const uint32_t lane_lds = stage_lds + 4u * (uint32_t)fresh_lane() + (uint32_t)(buf * sizeof(stage[0][0]));
        auto lines = [&](auto n_tag, auto first_tag, int l0) {
            constexpr int N = decltype(n_tag)::value;
            constexpr bool FIRST = decltype(first_tag)::value;
            uint32_t wv[N][C], iv[N][C / 2];
            rl.load(wv, iv);
            uint32_t aw[N][R];
            lds_lines(aw, lane_lds + l0 * 512u);
#pragma unroll
            for (int l = 0; l < N; l++) {
                if (FIRST && l == 0)
                    rail_line_first(p0, p1, n0, n1, wv[0], iv[0], aw[0][0], aw[0][1]);
                else
                    rail_line(p0, p1, n0, n1, wv[l], iv[l], aw[l][0], aw[l][1]);
            }
            rl.advance(N);
        };
        using T3 = std::integral_constant<int, 3>;
        using T2 = std::integral_constant<int, 2>;
        if constexpr (HALF) {
            p0 = p1 = n0 = n1 = 0u;
            or_lines16_lds(lane_lds, right_w, right_f, rl.w, rl.f, p0, p1, n0, n1);
            rl.advance(LPG);
            right_w += LPG * (C / 2);
            right_f += LPG * (C / 4);
        } else {
            lines(T3(), std::true_type(), 0);
            lines(T3(), std::false_type(), 3);
            lines(T3(), std::false_type(), 6);
            lines(T3(), std::false_type(), 9);
            lines(T2(), std::false_type(), 12);
            lines(T2(), std::false_type(), 14);
        }
        static_assert(LPG == 16, "the trips above cover 16 lines");
#pragma unroll
        for (int i = 0; i < C; i++) {
            popc_diff(sum[i], p0[i], n0[i]);
            popc_diff(sum[C + i], p1[i], n1[i]);
        }
        arrive();
    }
    };
    if (half_lines)
        walk(std::true_type());
    else
        walk(std::false_type());

    const int lane_out = fresh_lane();
    // the two halves of a c_out tile add their sums in LDS: half 0 writes, half 1 adds
    if (half == 0) {
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int r = 0; r < R; r++) red[cw][(r * 64 + lane_out) * C + c] = sum[2 * c + r];
    }
    __syncthreads();
    if (half != 0) {
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int r = 0; r < R; r++) atomicAdd(&red[cw][(r * 64 + lane_out) * C + c], sum[2 * c + r]);
    }
    __syncthreads();
    // 128 items x (8 tiles x 16 channels): channel fastest across the tiles, 512-byte runs per item
    const size_t out_plane = (size_t)q.wo * q.ho;
    const int cot_first = (blockIdx.x % cot_groups) * NWV;
    for (int e = wave_all * 64 + lane_out; e < NWV * R * 64 * C; e += 64 * NWV * G) {
        const int c = e % C, tw = (e / C) % NWV, sl = (e / (C * NWV)) % 64, r = e / (C * NWV * 64);
        const long long s_out = slot_first + sl;
        const int co = (cot_first + tw) * C + c;
        if (s_out >= q.slots || co >= q.c_out) continue;
        const long long item = s_out % q.row_groups + (long long)r * q.row_groups;
        if (item >= q.n) continue;
        q.y[((size_t)item * q.c_out + co) * out_plane + (size_t)(s_out / q.row_groups)] = red[tw][(r * 64 + sl) * C + c];
    }
}

// Rail-packed weight lines from the two-rail lines [line][cot][2][16]: word = pos | neg (at most one is non-zero), stored
// [cot][line][slot] with the zero words in front, and a 16-bit field per slot with what the rail kernels move into M0 (rail_slot,
// rail_field).  A thread per channel, so that a line is read and written by 16 consecutive lanes (random generator,
// 17 -> 441 channels, 3 x 3, L 128: 5 us less than a thread per line).
// `both` (one word, cleared by the launcher) is set when a channel of a line has two non-zero rails.
__global__ __launch_bounds__(256) void k_rail_pack(const uint32_t* __restrict__ lines2, uint32_t* __restrict__ words,
                                                   uint16_t* __restrict__ fields, size_t n_lines, int n_cotile,
                                                   uint32_t* __restrict__ both)
{
    constexpr int C = kCoTile;
    const size_t total = n_lines * n_cotile * C;  // whole lines: the lanes of a line take every step together
    const int c = threadIdx.x & (C - 1);
    bool two_rails = false;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
        const size_t l = e / C, line = l / n_cotile, cot = l - line * n_cotile;
        const uint32_t wp = lines2[l * 2 * C + c], wn = lines2[l * 2 * C + C + c];
        two_rails |= wp != 0u && wn != 0u;
        const uint32_t live = (uint32_t)(__ballot((wp | wn) != 0u) >> (threadIdx.x & 48)) & 0xffffu;
        const int at = rail_slot(live, c);
        const size_t dst = (cot * n_lines + line) * C + at;
        words[dst] = wp | wn;
        fields[dst] = (uint16_t)rail_field(live, at, c, wn != 0u);
    }
    if (two_rails) atomicOr(both, 1u);
}

__global__ __launch_bounds__(256) void k_zero_i32(int32_t* __restrict__ p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0;
}

// How a position-parallel launch (R accumulator rows per lane) is cut whose waves keep their sums in registers:
// waves of 64 lane slots per c_out tile, and the (pack, add group) pairs shared out over blockIdx.y.
struct SplitPlan {
    int row_groups;
    long long slots, tiles, waves;
    int pv, splits, pv_per_block;
};
SplitPlan plan_splits(const Geometry& g, int R, bool rows_in_n)
{
    SplitPlan sp;
    sp.row_groups = rows_in_n ? (g.n + R - 1) / R : (g.wo + R - 1) / R;
    sp.slots = rows_in_n ? (long long)sp.row_groups * g.ho : (long long)g.n * sp.row_groups * g.ho;
    sp.tiles = (sp.slots + 63) / 64;
    sp.waves = sp.tiles * g.n_cotile;
    // Fewer than four waves per SIMD (small layers): split the (pack, add group) sum over blockIdx.y until
    // about twelve waves per SIMD exist, so that three resident waves per SIMD stay available through the tail;
    // the partial sums meet in y through integer atomics.
    sp.pv = g.packs * g.add_outer * g.add_inner;
    int splits = 1;
    if (sp.waves < 4096) {
        splits = (int)((12288 + sp.waves - 1) / sp.waves);
        if (splits > sp.pv) splits = sp.pv;
    } else if (g.rail && !rows_in_n) {
        // Equal waves run in rounds of 4096 (four per SIMD): 3.06 rounds take the time of 4.  Splitting the
        // passes 2-, 3- or 4-fold makes the rounds shorter and the last one fuller; taken when it gains more than
        // the atomics cost.
        auto fill = [&](int k) { const double r = (double)sp.waves * k / 4096.0; return r / (double)(long long)(r + 0.999999); };
        double best = fill(1) * 1.08;
        for (int k = 2; k <= 4; k++)
            if (sp.pv % k == 0 && fill(k) > best) {
                best = fill(k);
                splits = k;
            }
    }
    sp.pv_per_block = (sp.pv + splits - 1) / splits;
    sp.splits = (sp.pv + sp.pv_per_block - 1) / sp.pv_per_block;
    return sp;
}

// The rail-skipping launches with two output rows per lane (position-major streams).
enum RailKernel { kRailPlain, kRailSplit, kRailPair, kRailTile };
struct RailPlan {
    RailKernel kernel;
    int shares, in_flight, per_slot;  // kRailTile
    int splits;                       // blockIdx.y
    // the launch adds to y (several blocks or waves hold a part of a count each): y is zeroed in front of it
    bool adds() const { return kernel == kRailSplit || kernel == kRailPair || splits > 1; }
};
constexpr long long kPairRound = 5 * 4 * 256;  // waves of a round with five waves per SIMD
RailPlan plan_rail_unbounded(const Geometry& g, const SplitPlan& sp)
{
    const long long lines = (long long)g.or_rows * g.or_ch_per_group * g.w_k;  // of an OR group
    const long long tiles = sp.waves, pairs = tiles * sp.pv;                   // (tile, pair) waves
    const int pv = sp.pv;
    RailPlan p = {kRailTile, 1, 4, 1, 1};
    // The lines between the forms were set on 2800 launches of random sizes (streams of 32 to 256 bits, kernels of 1, 3 and
    // 5, every accumulation), each timed in some forty forms with every word of a line ORed: what this rule took was 5.4 %
    // over the best form of each on the (geometric) average.  (Only the tile and pair kernels skip zero words.)
    // Short groups, where the 32 LDS additions at the end of a group weigh most, keep their sums in registers
    // once four waves per SIMD exist without splitting a tile (3 -> 32, 5 x 5, 32 x 32, batch 256, L 64: 64 us
    // against 72), where a tile has a single pair (4 -> 11 channels, 1 x 1, 13 x 31, batch 86: 5.3 against 7.1), with a dozen
    // or two of pairs in few tiles, where a wave is alone on its SIMD (16 pairs of 12 lines in 18 tiles: 8.1 against 10.8 as
    // the sixteen waves of a workgroup), or with so many groups per tile that the tile kernel's per-group work shows (z
    // mode, 3 x 3, 1320 groups of 309 tiles: 395 against 439 us; 1220 groups of 116 tiles: 146 against 162).
    const bool y_mode = g.mode == GEO_SC_ACC_Y;
    if (y_mode && tiles >= 4096 && lines <= 24) return {sp.splits == 1 ? kRailPlain : kRailSplit, 0, 0, 0, sp.splits};
    if (y_mode && pv == 1 && lines <= 32) return {kRailPlain, 0, 0, 0, 1};
    if ((lines <= 28 && pv >= 12 && pv <= 24 && pairs < 350) || (lines <= 12 && pairs >= 100000)) return {kRailSplit, 0, 0, 0, sp.splits};
    // Long groups, few of them per tile, in launches whose waves fill their rounds: the counts of a pair go
    // straight to y (64 -> 64, 3 x 3, 32 x 32, batch 128, L 64: 327 us against 336).  With twelve pairs per tile, with
    // image rows shorter than 16 (more lines per atomic), or with groups of under 128 lines (32 -> 16 channels, 3 x 3, L 64,
    // 801 tiles: 65 against 44) the atomics cost more than that gains.
    const long long rounds = (pairs + kPairRound - 1) / kPairRound;
    if (pv <= 10 && g.w_k >= 3 && lines >= 128 && g.ho >= 16 && pairs > 4096 && pairs * 5 >= rounds * kPairRound * 4)
        return {kRailPair, 0, 0, 0, pv};
    const int ch = g.or_ch_per_group;
    if (lines >= 48 && ch >= 4 && pairs < (lines < 96 ? 1024 : lines < 160 ? 1792 : lines >= 256 && pv <= 8 && g.w_k >= 3 ? 11000 : 8192)) {
        // Too few waves: the OR of a group shared out over four, eight or sixteen of them (a workgroup of a
        // multiple of four waves loads the four SIMDs alike: 512 -> 512 at 4 x 4, batch 50: 4 shares 300 us, 3: 337,
        // 6: 392).  Groups of under 160 lines are shared up to one or two waves per SIMD only (22 -> 311 channels at 5 x 3,
        // batch 122, L 128, 66 lines, 4320 pairs: shared 76 us, four pairs side by side 36; 1260 pairs of 156 lines: 32
        // against 41), longer ones as long as the launch is under two rounds (256 -> 256 at 8 x 8, batch 50, L 128: 4800
        // pairs of 768 lines: 266 against 303; 193 -> 360 at 9 x 9, batch 87, L 64: 8556 pairs of 579 lines: 356 against 494).
        p.in_flight = 1;
        p.shares = pairs * 4 >= 2048 || ch < 8 ? 4 : pairs * 8 >= 2048 || ch < 48 ? 8 : 16;
        p.splits = pv;
        // half a round of tiles, groups short enough for the atomics to show: all pairs
        // of a tile in one workgroup (32 -> 64, 5 x 5, 8 x 8, batch 256, L 64: 76 us; 88 with one pair each)
        if (p.shares == 4 && tiles >= 512 && lines < 192 && pv <= 16) {
            p.in_flight = pv > 1 ? 2 : 1;
            p.per_slot = (pv + 1) / 2;
            p.splits = 1;
        }
        return p;
    }
    if (lines <= 64 && tiles < 1024 && pv <= 24) {
        // few short groups
        if (pairs < 512 && ch >= 4 && lines >= 24) {
            p.shares = 4;
            p.in_flight = pv > 1 ? 2 : 1;
        } else {
            // all pairs of a tile in one workgroup where that leaves enough of them
            p.in_flight = pv <= 4 ? 4 : pv <= 8 || pv > 16 || tiles >= 256 ? 8 : 16;
            p.per_slot = tiles >= 128 ? (pv + p.in_flight - 1) / p.in_flight : 1;
        }
    } else {
        // pairs one after the other: fewer additions to y against a longer last round
        p.in_flight = tiles < 64 && pv >= 8 && pairs < 8000 ? 8 : pv <= 2 ? pv : 4;
        const int most = (pv + p.in_flight - 1) / p.in_flight;
        int want = lines >= 256 ? 2 : lines >= 80 ? 4 : lines >= 20 ? (int)(160 / lines) : 8;
        if (want > most) want = most;
        while (want > 1 && tiles * ((most + want - 1) / want) * p.in_flight < kPairRound) want--;
        p.per_slot = want;
    }
    if (pv / p.in_flight / p.per_slot >= 32768) p.per_slot = pv / p.in_flight / 32768 + 1;  // a grid's limit in y
    const int per_block = p.in_flight * p.per_slot;
    p.splits = (pv + per_block - 1) / per_block;
    return p;
}
RailPlan plan_rail(const Geometry& g, const SplitPlan& sp)
{
    const RailPlan p = plan_rail_unbounded(g, sp);
    // a grid has at most 2^32 - 1 threads in x (from 2^24 tiles of four waves on, 137 GB of counts): one wave per tile
    if (p.kernel == kRailTile && sp.waves * 64 * p.shares * p.in_flight > 0xffffffffLL)
        return {g.mode == GEO_SC_ACC_Y && sp.splits == 1 ? kRailPlain : kRailSplit, 0, 0, 0, sp.splits};
    return p;
}

template <int R, int WK, int CU, bool ROWS_IN_N>
int launch(const Geometry& g, FwdParams q, hipStream_t s)
{
    const SplitPlan sp = plan_splits(g, R, ROWS_IN_N);
    q.row_groups = sp.row_groups;
    q.slots = sp.slots;
    const long long tiles = sp.tiles, blocks = sp.waves;
    if (blocks <= 0 || blocks > 0x7fffffffLL) return GEO_SC_ERR_INVALID_ARGUMENT;
    // per-lane word offsets are 32-bit
    if ((unsigned long long)R * g.packs * g.act_plane >= 0xffffffffull) return GEO_SC_ERR_UNSUPPORTED;
    if (ROWS_IN_N != g.act_item_inner) return GEO_SC_ERR_INVALID_ARGUMENT;
    const int pv = sp.pv;
    q.pv_per_block = sp.pv_per_block;
    if constexpr (ROWS_IN_N) {
        static_assert(R == 2 && WK > 0, "item-innermost launches take two items per lane");
        // the kernel addresses the whole stream buffer with 32-bit byte offsets; y mode only
        if ((unsigned long long)g.act_words * 4 >= 0xffffffffull) return GEO_SC_ERR_UNSUPPORTED;
        if (!g.rail || g.mode != GEO_SC_ACC_Y) return GEO_SC_ERR_INVALID_ARGUMENT;  // make_geometry sets both with act_item_inner
        // OR groups of 16 one-wide lines with whole sets of 8 c_out tiles and enough of them to fill the
        // GPU: the workgroup that stages the activation words of its 8 tiles through LDS
        if (WK == 1 && lines16_lds(g)) {
            q.pv_per_block = pv / kLinHalves;
            hipLaunchKernelGGL(k_conv_fwd_items_rail_lds, dim3((unsigned)(tiles * (g.n_cotile / kLinTiles))),
                               dim3(64 * kLinTiles * kLinHalves), 0, s, q);
            return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
        }
        // Eight waves per workgroup share the (pack, kernel row) groups of their 128 items x 16 channels
        // (the 4096 x 4096 layer at batch 1024: 4 or 16 waves 3 - 10 % slower than 8).
        constexpr int S = 8;
        q.pv_per_block = (pv + S - 1) / S;
        hipLaunchKernelGGL((k_conv_fwd_items_rail_wg<WK, CU, S>), dim3((unsigned)blocks), dim3(64 * S), 0, s, q);
        return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
    }
    auto clear_y = [&]() {
        const size_t n_out = (size_t)g.n * g.c_out * g.wo * g.ho;
        const size_t zb = (n_out + 255) / 256;
        hipLaunchKernelGGL(k_zero_i32, dim3((unsigned)(zb > 4096 ? 4096 : zb)), dim3(256), 0, s, q.y, n_out);
    };
    if (g.rail) {
        if constexpr (R == 2 && WK > 0) {
            // two channels per trip for 1-wide kernels: with three, the six address pairs push the 32
            // sums out of the 128 registers
            constexpr int CR = WK == 1 ? 2 : 1;
            const RailPlan rp = plan_rail(g, sp);
            if (rp.adds()) clear_y();
            const dim3 grid((unsigned)blocks, (unsigned)rp.splits);
            if (rp.kernel == kRailPlain)
                hipLaunchKernelGGL((k_conv_fwd_rail<WK, CR>), grid, dim3(64), 0, s, q);
            else if (rp.kernel == kRailSplit)
                hipLaunchKernelGGL((k_conv_fwd_split_rail<WK, CR>), grid, dim3(64), 0, s, q);
            else if (rp.kernel == kRailPair)
                hipLaunchKernelGGL((k_conv_fwd_pair_rail<WK, CR>),
                                   dim3((unsigned)((blocks + kPairWaves - 1) / kPairWaves), (unsigned)rp.splits),
                                   dim3(64 * kPairWaves), 0, s, q, (unsigned)blocks);
            else {
                q.or_shares = rp.shares;
                q.pairs_per_slot = rp.per_slot;
                const size_t lds = sizeof(uint32_t) * 64 * kCoTile * (2 + (rp.shares > 1 ? 4 * rp.in_flight : 0));
                hipLaunchKernelGGL((k_conv_fwd_tile_rail<WK, CR>), grid,
                                   dim3((unsigned)(64 * rp.shares * rp.in_flight)), lds, s, q);
            }
        } else
            return GEO_SC_ERR_INVALID_ARGUMENT;  // make_geometry sets rail for two-row launches only
        return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
    }
    const dim3 grid((unsigned)blocks, (unsigned)sp.splits);
    if (sp.splits == 1 && g.mode == GEO_SC_ACC_Y)
        hipLaunchKernelGGL((k_conv_fwd<R, WK, CU, false>), grid, dim3(64), 0, s, q);
    else {
        clear_y();
        hipLaunchKernelGGL((k_conv_fwd_split<R, WK, CU, false>), grid, dim3(64), 0, s, q);
    }
    return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
}

}  // namespace

// positions per wave of k_conv_fwd_thin: one where waves of two are fewer than the CUs (both sides at 300 random sizes:
// under 128 waves one position is 1.1 - 1.5 times as fast, from 128 to 512 the two are equal, beyond that two positions
// are up to 2 times as fast)
static int thin_positions(const Geometry& g)
{
    const long long positions = (long long)g.n * g.wo * g.ho;
    return (positions + 1) / 2 * g.n_cotile * g.packs * g.add_outer * g.add_inner < 256 ? 1 : 2;
}

double conv_forward_cost(const Geometry& g)
{
    const double pv = (double)g.packs * g.add_outer * g.add_inner;
    if (g.thin || g.act_item_inner || g.wo < 2) {
        // lanes over OR members, or workgroups that share out the pairs themselves: no rounding modelled
        const double waves = ((double)g.n * g.wo * g.ho / 128.0 + 1.0) * g.n_cotile;
        return waves * pv / 4096.0;
    }
    // waves of one pair in rounds of five per SIMD; workgroups retire by themselves, so a round is not all or nothing
    const SplitPlan sp = plan_splits(g, g.rail ? 2 : 1, false);
    const double fifths = std::ceil((double)sp.waves * pv / (kPairRound / 5));
    return fifths < 5 ? 1.0 : fifths / 5;
}

int launch_rail_pack(const Geometry& g, uint32_t* wgt, hipStream_t s, bool from_generator)
{
    if (!g.wgt_rail) return GEO_SC_OK;
    if (from_generator && generator_packs_rails(g)) return GEO_SC_OK;  // written, flag area included, by the generator
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(256), 0, s, reinterpret_cast<int32_t*>(wgt + g.wgt_flag_off), (size_t)64);
    const size_t lines = g.wgt_rail_lines;
    size_t blocks = (lines * g.n_cotile * kCoTile + 255) / 256;
    hipLaunchKernelGGL(k_rail_pack, dim3((unsigned)(blocks > 4096 ? 4096 : blocks)), dim3(256), 0, s, wgt,
                       wgt + g.wgt_rail_off, reinterpret_cast<uint16_t*>(wgt + g.wgt_rail_idx_off), lines, g.n_cotile,
                       wgt + g.wgt_flag_off);
    return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
}

int launch_conv_forward(const Geometry& g, const uint32_t* act, const uint32_t* wgt, int32_t* y, hipStream_t s)
{
    FwdParams q;
    q.act = act;
    q.wgt = wgt;
    q.wgt_rail = g.wgt_rail ? wgt + g.wgt_rail_off : nullptr;
    q.wgt_rail_idx = g.wgt_rail ? wgt + g.wgt_rail_idx_off : nullptr;
    q.wgt_right = g.right_halves ? wgt : nullptr;
    q.wgt_right_idx = g.right_halves ? wgt + right_fields_off(g) : nullptr;
    q.rail_lines = g.wgt_rail_lines;
    q.y = y;
    q.c_in = g.c_in;
    q.wi = g.wi;
    q.hi = g.hi;
    q.c_out = g.c_out;
    q.w_k = g.w_k;
    q.h_k = g.h_k;
    q.packs = g.packs;
    q.wo = g.wo;
    q.ho = g.ho;
    q.n_cotile = g.n_cotile;
    q.act_plane = (unsigned)g.act_plane;
    q.row_groups = 0;
    q.or_shares = q.pairs_per_slot = 0;
    q.slots = 0;
    q.n = g.n;
    q.add_outer = g.add_outer;
    q.add_inner = g.add_inner;
    q.or_ch_total = g.or_ch_total;
    q.or_ch_per_group = g.or_ch_per_group;
    const unsigned ch_plane = (unsigned)g.wi * g.hi;
    q.add_stride = g.mode == GEO_SC_ACC_Z ? ch_plane : 1u;
    q.or_stride = g.mode == GEO_SC_ACC_Z ? 1u : ch_plane;
    q.or_rows = g.or_rows;
    if (g.thin) {
        const long long positions = (long long)g.n * g.wo * g.ho;
        const int per_wave = thin_positions(g);
        const long long blocks = (positions + per_wave - 1) / per_wave * g.n_cotile;
        const long long pv = (long long)g.packs * g.add_outer * g.add_inner;
        if (blocks > 0x7fffffffLL || pv > 65535 || g.act_item_inner) return GEO_SC_ERR_INVALID_ARGUMENT;
        const size_t n_out = (size_t)g.n * g.c_out * g.wo * g.ho;
        size_t zb = (n_out + 255) / 256;
        hipLaunchKernelGGL(k_zero_i32, dim3((unsigned)(zb > 4096 ? 4096 : zb)), dim3(256), 0, s, q.y, n_out);
        auto kernel = per_wave == 1 ? k_conv_fwd_thin<1> : k_conv_fwd_thin<2>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (unsigned)pv), dim3(64), 0, s, q, positions);
        return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
    }
    // Two accumulator rows per lane halve the weight traffic per instruction.  Outputs with
    // several rows take them along dim 2 (sliding-window reuse of activation words); outputs
    // with a single row (the SC-linear mapping, classifier layers) take two batch items.
    if (g.wo >= 2) {
        switch (g.w_k) {
        case 1: return launch<2, 1, 3, false>(g, q, s);
        case 3: return launch<2, 3, 1, false>(g, q, s);
        case 5: return launch<2, 5, 1, false>(g, q, s);
        default: return launch<1, 0, 1, false>(g, q, s);
        }
    }
    if (g.act_item_inner) {
        switch (g.w_k) {
        case 1: return launch<2, 1, 3, true>(g, q, s);
        case 3: return launch<2, 3, 1, true>(g, q, s);
        default: return launch<2, 5, 1, true>(g, q, s);
        }
    }
    switch (g.w_k) {
    case 1: return launch<1, 1, 3, false>(g, q, s);
    case 3: return launch<1, 3, 1, false>(g, q, s);
    case 5: return launch<1, 5, 1, false>(g, q, s);
    default: return launch<1, 0, 1, false>(g, q, s);
    }
}

}  // namespace geo_sc
