// Shared host/device definitions of the SC convolution kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "geo_sc.h"

namespace geo_sc {

// Output channels per weight tile: one tile = 16 positive-rail words + 16 negative-rail
// words = one 128-byte line, fetched by a wave as two scalar 16-dword loads.
constexpr int kCoTile = 16;

// Derived sizes of one problem; filled by make_geometry() after validation.
struct Geometry {
    int n, c_in, w_in, h_in, c_out, w_k, h_k, pad_w, pad_h;
    int L, n_bits, packs, bit_unit;
    int total_width, load_width, load_wait_w, load_wait_a;
    int mode;            // geo_sc_accumulate
    int z_unit;          // YZ: channels per OR group, clamped to c_in; otherwise c_in
    // Loop nest of the accumulation as the kernels walk it: for pack, for outer add group go <
    // add_outer, for inner add group gi < add_inner: OR over (or_ch channels of the group, w_k).
    //   Y : add_outer 1,              add_inner h_k,  OR channels = input channels
    //   YZ: add_outer channel groups, add_inner h_k,  OR channels = the group's input channels
    //   Z : add_outer 1,              add_inner c_in, OR channels = kernel rows (h_k)
    //   FULL: add_outer 1,            add_inner 1,    OR channels = input channels, and the OR also
    //         runs over or_rows = h_k kernel rows before the popcount (Y-mode weight line order)
    int add_outer, add_inner, or_ch_total, or_ch_per_group, or_rows;
    int generator;       // geo_sc_generator
    uint32_t seed;       // random generators
    size_t seed_wrap;    // activation seed index is (flat index % seed_wrap)
    int wi, hi;          // padded activation dims 2 / 3
    int wo, ho;          // output dims 2 / 3
    int k_or;            // OR-group size c_in * w_k
    int n_cotile;        // ceil(c_out / kCoTile)
    size_t act_plane;    // c_in * wi * hi words: one pack of one item
    // Activation stream layout.  false: [n][P][c_in][wi][hi].  true: [P][c_in][wi][hi][n] (batch item
    // innermost), used when the output has a single row so that the convolution kernel's lanes,
    // which then run over batch items, read consecutive words.
    bool act_item_inner;
    // Few output positions but large OR groups (classifier layers): the convolution runs with
    // lanes over the members of an OR group instead of over output positions.
    bool thin;
    size_t act_words;    // n * packs * act_plane
    // Weight stream buffer: lines [packs][h_k][k_or][n_cotile] of 2 x kCoTile words (both rails), then,
    // with rail, the same lines once more in the rail-packed form the plain y-mode kernel reads:
    // at wgt_rail_off kCoTile words per line (the non-zero rail's word, zero words in front), at wgt_rail_idx_off
    // kCoTile / 2 words per line (16 bits per word: rail_field), both ordered [n_cotile][line]
    // with wgt_rail_lines lines per tile.
    // Behind the rail-packed copy: wgt_flag_off, one word that the packing kernel sets when a caller's
    // line carries two non-zero rails for one channel (which the rail-packed form cannot hold), then
    // padding to 64 words.
    size_t wgt_words, wgt_rail_off, wgt_rail_idx_off, wgt_rail_lines, wgt_flag_off;
    // Position-major launches with two output rows per lane run the rail-skipping kernels: per weight
    // at most one rail's stream is non-zero (codes of clamp(w, 0, .) and -clamp(w, ., 0)), and only
    // that rail is processed.  wgt_rail: the weight stream buffer carries the rail-packed copy (a
    // property of the weights' shape alone); rail: this geometry's launch reads it.
    bool wgt_rail, rail;
    // The right halves of the rail-packed lines (slots 8 - 15) are written a second time, by themselves, into the two-rail lines'
    // place (right_words / right_fields): the whole-op forward of one-wide layers with OR groups of 16 lines, none of whose
    // launches reads two-rail lines.
    bool right_halves;
};

// A rail-packed line holds its 16 channels with the zero words in front, in channel order on either side; live: bit c set
// where channel c's word is not zero.  A wave that accumulates the line jumps over the zero words.
__device__ __forceinline__ int rail_slot(uint32_t live, int c)
{
    const int from = (int)__popc(live >> c), below = (int)__popc(~live & ((1u << c) - 1u));
    return (live >> c) & 1u ? kCoTile - from : below;
}
// The 16-bit field of channel c at slot `at`: bits 7:0 the register offset of its accumulators (2 c for the positive rail and
// for zero weights, 32 + 2 c for the negative one), bits 15:12 the SRC2 and DST enables of the VGPR index mode.  Two slots say in
// bits 11:8, which index mode ignores, how a wave reads the line:
//   slot 0: the zero words in front, at most 15: of those before the last slot the wave may jump over as many;
//   slot 8: bits 10:8 the zero words to jump over in the right half (at most 7), bit 11 set where the left half holds others.
// (A line or half without any other ORs one zero word.)
__device__ __forceinline__ uint32_t rail_field(uint32_t live, int at, int c, bool negative)
{
    constexpr int H = kCoTile / 2;
    const int zeros = min(kCoTile - (int)__popc(live), kCoTile - 1);  // (of unsigned and int, min is the one of doubles)
    uint32_t high = 0xC0u;
    if (at == 0) high |= (uint32_t)zeros;
    if (at == H) high |= zeros < H ? (uint32_t)H : (uint32_t)(zeros - H);
    return high << 8 | ((negative ? 2u * kCoTile : 0u) + 2u * (uint32_t)c);
}
static_assert(kCoTile == 16, "rail-packed lines hold 16 channels");

// Stream tables (one per stream length, constant data of the code object):
//   posp1[r], r < L-1 : 1 + index in the LFSR cycle of state r+1  (cycle[0] = 1)
//   thr[code][j]      : bit string, MSB-first, of [code > cycle[j mod (L-1)]] for
//                       j < 32 * words_per_code, long enough to read L bits from any
//                       offset <= L-1 plus one spare word for the funnel shift.
constexpr __host__ __device__ int table_words_per_code(int L) { return (2 * L + 31) / 32 + 2; }
inline __host__ __device__ size_t table_bytes(int L)
{
    return sizeof(uint32_t) * ((size_t)L + (size_t)L * table_words_per_code(L));
}

// k_conv_fwd_items_rail_lds: lines of an OR group, c_out tiles of a workgroup, shares that it cuts the groups into
constexpr int kLinLines = 16, kLinTiles = 8, kLinHalves = 2;
// whether launch_conv_forward takes that kernel: item-innermost, equal shares of the groups, 128 workgroups
inline bool lines16_lds(const Geometry& g)
{
    const long long tiles = ((long long)(g.n + 1) / 2 * g.ho + 63) / 64;
    return g.act_item_inner && g.w_k == 1 && g.c_in == kLinLines && g.n_cotile % kLinTiles == 0 &&
           g.packs * g.h_k % kLinHalves == 0 && tiles * (g.n_cotile / kLinTiles) >= 128;
}
// the right halves' words [n_cotile][line][8] and fields [n_cotile][line][8] of 16 bits, in the place of two-rail lines of 32 words
inline size_t right_fields_off(const Geometry& g) { return g.wgt_rail_lines * g.n_cotile * (kCoTile / 2); }

const uint32_t* stream_tables_host(int L, size_t* words);

int make_geometry(const geo_sc_conv_desc* d, Geometry* g);

// Caller's choices that are not part of the problem (geo_sc_options with its defaults filled in).
struct Options {
    size_t forward_stream_bytes;    // budget of the forward's activation stream buffer
    int backward_groups_per_round;  // cap on the add groups per round of backward launches; 0: none
    bool forward_single_stream;     // a cut batch runs on the caller's stream alone
    int backward_operand_bits;      // significant bits that x and w of the backward are expected to have; 0: not known
};
constexpr size_t kDefaultForwardStreamBytes = (size_t)256 << 20;

// launchers (each returns a geo_sc_status)
// item0: index of x's first item in the whole batch (the random generators number their sequences by it)
int launch_act_streams(const Geometry& g, const float* x, uint32_t* streams, hipStream_t s, size_t item0 = 0);
int launch_act_streams_q7(const Geometry& g, const uint8_t* x_q7, uint32_t* streams, hipStream_t s);
// rail_only: the caller's convolution kernel reads the rail-packed copy only; a generator that writes that
// copy itself may then leave the two-rail lines unwritten
int launch_weight_streams(const Geometry& g, const float* w, uint32_t* streams, hipStream_t s,
                          bool rail_only = false);
int launch_conv_forward(const Geometry& g, const uint32_t* act, const uint32_t* wgt, int32_t* y, hipStream_t s);
// Predicted duration of that launch in units of one wave walking one (pack, add group) pair on a full GPU:
// what the forward compares when it cuts a batch into chunks (waves run in rounds of five per SIMD, so a
// chunk of less than a round costs as much as a round; beyond one the cost is proportional).
double conv_forward_cost(const Geometry& g);
// fills the rail-packed part of a weight stream buffer from its two-rail lines (no-op unless g.wgt_rail;
// with from_generator also where launch_weight_streams has written that part itself)
int launch_rail_pack(const Geometry& g, uint32_t* wgt, hipStream_t s, bool from_generator);
// the LFSR weight generator writes the rail-packed copy (and clears the flag area) itself
inline bool generator_packs_rails(const Geometry& g) { return g.generator == GEO_SC_GEN_LFSR; }
// operand_bits: Options::backward_operand_bits
size_t backward_workspace_bytes(const Geometry& g, int groups_per_round, int operand_bits);
// GEO_SC_ERR_WORKSPACE when workspace_bytes is below backward_workspace_bytes(g, groups_per_round, operand_bits)
int launch_conv_backward(const Geometry& g, int groups_per_round, int operand_bits, const float* x, const float* w,
                         const float* gy, float* gx, float* gw, void* workspace, size_t workspace_bytes, hipStream_t s);

}  // namespace geo_sc
