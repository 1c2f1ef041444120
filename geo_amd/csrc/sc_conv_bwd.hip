// Surrogate-gradient backward of the SC convolution (gfx950, fp32 results, MFMA).
//
// The reference trains through a floating-point surrogate of the SC layer
// (utils_functional.py:611-634, :235-252): with wp = clamp(w,0,100), wn = -clamp(w,-100,0)
// and x the zero-padded activation,
//     z+-_v = corr2d(x[..., v : v+Ho], w+-[..., v:v+1])        (kernel W x 1, one per kernel row v)
//     y^    = sum_v (1 - exp(-z+_v)) - sum_v (1 - exp(-z-_v))
// and autograd differentiates y^.  Written out, with g the upstream gradient:
//     E+-_v      = g * exp(-z+-_v)
//     dL/dx      = sum_v corr2d^T(E+_v, wp_v) - corr2d^T(E-_v, wn_v)
//     dL/dw[..v] = [0 <= w <= 100] * sum x E+_v  +  [-100 <= w <= 0] * sum x E-_v
// (clamp passes its gradient on the closed interval, so both terms are live at w == 0).
//
// Per kernel row v this is three dense fp32 contractions over an im2col view of x:
//     Z  [m][j]  = sum_k col[m][k] * Wcat[k][j]        m=(n,a,b)  k=(ci,u)  j=(rail,co)
//     Gw [k][j]  = sum_m col[m][k] * E[m][j]
//     dcol[k][m] = sum_j Wd[j][k]  * E[m][j]           Wd = (wp ; -wn)
// All three run on MFMA kernels (fp32 in, fp32 accumulate, fp32 out) that take each operand either
// K-major or I-major: k_gemm_split forms every fp32 product from six bf16 MFMA products of a three-way
// split of the operands; k_gemm_big is the same product with eight waves on tiles of up to 256 x 256 for
// the large results.  Rows of col and E are padded to 16 bytes so that sizes that are no multiples of four take
// these kernels too (77 items of 45 x 27 x 19 -> 83 channels, z_unit 32: weight gradient 216 us on
// fp32 MFMAs with element-wise loads, 97 here; input gradient 136, 83);
// exp and the product with g are fused into the first GEMM's epilogue; the second is split over m
// and reduced deterministically.  Where every x and w is a bf16 number, as the 7-bit operands of the layers are
// (k / 128), eleven of the eighteen term products would multiply by zeros: a scan finds that out on the device and the
// products are left out (GemmParams::one_term), the same results bit for bit.  Three products of 64 -> 64 at 56 x 56,
// batch 128: 438 + 411 + 426 -> 349 + 303 + 349 us; 512 -> 512 at 4 x 4, batch 128, first product: 126 -> 61.  Up to 192
// members the first two are one kernel then, k_bwd_e_wgrad: 314 us there.
//
// The other accumulation modes have the same surrogate with other add groups
// (utils_functional.py:254-299): one exponential per add group, whose argument sums the OR
// members of the group.  "Kernel row" above generalises to a group g with members k:
//     Y : g = v,                      k = ci*w_k + u                       (conv2d_or_bin_1d)
//     Z : g = ci,                     k = u*h_k + v                        (conv2d_or_bin_z)
//     YZ: g = (ci / z_unit)*h_k + v,  k = (ci % z_unit)*w_k + u            (conv2d_or_bin_yz)
//     FULL: g = 0,                    k = (ci*w_k + u)*h_k + v             (conv2d_or_approx, :189-210)
// Members of a ragged last channel block that do not exist carry zero weights.
#include "sc_common.h"

#include <cstdint>
#include <cstdlib>

#include <algorithm>
#include <type_traits>

namespace geo_sc {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// exp(-z) of the surrogate's OR term, z >= 0: one multiply and v_exp_f32 (about 1 ulp of the result plus
// |z| 2^-24 from the rounded argument), far inside the gradients' 1e-5; the library expf costs five
// times the instructions and the fused kernels evaluate it once per (position, group, channel, rail)
__device__ __forceinline__ float exp_neg(float z) { return __expf(-z); }

constexpr int kTile = 128;   // block tile in I and J
constexpr int kChunk = 16;   // K per LDS stage

// the three products of the backward: E from col and wcat, the weight gradient from col and E, the input gradient from the
// weights and E
enum Product { PRODUCT_E = 0, PRODUCT_DW = 1, PRODUCT_DX = 2 };

enum Epilogue { EPI_STORE = 0, EPI_EXP_TIMES_G = 1, EPI_EXP_TIMES_G_PLANES = 2, EPI_STORE_ITEMS = 3 };

struct GemmParams {
    const float* __restrict__ a;
    const float* __restrict__ b;
    float* __restrict__ c;
    int I, J, K;              // C[I][J] = sum_k A(k,i) * B(k,j)
    long long lda, ldb, ldc;  // leading dimensions (elements)
    // z = batch * splits + split.  A batch member is one kernel row: its operands
    // and result start batch_stride elements further; a split takes k_per_split of K and
    // writes its own partial result c_split_stride further.
    int splits;
    int k_per_split;
    long long c_split_stride;
    long long a_batch_stride, b_batch_stride, c_batch_stride;
    // EPI_EXP_TIMES_G: c[i][j] = g[i * c_out + (j % c_out)] * exp(-acc), g = upstream gradient stored [m][c_out]
    // EPI_EXP_TIMES_G_PLANES (g_planes set; whole tiles only): the same from the gradient as the caller
    // has it, [n][c_out][npos] with i = n * npos + position; npos a multiple of 32, g 16-byte aligned
    const float* __restrict__ g;
    int c_out, npos, g_planes;
    // A as a view of the shifted input planes instead of a materialised col (kernels with VA): row r of
    // batch member z starts a_rows[z * a_rows_batch + r] elements into `a`, and position m of that row lies
    // m + (m / a_item) * a_skip elements further (a_item positions per item, a_skip elements between the
    // items' runs); lda and a_batch_stride are not used.
    const long long* __restrict__ a_rows;
    long long a_rows_batch;
    int a_item, a_skip;
    // B as a view of E shifted by image rows and columns (kernels with VB; the input-gradient product summed
    // over all sh_wk x sh_hk kernel taps (u, v) inside the GEMM): chunk c of the k dimension holds the columns
    // j = (c / (sh_wk sh_hk)) * kChunk ... of tap t = c % (sh_wk sh_hk), u = t % sh_wk, v = t / sh_wk, and column
    // i = (n, p, c) of B (an element of the input: sh_win rows of sh_hin) is row (n, p + sh_pad - u, c + sh_padh - v)
    // of E_v (sh_j floats per row, ldb apart; E_v starts v * b_batch_stride into b) where that output position
    // exists, zero elsewhere (read from sh_zero).
    const float* __restrict__ sh_zero;
    int sh_j, sh_wo, sh_ho, sh_win, sh_hin, sh_pad, sh_padh, sh_wk, sh_hk;
    // not null (LOOK): a word that says whether every x and w is a bf16 number (k_bwd_prep).  Where it is not zero, the
    // operands made from them are one term of the split instead of three, and the rows that `a` of the first two products
    // points to hold bf16 numbers (the same elements at the same indexes).
    const int* __restrict__ one_term;
    int one_term_elsewhere;  // another kernel (k_bwd_e_wgrad) does this product where they are
    // EPI_STORE_ITEMS: column j = (n, rest) of the result goes to c[(n * I + i) * c_plane + rest] (c_plane
    // columns per item): the input gradient in the caller's layout (n, c_in, w_in, h_in)
    int c_plane;
    // tile extent per workgroup in i and j: kTile, or kTile / 2 in at most one of them (set by
    // launch_gemm): the four waves then line up along the other dimension
    int tile_i, tile_j;
    // Workgroup numbering (set by launch_gemm).  The grid is one-dimensional and the hardware deals
    // consecutive workgroup ids to the 8 XCDs in turn, each with an L2 of its own.  Workgroups that read
    // the same operand tiles form a cluster of `cluster` members (the tiles along the short dimension of
    // the result, or all tiles of one split of a small result); cluster q runs on XCD q % 8 with its members
    // next to each other, so a tile comes from memory once instead of once per member.
    int ni, nj, nz;  // tiles in i and j, batch * splits
    int cluster;     // members per cluster
    int cluster_of;  // 0: members = j tiles of one i tile, 1: i tiles of one j tile, 2: all tiles of one z
};

// The tile (it, jt, z) of workgroup w under the numbering above.
__device__ __forceinline__ void gemm_tile_of(const GemmParams& q, int w, int& it, int& jt, int& z)
{
    const int c = q.cluster;
    const int n_clusters = q.cluster_of == 2 ? q.nz : q.cluster_of == 0 ? q.nz * q.ni : q.nz * q.nj;
    const int whole = (n_clusters / 8) * 8 * c;  // workgroups of the clusters that fill all 8 XCDs evenly
    int cl, member;
    if (w < whole) {
        const int xcd = w & 7, r = w >> 3;
        member = r % c;
        cl = (r / c) * 8 + xcd;
    } else {
        const int r = w - whole;
        member = r % c;
        cl = (n_clusters / 8) * 8 + r / c;
    }
    if (q.cluster_of == 2) {
        z = cl;
        it = member % q.ni;
        jt = member / q.ni;
    } else if (q.cluster_of == 0) {
        z = cl / q.ni;
        it = cl - z * q.ni;
        jt = member;
    } else {
        z = cl / q.nj;
        jt = cl - z * q.nj;
        it = member;
    }
}

// Epilogue of one wave: accumulator register r of lane l holds C[8*(r/4) + 4*(l/32) + r%4][l%32] of a
// 32 x 32 block; (iw, jw) is the wave's corner in the result.  No branches around the loads of the
// upstream gradient: they go out 16 at a time from clamped addresses, then the exponentials, then
// stores under the range conditions (a load inside a per-element branch is waited for element by
// element: 64 memory latencies in a row).
template <int EPI, int NX, int NY, int MAXB = 2, bool WHOLE = false>
__device__ __forceinline__ void store_tile(const GemmParams& q, const floatx16 (&acc)[NX ? NX : 1][NY ? NY : 1],
                                           float* __restrict__ out, int iw, int jw, int l32, int lk)
{
    // blocks in batches of up to MAXB: the gradient loads of a whole batch are in flight together.
    // WHOLE: the wave's blocks lie inside the result, no range conditions.
    constexpr int NB = NX * NY, NYd = NY ? NY : 1;
    constexpr int BB = (MAXB >= 4 && NB % 4 == 0) ? 4 : (MAXB >= 3 && NB % 3 == 0) ? 3 : (MAXB >= 2 && NB % 2 == 0) ? 2 : 1;
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += BB) {
        float gv[BB][16];
        if (EPI == EPI_EXP_TIMES_G_PLANES) {
            // a lane's 16 rows are four runs of four consecutive positions of one item: four 16-byte loads from
            // the plane of its channel (the 32 rows of a block lie in one item)
#pragma unroll
            for (int bb = 0; bb < BB; bb++) {
                const int x = (b0 + bb) / NYd, y = (b0 + bb) % NYd;
                const int j = jw + y * 32 + l32, ib = iw + x * 32 + 4 * lk;
                const int co = j >= q.c_out ? j - q.c_out : j;
                const int item = ib / q.npos;
                const float* gp = q.g + ((long long)item * q.c_out + co) * q.npos + (ib - item * q.npos);
#pragma unroll
                for (int rg = 0; rg < 4; rg++) {
                    const float4 v = *(const float4*)(gp + 8 * rg);
                    gv[bb][4 * rg] = v.x; gv[bb][4 * rg + 1] = v.y; gv[bb][4 * rg + 2] = v.z; gv[bb][4 * rg + 3] = v.w;
                }
            }
        }
        if (EPI == EPI_EXP_TIMES_G) {
#pragma unroll
            for (int bb = 0; bb < BB; bb++) {
                const int x = (b0 + bb) / NYd, y = (b0 + bb) % NYd;
                const int j = jw + y * 32 + l32, ib = iw + x * 32 + 4 * lk;
                const int jc = (WHOLE || j < q.J) ? j : q.J - 1;
                const int co = jc >= q.c_out ? jc - q.c_out : jc;
                const float* gp = q.g + (long long)ib * q.c_out + co;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int di = 8 * (r >> 2) + (r & 3);
                    gv[bb][r] = WHOLE ? gp[di * q.c_out] : q.g[(long long)min(ib + di, q.I - 1) * q.c_out + co];
                }
            }
        }
#pragma unroll
        for (int bb = 0; bb < BB; bb++) {
            const int x = (b0 + bb) / NYd, y = (b0 + bb) % NYd;
            const int j = jw + y * 32 + l32, ib = iw + x * 32 + 4 * lk;
            const bool j_ok = WHOLE || j < q.J;
            if constexpr (EPI == EPI_STORE_ITEMS) {
                // the lane's column is one element of one item: rows are c_plane apart
                const int jc = j_ok ? j : 0;
                const int item = jc / q.c_plane;
                float* op = out + ((long long)item * q.I + ib) * q.c_plane + (jc - item * q.c_plane);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int di = 8 * (r >> 2) + (r & 3);
                    if (WHOLE || (j_ok && ib + di < q.I)) op[(long long)di * q.c_plane] = acc[x][y][r];
                }
                continue;
            }
            float* op = out + (long long)ib * q.ldc + j;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int di = 8 * (r >> 2) + (r & 3);
                const float v = (EPI == EPI_EXP_TIMES_G || EPI == EPI_EXP_TIMES_G_PLANES) ? gv[bb][r] * exp_neg(acc[x][y][r])
                                                                                        : acc[x][y][r];
                if (WHOLE)
                    op[(long long)di * q.ldc] = v;
                else if (j_ok && ib + di < q.I)
                    out[(long long)(ib + di) * q.ldc + j] = v;
            }
        }
    }
}

// ---- the GEMM: fp32 operands and results on the bf16 matrix cores ----
// Every fp32 operand element is split into three bf16 terms (x = hi + mid + lo to 2^-27 |x|: each
// term is the round-to-nearest bf16 of what the previous ones leave) and a product is formed from
// the six term products of relative size >= 2^-18 (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi),
// each exact in fp32 and accumulated in fp32 by v_mfma_f32_32x32x16_bf16; the dropped ones
// (mid lo, lo mid, lo lo) are below 2^-26 of the product, less than the rounding of an fp32
// multiply.  Six bf16 MFMAs of 16 k take 6 x 8 passes where eight fp32 MFMAs of 2 k take
// 8 x 16.  The split happens once per element, when a staged chunk is written to LDS.
// Range: an operand above 3.39e38 is infinite to it, and an infinite one makes its products NaN (WgradOperands); the
// terms of one below 2^-109 reach into bf16's subnormal numbers and are exact to 2^-134 only, a hundredth of the smallest
// normal float.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr int kLdx = 132;  // LDS stride between the two k halves of a chunk, in 16-byte slots

// bf16(a) in the low half, bf16(b) in the high half (v_cvt_pk_bf16_f32, round to nearest even)
__device__ __forceinline__ unsigned pack_bf16(float a, float b)
{
    const floatx2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

__device__ __forceinline__ void split3(float a, float b, unsigned& hi, unsigned& mid, unsigned& lo)
{
    hi = pack_bf16(a, b);
    const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xffff0000u);
    mid = pack_bf16(ra, rb);
    lo = pack_bf16(ra - __uint_as_float(mid << 16), rb - __uint_as_float(mid & 0xffff0000u));
}

// What a thread holds of eight staged elements: fp32 values; bf16 bits, one element per register where the operand
// is K-major (eight loads), two where it is I-major (in the first four registers).
typedef unsigned short bf16_bits;
template <typename T>
using raw_of = typename std::conditional<std::is_same<T, float>::value, float, unsigned>::type;

// eight elements along k of an I-major row whose first element lies on an 8-byte (bf16) or 16-byte (fp32) boundary
__device__ __forceinline__ void load_row(const float* p, float (&r)[8])
{
    const float4 v0 = *(const float4*)p, v1 = *(const float4*)(p + 4);
    r[0] = v0.x; r[1] = v0.y; r[2] = v0.z; r[3] = v0.w;
    r[4] = v1.x; r[5] = v1.y; r[6] = v1.z; r[7] = v1.w;
}
__device__ __forceinline__ void load_row(const bf16_bits* p, unsigned (&r)[8])
{
    const uint2 v0 = *(const uint2*)p, v1 = *(const uint2*)(p + 4);
    r[0] = v0.x; r[1] = v0.y; r[2] = v1.x; r[3] = v1.y;
}
// the same of a partial chunk: elements from k_left on (counted from the chunk, this thread's start at k0) are read from
// the chunk's first element instead
__device__ __forceinline__ void load_row_part(const float* p, int k0, int k_left, float (&r)[8])
{
#pragma unroll
    for (int c = 0; c < 8; c++) r[c] = p[k0 + c < k_left ? c : -k0];
}
__device__ __forceinline__ void load_row_part(const bf16_bits* p, int k0, int k_left, unsigned (&r)[8])
{
#pragma unroll
    for (int c = 0; c < 4; c++)
        r[c] = (unsigned)p[k0 + 2 * c < k_left ? 2 * c : -k0] | (unsigned)p[k0 + 2 * c + 1 < k_left ? 2 * c + 1 : -k0] << 16;
}
// zeroes the elements from k_left on
template <typename T, bool KMAJOR>
__device__ __forceinline__ void zero_past(raw_of<T> (&r)[8], int k0, int k_left)
{
    if constexpr (std::is_same<T, float>::value || KMAJOR) {
#pragma unroll
        for (int c = 0; c < 8; c++) r[c] = k0 + c < k_left ? r[c] : (raw_of<T>)0;
    } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
            r[c] &= (k0 + 2 * c < k_left ? 0x0000ffffu : 0u) | (k0 + 2 * c + 1 < k_left ? 0xffff0000u : 0u);
    }
}
// pair c of eight staged elements as one term
template <typename T, bool KMAJOR>
__device__ __forceinline__ unsigned one_term_pair(const raw_of<T> (&r)[8], int c)
{
    if constexpr (std::is_same<T, float>::value)
        return pack_bf16(r[2 * c], r[2 * c + 1]);
    else
        return KMAJOR ? r[2 * c] | r[2 * c + 1] << 16 : r[c];
}
// eight staged elements as TERMS terms into LDS
template <int TERMS, typename T, bool KMAJOR>
__device__ __forceinline__ void commit_terms(uint4 (*s)[2][kLdx], int half, int ii, const raw_of<T> (&r)[8])
{
    unsigned hi[4], mid[4], lo[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        if constexpr (TERMS == 1)
            hi[c] = one_term_pair<T, KMAJOR>(r, c);
        else
            split3(r[2 * c], r[2 * c + 1], hi[c], mid[c], lo[c]);
    }
    s[0][half][ii] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    if constexpr (TERMS == 3) {
        s[1][half][ii] = make_uint4(mid[0], mid[1], mid[2], mid[3]);
        s[2][half][ii] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
}

// The term products of a product of operands with TA and TB terms, smallest first; 0 = hi, 1 = mid, 2 = lo.  An operand
// of one term leaves the products out that would multiply by its zero terms: the sums are the same bit for bit.
template <int TA, int TB>
struct TermProducts {
    static_assert((TA == 1 || TA == 3) && (TB == 1 || TB == 3), "one term or three");
    static constexpr int N = TA == 3 && TB == 3 ? 6 : TA == 3 || TB == 3 ? 3 : 1;
    static constexpr int a(int t) { constexpr int v[6] = {2, 0, 1, 1, 0, 0}; return TA == 1 ? 0 : TB == 1 ? 2 - t : v[t]; }
    static constexpr int b(int t) { constexpr int v[6] = {0, 2, 1, 0, 1, 0}; return TB == 1 ? 0 : TA == 1 ? 2 - t : v[t]; }
};

// Staging for the split kernel: a thread owns eight consecutive k (one half of the chunk) of one i,
// which is what one lane feeds to the MFMA, and commit() writes them as s[term][k half][i], 16 bytes
// (four words of two bf16) per term.
//   K-major operand (element (k, i) at p[k*ld + i]): eight element loads from a wave-uniform row pointer
//     each, lanes along i; the k half is the wave's (uniform)
//   I-major operand (element (k, i) at p[i*ld + k]): load_row along k
// Rows i outside the operand are clamped to its last row: what they produce is never stored.  Only a
// partial last chunk is zeroed beyond its k range.
template <bool KMAJOR, typename T = float>
struct SplitStager {
    const T* p;       // K-major: row k_begin + 8 * half of the operand (uniform); I-major: this thread's first element
    long long ld;
    int off;          // K-major: this thread's i (clamped)
    int half, ii;

    // (ii_, half_): the row of the tile and the k half this thread stages (stage_slot)
    __device__ __forceinline__ void init(const T* base, long long ld_, int i0, int k_begin, int I, int ii_, int half_)
    {
        ld = ld_;
        ii = ii_;
        half = half_;
        if (KMAJOR) {
            off = min(i0 + ii, I - 1);
            p = base + (long long)(k_begin + 8 * half) * ld;
        } else {
            p = base + (long long)min(i0 + ii, I - 1) * ld + k_begin + 8 * half;
        }
    }
    // past a chunk that another thread stages
    __device__ __forceinline__ void skip_chunk() { p += KMAJOR ? (long long)kChunk * ld : (long long)kChunk; }
    // a whole chunk, no branches
    __device__ __forceinline__ void fetch_whole(raw_of<T> (&r)[8])
    {
        if (KMAJOR) {
#pragma unroll
            for (int c = 0; c < 8; c++) r[c] = (p + (long long)c * ld)[off];
        } else {
            load_row(p, r);
        }
        skip_chunk();
    }
    // k_left: what is left of the k range from this chunk's start (a partial last chunk has < kChunk)
    __device__ __forceinline__ void fetch(raw_of<T> (&r)[8], int k_left)
    {
        const bool tail = k_left < kChunk;
        if (KMAJOR) {
#pragma unroll
            for (int c = 0; c < 8; c++) {
                // rows past the end of a partial chunk read the chunk's first row instead
                const long long row = (tail && 8 * half + c >= k_left) ? -8 * half : c;
                r[c] = (p + row * ld)[off];
            }
        } else {
            if (!tail)
                load_row(p, r);
            else
                load_row_part(p, 8 * half, k_left, r);
        }
        skip_chunk();
    }
    template <int TERMS>
    __device__ __forceinline__ void commit(uint4 (*s)[2][kLdx], raw_of<T> (&r)[8], int k_left) const
    {
        if (k_left < kChunk) zero_past<T, KMAJOR>(r, 8 * half, k_left);
        commit_terms<TERMS, T, KMAJOR>(s, half, ii, r);
    }
};

// The same stager for an A operand that is a view of the shifted input planes (GemmParams::a_rows): the
// rows start where a table says, and the positions of one item are a_skip elements away from the next
// item's.  As the K-major operand of the first product the positions are the rows' elements (a lane keeps
// its own position, shifted once); as the I-major operand of the weight-gradient product they are the k
// dimension: a thread's eight positions and a whole chunk lie inside one item (a_item is a multiple of
// kChunk), and the pointer jumps by a_skip when it passes an item's end.
// AHEAD (K-major only): the table entries of a chunk are read when the chunk before it is fetched, so that a
// fetch issues its loads without waiting for the table first; the entries read for the chunk behind the last
// one (up to 2 * kChunk + 8 entries behind the member's part of the table) are never used.
// Without AHEAD the table is read as constant memory (its kernel ran before): scalar loads, where the compiler otherwise
// takes vector loads, which the data loads then wait for (waves of 2 x 2 blocks, first product of 64 -> 64 at 28 x 28, batch
// 64, three terms: 69 us, now 57).  Waves of fewer blocks have registers for the entries ahead: a scalar load's wait takes
// in the LDS reads and each chunk's entries are a cache line of their own, a round trip to L2 per chunk in a short trip
// (256 -> 256 at 8 x 8, one item: 44 us, now 35; 512 -> 512 at 4 x 4, two items: 70, 53).
template <bool KMAJOR, typename T = float, bool AHEAD = false>
struct ViewStager {
    const T* base;
    const long long* rows;  // K-major: the table of this batch member (uniform)
    const T* p;             // I-major: this thread's first element
    int off;                // K-major: this thread's element of every row
    int kr;                 // K-major: first row of this thread's half of the current chunk
    int in_item, item, skip;
    int half, ii;
    long long ahead[(KMAJOR && AHEAD) ? 8 : 1];  // the rows' starts of the chunk to fetch next

    __device__ __forceinline__ long long row_at(int k) const
    {
        return ((const __attribute__((address_space(4))) long long*)rows)[k];
    }
    __device__ __forceinline__ void read_ahead()
    {
        if constexpr (KMAJOR && AHEAD) {
#pragma unroll
            for (int c = 0; c < 8; c++) ahead[c] = rows[kr + c];
        }
    }

    __device__ __forceinline__ void init(const GemmParams& q, int batch, int i0, int k_begin, int I, int ii_, int half_)
    {
        base = (const T*)q.a;
        rows = q.a_rows + batch * q.a_rows_batch;
        item = q.a_item;
        skip = q.a_skip;
        ii = ii_;
        half = half_;
        if (KMAJOR) {
            const int m = min(i0 + ii, I - 1);
            off = m + (m / item) * skip;
            kr = k_begin + 8 * half;
            read_ahead();
            if constexpr (AHEAD) {
                // wait for these entries here, where a tile is opened, and not where this path meets the one
                // of the later fetches: there the wait would also take in the data loads of the fetch before
#pragma unroll
                for (int c = 0; c < 8; c++) asm volatile("" ::"v"(ahead[c]));
            }
        } else {
            const int m = k_begin + 8 * half;
            in_item = m % item;
            p = base + rows[min(i0 + ii, I - 1)] + m + (long long)(m / item) * skip;
        }
    }
    __device__ __forceinline__ void advance()
    {
        if (KMAJOR) {
            kr += kChunk;
        } else {
            p += kChunk;
            in_item += kChunk;
            if (in_item >= item) {
                in_item -= item;
                p += skip;
            }
        }
    }
    __device__ __forceinline__ void skip_chunk()
    {
        advance();
        read_ahead();
    }
    __device__ __forceinline__ void fetch_whole(raw_of<T> (&r)[8])
    {
        if constexpr (KMAJOR && AHEAD) {
#pragma unroll
            for (int c = 0; c < 8; c++) r[c] = (base + ahead[c])[off];
            advance();
            read_ahead();
            return;
        }
        if (KMAJOR) {
#pragma unroll
            for (int c = 0; c < 8; c++) r[c] = (base + row_at(kr + c))[off];
        } else {
            load_row(p, r);
        }
        advance();
    }
    __device__ __forceinline__ void fetch(raw_of<T> (&r)[8], int k_left)
    {
        const bool tail = k_left < kChunk;
        if (KMAJOR) {
#pragma unroll
            for (int c = 0; c < 8; c++) {
                // rows past the end of a partial chunk read the chunk's first row instead
                const int row = (tail && 8 * half + c >= k_left) ? kr - 8 * half : kr + c;
                r[c] = (base + row_at(row))[off];
            }
        } else {
            if (!tail)
                load_row(p, r);
            else
                load_row_part(p, 8 * half, k_left, r);
        }
        skip_chunk();
    }
    template <int TERMS>
    __device__ __forceinline__ void commit(uint4 (*s)[2][kLdx], raw_of<T> (&r)[8], int k_left) const
    {
        if (k_left < kChunk) zero_past<T, KMAJOR>(r, 8 * half, k_left);
        commit_terms<TERMS, T, KMAJOR>(s, half, ii, r);
    }
};

// Stager of the B operand of the input-gradient product when it sums over the kernel taps inside the GEMM
// (GemmParams::sh_*): the k dimension runs over chunks of kChunk columns j of E with the tap (u, v) as the fast
// index (u fastest), and for tap (u, v) the column (n, p, c) of B - an element of the input - is the row
// (n, p + pad_w - u, c + pad_h - v) of E_v.  I-major: a thread keeps one column and eight consecutive j; from
// chunk to chunk it moves one image row up, then one column left, and after the last tap on to the next columns
// j - so the rows of E that the taps share are read in consecutive chunks, while they are still in the CU's
// cache.  Columns whose output position does not exist for a tap read a block of zeros instead (no select on the
// loaded data, so nothing waits for the load).  sh_j is a multiple of kChunk: there are no partial chunks.
struct ShiftStager {
    const float* e0;       // E_0; E_v is group_stride floats further per v
    const float* zero;
    const float* p;
    long long ld, group_stride;
    int j, u, v, prow, pcol, wo, ho;  // j: this thread's first column of E in the current chunk; prow = p + pad_w, pcol = c + pad_h
    long long row0;                   // (n * wo + prow) * ho + pcol: the row of E for the tap (0, 0)
    int half, ii, n_u, n_v;

    __device__ __forceinline__ void point()
    {
        const int r = prow - u, c = pcol - v;
        p = (r >= 0 && r < wo && c >= 0 && c < ho)
                ? e0 + (long long)v * group_stride + (row0 - (long long)u * ho - v) * ld + j
                : zero;
    }
    __device__ __forceinline__ void init(const GemmParams& q, int batch, int j0, int k_begin, int Jn, int ii_, int half_)
    {
        ii = ii_;
        half = half_;
        n_u = q.sh_wk;
        n_v = q.sh_hk;
        // all taps in one product (E_v chosen by the tap), or one product per kernel column (batch member) over
        // its kernel rows (sh_hk = 1, sh_hin = ho, sh_padh = 0)
        e0 = q.b + (n_v == 1 ? (long long)batch * q.b_batch_stride : 0);
        group_stride = q.b_batch_stride;
        zero = q.sh_zero;
        ld = q.ldb;
        wo = q.sh_wo;
        ho = q.sh_ho;
        const int m = min(j0 + ii, Jn - 1);
        const int per_item = q.sh_win * q.sh_hin;
        const int n = m / per_item, rem = m - n * per_item;
        const int pr = rem / q.sh_hin, c = rem - pr * q.sh_hin;
        prow = pr + q.sh_pad;
        pcol = c + q.sh_padh;
        row0 = ((long long)n * wo + prow) * ho + pcol;
        // chunk c of the k dimension: tap c % (w_k h_k) of the columns (c / (w_k h_k)) * kChunk ...
        const int chunk = k_begin / kChunk, taps = n_u * n_v, t = chunk % taps;
        u = t % n_u;
        v = t / n_u;
        j = (chunk / taps) * kChunk + 8 * half;
        point();
    }
    __device__ __forceinline__ void advance()
    {
        if (++u == n_u) {
            u = 0;
            if (++v == n_v) {
                v = 0;
                j += kChunk;
            }
        }
        point();
    }
    __device__ __forceinline__ void fetch_whole(float (&r)[8])
    {
        load_row(p, r);
        advance();
    }
    __device__ __forceinline__ void fetch(float (&r)[8], int) { fetch_whole(r); }
    template <int TERMS>
    __device__ __forceinline__ void commit(uint4 (*s)[2][kLdx], float (&r)[8], int) const
    {
        commit_terms<TERMS, float, false>(s, half, ii, r);
    }
};

// v_mfma_f32_32x32x16_bf16: lane l feeds A[i = l%32][k = 8 (l/32) .. + 7] and B[those k][j = l%32]:
// the 16 bytes at s[term][l/32][i]; results as in the fp32 instruction.
// TA, TB: terms of the operands; A: type of A's elements in memory (B's are fp32).
template <bool A_KMAJOR, bool B_KMAJOR, int EPI, int NX, int NY, bool VA, bool VB, int TA, int TB, typename A>
__device__ __forceinline__ void gemm_wave_split(const GemmParams& q, uint4 (*as)[3][2][kLdx], uint4 (*bs)[3][2][kLdx],
                                                int i0, int j0, int batch, int split, int k_begin, int k_end, int wi,
                                                int wj, int l32, int lk, int wave)
{
    floatx16 acc[NX ? NX : 1][NY ? NY : 1];
#pragma unroll
    for (int x = 0; x < NX; x++)
#pragma unroll
        for (int y = 0; y < NY; y++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[x][y][r] = 0.0f;

    constexpr bool BK = B_KMAJOR && !VB;
    typename std::conditional<VA, ViewStager<A_KMAJOR, A, NX * NY < 4>, SplitStager<A_KMAJOR, A>>::type sa;
    typename std::conditional<VB, ShiftStager, SplitStager<B_KMAJOR>>::type sb;
    // K-major operand: waves 0, 1 stage the first k half of the 128 rows, waves 2, 3 the second;
    // I-major operand: two threads per row, one k half each
    const int t = threadIdx.x;
    const int a_ii = A_KMAJOR ? (t & 127) : (t >> 1), a_half = A_KMAJOR ? (wave >> 1) : (t & 1);
    const int b_ii = BK ? (t & 127) : (t >> 1), b_half = BK ? (wave >> 1) : (t & 1);
    if constexpr (VA)
        sa.init(q, batch, i0, k_begin, min(q.I, i0 + q.tile_i), a_ii, a_half);
    else
        sa.init((const A*)q.a + batch * q.a_batch_stride, q.lda, i0, k_begin, min(q.I, i0 + q.tile_i), a_ii, a_half);
    if constexpr (VB)
        sb.init(q, batch, j0, k_begin, min(q.J, j0 + q.tile_j), b_ii, b_half);
    else
        sb.init(q.b + batch * q.b_batch_stride, q.ldb, j0, k_begin, min(q.J, j0 + q.tile_j), b_ii, b_half);
    // Two chunks ahead: while chunk c is multiplied out of LDS, chunk c + 1 sits in one register set
    // (its loads issued a whole trip ago) and the loads of chunk c + 2 go out into the other.
    raw_of<A> ra[2][8];
    float rb[2][8];
    const int k_len = k_end - k_begin;
    const int n_chunks = k_len > 0 ? (k_len + kChunk - 1) / kChunk : 0;
    if (n_chunks > 0) {
        sa.fetch(ra[0], k_len);
        sb.fetch(rb[0], k_len);
    }
    if (n_chunks > 1) {
        sa.fetch(ra[1], k_len - kChunk);
        sb.fetch(rb[1], k_len - kChunk);
    }
    if (n_chunks > 0) {
        sa.template commit<TA>(as[0], ra[0], k_len);
        sb.template commit<TB>(bs[0], rb[0], k_len);
    }
    __syncthreads();
    using Products = TermProducts<TA, TB>;
    auto multiply = [&](int buf) {
        bf16x8 a[NX ? NX : 1][TA], b[NY ? NY : 1][TB];
#pragma unroll
        for (int t = 0; t < TA; t++)
#pragma unroll
            for (int x = 0; x < NX; x++) a[x][t] = __builtin_bit_cast(bf16x8, as[buf][t][lk][wi + 32 * x + l32]);
#pragma unroll
        for (int t = 0; t < TB; t++)
#pragma unroll
            for (int y = 0; y < NY; y++) b[y][t] = __builtin_bit_cast(bf16x8, bs[buf][t][lk][wj + 32 * y + l32]);
#pragma unroll
        for (int t = 0; t < Products::N; t++)
#pragma unroll
            for (int x = 0; x < NX; x++)
#pragma unroll
                for (int y = 0; y < NY; y++)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[x][Products::a(t)], b[y][Products::b(t)], acc[x][y], 0, 0, 0);
    };
    int c = 0;
    // Whole chunks, no branches in the trip.  The split of chunk c + 1 (vector ALU, 24 steps of three terms: three per
    // pair of elements) is written between the MFMAs of chunk c, one step per MFMA with four blocks, so
    // that it issues while the matrix pipe is busy.  (Scheduling barriers that spelled this order out held in
    // the first of the loop's two trips only: in the second the compiler chained the six MFMAs of each
    // block back to back.  Without them both trips keep the written order.)
    const int n_whole = k_len > 0 ? k_len / kChunk : 0;
    constexpr int kMfmas = NX * NY > 0 ? Products::N * NX * NY : 1;  // per trip
    constexpr int kStepsA = 4 * TA, kSteps = kStepsA + 4 * TB;
    constexpr int kStepsPerMfma = (kSteps + kMfmas - 1) / kMfmas;
    auto multiply_and_split = [&](auto set) {
        constexpr int S = decltype(set)::value;
        sa.fetch_whole(ra[S]);
        sb.fetch_whole(rb[S]);
        bf16x8 a[NX ? NX : 1][TA], b[NY ? NY : 1][TB];
#pragma unroll
        for (int t = 0; t < TA; t++)
#pragma unroll
            for (int x = 0; x < NX; x++) a[x][t] = __builtin_bit_cast(bf16x8, as[S][t][lk][wi + 32 * x + l32]);
#pragma unroll
        for (int t = 0; t < TB; t++)
#pragma unroll
            for (int y = 0; y < NY; y++) b[y][t] = __builtin_bit_cast(bf16x8, bs[S][t][lk][wj + 32 * y + l32]);
        // pairs 0..3: this thread's elements of A, 4..7: of B
        unsigned hi[8], mid[8], lo[8];
        float r0[8], r1[8];
        auto split_step = [&](int pr, int st, const float (&src)[8]) {
            const int e = 2 * (pr & 3);
            if (st == 0) {
                hi[pr] = pack_bf16(src[e], src[e + 1]);
                r0[pr] = src[e] - __uint_as_float(hi[pr] << 16);
                r1[pr] = src[e + 1] - __uint_as_float(hi[pr] & 0xffff0000u);
            } else if (st == 1) {
                mid[pr] = pack_bf16(r0[pr], r1[pr]);
                r0[pr] -= __uint_as_float(mid[pr] << 16);
                r1[pr] -= __uint_as_float(mid[pr] & 0xffff0000u);
            } else {
                lo[pr] = pack_bf16(r0[pr], r1[pr]);
            }
        };
        auto step = [&](int n) {
            if (n < kStepsA) {
                if constexpr (TA == 1)
                    hi[n] = one_term_pair<A, A_KMAJOR>(ra[S ^ 1], n);
                else
                    split_step(n / 3, n % 3, ra[S ^ 1]);
            } else {
                const int m = n - kStepsA;
                if constexpr (TB == 1)
                    hi[4 + m] = one_term_pair<float, BK>(rb[S ^ 1], m);
                else
                    split_step(4 + m / 3, m % 3, rb[S ^ 1]);
            }
        };
#pragma unroll
        for (int m = 0; m < kMfmas; m++) {
            constexpr int kBlocks = NX * NY > 0 ? NX * NY : 1, kNy = NY > 0 ? NY : 1;
            const int t = m / kBlocks, x = (m % kBlocks) / kNy, y = m % kNy;
            acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[x][Products::a(t)], b[y][Products::b(t)], acc[x][y], 0, 0, 0);
#pragma unroll
            for (int n = m * kStepsPerMfma; n < (m + 1) * kStepsPerMfma && n < kSteps; n++) step(n);
        }
        auto write = [&](uint4 (*to)[2][kLdx], int half, int ii, int o, int terms) {
            to[0][half][ii] = make_uint4(hi[o], hi[o + 1], hi[o + 2], hi[o + 3]);
            if (terms == 3) {
                to[1][half][ii] = make_uint4(mid[o], mid[o + 1], mid[o + 2], mid[o + 3]);
                to[2][half][ii] = make_uint4(lo[o], lo[o + 1], lo[o + 2], lo[o + 3]);
            }
        };
        write(as[S ^ 1], sa.half, sa.ii, 0, TA);
        write(bs[S ^ 1], sb.half, sb.ii, 4, TB);
        __syncthreads();
    };
    if (NX * NY > 0) {
        for (; c + 3 < n_whole; c += 2) {
            multiply_and_split(std::integral_constant<int, 0>());
            multiply_and_split(std::integral_constant<int, 1>());
        }
    }
    for (; c + 1 < n_chunks; c += 2) {
        // chunk c from LDS buffer 0; register set 1 holds chunk c + 1
        if (c + 2 < n_chunks) {
            sa.fetch(ra[0], k_len - (c + 2) * kChunk);
            sb.fetch(rb[0], k_len - (c + 2) * kChunk);
        }
        multiply(0);
        sa.template commit<TA>(as[1], ra[1], k_len - (c + 1) * kChunk);
        sb.template commit<TB>(bs[1], rb[1], k_len - (c + 1) * kChunk);
        __syncthreads();
        // chunk c + 1 from LDS buffer 1; register set 0 holds chunk c + 2
        if (c + 3 < n_chunks) {
            sa.fetch(ra[1], k_len - (c + 3) * kChunk);
            sb.fetch(rb[1], k_len - (c + 3) * kChunk);
        }
        multiply(1);
        if (c + 2 < n_chunks) {
            sa.template commit<TA>(as[0], ra[0], k_len - (c + 2) * kChunk);
            sb.template commit<TB>(bs[0], rb[0], k_len - (c + 2) * kChunk);
        }
        __syncthreads();
    }
    if (c < n_chunks) multiply(0);  // an odd last chunk, already in buffer 0

    store_tile<EPI, NX, NY>(q, acc, q.c + batch * q.c_batch_stride + split * q.c_split_stride, i0 + wi, j0 + wj, l32, lk);
}

// Operands with 16-byte aligned rows and chunks (launch_gemm checks).  LOOK: one_term is there, operands of one term are
// taken as such; without it three terms are all there is (one body, and the code and registers that it had alone: the
// last product of 64 -> 64 channels in blocks of 16, 5 x 5, 16 x 16, 64 items takes 45 us beside the other body, 41 alone).
template <bool A_KMAJOR, bool B_KMAJOR, int EPI, int PRODUCT, bool VA, bool VB, bool LOOK>
// three waves per SIMD (at most 168 registers; three workgroups' LDS fit a CU)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_gemm_split(GemmParams q)
{
    __shared__ uint4 as[2][3][2][kLdx];
    __shared__ uint4 bs[2][3][2][kLdx];
    if (LOOK && q.one_term_elsewhere && *q.one_term) return;
    int it, jt, z;
    gemm_tile_of(q, blockIdx.x, it, jt, z);
    const int i0 = it * q.tile_i, j0 = jt * q.tile_j;
    const int batch = z / q.splits, split = z - batch * q.splits;
    const int k_begin = split * q.k_per_split;
    const int k_end = min(q.K, k_begin + q.k_per_split);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool narrow_j = q.tile_j < kTile, narrow_i = q.tile_i < kTile;
    const int wi = narrow_j ? wave * 32 : narrow_i ? 0 : (wave >> 1) * 64;
    const int wj = narrow_j ? 0 : narrow_i ? wave * 32 : (wave & 1) * 64;
    const int l32 = lane & 31, lk = lane >> 5;
    const bool x0 = i0 + wi < q.I, x1 = !narrow_j && i0 + wi + 32 < q.I;
    const bool y0 = j0 + wj < q.J, y1 = !narrow_i && j0 + wj + 32 < q.J;
    const int blocks_xy = (x0 && y0) ? 2 * (int)x1 + (int)y1 : -1;
    auto tile = [&](auto ta, auto tb, auto element) {
        constexpr int TA = decltype(ta)::value, TB = decltype(tb)::value;
        using A = decltype(element);
#define GEO_SC_GEMM_WAVE(NX, NY)                                                                                        \
    gemm_wave_split<A_KMAJOR, B_KMAJOR, EPI, NX, NY, VA, VB, TA, TB, A>(q, as, bs, i0, j0, batch, split, k_begin, k_end, wi, wj, l32, lk, wave)
        switch (blocks_xy) {
        case 3: GEO_SC_GEMM_WAVE(2, 2); break;
        case 2: GEO_SC_GEMM_WAVE(2, 1); break;
        case 1: GEO_SC_GEMM_WAVE(1, 2); break;
        case 0: GEO_SC_GEMM_WAVE(1, 1); break;
        default: GEO_SC_GEMM_WAVE(0, 0); break;
        }
#undef GEO_SC_GEMM_WAVE
    };
    using One = std::integral_constant<int, 1>;
    using Three = std::integral_constant<int, 3>;
    if (!LOOK || !*q.one_term)
        tile(Three(), Three(), 0.0f);
    else if constexpr (!LOOK)
        ;
    else if constexpr (PRODUCT == PRODUCT_E)
        tile(One(), One(), bf16_bits());
    else if constexpr (PRODUCT == PRODUCT_DW)
        tile(One(), Three(), bf16_bits());
    else
        tile(One(), Three(), 0.0f);
}

// ---- the split kernel with eight waves per workgroup and a tile of 64 NX x 256 ----
// What the 128 x 128 kernel waits for is its operands: every tile streams 128 + 128 rows of fp32 per 128 x 128
// results through L2, and three workgroups per CU ask for more than the caches deliver.  Here one workgroup
// per CU (2 x 4 waves, 32 NX x 64 results each; 2 waves per SIMD with up to 256 registers) multiplies
// 64 NX x 256: per result a half (NX = 4) to three quarters (NX = 2) of the operand traffic.  A wave reads
// the fragments of one term product at a time (NX + 2 reads for 2 NX MFMAs), so that the second wave of the
// SIMD and the wave's own next reads fill the matrix pipe's shadow; the three-way split of the next chunk
// is written between the MFMAs as in the small kernel.
// With nobody else on the CU, a tile's first loads and its epilogue would run with the matrix pipe idle, so
// the workgroups are persistent: workgroup w takes the tiles w, w + gridDim.x, ... and treats their chunks
// as one stream - while the last chunks of a tile are multiplied, the first chunks of the next are already
// loaded, split and written to LDS, and the epilogue runs with those loads in flight.
// Whole tiles and whole, non-empty chunk ranges only (launch_gemm checks); the stagers and the epilogue
// are the small kernel's.
constexpr int kBigJ = 256;
constexpr int kBigWorkgroups = 256;  // one per CU of an MI355X
// rows of a tile for a result with I rows: 256, 192 or 128 (NX = 4, 3, 2); 0: I is no multiple of any
inline int big_rows(int I) { return I % 256 == 0 ? 256 : I % 192 == 0 ? 192 : I % 128 == 0 ? 128 : 0; }

// KC: chunks per trip.  With NX = 2 a trip of one chunk holds 24 MFMAs per wave, too few for what every trip
// costs besides (barrier, the latency of the first LDS reads, the loads' address arithmetic); two chunks per
// trip (KC = 2, 150 KB of LDS) halve that share.
template <bool A_KMAJOR, bool B_KMAJOR, int EPI, bool VA, bool VB, int NX, int KC, int TA, int TB, typename A>
__device__ __forceinline__ void gemm_big_tiles(const GemmParams& q, uint4 (*as)[3][2 * KC][64 * NX + 4],
                                               uint4 (*bs)[3][2 * KC][kBigJ + 4])
{
    constexpr int RA = 64 * NX;
    constexpr int kUnit = KC * kChunk;  // k per trip
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int wi = (wave >> 2) * (32 * NX), wj = (wave & 3) * 64;
    const int l32 = lane & 31, lk = lane >> 5;
    // Staging slots.  A: 2 KC RA (row, eight k) pairs of a trip, one per thread (with fewer pairs than
    // threads the rest stage a pair a second time: same data to the same place); a K-major operand has
    // the lanes along the rows and the pair's k uniform in a wave, an I-major one neighbouring threads
    // along k.  B: 512 (row, k half) pairs per chunk, every thread one pair of each of the trip's chunks.
    static_assert(2 * KC * RA <= 512, "one pair of A per thread");
    constexpr bool BK = B_KMAJOR && !VB;
    const int wa = wave % (KC * RA / 32), ta = t % (2 * KC * RA);
    const int a_ii = A_KMAJOR ? (wa % NX) * 64 + lane : ta / (2 * KC);
    const int a_q = A_KMAJOR ? wa / NX : ta % (2 * KC);  // which eight k of the trip
    const int b_ii = BK ? (t & 255) : (t >> 1), b_half = BK ? (wave >> 2) : (t & 1);
    typename std::conditional<VA, ViewStager<A_KMAJOR, A, true>, SplitStager<A_KMAJOR, A>>::type sa;
    typename std::conditional<VB, ShiftStager, SplitStager<B_KMAJOR>>::type sb;

    const int n_tiles = q.ni * q.nj * q.nz;
    // the tile whose chunks are being loaded: the stagers point into it, left_f of its trips are still to load
    int w_f = blockIdx.x, left_f;
    auto open_tile = [&]() {
        int it, jt, z;
        gemm_tile_of(q, w_f, it, jt, z);
        const int batch = z / q.splits, split = z - batch * q.splits;
        const int k_begin = split * q.k_per_split;
        left_f = (min(q.K, k_begin + q.k_per_split) - k_begin) / kUnit;
        const int ka = k_begin + (a_q >> 1) * kChunk;  // A: this thread's chunk of every trip
        if constexpr (VA)
            sa.init(q, batch, it * RA, ka, q.I, a_ii, a_q & 1);
        else
            sa.init((const A*)q.a + batch * q.a_batch_stride, q.lda, it * RA, ka, q.I, a_ii, a_q & 1);
        if constexpr (VB)
            sb.init(q, batch, jt * kBigJ, k_begin, q.J, b_ii, b_half);
        else
            sb.init(q.b + batch * q.b_batch_stride, q.ldb, jt * kBigJ, k_begin, q.J, b_ii, b_half);
    };
    // The next trip's worth of the stream into a register set.  Once the last tile is through, the fetches go
    // round that tile again (loads of valid addresses that nobody uses): every path through here issues the
    // same loads, so the waits that the compiler places in front of the split count only the loads of the
    // set they need - with a path that issues none, they would wait for the newest loads as well.
    auto fetch_next = [&](raw_of<A> (&ra)[8], float (&rb)[KC][8]) {
        if (left_f == 0) {
            if (w_f + (int)gridDim.x < n_tiles) w_f += gridDim.x;
            open_tile();
        }
        sa.fetch_whole(ra);
#pragma unroll
        for (int kc = 1; kc < KC; kc++) sa.skip_chunk();
#pragma unroll
        for (int kc = 0; kc < KC; kc++) sb.fetch_whole(rb[kc]);
        --left_f;
    };
    // the tile being multiplied
    int w_m = blockIdx.x, left_m, i0_m, j0_m;
    float* out_m;
    auto describe_m = [&]() {
        int it, jt, z;
        gemm_tile_of(q, w_m, it, jt, z);
        const int batch = z / q.splits, split = z - batch * q.splits;
        const int k_begin = split * q.k_per_split;
        left_m = (min(q.K, k_begin + q.k_per_split) - k_begin) / kUnit;
        i0_m = it * RA;
        j0_m = jt * kBigJ;
        out_m = q.c + batch * q.c_batch_stride + split * q.c_split_stride;
    };

    floatx16 acc[NX][2];
    auto zero_acc = [&]() {
#pragma unroll
        for (int x = 0; x < NX; x++)
#pragma unroll
            for (int y = 0; y < 2; y++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[x][y][r] = 0.0f;
    };
    zero_acc();
    open_tile();
    describe_m();

    // Register set c % 2 holds trip c of the stream until it is split and written to LDS buffer c % 2, one
    // trip before it is multiplied; its loads go out two trips before that.
    constexpr int kPairs = 4 + 4 * KC;  // pairs of elements per thread and trip: A, then B chunk by chunk
    raw_of<A> ra[2][8];
    float rb[2][KC][8];
    auto write_split = [&](int buf, const unsigned (&hi)[kPairs], const unsigned (&mid)[kPairs], const unsigned (&lo)[kPairs]) {
        as[buf][0][a_q][a_ii] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        if (TA == 3) {
            as[buf][1][a_q][a_ii] = make_uint4(mid[0], mid[1], mid[2], mid[3]);
            as[buf][2][a_q][a_ii] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        }
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
            const int o = 4 + 4 * kc;
            bs[buf][0][2 * kc + b_half][b_ii] = make_uint4(hi[o], hi[o + 1], hi[o + 2], hi[o + 3]);
            if (TB == 3) {
                bs[buf][1][2 * kc + b_half][b_ii] = make_uint4(mid[o], mid[o + 1], mid[o + 2], mid[o + 3]);
                bs[buf][2][2 * kc + b_half][b_ii] = make_uint4(lo[o], lo[o + 1], lo[o + 2], lo[o + 3]);
            }
        }
    };
    // The split of a trip's elements: step n of kSteps, three per pair of an operand with three terms, one per pair else.
    constexpr int kStepsA = 4 * TA, kSteps = kStepsA + 4 * KC * TB;
    auto split_step = [](int pr, int st, float e0, float e1, unsigned (&hi)[kPairs], unsigned (&mid)[kPairs],
                         unsigned (&lo)[kPairs], float (&r0)[kPairs], float (&r1)[kPairs]) {
        if (st == 0) {
            hi[pr] = pack_bf16(e0, e1);
            r0[pr] = e0 - __uint_as_float(hi[pr] << 16);
            r1[pr] = e1 - __uint_as_float(hi[pr] & 0xffff0000u);
        } else if (st == 1) {
            mid[pr] = pack_bf16(r0[pr], r1[pr]);
            r0[pr] -= __uint_as_float(mid[pr] << 16);
            r1[pr] -= __uint_as_float(mid[pr] & 0xffff0000u);
        } else {
            lo[pr] = pack_bf16(r0[pr], r1[pr]);
        }
    };
    auto step = [&](int n, const raw_of<A> (&a)[8], const float (&b)[KC][8], unsigned (&hi)[kPairs], unsigned (&mid)[kPairs],
                    unsigned (&lo)[kPairs], float (&r0)[kPairs], float (&r1)[kPairs]) {
        if (n < kStepsA) {
            if constexpr (TA == 1)
                hi[n] = one_term_pair<A, A_KMAJOR>(a, n);
            else
                split_step(n / 3, n % 3, a[2 * (n / 3)], a[2 * (n / 3) + 1], hi, mid, lo, r0, r1);
        } else {
            const int m = (n - kStepsA) / TB, st = (n - kStepsA) % TB;  // pair of B, chunk m / 4
            if constexpr (TB == 1)
                hi[4 + m] = one_term_pair<float, BK>(b[m >> 2], m & 3);
            else
                split_step(4 + m, st, b[m >> 2][2 * (m & 3)], b[m >> 2][2 * (m & 3) + 1], hi, mid, lo, r0, r1);
        }
    };
    fetch_next(ra[0], rb[0]);
    fetch_next(ra[1], rb[1]);
    {
        unsigned hi[kPairs], mid[kPairs], lo[kPairs];
        float r0[kPairs], r1[kPairs];
#pragma unroll
        for (int n = 0; n < kSteps; n++) step(n, ra[0], rb[0], hi, mid, lo, r0, r1);
        write_split(0, hi, mid, lo);
    }
    fetch_next(ra[0], rb[0]);
    __syncthreads();

    // One trip: trip c of the stream out of LDS buffer S, trip c + 1 (register set S ^ 1) split and written
    // to the other buffer, the loads of trip c + 3 into that register set.  Past the end of the stream the
    // split works on stale registers and its result is never read.
    auto trip = [&](auto set) {
        constexpr int S = decltype(set)::value, R = S ^ 1;
        using Products = TermProducts<TA, TB>;
        constexpr int kMfmas = 2 * Products::N * NX * KC;
        unsigned hi[kPairs], mid[kPairs], lo[kPairs];
        float r0[kPairs], r1[kPairs];
#pragma unroll
        for (int kc = 0; kc < KC; kc++)
#pragma unroll
            for (int p6 = 0; p6 < Products::N; p6++) {
                bf16x8 a[NX], b[2];
#pragma unroll
                for (int x = 0; x < NX; x++)
                    a[x] = __builtin_bit_cast(bf16x8, as[S][Products::a(p6)][2 * kc + lk][wi + 32 * x + l32]);
#pragma unroll
                for (int y = 0; y < 2; y++)
                    b[y] = __builtin_bit_cast(bf16x8, bs[S][Products::b(p6)][2 * kc + lk][wj + 32 * y + l32]);
#pragma unroll
                for (int m = 0; m < 2 * NX; m++) {
                    acc[m >> 1][m & 1] =
                        __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m >> 1], b[m & 1], acc[m >> 1][m & 1], 0, 0, 0);
                    // the split's steps spread over the trip's MFMAs
                    const int gm = (kc * Products::N + p6) * 2 * NX + m;
#pragma unroll
                    for (int n = kSteps * gm / kMfmas; n < kSteps * (gm + 1) / kMfmas; n++)
                        step(n, ra[R], rb[R], hi, mid, lo, r0, r1);
                }
            }
        write_split(R, hi, mid, lo);
        fetch_next(ra[R], rb[R]);
        __syncthreads();
    };
    // after a trip: was that the tile's last?  Then its results go out.  Behind the last tile nothing is stored
    // any more (a trip that still follows multiplies what the fetches past the end left in LDS).
    auto tile_done = [&]() {
        if (--left_m > 0) return;
        store_tile<EPI, NX, 2, 2, true>(q, acc, out_m, i0_m + wi, j0_m + wj, l32, lk);
        if (w_m + (int)gridDim.x >= n_tiles) {
            left_m = 0x7fffffff;
            return;
        }
        w_m += gridDim.x;
        describe_m();
        zero_acc();
    };
    // The loop leaves at its end only, after a counted number of trip pairs (one trip more than the stream has
    // when that number is odd).  With an exit between the two trips the compiler's structured form of the loop
    // has a path from the first trip straight back to itself, and on that path the register set that the
    // first trip splits is the newest one loaded: its waits would then cover the loads of the trip before
    // instead of those of two trips before.
    int trips = 0;
    for (int w = blockIdx.x; w < n_tiles; w += gridDim.x) {
        int it, jt, z;
        gemm_tile_of(q, w, it, jt, z);
        const int k_begin = (z % q.splits) * q.k_per_split;
        trips += (min(q.K, k_begin + q.k_per_split) - k_begin) / kUnit;
    }
    for (int n = (trips + 1) >> 1; n > 0; n--) {
        trip(std::integral_constant<int, 0>());
        tile_done();
        trip(std::integral_constant<int, 1>());
        tile_done();
    }
}

template <bool A_KMAJOR, bool B_KMAJOR, int EPI, int PRODUCT, bool VA, bool VB, bool LOOK, int NX, int KC = 1>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_gemm_big(GemmParams q)
{
    __shared__ uint4 as[2][3][2 * KC][64 * NX + 4];
    __shared__ uint4 bs[2][3][2 * KC][kBigJ + 4];
    if (LOOK && q.one_term_elsewhere && *q.one_term) return;
    if (!LOOK || !*q.one_term)
        gemm_big_tiles<A_KMAJOR, B_KMAJOR, EPI, VA, VB, NX, KC, 3, 3, float>(q, as, bs);
    else if constexpr (!LOOK)
        ;
    else if constexpr (PRODUCT == PRODUCT_E)
        gemm_big_tiles<A_KMAJOR, B_KMAJOR, EPI, VA, VB, NX, KC, 1, 1, bf16_bits>(q, as, bs);
    else if constexpr (PRODUCT == PRODUCT_DW)
        gemm_big_tiles<A_KMAJOR, B_KMAJOR, EPI, VA, VB, NX, KC, 1, 3, bf16_bits>(q, as, bs);
    else
        gemm_big_tiles<A_KMAJOR, B_KMAJOR, EPI, VA, VB, NX, KC, 1, 3, float>(q, as, bs);
}

// ---- E and the weight gradient in one kernel, for operands of one term and up to 192 members ----
// What the two products by themselves spend their time on is E (M x 2 c_out floats per group: written, read once per 128
// members, split each time) and chunks of 16 members or positions, a barrier each, that hold four MFMAs per wave where
// operands are one term.  Here a wave keeps 32 columns: their weights for all members in registers (first product, 32x32x16:
// A = col[m][k], read transposed from LDS), and all members' sums of the weight gradient.  The first product's result
// E[m][j] is the second one's B operand as it is: lane -> column j, and of each 16 positions the eight that the lane
// holds (the order of a contraction is free; A = col[k][m] is read in the same order).  So E is split once and never read
// back; it is stored for the input gradient, and the same bits as the first product stores (not where nobody reads it:
// the weight gradient alone of 64 -> 64 at 56 x 56, batch 128: 430 us in all with the stores, 348).
// A workgroup is persistent: 4 waves, one group, NWJ * 32 columns, one part of the positions in tiles of 32 (64 where two
// waves cover the columns: the halves' sums meet at the end); col's next tile is loaded while this one is multiplied.
// 64 -> 64 at 56 x 56, batch 128: 314 us, the two products 354 + 306 us; without the stores of E it takes 40 less, without the
// gradient's loads 45 less, its matrix work is 108.  Ragged layer of 77 items, 45 -> 83, blocks of 32 channels: 93, 79 + 76.
// Three terms need three times the registers: those operands take the two products (which return at once otherwise).
struct EwParams {
    const bf16_bits* __restrict__ col;
    const float* __restrict__ wcat;
    const float* __restrict__ g;  // the gradient: [m][c_out], or as the caller has it (GemmParams::g_planes)
    float* __restrict__ e;
    float* __restrict__ part;
    const int* __restrict__ one_term;
    const long long* __restrict__ rows;  // the view's row table, or NULL: rows col_ld apart
    int rows_batch, item, skip;
    long long col_ld;
    size_t col_v, w_v, e_v, part_v;
    int M, K, J, e_ld, c_out, npos, m_per_split, jtiles;
    int splits, tiles_each, parts;  // partial sums as in SmallKParams
    int store_e;                    // somebody reads E: the input gradient, or wgrad_again
};
constexpr int kEwMembers = 192;     // six blocks of 32: 96 registers of sums
constexpr int kEwWorkgroups = 512;  // two per CU

// PLANES: the gradient as the caller has it, through LDS in runs along the positions (a lane's own loads, 16 bytes from
// each of 32 channels, thrash the CU's cache: 483 us instead of 314); otherwise [m][c_out], read by the lanes as it is.
template <int NKB, int NWJ, bool PLANES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_bwd_e_wgrad(EwParams q)
{
    static_assert(!PLANES || NWJ == 4, "tiles of 32 positions");
    constexpr int NWM = 4 / NWJ, TM = 32 * NWM, KR = 32 * NKB;
    constexpr int RQ = TM == 32 ? 9 : 18;            // 8-byte words per row of col: 8 or 16 and padding (no bank conflicts)
    constexpr int QPR = TM / 4, RPP = 256 / QPR, NP = KR / RPP;  // quads per row; rows per pass over the workgroup, passes
    __shared__ uint2 cs[2][KR][RQ];
    __shared__ long long row_at[KR];
    constexpr int GR = 128, GQ = 9;  // the gradient's rows in LDS (channels), 16-byte words per row: 8 and padding
    __shared__ floatx4 gs[2][PLANES ? GR : 1][GQ];
    static_assert(NWM == 1 || sizeof(cs[0]) >= NWJ * 16 * 64 * sizeof(float), "room for a block's sums of the waves");
    if (!*q.one_term) return;
    const int group = blockIdx.y;
    const int split = blockIdx.x / q.jtiles, jt = blockIdx.x - split * q.jtiles;
    const int m_begin = split * q.m_per_split, m_end = min(q.M, m_begin + q.m_per_split);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, lk = lane >> 5;
    const int wj = wave % NWJ, wm = wave / NWJ;
    const int j0 = (jt * NWJ + wj) * 32, j = j0 + l32;
    const bool j_ok = j < q.J;
    const bool has_columns = j0 < q.J;  // uniform

    for (int k = threadIdx.x; k < KR; k += 256) {
        const int kc = min(k, q.K - 1);
        row_at[k] = q.rows ? q.rows[(size_t)group * q.rows_batch + kc] : kc * q.col_ld;
    }
    // first product, B operand of step s: lane -> column j, members 16 s + 8 lk .. + 7
    bf16x8 wz[2 * NKB];
    {
        const float* wg = q.wcat + (size_t)group * q.w_v + min(j, q.J - 1);
#pragma unroll
        for (int s = 0; s < 2 * NKB; s++) {
            unsigned h[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int k = 16 * s + 8 * lk + 2 * c;
                const float v0 = wg[(size_t)min(k, q.K - 1) * q.J], v1 = wg[(size_t)min(k + 1, q.K - 1) * q.J];
                h[c] = pack_bf16(j_ok && k < q.K ? v0 : 0.0f, j_ok && k + 1 < q.K ? v1 : 0.0f);
            }
            wz[s] = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
        }
    }
    // col's tile: a thread moves quad tq of the rows tr, tr + RPP, ...; positions from the part's end on and rows
    // beyond the members are zero
    const int tq = threadIdx.x % QPR, tr = threadIdx.x / QPR;
    const bf16_bits* colg = q.col + (q.rows ? 0 : (size_t)group * q.col_v);
    // (in two halves where a thread moves up to 24 quads: registers)
    constexpr int HALVES = NWM, NH = NP / HALVES;
    static_assert(NH * HALVES == NP, "whole halves");
    uint2 keep;
    auto fetch = [&](int m0, int half, uint2 (&v)[NH]) {
        const int m = m0 + 4 * tq, left = m_end - m;
        keep.x = left >= 2 ? ~0u : left == 1 ? 0xffffu : 0u;
        keep.y = left >= 4 ? ~0u : left == 3 ? 0xffffu : 0u;
        const int mc = left > 0 ? m : m_begin;
        const long long at = q.rows ? mc + (long long)(mc / q.item) * q.skip : mc;
#pragma unroll
        for (int p = 0; p < NH; p++) v[p] = *(const uint2*)(colg + row_at[tr + RPP * (half * NH + p)] + at);
    };
    auto commit = [&](int buf, int half, const uint2 (&v)[NH]) {
#pragma unroll
        for (int p = 0; p < NH; p++) {
            const int k = tr + RPP * (half * NH + p);
            const bool in = k < q.K;
            cs[buf][k][tq] = make_uint2(in ? v[p].x & keep.x : 0u, in ? v[p].y & keep.y : 0u);
        }
    };
    floatx16 acc[NKB];
#pragma unroll
    for (int b = 0; b < NKB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[b][r] = 0.0f;
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4v* tr_ptr;
    const int co = j_ok ? (j >= q.c_out ? j - q.c_out : j) : 0;
    float* eg = q.e + (size_t)group * q.e_v;
    // the upstream gradient at the wave's positions mb + 8 (r / 4) + 4 lk + r % 4 (register r), a tile ahead (behind the
    // part's end: of its first positions)
    float gv[16];
    auto fetch_g = [&](int mb) {
        const int mi = (mb < m_end ? mb : m_begin) + 4 * lk;
#pragma unroll
        for (int r = 0; r < 16; r++) gv[r] = q.g[(size_t)min(mi + 8 * (r >> 2) + (r & 3), m_end - 1) * q.c_out + co];
    };
    // the same by rows of 32 positions, one per channel that the workgroup's columns have: all of them where they are few
    const int g_rows = min(q.c_out, GR), g_first = q.c_out <= GR ? 0 : jt * 128, g_row = q.c_out <= GR ? co : min(j, q.J - 1) - jt * 128;
    floatx4 g_next[GR / 32];
    auto fetch_planes = [&](int m0) {
        const int mc = m0 < m_end ? m0 : m_begin, item = mc / q.npos;
        const float* gp = q.g + (size_t)item * q.c_out * q.npos + (mc - item * q.npos) + 4 * (threadIdx.x & 7);
#pragma unroll
        for (int p = 0; p < GR / 32; p++) {
            const int row = min((int)(threadIdx.x >> 3) + 32 * p, g_rows - 1), jr = min(g_first + row, q.J - 1);
            g_next[p] = *(const floatx4*)(gp + (size_t)(jr >= q.c_out ? jr - q.c_out : jr) * q.npos);
        }
    };
    auto commit_planes = [&](int buf) {
#pragma unroll
        for (int p = 0; p < GR / 32; p++)
            gs[buf][(threadIdx.x >> 3) + 32 * p][threadIdx.x & 7] = g_next[p];
    };
    if constexpr (PLANES) {
        fetch_planes(m_begin);
        commit_planes(0);
    } else {
        fetch_g(m_begin + 32 * wm);
    }
    uint2 next[NH];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < HALVES; h++) {
        fetch(m_begin, h, next);
        commit(0, h, next);
    }
    __syncthreads();
    constexpr int kMfma = 0x008, kDsRead = 0x100;  // of __builtin_amdgcn_sched_group_barrier
    int part = 0, tiles_left = q.tiles_each;
    // the sums so far into their place, through a buffer of col that nobody reads or writes meanwhile
    auto store_part = [&](int free_buf) {
        // (opaque to the compiler, which would keep the stores' addresses in registers over the loop)
        int K = q.K, J = q.J;
        asm volatile("" : "+s"(K), "+s"(J));
        float* pg = q.part + (size_t)group * q.part_v + (size_t)(part * q.splits + split) * K * J;
        float* meet = (float*)&cs[free_buf][0][0];  // of the waves with the tile's other half: [column block][register][lane]
#pragma unroll
        for (int b = 0; b < NKB; b++) {
            if constexpr (NWM == 2) {
                __syncthreads();
                if (wm == 1) {
#pragma unroll
                    for (int r = 0; r < 16; r++) meet[(wj * 16 + r) * 64 + lane] = acc[b][r];
                }
                __syncthreads();
                if (wm == 0) {
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[b][r] += meet[(wj * 16 + r) * 64 + lane];
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int k = 32 * b + 8 * (r >> 2) + 4 * lk + (r & 3);
                if (wm == 0 && j_ok && k < K) pg[(size_t)k * J + j] = acc[b][r];
                acc[b][r] = 0.0f;
            }
        }
        if constexpr (NWM == 2) __syncthreads();
    };
    int buf = 0;
    for (int m0 = m_begin; m0 < m_end; m0 += TM, buf ^= 1) {
        const int mb = m0 + 32 * wm, mi = mb + 4 * lk;
        fetch(m0 + TM, 0, next);  // (zeros behind the part's end)
        if constexpr (PLANES) fetch_planes(m0 + TM);
        floatx16 z;
        if (has_columns) {
#pragma unroll
            for (int r = 0; r < 16; r++) z[r] = 0.0f;
#pragma unroll
            for (int s = 0; s < 2 * NKB; s++) {
                // 16 lanes read four members of 16 positions; each gets its position's four members
                const uint2* at = &cs[buf][16 * s + 8 * lk + ((lane & 15) >> 2)][8 * wm + 4 * (lane >> 4 & 1) + (lane & 3)];
                const short4v k0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at);
                const short4v k4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 4 * RQ));
                const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(k0, k4, 0, 1, 2, 3, 4, 5, 6, 7));
                z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, wz[s], z, 0, 0, 0);
            }
            // operands four steps ahead: a step alone waits for LDS longer than it multiplies
            constexpr int kAhead = 4;
            __builtin_amdgcn_sched_group_barrier(kDsRead, 2 * kAhead, 0);
#pragma unroll
            for (int s = 0; s < 2 * NKB; s++) {
                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                if (s + kAhead < 2 * NKB) __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 0);
            }
            if constexpr (PLANES) {
#pragma unroll
                for (int o = 0; o < 4; o++) {
                    const floatx4 v = gs[buf][g_row][2 * o + lk];
                    gv[4 * o] = v[0]; gv[4 * o + 1] = v[1]; gv[4 * o + 2] = v[2]; gv[4 * o + 3] = v[3];
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++) z[r] = gv[r] * exp_neg(z[r]);
            if constexpr (!PLANES) fetch_g(mb + TM);
            float* ep = eg + (size_t)mi * q.e_ld + j;
            if (mb + 32 <= m_end && j0 + 32 <= q.J) {
                if (q.store_e) {
#pragma unroll
                    for (int r = 0; r < 16; r++) ep[(size_t)(8 * (r >> 2) + (r & 3)) * q.e_ld] = z[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int d = 8 * (r >> 2) + (r & 3);
                    if (mi + d >= m_end)
                        z[r] = 0.0f;
                    else if (j_ok && q.store_e)
                        ep[(size_t)d * q.e_ld] = z[r];
                }
            }
        }
        if constexpr (HALVES > 1) {
            commit(buf ^ 1, 0, next);
            fetch(m0 + TM, 1, next);
        }
        if (has_columns) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                unsigned t3[3][4];
#pragma unroll
                for (int o = 0; o < 4; o++) split3(z[8 * c + 2 * o], z[8 * c + 2 * o + 1], t3[0][o], t3[1][o], t3[2][o]);
                bf16x8 bt[3];
#pragma unroll
                for (int t = 0; t < 3; t++) bt[t] = __builtin_bit_cast(bf16x8, make_uint4(t3[t][0], t3[t][1], t3[t][2], t3[t][3]));
#pragma unroll
                for (int b = 0; b < NKB; b++) {
                    const uint2* row = &cs[buf][32 * b + l32][8 * wm + 4 * c + lk];
                    const uint2 p0 = row[0], p1 = row[2];
                    const bf16x8 a = __builtin_bit_cast(bf16x8, make_uint4(p0.x, p0.y, p1.x, p1.y));
#pragma unroll
                    for (int t = 2; t >= 0; t--) acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bt[t], acc[b], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 1);
#pragma unroll
            for (int b = 0; b < 2 * NKB; b++) {
                __builtin_amdgcn_sched_group_barrier(kMfma, 3, 1);
                if (b + 2 < 2 * NKB) __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 1);
            }
        }
        commit(buf ^ 1, HALVES - 1, next);
        if constexpr (PLANES) commit_planes(buf ^ 1);
        __syncthreads();
        if (--tiles_left == 0) {
            store_part(buf);
            part++;
            tiles_left = q.tiles_each;
        }
    }
    for (; part < q.parts; part++) store_part(0);
}

// gt[n*npos + pos][co] = g[n][co][pos]: the upstream gradient with the channel innermost, so that the
// first GEMM's epilogue (lanes along the channel) reads it in contiguous runs instead of one
// cache line per lane.  32 x 32 tiles through LDS; blockIdx.z = n.
__global__ __launch_bounds__(256) void k_transpose_grad(const float* __restrict__ g, float* __restrict__ gt, int c_out,
                                                        int npos)
{
    __shared__ float tile[32][33];
    const size_t item = (size_t)blockIdx.z * c_out * npos;
    const int p0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int c = c0 + r, p = p0 + tx;
        tile[r][tx] = (c < c_out && p < npos) ? g[item + (size_t)c * npos + p] : 0.0f;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int p = p0 + r, c = c0 + tx;
        if (p < npos && c < c_out) gt[item + (size_t)p * c_out + c] = tile[tx][r];
    }
}

// Group structure of one accumulation mode: which weight element (ci, u, v) member k of add
// group g is, and the inverse.
struct Groups {
    int mode, c_in, w_k, h_k, zu;
    int n_groups, n_members;
};

struct Member {
    int ci, u, v;
    bool ok;
};

__host__ __device__ inline Member member_of(const Groups& G, int g, int k)
{
    Member e;
    if (G.mode == GEO_SC_ACC_Z) {
        e.ci = g;
        e.u = k / G.h_k;
        e.v = k - e.u * G.h_k;
        e.ok = true;
    } else if (G.mode == GEO_SC_ACC_FULL) {
        const int t = k / G.h_k;
        e.v = k - t * G.h_k;
        e.ci = t / G.w_k;
        e.u = t - e.ci * G.w_k;
        e.ok = true;
    } else if (G.mode == GEO_SC_ACC_YZ) {
        const int blk = g / G.h_k;
        const int cl = k / G.w_k;
        e.v = g - blk * G.h_k;
        e.u = k - cl * G.w_k;
        e.ci = blk * G.zu + cl;
        e.ok = e.ci < G.c_in;
    } else {
        e.ci = k / G.w_k;
        e.u = k - e.ci * G.w_k;
        e.v = g;
        e.ok = true;
    }
    return e;
}

// member k+1 of the same group from member k
__host__ __device__ inline void next_member(const Groups& G, Member& e)
{
    if (G.mode == GEO_SC_ACC_Z) {
        if (++e.v == G.h_k) {
            e.v = 0;
            ++e.u;
        }
    } else if (G.mode == GEO_SC_ACC_FULL) {
        if (++e.v == G.h_k) {
            e.v = 0;
            if (++e.u == G.w_k) {
                e.u = 0;
                ++e.ci;
            }
        }
    } else if (++e.u == G.w_k) {
        e.u = 0;
        ++e.ci;
        e.ok = e.ci < G.c_in;
    }
}

__host__ __device__ inline void group_of(const Groups& G, int ci, int u, int v, int& g, int& k)
{
    if (G.mode == GEO_SC_ACC_Z) {
        g = ci;
        k = u * G.h_k + v;
    } else if (G.mode == GEO_SC_ACC_FULL) {
        g = 0;
        k = (ci * G.w_k + u) * G.h_k + v;
    } else if (G.mode == GEO_SC_ACC_YZ) {
        const int blk = ci / G.zu;
        g = blk * G.h_k + v;
        k = (ci - blk * G.zu) * G.w_k + u;
    } else {
        g = v;
        k = ci * G.w_k + u;
    }
}

// The bf16 numbers that floats known to be such stand for, and whether a float is one: its low half is zero.  Infinities
// and NaN are left to three terms.
__device__ __forceinline__ bf16_bits exact_bf16(float v) { return (bf16_bits)(__float_as_uint(v) >> 16); }
__device__ __forceinline__ uint2 exact_bf16(const float4& v)
{
    return make_uint2(__float_as_uint(v.x) >> 16 | (__float_as_uint(v.y) & 0xffff0000u),
                      __float_as_uint(v.z) >> 16 | (__float_as_uint(v.w) & 0xffff0000u));
}
__device__ __forceinline__ bool takes_three_terms(float v)
{
    const unsigned u = __float_as_uint(v);
    return (u & 0xffffu) != 0 || (u & 0x7f800000u) == 0x7f800000u;
}

// Whether a call looks for operands of one term: what the caller expects says so (geo_sc_options.backward_operand_bits), and
// where it says nothing the products' size does (multiply-adds of one of them, both rails).  Other operands pay for the scan,
// for kernels that ask what it found and for one that returns at once: 40 -> 128, 1 x 1, 32 x 32, 256 items (2.7e9) 355 -> 373
// us, 64 -> 64 at 28 x 28, 128 items (7.4e9) 430 -> 443, at 56 x 56, 64 items (1.5e10) 788 -> 799, 128 items (3e10) 1469 ->
// 1472; small ones 3 - 7 us of 24 - 90.  7-bit operands gain 1 - 25 % of 35 - 130 us (33 members and more), more when larger.
constexpr double kLookWork = 2e10;
inline bool looks_for_one_term(int operand_bits, double products)
{
    return operand_bits ? operand_bits <= 8 : products >= kLookWork;
}

// Whether x and w are bf16 numbers throughout, which 7-bit operands (k / 128) are: the scan's blocks leave what they found
// (scan_operands), the launch behind them agrees on it (operands_are_bf16) and keeps it for those that follow, which
// read one word.  A thread stops at its first element that is none, so that the scan of other operands costs next to
// nothing; 25.7 M floats of x take 20 us (64 -> 64 at 56 x 56, batch 128), and bf16 planes alone give 24 back (94 -> 70).
// One row of kScanBlocks blocks, kScanRows from kScanFew elements on (36 us with 256 blocks).
constexpr int kScanRows = 4;
constexpr long long kScanFew = 1 << 21;
inline int scan_rows(long long elements) { return elements < kScanFew ? 1 : kScanRows; }
constexpr int kScanBlocks = 256;
__device__ __forceinline__ void scan_operands(const float* __restrict__ x, long long nx, const float* __restrict__ w,
                                              long long nw, int block, int blocks, int* __restrict__ found)
{
    bool three = false;
    auto scan = [&](const float* __restrict__ p, long long n) {
        const long long lead = min(n, (long long)((4 - (((uintptr_t)p >> 2) & 3)) & 3));  // floats in front of a quad
        const long long quads = (n - lead) >> 2;
        const float4* p4 = (const float4*)(p + lead);
        if (block == 0 && threadIdx.x < 8) {
            // the ends: what lies in front of the first quad and behind the last one
            const long long e = threadIdx.x < 4 ? (long long)threadIdx.x : lead + 4 * quads + (threadIdx.x - 4);
            if (threadIdx.x < 4 ? e < lead : e < n) three |= takes_three_terms(p[e]);
        }
        constexpr int kStep = 4;
        const long long stride = (long long)blocks * 256;
        for (long long i = (long long)block * 256 + threadIdx.x; i < quads && !three; i += kStep * stride) {
            float4 v[kStep];
#pragma unroll
            for (int q = 0; q < kStep; q++) v[q] = p4[i + q * stride < quads ? i + q * stride : i];
#pragma unroll
            for (int q = 0; q < kStep; q++)
                three |= takes_three_terms(v[q].x) || takes_three_terms(v[q].y) || takes_three_terms(v[q].z) ||
                         takes_three_terms(v[q].w);
        }
    };
    scan(w, nw);
    scan(x, nx);
    const int any = __syncthreads_or(three);
    if (threadIdx.x == 0) found[block] = any;
}
// every thread of a block of 256; rows of the scan; found NULL: nobody looked
__device__ __forceinline__ bool operands_are_bf16(const int* __restrict__ found, int rows)
{
    if (!found) return false;
    static_assert(kScanBlocks == 256, "one word per thread and row");
    int any = 0;
    for (int r = 0; r < rows; r++) any |= found[r * 256 + threadIdx.x];
    return !__syncthreads_or(any);
}

// Per output position m = (n, a, b): where its receptive field starts in the unpadded input.
//   base[m] = ((n*c_in)*w_in + (a - pad_w))*h_in + (b - pad_h),  arow[m] = a - pad_w,  bcol[m] = b - pad_h
// Built once per call; it keeps integer divisions out of the per-element kernels.
struct PositionTable {
    int* base;
    int* arow;
    int* bcol;
    int m_total, c_in, w_in, h_in, pad_w, pad_h, wo, ho;
    // by `blocks` blocks of 256
    __device__ __forceinline__ void fill(int block, int blocks) const
    {
        for (int m = block * 256 + threadIdx.x; m < m_total; m += blocks * 256) {
            const int b = m % ho;
            const int t = m / ho;
            const int a = t % wo;
            const int n = t / wo;
            base[m] = ((n * c_in) * w_in + (a - pad_w)) * h_in + (b - pad_h);
            arow[m] = a - pad_w;
            bcol[m] = b - pad_h;
        }
    }
};
// For the fused kernels; rows of blocks behind the first scan x_total elements of x.
__global__ __launch_bounds__(256) void k_position_table(PositionTable p, const float* __restrict__ scan_x, long long x_total,
                                                        int* __restrict__ scan_found)
{
    if (blockIdx.y == 0)
        p.fill(blockIdx.x, gridDim.x);
    else if (blockIdx.x < kScanBlocks)
        scan_operands(scan_x, x_total, nullptr, 0, (blockIdx.y - 1) * kScanBlocks + blockIdx.x, (gridDim.y - 1) * kScanBlocks,
                      scan_found);
}

// col[g][k][m] = x~[n, ci, a+u, b+v] for groups g0 + blockIdx.z, (ci, u, v) = member k of the
// group, m = (n, a, b); x~ is the zero-padded activation, read straight from the unpadded
// tensor.  blockIdx.y selects kIm2colMembers consecutive members; a thread reads its position's
// table entry once and moves those members.  Reads and writes run along m; rows are ld elements apart.  Where x and w hold
// bf16 numbers, so does col, which the first block tells the products (*one_term).
constexpr int kIm2colMembers = 12;
__global__ __launch_bounds__(256) void k_im2col_rows(const float* __restrict__ x, float* __restrict__ col,
                                                     const int* __restrict__ found, int found_rows,
                                                     int* __restrict__ one_term,
                                                     const int* __restrict__ base, const int* __restrict__ arow,
                                                     const int* __restrict__ bcol, int g0, int m_total, int ld,
                                                     Groups G, int w_in, int h_in, size_t g_stride)
{
    const int g = g0 + blockIdx.z;
    const int k0 = blockIdx.y * kIm2colMembers;
    const int k1 = min(G.n_members, k0 + kIm2colMembers);
    float* colg = col + (size_t)blockIdx.z * g_stride;
    const bool bf16_col = operands_are_bf16(found, found_rows);
    if (found && blockIdx.x + blockIdx.y + blockIdx.z == 0 && threadIdx.x == 0) *one_term = bf16_col;
    for (int m = blockIdx.x * 256 + threadIdx.x; m < m_total; m += gridDim.x * 256) {
        const int r0 = arow[m], c0 = bcol[m], b0 = base[m];
        // all loads first, from x[0] where the member lies in the padding (a load inside a branch is
        // waited for before the next one is issued), then the stores
        float vals[kIm2colMembers];
        Member e = member_of(G, g, k0);
#pragma unroll
        for (int q = 0; q < kIm2colMembers; q++) {
            const int r = r0 + e.u, c = c0 + e.v;
            const bool ok = k0 + q < k1 && e.ok && c >= 0 && c < h_in && r >= 0 && r < w_in;
            const float val = x[ok ? b0 + (e.ci * w_in + e.u) * h_in + e.v : 0];
            vals[q] = ok ? val : 0.0f;
            next_member(G, e);
        }
        if (bf16_col) {
#pragma unroll
            for (int q = 0; q < kIm2colMembers; q++)
                if (k0 + q < k1) ((bf16_bits*)col)[blockIdx.z * g_stride + (size_t)(k0 + q) * ld + m] = exact_bf16(vals[q]);
            continue;
        }
#pragma unroll
        for (int q = 0; q < kIm2colMembers; q++)
            if (k0 + q < k1) colg[(size_t)(k0 + q) * ld + m] = vals[q];
    }
}

// Four consecutive values of a row of floats starting `sh` (0..3) floats into the aligned quad a,
// continued in the next quad b.
__device__ __forceinline__ float4 shifted_quad(const float4& a, const float4& b, int sh)
{
    float4 r;
    r.x = sh == 0 ? a.x : sh == 1 ? a.y : sh == 2 ? a.z : a.w;
    r.y = sh == 0 ? a.y : sh == 1 ? a.z : sh == 2 ? a.w : b.x;
    r.z = sh == 0 ? a.z : sh == 1 ? a.w : sh == 2 ? b.x : b.y;
    r.w = sh == 0 ? a.w : sh == 1 ? b.x : sh == 2 ? b.y : b.z;
    return r;
}

// k_im2col_rows with four positions per thread, for image rows of a multiple of four elements on both
// sides (h_in, ho) and a 16-byte aligned x: the four positions are neighbours in one output row, so a
// member's four values are four consecutive elements of one input row, cut out of one or two aligned
// quads (the kernel tap shifts them by v - pad_h) and stored as one quad: a quarter of the loads,
// stores and table reads of the one-position kernel.
__global__ __launch_bounds__(256) void k_im2col_rows_v4(const float* __restrict__ x, float* __restrict__ col,
                                                        const int* __restrict__ found, int found_rows,
                                                        int* __restrict__ one_term,
                                                        const int* __restrict__ base, const int* __restrict__ arow,
                                                        const int* __restrict__ bcol, int g0, int m_total, Groups G,
                                                        int w_in, int h_in, size_t g_stride)
{
    const int g = g0 + blockIdx.z;
    const int k0 = blockIdx.y * kIm2colMembers;
    const int k1 = min(G.n_members, k0 + kIm2colMembers);
    float* colg = col + (size_t)blockIdx.z * g_stride;
    const float4* x4 = (const float4*)x;
    const int quads = m_total >> 2;
    const bool bf16_col = operands_are_bf16(found, found_rows);
    if (found && blockIdx.x + blockIdx.y + blockIdx.z == 0 && threadIdx.x == 0) *one_term = bf16_col;
    for (int mq = blockIdx.x * 256 + threadIdx.x; mq < quads; mq += gridDim.x * 256) {
        const int m = mq << 2;
        const int r0 = arow[m], c0 = bcol[m], b0 = base[m];
        float4 vals[kIm2colMembers];
        Member e = member_of(G, g, k0);
#pragma unroll
        for (int q = 0; q < kIm2colMembers; q++) {
            const int r = r0 + e.u, c = c0 + e.v;  // c: column of the first of the four values
            const int sh = c & 3, ca = c - sh;     // the aligned quads at columns ca and ca + 4 hold them
            const bool row_ok = k0 + q < k1 && e.ok && r >= 0 && r < w_in;
            const bool ok_a = row_ok && ca >= 0 && ca < h_in;
            const bool ok_b = row_ok && sh != 0 && ca + 4 >= 0 && ca + 4 < h_in;
            const int at = (b0 + (e.ci * w_in + e.u) * h_in + e.v - sh) >> 2;  // quad index of column ca of that row
            float4 a = x4[ok_a ? at : 0], b = x4[ok_b ? at + 1 : 0];
            if (!ok_a) a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!ok_b) b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            vals[q] = shifted_quad(a, b, sh);
            next_member(G, e);
        }
        if (bf16_col) {
#pragma unroll
            for (int q = 0; q < kIm2colMembers; q++)
                if (k0 + q < k1)
                    *(uint2*)((bf16_bits*)col + blockIdx.z * g_stride + (size_t)(k0 + q) * m_total + m) = exact_bf16(vals[q]);
            continue;
        }
#pragma unroll
        for (int q = 0; q < kIm2colMembers; q++)
            if (k0 + q < k1) *(float4*)(colg + (size_t)(k0 + q) * m_total + m) = vals[q];
    }
}

// The input as col without the copies: planes xs[v][ci][n][r][b] = x~[n, ci, r, b + v] over the padded
// rows r (w_in + 2 pad_w of them) and the output columns b, one per kernel column v and channel.  Member
// (ci, u, v) at position m = (n, a, b) is xs[v][ci][n][a + u][b]: row (ci, u) of col for kernel column v is
// the plane (v, ci) read from u * ho elements in, with the positions of item n shifted by
// n * (w_k - 1) * ho -- a third of col's bytes for a 3-wide kernel, and the rows of one channel share
// their cache lines.  Four columns per thread (ho and h_in multiples of four, 16-byte aligned x), as in
// k_im2col_rows_v4.  `total` quads; the (w_k - 1) * ho elements behind the last plane are never read.  Planes of bf16
// numbers where x and w are such throughout, which the first block tells the products.
// Q quads per thread and trip, a block's width apart: their loads go out together.  Four where that leaves every CU two
// workgroups, one below: 20 M quads (64 x 56 x 56, 128 items) 98 us with one, 94 with four; 645 k 7.1 and 6.6; 322 k 6.2
// and 7.5; 15 k 2.8 and 4.5 (bf16 planes 3.2 and 4.8).
constexpr long long kShiftMany = 1 << 19;
template <int Q>
__global__ __launch_bounds__(256) void k_shift_planes(const float* __restrict__ x, float* __restrict__ xs,
                                                      const int* __restrict__ found, int found_rows,
                                                      int* __restrict__ one_term, unsigned total,
                                                      unsigned n_items, unsigned c_in, int w_in, int h_in, int pad_w, int pad_h,
                                                      int ho)
{
    const unsigned wp = w_in + 2 * pad_w, hq = ho >> 2;
    const float4* x4 = (const float4*)x;
    const bool one = operands_are_bf16(found, found_rows);
    if (found && blockIdx.x == 0 && threadIdx.x == 0) *one_term = one;
    for (unsigned e0 = blockIdx.x * (256 * Q) + threadIdx.x; e0 < total; e0 += gridDim.x * (256 * Q)) {
        float4 a[Q], b[Q];
        int sh[Q];
        bool ok_a[Q], ok_b[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const unsigned e = min(e0 + q * 256, total - 1);
            // e = (((v * c_in + ci) * n_items + n) * wp + r) * hq + quad
            unsigned t = e / hq;
            const int bq = (int)(e - t * hq);
            const unsigned pr = t / wp;
            const int r = (int)(t - pr * wp);
            t = pr / n_items;
            const unsigned n = pr - t * n_items;
            const int v = (int)(t / c_in);
            const unsigned ci = t - v * c_in;
            const int row = r - pad_w, c = 4 * bq + v - pad_h;  // input row, and input column of the first of the four
            sh[q] = c & 3;
            const int ca = c - sh[q];
            const bool row_ok = row >= 0 && row < w_in;
            ok_a[q] = row_ok && ca >= 0 && ca < h_in;
            ok_b[q] = row_ok && sh[q] != 0 && ca + 4 >= 0 && ca + 4 < h_in;
            const long long at = (((long long)(n * c_in + ci) * w_in + row) * h_in + ca) >> 2;
            a[q] = x4[ok_a[q] ? at : 0];
            b[q] = x4[ok_b[q] ? at + 1 : 0];
        }
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const unsigned e = e0 + q * 256;
            if (!ok_a[q]) a[q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!ok_b[q]) b[q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const float4 quad = shifted_quad(a[q], b[q], sh[q]);
            if (e >= total) break;
            if (one)
                ((uint2*)xs)[e] = exact_bf16(quad);
            else
                ((float4*)xs)[e] = quad;
        }
    }
}

// Weight operands of groups g0 + blockIdx.y:
//   wcat[g][k][j]: j < c_out -> clamp(w,0,100), j >= c_out -> -clamp(w,-100,0)   (utils_functional.py:611-612)
//   wd[g][j][k]  : the same with the negative rail negated (it enters dL/dx with a minus sign)
// Members that do not exist (ragged last channel block) get zeros.
__global__ __launch_bounds__(256) void k_weight_operands(const float* __restrict__ w, float* __restrict__ wcat,
                                                         float* __restrict__ wd, int g0, int c_out, Groups G,
                                                         size_t g_stride)
{
    const int K = G.n_members;
    const int total = K * c_out;
    const int g = g0 + blockIdx.y;
    float* wcatg = wcat + (size_t)blockIdx.y * g_stride;
    float* wdg = wd + (size_t)blockIdx.y * g_stride;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < total; e += gridDim.x * 256) {
        const int co = e % c_out, k = e / c_out;
        const Member mb = member_of(G, g, k);
        const float wv = mb.ok ? w[(((long long)co * G.c_in + mb.ci) * G.w_k + mb.u) * G.h_k + mb.v] : 0.0f;
        const float wp = fminf(fmaxf(wv, 0.0f), 100.0f);
        const float wn = -fminf(fmaxf(wv, -100.0f), 0.0f);
        wcatg[(long long)k * 2 * c_out + co] = wp;
        wcatg[(long long)k * 2 * c_out + c_out + co] = wn;
        wdg[(long long)co * K + k] = wp;
        wdg[(long long)(c_out + co) * K + k] = -wn;
    }
}

// What a weight gradient is formed again from where its partial sums came out NaN (col NULL: nothing is; M positions,
// rows of col and E col_ld and e_ld apart, groups col_v and e_v).  An infinite element of E, or one that rounds to a
// bf16 infinity (above 3.39e38), is inf + (inf - inf) after its split into three bf16 terms: the product is NaN where an
// fp32 product is infinite (or finite).  The sizes whose rows are no whole quads, which an fp32 product would serve, take
// the split as well, so theirs is put right here: col E in fp32, one multiply-add after the other.  A sum that is NaN
// by its operands ends at the element that makes it so.
struct WgradOperands {
    const float* col;
    const int* one_term;  // col holds bf16 numbers
    const float* e;
    long long m, col_ld, e_ld;
    size_t col_v, e_v;
};
// The partial sums to add: `splits`, or `one` where operands of one term take k_bwd_e_wgrad.
struct WgradSplits {
    int splits, one;
    const int* one_term;  // NULL: they don't
    __device__ __forceinline__ int count() const { return one_term && *one_term ? one : splits; }
};
__device__ __forceinline__ float wgrad_again(const WgradOperands& o, int group, int k, int j, long long begin, long long end)
{
    const size_t c0 = group * o.col_v + k * o.col_ld;
    const bool one = o.one_term && *o.one_term;
    const float* e = o.e + group * o.e_v + j;
    float sum = 0.0f;
#pragma unroll 1
    for (long long m = begin; m < end && sum == sum; m++) {
        const float c = one ? __uint_as_float((unsigned)((const bf16_bits*)o.col)[c0 + m] << 16) : o.col[c0 + m];
        sum = fmaf(c, e[m * o.e_ld], sum);
    }
    return sum;
}

// dL/dw of the members of group g0 + blockIdx.y from the split partial sums part[g][s][k][j].  A
// block takes 32 consecutive (k, co) entries; 8 sets of threads each sum every 8th split, the
// sets are then added in a fixed order, so the result does not depend on scheduling.
__global__ __launch_bounds__(256) void k_reduce_wgrad(const float* __restrict__ part, const float* __restrict__ w,
                                                      float* __restrict__ gw, int g0, WgradSplits parts, int c_out, Groups G,
                                                      size_t g_stride, WgradOperands again)
{
    const int splits = parts.count();
    __shared__ float red[2][8][32];
    const int K = G.n_members;
    const int total = K * c_out;
    const long long stride = (long long)K * 2 * c_out;
    const int g = g0 + blockIdx.y;
    const float* partg = part + (size_t)blockIdx.y * g_stride;
    const int lane = threadIdx.x & 31, grp = threadIdx.x >> 5;
    const int e = blockIdx.x * 32 + lane;
    const bool ok = e < total;
    const int co = ok ? e % c_out : 0, k = ok ? e / c_out : 0;
    float sp = 0.0f, sn = 0.0f;
    if (ok)
        for (int s = grp; s < splits; s += 8) {
            sp += partg[s * stride + (long long)k * 2 * c_out + co];
            sn += partg[s * stride + (long long)k * 2 * c_out + c_out + co];
        }
    red[0][grp][lane] = sp;
    red[1][grp][lane] = sn;
    __syncthreads();
    auto add_sets = [&]() {
        sp = sn = 0.0f;
#pragma unroll
        for (int gidx = 0; gidx < 8; gidx++) {
            sp += red[0][gidx][lane];
            sn += red[1][gidx][lane];
        }
    };
    add_sets();
    // (every set holds the same 32 sums here: all waves agree)
    if (again.col && __any(ok && (sp != sp || sn != sn))) {
        __syncthreads();
        const long long share = (again.m + 7) / 8, begin = min(again.m, grp * share), end = min(again.m, begin + share);
        red[0][grp][lane] = ok && sp != sp ? wgrad_again(again, blockIdx.y, k, co, begin, end) : grp ? 0.0f : sp;
        red[1][grp][lane] = ok && sn != sn ? wgrad_again(again, blockIdx.y, k, c_out + co, begin, end) : grp ? 0.0f : sn;
        __syncthreads();
        add_sets();
    }
    const Member mb = member_of(G, g, k);
    if (grp == 0 && ok && mb.ok) {
        const long long wi = (((long long)co * G.c_in + mb.ci) * G.w_k + mb.u) * G.h_k + mb.v;
        const float wv = w[wi];
        float r = 0.0f;
        if (wv >= 0.0f && wv <= 100.0f) r += sp;
        if (wv >= -100.0f && wv <= 0.0f) r += sn;
        gw[wi] = r;
    }
}

// dL/dx[n][ci][p][q] (+)= sum over the kernel taps (u, v) whose group lies in [g0, g0 + ng) of
// dcol[g][k][(n, p+pad_w-u, q+pad_h-v)] over the valid output positions; the first chunk of
// groups writes, later chunks add.  One grid-stride loop over the elements with the item inside the channel: neighbouring
// threads read one row of dcol along its positions whatever the size of an item (blocks of whole planes left 252 of
// 256 threads idle on 2 x 2 images; 512 channels of them, batch 128: 41 -> 4 us).
__global__ __launch_bounds__(256) void k_col2im_rows(const float* __restrict__ dcol, float* __restrict__ gx, int g0,
                                                     int ng, long long m_total, unsigned total, unsigned n_items, Groups G, int w_in,
                                                     int h_in, int pad_w, int pad_h, int wo, int ho, size_t g_stride)
{
    const unsigned plane = w_in * h_in;
    const int k_step = (G.mode == GEO_SC_ACC_Z || G.mode == GEO_SC_ACC_FULL) ? G.h_k : 1;
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const unsigned cn = i / plane, e = i - cn * plane;
        const int ci = (int)(cn / n_items), n = (int)(cn - ci * n_items);
        const int p = (int)e / h_in, qq = (int)e - p * h_in;
        const float* src = dcol + (size_t)n * wo * ho;
        float* dst = gx + ((size_t)n * G.c_in + ci) * plane + e;
        float s = 0.0f;
        // kernel rows v whose output column b = qq + pad_h - v exists (a 1 x 256 kernel on a 256-wide
        // input has one such row per element, not 256)
        const int v_lo = max(0, qq + pad_h - (ho - 1)), v_hi = min(G.h_k - 1, qq + pad_h);
        for (int v = v_lo; v <= v_hi; v++) {
            const int b = qq + pad_h - v;
            // the group does not depend on u, and the member index advances by k_step per tap
            int g, k;
            group_of(G, ci, 0, v, g, k);
            if (g < g0 || g >= g0 + ng) continue;
            const float* sg = src + (size_t)(g - g0) * g_stride + (size_t)k * m_total + b;
            // four taps at a time: loads from clamped addresses first, then the sum
            for (int u0 = 0; u0 < G.w_k; u0 += 4) {
                float t[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int u = u0 + q, a = p + pad_w - u;
                    const bool ok = u < G.w_k && a >= 0 && a < wo;
                    const float val = sg[ok ? (size_t)u * k_step * m_total + a * ho : 0];
                    t[q] = ok ? val : 0.0f;
                }
                s += (t[0] + t[1]) + (t[2] + t[3]);
            }
        }
        *dst = g0 == 0 ? s : *dst + s;
    }
}

// The same for outputs of one position (a classifier, a linear layer): an element has the one term of the tap that lies on
// it, and the sum is a transposition of dcol's rows [element][n] to dL/dx [n][element], in tiles of 32 x 32 through LDS.
// The kernel above reads one element per cache line here (4096 elements in 256 groups, batch 1024: 47 -> 15 us).
// blockIdx = (element tile, item tile); gridDim.y strides over the item tiles.
__global__ __launch_bounds__(256) void k_col2im_one(const float* __restrict__ dcol, float* __restrict__ gx, int g0, int ng,
                                                    int n_items, Groups G, int w_in, int h_in, int pad_w, int pad_h,
                                                    size_t g_stride)
{
    __shared__ float tile[32][33];  // [element][item]
    const int plane = w_in * h_in, elements = G.c_in * plane;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int e0 = blockIdx.x * 32;
    for (int n0 = blockIdx.y * 32; n0 < n_items; n0 += gridDim.y * 32) {
        __syncthreads();
        for (int q = ty; q < 32; q += 8) {
            const int e = min(e0 + q, elements - 1), n = min(n0 + tx, n_items - 1);
            const int ci = e / plane, p = (e - ci * plane) / h_in, qq = e - ci * plane - p * h_in;
            int g, k;
            const int u = p + pad_w, v = qq + pad_h;
            group_of(G, ci, u, v, g, k);
            const bool ok = u < G.w_k && v < G.h_k && g >= g0 && g < g0 + ng;
            const float val = dcol[ok ? (size_t)(g - g0) * g_stride + (size_t)k * n_items + n : 0];
            tile[q][tx] = ok ? val : 0.0f;
        }
        __syncthreads();
        for (int q = ty; q < 32; q += 8) {
            const int n = n0 + q, e = e0 + tx;
            if (n < n_items && e < elements) {
                float* dst = gx + (size_t)n * elements + e;
                *dst = g0 == 0 ? tile[tx][q] : *dst + tile[tx][q];
            }
        }
    }
}

// k_col2im_rows with four elements of an input row per thread, for image rows of a multiple of four
// elements on both sides, kernels of at most eight columns and 16-byte aligned buffers: a tap's four
// terms are four consecutive elements of one dcol row, cut out of one or two aligned quads.  One
// grid-stride loop over the quads of all planes.
__global__ __launch_bounds__(256) void k_col2im_rows_v4(const float* __restrict__ dcol, float* __restrict__ gx, int g0,
                                                        int ng, long long m_total, int n_planes, Groups G, int w_in,
                                                        int h_in, int pad_w, int pad_h, int wo, int ho, size_t g_stride)
{
    const int plane = w_in * h_in, plane_quads = plane >> 2;
    const int k_step = (G.mode == GEO_SC_ACC_Z || G.mode == GEO_SC_ACC_FULL) ? G.h_k : 1;
    const long long total = (long long)n_planes * plane_quads;
    for (long long idx = (long long)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (long long)gridDim.x * 256) {
        const int nc = (int)(idx / plane_quads), eq = (int)(idx - (long long)nc * plane_quads);
        const int n = nc / G.c_in, ci = nc - n * G.c_in;
        float4* dst = (float4*)(gx + (size_t)nc * plane);
        const float* src = dcol + (size_t)n * wo * ho;
        const int e = eq << 2;
        const int p = e / h_in, qq = e - p * h_in;  // the thread's elements are (p, qq .. qq + 3)
        float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int v = 0; v < G.h_k; v++) {
            int g, k;
            group_of(G, ci, 0, v, g, k);
            if (g < g0 || g >= g0 + ng) continue;
            const int b = qq + pad_h - v;  // output column of the first element's term
            const int sh = b & 3, ba = b - sh;
            const bool ok_a = ba >= 0 && ba < ho, ok_b = sh != 0 && ba + 4 >= 0 && ba + 4 < ho;
            const float* sg = src + (size_t)(g - g0) * g_stride + (size_t)k * m_total;
            for (int u = 0; u < G.w_k; u++) {
                const int a = p + pad_w - u;
                const bool row_ok = a >= 0 && a < wo;
                const float4* row = (const float4*)(sg + (size_t)u * k_step * m_total + (row_ok ? a : 0) * ho);
                float4 qa = row[(row_ok && ok_a) ? ba >> 2 : 0], qb = row[(row_ok && ok_b) ? (ba >> 2) + 1 : 0];
                if (!(row_ok && ok_a)) qa = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (!(row_ok && ok_b)) qb = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                const float4 t = shifted_quad(qa, qb, sh);
                s.x += t.x;
                s.y += t.y;
                s.z += t.z;
                s.w += t.w;
            }
        }
        if (g0 != 0) {
            const float4 o = dst[eq];
            s.x += o.x;
            s.y += o.y;
            s.z += o.z;
            s.w += o.w;
        }
        dst[eq] = s;
    }
}

// (ci, u, v) of the flat index i of one output channel's weights
__device__ __forceinline__ void weight_coords(const Groups& G, int i, int& ci, int& u, int& v)
{
    const int t = i / G.h_k;
    v = i - t * G.h_k;
    ci = t / G.w_k;
    u = t - ci * G.w_k;
}

// wcat of the groups [g0, g0 + ng) for the fused kernel (which forms wd from it): a block moves a
// tile of 32 output channels x 32 consecutive weights of each through LDS, so that w is read and wcat
// written in 128-byte runs whatever the accumulation mode (k_weight_operands reads or writes one
// element per cache line when the members of a group are not neighbours in w).  Only members that
// exist are written: not for ragged channel blocks.  blockIdx = (weight tile, channel tile).
__global__ __launch_bounds__(256) void k_weight_cat_tiled(const float* __restrict__ w, float* __restrict__ wcat, int g0,
                                                          int ng, int c_out, Groups G, size_t g_stride)
{
    __shared__ float t[32][33];  // [channel][weight]
    const int per_channel = G.c_in * G.w_k * G.h_k;
    const int i0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int q = ty; q < 32; q += 8) {
        const int co = c0 + q, i = i0 + tx;
        t[q][tx] = (co < c_out && i < per_channel) ? w[(size_t)co * per_channel + i] : 0.0f;
    }
    __syncthreads();
    for (int q = ty; q < 32; q += 8) {
        const int i = i0 + q, co = c0 + tx;
        if (i >= per_channel || co >= c_out) continue;
        int ci, u, v, g, k;
        weight_coords(G, i, ci, u, v);
        group_of(G, ci, u, v, g, k);
        if (g < g0 || g >= g0 + ng) continue;
        const float wv = t[tx][q];
        float* row = wcat + (size_t)(g - g0) * g_stride + (size_t)k * 2 * c_out;
        row[co] = fminf(fmaxf(wv, 0.0f), 100.0f);
        row[c_out + co] = -fminf(fmaxf(wv, -100.0f), 0.0f);
    }
}

// k_reduce_wgrad with the same tiles: the partial sums part[g][s][k][j] of 32 weights x 32 channels
// are read in 128-byte runs along the channel, added over the splits in their order, and dL/dw is
// written in 128-byte runs along the weights of one channel.
__global__ __launch_bounds__(256) void k_reduce_wgrad_tiled(const float* __restrict__ part, const float* __restrict__ w,
                                                            float* __restrict__ gw, int g0, int ng, WgradSplits parts, int c_out,
                                                            Groups G, size_t g_stride, WgradOperands again)
{
    const int splits = parts.count();
    __shared__ float tp[32][33], tn[32][33];  // [weight][channel]
    const int per_channel = G.c_in * G.w_k * G.h_k;
    const long long stride = (long long)G.n_members * 2 * c_out;
    const int i0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int q = ty; q < 32; q += 8) {
        const int i = i0 + q, co = c0 + tx;
        float sp = 0.0f, sn = 0.0f;
        if (i < per_channel && co < c_out) {
            int ci, u, v, g, k;
            weight_coords(G, i, ci, u, v);
            group_of(G, ci, u, v, g, k);
            if (g >= g0 && g < g0 + ng) {
                const float* src = part + (size_t)(g - g0) * g_stride + (size_t)k * 2 * c_out + co;
                for (int s0 = 0; s0 < splits; s0++) {
                    sp += src[s0 * stride];
                    sn += src[s0 * stride + c_out];
                }
                if (again.col && sp != sp) sp = wgrad_again(again, g - g0, k, co, 0, again.m);
                if (again.col && sn != sn) sn = wgrad_again(again, g - g0, k, c_out + co, 0, again.m);
            }
        }
        tp[q][tx] = sp;
        tn[q][tx] = sn;
    }
    __syncthreads();
    for (int q = ty; q < 32; q += 8) {
        const int co = c0 + q, i = i0 + tx;
        if (i >= per_channel || co >= c_out) continue;
        int ci, u, v, g, k;
        weight_coords(G, i, ci, u, v);
        group_of(G, ci, u, v, g, k);
        if (g < g0 || g >= g0 + ng) continue;
        const size_t wi = (size_t)co * per_channel + i;
        const float wv = w[wi];
        float r = 0.0f;
        if (wv >= 0.0f && wv <= 100.0f) r += tp[tx][q];
        if (wv >= -100.0f && wv <= 0.0f) r += tn[tx][q];
        gw[wi] = r;
    }
}

// What a round of GEMM launches needs beforehand, in one launch (grid: blocks x groups of the round):
//  * the weight operands wcat / wd of k_weight_operands, for group g0 + blockIdx.y;
//  * with dx_rows, in wd's place, the A operand of the input-gradient product that sums kernel taps inside
//    the GEMM (y accumulation: group = kernel column v, members (ci, u)): wdx[k][ci] = wd[v][j][(ci, u)], i.e.
//    clamp(w, 0, 100) for the positive rail j < c_out and clamp(w, -100, 0) for the negative one, with the tap
//    as the fast index over chunks of kChunk columns - dx_rows = 1: one operand per group,
//    k = ((j / kChunk) * w_k + u) * kChunk + j % kChunk (the kernel rows inside the product); dx_rows = 2: one
//    operand for all groups, k = (((j / kChunk) * h_k + v) * w_k + u) * kChunk + j % kChunk (all taps inside):
//    consecutive chunks of the product then read the same columns of E one image row, then one image column
//    apart (ShiftStager);
//  * from the blocks of the round's first group: view_rows[g][k], where row k of group g's col starts in the
//    planes of k_shift_planes (elements), for every group; and 64 zeros for the shifted view of E (a store
//    rather than a memset, so that a caller may capture the launch sequence in a graph);
//  * by blocks of their own in rows behind the groups': the scan of x and w, and the position table (a launch less in front of
//    im2col: 4 us).  They are as many as they take, in rows as wide as the weight operands' (rows of 256 blocks for every
//    group, nearly all of them without work: 5 x 5, 468 -> 26, 295 groups, 29 us for 5.6).
struct PrepParams {
    const float* __restrict__ w;
    float* __restrict__ wcat;
    float* __restrict__ wd;
    int g0, c_out;
    Groups G;
    size_t g_stride;
    int dx_rows;            // wd holds the wdx operand (y accumulation: c_in, w_k, h_k from G): 1 per group, 2 one for all
    long long* view_rows;   // null: no view
    int view_groups, view_k_pad, ho;
    long long plane;
    float* zero;            // null: no block of zeros wanted
    int groups;             // rows of blocks (blockIdx.y) that make weight operands: one per group of the round
    int scan_blocks;        // blocks that scan x and w; 0: no scan wanted
    const float* __restrict__ x;
    long long x_total, w_total;
    int* found;             // what the scan's blocks found
    PositionTable positions;
    int position_blocks;    // blocks that fill it; 0: none wanted
};
constexpr int kPrepColumns = 8;  // least blocks in a row, so that those rows are few
constexpr int kPrepRows = (kScanRows * kScanBlocks + kScanBlocks) / kPrepColumns;
// what is no weight operand: the blocks of the scan and the positions (true: the block is one of them), the view's row
// table, the zeros
__device__ __forceinline__ bool prep_scans(const PrepParams& q)
{
    if ((int)blockIdx.y < q.groups) return false;
    const int block = (blockIdx.y - q.groups) * gridDim.x + blockIdx.x;
    if (block < q.scan_blocks)
        scan_operands(q.x, q.x_total, q.w, q.w_total, block, q.scan_blocks, q.found);
    else if (block < q.scan_blocks + q.position_blocks)
        q.positions.fill(block - q.scan_blocks, q.position_blocks);
    return true;
}
__device__ __forceinline__ void prep_tables(const PrepParams& q)
{
    if (blockIdx.y != 0) return;
    if (q.view_rows)
        for (int e = blockIdx.x * 256 + threadIdx.x; e < q.view_groups * q.view_k_pad; e += gridDim.x * 256) {
            const int gi = e / q.view_k_pad, k = e - gi * q.view_k_pad;
            const Member mb = member_of(q.G, gi, min(k, q.G.n_members - 1));
            q.view_rows[e] = ((long long)mb.v * q.G.c_in + mb.ci) * q.plane + (long long)mb.u * q.ho;
        }
    if (q.zero && blockIdx.x == 0 && threadIdx.x < 64) q.zero[threadIdx.x] = 0.0f;
}

__global__ __launch_bounds__(256) void k_bwd_prep(PrepParams q)
{
    if (prep_scans(q)) return;
    const int K = q.G.n_members, c_out = q.c_out;
    const int g = q.g0 + blockIdx.y;
    float* wcatg = q.wcat + (size_t)blockIdx.y * q.g_stride;
    float* wdg = q.wd + (size_t)blockIdx.y * q.g_stride;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < K * c_out; e += gridDim.x * 256) {
        const int co = e % c_out, k = e / c_out;
        const Member mb = member_of(q.G, g, k);
        const float wv = mb.ok ? q.w[(((long long)co * q.G.c_in + mb.ci) * q.G.w_k + mb.u) * q.G.h_k + mb.v] : 0.0f;
        const float wp = fminf(fmaxf(wv, 0.0f), 100.0f);
        const float wn = -fminf(fmaxf(wv, -100.0f), 0.0f);
        wcatg[(long long)k * 2 * c_out + co] = wp;
        wcatg[(long long)k * 2 * c_out + c_out + co] = wn;
        if (!q.dx_rows) {
            wdg[(long long)co * K + k] = wp;
            wdg[(long long)(c_out + co) * K + k] = -wn;
        }
    }
    if (q.dx_rows) {
        // this block row's kernel column g: its own operand, or its part of the one operand (which starts where
        // the round's wd starts)
        const int J = 2 * c_out, c_in = q.G.c_in, w_k = q.G.w_k, h_k = q.G.h_k;
        for (int e = blockIdx.x * 256 + threadIdx.x; e < w_k * J * c_in; e += gridDim.x * 256) {
            const int ci = e % c_in, r = e / c_in;
            const int chunk = r / kChunk, u = chunk % w_k, jc = chunk / w_k, jj = r % kChunk, j = jc * kChunk + jj;
            const int co = j >= c_out ? j - c_out : j;
            const float wv = q.w[(((size_t)co * c_in + ci) * w_k + u) * h_k + g];
            const float val = j < c_out ? fminf(fmaxf(wv, 0.0f), 100.0f) : fminf(fmaxf(wv, -100.0f), 0.0f);
            if (q.dx_rows == 2)
                q.wd[((((size_t)jc * h_k + g) * w_k + u) * kChunk + jj) * c_in + ci] = val;
            else
                wdg[e] = val;
        }
    }
    prep_tables(q);
}

// The same operands in tiles of 32 output channels x `channels` input channels with all their taps, which pass through LDS:
// w is read in the runs that it has along an output channel, and every operand is written along its innermost dimension
// (element by element, k_bwd_prep reads one weight per cache line: 512 -> 512, 3 x 3: 35 -> 15 us with
// the scan).  The
// first q.groups rows of blocks take the tiles of all groups of the round.  For taps that fit (prep_tile_channels) and groups whose members all exist.
constexpr int kPrepRow = 288;  // floats per output channel of a tile
// What it takes is one long pass per tile, element by element a line per weight.  Few weights are few tiles: from 2^18 weights on
// (25 600 of 5 x 5: 14 us in tiles, 7 element by element; 205 k: 11 and 7.4; 410 k: 12 and 13), or 2^17 in tiles of few
// weights per output channel (230 k of 3 x 3: 6.6 and 7.9; 147 k, channel blocks of 32: 6.1 and 8.1).  Where the input gradient's
// operand is that of several taps (dx_rows) a tile writes it tap by tap: from two tiles per CU on (3 x 3, 128 -> 128, 128 tiles: 8.0
// and 5.0; 224 -> 224, 392: 9.1 and 8.1; 256 -> 256, 512: 10.0 and 10.6; 512 -> 512: 18.5 and 25.4; 5 x 5, 128 -> 256, 256 tiles: 15.4
// and 13.6; 128 -> 512, 512: 18.4 and 20.8).
inline int prep_tile_channels(int c_in, int c_out, int taps, bool dx_rows)
{
    const long long weights = (long long)c_in * c_out * taps;
    if (weights < 1 << 17) return 0;
    int channels = 32;
    while (channels > 1 && channels * taps > kPrepRow) channels /= 2;
    if (channels * taps > kPrepRow) return 0;
    // two tiles per CU, where narrower ones make them
    auto tiles = [&] { return (long long)((c_out + 31) / 32) * ((c_in + channels - 1) / channels); };
    while (channels > 4 && tiles() < 512) channels /= 2;
    return (dx_rows ? weights >= 1 << 18 && tiles() >= 512 : weights >= 1 << 18 || channels * taps <= 48) ? channels : 0;
}
__global__ __launch_bounds__(256) void k_bwd_prep_tiled(PrepParams q, int n_groups, int channels_log2)
{
    __shared__ float tile[32][kPrepRow + 1];
    __shared__ long long cat_at[kPrepRow];  // where weight i of a channel goes in wcat, and in wd without its channel; -1: nowhere
    __shared__ int wd_at[kPrepRow];
    if (prep_scans(q)) return;
    const Groups& G = q.G;
    const int K = G.n_members, c_out = q.c_out, J = 2 * c_out, c_in = G.c_in, taps = G.w_k * G.h_k;
    const int channels = 1 << channels_log2;
    const int ci_tiles = (c_in + channels - 1) >> channels_log2, tiles = ci_tiles * ((c_out + 31) / 32);
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int t = blockIdx.y * gridDim.x + blockIdx.x; t < tiles; t += q.groups * gridDim.x) {
        const int ct = t / ci_tiles, c0 = (t - ct * ci_tiles) << channels_log2, o0 = ct * 32;
        const int nc = min(channels, c_in - c0), no = min(32, c_out - o0), row = nc * taps;
        __syncthreads();
        for (int i = threadIdx.x; i < row; i += 256) {
            const int c = i / taps, tap = i - c * taps, u = tap / G.h_k, v = tap - u * G.h_k;
            int g, k;
            group_of(G, c0 + c, u, v, g, k);
            const bool mine = g >= q.g0 && g < q.g0 + n_groups;
            cat_at[i] = mine ? (long long)(g - q.g0) * (long long)q.g_stride + (long long)k * J : -1;
            wd_at[i] = k;
        }
        // (twelve loads in flight: one after the other they take most of the kernel's time)
        for (int e0 = threadIdx.x; e0 < no * row; e0 += 12 * 256) {
            float v[12];
            int o[12], i[12];
#pragma unroll
            for (int n = 0; n < 12; n++) {
                const int e = min(e0 + n * 256, no * row - 1);
                o[n] = (int)((unsigned)e / (unsigned)row);
                i[n] = e - o[n] * row;
                v[n] = q.w[((size_t)(o0 + o[n]) * c_in + c0) * taps + i[n]];
            }
#pragma unroll
            for (int n = 0; n < 12; n++) tile[o[n]][i[n]] = v[n];
        }
        __syncthreads();
        // wcat: along the output channels
        if (tx < no)
#pragma unroll 4
            for (int i = ty; i < row; i += 8) {
                const long long at = cat_at[i];
                if (at < 0) continue;
                float* r = q.wcat + at + o0 + tx;
                const float wv = tile[tx][i];
                r[0] = fminf(fmaxf(wv, 0.0f), 100.0f);
                r[c_out] = -fminf(fmaxf(wv, -100.0f), 0.0f);
            }
        if (!q.dx_rows) {
            // wd: along the members
            for (int o = ty; o < no; o += 8)
#pragma unroll 4
                for (int i = tx; i < row; i += 32) {
                    if (cat_at[i] < 0) continue;
                    float* r = q.wd + (cat_at[i] - (long long)wd_at[i] * J) + (size_t)(o0 + o) * K + wd_at[i];
                    const float wv = tile[o][i];
                    r[0] = fminf(fmaxf(wv, 0.0f), 100.0f);
                    r[(size_t)c_out * K] = fminf(fmaxf(wv, -100.0f), 0.0f);
                }
            continue;
        }
        // wdx: along the input channels, 256 / channels (output channel, tap) pairs at a time (every group in the round)
        const int c = threadIdx.x & (channels - 1), pair0 = threadIdx.x >> channels_log2, pairs = 256 >> channels_log2;
        if (c < nc)
            for (int tap = 0; tap < taps; tap++) {
                const int u = tap / G.h_k, v = tap - u * G.h_k;
                float* out = (q.dx_rows == 2 ? q.wd + ((size_t)v * G.w_k + u) * kChunk * c_in
                                             : q.wd + (size_t)v * q.g_stride + (size_t)u * kChunk * c_in) + c0 + c;
                const size_t jc_stride = (size_t)(q.dx_rows == 2 ? taps : G.w_k) * kChunk * c_in;
#pragma unroll 4
                for (int o = pair0; o < 2 * no; o += pairs) {
                    const int rail = o >= no, oo = rail ? o - no : o;
                    const float wv = tile[oo][c * taps + tap];
                    const int j = rail * c_out + o0 + oo, jc = j / kChunk, jj = j % kChunk;
                    out[jc * jc_stride + (size_t)jj * c_in] = rail ? fminf(fmaxf(wv, -100.0f), 0.0f) : fminf(fmaxf(wv, 0.0f), 100.0f);
                }
            }
    }
    prep_tables(q);
}

// dL/dx[n][ci][p][q] = sum over the kernel columns v of d[v][ci][(n, p, q + pad_h - v)] where that output
// column exists: what is left of col2im when the GEMM has summed the kernel rows.  Four elements of an
// input row per thread (rows of whole quads on both sides, 16-byte aligned buffers), one grid-stride loop
// over the quads of dL/dx.
__global__ __launch_bounds__(256) void k_shift_sum_v4(const float* __restrict__ d, float* __restrict__ gx, long long quads,
                                                      int n_items, int c_in, int w_in, int h_in, int h_k, int pad_h,
                                                      int ho)
{
    const int hq = h_in >> 2;
    const long long per_v = (long long)c_in * n_items * w_in * ho;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < quads; e += (long long)gridDim.x * 256) {
        // e = ((n * c_in + ci) * w_in + p) * hq + quad
        long long t = e;
        const int qq = (int)(t % hq) << 2;
        t /= hq;
        const int p = (int)(t % w_in);
        t /= w_in;
        const int ci = (int)(t % c_in), n = (int)(t / c_in);
        const float* row = d + (((long long)ci * n_items + n) * w_in + p) * ho;
        float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int v = 0; v < h_k; v++) {
            const int b = qq + pad_h - v;
            const int sh = b & 3, ba = b - sh;
            const bool ok_a = ba >= 0 && ba < ho, ok_b = sh != 0 && ba + 4 >= 0 && ba + 4 < ho;
            const float4* r4 = (const float4*)(row + v * per_v);
            float4 qa = r4[ok_a ? ba >> 2 : 0], qb = r4[ok_b ? (ba >> 2) + 1 : 0];
            if (!ok_a) qa = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!ok_b) qb = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const float4 tq = shifted_quad(qa, qb, sh);
            s.x += tq.x;
            s.y += tq.y;
            s.z += tq.z;
            s.w += tq.w;
        }
        ((float4*)gx)[e] = s;
    }
}

// a[i] += b_1[i] + ... + b_{n-1}[i] for n arrays `stride` floats apart (a is the first), four floats
// per thread, the arrays added in their order: the dcol slices of the fused kernel's column blocks.
// count and stride are multiples of 4.
__global__ __launch_bounds__(256) void k_sum_slices(float* __restrict__ a, size_t count, int n, size_t stride)
{
    const size_t n4 = count / 4;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        float4 acc = ((const float4*)a)[i];
        for (int s0 = 1; s0 < n; s0 += 8) {
            float4 v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = ((const float4*)(a + (size_t)(s0 + q < n ? s0 + q : 0) * stride))[i];
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (s0 + q < n) {
                    acc.x += v[q].x;
                    acc.y += v[q].y;
                    acc.z += v[q].z;
                    acc.w += v[q].w;
                }
        }
        ((float4*)a)[i] = acc;
    }
}

// Whole backward of layers with small OR groups (K <= 32 members: z accumulation has K = W * H,
// yz with small channel blocks K = z_unit * W, the SC linear layer K = 16) in one kernel.  With few
// members per group the general path's scratch array E[g][m][j] is c_in (z) times larger than the
// problem's tensors and its GEMMs use a fraction of each MFMA; here a workgroup loops over tiles of
// 32 output positions of one group, gathers the im2col columns into LDS, forms Z = col^T wcat with
// MFMAs, turns it into E = g exp(-Z) in LDS and feeds both Gw += col E (accumulators live over all
// tiles) and dcol = wd^T E^T from it; only dcol (the size of col) reaches memory, for the common
// col2im.  The weights of both products sit in registers for the life of the workgroup.
//   KS: k-steps of the first product (ceil(K / 2), rounded up to 5, 8, 12 or 16)
//   NB: 32-column blocks of E per wave; a workgroup covers NB * 128 columns, wider layers take
//       several column blocks, each writing a slice dcol[block][g][k][m] of its own that
//       k_sum_slices adds in a fixed order
//   DX: the input gradient is wanted
// A workgroup handles tiles s, s + S, ... of one column block of group g0 + blockIdx.y and writes
// its columns of one partial sum part[g][s][k][j] for the common split reduction.
//
// The vector ALU shares its issue slots with the MFMAs, so every instruction per element of E counts:
// the upstream gradient comes in the register order of the first product's result (k_tile_grad: four
// 16-byte loads per 32 x 32 block, no address arithmetic per element), E is stored transposed
// (E^T[j][m], rows of kFusedLd floats) with 16-byte stores, and no element is range-checked: rows
// beyond M hold zeros in col and in the gradient, columns beyond 2 * c_out meet zero weights in the
// input-gradient product and are never stored by the weight-gradient one.
constexpr int kFusedK = 32;
constexpr int kFusedTile = 32;
constexpr int kFusedLd = 36;  // floats per LDS row of a tile: 16-byte aligned rows, conflict-free MFMA operand reads

// Upstream gradient in tiles of 32 positions x 32 columns, each stored in the register order of a
// 32 x 32 MFMA result: gtt[(tile * n_blocks + block) * 1024 + lane * 16 + r] = g[m][co] with
// m = 32 tile + 8 (r / 4) + 4 (lane / 32) + r % 4 and column 32 block + lane % 32; rows beyond M and
// columns beyond the last one are zero.  With dedupe (c_out a multiple of 32) the blocks run over
// c_out and serve both rails, otherwise over the 2 * c_out rails (column j -> channel j mod c_out).
// g is [n][c_out][npos]; blockIdx = (tile, block).
__global__ __launch_bounds__(256) void k_tile_grad(const float* __restrict__ g, float* __restrict__ gtt, int M, int c_out,
                                                   int npos, int n_blocks, int dedupe)
{
    __shared__ float t[32][33];  // [position][column]
    const int m0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int n_cols = dedupe ? c_out : 2 * c_out;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    // lanes along the positions where an item has many of them, along the channels otherwise
    const bool along_m = npos >= 8;
    for (int q = ty; q < 32; q += 8) {
        const int mi = along_m ? tx : q, ci = along_m ? q : tx;
        const int m = m0 + mi, c = c0 + ci;
        const int co = c >= c_out ? c - c_out : c;
        float v = 0.0f;
        if (m < M && c < n_cols) {
            const int n = m / npos, pos = m - n * npos;
            v = g[((size_t)n * c_out + co) * npos + pos];
        }
        t[mi][ci] = v;
    }
    __syncthreads();
    const int o = threadIdx.x * 4, lane = o >> 4, r = o & 15;
    const int i = 8 * (r >> 2) + 4 * (lane >> 5), l32 = lane & 31;
    float4 v = make_float4(t[i][l32], t[i + 1][l32], t[i + 2][l32], t[i + 3][l32]);
    *(float4*)(gtt + ((size_t)blockIdx.x * n_blocks + blockIdx.y) * 1024 + o) = v;
}

template <int KS, int NB, bool DX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_bwd_small_k(
    const float* __restrict__ x, const float* __restrict__ wcat, const float* __restrict__ gtt,
    const int* __restrict__ base, const int* __restrict__ arow,
    const int* __restrict__ bcol, float* __restrict__ part, float* __restrict__ dcol, Groups G, int g0, int M, int w_in,
    int h_in, int c_out, int jblocks, int splits, int store_part, int gt_blocks, int gt_dedupe, size_t w_stride,
    size_t part_stride, size_t dcol_stride, size_t dcol_slice)
{
    constexpr int KP = KS <= 8 ? 16 : 32;       // member rows held in LDS and in the weight gradient
    constexpr int TM = kFusedTile, LD = kFusedLd;
    constexpr int JW = NB * 128;                // columns of E per workgroup
    constexpr int DPARTS = KP == 16 ? 2 : 1;    // waves that share one 16 x 16 block of dcol and split j
    constexpr int DSTEPS = JW / DPARTS / 4;     // 16x16x4 MFMAs per wave and tile in the dcol product
    constexpr int GQ = KP / 8;                  // members gathered per thread
    __shared__ __attribute__((aligned(16))) float cs[KP][LD];  // col tile [k][m]
    __shared__ __attribute__((aligned(16))) float es[JW][LD];  // E^T tile [j][m]
    __shared__ float red[2][16][17];            // second j-half's partial dcol blocks (KP == 16)
    const int K = G.n_members, J = 2 * c_out;
    const int g = g0 + blockIdx.y;
    // blockIdx.x = split * jblocks + column block: the workgroups that gather the same columns of x run together
    const int split = blockIdx.x / jblocks, jblock = blockIdx.x - split * jblocks;
    const int j_begin = jblock * JW;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, lk = lane >> 5, l16 = lane & 15, lq = lane >> 4;

    // this group's wcat[k][j_begin .. j_begin + JW) through LDS (the space of es), read in 128-byte
    // runs; zero outside the problem
    constexpr int WLD = JW + 1;
    float* wl = &es[0][0];
    {
        const float* wg = wcat + (size_t)blockIdx.y * w_stride;
        for (int e = threadIdx.x; e < KP * JW; e += 256) {
            const int k = e / JW, jl = e - k * JW, j = j_begin + jl;
            const bool ok = k < K && j < J;
            const float v = wg[ok ? (size_t)k * J + j : 0];
            wl[k * WLD + jl] = ok ? v : 0.0f;
        }
    }
    __syncthreads();
    // weights of the first product, B operand of step t: wcat[k = 2 t + lk][j]
    float w_s[NB][KS];
#pragma unroll
    for (int y = 0; y < NB; y++)
#pragma unroll
        for (int t = 0; t < KS; t++) w_s[y][t] = wl[(2 * t + lk) * WLD + 32 * (NB * wave + y) + l32];
    // dcol: wave -> (member block kb, position block mb, j part); A operand of step t: wd[j][k = 16 kb + l16],
    // which is wcat[k][j] with the negative rail (j >= c_out) negated (it enters dL/dx with a minus sign)
    const int kb = KP == 32 ? wave >> 1 : 0, mb = wave & 1, jpart = KP == 32 ? 0 : wave >> 1;
    const int jd0 = jpart * (JW / DPARTS);
    float w_d[DX ? DSTEPS : 1];
    if (DX) {
#pragma unroll
        for (int t = 0; t < DSTEPS; t++) {
            const int jl = jd0 + 4 * t + lq;
            const float v = wl[(16 * kb + l16) * WLD + jl];
            w_d[t] = j_begin + jl >= c_out ? -v : v;
        }
    }
    // (the tile loop's first barriers come before anything is written to es)
    // im2col gather: thread -> position (t & 31) of the tile, members (t >> 5) + 8 q
    const int ml = threadIdx.x & 31, slot = threadIdx.x >> 5;
    int g_off[GQ], g_u[GQ], g_v[GQ];
    bool g_ok[GQ];
#pragma unroll
    for (int q4 = 0; q4 < GQ; q4++) {
        const int k = slot + 8 * q4;
        const Member e = member_of(G, g, k < K ? k : 0);
        g_ok[q4] = k < K && e.ok;
        g_off[q4] = (e.ci * w_in + e.u) * h_in + e.v;
        g_u[q4] = e.u;
        g_v[q4] = e.v;
    }
    // this lane's 16 values of each 32 x 32 block of the upstream gradient: block of tile 0, and the
    // distance to the next tile of this workgroup
    const float* gp[NB];
#pragma unroll
    for (int y = 0; y < NB; y++) {
        const int j0 = j_begin + 32 * (NB * wave + y);
        int blk = gt_dedupe ? (j0 >= c_out ? j0 - c_out : j0) >> 5 : j0 >> 5;
        if (j0 >= J) blk = 0;  // columns outside the problem: any finite values will do
        gp[y] = gtt + ((size_t)split * gt_blocks + blk) * 1024 + lane * 16;
    }
    const size_t g_step = (size_t)splits * gt_blocks * 1024;

    // weight-gradient accumulators: 32 x 32 blocks (lane holds rows 8 (r/4) + 4 lk + r%4 of column l32),
    // or, with at most 16 members, 16 x 16 blocks (rows 4 lq + r of column l16) at half the MFMA time
    floatx16 gw_acc[KP == 32 ? NB : 1];
    floatx4 gw_acc4[KP == 16 ? 2 * NB : 1];
    if constexpr (KP == 32) {
#pragma unroll
        for (int y = 0; y < NB; y++)
#pragma unroll
            for (int r = 0; r < 16; r++) gw_acc[y][r] = 0.0f;
    } else {
#pragma unroll
        for (int b = 0; b < 2 * NB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) gw_acc4[b][r] = 0.0f;
    }

    float* dg = dcol + (size_t)jblock * dcol_slice + (size_t)blockIdx.y * dcol_stride;
    const int n_tiles = (M + TM - 1) / TM;
    for (int tile = split; tile < n_tiles; tile += splits) {
        const int m0 = tile * TM;
        // the tile's upstream gradient, asked for before anything waits: it is needed after the first product
        float4 gv[NB][4];
#pragma unroll
        for (int y = 0; y < NB; y++) {
#pragma unroll
            for (int q = 0; q < 4; q++) gv[y][q] = ((const float4*)gp[y])[q];
            gp[y] += g_step;
        }
        __syncthreads();  // the previous tile's products have read cs, es and red
        {
            const bool m_ok = m0 + ml < M;
            const int mc = m_ok ? m0 + ml : 0;
            const int r0 = arow[mc], c0 = bcol[mc], b0 = base[mc];
            float vals[GQ];
#pragma unroll
            for (int q4 = 0; q4 < GQ; q4++) {
                const int rr = r0 + g_u[q4], cc = c0 + g_v[q4];
                const bool ok = m_ok && g_ok[q4] && cc >= 0 && cc < h_in && rr >= 0 && rr < w_in;
                const float v = x[ok ? b0 + g_off[q4] : 0];
                vals[q4] = ok ? v : 0.0f;
            }
#pragma unroll
            for (int q4 = 0; q4 < GQ; q4++) cs[slot + 8 * q4][ml] = vals[q4];
        }
        __syncthreads();
#pragma unroll
        for (int y = 0; y < NB; y++) {
            // Z[m][j] = sum_k col[k][m] * wcat[k][j] for one 32 x 32 block
            floatx16 z;
#pragma unroll
            for (int r = 0; r < 16; r++) z[r] = 0.0f;
#pragma unroll
            for (int t = 0; t < KS; t++) z = __builtin_amdgcn_mfma_f32_32x32x2f32(cs[2 * t + lk][l32], w_s[y][t], z, 0, 0, 0);
            // E^T[j][m] = g[m][co] * exp(-Z): register r of the result is position 8 (r / 4) + 4 lk + r % 4
            float* er = &es[32 * (NB * wave + y) + l32][4 * lk];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float4 e;
                e.x = gv[y][q].x * exp_neg(z[4 * q + 0]);
                e.y = gv[y][q].y * exp_neg(z[4 * q + 1]);
                e.z = gv[y][q].z * exp_neg(z[4 * q + 2]);
                e.w = gv[y][q].w * exp_neg(z[4 * q + 3]);
                *(float4*)(er + 8 * q) = e;
            }
        }
        __syncthreads();
        // Gw[k][j] += sum_m col[k][m] * E[m][j] on this wave's column blocks; a lane's share of the sum
        // over m is a run of consecutive positions, read with 16-byte loads
        if constexpr (KP == 32) {
            float a[16];
#pragma unroll
            for (int q = 0; q < 4; q++) *(float4*)&a[4 * q] = *(const float4*)&cs[l32][16 * lk + 4 * q];
#pragma unroll
            for (int y = 0; y < NB; y++) {
                float b[16];
#pragma unroll
                for (int q = 0; q < 4; q++) *(float4*)&b[4 * q] = *(const float4*)&es[32 * (NB * wave + y) + l32][16 * lk + 4 * q];
#pragma unroll
                for (int st = 0; st < 16; st++) gw_acc[y] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[st], b[st], gw_acc[y], 0, 0, 0);
            }
        } else {
            float a[8];
#pragma unroll
            for (int q = 0; q < 2; q++) *(float4*)&a[4 * q] = *(const float4*)&cs[l16][8 * lq + 4 * q];
#pragma unroll
            for (int bq = 0; bq < 2 * NB; bq++) {
                float b[8];
#pragma unroll
                for (int q = 0; q < 2; q++) *(float4*)&b[4 * q] = *(const float4*)&es[32 * NB * wave + 16 * bq + l16][8 * lq + 4 * q];
#pragma unroll
                for (int st = 0; st < 8; st++) gw_acc4[bq] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st], b[st], gw_acc4[bq], 0, 0, 0);
            }
        }
        if (DX) {
            // dcol[k][m] = sum_j wd[j][k] * E[m][j]: one 16 x 16 block per wave (v_mfma_f32_16x16x4_f32:
            // lane l feeds A[i = l%16][k' = l/16] and B[k' = l/16][j = l%16], holds D[4 (l/16) + r][l%16])
            floatx4 d = {0.0f, 0.0f, 0.0f, 0.0f};
            const float* eb = &es[jd0 + lq][16 * mb + l16];
#pragma unroll
            for (int t = 0; t < DSTEPS; t++) d = __builtin_amdgcn_mfma_f32_16x16x4f32(w_d[t], eb[4 * t * LD], d, 0, 0, 0);
            if (DPARTS == 2) {
                if (jpart == 1) {
#pragma unroll
                    for (int r = 0; r < 4; r++) red[mb][4 * lq + r][l16] = d[r];
                }
                __syncthreads();
                if (jpart == 0) {
#pragma unroll
                    for (int r = 0; r < 4; r++) d[r] += red[mb][4 * lq + r][l16];
                }
            }
            if (jpart == 0) {
                const int m = m0 + 16 * mb + l16;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int k = 16 * kb + 4 * lq + r;
                    if (k < K && m < M) dg[(size_t)k * M + m] = d[r];
                }
            }
        }
    }
    if (store_part) {
        float* pg = part + (size_t)blockIdx.y * part_stride + (size_t)split * K * J;
        if constexpr (KP == 32) {
#pragma unroll
            for (int y = 0; y < NB; y++) {
                const int j = j_begin + 32 * (NB * wave + y) + l32;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int k = 8 * (r >> 2) + 4 * lk + (r & 3);
                    if (k < K && j < J) pg[(size_t)k * J + j] = gw_acc[y][r];
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < 2 * NB; b++) {
                const int j = j_begin + 32 * NB * wave + 16 * b + l16;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int k = 4 * lq + r;
                    if (k < K && j < J) pg[(size_t)k * J + j] = gw_acc4[b][r];
                }
            }
        }
    }
}

// The fused kernel on the bf16 matrix cores, for K <= 16 members.  The fp32 MFMAs of k_bwd_small_k run on the vector
// ALU's multipliers: while one executes, no wave of the SIMD issues vector instructions, and the kernel's time is the
// sum of its MFMA and vector work.  The bf16 MFMAs have a pipe of their own; what bounds this kernel is the vector work
// per element of E: the exponential, the factor g and the split into three bf16 terms (5.5 instructions).  So E makes
// no detour that costs more of it.  All products are 16x16x32:
//   first product    A = col[m][k] (csz), B = wcat[k][j] (registers).  The 16 members are half of the instruction's k:
//                    operands of three terms put two term products into one instruction.  Row i of its two blocks is
//                    position 16 (i / 8) + i % 8 and that + 8, so that a lane's eight results are eight consecutive
//                    floats of the tiled gradient (k_tile_grad).
//   weight gradient  A = col[k][m] (csg), B = E[m][j]: the lane's eight results as they are - the order of a
//                    contraction is free, col's words are read in E's order.
//   input gradient   A = wd[k][j] (registers), B = E[m][j] along j: one term of a 32 x 32 block at a time through an
//                    LDS block of the wave's own, written as E^T[j][m] and read transposed (ds_read_b64_tr_b16), no
//                    barrier.  The waves' sums meet in LDS, once per tile.
// A wave has NB blocks of 32 columns.  Where x and the workgroup's weights are bf16 numbers (the layers' 7-bit operands)
// they are one term, 1, 3 and 3 products instead of 6, 6 and 6; otherwise a wave takes its blocks one after the other,
// each over all tiles (two blocks' operands of three terms need more than the 128 registers that four waves per SIMD
// have), and adds to the dcol of the first.  4096 x 4096 linear layer, batch 1024: 1965 us with three terms
// throughout and E in LDS for both gradients, 1096 now, of which the vector work of E is 630 (the sum of the slices of
// dcol, 16 with NB = 2 and 32 with NB = 1: 119 -> 62); unquantised operands, step 4.20 -> 4.17 ms; first layer of the
// 4-layer CNN 92 -> 56, half of that the gather's.
// Same grid, tiles and outputs as k_bwd_small_k.  LOOK: the call has scanned x; without it three terms are all there is.
constexpr int kBfEw = 18;  // words per row of E^T: 32 bf16 and padding (8-byte accesses of 16 rows meet no bank twice)
constexpr int kBfCw = 20;  // words per row of col[k][m]: 16-byte aligned rows

struct SmallKParams {
    const float* __restrict__ x;
    const float* __restrict__ wcat;
    const float* __restrict__ gtt;
    const int* __restrict__ base;
    const int* __restrict__ arow;
    const int* __restrict__ bcol;
    const int* __restrict__ found;  // what the scan of x left (scan_operands)
    float* __restrict__ part;
    float* __restrict__ dcol;
    Groups G;
    int g0, M, w_in, h_in, c_out, jblocks, splits, store_part, gt_blocks, gt_dedupe, found_rows;
    // partial sums of the weight gradient: one per `tiles_each` of a workgroup's tiles (longer sums in fp32 round more: 14
    // items of 7 x 37, 31 -> 280, z accumulation: 2.4e-7 against float64 over 23 tiles, 1.3e-7 over 6), n of them per workgroup
    int tiles_each, parts, sums;  // sums: those with tiles at all, the first ones
    size_t w_stride, part_stride, dcol_stride, dcol_slice;
};

template <int NW, int NB, bool DX>
struct SmallKShared {
    // col of two tiles in turn: the next tile's is written while this tile's products run
    uint4 csz[2][3][2][kFusedTile];      // first product: (term, k half, m) -> 8 bf16 along k
    unsigned csg[2][3][16][kBfCw];       // weight gradient: [term][k][m], two m per word
    union {
        float wl[16][32 * NW * NB + 1];  // the group's weights on their way into registers
        struct {
            uint2 est[DX ? NW : 1][32][kBfEw / 2];  // per wave: one term of E^T[j][m]
            float4 red[2][DX ? NW : 1][2][64];      // per wave: its part of dcol, 16 x 16 blocks in the order of an MFMA result
        } t;
    } u;
};

// this group's wcat[k][j_begin ..] into wl; zero outside the problem.  Whether an element takes three terms.
template <int NW, int NB, bool DX>
__device__ __forceinline__ bool small_k_weights(const SmallKParams& q, SmallKShared<NW, NB, DX>& sh, int j_begin)
{
    constexpr int JW = 32 * NW * NB;
    const int K = q.G.n_members, J = 2 * q.c_out;
    const float* wg = q.wcat + (size_t)blockIdx.y * q.w_stride;
    bool three = false;
    for (int e = threadIdx.x; e < 16 * JW; e += 64 * NW) {
        const int k = e / JW, jl = e - k * JW, j = j_begin + jl;
        const bool ok = k < K && j < J;
        const float v = wg[ok ? (size_t)k * J + j : 0];
        sh.u.wl[k][jl] = ok ? v : 0.0f;
        three |= ok && takes_three_terms(v);
    }
    return three;
}

// columns c0 + 32 (b NW + wave) .. + 31, b < NB, of the workgroup's (from j_begin on, weights in wl) over its tiles; ADD: to
// the dcol that is there; PARTS: more than one partial sum
template <int TERMS, int NW, int NB, bool DX, bool ADD, bool PARTS, typename Shared>
__device__ __forceinline__ void small_k_columns(const SmallKParams& q, Shared& sh, int split, int jblock, int j_begin, int c0)
{
    constexpr int KP = 16, TM = kFusedTile, NT = 64 * NW;
    constexpr int EP = NW == 8 ? 1 : 2;                    // members gathered per slot of a thread
    constexpr int GP = KP * TM / EP / NT;                  // slots per thread
    static_assert(GP * EP * NT == KP * TM, "every thread gathers");
    const int K = q.G.n_members, J = 2 * q.c_out, M = q.M, c_out = q.c_out;
    const int g = q.g0 + blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l16 = lane & 15, lq = lane >> 4;

    // im2col gather: slot = (position t % 32 of the tile, members EP (t / 32) ..)
    const int ml = threadIdx.x & 31;
    int kg[GP], g_off[GP][EP], g_u[GP][EP], g_v[GP][EP];
    bool g_ok[GP][EP];
#pragma unroll
    for (int gp = 0; gp < GP; gp++) {
        kg[gp] = (threadIdx.x >> 5) + gp * (NT / 32);
#pragma unroll
        for (int p = 0; p < EP; p++) {
            const int k = EP * kg[gp] + p;
            const Member e = member_of(q.G, g, k < K ? k : 0);
            g_ok[gp][p] = k < K && e.ok;
            g_off[gp][p] = (e.ci * q.w_in + e.u) * q.h_in + e.v;
            g_u[gp][p] = e.u;
            g_v[gp][p] = e.v;
        }
    }
    float* dg = q.dcol + (size_t)jblock * q.dcol_slice + (size_t)blockIdx.y * q.dcol_stride;
    const int n_tiles = (M + TM - 1) / TM;
    // The gather runs a tile ahead and its table entries two: a tile's columns of x are asked for at the
    // top of the tile before and its table entries at the top of the one before that, so that no tile
    // waits for two dependent loads in a row.  The first tile's are on their way while the weights become operands: with few
    // tiles per workgroup that is most of its time (16 x 1 x 256 -> 1000, 8 items, three terms: 48 us, now 41).
    struct Where {
        int r0, c0, b0;
        bool ok;
    };
    auto where = [&](int tile) {
        Where p;
        p.ok = tile < n_tiles && tile * TM + ml < M;
        const int mc = p.ok ? tile * TM + ml : 0;
        p.r0 = q.arow[mc];
        p.c0 = q.bcol[mc];
        p.b0 = q.base[mc];
        return p;
    };
    auto fetch = [&](const Where& p, float (&v)[GP][EP]) {  // returns which of them exist, one bit each
        unsigned exist = 0;
#pragma unroll
        for (int gp = 0; gp < GP; gp++)
#pragma unroll
            for (int e = 0; e < EP; e++) {
                const int rr = p.r0 + g_u[gp][e], cc = p.c0 + g_v[gp][e];
                const bool ok = p.ok && g_ok[gp][e] && cc >= 0 && cc < q.h_in && rr >= 0 && rr < q.w_in;
                v[gp][e] = q.x[ok ? p.b0 + g_off[gp][e] : 0];
                exist |= (unsigned)ok << (gp * EP + e);
            }
        return exist;
    };
    auto commit = [&](int buf, const float (&v)[GP][EP], unsigned exist) {
#pragma unroll
        for (int gp = 0; gp < GP; gp++) {
            float v2[2] = {0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < EP; e++) v2[e] = exist >> (gp * EP + e) & 1 ? v[gp][e] : 0.0f;
            unsigned t3[3];
            split3(v2[0], v2[1], t3[0], t3[1], t3[2]);
#pragma unroll
            for (int t = 0; t < TERMS; t++) {
                if constexpr (EP == 2) {
                    ((unsigned*)&sh.csz[buf][t][kg[gp] >> 2][ml])[kg[gp] & 3] = t3[t];
                    ((unsigned short*)&sh.csg[buf][t][2 * kg[gp] + 1][0])[ml] = (unsigned short)(t3[t] >> 16);
                } else {
                    ((unsigned short*)&sh.csz[buf][t][kg[gp] >> 3][ml])[kg[gp] & 7] = (unsigned short)t3[t];
                }
                ((unsigned short*)&sh.csg[buf][t][EP * kg[gp]][0])[ml] = (unsigned short)t3[t];
            }
        }
    };
    float x_next[GP][EP], x_after[GP][EP], x_first[GP][EP];
    const Where w_first = where(split), w_next = where(split + q.splits);
    Where w_after = where(split + 2 * q.splits);
    const unsigned ok_first = fetch(w_first, x_first);
    unsigned ok_next = fetch(w_next, x_next), ok_after;
    // first product, B operand of 16 columns: lane -> column l16, k = 8 (lq % 2) .. + 7 of one term; lanes from 32 on
    // have the second of two terms (hi and lo, mid and hi), or zeros
    constexpr int ZB = TERMS == 3 ? 2 : 1;
    const unsigned first = lq < 2 ? ~0u : 0u;
    bf16x8 wz[NB][2][ZB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int s = 0; s < 2; s++) {
            unsigned t3[3][4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int k = 8 * (lq & 1) + 2 * c, jl = c0 + 32 * (b * NW + wave) + 16 * s + l16;
                split3(sh.u.wl[k][jl], sh.u.wl[k + 1][jl], t3[0][c], t3[1][c], t3[2][c]);
            }
            unsigned o[2][4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                o[0][c] = (t3[0][c] & first) | (TERMS == 3 ? t3[2][c] & ~first : 0u);
                o[1][c] = (t3[1][c] & first) | (t3[0][c] & ~first);
            }
#pragma unroll
            for (int z = 0; z < ZB; z++) wz[b][s][z] = __builtin_bit_cast(bf16x8, make_uint4(o[z][0], o[z][1], o[z][2], o[z][3]));
        }
    // input gradient, A operand of 32 columns: lane -> wd[j][k = l16], j = 8 lq .. + 7, which is wcat[k][j] with the
    // negative rail (j >= c_out) negated
    bf16x8 wd[DX ? NB : 1][TERMS];
    if constexpr (DX) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            unsigned t3[3][4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int jl = c0 + 32 * (b * NW + wave) + 8 * lq + 2 * c;
                float v0 = sh.u.wl[l16][jl], v1 = sh.u.wl[l16][jl + 1];
                if (j_begin + jl >= c_out) v0 = -v0;
                if (j_begin + jl + 1 >= c_out) v1 = -v1;
                split3(v0, v1, t3[0][c], t3[1][c], t3[2][c]);
            }
#pragma unroll
            for (int t = 0; t < TERMS; t++) wd[b][t] = __builtin_bit_cast(bf16x8, make_uint4(t3[t][0], t3[t][1], t3[t][2], t3[t][3]));
        }
    }
    // where the upstream gradient of the wave's blocks lies in tile `split`: this lane's first eight values (columns 0 - 15;
    // those of columns 16 - 31 are 256 floats further), and the distance to the next tile of this workgroup
    int g_blk[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int j0 = j_begin + c0 + 32 * (b * NW + wave);
        g_blk[b] = q.gt_dedupe ? (j0 >= c_out ? j0 - c_out : j0) >> 5 : j0 >> 5;
        if (j0 >= J) g_blk[b] = 0;  // columns outside the problem: any finite values will do
    }
    const float* g_at = q.gtt + (size_t)split * q.gt_blocks * 1024 + ((lq & 1) * 32 + l16) * 16 + 8 * (lq >> 1);
    const size_t g_step = (size_t)q.splits * q.gt_blocks * 1024;
    float4 gv[2][2];
    auto fetch_g = [&](int b) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int h = 0; h < 2; h++) gv[s][h] = *(const float4*)(g_at + (size_t)g_blk[b] * 1024 + 256 * s + 4 * h);
    };

    fetch_g(0);

    floatx4 gw_acc[NB][2];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int s = 0; s < 2; s++) gw_acc[b][s] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    commit(0, x_first, ok_first);
    __syncthreads();  // the first tile's col is in place, and every wave has taken its weights out of wl
    // row i of the first product's two blocks is position zrow + 8 h; lane's results: positions ep + r and ep + 8 + r
    const int zrow = 16 * (l16 >> 3) + (l16 & 7), ep = 16 * (lq >> 1) + 4 * (lq & 1);
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4v* tr_ptr;
    int part = 0, tiles_left = q.tiles_each;
    auto store_part = [&]() {
        if (!q.store_part) return;
        // (opaque to the compiler, which would keep the stores' addresses in registers over the loop)
        int K = q.G.n_members, J = 2 * q.c_out;
        if constexpr (PARTS) asm volatile("" : "+s"(K), "+s"(J));
        float* pg = q.part + (size_t)blockIdx.y * q.part_stride + (size_t)(part * q.splits + split) * K * J;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const int j = j_begin + c0 + 32 * (b * NW + wave) + 16 * s + l16;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int k = 4 * lq + r;
                    if (k < K && j < J) pg[(size_t)k * J + j] = gw_acc[b][s][r];
                    if constexpr (PARTS) gw_acc[b][s][r] = 0.0f;
                }
            }
    };
    int buf = 0;
    for (int tile = split; tile < n_tiles; tile += q.splits, buf ^= 1) {
        ok_after = fetch(w_after, x_after);
        w_after = where(tile + 3 * q.splits);
        bf16x8 ag[TERMS];
#pragma unroll
        for (int t = 0; t < TERMS; t++) {
            const unsigned* row = sh.csg[buf][t][l16];
            const uint2 p0 = *(const uint2*)(row + ep / 2), p1 = *(const uint2*)(row + ep / 2 + 4);
            ag[t] = __builtin_bit_cast(bf16x8, make_uint4(p0.x, p0.y, p1.x, p1.y));
        }
        floatx4 d[2] = {floatx4{0.0f, 0.0f, 0.0f, 0.0f}, floatx4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int b = 0; b < NB; b++) {
            // Z[m][j] = sum_k col[k][m] * wcat[k][j], E = g * exp(-Z): eight positions of column 16 s + l16 per lane
            float e[2][8];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                // of three terms: lo hi + hi lo, mid mid + mid hi, hi mid + hi hi
                bf16x8 az[TERMS];
                if constexpr (TERMS == 3) {
                    az[0] = __builtin_bit_cast(bf16x8, sh.csz[buf][lq < 2 ? 2 : 0][lq & 1][zrow + 8 * h]);
                    az[1] = __builtin_bit_cast(bf16x8, sh.csz[buf][1][lq & 1][zrow + 8 * h]);
                    az[2] = __builtin_bit_cast(bf16x8, sh.csz[buf][0][lq & 1][zrow + 8 * h]);
                } else {
                    // (lanes from 32 on meet zero weights; what they read is finite)
                    az[0] = __builtin_bit_cast(bf16x8, sh.csz[buf][0][lq & 1][zrow + 8 * h]);
                }
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    floatx4 z = {0.0f, 0.0f, 0.0f, 0.0f};
                    if constexpr (TERMS == 3) {
                        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(az[0], wz[b][s][0], z, 0, 0, 0);
                        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(az[1], wz[b][s][1], z, 0, 0, 0);
                        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(az[2], wz[b][s][1], z, 0, 0, 0);
                    } else {
                        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(az[0], wz[b][s][0], z, 0, 0, 0);
                    }
                    const float4 gq = gv[s][h];
                    e[s][4 * h + 0] = gq.x * exp_neg(z[0]);
                    e[s][4 * h + 1] = gq.y * exp_neg(z[1]);
                    e[s][4 * h + 2] = gq.z * exp_neg(z[2]);
                    e[s][4 * h + 3] = gq.w * exp_neg(z[3]);
                }
            }
            // the next block's gradient, of this tile or of the workgroup's next one
            if (b + 1 == NB && tile + q.splits < n_tiles) g_at += g_step;
            fetch_g(b + 1 == NB ? 0 : b + 1);
            unsigned et[3][2][4];  // term, half of the columns, pairs of positions
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int c = 0; c < 4; c++) split3(e[s][2 * c], e[s][2 * c + 1], et[0][s][c], et[1][s][c], et[2][s][c]);
            // Gw[k][j] += sum_m col[k][m] * E[m][j], smallest terms first
            using Products = TermProducts<TERMS, 3>;
#pragma unroll
            for (int t = 0; t < Products::N; t++)
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const unsigned(&o)[4] = et[Products::b(t)][s];
                    gw_acc[b][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        ag[Products::a(t)], __builtin_bit_cast(bf16x8, make_uint4(o[0], o[1], o[2], o[3])), gw_acc[b][s], 0, 0, 0);
                }
            if constexpr (DX) {
                // dcol[k][m] = sum_j wd[j][k] * E[m][j] over this block's 32 columns, for positions 16 mb + l16; the wave
                // is alone in its block of LDS, whose accesses stay in the order that they are written here
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const int t = 2 - i;  // smallest first
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        uint2* row = sh.u.t.est[wave][16 * s + l16];
                        row[ep / 4] = make_uint2(et[t][s][0], et[t][s][1]);
                        row[ep / 4 + 2] = make_uint2(et[t][s][2], et[t][s][3]);
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int mb = 0; mb < 2; mb++) {
                        // 16 lanes read four columns of 16 positions; each gets its position's four columns
                        const uint2* at = &sh.u.t.est[wave][8 * lq + (l16 >> 2)][4 * mb + (l16 & 3)];
                        const short4v j0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at);
                        const short4v j4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 4 * (kBfEw / 2)));
                        const bf16x8 bd = __builtin_bit_cast(bf16x8, __builtin_shufflevector(j0, j4, 0, 1, 2, 3, 4, 5, 6, 7));
                        if constexpr (TERMS == 3) {
                            if (i > 1) d[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wd[b][2], bd, d[mb], 0, 0, 0);
                            if (i > 0) d[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wd[b][1], bd, d[mb], 0, 0, 0);
                        }
                        d[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wd[b][0], bd, d[mb], 0, 0, 0);
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
            }
        }
        // the next tile's col, into the buffer whose readers finished before the last barrier
        commit(buf ^ 1, x_next, ok_next);
        if constexpr (DX) {
#pragma unroll
            for (int mb = 0; mb < 2; mb++)
                sh.u.t.red[buf][wave][mb][lane] = make_float4(d[mb][0], d[mb][1], d[mb][2], d[mb][3]);
        }
        // every wave has read this tile's col, and written the next tile's and its share of red (whose other buffer
        // was read before this barrier)
        __syncthreads();
        if constexpr (DX) {
#pragma unroll
            for (int o = threadIdx.x; o < 2 * 64 * 4; o += NT) {
                const float* r = (const float*)&sh.u.t.red[buf][0][0][0] + o;
                float sum = r[0];
#pragma unroll
                for (int w = 1; w < NW; w++) sum += r[w * 2 * 64 * 4];
                const int k = 4 * (o >> 6 & 3) + (o & 3), m = tile * TM + 16 * (o >> 8) + (o >> 2 & 15);
                if (k < K && m < M) {
                    float* to = dg + (size_t)k * M + m;
                    *to = ADD ? *to + sum : sum;
                }
            }
        }
#pragma unroll
        for (int gp = 0; gp < GP; gp++)
#pragma unroll
            for (int e = 0; e < EP; e++) x_next[gp][e] = x_after[gp][e];
        ok_next = ok_after;
        if (PARTS && --tiles_left == 0) {
            store_part();
            part++;
            tiles_left = q.tiles_each;
        }
    }
    if constexpr (PARTS)
        for (; part < q.parts && part * q.splits + split < q.sums; part++) store_part();
    else
        store_part();
}

template <int NW, int NB, bool DX, bool LOOK>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 8 ? 4 : 3))) void k_bwd_small_k_bf16(SmallKParams q)
{
    constexpr int NT = 64 * NW, JW = 32 * NW * NB;
    __shared__ __attribute__((aligned(16))) SmallKShared<NW, NB, DX> sh;
    const int split = blockIdx.x / q.jblocks, jblock = blockIdx.x - split * q.jblocks, j_begin = jblock * JW;
    bool three = small_k_weights(q, sh, j_begin);
    if constexpr (LOOK) {
        // whether x and this workgroup's weights are bf16 numbers
        for (int e = threadIdx.x; e < q.found_rows * kScanBlocks; e += NT) three |= q.found[e] != 0;
        if (!__syncthreads_or(three)) {
            small_k_columns<1, NW, NB, DX, false, NB == 1>(q, sh, split, jblock, j_begin, 0);
            return;
        }
    } else {
        __syncthreads();
    }
    small_k_columns<3, NW, 1, DX, false, NB == 1>(q, sh, split, jblock, j_begin, 0);
    if constexpr (NB > 1) {
        static_assert(NB == 2, "one more pass");
        __syncthreads();
        small_k_weights(q, sh, j_begin);
        __syncthreads();
        small_k_columns<3, NW, 1, DX, true, false>(q, sh, split, jblock, j_begin, 32 * NW);
    }
}

int grid1d(long long total)
{
    long long blocks = (total + 255) / 256;
    if (blocks > 256 * 32) blocks = 256 * 32;
    return (int)(blocks < 1 ? 1 : blocks);
}

// VA: the A operand is a view of the shifted input planes (GemmParams::a_rows); the caller has checked that
// its rows and chunks are 16-byte aligned.
// Whether a product of views takes the eight-wave kernel, and with which NX (0: no): whole tiles of 64 NX x 256,
// whole chunks in every split, no empty split, an aligned B where B is read along k, and tiles for at least three
// quarters of the CUs (the callers have checked the views' alignment).
inline int big_tile_nx(const GemmParams& q, int batch, bool b_along_k)
{
    const int nx = big_rows(q.I) / 64;
    const bool b_ok = !b_along_k || (q.ldb % 4 == 0 && ((uintptr_t)q.b & 15) == 0 && q.b_batch_stride % 4 == 0);
    const bool ok = nx && q.J % kBigJ == 0 && q.K % kChunk == 0 && q.k_per_split % kChunk == 0 && b_ok &&
                    (long long)(q.splits - 1) * q.k_per_split < q.K &&
                    (long long)(q.I / (64 * nx)) * (q.J / kBigJ) * q.splits * batch >= 3 * kBigWorkgroups / 4;
    return ok ? nx : 0;
}

// Tile extents of the 128 x 128 kernel.  A dimension of at most 192 whose last (or only) 128-tile would be at
// most half full takes tiles of 64: the 2 x 2 wave arrangement would leave half of the waves of such a tile
// without work (one dimension only, j first).
inline void split_tile_extents(int I, int J, int& tile_i, int& tile_j)
{
    auto half_tiles = [](int n) { return n <= 3 * kTile / 2 && (n - 1) % kTile < kTile / 2; };
    tile_j = half_tiles(J) ? kTile / 2 : kTile;
    tile_i = tile_j == kTile && half_tiles(I) ? kTile / 2 : kTile;
}
// its tiles are all whole: what the epilogue that reads the upstream gradient in the caller's layout asks for
inline bool split_tiles_whole(int I, int J)
{
    int ti, tj;
    split_tile_extents(I, J, ti, tj);
    return I % ti == 0 && J % tj == 0;
}

template <bool AK, bool BK, int EPI, int PRODUCT, bool VA, bool VB, bool LOOK>
int launch_gemm_of(const GemmParams& q0, int batch, hipStream_t s)
{
    GemmParams q = q0;
    if constexpr (VA || VB) {
        const int nx = big_tile_nx(q, batch, !VB && !BK);
        // rows of 128: two chunks per trip where the chunks pair up
        const bool kc2 = nx == 2 && q.K % (2 * kChunk) == 0 && q.k_per_split % (2 * kChunk) == 0;
        if (nx) {
            q.tile_i = 64 * nx;
            q.tile_j = kBigJ;
            q.ni = q.I / q.tile_i;
            q.nj = q.J / q.tile_j;
            q.nz = q.splits * batch;
            if ((long long)q.ni * q.nj <= 16) {
                q.cluster_of = 2;
                q.cluster = q.ni * q.nj;
            } else if (q.nj <= q.ni) {
                q.cluster_of = 0;
                q.cluster = q.nj;
            } else {
                q.cluster_of = 1;
                q.cluster = q.ni;
            }
            const long long n_wg = (long long)q.ni * q.nj * q.nz;
            if (n_wg > 0x7fffffffLL) return GEO_SC_ERR_UNSUPPORTED;
            const dim3 grid((unsigned)std::min<long long>(n_wg, kBigWorkgroups));
            auto launch = [&](auto epi) {
                constexpr int E = decltype(epi)::value;
                if (nx == 4)
                    hipLaunchKernelGGL((k_gemm_big<AK, BK, E, PRODUCT, VA, VB, LOOK, 4>), grid, dim3(512), 0, s, q);
                else if (nx == 3)
                    hipLaunchKernelGGL((k_gemm_big<AK, BK, E, PRODUCT, VA, VB, LOOK, 3>), grid, dim3(512), 0, s, q);
                else if (kc2)
                    hipLaunchKernelGGL((k_gemm_big<AK, BK, E, PRODUCT, VA, VB, LOOK, 2, 2>), grid, dim3(512), 0, s, q);
                else
                    hipLaunchKernelGGL((k_gemm_big<AK, BK, E, PRODUCT, VA, VB, LOOK, 2>), grid, dim3(512), 0, s, q);
            };
            if constexpr (EPI == EPI_EXP_TIMES_G) {
                if (q.g_planes)
                    launch(std::integral_constant<int, EPI_EXP_TIMES_G_PLANES>());
                else
                    launch(std::integral_constant<int, EPI>());
            } else {
                launch(std::integral_constant<int, EPI>());
            }
            return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
        }
    }
    // the gradient in the caller's layout: views with whole tiles only (the caller decides with big_tile_nx and
    // split_tiles_whole)
    if (EPI == EPI_EXP_TIMES_G && q.g_planes && !(VA && split_tiles_whole(q.I, q.J))) return GEO_SC_ERR_UNSUPPORTED;
    split_tile_extents(q.I, q.J, q.tile_i, q.tile_j);
    q.ni = (q.I + q.tile_i - 1) / q.tile_i;
    q.nj = (q.J + q.tile_j - 1) / q.tile_j;
    q.nz = q.splits * batch;
    if ((long long)q.ni * q.nj <= 16) {
        q.cluster_of = 2;
        q.cluster = q.ni * q.nj;
    } else if (q.nj <= q.ni) {
        q.cluster_of = 0;
        q.cluster = q.nj;
    } else {
        q.cluster_of = 1;
        q.cluster = q.ni;
    }
    const long long n_groups = (long long)q.ni * q.nj * q.nz;
    if (n_groups > 0x7fffffffLL) return GEO_SC_ERR_UNSUPPORTED;
    dim3 grid((unsigned)n_groups);
    // The split kernel reads a K-major operand with dword loads and an I-major one with float4 along k:
    // every row start and every chunk start of the latter must lie on a 16-byte boundary.
    auto rows_aligned = [&](const float* base, long long ld, long long batch_stride) {
        return ld % 4 == 0 && ((uintptr_t)base & 15) == 0 && batch_stride % 4 == 0 && q.k_per_split % 4 == 0;
    };
    const bool a_vec = VA || AK || rows_aligned(q.a, q.lda, q.a_batch_stride);
    const bool b_vec = BK || rows_aligned(q.b, q.ldb, q.b_batch_stride);
    if constexpr (VB) {
        // (the caller has checked the view's alignment: rows of E and the runs of eight columns)
        hipLaunchKernelGGL((k_gemm_split<AK, BK, EPI, PRODUCT, false, true, LOOK>), grid, dim3(256), 0, s, q);
    } else if constexpr (VA) {
        if (!b_vec) return GEO_SC_ERR_UNSUPPORTED;
        if constexpr (EPI == EPI_EXP_TIMES_G) {
            if (q.g_planes)
                hipLaunchKernelGGL((k_gemm_split<AK, BK, EPI_EXP_TIMES_G_PLANES, PRODUCT, true, false, LOOK>), grid, dim3(256), 0, s, q);
            else
                hipLaunchKernelGGL((k_gemm_split<AK, BK, EPI, PRODUCT, true, false, LOOK>), grid, dim3(256), 0, s, q);
        } else {
            hipLaunchKernelGGL((k_gemm_split<AK, BK, EPI, PRODUCT, true, false, LOOK>), grid, dim3(256), 0, s, q);
        }
    } else {
        // (the scratch layout aligns the rows)
        if (!a_vec || !b_vec) return GEO_SC_ERR_UNSUPPORTED;
        hipLaunchKernelGGL((k_gemm_split<AK, BK, EPI, PRODUCT, false, false, LOOK>), grid, dim3(256), 0, s, q);
    }
    return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
}

template <bool AK, bool BK, int EPI, int PRODUCT, bool VA = false, bool VB = false>
int launch_gemm(const GemmParams& q, int batch, hipStream_t s)
{
    return q.one_term ? launch_gemm_of<AK, BK, EPI, PRODUCT, VA, VB, true>(q, batch, s)
                      : launch_gemm_of<AK, BK, EPI, PRODUCT, VA, VB, false>(q, batch, s);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct BwdLayout {
    long long m_total;
    int splits, m_per_split;
    Groups G;
    bool look;           // whether x and w are bf16 numbers is found out on the device
    bool fused_k;        // OR groups of at most 32 members: whole backward in one kernel, no col / E scratch
    int fused_jw;        // columns of E per workgroup of that kernel
    int fused_jblocks;   // its column blocks: each writes a dcol slice of its own
    int fused_splits;    // its workgroups per add group and column block
    int fused_tiles_each, fused_parts;  // of the bf16 kernel: tiles in a partial sum, partial sums per workgroup
    int fused_sums;      // partial sums with tiles at all
    int gt_dedupe;       // its upstream-gradient tiles serve both rails (c_out a multiple of 32)
    int gt_blocks;       // 32-column blocks of those tiles
    int ew_splits;       // parts of the positions in k_bwd_e_wgrad; 0: more members than it takes
    int ew_m_per_split, ew_tiles_each, ew_parts;  // tiles in a partial sum, partial sums per part of the positions
    int rows_per_chunk;  // add groups processed by one round of launches
    int dcol_slices;     // partial dcol arrays per round (column blocks of the fused kernel), rows_per_chunk * col_v apart
    bool dx_rows;        // the input-gradient GEMM sums the kernel rows itself (E read as a view shifted by image rows)
    bool dx_taps;        // it sums all kernel taps and writes dL/dx itself (E read as a view shifted by rows and columns)
    size_t off_zero;     // a block of zeros for that view
    size_t off_scan;     // what the scan's blocks found, and behind it the word that the products read
    bool view_col;       // the GEMMs read col as a view of the shifted input planes (k_shift_planes) kept in col's space
    int view_k_pad;      // entries per group of the view's row table
    size_t off_rows;     // the row table
    size_t col_v, e_v, part_v, w_v;  // floats per add group of each scratch array
    size_t off_col, off_e, off_dcol, off_part, off_wcat, off_wd, off_pos, off_gt, bytes;
};

// floats of the shifted input planes (one per kernel column and channel, over the padded rows and the
// output columns) including the run behind the last plane that a shifted row may touch
size_t view_floats(const Geometry& g)
{
    return (size_t)g.h_k * g.c_in * g.n * (g.w_in + 2 * g.pad_w) * g.ho + (size_t)g.w_k * g.ho;
}

inline long long pad4(long long v) { return (v + 3) & ~3LL; }

BwdLayout bwd_layout(const Geometry& g, int groups_per_round, int operand_bits)
{
    BwdLayout b;
    b.m_total = (long long)g.n * g.wo * g.ho;
    b.G.mode = g.mode;
    b.G.c_in = g.c_in;
    b.G.w_k = g.w_k;
    b.G.h_k = g.h_k;
    b.G.zu = g.z_unit;
    if (g.mode == GEO_SC_ACC_Z) {
        b.G.n_groups = g.c_in;
        b.G.n_members = g.w_k * g.h_k;
    } else if (g.mode == GEO_SC_ACC_FULL) {
        b.G.n_groups = 1;
        b.G.n_members = g.k_or * g.h_k;
    } else if (g.mode == GEO_SC_ACC_YZ) {
        b.G.n_groups = g.add_outer * g.h_k;
        b.G.n_members = g.z_unit * g.w_k;
    } else {
        b.G.n_groups = g.h_k;
        b.G.n_members = g.k_or;
    }
    const int K = b.G.n_members;
    b.look = looks_for_one_term(operand_bits, 2.0 * b.m_total * g.c_out * K * b.G.n_groups);
    b.fused_k = K <= kFusedK;
    // the bf16 kernel (at most 16 members) comes with 2, 4 or 8 waves of 32 columns, or 8 of 64 where under four of the
    // waves' 16 blocks stay empty (with 260 columns, operands of three terms: 417 us against 398 of 256-wide ones for
    // 64 -> 130 at 20 x 20, z_unit 4, batch 32) and the groups alone are two rounds of workgroups (otherwise three terms lose
    // more than one wins: 5 -> 250 at 28 x 28, batch 64: 405 us against 367); the fp32 one with 128 or 256 columns
    const long long fused_tiles = (b.m_total + kFusedTile - 1) / kFusedTile;
    const bool wide = b.look && K <= 16 && (512 - 2 * g.c_out % 512) % 512 < 128 &&
                      (long long)b.G.n_groups * ((2 * g.c_out + 511) / 512) >= 1024;
    b.fused_jw = 2 * g.c_out <= 64 && K <= 16 ? 64 : 2 * g.c_out <= 128 ? 128 : wide ? 512 : 256;
    b.fused_jblocks = (2 * g.c_out + b.fused_jw - 1) / b.fused_jw;
    b.gt_dedupe = g.c_out % 32 == 0;
    b.gt_blocks = b.gt_dedupe ? g.c_out / 32 : (2 * g.c_out + 31) / 32;
    {
        // about eight workgroups per CU in all, each looping over its share of the tiles
        const long long n_tiles = fused_tiles;
        const long long per_split = (long long)b.G.n_groups * b.fused_jblocks;
        long long want = 2048 / per_split;
        if (K <= 16) {
            // the bf16 kernel: the number of full rounds of workgroups that takes least, where one begins with what costs
            // it two tiles (its weights' terms).  12 -> 100, 1 x 1, 28 x 28, batch 64, step on floats: 161 us, 110; with
            // 2048 workgroups whatever their tiles 12 -> 200 took 289, now 163 (182 before)
            const long long at_once = b.fused_jw == 64 ? 1536 : b.fused_jw == 128 ? 768 : 512;
            long long least = 0;
            // (64 columns per wave: one workgroup per group and block, one partial sum)
            for (int rounds = 1; rounds <= 4; rounds++) {
                const long long splits = std::max(1LL, std::min(n_tiles, at_once * rounds / per_split));
                const long long cost = (splits * per_split + at_once - 1) / at_once * (2 + (n_tiles + splits - 1) / splits);
                if (!least || cost < least) {
                    least = cost;
                    want = splits;
                }
            }
        }
        if (want > n_tiles) want = n_tiles;
        if (want > 65535) want = 65535;
        b.fused_splits = (int)(want < 1 ? 1 : want);
        // (sums no longer than eight workgroups per CU would form)
        const long long most = std::max(1LL, std::min(n_tiles, 2048 / per_split));
        const long long each_wg = (n_tiles + b.fused_splits - 1) / b.fused_splits;
        b.fused_tiles_each = K > 16 ? 0 : b.fused_jw == 512 ? (int)each_wg : (int)std::min(each_wg, (n_tiles + most - 1) / most);
        b.fused_parts = K <= 16 ? (int)((each_wg + b.fused_tiles_each - 1) / b.fused_tiles_each) : 1;
        // Partial sum (part, split) has tiles where split + splits * part * tiles_each is one; they are numbered part * splits +
        // split, so those that have are the first ones, and what is left of the last parts is neither written nor read
        // (54 items of 3 x 22 x 17 -> 11, 632 tiles in 512 workgroups: 1024 sums 36 us to add, 632 of them 23)
        const long long before_last = (long long)b.fused_splits * (b.fused_parts - 1);
        b.fused_sums = (int)(before_last + std::min<long long>(b.fused_splits, n_tiles - before_last * b.fused_tiles_each));
    }
    // split the m-reduction of the weight gradient so that all groups' tiles together make about one
    // round of workgroups: three per CU for the 128 x 128 kernel (more splits only add partial sums to write
    // and reduce; C3: 0.85 ms with two rounds, 0.82 with one, 0.85 with a third of one), one per CU where the
    // eight-wave kernel will take the product (the shapes that read col as a view, with whole tiles)
    const bool quads = g.ho % 4 == 0 && g.h_in % 4 == 0 && (g.wo * g.ho) % kChunk == 0 && g.c_out % 2 == 0;
    const int big_i = !b.fused_k && quads && (2 * g.c_out) % kBigJ == 0 ? big_rows(K) : 0;
    const long long tiles = big_i ? (long long)(K / big_i) * (2 * g.c_out / kBigJ)
                                  : (long long)((K + kTile - 1) / kTile) * ((2 * g.c_out + kTile - 1) / kTile);
    long long want = (big_i ? kBigWorkgroups : 768) / (tiles * b.G.n_groups);
    if (want < 1) want = 1;
    long long per = (b.m_total + want - 1) / want;
    per = (per + kChunk - 1) / kChunk * kChunk;
    if (per < 256) per = 256;
    b.m_per_split = (int)(per > 0x7fffffffLL ? 0x7fffffffLL : per);
    b.splits = (int)((b.m_total + b.m_per_split - 1) / b.m_per_split);
    // one round of persistent workgroups for E and the weight gradient of operands of one term
    b.ew_splits = b.ew_m_per_split = b.ew_tiles_each = b.ew_parts = 0;
    if (b.look && !b.fused_k && K <= kEwMembers) {
        const int tm = 2 * g.c_out <= 64 ? 64 : 32;
        const long long jtiles = (2 * g.c_out + 127) / 128, m_tiles = (b.m_total + tm - 1) / tm;
        const long long parts = std::max(1LL, std::min(kEwWorkgroups / (jtiles * b.G.n_groups), m_tiles / 2));
        const long long tiles_each = (m_tiles + parts - 1) / parts;
        b.ew_m_per_split = (int)std::min<long long>(tiles_each * tm, 0x7fffffc0);
        b.ew_splits = (int)((b.m_total + b.ew_m_per_split - 1) / b.ew_m_per_split);
        // (sums over no more positions than those of the weight gradient's own product)
        b.ew_tiles_each = (int)std::min<long long>(tiles_each, std::max(1, b.m_per_split / tm));
        b.ew_parts = (int)((tiles_each + b.ew_tiles_each - 1) / b.ew_tiles_each);
    }
    // per-row scratch, each row's part padded to 64 floats so that float4 staging stays aligned
    auto pad64 = [](size_t v) { return (v + 63) & ~(size_t)63; };
    // (rows of col and of E start on 16-byte boundaries: the products that read them along a row do so four at a time)
    b.col_v = pad64((size_t)pad4(b.m_total) * K);
    b.e_v = pad64((size_t)b.m_total * pad4(2 * g.c_out));
    b.part_v = pad64((size_t)std::max(b.splits, b.fused_k ? b.fused_sums : b.ew_splits * b.ew_parts) * K * 2 * g.c_out);
    b.w_v = pad64((size_t)K * 2 * g.c_out);
    // the fused kernel needs neither col nor E
    const size_t col_alloc = b.fused_k ? 0 : b.col_v, e_alloc = b.fused_k ? 0 : b.e_v;
    b.dcol_slices = b.fused_k ? b.fused_jblocks : 1;
    // all groups in one round of launches unless that needs more than ~3 GB of scratch
    const size_t per_row = sizeof(float) * (col_alloc + b.dcol_slices * b.col_v + e_alloc + b.part_v + 2 * b.w_v);
    size_t rows = ((size_t)3 << 30) / per_row;
    if (rows < 1) rows = 1;
    if (rows > (size_t)b.G.n_groups) rows = b.G.n_groups;
    // the caller's cap on the add groups per round (less scratch, more launches)
    if (groups_per_round >= 1 && (size_t)groups_per_round < rows) rows = (size_t)groups_per_round;
    if (rows * b.splits > 65535 - kPrepRows) rows = (65535 - kPrepRows) / b.splits;  // grid.y = rows, the scan's and the positions', grid.z = rows * splits
    if (rows < 1) rows = 1;
    b.rows_per_chunk = (int)rows;
    // col as a view: whole quads in every row on both sides, chunks of kChunk positions inside one item, an
    // even number of rails' worth of columns (16-byte aligned rows of E), every group in one round, members
    // that all exist, and offsets that fit the stagers' 32-bit position index
    b.view_k_pad = (K + kChunk - 1) / kChunk * kChunk;
    b.view_col = !b.fused_k && g.ho % 4 == 0 && g.h_in % 4 == 0 && (g.wo * g.ho) % kChunk == 0 && g.c_out % 2 == 0 &&
                 rows == (size_t)b.G.n_groups && !(g.mode == GEO_SC_ACC_YZ && g.c_in % g.z_unit != 0) &&
                 view_floats(g) <= rows * col_alloc &&
                 (long long)g.n * (g.w_in + 2 * g.pad_w) * g.ho + (long long)g.w_k * g.ho < 0x7fffffffLL &&
                 view_floats(g) < ((size_t)1 << 33);  // 32-bit numbers of their quads
    // the kernel rows summed inside the input-gradient GEMM: y accumulation (group = kernel column, members =
    // (channel, kernel row)), whole quads in the rows of input and output, whole chunks of rails, every group in
    // one round, and the per-column result inside dcol's space
    b.dx_rows = !b.fused_k && g.mode == GEO_SC_ACC_Y && g.ho % 4 == 0 && g.h_in % 4 == 0 && g.h_k <= 8 &&
                (2 * g.c_out) % kChunk == 0 && rows == (size_t)b.G.n_groups &&
                (size_t)g.h_k * g.c_in * g.n * g.w_in * g.ho <= rows * b.col_v &&
                (long long)g.n * g.w_in * g.ho < 0x7fffffffLL && (long long)g.w_k * 2 * g.c_out < 0x7fffffffLL;
    // all kernel taps summed inside that GEMM, which then writes dL/dx itself (no per-column results, no pass that
    // adds them): the same without the conditions of that pass, where the result alone has tiles for the GPU
    // (a product per kernel column has h_k times as many)
    {
        int ti, tj;
        const long long m2 = (long long)g.n * g.w_in * g.h_in;
        split_tile_extents(g.c_in, m2 > 0x7fffffffLL ? 0x7fffffff : (int)m2, ti, tj);
        const long long tiles = (long long)((g.c_in + ti - 1) / ti) * ((m2 + tj - 1) / tj);
        b.dx_taps = !b.fused_k && g.mode == GEO_SC_ACC_Y && (2 * g.c_out) % kChunk == 0 &&
                    rows == (size_t)b.G.n_groups && m2 < 0x7fff0000LL &&
                    (long long)g.w_k * g.h_k * 2 * g.c_out < 0x7fffffffLL && tiles >= 2 * kBigWorkgroups;
    }
    size_t o = 0;
    b.off_col = o;  o += align256(sizeof(float) * rows * col_alloc);
    b.off_e = o;    o += align256(sizeof(float) * rows * e_alloc);
    // (no per-group input gradients where the product over all taps writes dL/dx itself)
    b.off_dcol = o; o += b.dx_taps ? 0 : align256(sizeof(float) * rows * b.col_v * b.dcol_slices);
    b.off_part = o; o += align256(sizeof(float) * rows * b.part_v);
    b.off_wcat = o; o += align256(sizeof(float) * rows * b.w_v);
    b.off_wd = o;   o += align256(sizeof(float) * rows * b.w_v);
    b.off_pos = o;  o += 3 * align256(sizeof(int) * (size_t)b.m_total);
    {
        // [m][c_out], or the fused kernel's tiles of 32 positions x 32 columns
        const size_t tiled = (size_t)((b.m_total + kFusedTile - 1) / kFusedTile) * b.gt_blocks * 1024;
        const size_t plain = (size_t)b.m_total * g.c_out;
        b.off_gt = o;
        o += align256(sizeof(float) * (b.fused_k && tiled > plain ? tiled : plain));
    }
    b.off_rows = o;
    // (and behind it the entries that the eight-wave kernel reads ahead of the last chunk)
    o += align256(sizeof(long long) * ((size_t)b.G.n_groups * b.view_k_pad + 2 * kChunk + 8));
    b.off_zero = o;
    o += 256;
    b.off_scan = o;
    o += align256(sizeof(int) * (kScanBlocks * kScanRows + 1));
    b.bytes = o;
    return b;
}

}  // namespace

size_t backward_workspace_bytes(const Geometry& g, int groups_per_round, int operand_bits)
{
    return bwd_layout(g, groups_per_round, operand_bits).bytes;
}

int launch_conv_backward(const Geometry& g, int groups_per_round, int operand_bits, const float* x, const float* w,
                         const float* gy, float* gx, float* gw, void* workspace, size_t workspace_bytes, hipStream_t s)
{
    const BwdLayout L = bwd_layout(g, groups_per_round, operand_bits);  // once per call: sizes the check and the launches alike
    if (workspace_bytes < L.bytes) return GEO_SC_ERR_WORKSPACE;
    if (L.m_total > 0x7fffffffLL) return GEO_SC_ERR_INVALID_ARGUMENT;
    char* ws = (char*)workspace;
    float* col = (float*)(ws + L.off_col);
    float* e = (float*)(ws + L.off_e);
    float* dcol = (float*)(ws + L.off_dcol);
    float* part = (float*)(ws + L.off_part);
    float* wcat = (float*)(ws + L.off_wcat);
    float* wd = (float*)(ws + L.off_wd);
    const Groups& G = L.G;
    const int M = (int)L.m_total, K = G.n_members, J = 2 * g.c_out;
    const int col_ld = (int)pad4(M), e_ld = (int)pad4(J);  // row strides of col and E
    const long long x_total = (long long)g.n * g.c_in * g.w_in * g.h_in;
    if (x_total > 0x7fffffffLL || K > 65535 * kIm2colMembers) return GEO_SC_ERR_UNSUPPORTED;
    if ((long long)g.n * g.c_out * g.wo * g.ho > 0x7fffffffLL) return GEO_SC_ERR_UNSUPPORTED;
    const size_t pos_stride = align256(sizeof(int) * (size_t)M) / sizeof(int);
    int* pos_base = (int*)(ws + L.off_pos);
    int* pos_arow = pos_base + pos_stride;
    int* pos_bcol = pos_arow + pos_stride;
    float* gt = (float*)(ws + L.off_gt);
    const int m_blocks = grid1d(M);
    // four elements per thread in im2col / col2im where rows of the input and of the output are whole quads
    const bool quad_rows = g.h_in % 4 == 0 && g.ho % 4 == 0;
    const bool im2col_v4 = quad_rows && ((uintptr_t)x & 15) == 0;
    const bool col2im_v4 = quad_rows && g.h_k <= 8 && gx && ((uintptr_t)gx & 15) == 0;
    const bool fused = L.fused_k;
    // col as a view of the shifted input planes (one round holds every group then)
    const bool view = L.view_col && ((uintptr_t)x & 15) == 0;
    // what the scan of the operands leaves, and the word that it comes down to; NULL: three terms, nobody looks
    const bool look = L.look;
    int* found = look ? (int*)(ws + L.off_scan) : nullptr;
    int* one_term = look ? found + kScanBlocks * kScanRows : nullptr;
    const int n_scan_rows = look ? scan_rows(x_total) : 0;
    // the position tables serve the gathers of im2col and of the fused kernels
    const PositionTable positions = {pos_base, pos_arow, pos_bcol, M, g.c_in, g.w_in, g.h_in, g.pad_w, g.pad_h, g.wo, g.ho};
    if (fused) {
        // (the kernel for up to 16 members takes operands of one term as such)
        const int rows = K <= 16 ? n_scan_rows : 0;
        hipLaunchKernelGGL(k_position_table, dim3(rows ? std::max(m_blocks, kScanBlocks) : m_blocks, 1 + rows), dim3(256), 0, s,
                           positions, x, x_total, found);
    }
    // Where the first product reads col as a view and its tiles are whole (the eight-wave kernel in every round,
    // or the 128 x 128 kernel), its epilogue reads the upstream gradient as it is (items of whole 32-position
    // blocks, 16-byte aligned): no transposed copy.
    // (the 128 x 128 kernel with full-width tiles only: with tiles of 64 columns the strided loads cost what the
    // small transposed copy does)
    bool g_planes = !fused && view && (g.wo * g.ho) % 32 == 0 && ((uintptr_t)gy & 15) == 0;
    if (g_planes && !(split_tiles_whole(M, J) && J % kTile == 0)) {
        GemmParams t = {};
        t.I = M; t.J = J; t.K = K; t.splits = 1; t.k_per_split = K;
        for (int v0 = 0; v0 < G.n_groups; v0 += L.rows_per_chunk) {
            const int nv = G.n_groups - v0 < L.rows_per_chunk ? G.n_groups - v0 : L.rows_per_chunk;
            if (!big_tile_nx(t, nv, false)) g_planes = false;
        }
    }
    {
        const int npos = g.wo * g.ho;
        if (fused) {
            hipLaunchKernelGGL(k_tile_grad, dim3((M + kFusedTile - 1) / kFusedTile, L.gt_blocks), dim3(256), 0, s, gy, gt, M,
                               g.c_out, npos, L.gt_blocks, L.gt_dedupe);
        } else if (!g_planes) {
            if (g.n > 65535) return GEO_SC_ERR_UNSUPPORTED;  // grid.z of the transpose
            hipLaunchKernelGGL(k_transpose_grad, dim3((npos + 31) / 32, (g.c_out + 31) / 32, g.n), dim3(256), 0, s, gy, gt,
                               g.c_out, npos);
        }
    }
    // dL/dx from dcol of the groups [v0, v0 + nv)
    auto col2im = [&](int v0, int nv) {
        const int n_planes = g.n * g.c_in;
        // (from two tiles of items and 2^18 elements on: 1024 elements, 64 items 4.6 us and 3.5 with the other kernel, 128 items 4.2
        // and 3.9, 256 items 4.9 and 5.4, 1024 items 5.2 and 11.5; 4096 elements, 64 items 4.6 and 6.3)
        if (g.wo * g.ho == 1 && g.n >= 64 && x_total >= 1 << 18) {
            const int tiles = (g.c_in * g.w_in * g.h_in + 31) / 32, rows = (g.n + 31) / 32;
            hipLaunchKernelGGL(k_col2im_one, dim3(tiles, std::min(rows, 1024)), dim3(256), 0, s, dcol, gx, v0, nv, g.n, G, g.w_in,
                               g.h_in, g.pad_w, g.pad_h, L.col_v);
        } else if (col2im_v4) {
            hipLaunchKernelGGL(k_col2im_rows_v4, dim3(grid1d((long long)n_planes * (g.w_in * g.h_in / 4))), dim3(256), 0, s, dcol, gx,
                               v0, nv, L.m_total, n_planes, G, g.w_in, g.h_in, g.pad_w, g.pad_h, g.wo, g.ho, L.col_v);
        } else {
            hipLaunchKernelGGL(k_col2im_rows, dim3(grid1d(x_total)), dim3(256), 0, s, dcol, gx, v0, nv, L.m_total,
                               (unsigned)x_total, (unsigned)g.n, G, g.w_in, g.h_in, g.pad_w, g.pad_h, g.wo, g.ho, L.col_v);
        }
    };
    int rc;
    if (fused) {
        if (!gx && !gw) return GEO_SC_OK;
        const int ks = (K + 1) / 2;
        const int jw = L.fused_jw;
        const size_t slice = (size_t)L.rows_per_chunk * L.col_v;
        if ((long long)L.fused_splits * L.fused_jblocks > 0x7fffffffLL) return GEO_SC_ERR_UNSUPPORTED;
        for (int v0 = 0; v0 < G.n_groups; v0 += L.rows_per_chunk) {
            const int nv = G.n_groups - v0 < L.rows_per_chunk ? G.n_groups - v0 : L.rows_per_chunk;
            // channel blocks with a ragged end have members that do not exist: their zeros come from the plain kernel
            const bool ragged = G.mode == GEO_SC_ACC_YZ && g.c_in % G.zu != 0;
            const dim3 w_tiles((g.c_in * g.w_k * g.h_k + 31) / 32, (g.c_out + 31) / 32);
            if (ragged) {
                int wb = grid1d((long long)K * g.c_out);
                hipLaunchKernelGGL(k_weight_operands, dim3(wb > 256 ? 256 : wb, nv), dim3(256), 0, s, w, wcat, wd, v0,
                                   g.c_out, G, L.w_v);
            } else {
                hipLaunchKernelGGL(k_weight_cat_tiled, w_tiles, dim3(256), 0, s, w, wcat, v0, nv, g.c_out, G, L.w_v);
            }
            const dim3 grid(L.fused_splits * L.fused_jblocks, nv);
            {
#define GEO_SC_FUSED_K(KS, NB, DX)                                                                                     \
    hipLaunchKernelGGL((k_bwd_small_k<KS, NB, DX>), grid, dim3(256), 0, s, x, wcat, gt, pos_base, pos_arow,             \
                       pos_bcol, part, dcol, G, v0, M, g.w_in, g.h_in, g.c_out, L.fused_jblocks, L.fused_splits,        \
                       gw ? 1 : 0, L.gt_blocks, L.gt_dedupe, L.w_v, L.part_v, L.col_v, slice)
#define GEO_SC_FUSED_NB_DX(KS)                                                                                         \
    do {                                                                                                               \
        if (jw == 128) {                                                                                               \
            if (gx) GEO_SC_FUSED_K(KS, 1, true); else GEO_SC_FUSED_K(KS, 1, false);                                    \
        } else {                                                                                                       \
            if (gx) GEO_SC_FUSED_K(KS, 2, true); else GEO_SC_FUSED_K(KS, 2, false);                                    \
        }                                                                                                              \
    } while (0)
                if (ks <= 8) {
                    SmallKParams p = {x, wcat, gt, pos_base, pos_arow, pos_bcol, found, part, dcol, G, v0, M, g.w_in, g.h_in,
                                      g.c_out, L.fused_jblocks, L.fused_splits, gw ? 1 : 0, L.gt_blocks, L.gt_dedupe, n_scan_rows,
                                      L.fused_tiles_each, L.fused_parts, L.fused_sums,
                                      L.w_v, L.part_v, L.col_v, slice};
                    auto launch = [&](auto dx, auto looks) {
                        constexpr bool DX = decltype(dx)::value, LOOK = decltype(looks)::value;
                        if (jw == 64)
                            hipLaunchKernelGGL((k_bwd_small_k_bf16<2, 1, DX, LOOK>), grid, dim3(128), 0, s, p);
                        else if (jw == 128)
                            hipLaunchKernelGGL((k_bwd_small_k_bf16<4, 1, DX, LOOK>), grid, dim3(256), 0, s, p);
                        else if (jw == 256)
                            hipLaunchKernelGGL((k_bwd_small_k_bf16<8, 1, DX, LOOK>), grid, dim3(512), 0, s, p);
                        else  // (only where a call looks)
                            hipLaunchKernelGGL((k_bwd_small_k_bf16<8, 2, DX, true>), grid, dim3(512), 0, s, p);
                    };
                    if (gx && look)
                        launch(std::true_type(), std::true_type());
                    else if (gx)
                        launch(std::true_type(), std::false_type());
                    else if (look)
                        launch(std::false_type(), std::true_type());
                    else
                        launch(std::false_type(), std::false_type());
                }
                else if (ks <= 12) GEO_SC_FUSED_NB_DX(12);
                else GEO_SC_FUSED_NB_DX(16);
#undef GEO_SC_FUSED_NB_DX
#undef GEO_SC_FUSED_K
            }
            if (gw) {
                // few partial sums (wide layers): coalesced tiles; many: the kernel that adds eight splits side by side
                if (L.fused_sums <= 4)
                    hipLaunchKernelGGL(k_reduce_wgrad_tiled, w_tiles, dim3(256), 0, s, part, w, gw, v0, nv,
                                       WgradSplits{L.fused_sums, 0, nullptr}, g.c_out, G, L.part_v, WgradOperands{});
                else
                    hipLaunchKernelGGL(k_reduce_wgrad, dim3((K * g.c_out + 31) / 32, nv), dim3(256), 0, s, part, w, gw, v0,
                                       WgradSplits{L.fused_sums, 0, nullptr}, g.c_out, G, L.part_v, WgradOperands{});
            }
            if (gx && L.dcol_slices > 1)
                hipLaunchKernelGGL(k_sum_slices, dim3(grid1d((long long)((size_t)nv * L.col_v / 4))), dim3(256), 0, s, dcol,
                                   (size_t)nv * L.col_v, L.dcol_slices, slice);
            if (gx) col2im(v0, nv);
        }
        return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
    }
    long long* view_rows = (long long*)(ws + L.off_rows);
    for (int v0 = 0; v0 < G.n_groups; v0 += L.rows_per_chunk) {
        const int nv = G.n_groups - v0 < L.rows_per_chunk ? G.n_groups - v0 : L.rows_per_chunk;
        const bool dx_taps = gx && L.dx_taps;
        const bool dx_rows = dx_taps || (gx && L.dx_rows && ((uintptr_t)gx & 15) == 0);
        {
            // weight operands of the round's groups; with the first round the view's row table and the block of zeros
            PrepParams pp = {};
            pp.w = w; pp.wcat = wcat; pp.wd = wd; pp.g0 = v0; pp.c_out = g.c_out; pp.G = G; pp.g_stride = L.w_v;
            pp.dx_rows = dx_taps ? 2 : dx_rows ? 1 : 0;
            if (v0 == 0 && view) {
                pp.view_rows = view_rows; pp.view_groups = G.n_groups; pp.view_k_pad = L.view_k_pad; pp.ho = g.ho;
                pp.plane = (long long)g.n * (g.w_in + 2 * g.pad_w) * g.ho;
            }
            if (dx_rows) pp.zero = (float*)(ws + L.off_zero);
            long long work = (long long)K * g.c_out;
            if (dx_rows && (long long)g.w_k * J * g.c_in > work) work = (long long)g.w_k * J * g.c_in;
            if (pp.view_rows && (long long)G.n_groups * L.view_k_pad > work) work = (long long)G.n_groups * L.view_k_pad;
            pp.groups = nv;
            int wb = std::min(grid1d(work), 256);
            if (v0 == 0) {
                pp.x = x; pp.x_total = x_total; pp.w_total = (long long)g.c_out * g.c_in * g.w_k * g.h_k; pp.found = found;
                pp.scan_blocks = n_scan_rows * kScanBlocks;
                pp.positions = positions;
                pp.position_blocks = view ? 0 : std::min(m_blocks, kScanBlocks);
                wb = std::max(wb, kPrepColumns);
            }
            auto more_rows = [&](int columns) { return (pp.scan_blocks + pp.position_blocks + columns - 1) / columns; };
            const bool ragged = G.mode == GEO_SC_ACC_YZ && g.c_in % G.zu != 0;
            const int channels = ragged ? 0 : prep_tile_channels(g.c_in, g.c_out, g.w_k * g.h_k, dx_rows);
            if (channels) {
                const long long tiles = (long long)((g.c_out + 31) / 32) * ((g.c_in + channels - 1) / channels);
                pp.groups = (int)std::min<long long>((tiles + kScanBlocks - 1) / kScanBlocks, 8);  // rows of tiles
                hipLaunchKernelGGL(k_bwd_prep_tiled, dim3(kScanBlocks, pp.groups + more_rows(kScanBlocks)), dim3(256), 0, s, pp, nv,
                                   __builtin_ctz((unsigned)channels));
            } else {
                hipLaunchKernelGGL(k_bwd_prep, dim3(wb, nv + more_rows(wb)), dim3(256), 0, s, pp);
            }
        }
        if (view) {
            const long long plane = (long long)g.n * (g.w_in + 2 * g.pad_w) * g.ho;
            const long long quads = (long long)g.h_k * g.c_in * plane / 4;
            auto shift = [&](auto per_thread) {
                constexpr int Q = decltype(per_thread)::value;
                hipLaunchKernelGGL((k_shift_planes<Q>), dim3(grid1d((quads + Q - 1) / Q)), dim3(256), 0, s, x, col, found,
                                   n_scan_rows, one_term, (unsigned)quads, g.n, g.c_in, g.w_in, g.h_in, g.pad_w, g.pad_h, g.ho);
            };
            if (quads >= kShiftMany)
                shift(std::integral_constant<int, 4>());
            else
                shift(std::integral_constant<int, 1>());
        } else if (im2col_v4) {
            const int q_blocks = grid1d(M / 4);
            hipLaunchKernelGGL(k_im2col_rows_v4,
                               dim3(q_blocks > 1024 ? 1024 : q_blocks, (K + kIm2colMembers - 1) / kIm2colMembers, nv),
                               dim3(256), 0, s, x, col, found, n_scan_rows, one_term, pos_base, pos_arow, pos_bcol, v0, M, G, g.w_in, g.h_in, L.col_v);
        } else {
            hipLaunchKernelGGL(k_im2col_rows,
                               dim3(m_blocks > 1024 ? 1024 : m_blocks, (K + kIm2colMembers - 1) / kIm2colMembers, nv),
                               dim3(256), 0, s, x, col, found, n_scan_rows, one_term, pos_base, pos_arow, pos_bcol, v0, M, col_ld, G, g.w_in, g.h_in, L.col_v);
        }
        // E[v][m][j] = g * exp(-(col_v^T . wcat_v)), col stored [K][M]
        GemmParams q1 = {};
        q1.one_term = one_term;
        q1.a = col; q1.b = wcat; q1.c = e;
        q1.I = M; q1.J = J; q1.K = K;
        q1.lda = col_ld; q1.ldb = J; q1.ldc = e_ld;
        q1.splits = 1; q1.k_per_split = K; q1.c_split_stride = 0;
        q1.a_batch_stride = (long long)L.col_v; q1.b_batch_stride = (long long)L.w_v;
        q1.c_batch_stride = (long long)L.e_v;
        q1.g = g_planes ? gy : gt; q1.g_planes = g_planes; q1.c_out = g.c_out; q1.npos = g.wo * g.ho;
        const bool ew = gw && L.ew_splits;
        if (ew) {
            // E and the partial sums of the weight gradient at once where the operands are one term
            EwParams p = {};
            p.col = (const bf16_bits*)col; p.wcat = wcat; p.g = g_planes ? gy : gt; p.e = e; p.part = part; p.one_term = one_term;
            p.rows = view ? view_rows : nullptr; p.rows_batch = L.view_k_pad; p.item = g.wo * g.ho; p.skip = (g.w_k - 1) * g.ho;
            p.col_ld = col_ld; p.col_v = L.col_v; p.w_v = L.w_v; p.e_v = L.e_v; p.part_v = L.part_v;
            p.M = M; p.K = K; p.J = J; p.e_ld = e_ld; p.c_out = g.c_out; p.npos = g.wo * g.ho;
            p.m_per_split = L.ew_m_per_split; p.jtiles = (J + 127) / 128;
            p.splits = L.ew_splits; p.tiles_each = L.ew_tiles_each; p.parts = L.ew_parts;
            p.store_e = gx || !view;
            const dim3 grid((unsigned)(L.ew_splits * p.jtiles), nv);
            auto launch = [&](auto blocks) {
                constexpr int B = decltype(blocks)::value;
                if (J <= 64)  // (never the gradient as it is: whole tiles of 128 columns)
                    hipLaunchKernelGGL((k_bwd_e_wgrad<B, 2, false>), grid, dim3(256), 0, s, p);
                else if (g_planes)
                    hipLaunchKernelGGL((k_bwd_e_wgrad<B, 4, true>), grid, dim3(256), 0, s, p);
                else
                    hipLaunchKernelGGL((k_bwd_e_wgrad<B, 4, false>), grid, dim3(256), 0, s, p);
            };
            switch ((K + 31) / 32) {
            case 2: launch(std::integral_constant<int, 2>()); break;
            case 3: launch(std::integral_constant<int, 3>()); break;
            case 4: launch(std::integral_constant<int, 4>()); break;
            case 5: launch(std::integral_constant<int, 5>()); break;
            default: launch(std::integral_constant<int, 6>()); break;
            }
            q1.one_term_elsewhere = 1;
        }
        q1.a_rows = view_rows; q1.a_rows_batch = L.view_k_pad; q1.a_item = g.wo * g.ho; q1.a_skip = (g.w_k - 1) * g.ho;
        rc = view ? launch_gemm<true, true, EPI_EXP_TIMES_G, PRODUCT_E, true>(q1, nv, s)
                  : launch_gemm<true, true, EPI_EXP_TIMES_G, PRODUCT_E>(q1, nv, s);
        if (rc != GEO_SC_OK) return rc;
        if (gw) {
            // partial Gw[v][s][k][j] = sum_{m in split s} col_v[k][m] * E_v[m][j]
            GemmParams q2 = {};
            q2.one_term = one_term;
            q2.one_term_elsewhere = ew;
            q2.a = col; q2.b = e; q2.c = part;
            q2.I = K; q2.J = J; q2.K = M;
            q2.lda = col_ld; q2.ldb = e_ld; q2.ldc = J;
            q2.splits = L.splits; q2.k_per_split = L.m_per_split; q2.c_split_stride = (long long)K * J;
            q2.a_batch_stride = (long long)L.col_v; q2.b_batch_stride = (long long)L.e_v;
            q2.c_batch_stride = (long long)L.part_v;
            q2.a_rows = view_rows; q2.a_rows_batch = L.view_k_pad; q2.a_item = g.wo * g.ho; q2.a_skip = (g.w_k - 1) * g.ho;
            rc = view ? launch_gemm<false, true, EPI_STORE, PRODUCT_DW, true>(q2, nv, s)
                      : launch_gemm<false, true, EPI_STORE, PRODUCT_DW>(q2, nv, s);
            if (rc != GEO_SC_OK) return rc;
            WgradOperands again = {};
            if (!view) again = {col, one_term, e, M, col_ld, e_ld, L.col_v, L.e_v};
            // Few partial sums and many weights: coalesced tiles (512 -> 512, 3 x 3, three partial sums: 50 -> 15.6 us;
            // the other kernel reads w and writes dL/dw one element per line).  Not where eight splits side by side are
            // what fills the GPU.
            const dim3 w_tiles((g.c_in * g.w_k * g.h_k + 31) / 32, (g.c_out + 31) / 32);
            const WgradSplits parts = {L.splits, L.ew_splits * L.ew_parts, ew ? one_term : nullptr};
            if (std::max(L.splits, L.ew_splits * L.ew_parts) <= 8 && (long long)w_tiles.x * w_tiles.y >= 512 && w_tiles.y <= 65535)
                hipLaunchKernelGGL(k_reduce_wgrad_tiled, w_tiles, dim3(256), 0, s, part, w, gw, v0, nv, parts,
                                   g.c_out, G, L.part_v, again);
            else
                hipLaunchKernelGGL(k_reduce_wgrad, dim3((K * g.c_out + 31) / 32, nv), dim3(256), 0, s, part, w, gw, v0, parts,
                                   g.c_out, G, L.part_v, again);
        }
        if (!gx) continue;
        if (dx_taps) {
            // gx[n][ci][(p, c)] = sum_(u, v, j) wdx[(j, v, u)][ci] * E_v[(n, p + pad_w - u, c + pad_h - v)][j]: every
            // kernel tap summed inside one GEMM (w_k h_k times the k of the product per tap, one output instead of one
            // per tap, stored in the caller's layout); the operand wdx and the block of zeros come from k_bwd_prep
            float* zero = (float*)(ws + L.off_zero);
            const int k9 = g.w_k * g.h_k * J;
            const long long m2 = (long long)g.n * g.w_in * g.h_in;
            GemmParams q3 = {};
            q3.one_term = one_term;
            q3.a = wd; q3.b = e; q3.c = gx;
            q3.I = g.c_in; q3.J = (int)m2; q3.K = k9;
            q3.lda = g.c_in; q3.ldb = e_ld; q3.ldc = m2;
            q3.splits = 1; q3.k_per_split = k9; q3.c_split_stride = 0;
            q3.a_batch_stride = 0; q3.b_batch_stride = (long long)L.e_v; q3.c_batch_stride = 0;
            q3.sh_zero = zero; q3.sh_j = J; q3.sh_wo = g.wo; q3.sh_ho = g.ho; q3.sh_win = g.w_in; q3.sh_hin = g.h_in;
            q3.sh_pad = g.pad_w; q3.sh_padh = g.pad_h; q3.sh_wk = g.w_k; q3.sh_hk = g.h_k;
            q3.c_plane = g.w_in * g.h_in;
            if ((rc = launch_gemm<true, false, EPI_STORE_ITEMS, PRODUCT_DX, false, true>(q3, 1, s)) != GEO_SC_OK) return rc;
            continue;
        }
        if (dx_rows) {
            // d[v][ci][(n, p, b)] = sum_(u, j) wd_v[j][(ci, u)] * E_v[(n, p + pad - u, b)][j]: the kernel rows
            // summed inside the GEMM (three times the k of the product per (ci, u), a third of its rows and of
            // its output), then the kernel columns by k_shift_sum_v4; the operand wdx and the block of zeros
            // come from k_bwd_prep
            float* zero = (float*)(ws + L.off_zero);
            const int k3 = g.w_k * J;
            const long long m2 = (long long)g.n * g.w_in * g.ho;
            GemmParams q3 = {};
            q3.one_term = one_term;
            q3.a = wd; q3.b = e; q3.c = dcol;
            q3.I = g.c_in; q3.J = (int)m2; q3.K = k3;
            q3.lda = g.c_in; q3.ldb = e_ld; q3.ldc = m2;
            q3.splits = 1; q3.k_per_split = k3; q3.c_split_stride = 0;
            q3.a_batch_stride = (long long)L.w_v; q3.b_batch_stride = (long long)L.e_v;
            q3.c_batch_stride = (long long)g.c_in * m2;
            q3.sh_zero = zero; q3.sh_j = J; q3.sh_wo = g.wo; q3.sh_ho = g.ho; q3.sh_win = g.w_in; q3.sh_hin = g.ho;
            q3.sh_pad = g.pad_w; q3.sh_padh = 0; q3.sh_wk = g.w_k; q3.sh_hk = 1;
            if ((rc = launch_gemm<true, false, EPI_STORE, PRODUCT_DX, false, true>(q3, nv, s)) != GEO_SC_OK) return rc;
            const long long quads = (long long)g.n * g.c_in * g.w_in * g.h_in / 4;
            hipLaunchKernelGGL(k_shift_sum_v4, dim3(grid1d(quads)), dim3(256), 0, s, dcol, gx, quads, g.n, g.c_in, g.w_in,
                               g.h_in, g.h_k, g.pad_h, g.ho);
            continue;
        }
        // dcol[v][k][m] = sum_j wd_v[j][k] * E_v[m][j]
        GemmParams q3 = {};
        q3.one_term = one_term;
        q3.a = wd; q3.b = e; q3.c = dcol;
        q3.I = K; q3.J = M; q3.K = J;
        q3.lda = K; q3.ldb = e_ld; q3.ldc = M;
        q3.splits = 1; q3.k_per_split = e_ld; q3.c_split_stride = 0;
        q3.a_batch_stride = (long long)L.w_v; q3.b_batch_stride = (long long)L.e_v;
        q3.c_batch_stride = (long long)L.col_v;
        if ((rc = launch_gemm<true, false, EPI_STORE, PRODUCT_DX>(q3, nv, s)) != GEO_SC_OK) return rc;
        col2im(v0, nv);
    }
    return hipGetLastError() == hipSuccess ? GEO_SC_OK : GEO_SC_ERR_LAUNCH;
}

}  // namespace geo_sc
