// Row-block kernels of the SDDMM engine for gfx950 (MI355X), for patterns that are locally dense: neighbouring rows with
// mostly the same columns (the window of local attention).  32 rows are a row block; the columns that any of them has,
// in ascending order, are cut into tiles of 32; a (row block, tile) pair is computed whole on the matrix cores.  A row's
// nonzeros of a tile are consecutive in the sorted S, so a 32-bit mask and the position of the first one say where every
// entry lies.  No list of nonzeros, no column per nonzero: 384 bytes per tile of up to 1024 nonzeros.
//
// Arithmetic: fp32 operands as three bf16 parts, eight products of parts, added up as in add_products (bf16_parts.hpp).
// What parts cannot carry is found and computed once more: with scaled operands where bits lie under bf16's smallest subnormal,
// in fp32 where there are infinities, NaNs or sums beyond the range.
//
// A unit is a row block and a range of its tiles, dealt tile by tile to the four waves of a workgroup.  A row block of
// long rows (tokens that look at all others) is several units.
//   sddmm_block_kernel: out = val * (W H^T).  A wave keeps the parts of the 32 rows of W in registers (12 for every 16
//     elements of K) and streams the H rows of its tiles past them, requested two steps ahead, straight into the
//     operands' lanes.  The dot products go through LDS, from where half a wave takes a row: entries found by mask,
//     epilogue, stores of up to 32 neighbours.  SOFTMAX: all scores of a row block stay there, and what is written is
//     their softmax: no second pass over out.
//   sddmm_block_spmm_kernel: Y = X H.  The tile of X is put together from the nonzeros in LDS, the 32 columns' rows of H
//     are the other operand; the waves' sums are added up in order through LDS.
//
// What bounds it: vector instructions, 3640 clocks of them per tile for scores and softmax (cutting H into parts and adding
// 1500, masks, exponentials, stores and the cutting of W the rest) and 3320 for the product, beside 1024 of matrix
// instructions, 27 and 35 % of which lie under vector ones; that fills a SIMD for 59 and 53 % of the time its compute unit
// has work, waits the rest: 2.5 units per compute unit, first loads, the barrier between tiles and rows
// (profiles/row_blocks_attention_k64.txt).  Window of 128 on either side of 16,384 tokens, 32 full rows and columns, K = 64
// (5.2 M nonzeros, 5602 tiles), us: scores and softmax 22 + 5.5 for the long rows (tile kernel and three softmax kernels 41 +
// 34), product 19 + 4 (walk over the pattern 66 + 5).  The relative error against 64 bits is smaller than that of those:
// scores 5.2e-8 (8.3e-8), product 6.6e-8 (11e-8), at K = 128 6.4e-8 (8.8e-8) and 6.6e-8 (15e-8).
// Measured on the way, us of the two kernels: epilogue from the accumulators' layout, tiles' scores read back one at a time
// 40; three waves per SIMD for all with 170 registers spilling 41 and 65 (a kernel that uses scratch memory starts late as
// well); long rows' units of 12 tiles, in front, 30 (a second round of workgroups), of 4, behind, 23.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "bf16_parts.hpp"
#include "kernels.hpp"
#include "launch.hpp"
#include "softmax_exp.hpp"

using namespace sddmm;

namespace {

constexpr int kRows = kBlockRows;     // 32
// A power of two that operands are multiplied by before they are cut into parts where they may be small, and that results are
// divided by: parts then hold every bit of a value down to the smallest subnormal, of which they lose some from 2^-110 down.
// The product's X always: softmax weights have all sizes below 1, and one whose score lies 77 below its row's maximum is
// smaller than that.  W and H only where a unit meets such values: the unit is done once more, with both scaled.  At the other
// end of the range sums overflow earlier, which is found as all overflow is: scaled dot products from 2^48 on, the product's
// sums from 2^84, with H scaled from 2^44.  us, 16,384 tokens, K = 64, and when such units were computed in fp32, entry by
// entry: product with scores of standard deviation 1 / 8 / 12 / 40 24.2 / 23.5 / 23.5 / 23.5, and 23.7 / 316 / 457 / 457; one
// element of H (1.2e-36) softmax 30 and product 26, and 115 and 322; a whole column of H 38 and 38, and 221 and 451.
constexpr float kScale = 0x1p40f;
constexpr int kXRow = 16 + 4;         // floats per row of half a tile of X in LDS: 16 rows' 16-byte reads fall into different banks

// the product's LDS: the waves' tiles of X or their sums, then masks and columns of a unit's tiles
constexpr int spmm_sum_floats(int KT, int nw) { return 4 * KT * 1024 > nw * kRows * kXRow ? 4 * KT * 1024 : nw * kRows * kXRow; }
constexpr size_t spmm_lds_bytes(int KT, int nw) { return (size_t)spmm_sum_floats(KT, nw) * 4 + kBlockTiles * kRows * 12; }

// accumulator register v of lane (m, kh) holds the result of row result_row(v, kh), column m
__device__ __forceinline__ int result_row(int v, int kh) { return 8 * (v >> 2) + 4 * kh + (v & 3); }

template <int CTRL>
__device__ __forceinline__ float from_dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
// over the 32 lanes of this lane's half
template <bool MAX>
__device__ __forceinline__ float over_half(float v)
{
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    v = op(v, from_dpp<0xB1>(v));   // quad_perm [1,0,3,2]
    v = op(v, from_dpp<0x4E>(v));   // quad_perm [2,3,0,1]
    v = op(v, from_dpp<0x141>(v));  // row_half_mirror
    v = op(v, from_dpp<0x140>(v));  // row_mirror
    return op(v, __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (16 << 10) | 0x1f)));  // lane ^ 16
}

// a short block's last row stands in the places behind it, too: no results there
__device__ __forceinline__ bool repeated_row(const int32_t *block_rows, int r) { return r > 0 && block_rows[r] == block_rows[r - 1]; }

// KS: K / 16.  SOFTMAX: units that are whole row blocks leave the softmax of their rows, the others their scores.
// NW: waves per workgroup.
template <int KS, bool SOFTMAX, int NW>
__global__ __launch_bounds__(64 * NW, NW == 4 && KS <= 4 ? 3 : 2)
void sddmm_block_kernel(const BlockArgs a)
{
    extern __shared__ float kept[];  // dot products [tile][result register][lane]; behind them the tiles' masks, [tile][row]
    const int lane = threadIdx.x & 63, m = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t K4 = (uint32_t)(a.K >> 2), lane_bit = 1u << m, lane_lt = lane_bit - 1u;
    const vec4f *__restrict__ W4 = reinterpret_cast<const vec4f *>(a.W);
    const vec4f *__restrict__ H4 = reinterpret_cast<const vec4f *>(a.H);
    const int4 unit = a.units[blockIdx.x];
    const int *block_rows = a.rows + unit.x * kRows;
    const bool softmax = SOFTMAX && unit.w < 0;  // (uniform)

    // Element 16 s + 8 kh + e of a row is element e of step s in this lane: the same order for both operands.
    // A step's operands are requested AHEAD steps before their use, a whole tile where the registers hold that (AHEAD
    // divides KS: the slots of the steps go round).
    constexpr int AHEAD = KS == 6 ? 3 : KS == 8 ? 4 : KS;
    uint32_t lost = 0;
    vec4w pa[KS][3];
    int t = unit.y + wave;
    int col = 0, col_next = 0;
    vec4f h[AHEAD][2];
    auto request = [&](int of, int s) {
        const vec4f *hr = H4 + ((uint32_t)of * K4 + 2 * kh);
        h[s % AHEAD][0] = hr[4 * s];
        h[s % AHEAD][1] = hr[4 * s + 1];
    };
    // What the wave's tiles from t on begin with.  SCALED: both operands are multiplied by a power of two before they are cut.
    auto begin = [&]<bool SCALED>(std::bool_constant<SCALED>) {
        if (t < unit.z) {
            col = a.cols[t * kRows + m];
            col_next = a.cols[min(t + NW, unit.z - 1) * kRows + m];
        }
        const vec4f *w = W4 + ((uint32_t)block_rows[m] * K4 + 2 * kh);
        vec4f raw[KS][2];
#pragma unroll
        for (int s = 0; s < KS; ++s) { raw[s][0] = w[4 * s]; raw[s][1] = w[4 * s + 1]; }
        if (t < unit.z) {
#pragma unroll
            for (int s = 0; s < AHEAD; ++s) request(col, s);
        }
        __builtin_amdgcn_sched_barrier(0);
        constexpr float f = SCALED ? kScale : 1.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s) split8(raw[s][0] * f, raw[s][1] * f, pa[s], lost);
    };
    begin(std::false_type{});
    bool scaled = false;  // (uniform) W or H has values below 2^-110: from there on both scaled, so that parts hold them
    // A softmax needs all of a row's scores at once; otherwise the tiles are taken a few at a time, for the LDS.
    const int round = SOFTMAX ? kBlockTiles : kRoundTiles;
    for (int t0 = unit.y; t0 < unit.z; t0 += round) {
        const int t1 = min(t0 + round, unit.z), nt = t1 - t0;
        uint2 *kept_info = reinterpret_cast<uint2 *>(kept + (size_t)(SOFTMAX ? unit.z - unit.y : min(kRoundTiles, unit.z - unit.y)) * 1024);
        if (t0 > unit.y) __syncthreads();  // (the round before has been read)
        for (int i = threadIdx.x; i < nt * kRows; i += 64 * NW) kept_info[i] = a.info[t0 * kRows + i];
        const int first = t;
        auto dots = [&]<bool SCALED>(std::bool_constant<SCALED>) {
            constexpr float f = SCALED ? kScale : 1.0f;
            for (; t < t1; t += NW) {
                // (behind the wave's last tile: the unit's last one again, never used)
                const int col_after = a.cols[min(t + 2 * NW, unit.z - 1) * kRows + m];
                floatx16 dot = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    vec4w pb[3];
                    split8(h[s % AHEAD][0] * f, h[s % AHEAD][1] * f, pb, lost);
                    if (s + AHEAD < KS) request(col, s + AHEAD);
                    else request(col_next, s + AHEAD - KS);
                    __builtin_amdgcn_sched_barrier(0);
                    add_products(dot, pa[s], pb);
                    __builtin_amdgcn_sched_barrier(0);  // (more than one step's sums at a time do not fit the registers)
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) kept[(t - t0) * 1024 + v * 64 + lane] = SCALED ? dot[v] * (1.0f / kScale / kScale) : dot[v];
                col = col_next;
                col_next = col_after;
            }
        };
        if (!scaled) {
            dots(std::false_type{});
            scaled = __syncthreads_or((lost & 0xffffu) != 0) != 0;
            if (scaled) {
                t = first;
                begin(std::true_type{});
            }
        }
        if (scaled) {
            dots(std::true_type{});
            __syncthreads();
        }
        // Each wave takes a quarter of the result registers, each half of it one row per register, all tiles.
        // the dot product of tile u's column in this lane once more, in fp32: where parts cannot carry it
        auto exact = [&](int u, int row) {
            const vec4f *w = W4 + (uint32_t)block_rows[row] * K4, *h = H4 + (uint32_t)a.cols[(t0 + u) * kRows + m] * K4;
            float d = 0.f;
#pragma unroll 1
            for (uint32_t k = 0; k < K4; ++k) {
                const vec4f x = w[k], y = h[k];
                d = fmaf(x.x, y.x, d); d = fmaf(x.y, y.y, d); d = fmaf(x.z, y.z, d); d = fmaf(x.w, y.w, d);
            }
            return d;
        };
        // the rows of result register v, up to T tiles: held in registers, all reads in flight together
        auto rows_of = [&]<int T>(std::integral_constant<int, T>, int v) {
            const int row = result_row(v, kh);
            float score[T];
            int at[T];       // -1: not an entry
            float odd = 0.f;  // NaN: an infinity or a NaN among the dot products
#pragma unroll
            for (int u = 0; u < T; ++u) {
                const int of = min(u, nt - 1);
                const uint2 r = kept_info[of * kRows + row];
                score[u] = kept[of * 1024 + v * 64 + lane];
                at[u] = u < nt && (r.x & lane_bit) ? (int)(r.y + (uint32_t)__builtin_popcount(r.x & lane_lt)) : -1;
            }
#pragma unroll
            for (int u = 0; u < T; ++u) odd = fmaf(score[u], 0.f, odd);
            if (!__all(odd == 0.f)) {
#pragma unroll 1
                for (int u = 0; u < nt; ++u) {
                    float &place = kept[u * 1024 + v * 64 + lane];
                    if ((kept_info[u * kRows + row].x & lane_bit) && !(fabsf(place) < INFINITY)) place = exact(u, row);
                }
#pragma unroll
                for (int u = 0; u < T; ++u) score[u] = kept[min(u, nt - 1) * 1024 + v * 64 + lane];
            }
            if (a.val) {
                float val[T];
#pragma unroll
                for (int u = 0; u < T; ++u) val[u] = a.val[(uint32_t)max(at[u], 0)];
#pragma unroll
                for (int u = 0; u < T; ++u) score[u] = a.residual ? val[u] - score[u] : val[u] * score[u];
            }
            float inv = 1.0f;
            if (softmax) {
                float most = -INFINITY, sum = 0.f;
#pragma unroll
                for (int u = 0; u < T; ++u) {
                    score[u] = at[u] >= 0 ? score[u] : -INFINITY;
                    most = fmaxf(most, score[u]);
                }
                most = over_half<true>(most);
#pragma unroll
                for (int u = 0; u < T; ++u) {
                    score[u] = exp_nonpositive(score[u] - most);
                    sum += score[u];
                }
                inv = 1.0f / over_half<false>(sum);
            }
#pragma unroll
            for (int u = 0; u < T; ++u)
                if (at[u] >= 0) a.out[(uint32_t)at[u]] = softmax ? score[u] * inv : score[u];
        };
#pragma unroll 1
        for (int v = wave; v < 16; v += NW) {
            if (nt <= 4) rows_of(std::integral_constant<int, 4>{}, v);
            else if (nt <= 6) rows_of(std::integral_constant<int, 6>{}, v);
            else if (nt <= 8) rows_of(std::integral_constant<int, 8>{}, v);
            else if (nt <= 10) rows_of(std::integral_constant<int, 10>{}, v);
            else if (nt <= 12) rows_of(std::integral_constant<int, 12>{}, v);
            else if (!SOFTMAX || NW == 4 || nt <= 16) rows_of(std::integral_constant<int, 16>{}, v);  // (NW = 4: up to kBlockTilesFew)
            else if (nt <= 20) rows_of(std::integral_constant<int, 20>{}, v);
            else if (nt <= 24) rows_of(std::integral_constant<int, 24>{}, v);
            else rows_of(std::integral_constant<int, kBlockTiles>{}, v);
        }
        if constexpr (SOFTMAX) return;  // (all tiles in one round)
    }
}

// The softmax of the rows whose blocks are several units, in place, in pieces of up to 16,384 entries, each held in the
// registers of a workgroup.  A row of one piece is done at once; of a longer one the first pass (RECORD) leaves the
// pieces' (max, sum), the second joins them and writes.  A few workgroups, bound by their chain of loads, so a piece says where
// its entries lie (looked up in the row pointers, and with the sum kernel below asking for its row only after its sums: scores,
// softmax and product of 16,384 tokens, K = 64, 48.6 us, now 47.9; 32,359 tokens 63.4 and 62.8).
constexpr int kLongThreads = 1024, kLongEach = kLongPiece / kLongThreads;

template <bool RECORD>
__global__ __launch_bounds__(kLongThreads)
void sddmm_block_long_rows_kernel(const BlockArgs a)
{
    __shared__ float red[2][kLongThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int4 piece = a.long_pieces[blockIdx.x];  // first entry, entries, the row's first piece, its pieces
    if (!RECORD && piece.w == 1) return;
    const int len = piece.y;
    float *o = a.out + piece.x;
    float v[kLongEach];
#pragma unroll
    for (int i = 0; i < kLongEach; ++i) {
        const int p = threadIdx.x + i * kLongThreads;
        v[i] = p < len ? o[p] : -INFINITY;
    }
    float all = -INFINITY, s = 0.f;
    if (RECORD) {
#pragma unroll
        for (int i = 0; i < kLongEach; ++i) all = fmaxf(all, v[i]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) all = fmaxf(all, __shfl_xor(all, off));
        if (lane == 0) red[0][wave] = all;
        __syncthreads();
        for (int w = 0; w < kLongThreads / 64; ++w) all = fmaxf(all, red[0][w]);
#pragma unroll
        for (int i = 0; i < kLongEach; ++i) {
            const float e = v[i] == -INFINITY ? 0.f : exp_nonpositive(v[i] - all);  // (a piece's maximum may be that)
            v[i] = piece.w == 1 && all == -INFINITY ? NAN : e;                      // (a row's: no weights)
            s += e;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (lane == 0) red[1][wave] = s;
        __syncthreads();
        s = 0.f;
        for (int w = 0; w < kLongThreads / 64; ++w) s += red[1][w];
        if (piece.w > 1) {
            if (threadIdx.x == 0) a.long_records[blockIdx.x] = make_float2(all, s);
            return;
        }
    } else {
        for (int k = 0; k < piece.w; ++k) all = fmaxf(all, a.long_records[piece.z + k].x);
        for (int k = 0; k < piece.w; ++k) {
            const float2 r = a.long_records[piece.z + k];
            s += r.y == 0.f ? 0.f : r.y * exp_nonpositive(r.x - all);
        }
#pragma unroll
        for (int i = 0; i < kLongEach; ++i) v[i] = exp_nonpositive(v[i] - all);
    }
    const float inv = 1.0f / s;
#pragma unroll
    for (int i = 0; i < kLongEach; ++i) {
        const int p = threadIdx.x + i * kLongThreads;
        if (p < len) o[p] = v[i] * inv;
    }
}

// KT: K / 32 rounded up
template <int KT, int NW>
__global__ __launch_bounds__(64 * NW, KT == 2 && NW == 4 ? 3 : 2)
void sddmm_block_spmm_kernel(const BlockArgs a)
{
    extern __shared__ float lds[];  // the waves' tiles of X, afterwards their sums; behind them the unit's masks and columns
    const int lane = threadIdx.x & 63, m = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = a.K;
    const uint32_t last = (uint32_t)(a.nnz - 1);
    const int4 unit = a.units[blockIdx.x];
    const int t0 = unit.y, nt = unit.z - t0;
    float *xt = lds + wave * kRows * kXRow;
    uint2 *info = reinterpret_cast<uint2 *>(lds + spmm_sum_floats(KT, NW));
    uint32_t *row_bytes = reinterpret_cast<uint32_t *>(info + kBlockTiles * kRows);  // where the columns' rows of H begin
    for (int i = threadIdx.x; i < nt * kRows; i += 64 * NW) {
        info[i] = a.info[t0 * kRows + i];
        row_bytes[i] = (uint32_t)a.cols[t0 * kRows + i] * (uint32_t)K * 4u;
    }
    uint32_t lost = 0;
    floatx16 sum[KT];
    __syncthreads();
    // What a tile needs is requested while the one before is multiplied.
    // X comes half a tile at a time, H in portions: portion q is the elements 32 (q % KT) on of the columns' rows of step
    // q / KT, and portion q + AHEAD is requested when portion q has been multiplied.
    // (K = 33 to 64 in workgroups of four waves: two portions ahead instead of four leave 168 registers of 185, and a SIMD holds three
    // waves instead of two; 16,384 tokens, K = 64, window of 128 on either side, us of this kernel 22.0 and 18.7, scores, softmax
    // and product of 32,359 tokens, 73 on either side, 67.5 and 62.7; level below 10,000 tokens)
    constexpr int AHEAD = KT == 3 ? 3 : KT == 1 || (KT == 2 && NW == 4) ? 2 : 4;
    float x[8], h[AHEAD][8];
    const int xc = lane & 15, xr0 = lane >> 4;  // this lane's column in half a tile, its first row
    auto fetch = [&](int s, int u) {  // half a tile: columns 16 s on, rows xr0 + 4 i
        const int c = 16 * s + xc;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint2 r = info[u * kRows + xr0 + 4 * i];
            x[i] = a.x[min(r.y + (uint32_t)__builtin_popcount(r.x & ((1u << c) - 1u)), last)];
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (the addresses of all at a time do not fit the registers)
        }
    };
    auto stage = [&](int s, int u) {  // (what a row does not have becomes 0 here: the entries need not have arrived before)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int has = __builtin_amdgcn_sbfe((int)info[u * kRows + xr0 + 4 * i].x, 16 * s + xc, 1);  // 0 or -1
            xt[(xr0 + 4 * i) * kXRow + xc] = __int_as_float(__float_as_int(x[i]) & has) * kScale;
        }
    };
    // Operand element e of step s is column 16 s + 8 kh + e of the tile.
    auto request = [&](int q, int u) {
        const int s = q / KT, n = q % KT;
        const uint4 *b4 = reinterpret_cast<const uint4 *>(row_bytes + u * kRows + 16 * s + 8 * kh);
        const uint4 lo = b4[0], hi = b4[1];
        const uint32_t b[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int e = 0; e < 8; ++e)  // (uniform base + 32-bit offset: no 64-bit addresses to compute and to keep)
            h[q % AHEAD][e] = 32 * n + m < K ? *reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.H) + (b[e] + 4 * m) + 128 * n) : 0.f;
    };
    // The wave's sums over its tiles.  SCALED: H is multiplied by the power of two as well.
    auto add_tiles = [&]<bool SCALED>(std::bool_constant<SCALED>) {
#pragma unroll
        for (int n = 0; n < KT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) sum[n][v] = 0.f;
        int u = wave;
        if (u < nt) {
            request(0, u);
            fetch(0, u);
#pragma unroll
            for (int q = 1; q < AHEAD; ++q) request(q, u);
        }
        for (; u < nt; u += NW) {
            const int next = min(u + NW, nt - 1);  // (behind the wave's last tile: the unit's last one, never used)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                stage(s, u);
                __builtin_amdgcn_wave_barrier();  // (written and read by this wave alone: its LDS operations complete in order)
                vec4w pa[3];
                const vec4f *xr = reinterpret_cast<const vec4f *>(xt + m * kXRow + 8 * kh);
                split8(xr[0], xr[1], pa, lost);
                __builtin_amdgcn_wave_barrier();
                if (s == 0) fetch(1, u);
                else fetch(0, next);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < KT; ++n) {
                    vec4w pb[3];
                    const int q = s * KT + n;
                    const float *b = h[q % AHEAD];
                    constexpr float f = SCALED ? kScale : 1.0f;
                    split8(vec4f{b[0], b[1], b[2], b[3]} * f, vec4f{b[4], b[5], b[6], b[7]} * f, pb, lost);
                    if (q + AHEAD < 2 * KT) request(q + AHEAD, u);
                    else request(q + AHEAD - 2 * KT, next);
                    add_products(sum[n], pa, pb);
                    __builtin_amdgcn_sched_barrier(0);  // (more than one portion's sums at a time do not fit the registers)
                }
            }
        }
    };
    auto beyond = [&]() {
        bool bad = false;
#pragma unroll
        for (int n = 0; n < KT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) bad |= !(fabsf(sum[n][v]) < 0x1p124f);  // (the sum of all waves' must not overflow either)
        return bad;
    };
    add_tiles(std::false_type{});
    float unscale = 1.0f / kScale;
    bool redo = false;
    if (__syncthreads_or(beyond() || (lost & 0xffffu) != 0)) {  // (the tiles of X have been read, too)
        redo = true;
        if (__syncthreads_or((lost & 0xffffu) != 0)) {  // H has values below 2^-110: once more, where parts hold them
            add_tiles(std::true_type{});
            unscale = 1.0f / kScale / kScale;
            redo = __syncthreads_or(beyond()) != 0;
        }
    }
    float *record = a.part + (size_t)max(unit.w, 0) * (KT * 1024);
    auto put = [&](int n, int v, int lane_of, float y) {  // result register v of lane lane_of, elements 32 n on
        if (unit.w >= 0) {
            record[n * 1024 + v * 64 + lane_of] = y;
        } else {
            const int r = result_row(v, lane_of >> 5), k = 32 * n + (lane_of & 31);
            if (k < K && !repeated_row(a.rows + unit.x * kRows, r)) a.Y[(size_t)a.rows[unit.x * kRows + r] * K + k] = y;
        }
    };
    if (redo) {
        for (int r = wave; r < kRows; r += NW)
            for (int k = lane; k < K; k += 64) {
                float y = 0.f;
                for (int i = 0; i < nt; ++i) {
                    uint32_t p = info[i * kRows + r].y;
                    for (uint32_t mask = info[i * kRows + r].x; mask; mask &= mask - 1, ++p)
                        y = fmaf(a.x[p], *reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.H) + row_bytes[i * kRows + __builtin_ctz(mask)] + 4 * k), y);
                }
                put(k >> 5, 4 * (r >> 3) + (r & 3), 32 * ((r >> 2) & 1) + (k & 31), y);
            }
        return;
    }
    // the waves' sums, in order: room for four at a time
    if constexpr (NW == 8) {
        if (wave >= 4) {
#pragma unroll
            for (int n = 0; n < KT; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) lds[((wave - 4) * KT + n) * 1024 + v * 64 + lane] = sum[n][v];
        }
        __syncthreads();
        if (wave < 4) {
#pragma unroll
            for (int n = 0; n < KT; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) sum[n][v] += lds[(wave * KT + n) * 1024 + v * 64 + lane];
        }
    }
    if (wave < 4) {
#pragma unroll
        for (int n = 0; n < KT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) lds[(wave * KT + n) * 1024 + v * 64 + lane] = sum[n][v];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < KT; ++n)
#pragma unroll
        for (int i = 0; i < 16 / NW; ++i) {
            const int v = wave * (16 / NW) + i;
            float y = lds[n * 1024 + v * 64 + lane];
#pragma unroll
            for (int w = 1; w < 4; ++w) y += lds[(w * KT + n) * 1024 + v * 64 + lane];
            put(n, v, lane, y * unscale);
        }
}

// What the product's first kernel leaves: the sums over the units of a row block that is several, 64 results per workgroup,
// each wave a quarter of the units, in order; and the rows without nonzeros, which become 0.
__global__ __launch_bounds__(256)
void sddmm_block_sum_kernel(const BlockArgs a, int results, int sum_groups)
{
    __shared__ float quarter[4][64];
    const int K = a.K;
    if ((int)blockIdx.x < sum_groups) {
        const int parts = results / 64, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int4 block = a.sums[blockIdx.x / parts];  // row block, first record, records
        const int e = (blockIdx.x % parts) * 64 + lane;
        const float *rec = a.part + (size_t)block.y * results + e;
        const int k = 32 * (e >> 10) + (e & 31), r = result_row((e >> 6) & 15, (e >> 5) & 1);
        const int32_t *rows = a.rows + block.x * kRows;
        const int row = rows[r], row_before = rows[max(r, 1) - 1];  // (on their way beside the records)
        __builtin_amdgcn_sched_barrier(0);
        const int k1 = block.z * (wave + 1) / 4;
        float y = 0.f;
        for (int k0 = block.z * wave / 4; k0 < k1; k0 += 16) {  // (sixteen records in flight)
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = rec[(size_t)min(k0 + u, k1 - 1) * results];
#pragma unroll
            for (int u = 0; u < 16; ++u) y += k0 + u < k1 ? v[u] : 0.f;
        }
        quarter[wave][lane] = y;
        __syncthreads();
        if (wave == 0 && k < K && !(r > 0 && row == row_before))
            a.Y[(size_t)row * K + k] = (quarter[0][lane] + quarter[1][lane]) + (quarter[2][lane] + quarter[3][lane]);
        return;
    }
    const int64_t n = (int64_t)a.n_empty * K, stride = (int64_t)(gridDim.x - sum_groups) * 256;
    for (int64_t i = (int64_t)(blockIdx.x - sum_groups) * 256 + threadIdx.x; i < n; i += stride)
        a.Y[(size_t)a.empty_rows[i / K] * K + i % K] = 0.f;
}

template <bool SOFTMAX, int NW>
BlockFn block_kernel_of(int K)
{
    switch (K / 16) {
    case 2: return sddmm_block_kernel<2, SOFTMAX, NW>;
    case 3: return sddmm_block_kernel<3, SOFTMAX, NW>;
    case 4: return sddmm_block_kernel<4, SOFTMAX, NW>;
    case 5: return sddmm_block_kernel<5, SOFTMAX, NW>;
    case 6: return sddmm_block_kernel<6, SOFTMAX, NW>;
    case 7: return sddmm_block_kernel<7, SOFTMAX, NW>;
    case 8: return sddmm_block_kernel<8, SOFTMAX, NW>;
    }
    return nullptr;
}

BlockFn block_spmm_of(int K, int nwaves)
{
    switch ((K + 31) / 32) {
    case 1: return nwaves == 4 ? sddmm_block_spmm_kernel<1, 4> : sddmm_block_spmm_kernel<1, 8>;
    case 2: return nwaves == 4 ? sddmm_block_spmm_kernel<2, 4> : sddmm_block_spmm_kernel<2, 8>;
    case 3: return nwaves == 4 ? sddmm_block_spmm_kernel<3, 4> : sddmm_block_spmm_kernel<3, 8>;
    case 4: return nwaves == 4 ? sddmm_block_spmm_kernel<4, 4> : sddmm_block_spmm_kernel<4, 8>;
    }
    return nullptr;
}

}  // namespace

namespace sddmm {

bool block_supported(int K) { return K % 16 == 0 && K >= 32 && K <= 128; }

BlockFn block_kernel(int K, bool softmax, int nwaves)
{
    if (!block_supported(K) || (nwaves != 4 && nwaves != 8)) return nullptr;
    if (softmax) return nwaves == 4 ? block_kernel_of<true, 4>(K) : block_kernel_of<true, 8>(K);
    return nwaves == 4 ? block_kernel_of<false, 4>(K) : block_kernel_of<false, 8>(K);
}

hipError_t block_spmm_set_lds(int K, int nwaves)
{
    return hipFuncSetAttribute((const void *)block_spmm_of(K, nwaves), hipFuncAttributeMaxDynamicSharedMemorySize, (int)spmm_lds_bytes((K + 31) / 32, nwaves));
}

hipError_t launch_block_long_rows(const BlockArgs &a, void *stream)
{
    if (a.n_long_pieces <= 0) return hipSuccess;
    const dim3 grid((unsigned)a.n_long_pieces), block(kLongThreads);
    hipError_t e = launch(sddmm_block_long_rows_kernel<true>, grid, block, 0, (hipStream_t)stream, a);
    if (e == hipSuccess && a.long_records) e = launch(sddmm_block_long_rows_kernel<false>, grid, block, 0, (hipStream_t)stream, a);
    return e;
}

hipError_t launch_block_spmm(const BlockArgs &a, int nwaves, void *stream)
{
    const hipStream_t st = (hipStream_t)stream;
    const int KT = (a.K + 31) / 32;
    if (hipError_t e = launch(block_spmm_of(a.K, nwaves), dim3((unsigned)a.n_units), dim3((unsigned)(64 * nwaves)), spmm_lds_bytes(KT, nwaves), st, a))
        return e;
    const int results = KT * 1024, sum_groups = a.n_sums * (results / 64);
    const int zero_groups = (int)std::min<int64_t>(((int64_t)a.n_empty * a.K + 255) / 256, 4096);
    if (sum_groups + zero_groups == 0) return hipSuccess;
    return launch(sddmm_block_sum_kernel, dim3((unsigned)(sum_groups + zero_groups)), dim3(256), 0, st, a, results, sum_groups);
}

}  // namespace sddmm
