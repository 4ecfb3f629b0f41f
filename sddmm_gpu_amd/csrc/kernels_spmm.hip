// The sparse-times-dense product Y = X H on a plan's column tiles, for gfx950 (MI355X):
// X has the pattern of S and one fp32 per nonzero (in sorted order), H is n_cols x K.
//
// Like the SDDMM's tile kernel a workgroup holds a column tile of H in LDS.  A (row, tile) run
// -- the nonzeros of one row inside one tile -- belongs to one group of 8 lanes from its first
// nonzero to its last: lane l keeps its 16 elements of the row of Y in registers and adds
// x[p] times its slice of the H row of every nonzero of the run, read from LDS.  No two groups
// ever add to the same row of Y: a run ends in one partial row, written once, in the order the
// runs are walked, and a second kernel adds the partial rows of every row of S (at most one per
// column tile).  No atomics, so the result has the same bits on every call.  The 8 groups of a
// wave walk 8 runs side by side ("bundle"); the planner sorts an item's runs by length, so a
// bundle's runs are about equally long.  Rows too short for the tiles gather their H rows from
// global memory, one group of lanes per row.
//
// RAGGED: K is no multiple of the kernel's width, and K needs no alignment: tiles and partial rows have the full width, with
// the tail of H rows filled up with zeros, the last piece of a row is read from its last four floats on (see RowPiece) and
// only what is new in it goes to Y.  us per product, by the walk over the CSR pattern and so: ratings of 4.9 million nonzeros,
// K = 50 / 100 / 250 / 300 68 / 102 / 240 / 395 and 54 / 88 / 183 / 273; 15.9 million, K = 50 / 100 / 250 / 300 175 / 286 / 984 /
// 1672 and 122 / 258 / 553 / 804 (when it is chosen: ragged_product_tiles).
#include <hip/hip_runtime.h>
#include <utility>
#include "csr_walk.hpp"
#include "kernels.hpp"

using namespace sddmm;

namespace {

typedef float vec4f __attribute__((ext_vector_type(4)));

// The value that lane I of this lane's group of 8 holds, by two row broadcasts of the data-parallel primitives, the second
// for the upper half of a 16-lane row only: vector-ALU work with no trip through the LDS pipe, which the H reads keep busy
// and whose latency would sit in front of every round.
template <int I>
__device__ __forceinline__ int from_group_lane(int v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, v, 0x150 + I, 0xf, 0xf, false);   // row_newbcast:I
    return __builtin_amdgcn_update_dpp(lo, v, 0x150 + I + 8, 0xf, 0xc, false);      // row_newbcast:I+8
}
// base + what lane 0, 1, ... 7 of this lane's group holds in v: the broadcasts as operands of the additions, which the
// compiler does not find.  (The s_nop covers the two wait states between a vector write of v and its use as such an operand.)
__device__ __forceinline__ void add_of_group(int v, int base, int (&sum)[8])
{
#define SDDMM_ADD_OF(i, j)                                                       \
    "v_add_u32_dpp %" #i ", %8, %9 row_newbcast:" #i " row_mask:0xf bank_mask:0x3\n\t" \
    "v_add_u32_dpp %" #i ", %8, %9 row_newbcast:" #j " row_mask:0xf bank_mask:0xc\n\t"
    asm("s_nop 1\n\t" SDDMM_ADD_OF(0, 8) SDDMM_ADD_OF(1, 9) SDDMM_ADD_OF(2, 10) SDDMM_ADD_OF(3, 11) SDDMM_ADD_OF(4, 12) SDDMM_ADD_OF(5, 13)
        SDDMM_ADD_OF(6, 14) SDDMM_ADD_OF(7, 15)
        : "=&v"(sum[0]), "=&v"(sum[1]), "=&v"(sum[2]), "=&v"(sum[3]), "=&v"(sum[4]), "=&v"(sum[5]), "=&v"(sum[6]), "=&v"(sum[7])
        : "v"(v), "v"(base));
#undef SDDMM_ADD_OF
}

// KPL float4 per lane: a K slice of 32 * KPL elements on groups of 8 lanes
template <int KPL, int NW, bool RAGGED>
__global__ __launch_bounds__(NW * 64)
void sddmm_spmm_tile_kernel(const SpmmArgs a)
{
    extern __shared__ float4 lds_tile[];
    constexpr int G = 8, K4 = G * KPL;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = lane & 7, g = lane >> 3;
    // the two groups of a 16-lane LDS phase read the halves of a 256-byte block in opposite order
    const int rot = KPL > 1 ? (g & 1) : 0;
    using lds_f4_ptr = const __attribute__((address_space(3))) vec4f *;
    const int lds_base = (int)(uint32_t)(uintptr_t)(lds_f4_ptr)reinterpret_cast<const vec4f *>(lds_tile);
    int piece[KPL];  // float4 index inside a row of this lane's j-th piece
#pragma unroll
    for (int j = 0; j < KPL; ++j) piece[j] = (j ^ rot) * G + l;
    // (its address is the row's + lane_e + 128 j for even j, that + odd for odd j)
    const int lane_e = lds_base + (l + rot * G) * 16, odd = -2 * rot * G * 16;
    const int row_k4 = a.K >> 2;
    const float4 *__restrict__ H4 = reinterpret_cast<const float4 *>(a.H) + (a.k_off >> 2);
    float4 *__restrict__ part4 = reinterpret_cast<float4 *>(a.part);
    const int n_steps = (a.n_items - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    int cur_tile = -1;
    for (int step = 0; step < n_steps; ++step) {
        const WorkItem wi = a.items[blockIdx.x + step * gridDim.x];  // [begin, end): the item's bundles
        if (wi.end <= wi.begin) continue;
        if (wi.tile != cur_tile) {
            if (cur_tile >= 0) __syncthreads();
            cur_tile = wi.tile;
            const int tile_base = wi.tile * a.tile_x;
            const int rows = min(a.tile_x, a.n_cols - tile_base);
            const float4 *src = H4 + (size_t)tile_base * row_k4;
            const int n4 = rows * K4;
            for (int i = threadIdx.x; i < n4; i += NW * 64) {
                const int r = i / K4, q = i - r * K4;
                if constexpr (RAGGED) {
                    const RowPiece pc = row_piece(q, a.K - a.k_off);
                    const vec4u v = *reinterpret_cast<const vec4u *>(a.H + ((size_t)(tile_base + r) * a.K + a.k_off) + pc.off);
                    lds_tile[i] = make_float4(pc.first > 0 ? 0.f : v.x, pc.first > 1 ? 0.f : v.y, pc.first > 2 ? 0.f : v.z, pc.first > 3 ? 0.f : v.w);
                } else {
                    lds_tile[i] = src[(size_t)r * row_k4 + q];
                }
            }
            __syncthreads();
        }
        // A wave takes the bundles wave, wave + NW, ... of the item, round by round; a round is 8 steps: lane l of a group
        // fetches the column and the value of the group's step 8 r + l, and the group's lanes take them from each other
        // (from_group_lane).  Three rounds are in flight, whatever the bundles' ends, and the header of the bundle behind the
        // one that they come from.  The rounds' registers go round by name, four in turn: a copy of what is in flight from one
        // name to another waits for it, and with three names that were shifted every round and every bundle waited for its
        // latest loads.  Nor are steps behind a bundle's longest run done, but for one where that is odd.  us of residual and
        // product together, with those waits, steps and a select per broadcast, and so: ratings of 4.9 million nonzeros, K = 50
        // 91.7 and 84.9; 15 million, K = 32 157.7 and 136.6; 98 million, K = 128 2249 and 2079; 17 million, K = 200 874 and 830.
        // (More loads in flight while a tile is staged give nothing.)
        if (wi.begin + wave >= wi.end) continue;
        struct Header { int p0, len, off, end; };
        auto header = [&](int b) -> Header {
            const int bc = min(b, wi.end - 1);  // (beyond the item: the last bundle again, never used)
            return {a.b_p0[bc * 8 + g], a.b_len[bc * 8 + g], a.b_off[bc], a.b_off[bc + 1]};
        };
        struct Round {
            uint32_t c;  // column of step l
            float x;     // its value, or that of the group's last step
            int rem;     // the group's steps from the lane's one on
            int bundle, steps, before;  // (uniform) bundle, its steps from here on, those of the rounds before
            bool last;
        };
        int bundle = wi.begin + wave, r = 0, off, n8, longest;  // what is fetched next: round r of the bundle's n8
        int first, last, lim;  // of the lane's step in the bundle's round 0, of the group's last one; the group's steps from the former on
        auto enter = [&](const Header &h) {
            off = __builtin_amdgcn_readfirstlane(h.off);
            n8 = __builtin_amdgcn_readfirstlane(h.end) - off;
            longest = __builtin_amdgcn_readfirstlane(h.len);  // (the bundle's first run)
            first = h.p0 + l;
            last = h.p0 + (max(h.len, 1) - 1);
            lim = h.len - l;
        };
        enter(header(bundle));
        Header ahead = header(bundle + NW);
        auto fetch = [&]() -> Round {
            if (r == n8) {
                bundle += NW;
                r = 0;
                enter(ahead);
                ahead = header(bundle + NW);
            }
            const uint16_t *cols = a.cols + (size_t)(off + r) * 64;
            const Round q = {cols[lane], a.x[min(first + 8 * r, last)], lim - 8 * r, bundle, longest - 8 * r, 8 * r, r + 1 == n8};
            ++r;
            return q;
        };
        float4 acc[KPL];
#pragma unroll
        for (int j = 0; j < KPL; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        auto rd = [&](vec4f (&h)[KPL], int addr_e) {
            const int addr_o = addr_e + odd;
#pragma unroll
            for (int j = 0; j < KPL; ++j) h[j] = *(lds_f4_ptr)(uintptr_t)(uint32_t)(((j & 1) ? addr_o : addr_e) + j * 128);
        };
        auto compute = [&](const Round &q) {
            // where this lane's pieces of the H rows of the round's eight steps begin, and the values, taken from the
            // group's lanes
            int at[8];
            float xs[8];
            add_of_group((int)q.c * (K4 * 16), lane_e, at);
            const int my_x = __float_as_int(q.rem > 0 ? q.x : 0.f);
            [&]<int... I>(std::integer_sequence<int, I...>) {
                ((xs[I] = __int_as_float(from_group_lane<I>(my_x))), ...);
            }(std::make_integer_sequence<int, 8>{});
            // the H pieces of step i + 1 are requested before the arithmetic of step i
            vec4f hb[2][KPL];
            rd(hb[0], at[0]);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (i > 0 && i % 2 == 0 && i >= q.steps) break;
                if (i + 1 < 8) rd(hb[(i + 1) & 1], at[i + 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < KPL; ++j) {
                    const vec4f h = hb[i & 1][j];
                    acc[j].x = fmaf(xs[i], h.x, acc[j].x); acc[j].y = fmaf(xs[i], h.y, acc[j].y);
                    acc[j].z = fmaf(xs[i], h.z, acc[j].z); acc[j].w = fmaf(xs[i], h.w, acc[j].w);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (q.last) {
                float4 *dst = part4 + ((size_t)q.bundle * 8 + g) * K4;
#pragma unroll
                for (int j = 0; j < KPL; ++j) {
                    if (q.rem + q.before + l > 0) dst[piece[j]] = acc[j];
                    acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
        };
        Round q0 = fetch(), q1 = fetch(), q2 = fetch();
        for (;;) {
            const Round q3 = fetch();
            if (q0.bundle >= wi.end) break;
            compute(q0);
            q0 = fetch();
            if (q1.bundle >= wi.end) break;
            compute(q1);
            q1 = fetch();
            if (q2.bundle >= wi.end) break;
            compute(q2);
            q2 = fetch();
            if (q3.bundle >= wi.end) break;
            compute(q3);
        }
    }
}

// A lane's piece of a row of Y.
template <bool RAGGED>
__device__ __forceinline__ void store_piece(const SpmmArgs &a, int row, int slot, const float4 &v)
{
    if constexpr (RAGGED) {
        const RowPiece pc = row_piece(slot, a.K - a.k_off);
        float *y = a.Y + ((size_t)row * a.K + a.k_off) + pc.off;
        if (pc.first == 0) {
            *reinterpret_cast<vec4u *>(y) = vec4u{v.x, v.y, v.z, v.w};
        } else {
            if (pc.first <= 1) y[1] = v.y;
            if (pc.first <= 2) y[2] = v.z;
            if (pc.first <= 3) y[3] = v.w;
        }
    } else {
        reinterpret_cast<float4 *>(a.Y)[(size_t)row * (a.K >> 2) + (a.k_off >> 2) + slot] = v;
    }
}

// Y[row, slice] = sum of the row's partial rows: one wave per listed row, group g takes the partial
// rows g, g + 8, ... and the groups' sums are added across the wave.
template <int KPL, bool RAGGED>
__device__ __forceinline__ void spmm_sum_rows(const SpmmArgs &a, int64_t block)
{
    constexpr int G = 8, K4 = G * KPL;
    const int lane = threadIdx.x & 63, l = lane & 7, g = lane >> 3;
    const int64_t w = (block * 256 + threadIdx.x) >> 6;
    if (w >= a.n_sum_rows) return;
    const int b = a.row_part_ptr[w], e = a.row_part_ptr[w + 1];
    const float4 *__restrict__ part4 = reinterpret_cast<const float4 *>(a.part);
    float4 acc[KPL];
#pragma unroll
    for (int j = 0; j < KPL; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k = b + g; k < e; k += 8) {
        const float4 *src = part4 + (size_t)a.part_slot[k] * K4;
#pragma unroll
        for (int j = 0; j < KPL; ++j) {
            const float4 v = src[j * G + l];
            acc[j].x += v.x; acc[j].y += v.y; acc[j].z += v.z; acc[j].w += v.w;
        }
    }
#pragma unroll
    for (int off = 8; off < 64; off <<= 1) {
#pragma unroll
        for (int j = 0; j < KPL; ++j) {
            acc[j].x += __shfl_xor(acc[j].x, off); acc[j].y += __shfl_xor(acc[j].y, off);
            acc[j].z += __shfl_xor(acc[j].z, off); acc[j].w += __shfl_xor(acc[j].w, off);
        }
    }
    if (g == 0) {
        const int row = a.sum_rows[w];
#pragma unroll
        for (int j = 0; j < KPL; ++j) store_piece<RAGGED>(a, row, j * G + l, acc[j]);
    }
}

// The rows outside the tiles (short ones, and rows without entries, which become 0): one group of 8
// lanes per row, H rows gathered from global memory, four nonzeros in flight per step; the planner lists
// the rows longest first, so that the eight rows of a wave are about equally long.
template <int KPL, bool RAGGED>
__device__ __forceinline__ void spmm_gather_rows(const SpmmArgs &a, int64_t block)
{
    constexpr int G = 8;
    const int lane = threadIdx.x & 63, l = lane & 7;
    const int64_t grp = (block * 256 + threadIdx.x) >> 3;
    if (grp >= a.n_gather_rows) return;
    const int row = a.gather_rows[grp];
    const int b = a.row_ptr[row], e = a.row_ptr[row + 1];
    const int row_k4 = a.K >> 2;
    const float4 *__restrict__ H4 = reinterpret_cast<const float4 *>(a.H) + (a.k_off >> 2) + l;
    int off[RAGGED ? KPL : 1];
    if constexpr (RAGGED) {
#pragma unroll
        for (int j = 0; j < KPL; ++j) off[j] = row_piece(j * G + l, a.K - a.k_off).off;
    }
    auto h_piece = [&](int c, int j) -> float4 {
        if constexpr (RAGGED) {  // (what is not new in a piece is added up as well, and not stored)
            const vec4u v = *reinterpret_cast<const vec4u *>(a.H + ((size_t)c * a.K + a.k_off) + off[j]);
            return make_float4(v.x, v.y, v.z, v.w);
        } else {
            return H4[(size_t)c * row_k4 + j * G];
        }
    };
    float4 acc[KPL];
#pragma unroll
    for (int j = 0; j < KPL; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](int c, float xs) {
#pragma unroll
        for (int j = 0; j < KPL; ++j) {
            const float4 h = h_piece(c, j);
            acc[j].x = fmaf(xs, h.x, acc[j].x); acc[j].y = fmaf(xs, h.y, acc[j].y);
            acc[j].z = fmaf(xs, h.z, acc[j].z); acc[j].w = fmaf(xs, h.w, acc[j].w);
        }
    };
    int p = b;
    for (; p + 3 < e; p += 4) {
        int cc[4]; float xx[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) { cc[i] = a.col_ind[p + i]; xx[i] = a.x[p + i]; }
        float4 hh[4][KPL];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < KPL; ++j) hh[i][j] = h_piece(cc[i], j);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < KPL; ++j) {
                acc[j].x = fmaf(xx[i], hh[i][j].x, acc[j].x); acc[j].y = fmaf(xx[i], hh[i][j].y, acc[j].y);
                acc[j].z = fmaf(xx[i], hh[i][j].z, acc[j].z); acc[j].w = fmaf(xx[i], hh[i][j].w, acc[j].w);
            }
    }
    for (; p < e; ++p) add(a.col_ind[p], a.x[p]);
#pragma unroll
    for (int j = 0; j < KPL; ++j) store_piece<RAGGED>(a, row, j * G + l, acc[j]);
}

// Second kernel of a slice: the sums of the partial rows (a stream through memory) and the rows outside
// the tiles (gathers from L2) side by side, sum_blocks and gather_blocks workgroups of each spread evenly
// over the grid, so that the two kinds of traffic overlap.
template <int KPL, bool RAGGED>
__global__ __launch_bounds__(256)
void sddmm_spmm_rows_kernel(const SpmmArgs a, int64_t sum_blocks, int64_t gather_blocks)
{
    const int64_t i = blockIdx.x, n = sum_blocks + gather_blocks;
    const int64_t sums_before = i * sum_blocks / n;  // (of the workgroups 0 .. i - 1)
    if ((i + 1) * sum_blocks / n > sums_before) spmm_sum_rows<KPL, RAGGED>(a, sums_before);
    else spmm_gather_rows<KPL, RAGGED>(a, i - sums_before);
}

}  // namespace

namespace sddmm {

bool spmm_tile_supported(int k_slice)
{
    return k_slice == 32 || k_slice == 64 || k_slice == 128;
}

using SpmmFn = void (*)(const SpmmArgs);

int spmm_tile_set_lds(int k_slice, int nwaves, bool ragged, int lds_bytes)
{
    SpmmFn fn = nullptr;
#define SDDMM_SPMM_FN(kpl) (ragged ? (nwaves == 12 ? (SpmmFn)sddmm_spmm_tile_kernel<kpl, 12, true> : (SpmmFn)sddmm_spmm_tile_kernel<kpl, 16, true>) \
                                   : (nwaves == 12 ? (SpmmFn)sddmm_spmm_tile_kernel<kpl, 12, false> : (SpmmFn)sddmm_spmm_tile_kernel<kpl, 16, false>))
    if (k_slice == 128) fn = SDDMM_SPMM_FN(4);
    else if (k_slice == 64) fn = SDDMM_SPMM_FN(2);
    else if (k_slice == 32) fn = SDDMM_SPMM_FN(1);
    if (!fn) return 1;
    return hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) == hipSuccess ? 0 : 2;
}

// one K slice of the product: the tile kernel over the bundles, the sum of the partial rows, the gathered rows
void launch_spmm_slice(const SpmmArgs &a, int k_slice, int nwaves, int grid, int lds_bytes, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    const unsigned sum_grid = (unsigned)((a.n_sum_rows + 3) / 4);
    const unsigned rows_grid = (unsigned)((a.n_gather_rows + 31) / 32);
    const bool ragged = a.K % k_slice != 0;
#define SDDMM_SPMM_LAUNCH(kpl)                                                                                          \
    do {                                                                                                                \
        if (a.n_items > 0)                                                                                              \
            hipLaunchKernelGGL(SDDMM_SPMM_FN(kpl), dim3((unsigned)grid), dim3(nwaves == 12 ? 12 * 64 : 16 * 64), (size_t)lds_bytes, st, a); \
        if (sum_grid + rows_grid > 0)                                                                                   \
            hipLaunchKernelGGL((ragged ? sddmm_spmm_rows_kernel<kpl, true> : sddmm_spmm_rows_kernel<kpl, false>), dim3(sum_grid + rows_grid), dim3(256), 0, st, \
                               a, (int64_t)sum_grid, (int64_t)rows_grid);                                               \
    } while (0)
    if (k_slice == 128) SDDMM_SPMM_LAUNCH(4);
    else if (k_slice == 64) SDDMM_SPMM_LAUNCH(2);
    else if (k_slice == 32) SDDMM_SPMM_LAUNCH(1);
#undef SDDMM_SPMM_LAUNCH
#undef SDDMM_SPMM_FN
}

}  // namespace sddmm
