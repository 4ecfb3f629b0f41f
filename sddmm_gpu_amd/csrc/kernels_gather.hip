// Row-gather kernel of the SDDMM engine for gfx950 (MI355X): S walked in sorted order, H rows read from
// global memory.  It serves plans of the row-gather family (rows of each batch from the plan's side arrays)
// and the plan-free entry point (rows from the row pointers).
//
// A wave takes up to 8 batches of 64 consecutive nonzeros, one per lane.  In a batch a group of G lanes works
// on its own G nonzeros, all lanes of the group on one nonzero per step: each lane keeps KPL pieces of four
// floats of the W row, reads the same pieces of the nonzero's H row, and the G partial sums of the G nonzeros
// are reduced together by a halving exchange that leaves nonzero i's dot product in lane i.
//
// What bounds it is the load path (64 bytes per clock and compute unit for everything read, cached or not) and,
// where H and W are larger than the caches, the traffic across the fabric.  So: the W row is read again only in
// steps in which some group's row changes (a uniform branch on a bit mask made once per batch), and the pieces
// of step i + 1 are requested before the arithmetic of step i, across batches too; index data is requested a
// batch ahead.  K needs no alignment (see RowPiece): the pieces behind the end of a row read its last four
// floats again, with what they share with the piece before masked to zero in both factors.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <utility>
#include "kernels.hpp"
#include "csr_walk.hpp"
#include "launch.hpp"

using namespace sddmm;

namespace {

// value held by lane I of the caller's group of G lanes
template <int G, int I>
__device__ __forceinline__ int group_bcast(int v)
{
    if constexpr (G == 64) return __builtin_amdgcn_readlane(v, I);
    else if constexpr (G == 4) return __builtin_amdgcn_mov_dpp(v, I * 0x55, 0xf, 0xf, true);  // quad_perm [I, I, I, I]
    else return __builtin_amdgcn_ds_swizzle(v, (I << 5) | (0x1f & ~(G - 1)));                 // src = (lane & ~(G-1)) | I
}

// value of lane (lane ^ S)
template <int S>
__device__ __forceinline__ float xor_lane(float v)
{
    if constexpr (S == 1)
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));  // quad_perm [1,0,3,2]
    else if constexpr (S == 2)
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));  // quad_perm [2,3,0,1]
    else if constexpr (S < 32)
        return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (S << 10) | 0x1f));
    else
        return __shfl_xor(v, S, 64);
}

// Running halving reduction: acc[i] is this lane's share of nonzero i; lane i of the group ends with the sum.
template <int G, int S = G / 2>
__device__ __forceinline__ void transpose_reduce_step(float (&acc)[G], int l)
{
    if constexpr (S >= 1) {
        const bool upper = (l & S) != 0;
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const float keep = upper ? acc[j + S] : acc[j];
            const float send = upper ? acc[j] : acc[j + S];
            acc[j] = keep + xor_lane<S>(send);
        }
        transpose_reduce_step<G, S / 2>(acc, l);
    }
}

// bit 0 of every group of G lanes
template <int G> constexpr uint64_t group_bits()
{
    uint64_t m = 0;
    for (int i = 0; i < 64; i += G) m |= 1ull << i;
    return m;
}

// Pieces that lie inside every row a variant is picked for (see pick_gather_variant): they need no mask.
constexpr int whole_pieces(int G, int KPL) { return KPL == 8 ? 4 * G : (KPL - 1) * G; }

// Where a row of W or H begins for a lane that knows its number: the number itself (WIDE), or the offset of its first float,
// as long as byte offsets have 32 bits: the multiplication is then done once per nonzero, not in every lane and step,
// and the load takes the matrix's address from scalar registers.  (us with a multiplication in every step and masks on every
// piece of a ragged row, and so: uniform, 0.9 million nonzeros of 4000 rows, K = 32 / 100 / 200: 9.6 / 23.8 / 41 and 9.1 /
// 22.3 / 38; 18 thousand, K = 100 / 200: 4.9 / 7.3 and 4.6 / 6.3; where the fabric bounds it the same.)
template <bool WIDE>
__device__ __forceinline__ vec4u row_piece_of(const float *m, uint32_t at, int off, int ld)
{
    if constexpr (WIDE) return *reinterpret_cast<const vec4u *>(m + (size_t)at * ld + off);
    else return *reinterpret_cast<const vec4u *>(reinterpret_cast<const char *>(m) + ((at << 2) + ((uint32_t)off << 2)));
}

// What a launch takes of the rows: all K elements at once; K elements of rows that are ld long, the dot products so far in out; all
// of those slices one after the other, the dot products so far in the kernel (values lie where the results go then, see
// launch_gather_slices).  Every dot product is added up in the same order in the last two.
enum class Take { Rows, Slice, Slices };

// The dot product of sorted position p, complete or a slice's share of it.
template <Take TAKE>
__device__ __forceinline__ void finish(const KArgs &a, int p, float v, float dot)
{
    if constexpr (TAKE == Take::Slice) {
        if (a.add) dot += a.out[p];
        if (a.part) {
            a.out[p] = dot;
            return;
        }
    }
    a.out[p] = a.residual ? v - dot : dot * v;
}

// RAGGED: K is not 4 * G * KPL (its pieces are masked; any K > 4 * G * (KPL - 1) up to 4 * G * KPL, K >= 4).
// (Slices are forms of their own: what they take costs small calls 0.2 us of 3.8, K = 21.)
template <int G, int KPL, bool RAGGED, bool WIDE, Take TAKE = Take::Rows>
__global__ __launch_bounds__(kRowGatherBlock)
void sddmm_gather_kernel(const KArgs a)
{
    constexpr int NW = kRowGatherBlock / 64;
    __shared__ int row_tab[NW][64 * kRowGatherBatchesPerWave + 1];  // (plan-free form)
    __shared__ float so_far[TAKE == Take::Slices ? NW : 1][TAKE == Take::Slices ? 64 * kRowGatherBatchesPerWave : 1];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = lane & (G - 1);
    const int K = a.K, ld = TAKE == Take::Rows ? K : a.ld;
    const float *W = a.W, *H = a.H;  // (their first elements that are taken)
    const uint64_t le = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);

    int off[KPL];
    int first[KPL];
#pragma unroll
    for (int j = 0; j < KPL; ++j) {
        const RowPiece r = row_piece(j * G + l, K);
        off[j] = RAGGED ? r.off : 4 * (j * G + l);
        first[j] = r.first;
    }

    const int begin = blockIdx.x * a.chunk;
    const int end = min(a.nnz, begin + a.chunk);
    const int nb = (end - begin + 63) >> 6;
    const int b0 = __builtin_amdgcn_readfirstlane((int)((int64_t)nb * wave / NW));
    const int b1 = __builtin_amdgcn_readfirstlane((int)((int64_t)nb * (wave + 1) / NW));
    if (b0 >= b1) return;
    const int batch_base = begin >> 6;
    const bool planned = a.batch_seg != nullptr;
    int *tab = row_tab[wave];
    if (!planned) {
        const int p0 = begin + (b0 << 6);
        rows_of_range(a.row_ptr, a.n_rows, a.nnz, p0, (b1 - b0) << 6, tab, lane);
    }

    struct Batch {
        int row, p, col;
        float v;
    };
    // (lanes past the end repeat the last nonzero and store nothing; beyond a wave's last batch its last one again)
    auto load_batch = [&](int bi_in) -> Batch {
        const int bi = min(bi_in, b1 - 1);
        const int pos = min(begin + (bi << 6) + lane, end - 1);
        Batch b;
        if (planned) {
            const int gb = batch_base + bi;
            const int seg = a.batch_seg[gb] + __popcll(a.batch_mask[gb] & le);  // (lanes past the end: the last segment)
            b.row = a.seg_row ? a.seg_row[seg] : seg;
        } else {
            b.row = tab[pos - begin - (b0 << 6)];
        }
        b.p = a.perm ? a.perm[pos] : pos;
        b.col = a.col_ind[b.p];
        if constexpr (!WIDE) b.col = (int)((uint32_t)b.col * (uint32_t)ld);
        b.v = a.sval ? a.sval[pos] : (a.val ? a.val[b.p] : 1.0f);
        return b;
    };

    vec4u w[2][KPL], h[2][KPL];
#pragma unroll
    for (int j = 0; j < KPL; ++j) w[0][j] = w[1][j] = vec4u{0.f, 0.f, 0.f, 0.f};
    auto mask_piece = [&](vec4u &v, int j) {
        if (RAGGED && (j + 1) * G > whole_pieces(G, KPL)) {
            v.x = first[j] > 0 ? 0.f : v.x;
            v.y = first[j] > 1 ? 0.f : v.y;
            v.z = first[j] > 2 ? 0.f : v.z;
            v.w = first[j] > 3 ? 0.f : v.w;
        }
    };
    // requests the pieces of step I of a batch; changed: the lanes whose nonzero is in another row than the one before
    auto issue = [&]<int I>(std::integral_constant<int, I>, const Batch &b, uint64_t changed) {
        if (changed & (group_bits<G>() << I)) {
            const uint32_t wr = (uint32_t)group_bcast<G, I>(WIDE ? b.row : b.row * ld);
#pragma unroll
            for (int j = 0; j < KPL; ++j) w[I & 1][j] = row_piece_of<WIDE>(W, wr, off[j], ld);
        } else {
#pragma unroll
            for (int j = 0; j < KPL; ++j) w[I & 1][j] = w[(I & 1) ^ 1][j];
        }
        const uint32_t hr = (uint32_t)group_bcast<G, I>(b.col);
#pragma unroll
        for (int j = 0; j < KPL; ++j) h[I & 1][j] = row_piece_of<WIDE>(H, hr, off[j], ld);
    };
    // rows of a batch that differ from the row before: inside a group the lane before, for its first lane the
    // group's row at the end of the batch before
    auto row_changes = [&](const Batch &b, int last_row) -> uint64_t {
        int before = __shfl_up(b.row, 1);
        if (l == 0) before = last_row;
        return __ballot(b.row != before);
    };

    for (int k = 0;; k += K, W += K, H += K) {  // (once, but for Slices)
        Batch cur = load_batch(b0);
        Batch nxt = load_batch(b0 + 1);
        uint64_t changed = row_changes(cur, -1);
        issue(std::integral_constant<int, 0>{}, cur, changed);
        for (int bi = b0; bi < b1; ++bi) {
            float acc[G];
            const Batch after = load_batch(bi + 2);
            const uint64_t changed_next = row_changes(nxt, group_bcast<G, G - 1>(cur.row));
            [&]<int... I>(std::integer_sequence<int, I...>) {
                ((void)[&] {
                    if constexpr (I + 1 < G) issue(std::integral_constant<int, I + 1>{}, cur, changed);
                    __builtin_amdgcn_sched_barrier(0);
                    float s = 0.f;
#pragma unroll
                    for (int j = 0; j < KPL; ++j) {
                        vec4u hv = h[I & 1][j], wv = w[I & 1][j];
                        mask_piece(hv, j);
                        mask_piece(wv, j);
                        s = fmaf(wv.x, hv.x, s); s = fmaf(wv.y, hv.y, s);
                        s = fmaf(wv.z, hv.z, s); s = fmaf(wv.w, hv.w, s);
                    }
                    asm volatile("" : "+v"(s));  // (computed here: left alone the compiler sinks it behind the branches of the later steps)
                    acc[I] = s;
                    // (the last step's: the next batch's first, requested before the reduction)
                    if constexpr (I + 1 == G) issue(std::integral_constant<int, 0>{}, nxt, changed_next);
                    __builtin_amdgcn_sched_barrier(0);
                }(), ...);
            }(std::make_integer_sequence<int, G>{});
            transpose_reduce_step<G>(acc, l);
            float dot = acc[0];
            bool done = begin + (bi << 6) + lane < end;
            if constexpr (TAKE == Take::Slices) {
                float &sum = so_far[wave][((bi - b0) << 6) + lane];
                if (k > 0) dot += sum;
                sum = dot;
                done = done && k + K == ld;
            }
            if (done) finish<TAKE>(a, cur.p, cur.v, dot);
            cur = nxt;
            nxt = after;
            changed = changed_next;
        }
        if (TAKE != Take::Slices || k + K == ld) break;
    }
}

// The same with one batch a wave, for what the chain of loads bounds rather than the load path: the pieces of up to
// eight steps, W's and H's, are requested together instead of one step ahead, and a step's W row is read whether it is
// another one or not (a copy of the step before would have to wait for that step's).  The sums are the same, bit for bit.
// us per launch from a graph, the kernel above and this one: 18 thousand nonzeros, K = 16 / 32 / 64 / 128: 3.8 / 4.6 / 4.7 / 5.1
// and 3.0 / 3.3 / 3.6 / 4.4; R-MAT, 1.86 million, K = 32 / 100 / 256: 43 / 86 / 257 and 30 / 77 / 230.  Where it is chosen:
// gather_shape.
template <int G, int KPL, bool RAGGED, bool WIDE, Take TAKE = Take::Rows>
__global__ __launch_bounds__(kRowGatherBlock)
void sddmm_gather_once_kernel(const KArgs a)
{
    constexpr int ROUND = KPL <= 2 ? (G < 8 ? G : 8) : KPL <= 4 ? 4 : 2;  // steps whose pieces are requested together
    static_assert(G % ROUND == 0);
    __shared__ int row_tab[kRowGatherBlock / 64][64 + 1];  // (plan-free form)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = lane & (G - 1);
    const int K = a.K, ld = TAKE == Take::Rows ? K : a.ld;
    const float *W = a.W, *H = a.H;  // (their first elements that are taken)
    const int batch = blockIdx.x * (kRowGatherBlock / 64) + wave;
    const int p0 = batch << 6;
    if (p0 >= a.nnz) return;
    int off[KPL], first[KPL];
#pragma unroll
    for (int j = 0; j < KPL; ++j) {
        const RowPiece r = row_piece(j * G + l, K);
        off[j] = RAGGED ? r.off : 4 * (j * G + l);
        first[j] = r.first;
    }
    // (lanes past the end repeat the last nonzero and store nothing)
    const int pos = min(p0 + lane, a.nnz - 1);
    const int p = a.perm ? a.perm[pos] : pos;
    const int col = a.col_ind[p];
    const float v = a.sval ? a.sval[pos] : (a.val ? a.val[p] : 1.0f);
    int row;
    if (a.batch_seg) {
        const uint64_t le = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
        const int seg = a.batch_seg[batch] + __popcll(a.batch_mask[batch] & le);
        row = a.seg_row ? a.seg_row[seg] : seg;
    } else {
        int *tab = row_tab[wave];
        rows_of_range(a.row_ptr, a.n_rows, a.nnz, p0, 64, tab, lane);
        row = tab[pos - p0];
    }
    const int h_at = WIDE ? col : (int)((uint32_t)col * (uint32_t)ld), w_at = WIDE ? row : (int)((uint32_t)row * (uint32_t)ld);
    auto mask_piece = [&](vec4u &x, int j) {
        if (RAGGED && (j + 1) * G > whole_pieces(G, KPL)) {
            x.x = first[j] > 0 ? 0.f : x.x;
            x.y = first[j] > 1 ? 0.f : x.y;
            x.z = first[j] > 2 ? 0.f : x.z;
            x.w = first[j] > 3 ? 0.f : x.w;
        }
    };
    float acc[G];
    auto round = [&]<int BASE, int... I>(std::integer_sequence<int, BASE>, std::integer_sequence<int, I...>) {
        vec4u h[ROUND][KPL], w[ROUND][KPL];
        ((void)[&] {
            const uint32_t hr = (uint32_t)group_bcast<G, BASE + I>(h_at);
#pragma unroll
            for (int j = 0; j < KPL; ++j) h[I][j] = row_piece_of<WIDE>(H, hr, off[j], ld);
            const uint32_t wr = (uint32_t)group_bcast<G, BASE + I>(w_at);
#pragma unroll
            for (int j = 0; j < KPL; ++j) w[I][j] = row_piece_of<WIDE>(W, wr, off[j], ld);
        }(), ...);
        __builtin_amdgcn_sched_barrier(0);
        ((void)[&] {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < KPL; ++j) {
                vec4u hv = h[I][j], wv = w[I][j];
                mask_piece(hv, j);
                mask_piece(wv, j);
                s = fmaf(wv.x, hv.x, s); s = fmaf(wv.y, hv.y, s);
                s = fmaf(wv.z, hv.z, s); s = fmaf(wv.w, hv.w, s);
            }
            acc[BASE + I] = s;
        }(), ...);
    };
    float dot = 0.f;
    for (int k = 0;; k += K, W += K, H += K) {  // (once, but for Slices)
        [&]<int... R>(std::integer_sequence<int, R...>) {
            (round(std::integer_sequence<int, R * ROUND>{}, std::make_integer_sequence<int, ROUND>{}), ...);
        }(std::make_integer_sequence<int, G / ROUND>{});
        transpose_reduce_step<G>(acc, l);
        dot = TAKE == Take::Slices && k > 0 ? acc[0] + dot : acc[0];
        if (TAKE != Take::Slices || k + K == ld) break;
    }
    if (p0 + lane < a.nnz) finish<TAKE>(a, p, v, dot);
}

// Any K >= 1 (used below 4 and beyond 2048): 8 lanes per nonzero striding over the row one float at a time,
// W re-read through the cache.  The slow, always-correct path.
__global__ __launch_bounds__(kRowGatherBlock)
void sddmm_generic_kernel(const KArgs a)
{
    constexpr int G = 8;
    constexpr int NW = kRowGatherBlock / 64;
    __shared__ int row_tab[NW][64 * kRowGatherBatchesPerWave + 1];  // (plan-free form)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = lane & (G - 1);
    const int begin = blockIdx.x * a.chunk;
    const int end = min(a.nnz, begin + a.chunk);
    const int batch_base = begin >> 6;
    const int nb = (end - begin + 63) >> 6;
    const int b0 = __builtin_amdgcn_readfirstlane((int)((int64_t)nb * wave / NW));
    const int b1 = __builtin_amdgcn_readfirstlane((int)((int64_t)nb * (wave + 1) / NW));
    if (b0 >= b1) return;
    const bool planned = a.batch_seg != nullptr;
    int *tab = row_tab[wave];
    if (!planned) {
        const int p0 = begin + (b0 << 6);
        rows_of_range(a.row_ptr, a.n_rows, a.nnz, p0, (b1 - b0) << 6, tab, lane);
    }
    for (int bi = b0; bi < b1; ++bi) {
        const int pos = begin + (bi << 6) + lane;
        const bool valid = pos < end;
        const int gb = batch_base + bi;
        const uint64_t le = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
        int row = -1, col = 0, p = 0;
        float v = 0.f;
        if (valid) {
            if (planned) {
                const int seg = a.batch_seg[gb] + __popcll(a.batch_mask[gb] & le);
                row = a.seg_row ? a.seg_row[seg] : seg;
            } else {
                row = tab[pos - begin - (b0 << 6)];
            }
            p = a.perm ? a.perm[pos] : pos;
            col = a.col_ind[p];
            v = a.val ? a.val[p] : 1.0f;
        }
        float acc[G];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const int r_i = __shfl(row, i, G);
            const int c_i = __shfl(col, i, G);
            float s = 0.f;
            if (r_i >= 0) {
                const float *wr = a.W + (size_t)r_i * a.K;
                const float *hr = a.H + (size_t)c_i * a.K;
                for (int t = l; t < a.K; t += G) s = fmaf(wr[t], hr[t], s);
            }
            acc[i] = s;
        }
        transpose_reduce_step<G>(acc, l);
        if (valid) a.out[p] = a.residual ? v - acc[0] : acc[0] * v;
    }
}

}  // namespace

namespace sddmm {

// The smallest number of lanes whose pieces cover a row, at least 8 (128 contiguous bytes per gathered row) from
// K = 17 on; K < 4 and K > 2048 are left to the generic kernel (G == 0).
static Variant pick_gather_variant(int K)
{
    const int K4 = (K + 3) / 4;
    const int cand[][2] = {{4, 1}, {8, 1}, {8, 2}, {8, 3}, {8, 4}, {16, 3}, {16, 4}, {32, 3}, {32, 4}, {64, 3}, {64, 4}, {64, 8}};
    if (K < 4) return {0, 0, false};
    for (auto &c : cand)
        if (c[0] * c[1] >= K4) return {c[0], c[1], c[0] * c[1] * 4 == K};
    return {0, 0, false};
}

// One batch a wave (once), or several?  Reading every step's W row costs load path, the more the longer the rows: a row's
// nonzeros are next to each other, and the kernel with several batches reads it once.  What it saves is waiting.
// profiles/row_gather_batches.txt has both at up to 17 ranks on 40 patterns; us, several batches a wave and one:
//   rows of up to 16 nonzeros: R-MAT, 0.44 million, K = 32 / 96 / 128 18 / 28 / 38 and 15 / 25 / 32, 2.1 million 48 / 95 /
//       163 and 37 / 75 / 130.  Of up to 32 where nonzeros times pieces are many: 0.38 million of 24 a row, K = 96 / 128 /
//       256 18 / 24 / 56 and 16 / 22 / 49, 3.9 million of 30, K = 32 / 96 72 / 218 and 69 / 199; but 0.24 million of 30, K =
//       100 / 128 / 256 11.3 / 12.0 / 28.0 and 12.7 / 13.0 / 25.8, 0.9 million, K = 32 13.2 and 14.3, and up to K = 16
//       R-MAT, 28 million of 27, 344 and 381.
//   K = 33 to 64: one batch where sixteen lanes take a piece each (see below); with eight lanes and two pieces one batch was
//       the slower form (R-MAT, 1.4 / 3.4 / 28 million, K = 40 35 / 80 / 648 and 40 / 89 / 835).
//   longer rows: only up to K = 32 and 2^18 nonzeros (0.19 million of 323 a row, K = 16 / 32 / 64 4.5 / 4.7 / 5.5 and 3.8 /
//       4.5 / 5.8; 0.8 million, K = 32 8.9 and 11.0).
// Batches a wave: up to 8, which is as many as share a search for the rows, but fewer where that would leave less than 4096
// waves (16 per compute unit): 0.9 million nonzeros, K = 32 / 64 / 128 with 2048 waves 27 / 30 / 49, with 4096 19 / 23 / 44; from
// 1.5 million on all take 8 (two million of 20,000 rows, K = 64: 35, and 38 with 7).
//
// With one batch a wave, from 2^18 nonzeros on, a row of up to 64 floats, or of 97 to 127, is read by as many lanes as it has
// pieces, in one request a line (rows of such lengths begin anywhere in a line: eight lanes' 128 bytes lie in two lines each,
// and the next piece's in the second of them again).  us, 8 lanes and 16 or 32: R-MAT, 0.55 million, K = 45 / 50 / 60 / 64 /
// 100 / 120 20.8 / 20.4 / 21.5 / 17.5 / 26.7 / 28.4 and 16.7 / 16.6 / 17.2 / 15.9 / 25.7 / 26.7; 1.8 million 45 / 46 / 50 / 49 /
// 76 / 81 and 43 / 43 / 46 / 42 / 71 / 78; 8.4 million 211 / 225 / 254 / 250 / 412 / 454 and 202 / 210 / 234 / 237 / 393 / 442.  Not
// where a third of the lanes would idle in large matrices (K = 36, 1.8 / 8.4 million: 41 / 176 and 41 / 180), nor at K = 65 to
// 96 (1.8 million, K = 72 / 90 57 / 65 and 66 / 69) and beyond 128 (K = 150 / 200 104 / 137 and 113 / 135), nor below (0.17
// million, K = 50 / 100: 6.7 / 10.1 and 6.8 / 10.4), nor with several batches (R-MAT 2^15, 1.2 million, K = 100: 41 and 46).
//
// The form decides the order a dot product is added up in, and a plan and the call without one give the same bits: it goes by
// n_rows, empty rows among them, which is what both know; listed_rows, the rows a plan has listed, decides the rest.
GatherShape gather_shape(int64_t nnz, int64_t n_rows, int64_t listed_rows, int K)
{
    Variant v = pick_gather_variant(K);
    const int pieces = v.G * v.KPL, used = (K + 3) / 4;
    auto short_rows = [&](int64_t rows) { return nnz <= (pieces > 4 && nnz * pieces >= 8000000 ? 32 : 16) * rows; };
    const bool line_wise = nnz >= 1 << 18 && short_rows(n_rows) && ((pieces == 16 && (used >= 10 || nnz < 1 << 20)) || (pieces == 32 && !v.exact));
    const bool once = v.G != 0 && (line_wise || nnz <= 1 << 16 || (short_rows(listed_rows) ? pieces != 16 : pieces <= 8 && nnz <= 1 << 18));
    if (line_wise) v = {pieces, 1, v.exact};
    const int64_t waves_wanted = 4096;
    const int per_wave = once ? 1 : nnz >= 1500000 ? kRowGatherBatchesPerWave
                                                   : (int)std::clamp<int64_t>(nnz / (64 * waves_wanted), 1, kRowGatherBatchesPerWave);
    return {v, 64 * per_wave * (kRowGatherBlock / 64), once};
}

KernelFn gather_kernel(const Variant &v, bool once, bool wide)
{
#define SDDMM_FORM(g, kpl, ragged)                                                                                        \
    (once ? (wide ? (KernelFn)sddmm_gather_once_kernel<g, kpl, ragged, true> : (KernelFn)sddmm_gather_once_kernel<g, kpl, ragged, false>) \
          : (wide ? (KernelFn)sddmm_gather_kernel<g, kpl, ragged, true> : (KernelFn)sddmm_gather_kernel<g, kpl, ragged, false>))
    // (read line by line: one batch a wave only, and 32 lanes for ragged ranks only)
#define SDDMM_LINE_WISE(g, ragged) (wide ? (KernelFn)sddmm_gather_once_kernel<g, 1, ragged, true> : (KernelFn)sddmm_gather_once_kernel<g, 1, ragged, false>)
    if (v.KPL == 1 && v.G == 16) return !once ? nullptr : v.exact ? SDDMM_LINE_WISE(16, false) : SDDMM_LINE_WISE(16, true);
    if (v.KPL == 1 && v.G == 32) return !once || v.exact ? nullptr : SDDMM_LINE_WISE(32, true);
#undef SDDMM_LINE_WISE
#define SDDMM_CASE(g, kpl) \
    if (v.G == g && v.KPL == kpl) return v.exact ? SDDMM_FORM(g, kpl, false) : SDDMM_FORM(g, kpl, true);
    SDDMM_CASE(4, 1) SDDMM_CASE(8, 1) SDDMM_CASE(8, 2) SDDMM_CASE(8, 3) SDDMM_CASE(8, 4) SDDMM_CASE(16, 3) SDDMM_CASE(16, 4)
    SDDMM_CASE(32, 3) SDDMM_CASE(32, 4) SDDMM_CASE(64, 3) SDDMM_CASE(64, 4) SDDMM_CASE(64, 8)
#undef SDDMM_CASE
#undef SDDMM_FORM
    return nullptr;
}

// Elements of a row that one launch takes: K, or 64 in turn where the rows of H do not fit a die's 4 MB of L2 and slices of them
// are found there more often.  The dot products so far wait in out, and columns and rows are read once more for every slice,
// which it takes long rows and enough nonzeros to pay.  us at K = 256 / 512, whole rows and slices: R-MAT 2^17, 2.6 / 6.1 million
// nonzeros, K = 256 320 / 801 and 259 / 616, 1.5 million, K = 512 459 and 369; 2^18, 6.5 million, K = 256 886 and 681, 4.1 million, K =
// 512 1236 and 931; uniform, 3.1 million of 57,000 columns 430 / 812 and 384 / 735; word counts, 3 million of 40,000 240 / 556 and
// 193 / 380; band of 3 million 429 / 814 and 420 / 808; K = 448, R-MAT 2^17, 5.7 million 1072 and 825.  Not
//   below (R-MAT 2^15, 1.4 million, K = 256 103 and 121; 2^18, 1.1 million, K = 512 359 and 377; 1.6 million, K = 448 343 and 367),
//   where few columns take most nonzeros and their rows fit (R-MAT 2^14, 3.0 million, K = 256 162 and 191; ratings of 6.2 million,
//       5600 columns 284 and 300; uniform over 17,000 columns would gain: 3.2 million, K = 256 368 and 219),
//   where most columns are used once (R-MAT 2^20, 1.6 million, K = 512 647 and 687; 3.3 million, K = 448 808 and 820),
//   beyond K = 512, where the sums of slices have the larger error against 64 bits (R-MAT 2^17, K = 576 / 1024 9.2e-8 / 10.3e-8 whole,
//       9.3e-8 / 10.6e-8 in slices, but K = 256 / 512 9.5e-8 / 9.9e-8 and 8.3e-8 / 9.2e-8); they would gain as at 512 (5.8 million, K = 640 /
//       1024 1693 / 3498 and 1262 / 2409),
//   at other ranks: at K = 192, 320 and 384 the lanes hold three pieces of whole rows instead of four, at 448 nearly four, so that
//       slices gain less and lose more (K = 192 / 320 / 384, R-MAT 2^17, 2.6 million 167 / 319 / 405 and 178 / 310 / 398, band of 3 million 299 /
//       494 / 598 and 327 / 498 / 656; large ones would gain, 5.8 million 386 / 740 / 951 and 330 / 609 / 751); K = 128, R-MAT 2^15, 1.0
//       million 40 and 48, band 182 and 195, R-MAT 2^17, 5.8 million 283 and 232; ranks that 64 does not divide have a last slice across lines.
// Slices of 128 are faster on half of these, but at K = 512 their error is larger (9.9e-8 whole, 10.0e-8; of 64 9.4e-8; K = 256 9.5e-8,
// 9.5e-8 and 8.6e-8).
int gather_slice(int64_t nnz, int64_t n_cols, int K)
{
    const int64_t least = K == 256 ? 2500000 : K == 512 ? 1400000 : K == 448 ? 3000000 : INT64_MAX;
    return nnz >= std::max(least, 4 * n_cols) && n_cols >= (K == 256 ? 24000 : 11000) ? 64 : K;
}

// Do values lie where the results go?  The first slice's dot products would overwrite them.
static bool values_in_results(const KArgs &a)
{
    const uintptr_t v = (uintptr_t)(a.sval ? a.sval : a.val), o = (uintptr_t)a.out, bytes = (uintptr_t)a.nnz * 4;
    return v && v < o + bytes && o < v + bytes;
}

int gather_slice_launches(const KArgs &a, int slice) { return values_in_results(a) ? 1 : a.K / slice; }

// The kernel for slices of 64 elements.  gather_shape gives sixteen lanes of one piece with one batch a wave there, or eight of two with
// several (slices begin far above the sizes where eight have one).
template <Take TAKE>
static KernelFn gather_slice_kernel(const GatherShape &s, bool wide)
{
    if (s.v.G == 16 && s.v.KPL == 1 && s.once) return wide ? (KernelFn)sddmm_gather_once_kernel<16, 1, false, true, TAKE> : (KernelFn)sddmm_gather_once_kernel<16, 1, false, false, TAKE>;
    if (s.v.G == 8 && s.v.KPL == 2 && !s.once) return wide ? (KernelFn)sddmm_gather_kernel<8, 2, false, true, TAKE> : (KernelFn)sddmm_gather_kernel<8, 2, false, false, TAKE>;
    return nullptr;
}

// Values where the results go: one launch that takes the slices in turn keeps the sums so far in registers or LDS, so the results have
// the same bits; its waves are at about the same slice, which brings part of what separate launches gain.  us, whole rows, slices in a
// launch each and in one: R-MAT 2^17, 5.8 million, K = 256 / 512 767 / 1785, 600 / 1237 and 680 / 1537; ratings of 7.8 million, K = 256 / 448
// 630 / 1337, 450 / 871 and 542 / 1108; band of 3 million, K = 448 717, 714 and 717.
hipError_t launch_gather_slices(KArgs a, int64_t listed_rows, int64_t n_rows, bool wide, int slice, void *stream)
{
    const GatherShape s = gather_shape(a.nnz, n_rows, listed_rows, slice);
    const int launches = gather_slice_launches(a, slice);
    const KernelFn fn = launches == 1 ? gather_slice_kernel<Take::Slices>(s, wide) : gather_slice_kernel<Take::Slice>(s, wide);
    a.ld = a.K;
    a.K = slice;  // (divides it)
    a.chunk = s.chunk;
    const dim3 grid((unsigned)((a.nnz + (int64_t)a.chunk - 1) / a.chunk));
    for (int i = 0; i < launches; ++i, a.W += slice, a.H += slice) {
        a.add = i > 0; a.part = i + 1 < launches;
        if (hipError_t e = launch(fn, grid, dim3(kRowGatherBlock), 0, (hipStream_t)stream, a)) return e;
    }
    return hipSuccess;
}

KernelFn generic_kernel() { return (KernelFn)sddmm_generic_kernel; }

}  // namespace sddmm
