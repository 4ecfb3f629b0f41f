// Sparse-times-dense product Y = X H over a plain CSR pattern in device memory, for gfx950 (MI355X):
// Y[r, :] = sum over row r's entries p of x[p] * H[col_p, :].
//
// A wave takes n = S * 64 / G consecutive nonzeros, G lanes spanning a row of H (a slice of it beyond 256 floats)
// in pieces of four floats, and each group of G lanes S consecutive nonzeros of its own, so that the work is the
// same for every wave whatever the rows' lengths.  Columns, values and rows of the wave's nonzeros are put into
// LDS once, from where a group's lanes read them by broadcast; a group adds in registers while the row lasts and
// writes it when it changes.  The parts of a row cut between groups are added across the wave, those of a row cut
// between waves through LDS; a row cut between workgroups is completed with fp32 atomic adds (the only place where
// the order of additions can vary from run to run; with an add per group and cut row the atomics took half the
// time).  The rows that need it -- those, and empty ones -- are zeroed by a kernel before this one.
// Behind a plan (sddmm_plan_spmm) there is memory for a record per workgroup instead: the parts of rows cut between
// workgroups go there, and a kernel after this one adds them up in order -- no atomics, the same bits on every call.
//
// What bounds it is the load path (64 bytes per clock and compute unit) and, for an H larger than the caches, the
// fabric; what bounded the form before (a wave per 256 nonzeros, row by row: three dependent loads for every row)
// was latency: 429 us at 1.8 M nonzeros and K = 100, 129 us at 18 thousand and K = 16;
// now 81 and 8 us.  Where H stays in the caches the vector unit came next to the load path: 64-bit addresses from columns,
// a comparison of rows and two reads of LDS for each nonzero.  So an entry holds where its row of H begins, as a 32-bit offset
// while H has them, and a mark where a row of S begins: one read, ahead of use, and four nonzeros of every group at a time
// without a look at their rows where no mark is among them.  us, before and so: ratings of 5 million nonzeros in 5600
// columns, K = 16 / 50 / 128 / 200 / 256: 45 / 73 / 107 / 243 / 266 and 37 / 69 / 103 / 186 / 227 (25 TB/s of H rows at K =
// 128); uniform, 4 million, K = 32 40 and 35; R-MAT, 1.86 million, K = 100 83 and 81.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "internal.hpp"
#include "csr_walk.hpp"
#include "launch.hpp"

using namespace sddmm;

namespace {

constexpr int kSpmmMost = 512;  // nonzeros of a wave at most
constexpr int kSpmmUnroll = 4;  // H pieces requested together
constexpr int kMostSlices = 65535;  // (a grid's second dimension)
constexpr uint32_t kRowChange = 0x80000000u;

// Zeroes the rows of Y that the product adds to or leaves out: empty rows, and rows cut between workgroups (of 2^shift nonzeros).
// A wave looks at 64 rows, or fewer as in the kernel below: a small matrix of long rows of H has 16 to 64 nonzeros
// to a workgroup, so nearly all of its rows are cut.  us with 64 rows a wave and so: 1024 rows, K = 256 6.0 and 2.3;
// 4096, K = 384 10.0 and 3.3; 32,768, K = 192 7.2 and 5.6; with the product, 18 thousand nonzeros of 4096 rows, R-MAT, K = 16 / 32 / 64 /
// 100 7.0 / 7.2 / 8.5 / 9.6 and 6.8 / 6.9 / 7.8 / 8.2.  (Where few rows are cut there is nothing to gain: uniform, 0.2 million of 20,000
// rows, K = 16 / 32 / 64 7.9 / 8.1 / 10.2 and 8.0 / 8.3 / 10.4.)
__global__ __launch_bounds__(256)
void sddmm_spmm_zero_rows_kernel(const int32_t *__restrict__ row_ptr, float *Y, int64_t n_rows, int K, int shift, int rows_per_wave)
{
    __shared__ int list[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r = lane < rows_per_wave ? ((int64_t)blockIdx.x * 4 + wave) * rows_per_wave + lane : n_rows;
    bool zero = false;
    if (r < n_rows) {
        const int s = row_ptr[r], e = row_ptr[r + 1];
        zero = s >= e || (s >> shift) != ((e - 1) >> shift);
    }
    const uint64_t todo = __ballot(zero);
    if (zero) list[wave][__builtin_popcountll(todo & (((uint64_t)1 << lane) - 1))] = (int)r;
    __builtin_amdgcn_wave_barrier();
    const int pieces = (K + 3) >> 2, n = __builtin_popcountll(todo) * pieces;
    for (int t = lane; t < n; t += 64) {
        const int i = t / pieces, q = t - i * pieces;
        *reinterpret_cast<vec4u *>(Y + (size_t)list[wave][i] * K + row_piece(q, K).off) = vec4u{0.f, 0.f, 0.f, 0.f};
    }
}

// The rows that the product with records leaves: empty rows become 0, rows cut between workgroups (of 2^shift
// nonzeros) the sum of their records, workgroup by workgroup.  A wave looks at 64 rows, at fewer where that would leave
// less than 1024 waves, though not at fewer than fill its lanes with pieces: where rows are longer than a workgroup's share
// all of them are cut, and a few waves taking 64 each, piece after piece, are slower than the product itself.  us for both
// kernels with 64 rows a wave and with this: 2220 rows, K = 128 49 and 28, 1800 rows, K = 32 23 and 18.
__global__ __launch_bounds__(256)
void sddmm_spmm_cut_rows_kernel(const int32_t *__restrict__ row_ptr, const float *__restrict__ part, float *Y, int64_t n_rows, int K, int shift,
                                int rows_per_wave)
{
    __shared__ int list[4][64];
    __shared__ int2 range[4][64];  // first and last workgroup; (0, -1): an empty row
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r = lane < rows_per_wave ? ((int64_t)blockIdx.x * 4 + wave) * rows_per_wave + lane : n_rows;
    int s = 0, e = 1;
    if (r < n_rows) { s = row_ptr[r]; e = row_ptr[r + 1]; }
    const int w0 = s >> shift, w1 = (e - 1) >> shift;
    const bool mine = r < n_rows && (s >= e || w0 != w1);
    const uint64_t todo = __ballot(mine);
    if (mine) {
        const int i = __builtin_popcountll(todo & (((uint64_t)1 << lane) - 1));
        list[wave][i] = (int)r;
        range[wave][i] = s >= e ? make_int2(0, -1) : make_int2(w0, w1);
    }
    __builtin_amdgcn_wave_barrier();
    const int pieces = (K + 3) >> 2, n = __builtin_popcountll(todo) * pieces;
    for (int t = lane; t < n; t += 64) {
        const int i = t / pieces, q = t - i * pieces;
        const RowPiece pc = row_piece(q, K);
        const int2 w = range[wave][i];
        vec4u sum = {0.f, 0.f, 0.f, 0.f};
        // (eight records in flight: a row as long as the matrix is wide has a record per workgroup, and one at a
        // time they are the whole kernel's time: window, 60,000 tokens, K = 128: 48 us next to 449)
        for (int k0 = w.x; k0 <= w.y; k0 += 8) {
            vec4u v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = min(k0 + u, w.y);
                v[u] = *reinterpret_cast<const vec4u *>(part + (2 * (size_t)k + (k < w.y ? 1 : 0)) * K + pc.off);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (k0 + u <= w.y) sum += v[u];
        }
        // (pieces at the end of a row may overlap: they hold the same sums)
        *reinterpret_cast<vec4u *>(Y + (size_t)list[wave][i] * K + pc.off) = sum;
    }
}

// RECORDS: part[(2 wg + 0) K ..] takes the part of a row that ends in workgroup wg and began before it, part[(2 wg + 1) K ..]
// that of a row that goes on behind it.
// WIDE: H is too large for 32-bit byte offsets.
template <int G, bool RECORDS, bool WIDE>
__global__ __launch_bounds__(256)
void sddmm_spmm_csr_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_ind, const float *__restrict__ x,
                           const float *__restrict__ H, float *Y, float *part, int n_rows, int nnz, int K, int S, int slice_pieces)
{
    constexpr int NG = 64 / G, U = kSpmmUnroll, NW = 4;
    __shared__ int row_tab[NW][kSpmmMost + 1];
    __shared__ uint2 entry_tab[NW][kSpmmMost];  // column (WIDE) or where its row of H begins, kRowChange set where a row does; value
    __shared__ vec4u head_sum[NW][G], tail_sum[NW][G];
    __shared__ int head_row[NW], tail_row[NW];  // -1: none
    __shared__ bool tail_started[NW];
    const int lane = threadIdx.x & 63, l = lane & (G - 1), g = lane / G;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = S * NG;
    const int slot = blockIdx.y * slice_pieces + l;
    const RowPiece pc = row_piece(slot, K);
    const int first = l < slice_pieces ? pc.first : 4;  // (4: nothing of this lane's piece is written)
    auto put = [&](float *y, const vec4u &v) {
        if (first == 0) {
            *reinterpret_cast<vec4u *>(y) = v;
        } else {
            if (first <= 1) y[1] = v.y;
            if (first <= 2) y[2] = v.z;
            if (first <= 3) y[3] = v.w;
        }
    };
    auto store = [&](int row, const vec4u &v) {
        if (row < n_rows) put(Y + (size_t)row * K + pc.off, v);  // (n_rows: past the last nonzero)
    };
    auto add = [&](int row, const vec4u &v, int which) {
        if (row >= n_rows) return;
        if constexpr (RECORDS) {
            put(part + (2 * (size_t)blockIdx.x + which) * K + pc.off, v);
            return;
        }
        float *y = Y + (size_t)row * K + pc.off;
        if (first <= 0) unsafeAtomicAdd(y + 0, v.x);
        if (first <= 1) unsafeAtomicAdd(y + 1, v.y);
        if (first <= 2) unsafeAtomicAdd(y + 2, v.z);
        if (first <= 3) unsafeAtomicAdd(y + 3, v.w);
    };
    const vec4u zero = {0.f, 0.f, 0.f, 0.f};

    const int64_t p0l = ((int64_t)blockIdx.x * NW + wave) * n;
    if (lane == 0) { head_row[wave] = -1; tail_row[wave] = -1; tail_started[wave] = true; }
    if (p0l < nnz) {
        const int p0 = (int)p0l;
        int *rows = row_tab[wave];
        uint2 *entries = entry_tab[wave];
        uint32_t col[kSpmmMost / 64];
        float val[kSpmmMost / 64];
#pragma unroll
        for (int t = 0; t < kSpmmMost / 64; ++t)
            if (64 * t < n) {
                const int p = p0 + min(64 * t + lane, nnz - 1 - p0);
                col[t] = (uint32_t)col_ind[p];
                val[t] = 64 * t + lane < nnz - p0 ? x[p] : 0.f;
            }
        const int r0 = rows_of_range(row_ptr, n_rows, nnz, p0, n, rows, lane);

#pragma unroll
        for (int t = 0; t < kSpmmMost / 64; ++t)
            if (64 * t < n) {
                const int i = 64 * t + lane;
                const bool changes = (i & (S - 1)) && rows[i] != rows[i - 1];
                if (i < n) entries[i] = make_uint2((WIDE ? col[t] : col[t] * (uint32_t)K) | (changes ? kRowChange : 0u), __float_as_uint(val[t]));
            }
        __builtin_amdgcn_wave_barrier();  // (LDS operations of one wave complete in order)
        const int gb = g * S;
        const int row_first = rows[gb], row_last = rows[gb + S - 1];
        // does the group's first row begin with the group, its last one end with it
        const bool began = gb > 0 ? rows[gb - 1] != row_first : row_ptr[r0] == p0;
        const bool ended = rows[gb + S] != row_last;
        const char *Hb = reinterpret_cast<const char *>(H);
        const uint32_t piece_at = (uint32_t)pc.off * 4u;
        auto read = [&](uint2 (&e)[U], int i0) {
#pragma unroll
            for (int u = 0; u < U; ++u) e[u] = entries[gb + min(i0, S - U) + u];
        };
        auto request = [&](vec4u (&h)[U], const uint2 (&e)[U]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if constexpr (WIDE) h[u] = *reinterpret_cast<const vec4u *>(H + (size_t)(e[u].x & ~kRowChange) * K + pc.off);
                else h[u] = *reinterpret_cast<const vec4u *>(Hb + ((e[u].x << 2) + piece_at));  // (the mark is shifted out)
            }
        };
        vec4u acc = zero, head = zero;  // head: the part of a row that began before the group
        int cur = row_first;
        auto add_entry = [&](const vec4u &h, const uint2 &e) {
            const float xs = __uint_as_float(e.y);
            acc.x = fmaf(xs, h.x, acc.x); acc.y = fmaf(xs, h.y, acc.y);
            acc.z = fmaf(xs, h.z, acc.z); acc.w = fmaf(xs, h.w, acc.w);
        };
        // h, e: the pieces and entries from i0 on; hn, en: the entries after them, whose pieces are requested here; e then
        // takes the entries after those
        auto step = [&](vec4u (&h)[U], uint2 (&e)[U], vec4u (&hn)[U], uint2 (&en)[U], int i0) {
            if (i0 + U < S) request(hn, en);
            uint2 now[U];
            uint32_t marks = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                now[u] = e[u];
                marks |= e[u].x;
            }
            read(e, i0 + 2 * U);
            __builtin_amdgcn_sched_barrier(0);
            if (__ballot((int)marks < 0) == 0) {  // (in most steps no group's row changes)
#pragma unroll
                for (int u = 0; u < U; ++u) add_entry(h[u], now[u]);
                return;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (now[u].x & kRowChange) {
                    if (cur == row_first && !began) head = acc;
                    else store(cur, acc);
                    acc = zero;
                    cur = rows[gb + i0 + u];
                }
                add_entry(h[u], now[u]);
            }
        };
        vec4u h0[U], h1[U];
        uint2 e0[U], e1[U];
        read(e0, 0);
        read(e1, U);
        request(h0, e0);
        for (int i0 = 0; i0 < S; i0 += 2 * U) {
            step(h0, e0, h1, e1, i0);
            if (i0 + U < S) step(h1, e1, h0, e0, i0 + U);
        }
        // The rows cut between the groups: acc is the part of the group's last row; `started` says whether that
        // row's beginning is in it.  A running sum over the groups carries the part on while it stays open.
        bool has_head = !began && row_first != row_last, started = began || row_first != row_last;
        if (ended) {
            if (started) store(row_last, acc);
            else { head = acc; has_head = true; }
            acc = zero;
            started = true;
        }
#pragma unroll
        for (int d = G; d < 64; d *= 2) {
            vec4u up;
            up.x = __shfl_up(acc.x, d); up.y = __shfl_up(acc.y, d); up.z = __shfl_up(acc.z, d); up.w = __shfl_up(acc.w, d);
            const bool started_up = __shfl_up((int)started, d) != 0;
            if (lane >= d && !started) { acc += up; started = started_up; }
        }
        vec4u before = zero;
        bool started_before = false;
        if constexpr (NG > 1) {
            before.x = __shfl_up(acc.x, G); before.y = __shfl_up(acc.y, G); before.z = __shfl_up(acc.z, G); before.w = __shfl_up(acc.w, G);
            started_before = __shfl_up((int)started, G) != 0 && g > 0;
            if (g == 0) before = zero;
        }
        if (has_head) {
            head += before;
            if (started_before) {
                store(row_first, head);
            } else {  // (one group of a wave at most: the first whose row ends)
                head_sum[wave][l] = head;
                if (l == 0) head_row[wave] = row_first;
            }
        }
        if (g == NG - 1 && !ended) {
            tail_sum[wave][l] = acc;
            if (l == 0) { tail_row[wave] = row_last; tail_started[wave] = started; }
        }
    }
    __syncthreads();
    // The rows cut between the waves, the same way; only what is cut between workgroups is added atomically.
    // (a wave whose last row ends with it has tail_started, and no sum)
    auto with_waves_before = [&](int w, vec4u v, bool &started) -> vec4u {
        while (!started && --w >= 0) {
            if (tail_row[w] >= 0) v += tail_sum[w][l];
            started = tail_started[w];
        }
        return v;
    };
    if (g > 0) return;
    if (head_row[wave] >= 0) {
        bool started = false;
        const vec4u v = with_waves_before(wave, head_sum[wave][l], started);
        if (started) store(head_row[wave], v);
        else add(head_row[wave], v, 0);
    }
    if (wave == NW - 1 && tail_row[wave] >= 0) {
        bool started = tail_started[wave];
        add(tail_row[wave], with_waves_before(wave, tail_sum[wave][l], started), 1);
    }
}

// K < 4: one lane per output column
__global__ __launch_bounds__(256)
void sddmm_spmm_generic_kernel(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_ind, const float *__restrict__ x,
                               const float *__restrict__ H, float *Y, int64_t n_rows, int K)
{
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
    const int64_t n_waves = ((int64_t)gridDim.x * 256) >> 6;
    for (int64_t r = wave; r < n_rows; r += n_waves) {
        const int64_t b = row_ptr[r], e = row_ptr[r + 1];
        for (int k = 0; k < K; ++k) {
            float acc = 0.f;
            for (int64_t p = b + lane; p < e; p += 64) acc = fmaf(x[p], H[(int64_t)col_ind[p] * K + k], acc);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
            if (lane == 0) Y[r * (int64_t)K + k] = acc;
        }
    }
}

int checked(hipError_t e)
{
    if (e != hipSuccess) return fail(SDDMM_ERR_HIP, "sddmm_spmm_csr: %s", hipGetErrorString(e));
    return SDDMM_OK;
}

}  // namespace

namespace {

// How the product over nnz nonzeros at rank K >= 4 is dealt out: lanes per group, log2 of the nonzeros per group and
// of those per workgroup, slices of a row (of slice_pieces pieces each; the lanes of a group cover a slice).
struct CsrShape {
    int G, shift, wg_shift, slices, slice_pieces;
    int64_t workgroups;
};
// Pieces of four floats in a slice of a row, at most.  The slices of H follow each other over the whole matrix (the grid's
// second dimension), so a slice that fits a die's 4 MB of L2 is gathered from there, and the columns and values read once
// more per slice, 8 bytes a nonzero, cost less than that gives.  Where rows lie on lines of 128 bytes (K a multiple of 32):
// the widest slices of 32, 16 or 8 pieces that divide a row and fit, at least 16 below 1.5 million nonzeros, or the narrowest where
// none fits; whole rows where H fits as a whole, and at narrow ranks where there is too little to gain.  us, whole rows (two
// slices beyond K = 256) and so: band of 11.6 million in +-600 columns, K = 64 / 128 / 512 290 / 708 / 3067 and 193 / 385 / 1503; uniform, 3 million of 17,000
// columns, K = 128 / 256 128 / 337 and 85 / 156; word counts of 10 million, K = 96 / 256 267 / 973 and 213 / 558; ratings of
// 4.9 / 16.8 million, K = 256 225 / 1076 and 186 / 642; R-MAT of 1.8 / 7.5 million, K = 256 250 / 1236 and 165 / 785; window of
// 16,384 tokens, 5.2 million, K = 256 282 and 197.  Rows across lines of 128 bytes gain nothing up to K = 256 (a slice
// touches one line more); beyond, slices of 32 or 16 pieces fill their lanes better than two of up to 64 (K = 300: ratings of 4.9
// million 393 and 312, uniform of 3 million 579 and 440).
//   Beyond K = 512, where the rows of S are looked up once more per slice as well: band of 2.4 million, K = 1024 / 2048 1246 / 2468 and
// 818 / 2151, ratings of 5 million 937 / 1845 and 745 / 1469, R-MAT 2^18, 2.9 million, K = 1024 2001 and 1469.
//   Where not even slices of 8 pieces fit, it depends on how evenly the columns are used, which the call does not know: R-MAT of
// 2^18 to 2^20 vertices gains at five uses a column or more (2.9 / 4.9 million, K = 256 465 / 1074 and 301 / 810), uniform over
// 400,000 columns at 8 and 12 uses a column loses 3 to 8 % (4.7 million, K = 64 / 256 / 1024 174 / 673 / 2665 and 181 / 704 / 2833).  At
// less than four uses (few_uses) slices of 8 pieces lose below K = 256 (R-MAT 2^20, 1.6 million, K = 128 / 192 216 / 304 and 231 /
// 323, with 16 pieces 212 / 305; K = 96, 3.0 million of 1.5 million columns, 175 and 192), slices of 16 at K = 300 (uniform, 2
// million of a million columns 1116 and 1175) and below 1 to 1.5 million nonzeros (1.3 million of 400,000 columns, K = 256 248 and 265; R-MAT 2^17,
// 0.39 million, K = 512 129 and 141), and gain otherwise (R-MAT 2^20, 1.6 million, K = 256 / 512 488 / 1017 and 439 / 880).
//   Few nonzeros: a group has 4 of them, so a workgroup of whole rows has 16, and nearly every row of S is cut and added
// atomically; slices have more to a workgroup (14 thousand, K = 256 15.9 and 9.4).  Not where rows of S have next to no nonzeros
// (16 to 64 thousand in 65,536 rows, R-MAT, K = 160 / 200 17.8-22.4 / 19.6-24.6 and 22.3-25.1 / 25.0-27.7), from fewer rows on where slices
// of 16 pieces are not whole lines (uniform, 40 thousand in 30,000 rows, K = 200 16.1 and 19.0).
int slice_pieces_most(int64_t nnz, int64_t n_rows, int64_t n_cols, int K)
{
    constexpr int64_t kL2 = 4200000;
    const int pieces = (K + 3) / 4;
    const int64_t h = 16 * (int64_t)pieces * n_cols;
    if (nnz <= 65536) return K >= 160 && n_rows <= (K % 64 == 0 ? 40000 : nnz * 2 / 3) && pieces <= 16 * kMostSlices ? 16 : 64;
    const int wide = K <= 256 || pieces > 32 * kMostSlices ? 64 : 32;
    if (nnz < 300000 || h <= kL2 || pieces > 8 * kMostSlices) return wide;
    const bool few_uses = nnz < 4 * n_cols;
    if (K % 32 != 0) return K > 256 && nnz >= 1500000 && !few_uses ? 16 : wide;
    if (K < 192 && (nnz < (K < 96 ? 4000000 : K < 128 ? 2000000 : 1500000) || h <= (K < 96 ? 20000000 : K < 128 ? 6000000 : kL2))) return wide;
    if (few_uses && nnz < (K <= 256 ? 1500000 : 1000000)) return wide;
    int narrow = 0;  // the narrowest that divides a row
    for (int p : {32, 16, 8}) {
        if (p >= pieces || pieces % p != 0 || (p == 8 && (nnz < 1500000 || (few_uses && K < 256)))) continue;
        narrow = p;
        if (16 * (int64_t)p * n_cols <= kL2) break;
    }
    return narrow ? narrow : wide;
}
CsrShape csr_shape(int64_t nnz, int64_t n_rows, int64_t n_cols, int K)
{
    CsrShape c;
    const int pieces = (K + 3) / 4, most = slice_pieces_most(nnz, n_rows, n_cols, K);
    c.slices = (pieces + most - 1) / most;
    c.slice_pieces = (pieces + c.slices - 1) / c.slices;
    c.G = 4;
    while (c.G < c.slice_pieces) c.G *= 2;
    // Nonzeros per wave: up to 512 (a workgroup's cut rows cost atomic adds), as many as leave 8192 waves, but not fewer
    // than 64 until there are less than 2048 of them: too few waves leave the latency of the gathers bare.  Measured,
    // us at 32 / 64 / 128 / 256 / 512 per wave: 253 thousand nonzeros, K = 256: 42 / 37 / 38 / 54 / -; 1.8 million, K = 100:
    // 106 / 85 / 82 / 88 / 100; 98 million, K = 128: 5148 / 3483 / 3125 / 3029 / 2979.
    const int groups_log2 = __builtin_ctz(64 / c.G);
    c.shift = 9 - groups_log2;
    auto waves = [&] { return (nnz >> (c.shift + groups_log2)) * c.slices; };
    while (c.shift > 2 && c.shift + groups_log2 > 6 && waves() < 8192) --c.shift;
    while (c.shift > 2 && waves() < 2048) --c.shift;
    c.wg_shift = c.shift + groups_log2 + 2;
    c.workgroups = (nnz + ((int64_t)1 << c.wg_shift) - 1) >> c.wg_shift;
    return c;
}

template <bool RECORDS>
hipError_t launch_csr(const CsrShape &c, int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *row_ptr, const int32_t *col_ind, const float *x,
                      int K, const float *H, float *Y, float *part, hipStream_t st)
{
    const dim3 grid((unsigned)c.workgroups, (unsigned)c.slices);
    const bool wide = n_cols * K >= (int64_t)1 << 30;
#define SPMM(g)                                                                                                                          \
    case g:                                                                                                                              \
        return launch(wide ? sddmm_spmm_csr_kernel<g, RECORDS, true> : sddmm_spmm_csr_kernel<g, RECORDS, false>, grid, dim3(256), 0, st, \
                      row_ptr, col_ind, x, H, Y, part, (int)n_rows, (int)nnz, K, 1 << c.shift, c.slice_pieces)
    switch (c.G) { SPMM(4); SPMM(8); SPMM(16); SPMM(32); SPMM(64); }
#undef SPMM
    return hipErrorInvalidValue;
}

// Rows that a wave of the kernels beside the product looks at.
int rows_per_wave(int64_t n_rows, int K)
{
    int per_wave = 64;
    while (per_wave > 1 && n_rows < (int64_t)1024 * per_wave && per_wave / 2 * ((K + 3) / 4) >= 64) per_wave /= 2;
    return per_wave;
}

}  // namespace

namespace sddmm {

int64_t spmm_csr_records(int64_t nnz, int64_t n_rows, int64_t n_cols, int K) { return K < 4 ? 0 : 2 * csr_shape(nnz, n_rows, n_cols, K).workgroups; }

int launch_spmm_csr_records(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *d_row_ptr, const int32_t *d_col_ind, const float *d_x, int32_t K,
                            const float *d_H, float *d_Y, float *d_part, void *stream)
{
    const CsrShape c = csr_shape(nnz, n_rows, n_cols, K);
    hipStream_t st = (hipStream_t)stream;
    if (int rc = checked(launch_csr<true>(c, n_rows, n_cols, nnz, d_row_ptr, d_col_ind, d_x, K, d_H, d_Y, d_part, st))) return rc;
    const int per_wave = rows_per_wave(n_rows, K);
    return checked(launch(sddmm_spmm_cut_rows_kernel, dim3((unsigned)((n_rows + 4 * per_wave - 1) / (4 * per_wave))), dim3(256), 0, st, d_row_ptr,
                          d_part, d_Y, n_rows, (int)K, c.wg_shift, per_wave));
}

}  // namespace sddmm

extern "C" int sddmm_spmm_csr(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *d_row_ptr, const int32_t *d_col_ind,
                              const float *d_x, int32_t K, const float *d_H, float *d_Y, void *stream)
{
    if (n_rows < 0 || n_cols < 0 || nnz < 0 || K < 1) return fail(SDDMM_ERR_ARG, "sddmm_spmm_csr: bad sizes");
    if (n_rows == 0) return SDDMM_OK;
    if (!d_row_ptr || !d_Y || (nnz > 0 && (!d_col_ind || !d_x || !d_H))) return fail(SDDMM_ERR_ARG, "sddmm_spmm_csr: NULL argument");
    if (nnz >= INT32_MAX || n_rows >= INT32_MAX) return fail(SDDMM_ERR_RANGE, "sddmm_spmm_csr: sizes beyond int32 offsets");
    hipStream_t st = (hipStream_t)stream;
    if (K < 4) {
        const unsigned grid = (unsigned)std::min<int64_t>((n_rows + 3) / 4, 256 * 64);
        return checked(launch(sddmm_spmm_generic_kernel, dim3(grid), dim3(256), 0, st, d_row_ptr, d_col_ind, d_x, d_H, d_Y, n_rows, (int)K));
    }
    const CsrShape c = csr_shape(nnz, n_rows, n_cols, K);
    const int per_wave = rows_per_wave(n_rows, K);
    if (int rc = checked(launch(sddmm_spmm_zero_rows_kernel, dim3((unsigned)((n_rows + 4 * per_wave - 1) / (4 * per_wave))), dim3(256), 0, st, d_row_ptr,
                                d_Y, n_rows, (int)K, c.wg_shift, per_wave)))
        return rc;
    if (nnz == 0) return SDDMM_OK;
    return checked(launch_csr<false>(c, n_rows, n_cols, nnz, d_row_ptr, d_col_ind, d_x, K, d_H, d_Y, nullptr, st));
}
