// The row-wise softmax of the sampled products (attention scores restricted to the pattern of S),
// for gfx950 (MI355X).  It works on the sorted S directly (CSR pointers + one fp32 per nonzero), so it
// follows a plan's sddmm_execute on the same stream without any re-ordering.
#include <hip/hip_runtime.h>
#include <mutex>
#include "internal.hpp"
#include "launch.hpp"
#include "softmax_exp.hpp"

using namespace sddmm;

namespace {

// Row softmax.  An entry is read once and written once, and the work is dealt out by entries and rows whatever the rows'
// lengths (a matrix may hold a few rows of a million entries next to millions of rows of ten or of none): an entry counts
// 1 and a row kSmRow, the rows are laid end to end on that scale, and a wave takes an equal share of it, a workgroup a
// unit of four shares.  A row belongs to the wave in whose share it starts, which finds its first row by a search of the
// row pointers:
//   rows of up to kSmByWave entries are held whole in registers, 64 rows at a time: a lane per row of up to 8 entries, then
//        groups of 8 lanes (up to 96), of 32 lanes (up to 512), the whole wave;
//   longer rows (up to kSmLongMax entries) are worked on by the whole workgroup afterwards, in registers;
//   huge rows (longer still): every workgroup takes the piece that lies in its unit, stores it as exp(x - m) with the
//        piece's own maximum m and leaves (m, sum) and the row in a record of the unit; a second kernel, which finds
//        nothing to do on most matrices, merges the records of each huge row and scales its pieces.
// No staging: a row's loads are all in flight together, and 16 waves per compute unit hide their latency, which is
// what bounds it until the entries do (the recommender pattern moves 0.8 GB at 3.5 TB/s).  Before this a kernel of its own
// laid chunks of whole rows out, and rows that had been left over went through lists to a third one.  us, before and now: 18
// thousand entries 11.8 and 7.7; R-MAT, 1.9 million 34 and 18, 28 million 134 and 111, 84 million 297 and 266, 189 million
// 526 and 526; window of 320 a row, 5.2 million 24 and 19; 3 million rows of one
// entry 38 and 30; 20 thousand entries spread over 4 million rows 93 and 23; a row of 30 million 328 and 93; recommender,
// 100 million 235 and 231.  (Maximum and sum by scans over the entries, whatever the rows: 1072 there, bound by the vector
// ALU.)
constexpr int kSmBlock = 256;
constexpr int kSmWaves = kSmBlock / 64;
constexpr int kSmLongQ = 17;                             // float4 per thread of the long-row function
constexpr int kSmLongMax = kSmLongQ * 4 * kSmBlock - 8;  // (less what a misaligned start costs)
constexpr int kSmByLane = 8, kSmBy8 = 96, kSmBy32 = 512, kSmByWave = 1024;  // row lengths up to which a lane / 8 lanes / 32 lanes / the wave work on a row
constexpr int kSmRow = 4;                                // (with 16 R-MAT, 28 million: 155 instead of 131)
constexpr int kSmShareMax = 8192;                        // (recommender, rows counting 4: 241, with 4096 258)
constexpr int kSmLeft = (kSmShareMax - 1) / (kSmByWave + 1) + 1;  // rows of more than kSmByWave entries that start in a share, at most
constexpr int kSmPieceMax = 16384;                       // a unit of the largest share makes two pieces of a huge row, worked on like long rows
static_assert(kSmPieceMax <= kSmLongMax);
constexpr int64_t kSmScaleMax = (int64_t)1 << 32;        // (2^31 entries, and as much for the rows: see softmax_scale)
constexpr int64_t kSmMaxPieces = kSmScaleMax / kSmPieceMax;

// The scale: row r starts at row_ptr[r] + row * r and the last one ends at `total`.
struct SoftmaxScale {
    int64_t total;
    int row, share;
    __host__ __device__ int unit() const { return kSmWaves * share; }
    __host__ __device__ int64_t units() const { return (total + unit() - 1) / unit(); }
    __host__ __device__ int piece() const { return unit() < kSmPieceMax ? unit() : kSmPieceMax; }
    __host__ __device__ int64_t pieces() const { return (total + piece() - 1) / piece(); }
};
// Shares: from 2^21 on the scale as large as leaves 4096 of them, up to kSmShareMax; below as small as makes no more than
// 4096, which is what runs at a time, not below 64: what a share costs whatever it holds, a search and the row pointers, is
// most of the time there, and a second turn of workgroups pays for it again.  us of the kernel alone with 4096 shares at
// least and at most: rows of 14, 0.23 million entries 9.8 and 6.0; of 900, 0.9 million 11.4 and 7.4; of 40, 1.2 million 10.0
// and 7.9; R-MAT, 0.24 / 0.69 / 1.3 million 10.7 / 14.5 / 15.0 and 9.2 / 10.4 / 14.3, but 1.86 million (2.4 on the scale) 15.5
// and 18.2.  (By counting zeros: in two loops that double the share it cost the workgroups of a large grid that find no unit
// more than launching them.  4 million empty rows, softmax and merge, with loops 23.4 us, so 19.2; two million rows of one 26.1 and 24.4.)
__host__ __device__ inline SoftmaxScale softmax_scale(int64_t nnz, int64_t n_rows)
{
    SoftmaxScale s;
    s.row = n_rows <= (int64_t)1 << 27 ? kSmRow : 1;
    s.total = nnz + s.row * n_rows;
    const uint64_t t = s.total > 2 ? s.total : 2;
    // (log2 of a 4096th of the scale, rounded up and down)
    const int up = 64 - __builtin_clzll(t - 1) - 12, down = 63 - __builtin_clzll(t) - 12;
    s.share = 1 << (down < 10 ? (up < 6 ? 6 : up < 9 ? up : 9) : down < 13 ? down : 13);
    return s;
}

// Per unit, or half of one (see piece): (m, sum) of the piece of a huge row that began before it, [2i], and of one that starts
// in it, [2i + 1]; the rows themselves plus one (0: none).  The kernels take both arrays as arguments: a caller's workspace
// (sddmm_execute_ws), or these file-scope arrays, 4 + 2 MiB per device, held until the process ends -- softmax calls
// without a workspace that overlap in time on one device share them and must not (calls on one stream never do).
static __device__ __align__(256) float2 g_softmax_rec_store[2 * kSmMaxPieces];
static __device__ __align__(256) int2 g_softmax_rows_store[kSmMaxPieces];

template <int GW>
__device__ __forceinline__ float group_max(float v)
{
#pragma unroll
    for (int off = GW / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}
template <int GW>
__device__ __forceinline__ float group_sum(float v)
{
#pragma unroll
    for (int off = GW / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// One whole row of len entries at xr / outr by a group of GW lanes (GW = 1: the lane alone), R entries
// per lane, all of them requested before the first is used.  Every lane of the wave runs through this
// (the lane exchanges must not sit under a branch); `mine` says whether the lane's group has a row.
template <int GW, int R>
__device__ __forceinline__ void softmax_row_by_group(const float *xr, float *outr, int len, bool mine)
{
    const int gl = threadIdx.x & (GW - 1);
    if (!mine) len = 0;
    float v[R];
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = gl + k * GW < len ? xr[gl + k * GW] : -INFINITY;
    float m = v[0];
#pragma unroll
    for (int k = 1; k < R; ++k) m = fmaxf(m, v[k]);
    m = group_max<GW>(m);
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        v[k] = gl + k * GW < len ? exp_nonpositive(v[k] - m) : 0.f;
        sum += v[k];
    }
    sum = group_sum<GW>(sum);
    const float inv = 1.0f / sum;
#pragma unroll
    for (int k = 0; k < R; ++k) if (gl + k * GW < len) outr[gl + k * GW] = v[k] * inv;
}

// One long row, or one piece of a huge row, [rb, re) by a workgroup of kSmBlock threads, held in registers
// (4 * NQ floats per thread): read once, written once.  x 16-byte aligned: float4 pieces counted from the
// aligned address below the first entry (entries outside are masked); otherwise single entries, strided.
// rec = NULL: a whole row, normalised; otherwise a piece, stored as exp(x - max) with (max, sum) in *rec.
template <int NQ>
__device__ __forceinline__ void softmax_long_row(const float *x, float *out, int64_t rb, int64_t re, int64_t nnz, bool vec_in,
                                                 bool vec_out, float *red, float2 *rec)
{
    constexpr int NW = kSmBlock / 64;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // (offsets relative to the aligned address below the row's start fit 32 bits)
    const int64_t a0 = vec_in ? (rb & ~(int64_t)3) : rb;
    const float *xr = x + a0;
    float *outr = out + a0;
    const int head = (int)(rb - a0), end = (int)(re - a0);
    const int lim = (int)min(nnz - a0, (int64_t)INT32_MAX);  // entries of the array from a0 on
    float f[4 * NQ];
    if (vec_in) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            const int p = 4 * (t + k * kSmBlock);
            float4 v = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
            if (p < end) {
                if (p + 3 < lim) {
                    v = *reinterpret_cast<const float4 *>(xr + p);
                } else {
                    v.x = xr[p];
                    if (p + 1 < lim) v.y = xr[p + 1];
                    if (p + 2 < lim) v.z = xr[p + 2];
                }
            }
            f[4 * k + 0] = (p + 0 >= head && p + 0 < end) ? v.x : -INFINITY;
            f[4 * k + 1] = (p + 1 >= head && p + 1 < end) ? v.y : -INFINITY;
            f[4 * k + 2] = (p + 2 >= head && p + 2 < end) ? v.z : -INFINITY;
            f[4 * k + 3] = (p + 3 >= head && p + 3 < end) ? v.w : -INFINITY;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4 * NQ; ++k) {
            const int p = t + k * kSmBlock;
            f[k] = p < end ? xr[p] : -INFINITY;
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < 4 * NQ; ++k) m = fmaxf(m, f[k]);
    m = group_max<64>(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) m = fmaxf(m, red[w]);
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < 4 * NQ; ++k) {
        f[k] = f[k] == -INFINITY ? 0.f : exp_nonpositive(f[k] - m);
        sum += f[k];
    }
    sum = group_sum<64>(sum);
    if (lane == 0) red[NW + wave] = sum;
    __syncthreads();
    sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += red[NW + w];
    const float inv = rec ? 1.0f : 1.0f / sum;
    if (rec && t == 0) *rec = make_float2(m, sum);
    if (vec_in) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            const int p = 4 * (t + k * kSmBlock);
            if (p >= end) continue;
            if (vec_out && p >= head && p + 4 <= end) {
                *reinterpret_cast<float4 *>(outr + p) = make_float4(f[4 * k] * inv, f[4 * k + 1] * inv, f[4 * k + 2] * inv, f[4 * k + 3] * inv);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) if (p + j >= head && p + j < end) outr[p + j] = f[4 * k + j] * inv;
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4 * NQ; ++k) {
            const int p = t + k * kSmBlock;
            if (p < end) outr[p] = f[k] * inv;
        }
    }
    // (the next row writes its maxima after this row's second barrier and its sums after its own first: no barrier needed here)
}

// 64 rows by a wave: the lane's one has len entries from rb on (0: none, or not to be done here; at most kSmByWave).
// few: rows of up to kSmByLane entries go with the next longer ones where that saves a pass.
__device__ __forceinline__ void softmax_row_batch(const float *x, float *out, int rb, int len, int lane, bool few)
{
    const uint64_t by_lane = __ballot(len >= 1 && len <= kSmByLane);
    uint64_t todo = __ballot(len > kSmByLane && len <= kSmBy8);
    // a lane per row
    if (few && (__builtin_popcountll(todo) + 7) / 8 >= (__builtin_popcountll(by_lane | todo) + 7) / 8) todo |= by_lane;
    else if (by_lane) softmax_row_by_group<1, kSmByLane>(x + rb, out + rb, len, len <= kSmByLane);
    // groups of 8 lanes: eight rows at a time
    while (todo) {
        int src = -1;  // the lane that holds the row of this lane's group
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const int b = todo ? __builtin_ctzll(todo) : -1;
            if (todo) todo &= todo - 1;
            if ((lane >> 3) == g) src = b;
        }
        const int gb = __shfl(rb, src < 0 ? lane : src);
        const int gn = __shfl(len, src < 0 ? lane : src);
        softmax_row_by_group<8, kSmBy8 / 8>(x + gb, out + gb, gn, src >= 0);
    }
    // groups of 32 lanes: two rows at a time
    todo = __ballot(len > kSmBy8 && len <= kSmBy32);
    while (todo) {
        int src = -1;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int b = todo ? __builtin_ctzll(todo) : -1;
            if (todo) todo &= todo - 1;
            if ((lane >> 5) == g) src = b;
        }
        const int gb = __shfl(rb, src < 0 ? lane : src);
        const int gn = __shfl(len, src < 0 ? lane : src);
        softmax_row_by_group<32, kSmBy32 / 32>(x + gb, out + gb, gn, src >= 0);
    }
    // the whole wave: row by row
    todo = __ballot(len > kSmBy32);
    while (todo) {
        const int b = __builtin_ctzll(todo);
        todo &= todo - 1;
        const int gb = __shfl(rb, b);
        softmax_row_by_group<64, kSmByWave / 64>(x + gb, out + gb, __shfl(len, b), true);
    }
}

// The last row that starts at k on the scale or before it, by the whole wave: 64 probes a round.
__device__ __forceinline__ int softmax_row_at(const int32_t *__restrict__ row_ptr, int n_rows, int row, int64_t k, int lane)
{
    int lo = 0, hi = n_rows;  // (the answer lies in [lo, hi))
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) >> 6;
        const int64_t at = (int64_t)lo + (int64_t)step * (lane + 1);
        const bool below = at < hi && row_ptr[at] + (int64_t)row * at <= k;
        const int c = __builtin_popcountll(__ballot(below));  // (monotone: the first c lanes)
        const int base = lo;
        lo = base + step * c;
        hi = (int)min((int64_t)hi, (int64_t)base + (int64_t)step * (c + 1));
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// First kernel: see above.
__global__ __launch_bounds__(kSmBlock, 4)  // (four long rows in flight per compute unit)
void sddmm_row_softmax_kernel(const int32_t *__restrict__ row_ptr, int64_t n_rows_, const float *x, float *out, float2 *__restrict__ rec,
                              int2 *__restrict__ rec_rows)
{
    __shared__ float red[2 * kSmWaves];
    // rows that the waves leave to the workgroup: row, first entry, length (read once more from the row pointers, and the row
    // that began before the unit looked up there by all waves, they cost units without any such row 3 us)
    __shared__ int3 left[kSmWaves * kSmLeft + 1];
    __shared__ int n_left;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_rows = (int)n_rows_, nnz = row_ptr[n_rows];
    const SoftmaxScale scale = softmax_scale(nnz, n_rows);
    const int64_t unit = scale.unit(), n_units = scale.units(), piece = scale.piece();
    // (A share of 64 starts sixteen rows at most, two passes of groups of 8: a pass of lanes before them is one more chain of loads and
    // sums where it saves none of theirs, and one less where it does.  us of softmax and merge, a lane per short row never, always
    // and by that rule: R-MAT of 1024 rows, 25 / 36 thousand entries 7.9 / 7.9, 8.4 / 8.4 and 8.0 / 7.9; 4096 rows, 29 / 117 thousand 7.9 /
    // 8.7, 8.3 / 9.1 and 8.0 / 8.6 (18 thousand 7.8, 7.5 and 7.7); 20 thousand rows of one 8.3, 6.4 and 6.6.  In larger shares always:
    // 3.5 million, R-MAT, 20.9, never 22.5.)
    const bool few = scale.share == 64;
    const bool vec_in = (reinterpret_cast<uintptr_t>(x) & 15u) == 0, vec_out = (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
    for (int64_t u = blockIdx.x; u < n_units; u += gridDim.x) {
        const int64_t k0 = u * unit, k1 = min(scale.total, k0 + unit);
        if (u != blockIdx.x) __syncthreads();  // (left has been read)
        if (threadIdx.x == 0) n_left = 0;
        if (threadIdx.x * piece < k1 - k0) rec_rows[k0 / piece + threadIdx.x] = make_int2(0, 0);
        __syncthreads();
        const int64_t s0 = k0 + wave * scale.share, s1 = min(k1, s0 + scale.share);
        if (s0 < s1) {
            const int r0 = softmax_row_at(row_ptr, n_rows, scale.row, s0, lane);
            if (wave == 0) {  // (the row that began before the unit, if it is a huge one that goes on in it)
                const int rb = row_ptr[r0], re = row_ptr[r0 + 1];
                const int64_t at = rb + (int64_t)scale.row * r0;
                if (re - rb > kSmLongMax && at < k0 && at + (re - rb) > k0 && lane == 0) left[atomicAdd(&n_left, 1)] = make_int3(r0, rb, re - rb);
            }
            for (uint32_t w0 = r0;; w0 += 64) {
                const uint32_t r = w0 + lane;
                const int rb = row_ptr[min(r, (uint32_t)n_rows)], re = row_ptr[min(r + 1, (uint32_t)n_rows)];
                const int64_t at = rb + (int64_t)scale.row * r;
                const int len = at >= s0 && at < s1 ? re - rb : 0;  // (r0 may begin before the share)
                if (len > kSmByWave) left[atomicAdd(&n_left, 1)] = make_int3((int)r, rb, re - rb);
                softmax_row_batch(x, out, rb, len > kSmByWave ? 0 : len, lane, few);
                if (__ballot(r >= (uint32_t)n_rows || at >= s1)) break;
            }
        }
        __syncthreads();
        const int n = n_left;
#pragma unroll 1
        for (int w = 0; w < n; ++w) {
            const int3 l = left[w];
            const int r = l.x;
            const int64_t b = l.y, len = l.z, at = b + (int64_t)scale.row * r;
            const bool huge = len > kSmLongMax;
            if (len <= 4 * 4 * kSmBlock - 8) {
                softmax_long_row<4>(x, out, b, b + len, nnz, vec_in, vec_out, red, nullptr);
                continue;
            }
            // (of a huge row what lies in this unit, piece by piece)
            const int64_t stop = huge ? min(len, k1 - at) : len;
            for (int64_t p = huge ? max((int64_t)0, k0 - at) : 0; p < stop;) {
                const int64_t i = (at + p) / piece, e = huge ? min(stop, (i + 1) * piece - at) : len;
                const int which = at < i * piece ? 0 : 1;
                if (huge && threadIdx.x == 0) (which ? rec_rows[i].y : rec_rows[i].x) = r + 1;
                softmax_long_row<kSmLongQ>(x, out, b + p, b + e, nnz, vec_in, vec_out, red, huge ? &rec[2 * i + which] : nullptr);
                p = e;
            }
        }
    }
}

// (m, sum) of the huge row of len entries that starts at `at` on the scale from the records of its pieces: the second
// one of the piece it starts in, the first ones of the others; every wave of the workgroup computes the same pair.
__device__ __forceinline__ float2 merged_record(const float2 *__restrict__ rec, int64_t at, int64_t len, int piece)
{
    const int lane = threadIdx.x & 63;
    const int64_t ua = at / piece, ub = (at + len - 1) / piece;
    float m = -INFINITY, s = 0.f;
    for (int64_t k = ua + lane; k <= ub; k += 64) {
        const float2 r = rec[2 * k + (k == ua ? 1 : 0)];
        const float mn = fmaxf(m, r.x);
        // (no record yet, or one of nothing but -inf: its term must vanish without producing inf - inf)
        s = (s == 0.f ? 0.f : s * expf(m - mn)) + (r.y == 0.f ? 0.f : r.y * expf(r.x - mn));
        m = mn;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float m2 = __shfl_xor(m, off), s2 = __shfl_xor(s, off);
        const float mn = fmaxf(m, m2);
        // (a lane without records holds (-inf, 0), one with a record of NaNs alone (-inf, NaN))
        const float t1 = s == 0.f ? 0.f : s * expf(m - mn), t2 = s2 == 0.f ? 0.f : s2 * expf(m2 - mn);
        s = t1 + t2;
        m = mn;
    }
    return make_float2(m, s);
}

// out[b..e) *= f by the whole workgroup, eight entries per thread in flight
__device__ __forceinline__ void scale_range(float *out, int64_t b, int64_t e, float f)
{
    for (int64_t i0 = b + threadIdx.x; i0 < e; i0 += 8 * kSmBlock) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = i0 + u * kSmBlock < e ? out[i0 + u * kSmBlock] : 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) if (i0 + u * kSmBlock < e) out[i0 + u * kSmBlock] = v[u] * f;
    }
}

// Second kernel: the pieces of huge rows are scaled to the whole row's maximum and sum.  A workgroup takes four consecutive
// pieces at a time, which mostly are of one row, and merges that row's records once; four and not an equal range, since
// huge rows may lie together (R-MAT 2^22, 189 million, the whole softmax: 583 us with 1024 workgroups, 855 with a range for
// each of 256).
__global__ __launch_bounds__(kSmBlock)
void sddmm_row_softmax_merge_kernel(const int32_t *__restrict__ row_ptr, int64_t n_rows, float *out, const float2 *__restrict__ rec,
                                    const int2 *__restrict__ rec_rows)
{
    const SoftmaxScale scale = softmax_scale(row_ptr[n_rows], n_rows);
    const int64_t size = scale.piece(), n_pieces = scale.pieces();
    constexpr int kTogether = 4;
    int merged_row = -1;
    float2 all = make_float2(0.f, 1.f);
    for (int64_t base = (int64_t)blockIdx.x * kTogether; base < n_pieces; base += (int64_t)gridDim.x * kTogether) {
        for (int64_t u = base; u < min(n_pieces, base + kTogether); ++u) {
            const int2 rows = rec_rows[u];
            for (int which = 0; which < 2; ++which) {
                const int r = (which ? rows.y : rows.x) - 1;
                if (r < 0) continue;
                const int64_t rb = row_ptr[r], re = row_ptr[r + 1];
                const int64_t at = rb + (int64_t)scale.row * r;
                if (r != merged_row) all = merged_record(rec, at, re - rb, (int)size);
                merged_row = r;
                const float2 piece = rec[2 * u + which];
                scale_range(out, rb + max((int64_t)0, u * size - at), min(re, rb + ((u + 1) * size - at)), expf(piece.x - all.x) / all.y);
            }
        }
    }
}

}  // namespace

namespace sddmm {

// device addresses of the file-scope record arrays on the current device (looked up once per device)
static int softmax_store(float2 **rec, int2 **rows)
{
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static float2 *rec_of[kMaxDevices] = {};
    static int2 *rows_of[kMaxDevices] = {};
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(SDDMM_ERR_HIP, "sddmm_row_softmax: no usable current device");
    std::lock_guard<std::mutex> lock(mu);
    if (!rec_of[dev]) {
        void *a = nullptr, *b = nullptr;
        if ((e = hipGetSymbolAddress(&a, HIP_SYMBOL(g_softmax_rec_store))) != hipSuccess ||
            (e = hipGetSymbolAddress(&b, HIP_SYMBOL(g_softmax_rows_store))) != hipSuccess || !a || !b)
            return fail(SDDMM_ERR_HIP, "sddmm_row_softmax: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
        rec_of[dev] = static_cast<float2 *>(a);
        rows_of[dev] = static_cast<int2 *>(b);
    }
    *rec = rec_of[dev];
    *rows = rows_of[dev];
    return SDDMM_OK;
}

int64_t row_softmax_workspace_bytes(int64_t nnz, int64_t n_rows)
{
    return ((softmax_scale(nnz, n_rows).pieces() * 24 + 255) / 256) * 256;  // two float2 and one int2 per piece
}

int launch_row_softmax(int64_t n_rows, const int32_t *d_row_ptr, const float *d_x, float *d_out, void *stream, void *d_ws, int64_t nnz, int64_t longest_row)
{
    if (n_rows <= 0) return SDDMM_OK;
    float2 *rec = nullptr;
    int2 *rows = nullptr;
    if (d_ws) {  // [2 * pieces] records, then [pieces] pairs of rows
        rec = static_cast<float2 *>(d_ws);
        rows = reinterpret_cast<int2 *>(rec + 2 * softmax_scale(nnz, n_rows).pieces());
    } else if (int rc = softmax_store(&rec, &rows)) {
        return rc;
    }
    // The entry count lives on the device: the grids are sized by the rows, the kernels stride over the entries.  1024
    // workgroups run at a time, and a unit of heavy rows takes long: the more workgroups the units are dealt to, the more
    // evenly the machine is filled at the end, but a workgroup that finds nothing costs its launch.  us with 2048 / 4096 /
    // 8192 workgroups: R-MAT 2^22, 189 million entries 574 / 544 / 536, 2^21, 84 million 297 / 282 / 282; recommender, 480
    // thousand rows 239 / 231 / 231; 4096 rows, 18 thousand entries 8.8 / 8.9 / 11.1, 167 thousand 9.4 / 10.9.  With 1024 /
    // 4096 for the merge: 574 / 564, 297 / 275, 4096 rows 8.8 / 10.8.  What the larger grids cost a matrix of a million
    // rows or more with next to no entries: 4 million rows, 20 thousand entries 19.2 and 22.2.
    const int main_groups = n_rows >= (int64_t)1 << 20 ? 8192 : n_rows >= (int64_t)1 << 18 ? 4096 : 2048;
    const int merge_groups = n_rows >= (int64_t)1 << 20 ? 4096 : 1024;
    const hipStream_t st = (hipStream_t)stream;
    hipError_t e = launch(sddmm_row_softmax_kernel, dim3(main_groups), dim3(kSmBlock), 0, st, d_row_ptr, n_rows, d_x, d_out, rec, rows);
    if (e == hipSuccess && longest_row > kSmLongMax) e = launch(sddmm_row_softmax_merge_kernel, dim3(merge_groups), dim3(kSmBlock), 0, st, d_row_ptr, n_rows, d_out, rec, rows);
    if (e != hipSuccess) return fail(SDDMM_ERR_HIP, "sddmm_row_softmax: %s", hipGetErrorString(e));
    return SDDMM_OK;
}

}  // namespace sddmm

extern "C" {

int sddmm_row_softmax(int64_t n_rows, const int32_t *d_row_ptr, const float *d_x, float *d_out, void *stream)
{
    if (n_rows < 0 || (n_rows > 0 && (!d_row_ptr || !d_x || !d_out))) return fail(SDDMM_ERR_ARG, "sddmm_row_softmax: bad arguments");
    if (n_rows >= INT32_MAX) return fail(SDDMM_ERR_RANGE, "sddmm_row_softmax: more than 2^31 - 2 rows");
    return launch_row_softmax(n_rows, d_row_ptr, d_x, d_out, stream, nullptr, 0, INT64_MAX);
}

}  // extern "C"
