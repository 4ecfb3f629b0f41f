// Device helpers of the kernels that walk the sorted S by nonzeros (gfx950, wave64): finding the rows of a
// range of nonzeros from the row pointers alone, and reading rows of a dense factor whose length is no
// multiple of four.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace sddmm {

// A piece of four floats at any 4-byte boundary.  The hardware's 16-byte global loads and stores need no more,
// so rows of any length take the same instructions as aligned ones (a piece may touch one cache line more).
typedef float vec4u __attribute__((ext_vector_type(4), aligned(4)));

// The row in [lo, hi) that holds nonzero p (row_ptr[lo] <= p < row_ptr[hi], all uniform), by the whole wave: 64 probes a
// round, so three rounds of one load each for a quarter of a million rows where a binary search is a chain of eighteen.
__device__ __forceinline__ int wave_find_row(const int32_t *__restrict__ row_ptr, int lo, int hi, int p, int lane)
{
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) >> 6;
        const int64_t at = (int64_t)lo + (int64_t)step * (lane + 1);
        const bool below = at < hi && row_ptr[at] <= p;
        const int c = __builtin_popcountll(__ballot(below));  // (monotone: the first c lanes)
        const int base = lo;
        lo = base + step * c;
        hi = (int)min((int64_t)hi, (int64_t)base + (int64_t)step * (c + 1));
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Inclusive maximum over the lanes up to this one (v >= 0).
__device__ __forceinline__ int wave_max_scan(int v)
{
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));  // row_shr:1
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return v;
}

// tab[i] = the row of nonzero p0 + i for 0 <= i < n, tab in this wave's own LDS, n rounded up to 64, plus one entry;
// nnz = row_ptr[n_rows] > p0.  Returns the row of p0.  tab[n] becomes a row other than that of nonzero p0 + n - 1 if a row
// ends there. (Entries past the last nonzero hold n_rows.)  The row starts inside the range are marked, one coalesced read
// of the row pointers for 64 rows, and a running maximum fills the rest; of the rows that start at one nonzero (empty ones)
// the last counts.  Every read waits for the one before (0.34 us each), so the walk ends at the last nonzero, and after as
// many steps as the search takes it is given up for that: each lane looks for the rows of its own nonzeros among those
// left.  (20 thousand nonzeros, K = 16, us without / with both: 4 million empty rows behind them 20700 / 8, spread over 4
// million rows 59 / 15.)
__device__ __forceinline__ int rows_of_range(const int32_t *__restrict__ row_ptr, int n_rows, int nnz, int p0, int n, int *tab, int lane)
{
    const int n_pad = (n + 63) & ~63;
    const int end = min(n, nnz - p0);
    const int r0 = wave_find_row(row_ptr, 0, n_rows, p0, lane);
    for (int i = lane; i <= n_pad; i += 64) tab[i] = 0;
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) tab[0] = r0;
    __builtin_amdgcn_wave_barrier();
    const int most = 16 + (n >> 4);
    int base = r0 + 1, last = 0;  // the rows before base are marked; row base - 1 starts at nonzero p0 + last, or before p0
    for (int step = 0; step < most && last < end; ++step, base += 64) {
        const int r = base + lane;
        const int rel = r <= n_rows ? row_ptr[r] - p0 : INT32_MAX;
        const int next = __shfl_down(rel, 1);
        if (rel <= end && (rel != next || lane == 63)) tab[rel] = r;
        last = __builtin_amdgcn_readlane(rel, 63);
    }
    if (__builtin_expect(last < end, 0)) {
        const int r1 = wave_find_row(row_ptr, base - 1, n_rows, p0 + end - 1, lane);
        constexpr int U = 4;  // searches of a lane at a time
        for (int i0 = last & ~63; i0 < end; i0 += 64 * U) {
            int lo[U];
#pragma unroll
            for (int u = 0; u < U; ++u) lo[u] = base - 1;
            for (int span = r1 - (base - 1); span > 0; span >>= 1) {  // the row lies in [lo, lo + span]
                const int half = (span + 1) >> 1;
                int at[U];
#pragma unroll
                for (int u = 0; u < U; ++u) at[u] = row_ptr[lo[u] + half];
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (at[u] - p0 <= i0 + 64 * u + lane) lo[u] += half;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = i0 + 64 * u + lane;
                if (i >= last && i < end) tab[i] = lo[u];
            }
        }
        if (lane == 0 && r1 < n_rows && row_ptr[r1 + 1] == p0 + end) tab[end] = r1 + 1;
    }
    if (__builtin_expect(nnz - p0 <= n, 0) && lane == 0) tab[nnz - p0] = n_rows;
    __builtin_amdgcn_wave_barrier();  // (LDS operations of one wave complete in order)
    int carry = 0;
    for (int i = 0; i < n_pad; i += 64) {
        const int v = max(wave_max_scan(tab[i + lane]), carry);
        tab[i + lane] = v;
        carry = __builtin_amdgcn_readlane(v, 63);
    }
    if (lane == 0) tab[n_pad] = max(tab[n_pad], carry);
    __builtin_amdgcn_wave_barrier();
    return r0;
}

// Lane slot of a row of K >= 4 floats read in pieces of four, when K is no multiple of the lanes' pieces: piece
// `slot` starts at float min(4 slot, K - 4), and only its elements from `first` on are new (4: none of them).
struct RowPiece {
    int off, first;
};
__device__ __forceinline__ RowPiece row_piece(int slot, int K)
{
    RowPiece r;
    r.off = min(4 * slot, K - 4);
    r.first = min(4, 4 * slot - r.off);
    return r;
}

}  // namespace sddmm
