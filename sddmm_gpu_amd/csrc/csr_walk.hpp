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

// The row that holds nonzero p (0 <= p < row_ptr[n_rows], uniform), by the whole wave: 64 probes a round, so three
// rounds of one load each for a quarter of a million rows where a binary search is a chain of eighteen.
__device__ __forceinline__ int wave_find_row(const int32_t *__restrict__ row_ptr, int n_rows, int p, int lane)
{
    int lo = 0, hi = n_rows;  // row_ptr[lo] <= p < row_ptr[hi]
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
// r0 = the row of p0.  tab[n] becomes the row of nonzero p0 + n, or n_rows where the nonzeros end there.
// (Entries past the last nonzero hold n_rows.)  The row starts inside the range are marked, one coalesced read of
// the row pointers for 64 rows, and a running maximum fills the rest; of the rows that start at one nonzero (empty
// ones) the last counts.
__device__ __forceinline__ void rows_of_range(const int32_t *__restrict__ row_ptr, int n_rows, int r0, int p0, int n, int *tab, int lane)
{
    const int n_pad = (n + 63) & ~63;
    for (int i = lane; i <= n_pad; i += 64) tab[i] = 0;
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) tab[0] = r0;
    __builtin_amdgcn_wave_barrier();
    for (int base = r0 + 1; base <= n_rows; base += 64) {
        const int r = base + lane;
        const int rel = r <= n_rows ? row_ptr[r] - p0 : INT32_MAX;
        const int next = __shfl_down(rel, 1);
        if (rel <= n && (rel != next || lane == 63)) tab[rel] = r;
        if (__builtin_amdgcn_readlane(rel, 63) > n) break;
    }
    __builtin_amdgcn_wave_barrier();  // (LDS operations of one wave complete in order)
    int carry = 0;
    for (int i = 0; i < n_pad; i += 64) {
        const int v = max(wave_max_scan(tab[i + lane]), carry);
        tab[i + lane] = v;
        carry = __builtin_amdgcn_readlane(v, 63);
    }
    if (lane == 0) tab[n_pad] = max(tab[n_pad], carry);
    __builtin_amdgcn_wave_barrier();
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
