// Padded gather with groups of 4 positions: the stream of the tile kernel's gather form (H rows read from global memory),
// every (row, column slab) run padded to a multiple of 4, for patterns whose runs are short.
#include "kernels_tile_impl.hpp"

namespace {

// Eight lanes work on eight consecutive positions -- two groups, so up to two rows of W -- one position a step, and read a
// whole 128-byte line of its H row per request, KPL lines for a K slice of 32 KPL elements.  (With four lanes to a group
// and position, which a group of 4 suggests, a request takes half of each of 16 lines and the next one the other half:
// by then the line may have left the compute unit's 32 KB of L1, and where rows come from L2 and beyond in turn that
// costs bandwidth.  Random rows of 256 bytes, 57 % of them from 2 MB and the others from 1 GB: 10.8 TB/s by halves, 11.9
// by lines.)  What bounds it is the fabric (7.2 TB/s for rows that miss L2) together with the load path (28 TB/s for those
// that do not): on R-MAT 2^22, K = 64, 43 % of 60 GB of rows cross the fabric.
// us per product, with four lanes and so: R-MAT 2^22, 185 million nonzeros, K = 64 4896 and 4541; 2^20, K = 64 (28 million) 645 and
// 590, K = 128 (70 million) 2800 and 2741, K = 512 (33 million) 6457 and 6280; 2^18, 12 million, K = 128 466 and 446; uniform, 20
// million of 100,000 columns, K = 64 / 128 419 / 713 and 375 / 703 (all with 2048 positions a workgroup, which the planner chooses
// from 32 million on; below it takes 1024, see there): 1024 / 4096 / 8192 / 16384 on the first 4509 / 4419 / 4506 / 4763 where 2048
// takes 4415; neighbouring workgroups bound to one die, 4 to 1024 at a time: 4398 to 4453; four steps' pieces at a time instead of
// eight: the same.
// VMODE, SLICE: as in the tile kernel.  (SLICE 3, all K slices inside one launch: a wave's partial results are its own.)
template <int KPL, int VMODE, int SLICE>
__global__ __launch_bounds__(256)
void sddmm_slab_gather_kernel(const TileArgs a)
{
    constexpr int L = 8, G = 4, NW = 4;
    constexpr int ROUND = KPL <= 2 ? 8 : 4;  // steps whose pieces of H are requested together
    constexpr bool FUSED = SLICE == 3, ACC = SLICE == 2 || SLICE == 4, PART = SLICE >= 1, TO_OUT = SLICE == 0 || SLICE >= 3;
    constexpr bool RESIDUAL = VMODE >= 3, STREAM_VAL = VMODE == 0 || VMODE == 3, SORTED_VAL = VMODE == 1 || VMODE == 4;
    static_assert(TO_OUT || VMODE == 2);
    const int lane = threadIdx.x & 63, l = lane & (L - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the slabs follow each other in the stream: a workgroup takes an equal range of positions, a wave an equal part of its batches
    const int64_t total = a.unit_ptr[a.n_units];
    const int64_t lo = ((total * blockIdx.x / gridDim.x) + 63) & ~(int64_t)63;
    const int64_t hi = blockIdx.x + 1 == gridDim.x ? total : ((total * (blockIdx.x + 1) / gridDim.x) + 63) & ~(int64_t)63;
    const int nb = (int)((hi - lo + 63) >> 6);
    const int b0 = __builtin_amdgcn_readfirstlane(nb * wave / NW);
    const int b1 = __builtin_amdgcn_readfirstlane(nb * (wave + 1) / NW);
    if (b0 >= b1) return;
    const int32_t *perm = a.perm + lo, *scol = a.scol + lo, *grow = a.grow + lo / G;
    const float *sval = a.sval + lo;
    float *part = a.part + lo;
    const uint32_t last = (uint32_t)(total - 1 - lo);  // the stream's last position, counted from lo

    const int n_slices = FUSED ? a.n_slices : 1;
    for (int sl = 0; sl < n_slices; ++sl) {
    const bool first_slice = sl == 0, last_slice = sl + 1 == n_slices;  // (used by the FUSED form only)
    const float4 *__restrict__ W4 = reinterpret_cast<const float4 *>(a.W) + ((a.k_off >> 2) + sl * L * KPL + l);
    const float4 *__restrict__ H4 = reinterpret_cast<const float4 *>(a.H) + ((a.k_off >> 2) + sl * L * KPL + l);
    if (FUSED && sl > 0) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // the partial results before are stored

    // Index data of one batch: lanes past the end of the stream repeat its last position, and their results are dropped
    // like those of padding; what is requested past a wave's range is dropped.
    struct Meta { uint32_t wrow, p, o; int col; float sv, old; };
    uint32_t at = (uint32_t)(b0 << 6) + (uint32_t)lane;
    auto issue_meta = [&]() -> Meta {
        Meta m;
        m.o = min(at, last);
        m.wrow = (uint32_t)grow[m.o / G];
        if constexpr (TO_OUT) m.p = (uint32_t)perm[m.o] | (at > last ? 0x80000000u : 0u);
        m.col = scol[m.o];
        m.sv = STREAM_VAL ? sval[m.o] : 1.0f;
        at += 64;
        return m;
    };
    // (FUSED: the slot is read in every slice and ignored in the first: no load behind a branch)
    auto issue_old = [&](Meta &m) {
        m.old = ACC || FUSED ? part[m.o] : 0.f;
        if constexpr (FUSED) m.old = first_slice ? 0.f : m.old;
    };
    // both rows' pieces: lanes 0 to 3 of the eight hold the first group's row, lanes 4 to 7 the second one's
    auto issue_w = [&](float4 (&w)[2][KPL], uint32_t wrow) {
        const uint32_t other = (uint32_t)from_lane_xor<4>((int)wrow);
        const float4 *r0 = W4 + (l < 4 ? wrow : other), *r1 = W4 + (l < 4 ? other : wrow);
#pragma unroll
        for (int j = 0; j < KPL; ++j) w[0][j] = r0[j * L];
#pragma unroll
        for (int j = 0; j < KPL; ++j) w[1][j] = r1[j * L];
    };
    float pend_v;  // result of the batch before, not yet stored
    uint32_t pend_p, pend_o;
    auto flush = [&]() {
        float *dst;
        if constexpr (!TO_OUT) dst = part + pend_o;
        else dst = (int32_t)pend_p < 0 ? a.sink + (((blockIdx.x & 255) << 6) + lane) : a.out + pend_p;
        if constexpr (FUSED) dst = last_slice ? dst : part + pend_o;
        *dst = pend_v;
    };
    auto compute = [&](const float4 (&w)[2][KPL], const Meta &m) {
        float v = m.sv;
        if constexpr (SORTED_VAL) v = a.val[m.p & 0x7fffffffu];
        int c[L];
        columns_of_steps<L, false>(m.col, 0, c);
        float acc[L];
        auto round = [&]<int BASE, int... I>(std::integer_sequence<int, BASE>, std::integer_sequence<int, I...>) {
            float4 h[ROUND][KPL];
            ((void)[&] {
                const float4 *hr = H4 + (uint32_t)c[BASE + I];
#pragma unroll
                for (int j = 0; j < KPL; ++j) h[I][j] = hr[j * L];
            }(), ...);
            __builtin_amdgcn_sched_barrier(0);
            ((void)[&] {
                float s = 0.f;
#pragma unroll
                for (int j = 0; j < KPL; ++j) s = dot4(w[(BASE + I) / G][j], h[I][j], s);
                acc[BASE + I] = s;
            }(), ...);
        };
        [&]<int... R>(std::integer_sequence<int, R...>) {
            (round(std::integer_sequence<int, R * ROUND>{}, std::make_integer_sequence<int, ROUND>{}), ...);
        }(std::make_integer_sequence<int, L / ROUND>{});
        const Halves d = transpose_reduce<L, false>(acc, l);
        if constexpr (!PART) {
            pend_v = RESIDUAL ? v - (d.x + d.y) : (d.x + d.y) * v;
        } else if constexpr (SLICE == 1) {
            pend_v = d.x + d.y;
        } else {
            const Halves sum = add_to(m.old, d, (l & 1) != 0);
            if constexpr (SLICE == 2) pend_v = sum.x + sum.y;
            else pend_v = RESIDUAL ? (v - (d.x + d.y)) - m.old : VMODE == 2 ? sum.x + sum.y : fmaf(sum.x, v, sum.y * v);
            if constexpr (FUSED) pend_v = last_slice ? pend_v : sum.x + sum.y;
        }
        if constexpr (TO_OUT) pend_p = m.p;
        pend_o = m.o;
    };

    float4 wa[2][KPL], wb[2][KPL];
    Meta m0 = issue_meta(), m1 = issue_meta();
    issue_old(m0);
    issue_w(wa, m0.wrow);
    for (int bi = b0; bi < b1; bi += 2) {
        if (bi > b0) flush();
        Meta m2 = issue_meta();  // batch bi + 2
        issue_old(m1);
        issue_w(wb, m1.wrow);
        __builtin_amdgcn_sched_barrier(0);  // keep the requests ahead of the arithmetic
        compute(wa, m0);
        if (bi + 1 >= b1) break;
        flush();
        const Meta m3 = issue_meta();  // batch bi + 3
        issue_old(m2);
        issue_w(wa, m2.wrow);
        __builtin_amdgcn_sched_barrier(0);
        compute(wb, m1);
        m0 = m2;
        m1 = m3;
    }
    flush();
    }
}

template <int KPL, int VMODE>
TileFn slab_gather(int slice)
{
    if (slice == 0) return (TileFn)sddmm_slab_gather_kernel<KPL, VMODE, 0>;
    if constexpr (KPL == 4)
        if (slice == 3) return (TileFn)sddmm_slab_gather_kernel<KPL, VMODE, 3>;
    if (slice == 4) return (TileFn)sddmm_slab_gather_kernel<KPL, VMODE, 4>;
    if constexpr (VMODE == 2) {
        if (slice == 1) return (TileFn)sddmm_slab_gather_kernel<KPL, VMODE, 1>;
        if (slice == 2) return (TileFn)sddmm_slab_gather_kernel<KPL, VMODE, 2>;
    }
    return nullptr;
}

}  // namespace

namespace sddmm {

TileFn slab_gather_kernel(int k_slice, int vmode, int slice)
{
#define SDDMM_CASE(w)                                       \
    if (k_slice == w) switch (vmode) {                      \
        case 0: return slab_gather<w / 32, 0>(slice);       \
        case 1: return slab_gather<w / 32, 1>(slice);       \
        case 2: return slab_gather<w / 32, 2>(slice);       \
        case 3: return slab_gather<w / 32, 3>(slice);       \
        case 4: return slab_gather<w / 32, 4>(slice);       \
        }
    SDDMM_CASE(32) SDDMM_CASE(64) SDDMM_CASE(128)
#undef SDDMM_CASE
    return nullptr;
}

}  // namespace sddmm
