// What the planner, the launch code and the plan files of libsddmm_hip.so share: a plan, its launches,
// and the functions that build them.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <memory>
#include <mutex>
#include "internal.hpp"
#include "kernels.hpp"

#define HIP_TRY(expr)                                                                               \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess)                                                                       \
            return sddmm::fail(SDDMM_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

// One kernel launch of a plan.  A plan is a list of launches over disjoint
// sets of rows; together they write every nonzero's output exactly once.
struct Launch {
    int kind = 0;            // SDDMM_KERNEL_ROW_GATHER / LDS_TILE / PANEL
    sddmm::KernelFn fn = nullptr;   // stream kernels
    sddmm::PanelFn pfn = nullptr;   // panel kernel
    sddmm::TileFn tfn = nullptr;        // tile kernel (values in stream order, first K slice); null: not a tile launch
    sddmm::TileFn tfns[5][5] = {};      // [values in stream order / in sorted order / none / residual epilogue with values
                                 //  in stream order / in sorted order][the only K slice / first of several / a later one /
                                 //  all slices inside one launch (null: no such variant)]
    sddmm::KArgs ka{};
    sddmm::PanelArgs pa{};
    sddmm::TileArgs ta{};
    sddmm::DenseFn dfn = nullptr;       // dense-block kernel; null: not a dense launch
    sddmm::DenseArgs da{};
    sddmm::BlockFn bfns[2] = {};        // row-block kernel, without and with the row softmax; null: not a row-block launch
    sddmm::BlockArgs ba{};
    int32_t softmax_waves = 0;          // waves per workgroup of the form with the softmax
    float *sval = nullptr;        // the plan's values in stream order (launches that walk a permuted stream)
    const int32_t *perm = nullptr;  // stream position -> sorted position of that launch (null: identity)
    int32_t grid = 0, block = 0, lds = 0, k_slice = 0;
    int32_t tile_g = 0, gather_g = 8;
    int64_t nnz = 0, rows = 0, positions = 0;
    int64_t longest_row = 0;  // most nonzeros in a row of S (the same for all launches of a plan)
    // what the function pointers above were looked up with (they are looked up again when a saved plan is loaded)
    int32_t fn_kind = 0;  // 1 stream kernel (row gather), 2 stream kernel with an LDS tile, 3 tile kernel, 4 panel, 5 dense,
                          // 6 row blocks
    int32_t fn_g = 0, fn_kpl = 0, fn_exact = 0, fn_gather = 0, fn_nwaves = 0;
    int32_t fn_once = 0, fn_wide = 0;  // row gather: the kernel with one batch of 64 a wave; W or H beyond 32-bit byte offsets
    int32_t fn_ragged = 0;  // tile kernel: the form for ranks that are no multiple of its width
    int32_t fn_nwm = 0;  // tile kernel: waves per workgroup that run the launch's matrix-core share (0: none)
    int32_t fused_slices = 0;  // sliced tile launch small enough that its K slices run inside one kernel launch
    // Scratch memory of the launch (partial results between K slices; packed operands of the matrix-core share):
    // sizes, and where each lies in a caller's workspace (sddmm_execute_ws); the plan's own copies are in ta
    int64_t part_bytes = 0, hp_bytes = 0, wp_bytes = 0;
    int64_t ws_part = 0, ws_hp = 0, ws_wp = 0;
    // the product Y = X H (spmm_stream = 1): sp_on == 1 on this launch's tiles, 2 over the plan's CSR pattern with records
    // in sa.part (see add_tile), 3 on the row blocks, 0 not built
    sddmm::SpmmArgs sa{};
    int32_t sp_on = 0, sp_grid = 0, sp_nwaves = 16;  // (16 waves per workgroup: 1.54 against 1.59 ms with 12 on the recommender shape)
    int64_t sp_part_bytes = 0, ws_sp_part = 0;
};

namespace sddmm {
struct HostCall;  // host_call.hip
struct HostCallDelete { void operator()(HostCall *c) const; };
}  // namespace sddmm

struct sddmm_plan {
    sddmm_plan_info info{};
    std::vector<Launch> launches;
    struct Owned { void *p; size_t bytes; bool scratch = false; };  // scratch: contents need not be kept (plan files)
    std::vector<Owned> owned;   // device allocations freed with the plan (sizes kept for sddmm_plan_save)
    uint64_t pattern_hash = 0;  // of the CSR pattern the plan was built for (see pattern_hash_host)
    const int32_t *d_row_ptr = nullptr, *d_col = nullptr;
    float *d_val = nullptr;
    int32_t requested_kernel = 0;
    int64_t ws_softmax = 0, ws_bytes = 0;  // workspace layout: the launches' scratch, then the softmax pass's records
    sddmm_plan_options options{};  // what the plan was built with, environment overrides applied
    mutable std::mutex host_mu;    // sddmm_gpu: one call at a time, with the device arrays it keeps
    mutable std::unique_ptr<sddmm::HostCall, sddmm::HostCallDelete> host_call;
    mutable std::atomic<int64_t> host_bytes{0};  // size of those arrays
    ~sddmm_plan()
    {
        for (const Owned &o : owned) (void)hipFree(o.p);
    }
};

namespace sddmm {

constexpr size_t kStreamSlack = 5120;  // readable entries behind a tile stream's arrays: 16 waves' batches of 64, up to four ahead and one more

// (the word mixer of the pattern hash and of the plan files' checksums)
__host__ __device__ inline uint64_t mix64(uint64_t x)
{
    x ^= x >> 33; x *= 0xff51afd7ed558ccdull; x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ull; x ^= x >> 33;
    return x;
}

template <class T, class A>
int upload(T **dst, const std::vector<T, A> &src, int64_t *bytes)
{
    *dst = nullptr;
    if (src.empty()) return SDDMM_OK;
    HIP_TRY(hipMalloc((void **)dst, src.size() * sizeof(T)));
    HIP_TRY(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    *bytes += (int64_t)(src.size() * sizeof(T));
    return SDDMM_OK;
}

// Everything the launch builders need.
struct Ctx {
    sddmm_plan *P;
    int64_t n_rows, n_cols, nnz;
    const int32_t *row_ptr, *col_ind;  // host CSR
    const float *vals;                 // host values (indexed by position in the original S) or null
    int32_t K;
    int cus;
    int64_t dev_bytes = 0;
    // The CSR above may be what is left of S after the dense blocks were cut out; orig then maps
    // its positions to positions in the original S (null: the CSR is S itself).  Streams record
    // original positions: that is where outputs go and where values come from.
    const int32_t *orig = nullptr;
    sddmm_plan_options opt{};  // the caller's options with the environment overrides applied
    int64_t sp_min_row = 0;    // the product on column tiles: rows of fewer nonzeros gather their H rows
    bool sp_walk = false;      // the product over the CSR pattern whatever the runs of the tile launch
    int32_t pos(int64_t p) const { return orig ? orig[p] : (int32_t)p; }
    float value(int64_t p) const { return vals[orig ? orig[p] : p]; }

    template <class T, class A>
    int up(T **dst, const std::vector<T, A> &src)
    {
        int rc = upload(dst, src, &dev_bytes);
        if (rc == SDDMM_OK && *dst) P->owned.push_back({(void *)*dst, src.size() * sizeof(T)});
        return rc;
    }
    int need_row_ptr()
    {
        if (P->d_row_ptr) return SDDMM_OK;
        int32_t *d = nullptr;
        HIP_TRY(hipMalloc((void **)&d, (size_t)(n_rows + 1) * 4));
        P->owned.push_back({d, (size_t)(n_rows + 1) * 4});
        HIP_TRY(hipMemcpy(d, row_ptr, (size_t)(n_rows + 1) * 4, hipMemcpyHostToDevice));
        dev_bytes += (n_rows + 1) * 4;
        P->d_row_ptr = d;
        return SDDMM_OK;
    }
};

struct DenseBlocks;

// planner.hip
int device_ok();
void default_options(sddmm_plan_options &o);
void apply_env_overrides(sddmm_plan_options &o);  // the environment as an override layer over the caller's options
int resolve_functions(Launch &L);  // looks the launch's kernels up from its descriptor and allows them its LDS size
uint64_t pattern_hash_host(int64_t n_rows, int64_t nnz, const int32_t *row_ptr, const int32_t *col_ind);
int pattern_hash_device(int64_t n_rows, int64_t nnz, const int32_t *d_row_ptr, const int32_t *d_col_ind, uint64_t *out);
void build_batches(const std::vector<WorkItem> &items, const int32_t *seg_end, int64_t n_seg, std::vector<int32_t> &batch_seg,
                   std::vector<uint64_t> &batch_mask);
int64_t list_nnz(const Ctx &c, const std::vector<int32_t> &rows);
int add_row_gather(Ctx &c, const std::vector<int32_t> &rows, bool all_rows);
void assign_workspace(sddmm_plan *P);
int make_plan(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *row_ptr_all, const int32_t *col_ind_all,
              const float *vals, const int32_t *d_row_ptr_borrowed, const int32_t *d_col_borrowed, int32_t K,
              const sddmm_plan_options &opt_in, sddmm_plan **out);
// Is the product with the dense factor, behind a plan of a matrix of this size (tile slices of ks elements), a walk over
// the CSR pattern whatever the runs (see add_tile)?  From 4 million nonzeros on the rows are split by length, and tiles that
// hold long rows only are the faster ones; so they are when the walk, at 17 TB/s, has more than 1.8 GB of H rows to read,
// 2.8 where the tiles take slices of 64 (tiles against walk, ratings of 1.8, 2.4 and 3.6 M, K = 256: 108 / 101, 123 / 139 and
// 167 / 190 us; of 2.6 and 3.8 M, K = 192: 148 / 131 and 180 / 184; K = 320, 1.8 and 2.6 M: 231 / 171 and 240 / 259).  The walk's times from
// K = 192 on are those before it took slices of H; with them it is faster up to more nonzeros (ratings of 1.2 M, K = 384 120 / 82).
inline bool product_walks(int64_t nnz, int32_t K, int ks) { return nnz < 4000000 && nnz * K < (ks < 128 ? 700000000 : 450000000); }
// And at a rank that is no multiple of the tiles' width ks, which they work on up to the next multiple?  From 4 million nonzeros
// on, where little of that is padding (SDDMM + product, us, walk and tiles: ratings of 4.9 M, K = 20 / 36 / 50 / 75 / 120 68 / 95
// / 102 / 160 / 179 and 73 / 90 / 92 / 143 / 153, K = 150 / 180 / 200 / 250 / 300 / 380 274 / 285 / 313 / 368 / 577 / 624 and 282 /
// 290 / 293 / 305 / 441 / 457; 15.9 M, K = 50 / 120 / 150 / 200 / 300 257 / 506 / 780 / 964 / 2118 and 215 / 422 / 791 / 829 / 1250);
// below, where the walk has three slices or more (3.3 M, K = 200 / 220 / 250 / 280 / 340: 208 / 218 / 240 / 387 / 402 and 248 /
// 250 / 253 / 365 / 370).  And not at a width of 32: the work is little and the longest run, which eight lanes walk alone, sets
// the time (K = 28, product alone, ratings of 4.2 and 5.1 M 45 / 65 and 53 / 51, word counts of 5.9 and 7.4 M 57 / 72 and 69 / 75).
inline bool ragged_product_tiles(int64_t nnz, int32_t K, int ks)
{
    const int padded = (K + ks - 1) / ks * ks;
    return nnz < 4000000 ? K > 256 && !product_walks(nnz, K, ks) : K > 32 && (K <= 128 || K * 100 >= padded * 72);
}
// The runs it takes for that, in nonzeros per run on average: a run costs a partial row of the padded width, its nonzeros cost
// the walk K elements each.  So the line is one of run length times the used share of the width.  It is drawn on SDDMM + product
// one after the other: a product alone finds its partial rows in the caches, behind an SDDMM it does not (ratings of 4.9 M, K = 187:
// 184 / 172 alone and 302 / 336 together).  us, walk and tiles at (that figure):
//   width 64: uniform, 5.4 / 9.0 M, K = 55 100 / 89 (14.9), 155 / 138 (17.0), 11.4 M 252 / 198 (13.7); up to K = 48, whose rows are few
//       lines each to the walk, ratings of 5.1 M, K = 34 88 / 82 (18.1), and, product alone, with an H of more than 2.5 MB word counts of
//       8.9 M, K = 40 / 48 111 / 129 (15.0), 113 / 130 (18.0), with a smaller one of 7.4 M, K = 48 82 / 92 (14.4)
//   width 128: ratings of 4.5 / 5.6 / 7.3 M, K = 84 / 75 / 78 140 / 137 (10.7), 168 / 158 (10.6), 199 / 192 (12.5); of 8.2 / 11.8 / 12.3 M, K =
//       69 / 75 / 90 216 / 234 (9.5), 307 / 325 (12.5), 323 / 343 (14.8), 8.7 M, K = 89 235 / 227 (15.6); an H of more than 4.5 MB, word
//       counts of 6.1 / 4.4 M, K = 125 / 124 282 / 230 (11.9), 172 / 141 (13.2), 7.5 / 9.7 M, K = 110 / 92 360 / 359 (14.1), 388 / 408
//   two slices: ratings of 4.9 M, K = 195 / 200 303 / 315 (14.4), 299 / 298 (15.1), 5.9 M, K = 208 362 / 341 (16.8); uniform, 4.4 M, K = 189
//       222 / 257 (11.3); an H of more than 6 MB, word counts of 19 M, K = 238 2441 / 1634 (11.5), 5.5 M, K = 252 664 / 539 (12.8)
//   more: word counts of 4.1 / 12.8 M, K = 337 / 518 737 / 775 (7.3), 4600 / 3341 (7.3); below 4 M nonzeros, ratings of 2.9 M, K = 286
//       338 / 324 (10.1), 2.2 M, K = 352 / 357 259 / 265 (11.3), 275 / 266 (11.5), word counts of 3.0 M, K = 369 478 / 350 (10.9), and with
//       four slices and an H of up to 11 MB ratings of 2.9 / 3.2 M, K = 418 / 488 384 / 434 (10.6), 473 / 512 (12.4), uniform, 3.8 M, K =
//       496 428 / 472 (13.2), but H of 12.5 MB, 3.3 M, K = 450 630 / 409 (10.4)
// (The tiles have become 2 to 20 % faster since; of 302 pairs the slower form is taken by more than 5 % in 44, a walk in 39 of them:
// profiles/product_pairs_ragged.txt.)
inline double ragged_product_run(int64_t nnz, int64_t n_cols, int32_t K, int ks)
{
    const double padded = (K + ks - 1) / ks * ks, h = 4.0 * n_cols * K;
    double least;
    if (ks < 128) least = K > 48 ? 13.5 : h <= 2.5e6 ? 15.0 : 19.0;
    else if (K <= 128) least = nnz < 7500000 ? (h <= 4.5e6 ? 10.5 : 11.8) : h <= 4.5e6 ? 15.0 : 14.0;
    else if (K <= 256) least = h <= 6.0e6 ? 15.5 : 11.0;
    else if (nnz < 4000000) least = K > 384 && h <= 11.0e6 ? 16.0 : 10.0;
    else least = nnz < 6000000 ? 9.0 : 7.0;
    return least * padded / K;
}
// planner_tile.hip: the rows' nonzeros in tile order (tiles of x columns), every (row, tile) run padded
// ks: K elements per launch, a divisor of K or (ragged ranks) the width K is rounded up to
int add_tile(Ctx &c, const std::vector<int32_t> &rows_in, int32_t x, int32_t panel_rows, int want_g, int ks,
             sddmm_plan_info *I, bool gather = false, bool x_explicit = false);
// planner_block.hip: all of S on the row-block kernels, where that pays (*taken)
int add_blocks(Ctx &c, const std::vector<int32_t> &rows, bool *taken);
}  // namespace sddmm
